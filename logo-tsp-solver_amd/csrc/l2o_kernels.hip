// l2o_kernels.hip -- gfx950 kernels around the sweep (l2o_sweep.hip): move
// application, ILS bookkeeping, multi-start rounds, tour length.
//
// Replaces the host-side apply of the reference
// (src/solvers/twoOptLocalSolver.cpp:40-50) and its ILS loops.
#include <hip/hip_runtime.h>

#include "l2o_device.h"

namespace l2o {

// ---------------------------------------------------------------------------
// the end of a run of sweeps (l2o_state.h), or of one by itself (run = 0):
// apply the last one's move
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(L2O_APPLY_THREADS) void k_apply(const l2o_apply_item *__restrict__ items,
                                                             l2o_inst *__restrict__ insts,
                                                             unsigned *__restrict__ live, uint32_t run)
{
    const uint32_t t = run ? run : 1;
    const l2o_apply_item it = items[blockIdx.x];
    l2o_inst *in = insts + it.inst;
    const __attribute__((address_space(4))) l2o_inst *ci = (const __attribute__((address_space(4))) l2o_inst *)in;
    const unsigned long long key = ci->key[(t - 1) & 3];
    const uint32_t phase = ci->phase, b = (ci->base + t - 1) & 1;
    const int n = (int)ci->n;
    if (phase != L2O_LO) return;
    if (key == L2O_SENTINEL) {
        // no improving move: the local search has converged (sweeps = moves + 1)
        if (it.chunk == 0 && threadIdx.x < 64) local_optimum(in, live, b);
        return;
    }
    const move_map mm(key, n);
    // wave 0: the pool entries on the new tour (stored by the last chunk)
    static_assert(L2O_POOL == 64, "one lane per pool entry");
    unsigned long long *const pool = ci->pool;
    unsigned long long pk = L2O_SENTINEL;
    if (threadIdx.x < L2O_POOL) {
        pk = pool[((t - 1) & 3) * L2O_POOL + threadIdx.x];
        if (!run) pk = min(pk, pool[3 * L2O_POOL + threadIdx.x]);  // (a run's sweeps carry it over)
    }
    copy_chunk<L2O_APPLY_THREADS>(ci, b, mm, ci->metric, (int)(it.chunk * L2O_APPLY_CHUNK));
    pk = remap_key(pk, (uint32_t)mm.i, (uint32_t)mm.J, (uint32_t)n);
    const int cap = next_cap(pk, 0, (uint32_t)n);
    asm volatile("" ::"s"(cap));  // the pool loads have returned before the barrier
    // Every wave of the workgroup has read key, base and its sources once all
    // are past the barrier (each loaded value feeds a store issued before it),
    // so the last chunk to count may commit the move.  No memory fence: nothing
    // in this kernel reads the new buffers, and the next kernel sees them at the
    // kernel boundary; the empty asm keeps the compiler from moving memory
    // operations across the barrier.
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (threadIdx.x < 64) {
        const uint32_t nch = ((uint32_t)n + L2O_APPLY_CHUNK - 1) / L2O_APPLY_CHUNK;
        uint32_t prev = 0;
        if (threadIdx.x == 0) prev = atomicAdd(&in->apply_done, 1u);
        prev = (uint32_t)__builtin_amdgcn_readfirstlane((int)prev);
        if (prev != nch - 1) return;
        pool[3 * L2O_POOL + threadIdx.x] = pk;
        pool[threadIdx.x] = L2O_SENTINEL;
        if (threadIdx.x == 0) {
            in->apply_done = 0;
            in->parity = in->base = b ^ 1;
            in->cap = cap;
            if (key != L2O_KEY_NONE) log_move(in, key);
            in->key[3] = L2O_KEY_NONE;
            in->key[0] = L2O_SENTINEL;
        }
    }
}

// ---------------------------------------------------------------------------
// ILS bookkeeping: accept/revert, kick, restart (ILSGlobalSolverSequential.cpp:73-99)
// ---------------------------------------------------------------------------
// A plain ILS instance at L2O_LO_DONE: accept iff strictly shorter (copy to
// the best buffers), stop after `rounds` or once the best length is below
// stop_below, else kick its best and restart.
// A chain of a multi-start group at L2O_LO_DONE only accepts into its own best
// and waits (L2O_WAIT) for k_group; at L2O_KICK it kicks the best tour of
// `kick_src` that k_group chose.  While any chain of a group is at L2O_KICK,
// all of them are, so no best buffer is written while a kick reads it.
// The kicked tour goes where the run's next sweep, tnext, reads it.
__global__ __launch_bounds__(L2O_ILS_THREADS) void k_ils(l2o_inst *__restrict__ insts, unsigned *__restrict__ live,
                                                         uint32_t tnext)
{
    l2o_inst *in = insts + blockIdx.x;
    const uint32_t phase = in->phase;
    if (phase != L2O_LO_DONE && phase != L2O_KICK) return;
    const bool grouped = in->group_lead != L2O_NO_GROUP;
    __shared__ int s_accept, s_done;
    __shared__ uint32_t s_a, s_b, s_c;
    __shared__ unsigned long long s_sum[L2O_ILS_THREADS / 64];
    const uint32_t n = in->n;
    const uint32_t par = in->parity;
    if (threadIdx.x == 0) {
        int acc = 0, done = 0;
        if (phase == L2O_LO_DONE) {
            acc = !in->have_best || in->length < in->best_length;
            if (acc) {
                in->best_length = in->length;
                in->have_best = 1;
            }
            if (grouped) {
                in->improved = acc;
            } else {
                if (in->rlog) in->rlog[in->rounds_done] = in->best_length;
                done = in->rounds_done >= in->ils_rounds || in->best_length < in->stop_below;
            }
        }
        s_accept = acc;
        s_done = done;
        if (!done && (phase == L2O_KICK || !grouped)) {
            uint32_t cut[3];
            draw_kick(in->rng, in->kick, n, cut);
            s_a = cut[0];
            s_b = cut[1];
            s_c = cut[2];
        }
    }
    __syncthreads();
    if (s_accept) {
        const l2o_pt *__restrict__ P = in->pts[par];
        const uint32_t *__restrict__ R = in->tour[par];
        l2o_pt *__restrict__ BP = in->bpts;
        uint32_t *__restrict__ BR = in->btour;
        for (uint32_t k = threadIdx.x; k < n; k += L2O_ILS_THREADS) {
            BP[k] = P[k];
            BR[k] = R[k];
        }
    }
    __syncthreads();
    if (grouped && phase == L2O_LO_DONE) {
        if (threadIdx.x == 0) {
            __threadfence();
            in->phase = L2O_WAIT;
        }
        return;
    }
    if (s_done) {
        if (threadIdx.x == 0) {
            in->phase = L2O_DONE;
            atomicSub(live, 1u);
        }
        return;
    }
    // new current tour = kick(best of the source), written to the next sweep's buffer
    const l2o_inst *src = grouped ? insts + in->kick_src : in;
    const l2o_pt *__restrict__ BP = src->bpts;
    const uint32_t *__restrict__ BR = src->btour;
    const uint32_t a = s_a, b = s_b, c = s_c;
    const bool ref = in->kick == 1;
    auto src_of = [&](uint32_t k) -> uint32_t { return kick_source(k, n, ref, a, b, c); };
    const uint32_t nb = (in->base + (tnext ? tnext - 1 : 0)) & 1;
    l2o_pt *__restrict__ Pn = in->pts[nb];
    uint32_t *__restrict__ Rn = in->tour[nb];
    const uint32_t metric = in->metric;
    unsigned long long sum = 0;
    for (uint32_t k = threadIdx.x; k < n; k += L2O_ILS_THREADS) {
        const uint32_t s = src_of(k);
        const uint32_t sp = src_of(k == 0 ? n - 1 : k - 1);
        const l2o_pt p = BP[s], q = BP[sp];
        const int d = exact_dist(q.x, q.y, p.x, p.y, metric);
        sum += (unsigned long long)d;
        l2o_pt r;
        r.x = p.x;
        r.y = p.y;
        r.d = d;
        r.w = p.w;
        Pn[k] = r;
        Rn[k] = BR[s];
    }
    sum = wave_sum_u64(sum);
    if ((threadIdx.x & 63) == 0) s_sum[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long L = 0;
        for (int k = 0; k < L2O_ILS_THREADS / 64; ++k) L += s_sum[k];
        in->length = L;
        in->parity = nb;
        in->cap = -1;
        in->rounds_done += 1;
        in->key[(tnext - 1) & 3] = L2O_KEY_NONE;
        in->key[tnext & 3] = L2O_SENTINEL;
        in->apply_done = 0;
        __threadfence();
        in->phase = L2O_LO;
    }
}

// ---------------------------------------------------------------------------
// Multi-start ILS round barrier: ILSGlobalSolverMT::optimize with comm = 1
// (ILSGlobalSolverMT.cpp:86-195) shares a global best between threads under a
// mutex, so its result depends on timing.  Here the chains of a group advance
// round by round: once every chain has reached its local optimum (L2O_WAIT),
// one thread per group takes the group best (smallest best length, lowest
// chain on ties), logs it, and sends each chain on with a kick of its own
// tour if that improved its best this round, else of the group best (the
// reference's "route = bestGlobalMinima.back()"); after `rounds` kicks every
// chain stops.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(64) void k_group(l2o_inst *__restrict__ insts, uint32_t nslots,
                                              unsigned *__restrict__ live)
{
    const uint32_t id = blockIdx.x * 64 + threadIdx.x;
    if (id >= nslots) return;
    l2o_inst *lead = insts + id;
    if (lead->group_lead != id || lead->phase != L2O_WAIT) return;
    const uint32_t m = lead->group_size;
    uint32_t best = id;
    for (uint32_t c = 0; c < m; ++c) {
        const l2o_inst *in = insts + id + c;
        if (in->phase != L2O_WAIT) return;  // not all chains are done with this round
        if (in->best_length < insts[best].best_length) best = id + c;
    }
    const unsigned long long G = insts[best].best_length;
    const uint32_t rounds = lead->rounds_done;
    const bool done = rounds >= lead->ils_rounds || G < lead->stop_below;
    for (uint32_t c = 0; c < m; ++c) {
        l2o_inst *in = insts + id + c;
        if (in->rlog) in->rlog[rounds] = G;
        in->kick_src = in->improved ? id + c : best;
        in->phase = done ? L2O_DONE : L2O_KICK;
    }
    if (done) atomicSub(live, m);
}

// ---------------------------------------------------------------------------
// admission and release of a slot.  Kernels that read and write pinned host
// memory, in place of copies: a copy of a few hundred bytes between launches
// takes longer than a launch does.
// ---------------------------------------------------------------------------
// host memory to HBM: an instance's record, and its coordinates by city (int32
// x, y) and start tour (n times 12 bytes) into its other point buffer
__global__ __launch_bounds__(256) void k_stage(l2o_inst *__restrict__ in, const l2o_inst *__restrict__ rec,
                                               uint4 *__restrict__ raw, const uint4 *__restrict__ host, uint32_t words)
{
    if (blockIdx.x == 0)
        for (uint32_t k = threadIdx.x; k < sizeof(l2o_inst) / 4; k += 256) ((uint32_t *)in)[k] = ((const uint32_t *)rec)[k];
    for (uint32_t k = blockIdx.x * 256 + threadIdx.x; k < words; k += gridDim.x * 256) raw[k] = host[k];
}

// the tour-ordered points of an admitted instance: coordinates, exact edge
// lengths, quantised coordinates; city ids and the tour's length.  Behind the raw
// cities each wave leaves the position of its longest edge's end (0: none).
__global__ __launch_bounds__(256) void k_load(l2o_inst *__restrict__ insts, uint32_t slot, unsigned *__restrict__ live,
                                              int count)
{
    l2o_inst *in = insts + slot;
    const int n = (int)in->n;
    const uint32_t metric = in->metric;
    const int2 *__restrict__ xy = (const int2 *)in->pts[1];
    const uint32_t *__restrict__ route = (const uint32_t *)(xy + n);
    l2o_pt *__restrict__ P = in->pts[0];
    uint32_t *__restrict__ R = in->tour[0];
    unsigned long long sum = 0, longest = ~0ull;
    for (int k = (int)(blockIdx.x * 256 + threadIdx.x); k < n; k += (int)gridDim.x * 256) {
        const uint32_t c = route[k], pc = route[k ? k - 1 : n - 1];
        const int2 a = xy[c], b = xy[pc];
        l2o_pt r;
        r.x = a.x;
        r.y = a.y;
        r.d = exact_dist(b.x, b.y, a.x, a.y, metric);
        r.w = quant_xy(in->qs, in->qox, in->qoy, a.x, a.y);
        sum += (unsigned long long)r.d;
        P[k] = r;
        R[k] = c;
        const unsigned long long e = (unsigned long long)(uint32_t)~r.d << 32 | (uint32_t)k;
        if (k && e < longest) longest = e;  // (edge 0 closes the tour: no candidate's)
    }
    sum = wave_sum_u64(sum);
    longest = wave_min_u64(longest);
    if ((threadIdx.x & 63) == 0)
        ((uint32_t *)(route + n))[blockIdx.x * 4 + (threadIdx.x >> 6)] = longest == ~0ull ? 0u : (uint32_t)longest;
    if ((threadIdx.x & 63) == 0 && sum) atomicAdd(&in->length, sum);
    if (count && blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(live, 1u);
}

// A cap for the first sweep of an instance: the best candidate between the `m`
// long edges k_load found, into in->cap.  The best move of a tour nearly always
// removes two of them, so the sweep's test passes little else.  Latency: three
// dependent loads, one exact gain per lane and turn.
__global__ __launch_bounds__(256) void k_prime(l2o_inst *__restrict__ insts, uint32_t slot, uint32_t m)
{
    l2o_inst *in = insts + slot;
    const uint32_t metric = in->metric;
    const l2o_pt *__restrict__ P = in->pts[0];
    const uint32_t *__restrict__ ends = (const uint32_t *)in->pts[1] + 3 * in->n;
    __shared__ int s_best;
    if (threadIdx.x == 0) s_best = -1;
    __syncthreads();
    const uint32_t q = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t ka = q < m ? ends[q] : 0u;
    int best = -1;
    if (ka) {
        const l2o_pt a0 = P[ka - 1], a1 = P[ka];
        for (uint32_t r = q + 1 + lane; r < m; r += 64) {
            const uint32_t kb = ends[r];
            if (kb == 0 || (kb < ka ? ka - kb : kb - ka) < 2) continue;  // edges with a common end
            const l2o_pt b0 = P[kb - 1], b1 = P[kb];
            best = min(best, exact_dist(a0.x, a0.y, b0.x, b0.y, metric) + exact_dist(a1.x, a1.y, b1.x, b1.y, metric) -
                                 a1.d - b1.d);
        }
    }
    if (best < -1) atomicMin(&s_best, best);
    __syncthreads();
    if (threadIdx.x == 0 && s_best < __hip_atomic_load(&in->cap, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMin(&in->cap, s_best);
}

// release of a slot: its record blank, its pool empty (`running`: it was live)
__global__ __launch_bounds__(256) void k_free(l2o_inst *__restrict__ insts, uint32_t slot, unsigned *__restrict__ live,
                                              int running, int clear_pool)
{
    l2o_inst *in = insts + slot;
    unsigned long long *const pool = in->pool;
    if (clear_pool) pool[threadIdx.x] = L2O_SENTINEL;  // 4 L2O_POOL entries
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < sizeof(l2o_inst) / 4; k += 256) ((uint32_t *)in)[k] = 0;  // L2O_FREE
    if (running && threadIdx.x == 0) atomicSub(live, 1u);
}

// an instance's record and result tour into host memory
__global__ __launch_bounds__(256) void k_fetch(const l2o_inst *__restrict__ insts, uint32_t slot,
                                               l2o_inst *__restrict__ rec, uint32_t *__restrict__ tour)
{
    const l2o_inst *in = insts + slot;
    if (blockIdx.x == 0)
        for (uint32_t k = threadIdx.x; k < sizeof(l2o_inst) / 4; k += 256) ((uint32_t *)rec)[k] = ((const uint32_t *)in)[k];
    if (!tour) return;
    const uint32_t *src = in->ils_rounds && in->have_best ? in->btour : in->tour[in->parity];
    for (uint32_t k = blockIdx.x * 256 + threadIdx.x; k < in->n; k += gridDim.x * 256) tour[k] = src[k];
}

// ---------------------------------------------------------------------------
// exact tour length of the current buffer: sum of D (headers.h:170-189)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_length(const l2o_inst *__restrict__ insts, uint32_t slot,
                                                unsigned long long *__restrict__ out)
{
    const l2o_inst *in = insts + slot;
    const l2o_pt *P = in->pts[in->parity];
    const uint32_t n = in->n;
    unsigned long long sum = 0;
    for (uint32_t k = blockIdx.x * 256 + threadIdx.x; k < n; k += gridDim.x * 256) {
        const l2o_pt p = P[k], q = P[k == 0 ? n - 1 : k - 1];
        sum += (unsigned long long)exact_dist(q.x, q.y, p.x, p.y, in->metric);
    }
    sum = wave_sum_u64(sum);
    if ((threadIdx.x & 63) == 0 && sum) atomicAdd(out, sum);
}

// ---------------------------------------------------------------------------
// v_sqrt_f32 accuracy: max |ulp| distance from the correctly rounded sqrt
// over float bit patterns [lo, hi)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_sqrt_ulp(uint32_t lo, uint32_t hi, unsigned *__restrict__ max_ulp)
{
    unsigned m = 0;
    for (unsigned long long b = (unsigned long long)lo + blockIdx.x * 256ull + threadIdx.x; b < hi;
         b += (unsigned long long)gridDim.x * 256ull) {
        const float x = __uint_as_float((uint32_t)b);
        const float hw = __builtin_amdgcn_sqrtf(x);
        const float cr = (float)sqrt((double)x);  // correctly rounded (sqrt is double-rounding safe)
        const int d = (int)__float_as_uint(hw) - (int)__float_as_uint(cr);
        const unsigned ad = (unsigned)(d < 0 ? -d : d);
        m = ad > m ? ad : m;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned o = __shfl_xor(m, off);
        m = o > m ? o : m;
    }
    if ((threadIdx.x & 63) == 0) atomicMax(max_ulp, m);
}

}  // namespace l2o

// ---------------------------------------------------------------------------
// launch wrappers used by the host engine
// ---------------------------------------------------------------------------
#include "l2o_launch.h"

namespace l2o {

hipError_t launch_apply(const l2o_apply_item *items, uint32_t nitems, l2o_inst *insts, unsigned *live, uint32_t t,
                        hipStream_t stream)
{
    if (nitems == 0) return hipSuccess;
    hipLaunchKernelGGL(k_apply, dim3(nitems), dim3(L2O_APPLY_THREADS), 0, stream, items, insts, live, t);
    return hipGetLastError();
}

hipError_t launch_ils(l2o_inst *insts, uint32_t nslots, unsigned *live, uint32_t tnext, hipStream_t stream)
{
    if (nslots == 0) return hipSuccess;
    hipLaunchKernelGGL(k_ils, dim3(nslots), dim3(L2O_ILS_THREADS), 0, stream, insts, live, tnext);
    return hipGetLastError();
}

hipError_t launch_group(l2o_inst *insts, uint32_t nslots, unsigned *live, hipStream_t stream)
{
    if (nslots == 0) return hipSuccess;
    hipLaunchKernelGGL(k_group, dim3((nslots + 63) / 64), dim3(64), 0, stream, insts, nslots, live);
    return hipGetLastError();
}

static uint32_t blocks_for(uint32_t n) { return n < 256 * 256 ? (n + 255) / 256 : 256; }

hipError_t launch_load(l2o_inst *insts, uint32_t slot, uint32_t n, const l2o_inst *rec, const void *raw, unsigned *live,
                       bool count, hipStream_t stream)
{
    const uint32_t words = (12 * n + 15) / 16;  // (the point buffer holds 16 n bytes)
    hipLaunchKernelGGL(k_stage, dim3(blocks_for(words)), dim3(256), 0, stream, insts + slot, rec, (uint4 *)rec->pts[1],
                       (const uint4 *)raw, words);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL(k_load, dim3(blocks_for(n)), dim3(256), 0, stream, insts, slot, live, count ? 1 : 0);
    return hipGetLastError();
}

hipError_t launch_prime(l2o_inst *insts, uint32_t slot, uint32_t n, hipStream_t stream)
{
    const uint32_t blocks = blocks_for(n);  // as many waves as k_load's
    hipLaunchKernelGGL(k_prime, dim3(blocks), dim3(256), 0, stream, insts, slot, 4 * blocks);
    return hipGetLastError();
}

hipError_t launch_free(l2o_inst *insts, uint32_t slot, unsigned *live, bool running, bool clear_pool, hipStream_t stream)
{
    hipLaunchKernelGGL(k_free, dim3(1), dim3(256), 0, stream, insts, slot, live, running ? 1 : 0, clear_pool ? 1 : 0);
    return hipGetLastError();
}

hipError_t launch_fetch(const l2o_inst *insts, uint32_t slot, uint32_t n, l2o_inst *rec, uint32_t *tour,
                        hipStream_t stream)
{
    hipLaunchKernelGGL(k_fetch, dim3(tour ? blocks_for(n) : 1), dim3(256), 0, stream, insts, slot, rec, tour);
    return hipGetLastError();
}

hipError_t launch_length(const l2o_inst *insts, uint32_t slot, uint32_t n, unsigned long long *out,
                         hipStream_t stream)
{
    const uint32_t blocks = min(1024u, (n + 255) / 256);
    hipLaunchKernelGGL(k_length, dim3(blocks), dim3(256), 0, stream, insts, slot, out);
    return hipGetLastError();
}

hipError_t launch_sqrt_ulp(uint32_t lo, uint32_t hi, unsigned *max_ulp, hipStream_t stream)
{
    hipLaunchKernelGGL(k_sqrt_ulp, dim3(4096), dim3(256), 0, stream, lo, hi, max_ulp);
    return hipGetLastError();
}

}  // namespace l2o
