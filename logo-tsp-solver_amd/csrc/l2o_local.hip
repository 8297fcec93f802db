// l2o_local.hip -- whole local searches and ILS runs of small instances, one
// workgroup per instance.
//
// A step of a small instance through k_sweep and k_apply costs two launches
// (about 11 us however few candidates there are).  Here a workgroup keeps the
// tour in LDS and runs `steps` sweeps of its instance in one launch: the matrix
// test of l2o_sweep.hip over all pairs of 32-edge blocks, exact evaluation of
// the survivors from LDS, the winning move by a gather into the other copy of
// the tour, and for an ILS job the accept, kick and stop rules of k_ils.  Moves,
// keys, random numbers and counters are those of the launch path, step by step,
// so an instance may change path between launches.
//
// What bounds it: latency.  A step passes four barriers; at 200 cities (4.0 us,
// 11.3 us with two launches) about 2 us go into the few waves that find and
// evaluate survivors, 0.9 us into applying the move.  At 1,000 cities (10.2 us)
// the 528 tiles take four SIMDs about 4 us of matrix and v_or3 issue.  The work
// is dealt out in units of a column pair and up to four row blocks, taken in
// turn from an LDS counter, those at the diagonal (most survivors) first: a
// fixed deal took 13.8 us at 1,000 cities.
//
// LDS per city: 16 bytes twice (x and y with the city id in their upper 10
// bits, the edge length, the quantised coordinates) and the 16-byte record of
// its edge, from which both operands are made.
#include <hip/hip_runtime.h>

#include "l2o_device.h"
#include "l2o_quant.h"

namespace l2o {

#define L2O_LOCAL_XY 0x3FFFFFu

// column pairs of 64 edges
__host__ __device__ inline uint32_t local_pairs(uint32_t n) { return (n - 1 + 63) >> 6; }

// row blocks a unit of work spans: enough units for every wave to take several
__host__ __device__ inline uint32_t local_span(uint32_t pairs, uint32_t waves)
{
    const uint32_t s = pairs * (pairs + 1) / (6 * waves);  // pairs (pairs + 1) strips in all
    return s < 1 ? 1 : s > 4 ? 4 : s;
}

// units: each column pair p has the row blocks 0 .. 2p+1
__host__ __device__ inline uint32_t local_units(uint32_t pairs, uint32_t span)
{
    uint32_t u = 0;
    for (uint32_t p = 0; p < pairs; ++p) u += (2 * p + 1) / span + 1;
    return u;
}

uint32_t local_lds_bytes(uint32_t n, int waves)
{
    const uint32_t pairs = local_pairs(n);
    return 16u * (2u * n + 64u * pairs + 1u) + 8u * (2u * L2O_POOL + 4u) + 4u * 8u + (uint32_t)waves * 512u +
           4u * local_units(pairs, local_span(pairs, (uint32_t)waves));
}

// B operand from the record of an edge (l2o_quant.h: row_record)
__device__ __forceinline__ half8 col_operand(const uint4 &r, bool upper)
{
    const half2v m2 = {(_Float16)-2.0f, (_Float16)-2.0f};
    uint4 v;
    v.x = upper ? (r.w >> 16) | pk16(0.0f, -1.0f)
                : __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, r.x) * m2);
    v.y = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, r.y) * m2);
    v.z = (__builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, r.z) * m2) & 0xFFFFu) | r.w << 16;
    v.w = pk16(1.0f, 2048.0f);
    return __builtin_bit_cast(half8, v);
}

template <int NW>
__global__ __launch_bounds__(64 * NW) void k_local(const uint32_t *__restrict__ ids, l2o_inst *__restrict__ insts,
                                                   unsigned *__restrict__ live, uint32_t steps)
{
    constexpr int NTHR = 64 * NW;
    extern __shared__ __attribute__((aligned(16))) uint4 lds[];
    l2o_inst *in = insts + ids[blockIdx.x];
    // (scalar loads: nothing else writes these while the kernel runs)
    const __attribute__((address_space(4))) l2o_inst *ci = (const __attribute__((address_space(4))) l2o_inst *)in;
    if (ci->phase != L2O_LO) return;
    const int n = (int)ci->n;
    const uint32_t metric = ci->metric, par = ci->parity;
    const float slack = ci->slack, es = ci->est_scale, ea = ci->est_add, qk = ci->qk, qm = ci->qm;
    const uint32_t ils_rounds = ci->ils_rounds, kick = ci->kick;
    const bool chain = ci->group_lead != L2O_NO_GROUP;  // its rounds are k_ils's and k_group's
    const unsigned long long stop_below = ci->stop_below;
    l2o_move *const mlog = ci->log;
    const uint32_t log_cap = ci->log_cap;
    l2o_pt *const G = par ? ci->pts[1] : ci->pts[0];
    uint32_t *const R = par ? ci->tour[1] : ci->tour[0];
    l2o_pt *const BP = ci->bpts;
    uint32_t *const BR = ci->btour;
    unsigned long long *const rlog = ci->rlog, *const gpool = ci->pool;
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int np = (int)local_pairs((uint32_t)n), nrec = 64 * np, nblk = (n - 1 + 31) >> 5;
    uint4 *const rec = lds + 2 * n;
    unsigned long long *const s_pool = (unsigned long long *)(rec + nrec + 1);  // [2][L2O_POOL]
    unsigned long long *const s_key = s_pool + 2 * L2O_POOL;                    // [2]
    unsigned long long *const s_sum = s_key + 2;                                // [2]
    uint32_t *const s_misc = (uint32_t *)(s_sum + 2);                           // [8]
    uint32_t *const list = s_misc + 8 + 128 * w;
    uint32_t *const s_unit = s_misc + 8 + 128 * NW;
    const int span = (int)local_span((uint32_t)np, NW), nunit = (int)local_units((uint32_t)np, (uint32_t)span);
    // the units, those at the diagonal (where most survivors are) first: unit
    // (p, c) covers the row blocks [2p+2 - span (c+1), 2p+2 - span c)
    for (int p = tid; p < np; p += NTHR) {
        int before = 0;
        for (int q = 0; q < p; ++q) before += (2 * q + 1) / span + 1;
        for (int c = 0; c <= (2 * p + 1) / span; ++c) {
            const int q1 = 2 * p + 2 - span * c, q0 = max(q1 - span, 0);
            // position: the diagonal units of all pairs, then the rest
            const int at = c == 0 ? p : np + (before - p) + c - 1;
            s_unit[at] = (uint32_t)p | (uint32_t)q0 << 10 | (uint32_t)min(q1, nblk) << 20;
        }
    }
    if (tid < 2) s_misc[6 + tid] = NW;

    auto px = [](const uint4 &p) __attribute__((always_inline)) { return (int)(p.x & L2O_LOCAL_XY); };
    auto py = [](const uint4 &p) __attribute__((always_inline)) { return (int)(p.y & L2O_LOCAL_XY); };
    auto pack = [](int x, int y, int d, int qw, uint32_t id) __attribute__((always_inline)) {
        return make_uint4((uint32_t)x | id << 22, (uint32_t)y | (id >> 10) << 22, (uint32_t)d, (uint32_t)qw);
    };

    // the tour, the pool and the key
    {
        for (int k = tid; k < n; k += NTHR) {
            const l2o_pt p = G[k];
            lds[k] = pack(p.x, p.y, p.d, p.w, R[k]);
        }
        if (tid < L2O_POOL) s_pool[tid] = gpool[3 * L2O_POOL + tid];
    }
    // the best known move of the current tour, and the largest gain its sweep evaluates
    const unsigned long long known = gpool[3 * L2O_POOL + lane];
    unsigned long long pmin = wave_min_u64(known);
    int cap = (int)ci->cap;
    if (tid == 0) {
        s_key[0] = pmin;
        rec[nrec] = row_const();
    }
    unsigned long long length = uniform_u64(in->length), moves = uniform_u64(in->moves);
    uint32_t sweeps = 0;
    unsigned fb = 0;
    int cur = 0;  // the tour is lds[cur n .. cur n + n)
    bool done = false;
    __syncthreads();

    for (uint32_t t = 0;; t ^= 1) {
        const uint4 *const P = lds + cur * n;
        const float hc = half_cap(cap, qk);
        const float thr = (float)cap + slack;
        // records of the edges k -> k+1
        {
            for (int k = tid; k < nrec; k += NTHR) {
                const uint4 p = P[min(k, n - 1)], q = P[min(k + 1, n - 1)];
                const qedge e = quant_edge(p.w, q.w, q.z, qk, qm);
                rec[k] = row_record(e, edge_terms(e, hc, k <= n - 2));
            }
        }
        __syncthreads();

        // every pair of blocks: wave w takes units w, w + NW, ... of a pair of
        // column tiles and up to four row blocks
        unsigned long long lbest = L2O_SENTINEL;
        int cnt = 0;
        auto evaluate = [&]() __attribute__((always_inline)) {
            asm volatile("" ::: "memory");
            if (lane < cnt) {
                const uint32_t v = list[lane];
                const int a = (int)(v >> 16), b = (int)(v & 0xFFFFu);
                const uint4 A0 = P[a], A1 = P[a + 1], B0 = P[b], B1 = P[b + 1];
                const int da = (int)A1.z, db = (int)B1.z;
                const float w2 = (est_dist(px(A0), py(A0), px(B0), py(B0), es, ea) +
                                  est_dist(px(A1), py(A1), px(B1), py(B1), es, ea)) - (float)db;
                if (w2 <= thr + (float)da) {
                    ++fb;
                    const int gain = exact_dist(px(A0), py(A0), px(B0), py(B0), metric) +
                                     exact_dist(px(A1), py(A1), px(B1), py(B1), metric) - da - db;
                    if (gain < 0) {
                        const uint32_t i = (uint32_t)(a + 1);
                        const unsigned long long key = make_key(gain, i, (uint32_t)(b + 1));
                        lbest = key < lbest ? key : lbest;
                        atomicMin(&s_pool[t * L2O_POOL + ((i * 0x9E3779B1u) >> 26)], key);
                    }
                }
            }
            // what was not evaluated moves to the front of the list
            uint32_t rest = 0;
            if (lane < cnt - 64) rest = list[64 + lane];
            asm volatile("" ::: "memory");
            if (lane < cnt - 64) list[lane] = rest;
            asm volatile("" ::: "memory");
            cnt = max(cnt - 64, 0);
        };
        const bool upper = lane >= 32;
        const float16v zero = {0};
        // (the first unit by wave, the following ones in turn)
        for (int u = w; u < nunit;) {
            const uint32_t unit = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_unit[u]);
            int un = 0;
            if (lane == 0) un = (int)atomicAdd(&s_misc[6 + t], 1u);
            const int p = (int)(unit & 1023u), q0 = (int)(unit >> 10 & 1023u), q1 = (int)(unit >> 20);
            uint4 r0 = rec[64 * p + (lane & 31)], r1 = rec[64 * p + 32 + (lane & 31)];
            // (row operand of the next step in flight: `upper` lanes stay at the constant)
            int ra = upper ? nrec : 32 * q0 + lane;
            const int rstep = upper ? 0 : 32;
            uint4 an = rec[ra];
            // (whole loads before the selects of the column operand)
            asm volatile("" : "+v"(r0.x), "+v"(r0.y), "+v"(r0.z), "+v"(r0.w), "+v"(r1.x), "+v"(r1.y), "+v"(r1.z), "+v"(r1.w));
            const half8 B0 = col_operand(r0, upper), B1 = col_operand(r1, upper);
            for (int q = q0; q < q1; ++q) {
                const half8 A = __builtin_bit_cast(half8, an);
                ra += rstep;
                if (q + 1 < q1) an = rec[ra];
                const float16v c0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(A, B0, zero, 0, 0, 0);
                const float16v c1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(A, B1, zero, 0, 0, 0);
                uint32_t m = 0;
#pragma unroll
                for (int r = 0; r < 16; ++r) m |= __float_as_uint(c0[r]) | __float_as_uint(c1[r]);
                if (!__ballot((int)m < 0)) continue;
                uint32_t mask = sign_mask(c0, c1);
                if (64 * p < 32 * q + 33) {  // the pair meets the diagonal: candidates need a + 2 <= b
                    const int l = 64 * p + (lane & 31) - 2 - 32 * q - (lane >> 5) * 4;
                    mask &= rows_upto(l) | rows_upto(l + 32) << 16;
                }
                for (;;) {
                    const unsigned long long any = __ballot(mask != 0);
                    if (!any) break;
                    if (mask) {
                        const int bit = __builtin_ctz(mask);
                        mask &= mask - 1;
                        const uint32_t a = (uint32_t)(32 * q + (bit & 3) + ((bit >> 2) & 3) * 8 + (lane >> 5) * 4);
                        const uint32_t b = (uint32_t)(64 * p + (bit >> 4) * 32 + (lane & 31));
                        list[cnt + lanes_below(any)] = a << 16 | b;
                    }
                    cnt += __builtin_popcountll(any);
                    if (cnt >= 64) evaluate();
                }
            }
            u = __builtin_amdgcn_readfirstlane(un);
        }
        if (cnt) evaluate();
        if (__ballot(lbest != L2O_SENTINEL)) {
            const unsigned long long wb = wave_min_u64(lbest);
            if (lane == 0) atomicMin(&s_key[t], wb);
        }
        __syncthreads();

        const unsigned long long key = uniform_u64(s_key[t]);
        const uint32_t t1 = t ^ 1;
        uint4 *const Q = lds + (cur ^ 1) * n;
        ++sweeps;
        bool kicked = false;
        if (key != L2O_SENTINEL) {
            // r' = r[i..J-1] ++ r[i-1..0] ++ r[n-1..J]; edge lengths move with
            // their edges, the two new ones are at positions 0 and L
            const int gain = key_gain(key);
            const int i = (int)((uint32_t)(key >> 20) & 0xFFFFFu), J = (int)((uint32_t)key & 0xFFFFFu), L = J - i;
            for (int k = tid; k < n; k += NTHR) {
                const int sr = k < L ? i + k : k < J ? J - 1 - k : n - 1 + J - k;
                const int de = k < L ? sr : sr + 1 == n ? 0 : sr + 1;
                uint4 v = P[sr];
                v.z = P[de].z;
                if (k == 0 || k == L) {  // (the length is the last wave's, below)
                    Q[k].x = v.x;
                    Q[k].y = v.y;
                    Q[k].w = v.w;
                } else {
                    Q[k] = v;
                }
            }
            if (w == NW - 1 && lane < 2) {  // lane 0: P[i] -> P[J] at 0, lane 1: P[J-1] -> P[i-1] at L
                const uint4 u = P[lane == 0 ? i : J - 1], v = P[lane == 0 ? J : i - 1];
                Q[lane == 0 ? 0 : L].z = (uint32_t)exact_dist(px(u), py(u), px(v), py(v), metric);
            }
            const unsigned long long pk = remap_key(s_pool[t * L2O_POOL + lane], (uint32_t)i, (uint32_t)J, (uint32_t)n);
            pmin = wave_min_u64(pk);
            cap = next_cap(pk, 0, (uint32_t)n);
            if (w == 0) s_pool[t1 * L2O_POOL + lane] = pk;
            if (tid == 0) {
                if (moves < log_cap) {
                    l2o_move m;
                    m.i = (uint32_t)i;
                    m.j = (uint32_t)J;
                    m.gain = gain;
                    mlog[moves] = m;
                }
                s_key[t1] = pmin;
                s_misc[6 + t] = NW;  // (next used two steps on)
            }
            ++moves;
            length += (unsigned long long)(long long)gain;
        } else {
            if (!ils_rounds || chain) {
                done = true;
                break;
            }
            // a local optimum of an ILS run: accept, stop or kick (as k_ils)
            if (tid == 0) {
                const bool acc = !in->have_best || length < in->best_length;
                if (acc) {
                    in->best_length = length;
                    in->have_best = 1;
                }
                const unsigned long long best = acc ? length : in->best_length;
                if (rlog) rlog[in->rounds_done] = best;
                const bool stop = in->rounds_done >= ils_rounds || best < stop_below;
                uint32_t cut[3] = {0, 0, 0};
                if (!stop) {
                    draw_kick(in->rng, kick, (uint32_t)n, cut);
                    in->rounds_done += 1;
                }
                s_misc[0] = acc;
                s_misc[1] = stop;
                s_misc[2] = cut[0];
                s_misc[3] = cut[1];
                s_misc[4] = cut[2];
                s_sum[0] = 0;
                s_key[t1] = L2O_SENTINEL;
                s_misc[6 + t] = NW;
            }
            __syncthreads();
            auto misc = [&](int k) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)s_misc[k]); };
            const bool acc = misc(0) != 0, stop = misc(1) != 0;
            if (acc) {
                for (int k = tid; k < n; k += NTHR) {
                    const uint4 v = P[k];
                    l2o_pt r;
                    r.x = px(v);
                    r.y = py(v);
                    r.d = (int)v.z;
                    r.w = (int)v.w;
                    BP[k] = r;
                    BR[k] = v.x >> 22 | (v.y >> 22) << 10;
                }
            }
            if (stop) {
                done = true;
                break;
            }
            const uint32_t ca = misc(2), cb = misc(3), cc = misc(4);
            const bool ref = kick == 1;
            auto best_at = [&](uint32_t s) __attribute__((always_inline)) {
                if (acc) return P[s];  // the best tour is the current one
                const l2o_pt r = BP[s];
                return pack(r.x, r.y, r.d, r.w, BR[s]);
            };
            unsigned long long sum = 0;
            for (int k = tid; k < n; k += NTHR) {
                uint4 v = best_at(kick_source((uint32_t)k, (uint32_t)n, ref, ca, cb, cc));
                const uint4 u = best_at(kick_source((uint32_t)(k ? k - 1 : n - 1), (uint32_t)n, ref, ca, cb, cc));
                const int d = exact_dist(px(u), py(u), px(v), py(v), metric);
                sum += (unsigned long long)d;
                v.z = (uint32_t)d;
                Q[k] = v;
            }
            sum = wave_sum_u64(sum);
            if (lane == 0) atomicAdd(&s_sum[0], sum);
            if (tid < L2O_POOL) s_pool[t1 * L2O_POOL + tid] = L2O_SENTINEL;
            pmin = L2O_SENTINEL;
            cap = -1;
            kicked = true;
        }
        cur ^= 1;
        __syncthreads();
        if (kicked) length = uniform_u64(s_sum[0]);
        if (sweeps == steps) break;
    }

    // the state back to the instance's buffers
    const uint4 *const P = lds + cur * n;
    for (int k = tid; k < n; k += NTHR) {
        const uint4 v = P[k];
        l2o_pt r;
        r.x = px(v);
        r.y = py(v);
        r.d = (int)v.z;
        r.w = (int)v.w;
        G[k] = r;
        R[k] = v.x >> 22 | (v.y >> 22) << 10;
    }
    if (w == 0) {
        // the pool of the current tour: the last sweep's, mapped (empty at the end)
        gpool[3 * L2O_POOL + lane] = done ? L2O_SENTINEL : s_pool[(sweeps & 1) * L2O_POOL + lane];
    }
    const unsigned wfb = wave_sum_u32(fb);
    if (lane == 0 && wfb) atomicAdd(&in->fallbacks, (unsigned long long)wfb);
    __threadfence();
    __syncthreads();
    if (tid == 0) {
        in->length = length;
        in->moves = moves;
        in->sweeps += sweeps;
        in->cap = done ? -1 : cap;
        if (done && chain) {
            in->phase = L2O_LO_DONE;
        } else if (done) {
            // the host may look at both while other workgroups run
            in->phase = L2O_DONE;
            __threadfence();
            atomicSub(live, 1u);
        }
    }
}

#define L2O_LOCAL_WAVES(X) X(4) X(8) X(16)

hipError_t launch_local(int waves, const uint32_t *ids, uint32_t count, uint32_t max_n, l2o_inst *insts, unsigned *live,
                        uint32_t steps, hipStream_t stream)
{
    if (count == 0) return hipSuccess;
    const uint32_t bytes = local_lds_bytes(max_n, waves);
#define L2O_LOCAL_CASE(W_)                                                                                         \
    if (waves == W_) {                                                                                            \
        hipError_t e = hipFuncSetAttribute((const void *)k_local<W_>, hipFuncAttributeMaxDynamicSharedMemorySize, \
                                           (int)bytes);                                                           \
        if (e != hipSuccess) return e;                                                                            \
        hipLaunchKernelGGL((k_local<W_>), dim3(count), dim3(64 * W_), bytes, stream, ids, insts, live, steps);    \
        return hipGetLastError();                                                                                 \
    }
    L2O_LOCAL_WAVES(L2O_LOCAL_CASE)
    return hipErrorInvalidValue;
}

}  // namespace l2o
