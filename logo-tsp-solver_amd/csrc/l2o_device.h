// l2o_device.h -- device helpers shared by the kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "l2o_launch.h"
#include "l2o_state.h"

namespace l2o {

// ---------------------------------------------------------------------------
// exact metric length of the edge P1 -> P2 (metric_dist in l2o_launch.h) without
// FP64: with m an estimate of floor(sqrt(s / f)) from v_sqrt_f32, at most 3 off
// (s has a relative error of 2^-23, the root 3 ulp, and sqrt(s) < 2^22.5), the
// remainder r = s - f m^2 is below 2^28 in magnitude, so 32-bit arithmetic holds it.
// floor(r / (f (2m+1))) is the distance to the true root or one more, and one
// correction each way makes m exact; then s > f m^2 + e m is r > e m.
// ---------------------------------------------------------------------------
template <int F>
__device__ __forceinline__ int root_len(uint32_t s32, float fs, int e)
{
    int m = (int)__builtin_amdgcn_sqrtf(F == 1 ? fs : fs * 0.1f);
    int r = (int)(s32 - (uint32_t)F * ((uint32_t)m * (uint32_t)m));
    const int d = (int)__builtin_floorf((float)r * __builtin_amdgcn_rcpf((float)(F * (2 * m + 1))));
    r -= F * (d * (2 * m + d));
    m += d;
    if (r < 0) {
        m -= 1;
        r += F * (2 * m + 1);
    }
    if (r >= F * (2 * m + 1)) {
        r -= F * (2 * m + 1);
        m += 1;
    }
    return m + (r > e * m ? 1 : 0);
}

__device__ __forceinline__ int exact_dist(int x1, int y1, int x2, int y2, uint32_t metric)
{
    // coordinates lie in [0, 2^22)
    const int dx = x1 - x2, dy = y1 - y2;
    const uint32_t s32 = (uint32_t)dx * (uint32_t)dx + (uint32_t)dy * (uint32_t)dy;
    const float fs = __builtin_fmaf((float)dx, (float)dx, (float)dy * (float)dy);
    return metric == L2O_ATT ? root_len<10>(s32, fs, 0) : root_len<1>(s32, fs, metric == L2O_EUC_2D ? 1 : 0);
}

// FP32 estimate of the metric length: sqrt(s) * scale + add, with scale = 1,
// add = 0 for EUC_2D (D = nint(d)), scale = 1, add = 1/2 for CEIL_2D (D in
// [d, d+1)) and scale = 1/sqrt(10), add = 1/2 for ATT; |D - estimate| <= 1/2
// plus the FP32 error, which the instance's slack bounds.  The integer
// differences convert to FP32 exactly.
__device__ __forceinline__ float est_dist(int x1, int y1, int x2, int y2, float scale, float add)
{
    const float dx = (float)(x1 - x2), dy = (float)(y1 - y2);
    return __builtin_fmaf(__builtin_amdgcn_sqrtf(__builtin_fmaf(dx, dx, dy * dy)), scale, add);
}

__device__ __forceinline__ unsigned long long make_key(int gain, uint32_t i, uint32_t j)
{
    return ((unsigned long long)(gain + L2O_KEY_GAIN_BIAS) << 40) |
           ((unsigned long long)i << 20) | (unsigned long long)j;
}

__device__ __forceinline__ int key_gain(unsigned long long key)
{
    return (int)((long long)(key >> 40) - L2O_KEY_GAIN_BIAS);
}

// one step of a 64-bit minimum scan over the lanes: DPP CTRL moves both
// halves; lanes the move leaves without a source keep their own value
template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned long long dpp_min_u64(unsigned long long v)
{
    const int lo = (int)(uint32_t)v, hi = (int)(uint32_t)(v >> 32);
    const uint32_t l2 = (uint32_t)__builtin_amdgcn_update_dpp(lo, lo, CTRL, ROWS, 0xF, false);
    const uint32_t h2 = (uint32_t)__builtin_amdgcn_update_dpp(hi, hi, CTRL, ROWS, 0xF, false);
    const unsigned long long o = ((unsigned long long)h2 << 32) | l2;
    return o < v ? o : v;
}

// minimum over the 64 lanes, returned wave-uniform (in SGPRs): row_shr 1, 2,
// 4, 8 within each row of 16 lanes, then row_bcast 15 and 31 carry the rows
// below upwards, so lane 63 ends with the minimum (VALU only, no LDS)
__device__ __forceinline__ unsigned long long wave_min_u64(unsigned long long v)
{
    v = dpp_min_u64<0x111, 0xF>(v);
    v = dpp_min_u64<0x112, 0xF>(v);
    v = dpp_min_u64<0x114, 0xF>(v);
    v = dpp_min_u64<0x118, 0xF>(v);
    v = dpp_min_u64<0x142, 0xA>(v);
    v = dpp_min_u64<0x143, 0xC>(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, 63);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), 63);
    return ((unsigned long long)hi << 32) | lo;
}

// a wave-uniform 64-bit value moved to SGPRs (readfirstlane returns int: each
// half is taken as unsigned before it is widened)
__device__ __forceinline__ unsigned long long uniform_u64(unsigned long long v)
{
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return ((unsigned long long)hi << 32) | lo;
}

// The key of a known candidate (edges e-1 -> e of positions i2 and j2) on the
// tour after the move (i, J): r' = r[i..J-1] ++ r[i-1..0] ++ r[n-1..J].  An
// edge keeps its two cities unless it is one of the two removed ones; its
// direction is reversed outside [i, J-1].  Two edges of the same side keep
// their relative direction, so the candidate keeps its gain at the mapped
// positions; two edges of different sides would reconnect the other way.
// L2O_SENTINEL if the candidate is gone.
// (i = 0, J = n: no move.)
__device__ __forceinline__ unsigned long long remap_key(unsigned long long key, uint32_t i, uint32_t J, uint32_t n)
{
    const uint32_t i2 = (uint32_t)(key >> 20) & 0xFFFFFu, j2 = (uint32_t)key & 0xFFFFFu;
    const bool in1 = i2 > i && i2 < J, in2 = j2 > i && j2 < J;
    auto to = [&](uint32_t e) { return e > i && e < J ? e - i : e < i ? J - e : n + J - e; };
    const uint32_t e1 = to(i2), e2 = to(j2);
    if (key == L2O_SENTINEL || in1 != in2 || i2 == i || i2 == J || j2 == i || j2 == J) return L2O_SENTINEL;
    return (key & ~((1ull << 40) - 1)) | ((unsigned long long)min(e1, e2) << 20) | max(e1, e2);
}

// point records in global memory (address space 1: the pointers come from
// the instance record, so the space is stated for global_* instructions)
typedef __attribute__((address_space(1))) l2o_pt gpt;
typedef __attribute__((address_space(1))) uint32_t gu32;

__device__ __forceinline__ l2o_pt ld_pt(const gpt *P, uint32_t k)
{
    l2o_pt r;
    r.x = P[k].x;
    r.y = P[k].y;
    r.d = P[k].d;
    r.w = P[k].w;
    return r;
}

__device__ __forceinline__ void st_pt(gpt *P, uint32_t k, const l2o_pt r)
{
    P[k].x = r.x;
    P[k].y = r.y;
    P[k].d = r.d;
    P[k].w = r.w;
}

// The tour after a move (i, J), in terms of the one before:
// r' = r[i..J-1] ++ r[i-1..0] ++ r[n-1..J] (twoOptLocalSolver.cpp:41-48).  Without
// a move (L2O_KEY_NONE) i = 0, J = n: the identity.
struct move_map {
    int i, J, L, n;
    __device__ __forceinline__ move_map(unsigned long long key, int n_)
    {
        n = n_;
        i = key == L2O_KEY_NONE ? 0 : (int)((uint32_t)(key >> 20) & 0xFFFFFu);
        J = key == L2O_KEY_NONE ? n : (int)((uint32_t)key & 0xFFFFFu);
        L = J - i;
    }
    // position before the move of the city at k
    __device__ __forceinline__ int src(int k) const { return k < L ? k + i : k < J ? J - 1 - k : n - 1 + J - k; }
    // length of the edge k-1 -> k (k > 0) from l2o_pt.d of its ends before the
    // move (d0 of src(k-1), d1 of src(k)) and of the new edge at L
    __device__ __forceinline__ int len(int k, int d0, int d1, int dL) const { return k < L ? d1 : k == L ? dL : d0; }
};

__device__ __forceinline__ unsigned wave_sum_u32(unsigned v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// maximum over the 64 lanes, returned wave-uniform: the scan pattern of
// wave_min_u64 with max, where a lane that a shift leaves without a source keeps its value
__device__ __forceinline__ int wave_max_i32(int v)
{
    v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x111, 0xF, 0xF, false));
    v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x112, 0xF, 0xF, false));
    v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x114, 0xF, 0xF, false));
    v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x118, 0xF, 0xF, false));
    v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x142, 0xA, 0xF, false));
    v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x143, 0xC, 0xF, false));
    return __builtin_amdgcn_readlane(v, 63);
}

// The largest gain the next sweep evaluates, given the pool (one entry per
// lane) and the move (i, J) after it: the best gain of the entries that the move
// leaves (see remap_key) while it leaves enough of them, else a somewhat worse
// one, so that the sweep refills the pool before it runs out (a move invalidates
// up to half of it, and a sweep without a known move evaluates every improving
// candidate).
#ifndef L2O_POOL_LOW
#define L2O_POOL_LOW 16
#endif
#ifndef L2O_CAP_SHIFT
#define L2O_CAP_SHIFT 3
#endif
__device__ __forceinline__ int worse_gain(int gain) { return min(gain - (gain >> L2O_CAP_SHIFT), -1); }
__device__ __forceinline__ int next_cap(unsigned long long key, uint32_t i, uint32_t J)
{
    const uint32_t i2 = (uint32_t)(key >> 20) & 0xFFFFFu, j2 = (uint32_t)key & 0xFFFFFu;
    const bool stays = key != L2O_SENTINEL && (i2 > i && i2 < J) == (j2 > i && j2 < J) && i2 != i && i2 != J &&
                       j2 != i && j2 != J;
    const unsigned long long left = __ballot(stays);
    if (!left) return -1;
    const int gain = -wave_max_i32(stays ? -key_gain(key) : 0);
    return __builtin_popcountll(left) >= L2O_POOL_LOW ? gain : worse_gain(gain);
}

__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned lo = __shfl_xor((unsigned)v, off);
        const unsigned hi = __shfl_xor((unsigned)(v >> 32), off);
        v += ((unsigned long long)hi << 32) | lo;
    }
    return v;
}

// ---------------------------------------------------------------------------
// ILS kicks (xoshiro256**)
// ---------------------------------------------------------------------------
__device__ __forceinline__ unsigned long long rotl64(unsigned long long v, int k)
{
    return (v << k) | (v >> (64 - k));
}

__device__ inline unsigned long long xoshiro_next(unsigned long long *s)
{
    const unsigned long long result = rotl64(s[1] * 5ull, 7) * 9ull;
    const unsigned long long t = s[1] << 17;
    s[2] ^= s[0];
    s[3] ^= s[1];
    s[1] ^= s[2];
    s[0] ^= s[3];
    s[2] ^= t;
    s[3] = rotl64(s[3], 45);
    return result;
}

// cut points of a kick: the reference's a, b = rand() % n, sorted
// (ILSGlobalSolver.cpp:39-44), or for the double bridge 1 <= p1 < p2 < p3 <= n-1
__device__ inline void draw_kick(unsigned long long *rng, uint32_t kick, uint32_t n, uint32_t *cut)
{
    if (kick == 1) {
        const uint32_t a = (uint32_t)(xoshiro_next(rng) % n);
        const uint32_t b = (uint32_t)(xoshiro_next(rng) % n);
        cut[0] = min(a, b);
        cut[1] = max(a, b);
        cut[2] = 0;
        return;
    }
    int have = 0;
    while (have < 3) {
        const uint32_t v = 1u + (uint32_t)(xoshiro_next(rng) % (unsigned long long)(n - 1));
        bool dup = false;
        for (int q = 0; q < have; ++q) dup |= (cut[q] == v);
        if (!dup) cut[have++] = v;
    }
    const uint32_t lo = min(min(cut[0], cut[1]), cut[2]), hi = max(max(cut[0], cut[1]), cut[2]);
    cut[1] = cut[0] ^ cut[1] ^ cut[2] ^ lo ^ hi;
    cut[0] = lo;
    cut[2] = hi;
}

// position of the best tour that a kick puts at position k: rotate(a) then
// reverse from b-a (ILSGlobalSolver.cpp:46-47), or A C B D of A=[0,a) B=[a,b)
// C=[b,c) D=[c,n)
__device__ __forceinline__ uint32_t kick_source(uint32_t k, uint32_t n, bool ref, uint32_t a, uint32_t b, uint32_t c)
{
    if (ref) return k < b - a ? (a + k) % n : (n - 1 - k + b) % n;
    if (k < a) return k;
    if (k < a + (c - b)) return b + (k - a);
    if (k < c) return a + (k - a - (c - b));
    return k;
}

// ---------------------------------------------------------------------------
// the tour after a move, chunk of L2O_APPLY_CHUNK positions from k0: points, edge
// lengths and city ids gathered from buffer `b` into the other one.  A thread's
// elements are independent: the loads of four are issued before their stores.
// ---------------------------------------------------------------------------
template <int NTHR>
__device__ __forceinline__ void copy_chunk(const __attribute__((address_space(4))) l2o_inst *ci, uint32_t b,
                                           const move_map &mm, uint32_t metric, int k0)
{
    const gpt *P = (const gpt *)(b ? ci->pts[1] : ci->pts[0]);
    gpt *Pn = (gpt *)(b ? ci->pts[0] : ci->pts[1]);
    const gu32 *R = (const gu32 *)(b ? ci->tour[1] : ci->tour[0]);
    gu32 *Rn = (gu32 *)(b ? ci->tour[0] : ci->tour[1]);
    const int n = mm.n;
    const bool moved = mm.L < n;
    // the far ends of the two new edges: P[i] -> P[J] at position 0, P[J-1] -> P[i-1] at L
    const l2o_pt endJ = ld_pt(P, moved ? mm.J : 0), endJ1 = ld_pt(P, mm.J - 1);
    constexpr int PER = 4;
    for (int c = 0; c < L2O_APPLY_CHUNK; c += PER * NTHR) {
        l2o_pt p[PER];
        int dq[PER];
        uint32_t rid[PER];
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const int k = min(k0 + c + (int)threadIdx.x + e * NTHR, n - 1);
            const int s = mm.src(k);
            const int de = k < mm.L ? s : s + 1 >= n ? 0 : s + 1;
            p[e] = ld_pt(P, (uint32_t)s);
            dq[e] = P[de].d;
            rid[e] = R[s];
        }
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const int k = k0 + c + (int)threadIdx.x + e * NTHR;
            if (c + (int)threadIdx.x + e * NTHR >= L2O_APPLY_CHUNK || k >= n) continue;
            l2o_pt r = p[e];
            r.d = dq[e];
            if (moved && (k == 0 || k == mm.L)) {
                const l2o_pt o = k == 0 ? endJ : endJ1;
                r.d = exact_dist(r.x, r.y, o.x, o.y, metric);
            }
            st_pt(Pn, (uint32_t)k, r);
            Rn[k] = rid[e];
        }
    }
}

// a local optimum found: the pool is left empty, the instance goes to its next
// phase (one wave; `parity` is the buffer of its tour)
__device__ __forceinline__ void local_optimum(l2o_inst *in, unsigned *live, uint32_t parity)
{
    const int lane = (int)threadIdx.x & 63;
#pragma unroll
    for (int r = 0; r < 4; ++r) in->pool[r * L2O_POOL + lane] = L2O_SENTINEL;
    if (lane == 0) {
        in->sweeps += 1;
        in->parity = parity;
        if (in->ils_rounds == 0) {
            in->phase = L2O_DONE;
            atomicSub(live, 1u);
        } else {
            in->phase = L2O_LO_DONE;
        }
    }
}

// counters and log of an applied move (one thread)
__device__ __forceinline__ void log_move(l2o_inst *in, unsigned long long key)
{
    const int gain = key_gain(key);
    in->length += (unsigned long long)(long long)gain;
    if (in->moves < in->log_cap) {
        l2o_move m;
        m.i = (uint32_t)(key >> 20) & 0xFFFFFu;
        m.j = (uint32_t)key & 0xFFFFFu;
        m.gain = gain;
        in->log[in->moves] = m;
    }
    in->moves += 1;
    in->sweeps += 1;
}

}  // namespace l2o
