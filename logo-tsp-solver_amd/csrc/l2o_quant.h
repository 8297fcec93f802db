// l2o_quant.h -- operands of the matrix test (see l2o_sweep.hip).
#pragma once
#include "l2o_device.h"

namespace l2o {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float16v __attribute__((ext_vector_type(16)));

__device__ __forceinline__ uint32_t pk16(float a, float b)
{
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a, b));
}

// the wave's lanes below this one among `m`
__device__ __forceinline__ int lanes_below(unsigned long long m)
{
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// quantised edge k -> k+1: {X, Y} and {X1, Y1} as FP16 pairs (l2o_pt.w of its
// ends), U = |(X, Y, X1, Y1)|^2 and E of its length (l2o_pt.d of k+1)
struct qedge {
    uint32_t p0, p1;
    float u, e;
};

__device__ __forceinline__ qedge quant_edge(uint32_t w0, uint32_t w1, uint32_t d1, float qk, float qm)
{
    const half2v a = __builtin_bit_cast(half2v, w0), b = __builtin_bit_cast(half2v, w1);
    qedge r;
    r.p0 = w0;
    r.p1 = w1;
    r.u = __builtin_amdgcn_fdot2(a, a, __builtin_amdgcn_fdot2(b, b, 0.0f, false), false);
    r.e = __builtin_ceilf(__builtin_fmaf((float)(int)d1, qk, qm));
    return r;
}

// E' = max(E - hc, 0) and the limbs of N of an edge; one outside the range
// (valid false) gets an Nh that no other terms can outweigh
struct qterms {
    float e, nh, nl;
};
__device__ __forceinline__ qterms edge_terms(const qedge &q, float hc, bool valid)
{
    qterms t;
    t.e = __builtin_fmaxf(q.e - hc, 0.0f);
    const float nn = __builtin_fmaf(-t.e, t.e, q.u);
    t.nh = __builtin_floorf(nn * (1.0f / 2048.0f));
    t.nl = __builtin_fmaf(t.nh, -2048.0f, nn);
    t.nh = valid ? t.nh : 30000.0f;
    return t;
}

// A operand (rows), 16 FP16 terms: lanes 0..31 {X, Y, X1, Y1, E', 1, Nl, Nh},
// lanes 32..63 the same {2048, 1, 0, 0, 0, 0, 0, 0} for every row
__device__ __forceinline__ uint4 row_record(const qedge &q, const qterms &t)
{
    return make_uint4(q.p0, q.p1, pk16(t.e, 1.0f), pk16(t.nl, t.nh));
}
__device__ __forceinline__ uint4 row_const() { return make_uint4(pk16(2048.0f, 1.0f), 0u, 0u, 0u); }

// B operand (columns): lanes 0..31 {-2X, -2Y, -2X1, -2Y1, -2E', Nl, 1, 2048},
// lanes 32..63 {Nh, -1, any six finite numbers}
__device__ __forceinline__ uint4 col_record(const qedge &q, const qterms &t)
{
    const half2v m2 = {(_Float16)-2.0f, (_Float16)-2.0f};
    return make_uint4(__builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, q.p0) * m2),
                      __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, q.p1) * m2),
                      pk16(-2.0f * t.e, t.nl), pk16(1.0f, 2048.0f));
}
__device__ __forceinline__ uint32_t col_upper(const qterms &t) { return pk16(t.nh, -1.0f); }

// the rows up to l of a block of 32 as bits: bit r of a lane's 16 results is
// row (r & 3) + 8 (r >> 2) + 4 (lane >> 5)
__device__ __forceinline__ uint32_t rows_upto(int l)
{
    return l < 0 ? 0u : ((2u << (4 * min(l >> 3, 3) + min(l >= 32 ? 3 : l & 7, 3))) - 1u) & 0xFFFFu;
}

// sign bits of a pair of products: bit r of c0, bit 16 + r of c1
__device__ __forceinline__ uint32_t sign_mask(const float16v &c0, const float16v &c1)
{
    uint32_t m0 = 0, m1 = 0;  // two chains
#pragma unroll
    for (int r = 15; r >= 0; --r) {
        m0 = __builtin_amdgcn_alignbit(m0, __float_as_uint(c0[r]), 31);
        m1 = __builtin_amdgcn_alignbit(m1, __float_as_uint(c1[r]), 31);
    }
    return m0 | m1 << 16;
}

// half of -C for the largest gain `cap` still worth an exact evaluation
__device__ __forceinline__ float half_cap(int cap, float qk)
{
    return __builtin_fmaxf(__builtin_floorf((float)-cap * (qk * 0.49999f) - 0.01f), 0.0f);
}

}  // namespace l2o
