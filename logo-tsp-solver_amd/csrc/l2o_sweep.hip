// l2o_sweep.hip -- the sweep: every 2-opt candidate of a tour through a matrix
// test, the survivors through an FP32 estimate and the exact length.
//
// Candidates.  With a = i-1 and b = J-1 a candidate is a pair
// 0 <= a, a+2 <= b <= n-2 with exact gain
//     G = n(a,b) + n(a+1,b+1) - D[a+1] - D[b+1],
// n(x,y) the exact metric length of P[x] -> P[y] and D[k] = n(k-1,k).  The
// sweep returns the lexicographic minimum of (G, i, J) over G < 0 (the move the
// reference's strict-'<' scan keeps).
//
// Matrix test.  Take row a as the 4-vector u = (x_a, y_a, x_a+1, y_a+1) and
// column b as v likewise.  The new edges have Euclidean lengths d1, d2 with
// d1^2 + d2^2 = |u - v|^2, so |u - v| <= d1 + d2, and G <= cap needs
// d1 + d2 <= kappa (D[a+1] + D[b+1] + cap) + h (h = 1 for EUC_2D's two
// roundings, kappa = sqrt(10) for ATT).  With the coordinates quantised to
// whole numbers X = rint(x s + o) the vector |U - V| is at most 2 + s |u - v|
// (each of four components is off by at most 1), so with
//     E = ceil(s kappa D + s h / 2 + 1),   C = -2 floor(s kappa |cap| / 2)
// a candidate that can still win has |U - V|^2 <= (E_a + E_b + C)^2.  Both
// sides expand into an inner product of a row record and a column record
// (the cap goes in half to each side, E' = max(E + C/2, 0), N = |U|^2 - E'^2):
//     |U - V|^2 - (E'_a + E'_b)^2 - 1
//        = -2 U.V - 2 E'_a E'_b + N_a + N_b - 1 < 0,
// 5 products and N split into N = 2048 Nh + Nl on each side: 10 of the 16
// terms of v_mfma_f32_32x32x16_f16.  Every operand is a whole number of at
// most 11 bits, exact in FP16, and every partial sum stays below 2^24
// (L2O_QR, L2O_QE in l2o_launch.h), exact in FP32: the test has no rounding.
// One matrix instruction tests 32 x 32 candidates; 16 results per lane are
// combined by their sign bits (v_or3_b32, two results an instruction); a
// candidate costs 1.0 VALU instructions in all (33,810 clustered cities), where
// the 8-bit v_sad_u8 bound it replaces took 2.2.
//
// What bounds it.  A tile of 1,024 candidates holds the matrix unit for 32
// cycles and needs at least 8 v_or3 (32 cycles of VALU issue); the two overlap
// only in part (a loop of nothing else: 46 cycles a tile, 5.0e13 candidates/s).
// At 33,810 cities VALU issue takes 58% and the matrix unit 29% of a launch of
// 25 us.  Measured with one MI355X, whole steps: 100,000 cities 270 -> 133 us
// (3.8e13 candidates/s), 33,810 clustered 57 -> 27 us, 7,397 20 -> 7.9 us (a
// launch's latency).  Matrix results kept in AGPRs, as the compiler prefers,
// cost a copy each: 2.7e13 instead of 4.4e13 tests/s (-amdgpu-mfma-vgpr-form).
//
// E' is cut off at 0 (a larger sum only lets more pass): without it a pair of
// short edges has a negative sum under a strong cap, and its square lets
// thousands of candidates pass that cannot win.
//
// Survivors.  The 32 sign bits of a pair of tiles are stored in LDS per lane;
// every row block the wave compacts them into full waves of candidates, which
// load their four points, take the FP32 estimate and, if that passes, the exact
// length (integers, l2o_device.h).  Keys go to the instance's
// shared key by atomicMin; the result is exact and independent of wave order.
#include <hip/hip_runtime.h>

#include "l2o_device.h"
#include "l2o_quant.h"

namespace l2o {

// maximum over each half of the wave of a pair of FP16 numbers, in lanes 31 and
// 63 (the others hold partial ones)
__device__ __forceinline__ uint32_t half_max_pk(uint32_t v)
{
    auto step = [](uint32_t x, int y) {
        return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(half2v, x),
                                                                      __builtin_bit_cast(half2v, (uint32_t)y)));
    };
    v = step(v, __builtin_amdgcn_update_dpp((int)v, (int)v, 0x111, 0xF, 0xF, false));
    v = step(v, __builtin_amdgcn_update_dpp((int)v, (int)v, 0x112, 0xF, 0xF, false));
    v = step(v, __builtin_amdgcn_update_dpp((int)v, (int)v, 0x114, 0xF, 0xF, false));
    v = step(v, __builtin_amdgcn_update_dpp((int)v, (int)v, 0x118, 0xF, 0xF, false));
    v = step(v, __builtin_amdgcn_update_dpp((int)v, (int)v, 0x142, 0xA, 0xF, false));
    return v;
}

// Box of the 32 edges of each half of the wave, both ends of the valid ones:
// {max X, max Y}, {-min X, -min Y} and the largest E' (pairs of FP16 whole
// numbers); lanes 31 and 63 write it
__device__ __forceinline__ void edge_boxes(const qedge &q, float hc, bool valid, int lane, uint4 *out)
{
    const half2v a = __builtin_bit_cast(half2v, q.p0), b = __builtin_bit_cast(half2v, q.p1);
    const uint32_t none = 0xE800E800u;  // {-2048, -2048}
    const uint32_t hi = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(a, b));
    const uint32_t lo = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(-a, -b));
    uint4 r;
    r.x = half_max_pk(valid ? hi : none);
    r.y = half_max_pk(valid ? lo : none);
    r.z = half_max_pk(valid ? pk16(__builtin_fmaxf(q.e - hc, 0.0f), 0.0f) : none);
    r.w = 0;
    if ((lane & 31) == 31) out[lane >> 5] = r;
}

// whether a candidate of a row block and a column tile can pass: its |U - V|^2 is
// at least twice the squared distance of the boxes (both ends of an edge lie in
// its box) and its E'_a + E'_b at most the sum of the largest
__device__ __forceinline__ bool boxes_meet(const uint4 &r, const uint4 &c)
{
    auto h2 = [](uint32_t v) { return __builtin_bit_cast(half2v, v); };
    const half2v zero = {(_Float16)0.0f, (_Float16)0.0f};
    const half2v g = __builtin_elementwise_max(__builtin_elementwise_max(-(h2(r.y) + h2(c.x)), -(h2(c.y) + h2(r.x))), zero);
    const float s = (float)h2(r.z)[0] + (float)h2(c.z)[0];
    return s >= 0.0f && 2.0f * __builtin_amdgcn_fdot2(g, g, 0.0f, false) <= s * s;
}

// One work item: rows [a0, a0 + rows) and the 64 K WAVES columns from b0.  A wave
// keeps its columns' operands in registers; the rows stream through LDS in
// chunks of one row per thread, the next chunk's points loaded while this one
// is tested.
// RUN: sweep t of a run (l2o_state.h), on the tour after the move of the sweep
// before; otherwise t = 0 and the tour is the buffer's.
#define L2O_SWEEP_MAX_T 512
template <int K, int WAVES, int MODE, bool RUN>
__device__ __forceinline__ void sweep_item(const l2o_sweep_item it, l2o_inst *__restrict__ insts, uint32_t t_)
{
    const uint32_t t = RUN ? t_ : 0;
    l2o_inst *in = insts + it.inst;
    // The fields this kernel reads but no wave writes come in one batch of
    // scalar loads before any branch (constant address space: other kernels
    // and the host write them, and the scalar cache starts clean)
    const __attribute__((address_space(4))) l2o_inst *ci = (const __attribute__((address_space(4))) l2o_inst *)in;
    const uint32_t phase = ci->phase, buf = (ci->base + (t ? t - 1 : 0)) & 1;
    const unsigned long long kprev = RUN ? ci->key[(t - 1) & 3] : L2O_KEY_NONE;
    const int n = (int)ci->n;
    const float slack = ci->slack;
    const uint32_t metric = ci->metric;
    const float es = ci->est_scale, ea = ci->est_add;
    const float qk = ci->qk, qm = ci->qm;
    l2o_pt *const p0 = ci->pts[0], *const p1 = ci->pts[1];
    unsigned long long *const pool = ci->pool;
    asm volatile("" ::"s"(phase), "s"(buf), "s"(kprev), "s"(n), "s"(slack), "s"(p0), "s"(p1), "s"(it.a0), "s"(it.b0),
                 "s"(it.rows), "s"(metric), "s"(qk), "s"(pool));
    if (phase != L2O_LO || kprev == L2O_SENTINEL) return;
    const gpt *__restrict__ P = (const gpt *)(buf ? p1 : p0);
    // the tour of this sweep: that of the buffer after the move kprev
    const move_map mm(kprev, n);
    auto src = [&](int k) __attribute__((always_inline)) { return RUN ? mm.src(k) : k; };

    constexpr bool PRUNE = MODE == L2O_SWEEP_PRUNE;
    constexpr int NT = 2 * K;         // column tiles of a wave
    constexpr int WC = 64 * K;        // columns of a wave
    constexpr int CH = 64 * WAVES;    // rows of a chunk
    constexpr int HCAP = 4 * K;       // pairs of tiles kept until they are evaluated
    __shared__ __attribute__((aligned(16))) uint4 s_row[2 * CH + 1];
    __shared__ __attribute__((aligned(16))) uint4 s_col[WAVES * WC];
    __shared__ uint32_t s_nh[WAVES * WC];
    __shared__ uint32_t s_list[WAVES][128];
    __shared__ uint32_t s_hdr[WAVES][HCAP];
    __shared__ uint4 s_rbox[PRUNE ? L2O_SWEEP_MAX_T / 32 + 2 * WAVES : 1], s_cbox[PRUNE ? WAVES * NT : 1];
    __shared__ int s_any[PRUNE ? WAVES : 1];
    const int a0 = (int)it.a0;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tid = (int)threadIdx.x;
    const int lane = tid & 63;
    const int bw = (int)it.b0 + w * WC;                                         // first column of this wave
    const int ncol = min(n - 1 - (int)it.b0, WAVES * WC);
    // rows a <= n-4 have candidates, and only rows a <= b-2 of the last column b
    const int rows = min(min((int)it.rows, n - 3 - a0), (int)it.b0 + ncol - 2 - a0);
    if (rows <= 0) return;

    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    typedef const __attribute__((address_space(1))) u32x2 *gdw;
    auto dw = [&](int k) __attribute__((always_inline)) { return *(gdw)&P[src(min(k, n - 1))].d; };  // {d, w}
    auto ld4 = [&](int k) __attribute__((always_inline)) {
        const int s = src(k);
        return make_uint4((uint32_t)P[s].x, (uint32_t)P[s].y, (uint32_t)P[s].d, (uint32_t)P[s].w);
    };
    // the move's new edge at position L (the one at 0 is no candidate's)
    int dL = 0;
    if constexpr (RUN) {
        const __attribute__((address_space(4))) l2o_pt *S = (const __attribute__((address_space(4))) l2o_pt *)(buf ? p1 : p0);
        const int u = mm.J - 1, v = max(mm.i - 1, 0);
        dL = exact_dist(S[u].x, S[u].y, S[v].x, S[v].y, metric);
    }
    // A range of positions mostly lies in one piece of the move: position k is then
    // S k + O before it, and an edge's length its later (S = 1) or earlier end's.
    struct piece {
        int S, O;
    };
    auto len = [&](int k, int d0, int d1) __attribute__((always_inline)) { return RUN ? mm.len(k, d0, d1, dL) : d1; };
    auto piece_of = [&](int lo, int hi) __attribute__((always_inline)) {  // S = 0: no single piece
        piece r{0, 0};
        if (!RUN) {
            if (hi < n) r = {1, 0};
        } else if (hi < n) {
            if (hi < mm.L) r = {1, mm.i};
            else if (lo >= mm.J) r = {-1, n - 1 + mm.J};
            else if (lo >= mm.L && hi < mm.J) r = {-1, mm.J - 1};
        }
        return r;
    };
    // {d, w} of position k and of k + 1
    struct ends {
        u32x2 v0, v1;
    };
    auto load_edge = [&](const piece &r, int k) __attribute__((always_inline)) {
        ends v;
        if (r.S) {
            const int s = RUN ? r.S * k + r.O : k;
            v.v0 = *(gdw)&P[s].d;
            v.v1 = *(gdw)&P[s + (RUN ? r.S : 1)].d;
        } else {
            v.v0 = dw(k);
            v.v1 = dw(k + 1);
        }
        return v;
    };
    auto edge = [&](const piece &r, int k, const ends &v) __attribute__((always_inline)) {  // k -> k+1
        const int d = !RUN || r.S > 0 ? (int)v.v1.x : r.S < 0 ? (int)v.v0.x : len(k + 1, (int)v.v0.x, (int)v.v1.x);
        return quant_edge(v.v0.y, v.v1.y, (uint32_t)d, qk, qm);
    };
    // columns bw .. bw+WC-1 per wave, the first chunk of rows
    qedge qc[K], qr;
    {
        const piece pc = piece_of(bw, bw + WC), pr = piece_of(a0, a0 + CH);
        ends vc[K];
#pragma unroll
        for (int m = 0; m < K; ++m) vc[m] = load_edge(pc, bw + 64 * m + lane);
        const ends vr = load_edge(pr, a0 + tid);
#pragma unroll
        for (int m = 0; m < K; ++m) qc[m] = edge(pc, bw + 64 * m + lane, vc[m]);
        qr = edge(pr, a0 + tid, vr);
    }
    // cap = the largest gain still worth an exact evaluation: the instance's,
    // or without a known move the best key published so far, taken inclusively
    // (it may come from a larger i: a tie at a smaller i wins)
    unsigned long long *const row = pool + (t & 3) * L2O_POOL;
    const int cap0 = RUN ? next_cap(pool[((t - 1) & 3) * L2O_POOL + lane], (uint32_t)mm.i, (uint32_t)mm.J) : ci->cap;
    int cap = cap0;
    if (cap0 == -1) {
        const unsigned long long g =
            uniform_u64(__hip_atomic_load(&in->key[t & 3], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        if (g != L2O_SENTINEL) cap = min(cap, worse_gain(key_gain(g)));
    }
    // half of -C (waves may start with different caps: each is a valid one)
    const float hc = half_cap(cap, qk);
    float thr = (float)cap + slack;  // of the FP32 estimate

    // PRUNE: the boxes of the columns and of all rows; an item without a pair of
    // tiles whose boxes meet ends here, before any operand is made (60,000
    // cities: 44.3 -> 35.5 us a step, most items end here; with five FP32
    // maxima a box and the operands made first they spent 700 VALU instructions
    // a wave)
    // (bit q K + p of live_of(c): row block q of the chunk from c, column pair p)
    auto live_of = [&](int c) __attribute__((always_inline)) -> unsigned long long {
        const int q = lane / K, p = lane % K;
        bool ok = false;
        if (q < 2 * WAVES && c + 32 * q < rows && bw + 64 * p + 63 >= a0 + c + 32 * q + 2) {
            const uint4 r = s_rbox[c / 32 + q], *cb = s_cbox + w * NT + 2 * p;
            ok = boxes_meet(r, cb[0]) || boxes_meet(r, cb[1]);
        }
        return __ballot(ok);
    };
    bool wave_live = true;
    if constexpr (PRUNE) {
#pragma unroll
        for (int m = 0; m < K; ++m) edge_boxes(qc[m], hc, bw + 64 * m + lane <= n - 2, lane, s_cbox + w * NT + 2 * m);
        edge_boxes(qr, hc, tid < rows, lane, s_rbox + 2 * w);
        for (int c = CH; c < rows; c += CH) {
            const piece pr = piece_of(a0 + c, a0 + c + CH);
            const qedge q = edge(pr, a0 + c + tid, load_edge(pr, a0 + c + tid));
            edge_boxes(q, hc, c + tid < rows, lane, s_rbox + c / 32 + 2 * w);
        }
        if constexpr (WAVES > 1) __syncthreads();
        asm volatile("" ::: "memory");
        wave_live = false;
        for (int c = 0; c < rows; c += CH) wave_live = wave_live || live_of(c) != 0;
        bool item_live = wave_live;
        if constexpr (WAVES > 1) {
            if (lane == 0) s_any[w] = wave_live;
            __syncthreads();
            item_live = false;
#pragma unroll
            for (int q = 0; q < WAVES; ++q) item_live = item_live || __builtin_amdgcn_readfirstlane(s_any[q]) != 0;
        }
        if (!item_live) return;
    }

    const bool upper = lane >= 32;
    half8 B[NT];
    uint4 *const scol = s_col + w * WC;
    uint32_t *const snh = s_nh + w * WC;
#pragma unroll
    for (int m = 0; m < K; ++m) {
        const bool valid = bw + 64 * m + lane <= n - 2;
        const qterms t = edge_terms(qc[m], hc, valid);
        scol[64 * m + lane] = col_record(qc[m], t);
        snh[64 * m + lane] = col_upper(t);
    }
    asm volatile("" ::: "memory");  // (the wave's own columns: LDS keeps its order)
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        uint4 v = scol[32 * t + (lane & 31)];
        v.x = upper ? snh[32 * t + (lane & 31)] : v.x;
        B[t] = __builtin_bit_cast(half8, v);
    }
    // the column stage now holds the sign masks of tile pairs with survivors
    asm volatile("" ::: "memory");
    uint32_t *const smask = (uint32_t *)scol;
    uint32_t *const slist = s_list[w];
    // row r of the item into its half of the chunk buffer
    auto stage_row = [&](const qedge &q, int r, int half) __attribute__((always_inline)) {
        const bool valid = r < rows;
        const qterms t = edge_terms(q, hc, valid);
        s_row[half * CH + tid] = row_record(q, t);
    };
    stage_row(qr, tid, 0);
    if (tid == 0) s_row[2 * CH] = row_const();

    unsigned long long lbest = L2O_SENTINEL, published = L2O_SENTINEL;
    unsigned fb = 0;
    int nh = 0;  // pairs kept

    // exact evaluation of the kept pairs' survivors
    auto drain = [&]() __attribute__((always_inline)) {
        asm volatile("" ::: "memory");
        int e = 0, cnt = 0;
        uint32_t m = 0, hdr = 0;
        for (;;) {
            // fill the list to a full wave
            while (cnt < 64) {
                unsigned long long any = __ballot(m != 0);
                if (!any) {
                    if (e >= nh) break;
                    m = smask[64 * e + lane];
                    hdr = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_hdr[w][e]);
                    ++e;
                    any = __ballot(m != 0);
                }
                if (m) {
                    const int bit = __builtin_ctz(m);
                    m &= m - 1;
                    const uint32_t row = (hdr >> 12) + (uint32_t)((bit & 3) + ((bit >> 2) & 3) * 8 + (lane >> 5) * 4);
                    const uint32_t col = (hdr & 0xFFFu) + (uint32_t)((bit >> 4) * 32 + (lane & 31));
                    slist[cnt + lanes_below(any)] = (row << 12) | col;
                }
                cnt += __builtin_popcountll(any);
            }
            if (cnt == 0) break;
            asm volatile("" ::: "memory");
            unsigned long long key = L2O_SENTINEL;
            if (lane < cnt) {
                const uint32_t v = slist[lane];
                const int a = a0 + (int)(v >> 12), b = bw + (int)(v & 0xFFFu);
                const uint4 A0 = ld4(a), A1 = ld4(a + 1), B0 = ld4(b), B1 = ld4(b + 1);
                const int da = len(a + 1, (int)A0.z, (int)A1.z), db = len(b + 1, (int)B0.z, (int)B1.z);
                const float w2 = (est_dist((int)A0.x, (int)A0.y, (int)B0.x, (int)B0.y, es, ea) +
                                  est_dist((int)A1.x, (int)A1.y, (int)B1.x, (int)B1.y, es, ea)) - (float)db;
                if (w2 <= thr + (float)da) {
                    ++fb;
                    const int gain = exact_dist((int)A0.x, (int)A0.y, (int)B0.x, (int)B0.y, metric) +
                                     exact_dist((int)A1.x, (int)A1.y, (int)B1.x, (int)B1.y, metric) - da - db;
                    if (gain < 0) key = make_key(gain, (uint32_t)(a + 1), (uint32_t)(b + 1));
                }
            }
            // into the pool; of many, the best of each 16 lanes (atomics on one
            // line take their turns, about 14 ns each)
            const unsigned long long got = __ballot(key != L2O_SENTINEL);
            if (got) {
                lbest = key < lbest ? key : lbest;
                if (__builtin_popcountll(got) > 16) {
                    key = dpp_min_u64<0x111, 0xF>(key);
                    key = dpp_min_u64<0x112, 0xF>(key);
                    key = dpp_min_u64<0x114, 0xF>(key);
                    key = dpp_min_u64<0x118, 0xF>(key);
                    if ((lane & 15) != 15) key = L2O_SENTINEL;
                }
                if (key != L2O_SENTINEL)
                    atomicMin(&row[(((uint32_t)(key >> 20) & 0xFFFFFu) * 0x9E3779B1u) >> 26], key);
            }
            // what was not evaluated moves to the front of the list
            uint32_t rest = 0;
            if (lane < cnt - 64) rest = slist[64 + lane];
            asm volatile("" ::: "memory");
            if (lane < cnt - 64) slist[lane] = rest;
            asm volatile("" ::: "memory");
            cnt = max(cnt - 64, 0);
            // publish an improvement at once: other waves tighten their cap
            if (__ballot(lbest < published)) {
                published = wave_min_u64(lbest);
                if (cap0 == -1) {
                    cap = min(cap, worse_gain(key_gain(published)));
                    thr = (float)cap + slack;
                }
                if (lane == 0) atomicMin(&in->key[t & 3], published);
            }
        }
        nh = 0;
    };

    const float16v zero = {0};
    // keeps the survivors of pair p and 32 rows from a0 + r0 (the two products
    // again: the loop below keeps only the combined signs)
    auto keep = [&](const half8 &A, int r0, int p) __attribute__((always_inline)) {
        const float16v c0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(A, B[2 * p], zero, 0, 0, 0);
        const float16v c1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(A, B[2 * p + 1], zero, 0, 0, 0);
        const int aq = a0 + r0, bp = bw + 64 * p;
        uint32_t mask = sign_mask(c0, c1);
        if (bp < aq + 33) {  // the pair meets the diagonal: candidates need a + 2 <= b
            const int l = bp + (lane & 31) - 2 - aq - (lane >> 5) * 4;
            mask &= rows_upto(l) | rows_upto(l + 32) << 16;
        }
        if (__ballot(mask != 0)) {
            smask[64 * nh + lane] = mask;
            if (lane == 0) s_hdr[w][nh] = (uint32_t)r0 << 12 | (uint32_t)(64 * p);
            ++nh;
        }
    };
    for (int c = 0, half = 0; c < rows; c += CH, half ^= 1) {
        // the next chunk's points, in flight while this one is tested
        ends nv{};
        piece np{};
        const bool more = c + CH < rows;
        if (more) {
            np = piece_of(a0 + c + CH, a0 + c + 2 * CH);
            nv = load_edge(np, a0 + c + CH + tid);
        }
        if constexpr (WAVES > 1) __syncthreads();
        asm volatile("" ::: "memory");
        const unsigned long long live = !PRUNE ? ~0ull : wave_live ? live_of(c) : 0ull;
        // rows of the chunk that this wave's columns see
        const int cr = min(min(rows - c, CH), min(bw + WC - 1, n - 2) - 1 - a0 - c);
        const int nq = bw > n - 2 ? 0 : (cr + 31) >> 5;
        // lanes 0..31 step through the rows, lanes 32..63 stay at the constant
        int ra = upper ? 2 * CH : half * CH + lane;
        const int rstep = upper ? 0 : 32;
        for (int q = 0; q < nq; ++q, ra += rstep) {
            const int r0 = c + 32 * q;
            if (PRUNE && !((live >> (q * K)) & ((1ull << K) - 1))) continue;
            const half8 A = __builtin_bit_cast(half8, s_row[ra]);
            uint32_t m[K], all = 0;
            if (PRUNE || bw < a0 + r0 + 33) {
                // pruned, or at the diagonal: pair by pair
#pragma unroll
                for (int p = 0; p < K; ++p) {
                    m[p] = (PRUNE ? (live >> (q * K + p)) & 1 : bw + 64 * p + 63 >= a0 + r0 + 2) ? 0x80000000u : 0u;
                    all |= m[p];
                }
            } else {
#pragma unroll
                for (int p = 0; p < K; ++p) {
                    m[p] = 0;
                    const float16v c0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(A, B[2 * p], zero, 0, 0, 0);
                    const float16v c1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(A, B[2 * p + 1], zero, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 16; ++r) m[p] |= __float_as_uint(c0[r]) | __float_as_uint(c1[r]);
                    all |= m[p];
                }
            }
            if (__ballot((int)all < 0)) {
#pragma unroll
                for (int p = 0; p < K; ++p)
                    if (__ballot((int)m[p] < 0)) keep(A, r0, p);
                if (nh + K > HCAP) drain();
            }
        }
        if (more) {
            qr = edge(np, a0 + c + CH + tid, nv);
            stage_row(qr, c + CH + tid, half ^ 1);
        }
    }
    if (nh) drain();

    const unsigned wfb = wave_sum_u32(fb);
    if (lane == 0 && wfb) atomicAdd(&in->fallbacks, (unsigned long long)wfb);
}

// waves per SIMD that the columns' operands leave room for (8 K VGPRs and about 55)
#define L2O_WPE(K) ((K) <= 2 ? 6 : (K) <= 4 ? 5 : (K) <= 6 ? 4 : 3)
// In a run, the first workgroups of a launch (na of them) write the
// sweep's tour to the other buffer and keep the books of the move they apply;
// the first chunk of an instance also carries its pool over and empties the
// next sweep's key and pool row.
template <int NTHR>
__device__ __forceinline__ void apply_item(const l2o_apply_item it, l2o_inst *__restrict__ insts,
                                           unsigned *__restrict__ live, uint32_t t)
{
    l2o_inst *in = insts + it.inst;
    const __attribute__((address_space(4))) l2o_inst *ci = (const __attribute__((address_space(4))) l2o_inst *)in;
    const unsigned long long kprev = ci->key[(t - 1) & 3];
    const uint32_t phase = ci->phase, buf = (ci->base + (t ? t - 1 : 0)) & 1;
    if (phase != L2O_LO) return;
    if (kprev == L2O_SENTINEL) {
        // no improving move: the local search has converged (sweeps = moves + 1)
        if (it.chunk == 0 && threadIdx.x < 64) local_optimum(in, live, buf);
        return;
    }
    const move_map mm(kprev, (int)ci->n);
    if (it.chunk == 0 && threadIdx.x < 64) {
        unsigned long long *const pool = ci->pool;
        const unsigned long long known = remap_key(pool[((t - 1) & 3) * L2O_POOL + threadIdx.x], (uint32_t)mm.i,
                                                   (uint32_t)mm.J, (uint32_t)mm.n);
        if (known != L2O_SENTINEL) atomicMin(&pool[(t & 3) * L2O_POOL + threadIdx.x], known);
        pool[((t + 1) & 3) * L2O_POOL + threadIdx.x] = L2O_SENTINEL;
        if (threadIdx.x == 0) {
            in->key[(t + 1) & 3] = L2O_SENTINEL;
            if (kprev != L2O_KEY_NONE) log_move(in, kprev);
        }
    }
    if (t) copy_chunk<NTHR>(ci, buf, mm, ci->metric, (int)(it.chunk * L2O_APPLY_CHUNK));
}

template <int K, int WAVES, int MODE, bool RUN>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(L2O_WPE(K)))) void k_sweep(
    const l2o_sweep_item *__restrict__ items, const l2o_apply_item *__restrict__ aitems, uint32_t na,
    l2o_inst *__restrict__ insts, unsigned *__restrict__ live, uint32_t t)
{
    if (RUN && blockIdx.x < na) apply_item<64 * WAVES>(aitems[blockIdx.x], insts, live, t);
    else sweep_item<K, WAVES, MODE, RUN>(items[blockIdx.x - (RUN ? na : 0)], insts, t);
}

// column and wave counts compiled into the library, and the tile shapes {k, t,
// waves} the autotuner chooses among per n bucket (t, the rows of an item, is
// up to the host)
#define L2O_SWEEP_KERNELS(X) X(1, 1) X(2, 1) X(4, 1) X(6, 1) X(8, 1) X(4, 2) X(6, 2) X(8, 2) X(2, 4) X(4, 4) X(6, 4) X(8, 4)
static const int g_shapes[][3] = {  // t <= L2O_SWEEP_MAX_T
    {1, 32, 1}, {1, 64, 1}, {2, 64, 1}, {2, 128, 1}, {4, 64, 1}, {4, 128, 1}, {4, 256, 1}, {6, 64, 1}, {6, 128, 1},
    {8, 64, 1}, {8, 128, 1}, {8, 256, 1}, {4, 64, 2}, {4, 128, 2}, {6, 64, 2}, {8, 64, 2}, {8, 128, 2}, {8, 256, 2},
    {2, 64, 4}, {4, 64, 4}, {6, 64, 4}, {8, 64, 4}, {8, 128, 4}, {6, 128, 2}, {6, 160, 1}, {6, 128, 4}, {4, 256, 2},
    {4, 256, 4}, {2, 256, 4}, {2, 512, 4}, {4, 512, 4}};

template <int K, int W, int MODE>
static void launch_shape(uint32_t nitems, uint32_t na, bool run, hipStream_t stream, const l2o_sweep_item *items,
                         const l2o_apply_item *aitems, l2o_inst *insts, unsigned *live, uint32_t t)
{
    if (run)
        hipLaunchKernelGGL((k_sweep<K, W, MODE, true>), dim3(na + nitems), dim3(64 * W), 0, stream, items, aitems, na,
                           insts, live, t);
    else
        hipLaunchKernelGGL((k_sweep<K, W, MODE, false>), dim3(nitems), dim3(64 * W), 0, stream, items, aitems, 0u, insts,
                           live, 0u);
}

#define L2O_SWEEP_CASE(K_, W_)                                                                              \
    if (cfg.k == K_ && cfg.waves == W_) {                                                                  \
        if (mode == L2O_SWEEP_PRUNE)                                                                        \
            launch_shape<K_, W_, L2O_SWEEP_PRUNE>(nitems, na, run, stream, items, aitems, insts, live, t);  \
        else                                                                                                \
            launch_shape<K_, W_, L2O_SWEEP_FULL>(nitems, na, run, stream, items, aitems, insts, live, t);   \
        return hipGetLastError();                                                                           \
    }

hipError_t launch_sweep(const sweep_cfg &cfg, const l2o_sweep_item *items, uint32_t nitems,
                        const l2o_apply_item *aitems, uint32_t na, l2o_inst *insts, unsigned *live, bool run,
                        uint32_t t, hipStream_t stream, int mode)
{
    if (nitems == 0) return hipSuccess;
    if (mode != L2O_SWEEP_FULL && mode != L2O_SWEEP_PRUNE) return hipErrorInvalidValue;
    L2O_SWEEP_KERNELS(L2O_SWEEP_CASE)
    return hipErrorInvalidValue;
}

bool sweep_cfg_supported(const sweep_cfg &c)
{
    for (const auto &r : g_shapes)
        if (r[0] == c.k && r[1] == c.t && r[2] == c.waves) return true;
    return false;
}

int sweep_shapes(int (*out)[3], int cap)
{
    const int m = (int)(sizeof(g_shapes) / sizeof(g_shapes[0]));
    for (int q = 0; q < m && q < cap; ++q) {
        out[q][0] = g_shapes[q][0];
        out[q][1] = g_shapes[q][1];
        out[q][2] = g_shapes[q][2];
    }
    return m;
}

}  // namespace l2o
