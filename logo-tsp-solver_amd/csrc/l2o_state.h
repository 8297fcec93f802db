// l2o_state.h -- device-resident instance state shared by the host engine and
// the gfx950 kernels.
//
// Per instance (n cities) HBM holds, 16-byte aligned:
//   pts[2][n]  l2o_pt {x, y, D, W}   tour-ordered points (ping-pong): integer
//                                     coordinates shifted into [0, 2^22),
//                                     D[k] = exact metric length of the edge
//                                     P[k-1] -> P[k] (EUC_2D, CEIL_2D or ATT),
//                                     D[0] the closing edge, W[k] the
//                                     quantised coordinates of P[k]
//   tour[2][n] uint32                 city ids in the same order (ping-pong)
//   bpts[n], btour[n]                 best tour of an ILS run
//   log[log_cap]                      applied moves {i, J, gain}
// The reference keeps the tour on the host and re-uploads ordered
// coordinates every move (CUDASolver.cpp:316-329); here both stay resident and
// the move is applied by a device gather.
#pragma once
#include <stdint.h>

#define L2O_SENTINEL 0xFFFFFFFFFFFFFFFFull

// key = ((gain + 2^24) << 40) | (i << 20) | J   for gain < 0, i < J < 2^20.
// Unsigned order of keys is the lexicographic order of (gain, i, J), so the
// minimum key is the reference's strict-'<' scan winner
// (cpuSolver.cpp:140-145) and an atomicMin reduction is order independent.
#define L2O_KEY_GAIN_BIAS (1ll << 24)

enum l2o_phase : uint32_t {
    L2O_FREE = 0,     // slot unused
    L2O_LO = 1,       // local search running: sweep + apply every step
    L2O_LO_DONE = 2,  // local optimum reached, ILS bookkeeping pending
    L2O_DONE = 3,     // finished (result ready)
    L2O_WAIT = 4,     // chain of a group at a local optimum, waiting for the others
    L2O_KICK = 5,     // chain of a group: kick from `kick_src`'s best, then local search
};

#define L2O_NO_GROUP 0xFFFFFFFFu

struct __attribute__((aligned(16))) l2o_pt {
    int32_t x, y;  // coordinates, 0 <= x, y < 2^22
    int32_t d;     // exact metric length of the edge into this point
    int32_t w;     // the point's quantised coordinates (quant_xy in l2o_launch.h)
};

struct l2o_move {
    uint32_t i;
    uint32_t j;
    int32_t gain;
};

struct l2o_inst {
    // ---- fixed at admission
    l2o_pt *pts[2];
    uint32_t *tour[2];
    l2o_pt *bpts;
    uint32_t *btour;
    l2o_move *log;
    unsigned long long *rlog;  // ILS: best length after the first LO and each round
    uint32_t n;
    uint32_t log_cap;
    float slack;          // bound on |exact gain - FP32 estimate| (see l2o_kernels.hip)
    uint32_t ils_rounds;  // 0 = local search only
    uint32_t kick;
    uint32_t have_best;
    uint32_t metric;      // edge length: L2O_EUC_2D, L2O_CEIL_2D or L2O_ATT
    uint32_t group_lead;  // multi-start ILS: first slot of the group (L2O_NO_GROUP: none)
    uint32_t group_size;  // chains in the group (slots group_lead .. group_lead+size-1)
    uint32_t improved;    // the chain's last local search improved its own best
    uint32_t kick_src;    // slot whose best tour the next kick starts from
    float est_scale;      // FP32 estimate: D ~ sqrt(s) * est_scale + est_add
    float est_add;
    float qs, qox, qoy;   // matrix test: X ~ x qs + qox, Y ~ y qs + qoy,
    float qk, qm;         // and E = ceil(D qk + qm) (set_quant in l2o_launch.h)
    unsigned long long stop_below;  // ILS: done once best_length < stop_below (0: never)
    unsigned long long *pool;       // 4 rows of L2O_POOL keys of known improving moves (below)
    // ---- dynamic
    uint32_t phase;
    uint32_t parity;      // buffer of the current tour (outside of a run of sweeps)
    uint32_t base;        // buffer of the tour that a run's first sweep reads (below)
    int32_t cap;          // largest gain the sweep of T_0 evaluates (next_cap in l2o_device.h)
    uint32_t apply_done;  // last-workgroup counter of the apply kernel
    uint32_t rounds_done;
    unsigned long long key[4];
    unsigned long long length;
    unsigned long long best_length;
    unsigned long long moves;
    unsigned long long sweeps;
    unsigned long long fallbacks;
    unsigned long long rng[4];
};

// One workgroup of the sweep kernel: rows a in [a0, a0 + rows) and columns b
// in [b0, b0 + 64 * waves * k) of the candidate triangle a + 2 <= b <= n - 2;
// rows <= T of the launch's shape (the tail of a launch uses shorter items).
struct l2o_sweep_item {
    uint32_t inst;
    uint32_t a0;
    uint32_t b0;
    uint32_t rows;
};

// One workgroup of the apply kernel: elements [chunk*CHUNK, (chunk+1)*CHUNK).
struct l2o_apply_item {
    uint32_t inst;
    uint32_t chunk;
};

// A run of sweeps.  Sweep t of a run (t = 0, 1, ...) works on the tour T_t and
// leaves its best move in key[t & 3].  T_0 is in buffer `base`; T_t (t > 0) is
// the tour of buffer (base + t - 1) & 1 after the move key[(t-1) & 3], which the
// sweep applies to every index it reads while some of its workgroups write T_t
// to the other buffer.  So a move costs one launch.  key[(t-1) & 3] is
// L2O_KEY_NONE where there is no move to apply (t = 0, or a new tour from a
// kick) and L2O_SENTINEL where T_(t-1) was a local optimum.  Sweep t also
// empties key and pool row t+1.  After the last sweep k_apply brings the tour
// to a buffer of its own and the state back to t = 0: key[3] = L2O_KEY_NONE,
// key[0] = L2O_SENTINEL, the pool in row 3, row 0 empty.
#define L2O_KEY_NONE 0ull

// Keys of improving candidates the sweeps have evaluated exactly, bucketed by
// position: row t & 3 for those of T_t.  They are carried over to the next tour,
// whose sweep starts with the best of them as its bound.  All rows are
// L2O_SENTINEL at a local optimum.
#define L2O_POOL 64
#define L2O_MAX_GROUPS 32  // distinct sweep tile shapes in one engine step
#define L2O_APPLY_CHUNK 1024
#define L2O_APPLY_THREADS 256
#define L2O_ILS_THREADS 1024
