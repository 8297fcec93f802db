// l2o_launch.h -- host-side launch wrappers for the kernels in l2o_kernels.hip.
#pragma once
#include <hip/hip_runtime.h>

#include <math.h>

#include "l2o_state.h"

namespace l2o {

// Edge-length metrics (TSPLIB EDGE_WEIGHT_TYPE), for integer s = dx^2 + dy^2:
//   EUC_2D  nint(sqrt(s))
//   CEIL_2D ceil(sqrt(s))
//   ATT     ceil(sqrt(s / 10)): TSPLIB's t = nint(r), r = sqrt(s/10), plus 1
//           when t < r, equals ceil(r) for every s (when r is not an integer,
//           nint(r) < r exactly when the fraction of r is below 1/2)
enum : uint32_t { L2O_EUC_2D = 0, L2O_CEIL_2D = 1, L2O_ATT = 2 };

// Exact metric length.  With f = 10 for ATT and 1 otherwise,
// m = floor(sqrt(s / f)) satisfies f m^2 <= s < f (m+1)^2, and
//   EUC_2D  nint(sqrt(s)) = m + [s > m^2 + m]  (sqrt(s) is never m + 1/2)
//   CEIL_2D               = m + [s > m^2]
//   ATT                   = m + [s > 10 m^2]
// The FP64 square root starts m within one of the floor; the integer
// comparisons make it exact (s < 2^45 here).
__host__ __device__ inline int32_t metric_dist(long long s, uint32_t metric)
{
    const long long f = metric == L2O_ATT ? 10 : 1;
    const long long e = metric == L2O_EUC_2D ? 1 : 0;
    long long m = (long long)sqrt((double)s * (metric == L2O_ATT ? 0.1 : 1.0));
    if (f * m * m > s) m -= 1;
    else if (f * (m + 1) * (m + 1) <= s) m += 1;
    return (int32_t)(m + (s > f * m * m + e * m ? 1 : 0));
}

// Quantised geometry of the sweep's matrix test (see l2o_sweep.hip).  A city
// (x, y) becomes X and Y, x qs + qox and y qs + qoy rounded to whole numbers in
// [-L2O_QR, L2O_QR]; an edge of length D becomes E = ceil(D qk + qm) <= L2O_QE,
// where qk >= qs kappa (kappa = sqrt(10) for ATT, else 1) and qm covers half
// of the metric's rounding (d < D + 1/2 for EUC_2D) and of the rounding of the
// coordinates.  With these limits every partial sum of the test is a whole
// number below 2^24, exact in FP32 in any order.
#define L2O_QR 640
#define L2O_QE 1830
__host__ inline void set_quant(l2o_inst &in, double span_x, double span_y)
{
    const double half = 0.5 * (span_x > span_y ? span_x : span_y);
    in.qs = (float)(half * 4.0 <= 639.0 ? 4.0 : 639.0 / half);
    in.qox = (float)(-0.5 * span_x * (double)in.qs);
    in.qoy = (float)(-0.5 * span_y * (double)in.qs);
    const double kappa = in.metric == L2O_ATT ? sqrt(10.0) : 1.0;
    in.qk = nextafterf((float)((double)in.qs * kappa), 1e30f);
    in.qm = (float)(1.02 + (in.metric == L2O_EUC_2D ? 0.5 * (double)in.qs : 0.0));
}

// FP16 bits of a whole number |v| <= 2048 given as a float (exact)
__host__ __device__ inline uint32_t f16_of_whole(float v)
{
    union {
        float f;
        uint32_t u;
    } b;
    b.f = v;
    const uint32_t m = b.u & 0x7FFFFFFFu;
    return ((b.u >> 16) & 0x8000u) | (m ? (m >> 13) - (112u << 10) : 0u);
}

// l2o_pt.w of a city: X and Y as a pair of FP16 numbers (rounded to the nearest
// whole number by truncation of a positive one)
__host__ __device__ inline int32_t quant_xy(float qs, float qox, float qoy, int32_t x, int32_t y)
{
    const float fx = (float)x * qs + qox, fy = (float)y * qs + qoy;
    const int32_t X = (int32_t)(fx + 1024.5f) - 1024, Y = (int32_t)(fy + 1024.5f) - 1024;
    return (int32_t)(f16_of_whole((float)X) | (f16_of_whole((float)Y) << 16));
}

// Sweep tile shape: each workgroup has `waves` wave64s on the same `t` rows,
// each wave with 64 k columns of its own (2 k matrix tiles of 32 columns).
struct sweep_cfg {
    int k;
    int t;
    int waves;
    int cols() const { return waves * 64 * k; }
};

bool sweep_cfg_supported(const sweep_cfg &c);
// compiled shapes: fills up to cap rows {k, t, waves}, returns the total count
int sweep_shapes(int (*out)[3], int cap);
// Sweep variants (same results): every pair of tiles through the matrix test,
// or only those that a bounding-box bound does not rule out
enum { L2O_SWEEP_FULL = 0, L2O_SWEEP_PRUNE = 1 };
// one workgroup per item, of the variant `mode`: sweep t of a run (l2o_state.h),
// with one workgroup per apply item of the same instances, or a sweep by itself
hipError_t launch_sweep(const sweep_cfg &cfg, const l2o_sweep_item *items, uint32_t nitems,
                        const l2o_apply_item *aitems, uint32_t na, l2o_inst *insts, unsigned *live, bool run,
                        uint32_t t, hipStream_t stream, int mode);
// the end of a run of t sweeps, or of a sweep by itself (t = 0)
hipError_t launch_apply(const l2o_apply_item *items, uint32_t nitems, l2o_inst *insts, unsigned *live, uint32_t t,
                        hipStream_t stream);
// ILS bookkeeping before sweep tnext of a run
hipError_t launch_ils(l2o_inst *insts, uint32_t nslots, unsigned *live, uint32_t tnext, hipStream_t stream);
// `steps` sweeps of each of the instances ids[0 .. count), none larger than
// max_n cities: one workgroup each (a chain of a group stops at its local
// optimum, L2O_LO_DONE)
hipError_t launch_local(int waves, const uint32_t *ids, uint32_t count, uint32_t max_n, l2o_inst *insts, unsigned *live,
                        uint32_t steps, hipStream_t stream);
uint32_t local_lds_bytes(uint32_t n, int waves);
hipError_t launch_group(l2o_inst *insts, uint32_t nslots, unsigned *live, hipStream_t stream);
// admission, release and result of a slot (l2o_kernels.hip)
// (`rec` and `raw`: pinned host memory, 16-byte aligned, a multiple of 16 bytes;
// `count`: the slot was not live)
hipError_t launch_load(l2o_inst *insts, uint32_t slot, uint32_t n, const l2o_inst *rec, const void *raw, unsigned *live,
                       bool count, hipStream_t stream);
hipError_t launch_prime(l2o_inst *insts, uint32_t slot, uint32_t n, hipStream_t stream);  // after launch_load
hipError_t launch_free(l2o_inst *insts, uint32_t slot, unsigned *live, bool running, bool clear_pool, hipStream_t stream);
hipError_t launch_fetch(const l2o_inst *insts, uint32_t slot, uint32_t n, l2o_inst *rec, uint32_t *tour,
                        hipStream_t stream);
hipError_t launch_length(const l2o_inst *insts, uint32_t slot, uint32_t n, unsigned long long *out,
                         hipStream_t stream);
hipError_t launch_sqrt_ulp(uint32_t lo, uint32_t hi, unsigned *max_ulp, hipStream_t stream);

}  // namespace l2o
