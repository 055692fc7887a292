// Arithmetic shared by the field consumers: bins of uint16 values, division by
// a shared divisor, 16-byte chunk loads.
#ifndef MXB_HIST_H
#define MXB_HIST_H

#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "mxb_field_plan.h"

namespace mxb {

// bin(v) = floor(c * ((v - lo) / d)) in float64 (cpu/histograms.cc:62, :279,
// :292), counted where vlo <= v <= vhi and 0 <= bin <= c.
//
// A table over the 65536 values would make every voxel a scattered read (up
// to 64 cache lines per wave), so the kernels evaluate the expression.  The
// division is done with the correctly rounded reciprocal rd = 1/d and one
// residual: q0 = x rd, q = q0 + (x - q0 d) rd with FMAs, which is the
// correctly rounded x / d whenever d's significand is not all ones (Markstein,
// IBM J. Res. Dev. 34(1), 1990); `fast` says that this and the ranges hold,
// else the kernels divide.
struct BinMap {
    double lo, d, rd, c;
    uint32_t vlo, vhi;
    int fast;
};

// mask_range: values outside [lo, hi] are not counted (the voxel axis);
// otherwise every nonzero value with a bin in range is (the field axis).
BinMap make_bin_map(double lo, double hi, int64_t nbins, bool mask_range);

// The bin of v, or kNoBin (bin counts multiply to less than 2^32 - 1, so a bin
// may be 2^31 or more).
constexpr uint32_t kNoBin = 0xffffffffu;
template <bool FAST>
__device__ __forceinline__ uint32_t bin_of(uint32_t v, const BinMap &m) {
#pragma clang fp contract(off)
    const double x = (double)v - m.lo;
    double q;
    if constexpr (FAST) {
        q = x * m.rd;
        q = __builtin_fma(__builtin_fma(-q, m.d, x), m.rd, q);
    } else {
        q = x / m.d;
    }
    const double t = m.c * q;
    // t < c + 1 and t >= 0 exactly when floor(t) is a bin (false for NaN)
    const bool ok = v - m.vlo <= m.vhi - m.vlo && t >= 0.0 && t < m.c + 1.0;
    return ok ? (uint32_t)t : kNoBin;
}

// Float32 division of many values by one: the correctly rounded quotient from
// the correctly rounded reciprocal and one residual (Markstein, as above),
// where d is far from under- and overflow and its significand is not all
// ones (`exact`); the dividends must be 0 or within 2^40 of d.
struct SharedDiv {
    float d, r;
    bool exact;
    __device__ __forceinline__ explicit SharedDiv(float divisor) : d(divisor), r(1.0f / divisor) {
        const uint32_t b = __float_as_uint(d);
        exact = d > 0x1p-40f && d < 0x1p40f && (b & 0x7fffffu) != 0x7fffffu;
    }
    __device__ __forceinline__ float quick(float x) const {
        const float q = x * r;
        return __builtin_fmaf(__builtin_fmaf(-q, d, x), r, q);
    }
};

// Elements 8 c .. 8 c + 7 of `base` (16-byte aligned); those outside [b, e)
// are not read and come back as 0.
__device__ __forceinline__ void load_chunk(const uint16_t *__restrict__ base, int64_t c, int64_t b, int64_t e,
                                           uint16_t q[8]) {
    const int64_t e0 = c * 8;
    if (e0 >= b && e0 + 8 <= e) {
        const uint4 u = *reinterpret_cast<const uint4 *>(base + e0);
        const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int k = 0; k < 8; ++k) q[k] = (uint16_t)(w[k >> 1] >> (16 * (k & 1)));
    } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) q[k] = e0 + k >= b && e0 + k < e ? base[e0 + k] : (uint16_t)0;
    }
}

// Field histogram, enqueued on `s`.  `words` receives the host tables that are
// copied to the start of `ws`: they must outlive the copy.
hipError_t launch_field_histogram(const uint16_t *vox, int64_t nZ, int64_t nY, int64_t nX, const uint16_t *field,
                                  int64_t nz, int64_t ny, int64_t nx, uint64_t *bins, int64_t fb, int64_t vb,
                                  double vmin, double vmax, double fmin, double fmax, void *ws,
                                  std::vector<int32_t> &words, hipStream_t s);

}  // namespace mxb

#endif  // MXB_HIST_H
