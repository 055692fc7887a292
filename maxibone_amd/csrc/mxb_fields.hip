// Consumers of the diffusion field (gfx950): field combination, and the C
// entries of the 2D histograms (kernels in mxb_histograms.hip).  C ABI in
// include/maxibone_fields.h.
//
// Combination (0975_combine_fields.py:41-62, float32 in the script's order):
//   c = g/gmax - e/emax;  c' = c + |min c|;  w = c' / max c';  v = w * cyl;
//   out = cyl * (uint16)((v - min v) / (max v - min v) * 65535)
// Rounding is monotone, so max c' = fl(max c + a), and min/max of v follow
// from min/max of c over the cylinder; three passes therefore reproduce the
// script exactly: (1) max g, max e; (2) min/max of c overall and inside the
// cylinder; (3) the output.  Each pass reads the reductions of the one before
// from the workspace, so nothing returns to the host in between.
//
// The passes read 4, 4 and 4 bytes per voxel and write 2 in the last: 2.6 ms
// at the copy rate for 1024^3.  A volume is walked as planes (the cylinder
// mask is one plane, which a thread reads once), a thread taking 8 neighbours
// of a plane at any alignment through the planes of its block.  The divisors
// are shared by all voxels: SharedDiv (mxb_hist.h) divides in 3 instructions.
// 1024^3: 5.8 -> 2.6 ms; before, IEEE division sequences (up to three per
// voxel) bound the passes, and the host read the reductions back twice.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <type_traits>
#include <vector>

#include "maxibone_diffusion.h"
#include "maxibone_fields.h"
#include "mxb_hist.h"
#include "mxb_internal.h"

namespace mxb {

constexpr int kThreads = 256;
constexpr int kPerThread = 8;

// Orderable encoding of a float for atomic min / max on uint32.
__device__ __forceinline__ uint32_t f2ord(float f) {
    const uint32_t b = __float_as_uint(f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float ord2f(uint32_t o) {
    return __uint_as_float((o & 0x80000000u) ? (o & 0x7fffffffu) : ~o);
}

__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
    for (int o = 32; o > 0; o >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, o));
    return v;
}
__device__ __forceinline__ uint32_t wave_min(uint32_t v) {
    for (int o = 32; o > 0; o >>= 1) v = min(v, (uint32_t)__shfl_xor((int)v, o));
    return v;
}

// ws[0] = max g, ws[1] = max e, ws[2..5] = ord(min c), ord(max c),
// ord(min c | cyl), ord(max c | cyl); ws[6], ws[7]: some voxel lies inside,
// outside the cylinder.
constexpr int kWsWords = 8;

__global__ __launch_bounds__(64) void k_fields_init(uint32_t *ws) {
    if (threadIdx.x < kWsWords) ws[threadIdx.x] = threadIdx.x == 2 || threadIdx.x == 4 ? 0xffffffffu : 0u;
}

// A thread's 8 elements of a plane, at e0; `left` of them exist.
struct Piece {
    int64_t e0;
    int left;
    __device__ __forceinline__ explicit Piece(int64_t plane) {
        e0 = ((int64_t)blockIdx.x * kThreads + threadIdx.x) * kPerThread;
        left = plane - e0 < kPerThread ? (int)(plane - e0 > 0 ? plane - e0 : 0) : kPerThread;
    }
    // FULL: all 8 exist, one 16-byte load (through a whole vector: an array of
    // uint16 makes the compiler merge its first element with the other branch
    // and split the rest); else elements that do not exist read as 0
    template <bool FULL>
    __device__ __forceinline__ void load(const uint16_t *__restrict__ p, uint16_t v[kPerThread]) const {
        if constexpr (FULL) {
            uint4 q;
            __builtin_memcpy(&q, p + e0, 16);
            const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
            for (int k = 0; k < kPerThread; ++k) v[k] = (uint16_t)(w[k >> 1] >> (16 * (k & 1)));
        } else {
#pragma unroll
            for (int k = 0; k < kPerThread; ++k) v[k] = k < left ? p[e0 + k] : (uint16_t)0;
        }
    }
    // f(true_type) for whole pieces, f(false_type) for partial ones: the choice
    // stays outside the loops, whose loads then overlap
    template <typename F>
    __device__ __forceinline__ void each(F &&f) const {
        if (left == kPerThread) f(std::true_type{});
        else if (left > 0) f(std::false_type{});
    }
    // bit k: element k lies inside the cylinder
    __device__ __forceinline__ uint32_t inside(const uint8_t *__restrict__ cyl) const {
        uint32_t in = 0;
#pragma unroll
        for (int k = 0; k < kPerThread; ++k)
            if (k < left && (cyl == nullptr || cyl[e0 + k] != 0)) in |= 1u << k;
        return in;
    }
};

// Reduces v over the block with f (max or min) and folds it into *dst, one
// atomic, only where it improves what is there.
template <bool MAX>
__device__ __forceinline__ void fold(uint32_t v, uint32_t *dst) {
    __shared__ uint32_t red[kThreads / 64];
    v = MAX ? wave_max(v) : wave_min(v);
    __syncthreads();  // red is free again
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int i = 1; i < kThreads / 64; ++i) v = MAX ? max(v, red[i]) : min(v, red[i]);
    const uint32_t now = __hip_atomic_load(dst, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (MAX ? v > now : v < now) {
        if (MAX) atomicMax(dst, v);
        else atomicMin(dst, v);
    }
}

__global__ __launch_bounds__(kThreads) void k_max2(const uint16_t *__restrict__ a, const uint16_t *__restrict__ b,
                                                   int64_t nz, int64_t plane, uint32_t *ws) {
    const Piece p(plane);
    uint16_t ma[kPerThread] = {}, mb[kPerThread] = {};
    p.each([&](auto full) {
#pragma unroll 4
        for (int64_t z = blockIdx.y; z < nz; z += gridDim.y) {
            uint16_t va[kPerThread], vb[kPerThread];
            p.load<decltype(full)::value>(a + z * plane, va);
            p.load<decltype(full)::value>(b + z * plane, vb);
#pragma unroll
            for (int k = 0; k < kPerThread; ++k) {
                ma[k] = va[k] > ma[k] ? va[k] : ma[k];
                mb[k] = vb[k] > mb[k] ? vb[k] : mb[k];
            }
        }
    });
    uint32_t xa = 0, xb = 0;
#pragma unroll
    for (int k = 0; k < kPerThread; ++k) {
        xa = max(xa, (uint32_t)ma[k]);
        xb = max(xb, (uint32_t)mb[k]);
    }
    fold<true>(xa, ws);
    fold<true>(xb, ws + 1);
}

// g / gmax - e / emax: the maxima are whole numbers below 2^16, which SharedDiv
// divides exactly (all 2^32 quotients compared).
__device__ __forceinline__ float combine_c(uint16_t g, uint16_t e, const SharedDiv &gm, const SharedDiv &em) {
    return gm.quick((float)g) - em.quick((float)e);
}

__global__ __launch_bounds__(kThreads) void k_combine_minmax(const uint16_t *__restrict__ g,
                                                             const uint16_t *__restrict__ e,
                                                             const uint8_t *__restrict__ cyl, int64_t nz,
                                                             int64_t plane, uint32_t *ws) {
    if (ws[0] == 0 || ws[1] == 0) return;  // refused by the host
    const SharedDiv gm((float)ws[0]), em((float)ws[1]);
    const Piece p(plane);
    const uint32_t in = p.inside(cyl);
    float lo = INFINITY, hi = -INFINITY, lo_c = INFINITY, hi_c = -INFINITY;
    p.each([&](auto full) {
#pragma unroll 4
        for (int64_t z = blockIdx.y; z < nz; z += gridDim.y) {
            uint16_t vg[kPerThread], ve[kPerThread];
            p.load<decltype(full)::value>(g + z * plane, vg);
            p.load<decltype(full)::value>(e + z * plane, ve);
#pragma unroll
            for (int k = 0; k < kPerThread; ++k) {
                const float c = combine_c(vg[k], ve[k], gm, em);
                if (decltype(full)::value || k < p.left) {
                    lo = fminf(lo, c);
                    hi = fmaxf(hi, c);
                }
                if (in >> k & 1) {
                    lo_c = fminf(lo_c, c);
                    hi_c = fmaxf(hi_c, c);
                }
            }
        }
    });
    const uint32_t some_in = in != 0, some_out = in != (1u << p.left) - 1;
    fold<false>(lo <= hi ? f2ord(lo) : 0xffffffffu, ws + 2);
    fold<true>(lo <= hi ? f2ord(hi) : 0u, ws + 3);
    fold<false>(lo_c <= hi_c ? f2ord(lo_c) : 0xffffffffu, ws + 4);
    fold<true>(lo_c <= hi_c ? f2ord(hi_c) : 0u, ws + 5);
    if (blockIdx.y == 0) {
        fold<true>(some_in, ws + 6);
        fold<true>(some_out, ws + 7);
    }
}

__global__ __launch_bounds__(kThreads) void k_combine_out(const uint16_t *__restrict__ g,
                                                          const uint16_t *__restrict__ e,
                                                          const uint8_t *__restrict__ cyl, int64_t nz, int64_t plane,
                                                          const uint32_t *__restrict__ ws,
                                                          uint16_t *__restrict__ out) {
    if (ws[0] == 0 || ws[1] == 0) return;  // refused by the host
    const SharedDiv gm((float)ws[0]), em((float)ws[1]);
    const float cmin = ord2f(ws[2]), cmax = ord2f(ws[3]);
    const float a = fabsf(cmin);        // combined += np.abs(combined.min())
    const SharedDiv M(cmax + a);        // combined /= combined.max()
    float vmin = 0.0f, vmax = 0.0f;
    if (ws[6] != 0) {
        const float wmin = (ord2f(ws[4]) + a) / M.d;
        const float wmax = (ord2f(ws[5]) + a) / M.d;
        vmin = ws[7] != 0 ? fminf(0.0f, wmin) : wmin;
        vmax = ws[7] != 0 ? fmaxf(0.0f, wmax) : wmax;
    }
    // min_max starts vmax at numeric_limits<float>::min(), the smallest
    // positive normal (general.hh:78)
    vmax = fmaxf(vmax, FLT_MIN);
    const SharedDiv range(vmax - vmin);  // general.hh:100, (float)vmax - (float)vmin
    const Piece p(plane);
    const uint32_t in = p.inside(cyl);
    auto convert = [&](auto by) {
        p.each([&](auto full) {
#pragma unroll 2
            for (int64_t z = blockIdx.y; z < nz; z += gridDim.y) {
                uint16_t vg[kPerThread], ve[kPerThread];
                p.load<decltype(full)::value>(g + z * plane, vg);
                p.load<decltype(full)::value>(e + z * plane, ve);
                uint32_t q[kPerThread];
#pragma unroll
                for (int k = 0; k < kPerThread; ++k) {
                    const float v = by(combine_c(vg[k], ve[k], gm, em) + a, M);
                    const float s = by(v - vmin, range) * 65535.0f;  // general.hh:100
                    q[k] = (in >> k & 1) && range.d > 0.0f ? (uint32_t)s & 0xffffu : 0u;  // x cylinder mask
                }
                uint16_t *const o = out + z * plane + p.e0;
                if constexpr (decltype(full)::value) {
                    const uint4 w = make_uint4(q[0] | q[1] << 16, q[2] | q[3] << 16, q[4] | q[5] << 16, q[6] | q[7] << 16);
                    __builtin_memcpy(o, &w, 16);
                } else {
                    for (int k = 0; k < p.left; ++k) o[k] = (uint16_t)q[k];
                }
            }
        });
    };
    // a volume of one value has M or range 0 or tiny: IEEE division
    if (M.exact && range.exact) convert([](float x, const SharedDiv &d) { return d.quick(x); });
    else convert([](float x, const SharedDiv &d) { return x / d.d; });
}

#define MXB_FHIP(expr)                                                          \
    do {                                                                        \
        hipError_t _e = (expr);                                                 \
        if (_e != hipSuccess) {                                                 \
            set_error(std::string(#expr) + ": " + hipGetErrorString(_e));       \
            return _e == hipErrorOutOfMemory ? ENOMEM_ : EDEVICE;               \
        }                                                                       \
    } while (0)

// As MXB_FHIP, for calls made after a copy from a host table was queued on
// `s`: an error path first waits for the stream, so the copy never reads the
// table after it is freed.
#define MXB_FHIP_AFTER_COPY(expr, s)                                            \
    do {                                                                        \
        hipError_t _e = (expr);                                                 \
        if (_e != hipSuccess) {                                                 \
            set_error(std::string(#expr) + ": " + hipGetErrorString(_e));       \
            (void)hipStreamSynchronize(s);                                      \
            return _e == hipErrorOutOfMemory ? ENOMEM_ : EDEVICE;               \
        }                                                                       \
    } while (0)

// The device combine, enqueued on `s`; the maxima return to the host at the
// end (a zero one is refused, and the passes after the first left `out` alone).
static int device_combine(const uint16_t *g, const uint16_t *e, int64_t nz, int64_t ny, int64_t nx,
                          const uint8_t *cyl, uint16_t *out, uint32_t *ws, hipStream_t s) {
    const int64_t plane = ny * nx;
    if (nz * plane == 0) return OK;
    const int64_t chunks = (plane + kThreads * kPerThread - 1) / (kThreads * kPerThread);
    if (nz * ny * ((nx + 1023) / 1024) > 0x7fffffffLL || chunks > 0x7fffffffLL) {
        set_error("volume too large for one launch of the row kernels");
        return EINVAL_;
    }
    // Planes per block: 16 for the reductions, which fold with atomics, and 4
    // for the output, unless that leaves CUs empty (a block's planes apart, many
    // blocks at once: 1024^3, 128 planes per block 0.83 / 0.91 / 1.38 ms, 16
    // and 4 0.72 / 0.78 / 1.13; one plane per block costs 24 M voxels 193 us
    // against 134 for 6)
    auto grid_of = [&](int64_t planes, int64_t blocks) {
        const int64_t y = std::max((nz + planes - 1) / planes, std::min(nz, (blocks + chunks - 1) / chunks));
        return dim3((unsigned)chunks, (unsigned)std::min<int64_t>(y, 65535));
    };
    const dim3 grid = grid_of(16, 2048), out_grid = grid_of(4, 8192);
    hipLaunchKernelGGL(k_fields_init, dim3(1), dim3(64), 0, s, ws);
    hipLaunchKernelGGL(k_max2, grid, dim3(kThreads), 0, s, g, e, nz, plane, ws);
    hipLaunchKernelGGL(k_combine_minmax, grid, dim3(kThreads), 0, s, g, e, cyl, nz, plane, ws);
    hipLaunchKernelGGL(k_combine_out, out_grid, dim3(kThreads), 0, s, g, e, cyl, nz, plane, ws, out);
    MXB_FHIP(hipGetLastError());
    uint32_t h[2];
    MXB_FHIP(hipMemcpyAsync(h, ws, 8, hipMemcpyDeviceToHost, s));
    MXB_FHIP(hipStreamSynchronize(s));
    if (h[0] == 0 || h[1] == 0) {
        set_error("combine_fields: a field's maximum is zero");
        return EINVAL_;
    }
    return OK;
}

static int device_field_histogram(const uint16_t *vox, int64_t nZ, int64_t nY, int64_t nX,
                                  const uint16_t *field, int64_t nz, int64_t ny, int64_t nx,
                                  uint64_t *bins, int64_t fb, int64_t vb, double vmin, double vmax,
                                  double fmin, double fmax, void *ws, hipStream_t s) {
    if (nZ * nY * nX == 0) return OK;
    if (nz < 1 || ny < 1 || nx < 1 || fb < 1 || vb < 1 || fb * vb >= (int64_t)0xffffffffLL) {
        set_error("field_histogram: invalid field shape or bin counts");
        return EINVAL_;
    }
    std::vector<int32_t> words;  // host tables: outlive their copy
    MXB_FHIP_AFTER_COPY(launch_field_histogram(vox, nZ, nY, nX, field, nz, ny, nx, bins, fb, vb, vmin, vmax, fmin, fmax,
                                               ws, words, s), s);
    MXB_FHIP(hipStreamSynchronize(s));
    return OK;
}

static int device_axis_histograms(const uint16_t *vox, int64_t nz, int64_t ny, int64_t nx,
                                  int64_t z_offset, uint64_t *xb, uint64_t *yb, uint64_t *zb,
                                  uint64_t *rb, int64_t Nz, int64_t Nr, int64_t vb, uint64_t cy,
                                  uint64_t cx, double vmin, double vmax, hipStream_t s) {
    if (nz * ny * nx == 0) return OK;
    if (vb < 1 || z_offset < 0 || Nz < 0 || Nr < 0) {
        set_error("axis_histograms: invalid arguments");
        return EINVAL_;
    }
    if (nz * ny * ((nx + 1023) / 1024) > 0x7fffffffLL) {
        set_error("volume too large for one launch of the row kernels");
        return EINVAL_;
    }
    if (vb > 8192) {
        set_error("axis_histograms: at most 8192 voxel bins");
        return EINVAL_;
    }
    MXB_FHIP(launch_axis_histograms(vox, nz, ny, nx, z_offset, xb, yb, zb, rb, Nz, Nr, vb, (int64_t)cy, (int64_t)cx,
                                    vmin, vmax, s));
    MXB_FHIP(hipStreamSynchronize(s));
    return OK;
}

// RAII device buffer for the host entries.
struct FBuf {
    void *p = nullptr;
    ~FBuf() {
        if (p) (void)hipFree(p);
    }
    int alloc(size_t n) {
        if (n == 0) n = 1;
        hipError_t e = hipMalloc(&p, n);
        if (e != hipSuccess) {
            set_error(std::string("hipMalloc: ") + hipGetErrorString(e));
            return e == hipErrorOutOfMemory ? ENOMEM_ : EDEVICE;
        }
        return OK;
    }
};

}  // namespace mxb

using namespace mxb;

extern "C" {

int64_t mxb_combine_workspace_bytes(void) { return 256; }

int mxb_device_combine_fields(const uint16_t *dev_gauss, const uint16_t *dev_edt, int64_t nz,
                              int64_t ny, int64_t nx, const uint8_t *dev_cylinder,
                              uint16_t *dev_out, void *dev_workspace, void *stream) {
    if (nz < 0 || ny < 0 || nx < 0 || (nz * ny * nx > 0 && (!dev_gauss || !dev_edt || !dev_out || !dev_workspace))) {
        set_error("combine_fields: invalid arguments");
        return EINVAL_;
    }
    return device_combine(dev_gauss, dev_edt, nz, ny, nx, dev_cylinder, dev_out, (uint32_t *)dev_workspace,
                          (hipStream_t)stream);
}

int mxb_combine_fields(const uint16_t *gauss, const uint16_t *edt, int64_t nz, int64_t ny,
                       int64_t nx, const uint8_t *cylinder, uint16_t *out, int verbose) {
    (void)verbose;
    if (nz < 0 || ny < 0 || nx < 0 || (nz * ny * nx > 0 && (!gauss || !edt || !out))) {
        set_error("combine_fields: invalid arguments");
        return EINVAL_;
    }
    const int64_t n = nz * ny * nx;
    if (n == 0) return OK;
    FBuf g, e, o, c, ws;
    int rc;
    if ((rc = g.alloc(n * 2)) || (rc = e.alloc(n * 2)) || (rc = o.alloc(n * 2)) || (rc = ws.alloc(256))) return rc;
    if (cylinder != nullptr && (rc = c.alloc(ny * nx))) return rc;
    hipStream_t s = nullptr;
    MXB_FHIP(staged_copy(g.p, gauss, n * 2, true, nullptr));
    MXB_FHIP(staged_copy(e.p, edt, n * 2, true, nullptr));
    if (cylinder != nullptr) MXB_FHIP(hipMemcpy(c.p, cylinder, ny * nx, hipMemcpyHostToDevice));
    rc = device_combine((const uint16_t *)g.p, (const uint16_t *)e.p, nz, ny, nx,
                        cylinder != nullptr ? (const uint8_t *)c.p : nullptr, (uint16_t *)o.p, (uint32_t *)ws.p, s);
    if (rc != OK) return rc;
    MXB_FHIP(staged_copy(out, o.p, n * 2, false, nullptr));
    return OK;
}

int64_t mxb_histogram_workspace_bytes(int64_t nZ, int64_t nY, int64_t nX) {
    if (nZ < 0 || nY < 0 || nX < 0) return -1;
    return field_workspace_bytes(nZ, nY, nX);
}

int mxb_device_field_histogram(const uint16_t *dev_voxels, int64_t nZ, int64_t nY, int64_t nX,
                               const uint16_t *dev_field, int64_t nz, int64_t ny, int64_t nx,
                               uint64_t *dev_bins, int64_t field_bins, int64_t voxel_bins,
                               double vmin, double vmax, double fmin, double fmax,
                               void *dev_workspace, void *stream) {
    if (nZ < 0 || nY < 0 || nX < 0 || (nZ * nY * nX > 0 && (!dev_voxels || !dev_field || !dev_bins || !dev_workspace))) {
        set_error("field_histogram: invalid arguments");
        return EINVAL_;
    }
    return device_field_histogram(dev_voxels, nZ, nY, nX, dev_field, nz, ny, nx, dev_bins, field_bins,
                                  voxel_bins, vmin, vmax, fmin, fmax, dev_workspace, (hipStream_t)stream);
}

int mxb_field_histogram(const uint16_t *voxels, int64_t nZ, int64_t nY, int64_t nX,
                        const uint16_t *field, int64_t nz, int64_t ny, int64_t nx, uint64_t *bins,
                        int64_t field_bins, int64_t voxel_bins, double vmin, double vmax,
                        double fmin, double fmax, int verbose) {
    (void)verbose;
    if (nZ < 0 || nY < 0 || nX < 0 || nz < 0 || ny < 0 || nx < 0 || field_bins < 1 || voxel_bins < 1 ||
        (nZ * nY * nX > 0 && (!voxels || !field || !bins))) {
        set_error("field_histogram: invalid arguments");
        return EINVAL_;
    }
    const int64_t n = nZ * nY * nX, nf = nz * ny * nx, nb = field_bins * voxel_bins;
    if (n == 0) return OK;
    FBuf v, f, b, ws;
    int rc;
    if ((rc = v.alloc(n * 2)) || (rc = f.alloc(nf * 2)) || (rc = b.alloc(nb * 8)) ||
        (rc = ws.alloc(field_workspace_bytes(nZ, nY, nX))))
        return rc;
    MXB_FHIP(staged_copy(v.p, voxels, n * 2, true, nullptr));
    MXB_FHIP(staged_copy(f.p, field, nf * 2, true, nullptr));
    MXB_FHIP(hipMemcpy(b.p, bins, nb * 8, hipMemcpyHostToDevice));
    rc = device_field_histogram((const uint16_t *)v.p, nZ, nY, nX, (const uint16_t *)f.p, nz, ny, nx,
                                (uint64_t *)b.p, field_bins, voxel_bins, vmin, vmax, fmin, fmax, ws.p, nullptr);
    if (rc != OK) return rc;
    MXB_FHIP(hipMemcpy(bins, b.p, nb * 8, hipMemcpyDeviceToHost));
    return OK;
}

int mxb_device_axis_histograms(const uint16_t *dev_voxels, int64_t nz, int64_t ny, int64_t nx,
                               int64_t z_offset, uint64_t *dev_x_bins, uint64_t *dev_y_bins,
                               uint64_t *dev_z_bins, uint64_t *dev_r_bins, int64_t Nz, int64_t Nr,
                               int64_t voxel_bins, uint64_t cy, uint64_t cx, double vmin,
                               double vmax, void *dev_workspace, void *stream) {
    if (nz < 0 || ny < 0 || nx < 0 ||
        (nz * ny * nx > 0 && (!dev_voxels || !dev_x_bins || !dev_y_bins || !dev_z_bins || !dev_r_bins || !dev_workspace))) {
        set_error("axis_histograms: invalid arguments");
        return EINVAL_;
    }
    return device_axis_histograms(dev_voxels, nz, ny, nx, z_offset, dev_x_bins, dev_y_bins, dev_z_bins,
                                  dev_r_bins, Nz, Nr, voxel_bins, cy, cx, vmin, vmax, (hipStream_t)stream);
}

int mxb_axis_histograms(const uint16_t *voxels, int64_t nz, int64_t ny, int64_t nx,
                        int64_t z_offset, uint64_t *x_bins, uint64_t *y_bins, uint64_t *z_bins,
                        uint64_t *r_bins, int64_t Nz, int64_t Nr, int64_t voxel_bins, uint64_t cy,
                        uint64_t cx, double vmin, double vmax, int verbose) {
    (void)verbose;
    if (nz < 0 || ny < 0 || nx < 0 || voxel_bins < 1 || Nz < 0 || Nr < 0 ||
        (nz * ny * nx > 0 && (!voxels || !x_bins || !y_bins || !z_bins || !r_bins))) {
        set_error("axis_histograms: invalid arguments");
        return EINVAL_;
    }
    const int64_t n = nz * ny * nx;
    if (n == 0) return OK;
    FBuf v, xb, yb, zb, rb;
    int rc;
    if ((rc = v.alloc(n * 2)) || (rc = xb.alloc(nx * voxel_bins * 8)) || (rc = yb.alloc(ny * voxel_bins * 8)) ||
        (rc = zb.alloc(Nz * voxel_bins * 8)) || (rc = rb.alloc(Nr * voxel_bins * 8)))
        return rc;
    MXB_FHIP(staged_copy(v.p, voxels, n * 2, true, nullptr));
    MXB_FHIP(hipMemcpy(xb.p, x_bins, nx * voxel_bins * 8, hipMemcpyHostToDevice));
    MXB_FHIP(hipMemcpy(yb.p, y_bins, ny * voxel_bins * 8, hipMemcpyHostToDevice));
    if (Nz > 0) MXB_FHIP(hipMemcpy(zb.p, z_bins, Nz * voxel_bins * 8, hipMemcpyHostToDevice));
    if (Nr > 0) MXB_FHIP(hipMemcpy(rb.p, r_bins, Nr * voxel_bins * 8, hipMemcpyHostToDevice));
    rc = device_axis_histograms((const uint16_t *)v.p, nz, ny, nx, z_offset, (uint64_t *)xb.p, (uint64_t *)yb.p,
                                (uint64_t *)zb.p, (uint64_t *)rb.p, Nz, Nr, voxel_bins, cy, cx, vmin, vmax,
                                nullptr);
    if (rc != OK) return rc;
    MXB_FHIP(hipMemcpy(x_bins, xb.p, nx * voxel_bins * 8, hipMemcpyDeviceToHost));
    MXB_FHIP(hipMemcpy(y_bins, yb.p, ny * voxel_bins * 8, hipMemcpyDeviceToHost));
    if (Nz > 0) MXB_FHIP(hipMemcpy(z_bins, zb.p, Nz * voxel_bins * 8, hipMemcpyDeviceToHost));
    if (Nr > 0) MXB_FHIP(hipMemcpy(r_bins, rb.p, Nr * voxel_bins * 8, hipMemcpyDeviceToHost));
    return OK;
}

}  // extern "C"
