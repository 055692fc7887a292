// 2D histograms of uint16 volumes (gfx950): the axis histograms of
// src/lib/cpp/cpu/histograms.cc:14-78.  C entries in mxb_fields.hip.
//
// Every voxel adds one count to each histogram, so the work is counting, not
// arithmetic.  A count that goes straight to the 64-bit bins in memory is a
// device-scope atomic (about 20-60 G/s over the whole chip), so each block
// takes voxels that share a few coordinates, counts them in LDS and adds one
// atomic per nonzero bin at the end.  Which voxels share a coordinate differs
// per axis, and one LDS table holds few of them, so the volume is read once
// per histogram (0.33 ms each at 1024^3) rather than once for all with
// frequent flushes.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "mxb_hist.h"
#include "mxb_internal.h"

namespace mxb {

// ------------------------------------------------------------- bins of a value
BinMap make_bin_map(double lo, double hi, int64_t nbins, bool mask_range) {
    BinMap m{};
    m.lo = lo;
    m.d = hi - lo;
    m.rd = 1.0 / m.d;
    m.c = static_cast<double>(nbins - 1);
    m.vlo = 1;
    m.vhi = 65535;
    if (mask_range) {  // values outside [lo, hi] become 0, and 0 is not counted
        if (!(lo <= 65535.0) || !(hi >= 1.0) || !(lo <= hi)) {
            m.vlo = 1;
            m.vhi = 0;
        } else {
            if (lo > 1.0) m.vlo = (uint32_t)std::ceil(lo);
            if (hi < 65535.0) m.vhi = (uint32_t)std::floor(hi);
        }
    }
    // the reciprocal form needs a finite normal divisor whose significand is
    // not all ones, and operands far from under- and overflow
    uint64_t bits;
    std::memcpy(&bits, &m.d, 8);
    const uint64_t frac = bits & 0xfffffffffffffull;
    m.fast = m.d > 0x1p-200 && m.d < 0x1p200 && frac != 0xfffffffffffffull && std::fabs(lo) < 0x1p60 ? 1 : 0;
    return m;
}

namespace {

constexpr int kLineThreads = 256;
constexpr int kTableThreads = 1024;
constexpr int64_t kTableBytes = 128 * 1024;  // LDS of a column or ring block's tables
static_assert(8 * 8192 * 2 <= kTableBytes, "eight 16-bit rows (a 16-byte load's columns) at the most bins");

// The volume as 16-byte chunks: `base` is the data pointer rounded down to 16
// bytes, element e of the volume sits at base[off + e], 0 <= off < 8.
struct Vol {
    const uint16_t *base;
    int64_t off, n;
};

static Vol vol_of(const uint16_t *p, int64_t n) {
    const uintptr_t a = reinterpret_cast<uintptr_t>(p);
    return Vol{reinterpret_cast<const uint16_t *>(a & ~uintptr_t(15)), (int64_t)((a & 15) / 2), n};
}

// ------------------------------------------------------------- y and z
// Output row o counts `rows` pieces of `len` consecutive voxels, piece i at
// element o * out_stride + i * row_stride.  z: one piece, a whole plane;
// y: one piece per plane, a row.  A block takes one part of one output row
// (parts split the pieces, or the chunks of a single piece).
struct LineSet {
    int64_t out_stride, rows, row_stride, len;
    int64_t parts, per;  // parts per output row; pieces (rows > 1) or chunks per part
    int64_t bin_row0;    // first row of the bins
    int tx;              // threads along a piece's chunks (a power of two)
};

// One vb-entry table per block (32 KB at most, so the wave slots fill), 16
// bytes per lane and load.  1024^3 with 4096 bins of noisy data: 0.57-0.6 ms
// each for y and z (3.7 TB/s); both counted along rows, with a flush of the y
// table after every row, took 10.7 ms.  Bound by the LDS atomics (a wave's 64
// counts take several passes over the banks) and the read together.
template <bool FAST>
__global__ __launch_bounds__(kLineThreads) void k_axis_lines(Vol v, LineSet s, BinMap m, int64_t vb,
                                                             unsigned long long *__restrict__ bins) {
    extern __shared__ uint32_t hist[];
    for (int64_t i = threadIdx.x; i < vb; i += kLineThreads) hist[i] = 0;
    __syncthreads();
    const int64_t o = blockIdx.x / s.parts, part = blockIdx.x % s.parts;
    const int tx = s.tx, ty = kLineThreads / tx;
    const int cx = threadIdx.x & (tx - 1), ry = threadIdx.x / tx;
    int64_t r0 = 0, r1 = 1, p0 = 0, p1 = INT64_MAX;
    if (s.rows > 1) {
        r0 = part * s.per;
        r1 = r0 + s.per < s.rows ? r0 + s.per : s.rows;
    } else {
        p0 = part * s.per;
        p1 = p0 + s.per;
    }
    for (int64_t r = r0 + ry; r < r1; r += ty) {
        const int64_t b = v.off + o * s.out_stride + r * s.row_stride, e = b + s.len;
        const int64_t first = b >> 3;
        const int64_t last = (e + 7) >> 3;
        const int64_t cend = p1 < last - first ? first + p1 : last;
        for (int64_t c = first + p0 + cx; c < cend; c += tx) {
            uint16_t q[8];
            load_chunk(v.base, c, b, e, q);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int bin = bin_of<FAST>(q[k], m);
                if (bin >= 0) atomicAdd(&hist[bin], 1u);
            }
        }
    }
    __syncthreads();
    for (int64_t i = threadIdx.x; i < vb; i += kLineThreads) {
        const uint32_t c = hist[i];
        if (c != 0) atomicAdd(&bins[(s.bin_row0 + o) * vb + i], (unsigned long long)c);
    }
}

// ------------------------------------------------------------- x and r
// Tables of a block: NT rows of vb counters, 16 bits each, two to a word
// (WIDE: 32 bits).  The host bounds what a block may add to one row to 65535
// where it uses 16 bits, so a counter never carries into its neighbour.
template <bool WIDE>
__device__ __forceinline__ void count_in(uint32_t *t, uint32_t idx) {
    if constexpr (WIDE) atomicAdd(&t[idx], 1u);
    else atomicAdd(&t[idx >> 1], 1u << (16 * (idx & 1)));
}

// Adds the tables' rows to the bins (rows from row_end on do not exist).  The
// lanes take consecutive counters: their atomics then share cache lines (8
// counters per lane instead, skipping zero words, made the flush 2-3 times
// slower).
template <bool WIDE>
__device__ __forceinline__ void flush_tables(const uint32_t *t, int64_t nt, int64_t vb, int64_t row0, int64_t row_end,
                                             unsigned long long *__restrict__ bins) {
    const int live = (int)((nt < row_end - row0 ? nt : row_end - row0) * vb);
    unsigned long long *const dst = bins + row0 * vb;
    for (int i0 = threadIdx.x; i0 < live; i0 += 4 * kTableThreads) {
        uint32_t c[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int i = i0 + k * kTableThreads;
            c[k] = i >= live ? 0 : (WIDE ? t[i] : (t[i >> 1] >> (16 * (i & 1))) & 0xffffu);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (c[k] != 0) atomicAdd(&dst[i0 + k * kTableThreads], (unsigned long long)c[k]);
    }
}

// Clears `bytes` of tables, whole 16-byte pieces.
__device__ __forceinline__ void clear_tables(uint32_t *t, int bytes) {
    for (int i = threadIdx.x; i < bytes / 16; i += kTableThreads) reinterpret_cast<uint4 *>(t)[i] = make_uint4(0, 0, 0, 0);
    __syncthreads();
}

// LDS bytes of nt rows of vb counters.
__host__ __device__ inline int table_bytes(int64_t nt, int64_t vb, bool wide) {
    return (int)((nt * vb * (wide ? 4 : 2) + 15) / 16 * 16);
}

struct ColSet {
    int64_t nx, q;            // columns; rows (z, y) counted
    int64_t per;              // rows per block
    int64_t groups, chunks;   // groups of NT columns, row chunks
    int nt, lt;               // columns per block, a power of two, and its log2
    int sib;                  // blocks that share 64 columns, which one L2 serves together
};

// x: a block takes NT columns and `per` rows.  The blocks of one 64-column
// group read the same 128-byte lines, so they go to one XCD next to each
// other (block b runs on XCD b % 8).  VEC: 16-byte loads of 8 columns
// (aligned rows), else one voxel per lane, 2 NT contiguous bytes per row.
// 1024^3, 4096 bins: 0.87 ms (2.5 TB/s).
template <bool FAST, bool WIDE, bool VEC>
__global__ __launch_bounds__(kTableThreads) void k_axis_cols(const uint16_t *__restrict__ vox, ColSet s, BinMap m,
                                                             int64_t vb, unsigned long long *__restrict__ bins) {
    extern __shared__ __attribute__((aligned(16))) uint32_t tab[];
    const int64_t k = blockIdx.x / 8, xcd = blockIdx.x % 8;
    const int64_t wide_groups = (s.groups + s.sib - 1) / s.sib;
    const int64_t rest = (k / s.sib) * 8 + xcd;
    const int64_t grp = (rest % wide_groups) * s.sib + k % s.sib, chunk = rest / wide_groups;
    if (grp >= s.groups || chunk >= s.chunks) return;
    clear_tables(tab, table_bytes(s.nt, vb, WIDE));
    const int64_t x0 = grp * s.nt;
    const int64_t q0 = chunk * s.per, q1 = q0 + s.per < s.q ? q0 + s.per : s.q;
    if constexpr (VEC) {
        const int lc = s.lt - 3;  // log2 of chunks per row
        const int col = (threadIdx.x & ((1 << lc) - 1)) * 8;
        const int64_t step = kTableThreads >> lc;
        if (x0 + col < s.nx) {  // rows are whole 8-voxel chunks
            const uint16_t *p = vox + x0 + col;
            int64_t q = q0 + (threadIdx.x >> lc);
            auto add = [&](const uint4 &w4) {
                const uint32_t w[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int bin = bin_of<FAST>((w[j >> 1] >> (16 * (j & 1))) & 0xffffu, m);
                    if (bin >= 0) count_in<WIDE>(tab, (uint32_t)((col + j) * vb + bin));
                }
            };
            for (; q + 3 * step < q1; q += 4 * step) {
                uint4 w[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) w[u] = *reinterpret_cast<const uint4 *>(p + (q + u * step) * s.nx);
#pragma unroll
                for (int u = 0; u < 4; ++u) add(w[u]);
            }
            for (; q < q1; q += step) add(*reinterpret_cast<const uint4 *>(p + q * s.nx));
        }
    } else {
        const int col = threadIdx.x & (s.nt - 1);
        const int64_t step = kTableThreads >> s.lt;
        if (x0 + col < s.nx) {
            const uint16_t *p = vox + x0 + col;
            for (int64_t q = q0 + (threadIdx.x >> s.lt); q < q1; q += 8 * step) {
                uint16_t w[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) w[u] = q + u * step < q1 ? p[(q + u * step) * s.nx] : (uint16_t)0;
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int bin = bin_of<FAST>(w[u], m);  // 0 has no bin
                    if (bin >= 0) count_in<WIDE>(tab, (uint32_t)(col * vb + bin));
                }
            }
        }
    }
    __syncthreads();
    flush_tables<WIDE>(tab, s.nt, vb, x0, s.nx, bins);
}

__device__ __forceinline__ int64_t isqrt64(int64_t s) {
    int64_t r = (int64_t)sqrt((double)s);
    while (r * r > s) --r;
    while ((r + 1) * (r + 1) <= s) ++r;
    return r;
}

struct RingSet {
    int64_t ny, nx, nz;          // nz: layers counted
    int64_t cy, cx, Nr;
    int64_t a0, na, zc;          // first annulus, annuli, layers per block
    int nt;                      // radii per annulus
};

constexpr int kU = 4;  // layers whose loads a lane issues together (1024^3: 4 3.85, 8 4.13, 16 4.05 ms for the whole call)
// r: a block takes an annulus of nt radii and zc layers.  The annulus is a
// set of runs, at most two per image row; their lengths are scanned for up to
// kTableThreads rows at a time, and the threads take its pixels in order (a
// binary search finds a pixel's row), each pixel through all layers of the
// block.  A pixel's radius is so worked out once per block, no lane idles on
// short runs, and the layers' loads are independent.  1024^3, 4096 bins: 1.9
// ms; with x, one global atomic per voxel and lanes grouped by equal bins, it
// took 36.5 ms.
template <bool FAST, bool WIDE>
__global__ __launch_bounds__(kTableThreads) void k_axis_rings(const uint16_t *__restrict__ vox, RingSet s, BinMap m,
                                                              int64_t vb, unsigned long long *__restrict__ bins) {
    extern __shared__ __attribute__((aligned(16))) uint32_t tab[];
    __shared__ int32_t offs[kTableThreads + 1];   // pixels of the batch before a row
    __shared__ int32_t lbeg[kTableThreads], llen[kTableThreads], rbeg[kTableThreads];
    __shared__ int32_t wsum[kTableThreads / 64];
    const int64_t a = blockIdx.x % s.na + s.a0, z0 = (blockIdx.x / s.na) * s.zc;
    const int nzb = (int)(s.zc < s.nz - z0 ? s.zc : s.nz - z0);
    const int64_t r0 = a * s.nt, r1 = r0 + s.nt < s.Nr ? r0 + s.nt : s.Nr;
    clear_tables(tab, table_bytes(s.nt, vb, WIDE));
    const int64_t plane = s.ny * s.nx;
    const uint16_t *const base = vox + z0 * plane;
    const int64_t ylo = s.cy - r1 + 1 > 0 ? s.cy - r1 + 1 : 0, yhi = s.cy + r1 < s.ny ? s.cy + r1 : s.ny;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    for (int64_t yb = ylo; yb < yhi; yb += kTableThreads) {
        // the runs of row yb + tid: [lbeg, lbeg + llen) and, after the inner
        // circle, rbeg on
        const int64_t y = yb + tid;
        int lb = 0, ll = 0, rb = 0, rl = 0;
        if (y < yhi) {
            const int64_t dy2 = (y - s.cy) * (y - s.cy), room = r1 * r1 - 1 - dy2;
            if (room >= 0) {
                const int64_t wo = isqrt64(room), in = r0 * r0 - 1 - dy2;
                auto clip = [&](int64_t x) { return (int)(x < 0 ? 0 : (x > s.nx ? s.nx : x)); };
                if (in < 0) {  // the inner circle does not reach this row: one run
                    lb = clip(s.cx - wo);
                    ll = clip(s.cx + wo + 1) - lb;
                } else {
                    const int64_t wi = isqrt64(in);
                    lb = clip(s.cx - wo);
                    ll = clip(s.cx - wi) - lb;
                    rb = clip(s.cx + wi + 1);
                    rl = clip(s.cx + wo + 1) - rb;
                }
            }
        }
        int incl = ll + rl;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int u = __shfl_up(incl, d, 64);
            if (lane >= d) incl += u;
        }
        if (lane == 63) wsum[wv] = incl;
        __syncthreads();
        int before = 0;
        for (int w = 0; w < wv; ++w) before += wsum[w];
        offs[tid + 1] = before + incl;
        if (tid == 0) offs[0] = 0;
        lbeg[tid] = lb;
        llen[tid] = ll;
        rbeg[tid] = rb;
        __syncthreads();
        const int total = offs[kTableThreads];
        for (int p = tid; p < total; p += kTableThreads) {
            int lo = 0, hi = kTableThreads;  // the last row that starts at or before p
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (offs[mid] <= p) lo = mid;
                else hi = mid;
            }
            const int i = p - offs[lo];
            const int64_t x = i < llen[lo] ? lbeg[lo] + i : rbeg[lo] + (i - llen[lo]);
            const int64_t yy = yb + lo, dy = yy - s.cy, dx = x - s.cx;
            const uint32_t row = (uint32_t)(isqrt64(dy * dy + dx * dx) - r0) * (uint32_t)vb;
            const uint16_t *const px = base + yy * s.nx + x;
            for (int z = 0; z < nzb; z += kU) {
                uint16_t w[kU];
#pragma unroll
                for (int u = 0; u < kU; ++u) w[u] = z + u < nzb ? px[(z + u) * plane] : (uint16_t)0;
#pragma unroll
                for (int u = 0; u < kU; ++u) {
                    const int bin = bin_of<FAST>(w[u], m);  // 0 has no bin
                    if (bin >= 0) count_in<WIDE>(tab, row + (uint32_t)bin);
                }
            }
        }
        __syncthreads();
    }
    __syncthreads();
    flush_tables<WIDE>(tab, s.nt, vb, r0, r1, bins);
}

template <typename F>
hipError_t allow_lds(F *fn, size_t bytes) {
    if (bytes <= 64 * 1024) return hipSuccess;
    return hipFuncSetAttribute(reinterpret_cast<const void *>(fn), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)bytes);
}

hipError_t launch_lines(const Vol &v, LineSet s, int64_t outs, int64_t want, const BinMap &m, int64_t vb, uint64_t *bins,
                        hipStream_t st) {
    if (outs <= 0) return hipSuccess;
    const int64_t cpr = (s.len + 14) / 8;  // chunks a piece may touch
    // enough parts to fill the device, each of at least 16 table clears' work
    const int64_t work = s.rows * cpr;
    int64_t parts = std::max<int64_t>(1, (2 * want + outs - 1) / outs);
    parts = std::min(parts, std::max<int64_t>(1, work * 8 / std::max<int64_t>(4 * vb, 4096)));
    if (s.rows > 1) {
        parts = std::min(parts, s.rows);
        s.per = (s.rows + parts - 1) / parts;
        s.parts = (s.rows + s.per - 1) / s.per;
    } else {
        s.per = (cpr + parts - 1) / parts;
        s.parts = (cpr + s.per - 1) / s.per;
    }
    // threads along a piece: the power of two that leaves the fewest idle
    s.tx = kLineThreads;
    if (s.rows > 1)
        for (int t = kLineThreads / 2; t >= 8; t >>= 1)
            if ((cpr + t - 1) / t * t < (cpr + s.tx - 1) / s.tx * s.tx) s.tx = t;
    const size_t smem = (size_t)vb * 4;
    const unsigned grid = (unsigned)(outs * s.parts);
    if (m.fast) hipLaunchKernelGGL(k_axis_lines<true>, dim3(grid), dim3(kLineThreads), smem, st, v, s, m, vb, (unsigned long long *)bins);
    else hipLaunchKernelGGL(k_axis_lines<false>, dim3(grid), dim3(kLineThreads), smem, st, v, s, m, vb, (unsigned long long *)bins);
    return hipGetLastError();
}

// Rows of counters that a block's LDS holds: a power of two, at most 16.
// More rows mean fewer column groups or annuli, so more blocks along the
// other axes and a flush by each of them (512^3 with 1024 bins: 64 rows 685
// us, 16 rows 537, 8 rows 543; 1024^3 with 4096 bins: 16 rows 4.27 ms, 8 rows,
// which read 16 bytes of a cache line at a time, 4.83).
int table_rows(int64_t vb, int64_t counter_bytes) {
    int nt = 16;
    while (nt > 1 && nt * vb * counter_bytes > kTableBytes) nt >>= 1;
    return nt;
}

template <bool FAST, bool VEC>
hipError_t launch_cols(const uint16_t *vox, ColSet s, const BinMap &m, int64_t vb, uint64_t *bins, hipStream_t st) {
    const size_t smem = table_bytes(s.nt, vb, false);
    const int64_t wide_groups = (s.groups + s.sib - 1) / s.sib;
    const int64_t blocks = (wide_groups * s.chunks + 7) / 8 * 8 * s.sib;
    auto *fn = &k_axis_cols<FAST, false, VEC>;
    if (hipError_t e = allow_lds(fn, smem)) return e;
    hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3(kTableThreads), smem, st, vox, s, m, vb,
                       (unsigned long long *)bins);
    return hipGetLastError();
}

template <bool FAST, bool WIDE>
hipError_t launch_rings(const uint16_t *vox, const RingSet &s, const BinMap &m, int64_t vb, uint64_t *bins,
                        hipStream_t st) {
    const size_t smem = table_bytes(s.nt, vb, WIDE);
    const int64_t blocks = s.na * ((s.nz + s.zc - 1) / s.zc);
    auto *fn = &k_axis_rings<FAST, WIDE>;
    if (hipError_t e = allow_lds(fn, smem)) return e;
    hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3(kTableThreads), smem, st, vox, s, m, vb,
                       (unsigned long long *)bins);
    return hipGetLastError();
}

}  // namespace

// vb <= 8192, every extent at least 1, nz * ny within the launch limits.
hipError_t launch_axis_histograms(const uint16_t *vox, int64_t nz, int64_t ny, int64_t nx, int64_t z_offset,
                                  uint64_t *xb, uint64_t *yb, uint64_t *zb, uint64_t *rb, int64_t Nz, int64_t Nr,
                                  int64_t vb, int64_t cy, int64_t cx, double vmin, double vmax, hipStream_t st) {
    const int64_t nzc = std::min(nz, Nz - z_offset);  // layers at or beyond Nz are skipped
    if (nzc <= 0) return hipSuccess;
    const BinMap m = make_bin_map(vmin, vmax, vb, true);
    if (m.vlo > m.vhi) return hipSuccess;  // no value is counted
    const Vol v = vol_of(vox, nz * ny * nx);
    // Blocks per launch: every block flushes its tables, so small volumes take
    // one per CU of a 256-CU device (200^3, 256 bins: 256 blocks 109 us, 1024
    // 150) and large ones more, for the tail (1024^3: 2048 blocks 3 % faster
    // than 1024).
    const int64_t want = std::min<int64_t>(2048, std::max<int64_t>(256, (nzc * ny * nx) >> 17));
    hipError_t e;
    LineSet z{ny * nx, 1, 0, ny * nx, 1, 1, z_offset, 0};
    if ((e = launch_lines(v, z, nzc, want, m, vb, zb, st)) != hipSuccess) return e;
    LineSet y{nx, nzc, ny * nx, nx, 1, 1, 0, 0};
    if ((e = launch_lines(v, y, ny, want, m, vb, yb, st)) != hipSuccess) return e;

    // x: a 16-bit counter sees each row of a block once
    const bool vec = nx % 8 == 0 && reinterpret_cast<uintptr_t>(vox) % 16 == 0;
    ColSet c{};
    c.nx = nx;
    c.q = nzc * ny;
    c.nt = table_rows(vb, 2);
    while (c.nt > 8 && c.nt / 2 >= nx) c.nt >>= 1;
    c.lt = 0;
    while ((1 << c.lt) < c.nt) ++c.lt;
    c.groups = (nx + c.nt - 1) / c.nt;
    c.sib = std::max(1, 64 / c.nt);
    c.chunks = std::max<int64_t>((c.q + 65534) / 65535, std::min((want + c.groups - 1) / c.groups, (c.q + 511) / 512));
    c.per = (c.q + c.chunks - 1) / c.chunks;
    c.chunks = (c.q + c.per - 1) / c.per;
    if (m.fast) e = vec ? launch_cols<true, true>(vox, c, m, vb, xb, st) : launch_cols<true, false>(vox, c, m, vb, xb, st);
    else e = vec ? launch_cols<false, true>(vox, c, m, vb, xb, st) : launch_cols<false, false>(vox, c, m, vb, xb, st);
    if (e != hipSuccess || Nr <= 0) return e;

    // r: a centre this far out has no radius within any table
    constexpr int64_t kFar = int64_t(1) << 30;
    if (cy < -kFar || cy > kFar || cx < -kFar || cx > kFar) return hipSuccess;
    auto span = [](int64_t c0, int64_t n, int64_t &lo, int64_t &hi) {  // distances of [0, n) from c0
        lo = c0 < 0 ? -c0 : (c0 >= n ? c0 - (n - 1) : 0);
        hi = std::max(std::abs(c0), std::abs(n - 1 - c0));
    };
    int64_t ylo, yhi, xlo, xhi;
    span(cy, ny, ylo, yhi);
    span(cx, nx, xlo, xhi);
    const int64_t rmin = (int64_t)std::sqrt((double)(ylo * ylo + xlo * xlo));
    const int64_t rmax = (int64_t)std::sqrt((double)(yhi * yhi + xhi * xhi)) + 1;
    RingSet r{};
    r.ny = ny; r.nx = nx; r.nz = nzc; r.cy = cy; r.cx = cx; r.Nr = Nr;
    // a ring of radius rho holds at most 7 (rho + 1) pixels (2 pi rho and a
    // lattice remainder, 8 at rho = 1), each counted once per layer; beyond 16-bit counts even for one layer, 32-bit counters
    const int64_t rtop = std::min(Nr, rmax + 1), ring = 7 * (rtop + 1);
    const bool wide = ring > 65535;
    r.nt = table_rows(vb, wide ? 4 : 2);
    while (r.nt > 8 && r.nt / 2 >= rtop) r.nt >>= 1;
    r.a0 = std::max<int64_t>(0, rmin - 1) / r.nt;
    r.na = (rtop + r.nt - 1) / r.nt - r.a0;
    if (r.na <= 0) return hipSuccess;
    r.zc = wide ? (int64_t(1) << 32) / ring : 65535 / ring;
    r.zc = std::max<int64_t>(1, std::min(r.zc, (nzc * r.na + want - 1) / want));
    if (r.zc > kU) r.zc -= r.zc % kU;
    if (m.fast) return wide ? launch_rings<true, true>(vox, r, m, vb, rb, st) : launch_rings<true, false>(vox, r, m, vb, rb, st);
    return wide ? launch_rings<false, true>(vox, r, m, vb, rb, st) : launch_rings<false, false>(vox, r, m, vb, rb, st);
}

}  // namespace mxb
