// 2D histograms of uint16 volumes (gfx950): the axis histograms of
// src/lib/cpp/cpu/histograms.cc:14-78 and the field histogram of :231-306.
// C entries in mxb_fields.hip.
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
#include <type_traits>

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
// table after every row, took 10.7 ms.  Bound by its vector instructions (the
// float64 bin of each voxel): they fill 87 % of the SIMDs' cycles, the LDS 38 %
// of its own.
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
                const uint32_t bin = bin_of<FAST>(q[k], m);
                if (bin != kNoBin) atomicAdd(&hist[bin], 1u);
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
// 1024^3, 4096 bins: 0.87 ms (2.5 TB/s), 69 % of the SIMDs' cycles in vector
// instructions.
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
                    const uint32_t bin = bin_of<FAST>((w[j >> 1] >> (16 * (j & 1))) & 0xffffu, m);
                    if (bin != kNoBin) count_in<WIDE>(tab, (uint32_t)((col + j) * vb + bin));
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
                    const uint32_t bin = bin_of<FAST>(w[u], m);  // 0 has no bin
                    if (bin != kNoBin) count_in<WIDE>(tab, (uint32_t)(col * vb + bin));
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
// took 36.5 ms.  Three times k_axis_lines, with as many LDS atomics: a lane
// loads 2 bytes (eight times the loads) and each count takes 2.4 times the
// vector instructions (58 % of the SIMDs' cycles), while a wave waits 62 % of
// its time.  Where an annulus has fewer pixels than half the threads,
// lanes share a pixel's layers (4096x1x4096, 4096 bins, the whole call: 567 ->
// 211 us).
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
        auto count = [&](int p, int z0, auto step) {  // pixel p's layers z0 .. z0 + kU - 1, then `step` further
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
            for (int z = z0; z < nzb; z += step) {
                uint16_t w[kU];
#pragma unroll
                for (int u = 0; u < kU; ++u) w[u] = z + u < nzb ? px[(z + u) * plane] : (uint16_t)0;
#pragma unroll
                for (int u = 0; u < kU; ++u) {
                    const uint32_t bin = bin_of<FAST>(w[u], m);  // 0 has no bin
                    if (bin != kNoBin) count_in<WIDE>(tab, row + (uint32_t)bin);
                }
            }
        };
        // few pixels (thin slabs): several lanes share one's layers
        if (total > 0 && 2 * total <= kTableThreads) {
            const int share = kTableThreads / total, part = tid / total;
            if (part < share) count(tid % total, part * kU, share * kU);
        } else {
            for (int p = tid; p < total; p += kTableThreads) count(p, 0, std::integral_constant<int, kU>{});
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
    // lattice remainder, 8 at rho = 1), and in one row or column at most 2
    // ceil(sqrt(2 rho + 1)) (the widest chord of a ring 1 wide, on either side),
    // each counted once per layer; beyond 16-bit counts even for one layer,
    // 32-bit counters.  Without the second bound thin slabs got few layers per
    // block, and a table to clear and flush for each (4096x1x4096, 4096 bins: 5.0
    // ms, 0.57 with it).
    const int64_t rtop = std::min(Nr, rmax + 1), chord = 2 * ((int64_t)std::sqrt(2.0 * (double)rtop + 1.0) + 1);
    const int64_t ring = std::min({7 * (rtop + 1), ny * std::min(nx, chord), nx * std::min(ny, chord)});
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

// ------------------------------------------------------------- field histogram
// Voxels against a field sampled at floor(Z nz / nZ) etc.
// (cpu/histograms.cc:231-306): one count per voxel into bins[fb][vb], a table
// far larger than LDS (64 MB at 2048 x 4096).  Noisy voxels over a smooth
// field give nearly as many (field bin, voxel bin) pairs as voxels in any
// compact piece of the volume, so gathering pieces in LDS saves little
// (an LDS hash table per brick: 52 ms at 1024^3, nearly all of it global
// atomics).  The field is what is smooth: the voxels of a few neighbouring
// field bins lie in a shell, and their counts fit in LDS.  So:
//   k_field_ranges: per brick of field values, the least and greatest nonzero
//                   value;
//   k_field_plan:   per group of G field bins (an interval of field values,
//                   as bins are monotone in the value), how many bricks meet
//                   it, and how many blocks serve it;
//   k_field_groups: a block takes a group and a share of its bricks.  Its
//                   waves test the bricks' field values, queue the matches,
//                   and count the queued values' voxels in the block's
//                   G x vb table, which reaches the bins once.
// 1024^3 voxels, 512^3 field, 2048 x 4096 bins, calls back to back: 52.5 ->
// 4.8 ms (k_field_groups 4.5); with a 1024^3 field 53.5 -> 15.5 (tests of field values against about ten groups each);
// 240^3 with a 60^3 field 0.71 -> 0.15.  Extents that do not divide (boxes of
// two or three voxels a side): 301x257x263 and half, smooth field 0.43, noise 1.10
// (the hash form 1.37); with a place of the widest box per lane, and bricks
// weighed by it, 0.87 and 2.65.  Bound by vector
// instructions (64 % of a busy SIMD's cycles: tests, bins, the queue), beside
// scattered reads (a wave waits 47 % of its time) that only 16 waves per CU,
// which the table allows, can hide.
// A field that is not smooth (noise) makes every brick meet every group; then,
// and for tables or axes beyond the limits below, k_field_hash counts.
namespace {

constexpr int kGroupThreads = 1024, kGroupWaves = kGroupThreads / 64;
constexpr int kQueue = 368;              // field values queued per wave
constexpr int kList = kGroupThreads * 3 / 2; // bricks a block lists at a time
constexpr int kGroupBlocks = 1024;       // blocks wanted at most (one fits a CU at a time; 256 leave a long tail)
constexpr int64_t kBlockVoxels = 2048;   // and one per so many voxels: each clears and flushes its table

struct FieldGeom {
    int64_t n[3], nf[3];   // voxel and field extents (z, y, x)
    int32_t nb[3], lb[3];  // bricks, log2 of brick edges (x at least 16)
    int32_t width[3];      // widest segment
    int32_t lbox;          // every segment is as wide and a box holds 2^lbox <= 64 voxels; else -1
    int32_t bricks, ng, G;
    int32_t blocks_wanted;
    int32_t pairs;         // layer pairs per unit of work: 4, or 1 where a value stands for many voxels
    int64_t fb, vb;
    uint32_t box, mean;              // voxels per value, at most and on average
    uint32_t m_y, m_xy, m_x;         // magic reciprocals of widths
    const int32_t *starts[3];        // first voxel coordinate of every segment, and the extent
    uint32_t *ranges;                // per brick: least << 16 | greatest nonzero value
    uint32_t *start;                 // per group: first block; [ng]: blocks, [ng + 1]: brick visits, weighed
    const uint32_t *bound;           // per group: least field value, [ng]: end
    uint32_t visits_max;             // beyond, the hash form counts
    uint32_t few_weight;             // of a visit, in 16ths, where voxels have one value or two
};

// i / d for i < 2^20, d <= 512 by m = ceil(2^32 / d); d = 1: m = 0
__device__ __forceinline__ uint32_t div_magic(uint32_t i, uint32_t m) { return m == 0 ? i : __umulhi(i, m); }

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ void brick_origin(const FieldGeom &g, uint32_t brick, int o[3]) {
    const uint32_t bx = brick % (uint32_t)g.nb[2], r = brick / (uint32_t)g.nb[2];
    o[2] = (int)(bx << g.lb[2]);
    o[1] = (int)((r % (uint32_t)g.nb[1]) << g.lb[1]);
    o[0] = (int)((r / (uint32_t)g.nb[1]) << g.lb[0]);
}

// One wave per brick; lanes 16 x by 4 y.  Reads the field once.
__global__ __launch_bounds__(256) void k_field_ranges(const uint16_t *__restrict__ field, FieldGeom g) {
    const int lane = threadIdx.x & 63;
    const uint32_t brick = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (brick >= (uint32_t)g.bricks) return;
    int o[3];
    brick_origin(g, brick, o);
    uint32_t lo = 65535, hi = 0;
    const int lx = lane & 15, ly = lane >> 4;
    for (int z = 0; z < 1 << g.lb[0] && o[0] + z < g.nf[0]; ++z)
        for (int y = ly; y < 1 << g.lb[1] && o[1] + y < g.nf[1]; y += 4)
            for (int x = lx; x < 1 << g.lb[2] && o[2] + x < g.nf[2]; x += 16) {
                const uint32_t f = field[((o[0] + z) * g.nf[1] + o[1] + y) * g.nf[2] + o[2] + x];
                if (f != 0) {
                    lo = min(lo, f);
                    hi = max(hi, f);
                }
            }
    for (int d = 32; d > 0; d >>= 1) {
        lo = min(lo, (uint32_t)__shfl_xor((int)lo, d));
        hi = max(hi, (uint32_t)__shfl_xor((int)hi, d));
    }
    if (lane == 0) g.ranges[brick] = lo << 16 | hi;
}

// Blocks per group, in proportion to its work; one block.
//
// It also weighs the visits against the hash form (visits_max).  Voxels of very
// few values (a mask, a constant) stay as few pairs in a hash block's table: 11
// ps a voxel for one value, 14 for two, 20 for four to sixteen, instead of 50, so
// there a visit weighs more.  A sample of voxels tells how many values there
// are; kFewPairs bounds the pairs with the field bins that a brick meets, beyond
// which the table (8192 slots) overflows.  One value over noise, field of half
// the extents: 512^3 4.70 -> 1.24 ms, 1024^3 37.9 -> 9.1; over a smooth field as
// fine as the voxels, 1024^3 18.3 -> 11.2.  Four values there are faster grouped
// (15.6 against 17.9), hence the lesser weight from three on.
constexpr int64_t kFewPairs = 8192;
__global__ __launch_bounds__(kGroupThreads) void k_field_plan(const uint16_t *__restrict__ vox, FieldGeom g, BinMap vm) {
    __shared__ uint32_t bound[kMaxGroups + 1];
    __shared__ uint32_t seen[kGroupCells / 32];
    __shared__ int32_t diff[kMaxGroups + 1];
    __shared__ int32_t wsum[kGroupWaves];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    for (int i = tid; i <= g.ng; i += kGroupThreads) {
        bound[i] = g.bound[i];
        diff[i] = 0;
    }
    for (int i = tid; i < kGroupCells / 32; i += kGroupThreads) seen[i] = 0;
    __syncthreads();
    uint32_t sample = 0;
    if (g.few_weight > 16)
        sample = vox[__umul64hi((uint64_t)(tid + 1) * 0x9e3779b97f4a7c15u, (uint64_t)(g.n[0] * g.n[1] * g.n[2]))];
    auto last_at = [&](uint32_t f) {  // the last group that starts at or before f, or -1
        int lo = -1, hi = g.ng;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (bound[mid] <= f) lo = mid;
            else hi = mid;
        }
        return lo;
    };
    int met = 0;  // brick visits
    for (int i = tid; i < g.bricks; i += kGroupThreads) {
        const uint32_t r = g.ranges[i], lo = r >> 16, hi = r & 0xffffu;
        if (lo > hi || lo >= bound[g.ng] || hi < bound[0]) continue;
        int a = last_at(lo), b = last_at(hi);
        a = a < 0 ? 0 : a;
        // a visit tests all of the brick's values and counts its share of their voxels
        const int cost = 4 + 12 * (int)g.mean / (b - a + 1);
        atomicAdd(&diff[a], cost);
        atomicAdd(&diff[b + 1], -cost);
        met += b - a + 1;
    }
    if (g.few_weight > 16) {
        const uint32_t b = bin_of<true>(sample, vm);
        if (b != kNoBin) atomicOr(&seen[b >> 5], 1u << (b & 31));
    }
    __syncthreads();
    // two groups per thread: inclusive scans of diff (work per group), then of
    // the blocks per group; `before` is what lies before the thread's two
    auto scan = [&](int a, int b, int &before, int &total) {
        int incl = a + b;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int u = __shfl_up(incl, d, 64);
            if (lane >= d) incl += u;
        }
        if (lane == 63) wsum[wv] = incl;
        __syncthreads();
        before = incl - a - b;
        total = 0;
        for (int w = 0; w < kGroupWaves; ++w) {
            if (w < wv) before += wsum[w];
            total += wsum[w];
        }
        __syncthreads();
    };
    const int i0 = 2 * tid, i1 = i0 + 1;
    const int d0 = i0 < g.ng ? diff[i0] : 0, d1 = i1 < g.ng ? diff[i1] : 0;
    int before, total, visits, work;
    scan(met, 0, before, visits);
    scan(d0, d1, before, total);
    const int v0 = i0 < g.ng ? before + d0 : 0, v1 = i1 < g.ng ? before + d0 + d1 : 0;
    scan(v0, v1, before, work);
    const int64_t want = min(g.blocks_wanted, max(visits, 1));
    auto blocks = [&](int v) { return v == 0 ? 0 : (int)((v * want + work - 1) / work); };
    const int p0 = blocks(v0), p1 = blocks(v1);
    scan(p0, p1, before, total);
    int values = 0, unused;
    if (g.few_weight > 16) scan(__popc(seen[tid]), 0, unused, values);
    if (i0 < g.ng) g.start[i0] = (uint32_t)before;
    if (i1 < g.ng) g.start[i1] = (uint32_t)(before + p0);
    if (tid == 0) {
        g.start[g.ng] = (uint32_t)total;
        const bool few = g.few_weight > 16 && (int64_t)values * g.G * visits <= kFewPairs * g.bricks;
        const uint32_t w = values <= 2 ? g.few_weight : max(16u, g.few_weight * 6 / 16);
        g.start[g.ng + 1] = few ? (uint32_t)min((uint64_t)visits * w >> 4, (uint64_t)0xffffffffu) : (uint32_t)visits;
    }
}

// LDS: the table, the waves' queues and segment starts, the brick list.
constexpr int kUnitStarts = 17 + 9 + 9;  // x, y, z starts of a unit
constexpr int kGroupLds = kGroupCells * 4 + (kGroupWaves * (kQueue + kUnitStarts) + kList) * 4;
static_assert(kGroupLds <= 160 * 1024 - 256, "one block per CU");

__global__ __launch_bounds__(kGroupThreads) void k_field_groups(const uint16_t *__restrict__ vox,
                                                                const uint16_t *__restrict__ field, FieldGeom g,
                                                                BinMap vm, BinMap fm,
                                                                unsigned long long *__restrict__ bins) {
    extern __shared__ __attribute__((aligned(16))) uint32_t tab[];
    uint32_t *const queue = tab + kGroupCells + (threadIdx.x >> 6) * kQueue;
    int32_t *const starts = reinterpret_cast<int32_t *>(tab + kGroupCells + kGroupWaves * kQueue) + (threadIdx.x >> 6) * kUnitStarts;
    uint32_t *const list = tab + kGroupCells + kGroupWaves * (kQueue + kUnitStarts);
    __shared__ int32_t s_grp, s_part, s_parts, s_count, s_next;
    const int tid = threadIdx.x, lane = tid & 63;
    // neighbouring groups meet the same cache lines: each XCD (block x % 8) takes
    // a contiguous range of the blocks
    const uint32_t blocks = g.start[g.ng], each = (blocks + 7) / 8;
    const uint32_t blk = blockIdx.x % 8 * each + blockIdx.x / 8;
    if (blockIdx.x / 8 >= each || blk >= blocks || g.start[g.ng + 1] > g.visits_max) return;
    for (int i = tid; i < g.ng; i += kGroupThreads) {
        const uint32_t a = g.start[i], b = g.start[i + 1];
        if (a <= blk && blk < b) {
            s_grp = i;
            s_part = (int)(blk - a);
            s_parts = (int)(b - a);
        }
    }
    if (tid == 0) s_count = 0;
    clear_tables(tab, (int)(kGroupCells * 4));  // ends in a barrier
    const int grp = s_grp;
    const uint32_t part = (uint32_t)s_part, parts = (uint32_t)s_parts;
    const uint32_t lo = g.bound[grp], hi = g.bound[grp + 1] - 1;
    const int f0 = grp * g.G;
    if (lo > hi) return;  // no value has these bins

    // the voxels of the wave's queued field values: entry = local bin row << 10
    // | z << 7 | y << 4 | x within the unit at o, whose starts are in LDS
    const int64_t vplane = g.n[1] * g.n[2];
    // even boxes of 1, 2, 4 .. 64 voxels: a lane keeps one place in the box
    const int lw = lane & ((int)g.box - 1);
    const int ldz = (int)div_magic(lw, g.m_xy), ldy = (int)div_magic(lw - ldz * g.width[1] * g.width[2], g.m_x);
    const uint32_t place = (uint32_t)(ldz * vplane + ldy * g.n[2] + (lw - (ldz * g.width[1] + ldy) * g.width[2]));
    const int per_step = 64 >> g.lbox, e_lane = lane >> g.lbox;
    auto drain_even = [&](int n, const int o[3]) {
        wave_lds_sync();
        const uint16_t *const base = vox + ((int64_t)o[0] * g.width[0] * g.n[1] + (int64_t)o[1] * g.width[1]) * g.n[2] + (int64_t)o[2] * g.width[2];
        const uint32_t sz = (uint32_t)(g.width[0] * vplane), sy = (uint32_t)(g.width[1] * g.n[2]), sx = (uint32_t)g.width[2];
        auto step = [&](int e0, auto U) {
            constexpr int kU = decltype(U)::value;
            uint32_t v[kU], row[kU];
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                const int e = e0 + u * per_step;
                v[u] = 0;
                row[u] = 0;
                if (e < n) {
                    const uint32_t q = queue[e];
                    v[u] = base[place + (q >> 7 & 7) * sz + (q >> 4 & 7) * sy + (q & 15) * sx];
                    row[u] = (q >> 10) * (uint32_t)g.vb;
                }
            }
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                const int bin = (int)bin_of<true>(v[u], vm);  // at most 32768 of them; 0 has none
                if (bin >= 0) atomicAdd(&tab[row[u] + (uint32_t)bin], 1u);
            }
        };
        // whole steps of 8 loads per lane, then pairs
        int e0 = 0;
        for (; e0 + 6 * per_step < n; e0 += 8 * per_step) step(e0 + e_lane, std::integral_constant<int, 8>{});
        for (; e0 < n; e0 += 2 * per_step) step(e0 + e_lane, std::integral_constant<int, 2>{});
        wave_lds_sync();
    };
    auto drain = [&](int n, const int o[3]) {
        if (g.lbox >= 0) {
            drain_even(n, o);
            return;
        }
        wave_lds_sync();
        // a lane takes one row of a value's box, neighbouring values' rows first
        const uint32_t un = (uint32_t)n, m_n = un == 1 ? 0 : 0xffffffffu / un + 1;  // magic reciprocal of n
        const uint32_t items = un * (uint32_t)(g.width[0] * g.width[1]);
        constexpr int kU = 2, kX = 4;
        for (uint32_t i0 = lane; i0 < items; i0 += 64 * kU) {
            uint32_t row[kU];
            const uint16_t *p[kU];
            int len[kU], longest = 0;
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                const uint32_t i = i0 + 64 * u;
                row[u] = 0;
                p[u] = vox;
                len[u] = 0;
                if (i < items) {
                    const uint32_t w = div_magic(i, m_n), q = queue[i - w * un];
                    const uint32_t dz = div_magic(w, g.m_y), dy = w - dz * (uint32_t)g.width[1];
                    const int sz = (int)(q >> 7 & 7), sy = (int)(q >> 4 & 7), sx = (int)(q & 15);
                    const int z = starts[26 + sz] + (int)dz, y = starts[17 + sy] + (int)dy, x = starts[sx];
                    if (z < starts[27 + sz] && y < starts[18 + sy]) {
                        p[u] = vox + ((int64_t)z * g.n[1] + y) * g.n[2] + x;
                        len[u] = starts[sx + 1] - x;
                        row[u] = (q >> 10) * (uint32_t)g.vb;
                    }
                }
                longest = max(longest, len[u]);
            }
            for (int x = 0; x < longest; x += kX) {
                uint32_t v[kU][kX];
#pragma unroll
                for (int u = 0; u < kU; ++u)
#pragma unroll
                    for (int k = 0; k < kX; ++k) v[u][k] = x + k < len[u] ? p[u][x + k] : 0u;
#pragma unroll
                for (int u = 0; u < kU; ++u)
#pragma unroll
                    for (int k = 0; k < kX; ++k) {
                        const int bin = (int)bin_of<true>(v[u][k], vm);  // at most 32768 of them; 0 has none
                        if (bin >= 0) atomicAdd(&tab[row[u] + (uint32_t)bin], 1u);
                    }
            }
        }
        wave_lds_sync();
    };
    // a unit: 16 x 8 x 8 field values of a brick; a lane tests four neighbours
    // in x in each of four layer pairs
    const int lx = (lane & 3) * 4, ly = (lane >> 2) & 7, lz = lane >> 5;
    const int lux = g.lb[2] - 4, luy = g.lb[1] - 3, lp = g.pairs == 4 ? 0 : 2, lunits = lp + lux + luy + g.lb[0] - 3;
    struct Unit {
        int o[3];
        uint2 f[4];
    };
    auto fetch = [&](uint32_t brick, int unit, Unit &un) {
        int *const o = un.o;
        const int pair0 = unit & ((1 << lp) - 1);
        unit >>= lp;
        o[2] = (int)(brick & 0x7ff) << g.lb[2] | (unit & ((1 << lux) - 1)) << 4;
        o[1] = (int)(brick >> 11 & 0x3ff) << g.lb[1] | (unit >> lux & ((1 << luy) - 1)) << 3;
        o[0] = (int)(brick >> 21) << g.lb[0] | unit >> (lux + luy) << 3;
        const int left = (int)g.nf[2] - o[2] - lx;  // values of the row from the lane's first on
        const bool rows = o[1] + ly < g.nf[1];
        const int64_t plane = g.nf[1] * g.nf[2];
        const uint16_t *const p = field + ((int64_t)(o[0] + lz) * g.nf[1] + o[1] + ly) * g.nf[2] + o[2] + lx;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const bool mine = u >= pair0 && u < pair0 + g.pairs;
            const bool in = mine && rows && o[0] + lz + 2 * u < g.nf[0];
            const uint16_t *const q = p + 2 * u * plane;
            uint2 w = make_uint2(0, 0);
            if (in && left >= 4) {
                __builtin_memcpy(&w, q, 8);  // rows start at any 2-byte address
            } else if (in) {
                w.x = left > 0 ? q[0] | (left > 1 ? (uint32_t)q[1] << 16 : 0u) : 0u;
                w.y = left > 2 ? q[2] : 0u;
            }
            un.f[u] = w;
        }
    };
    auto count = [&](const Unit &un) {
        const int *const o = un.o;
        if (g.lbox < 0 && lane < kUnitStarts) {
            const int k = lane < 17 ? 2 : (lane < 26 ? 1 : 0), i = lane - (lane < 17 ? 0 : (lane < 26 ? 17 : 26));
            starts[lane] = g.starts[k][min(o[k] + i, (int)g.nf[k])];
        }
        // which of the lane's 16 values belong to the group
        uint32_t hits = 0;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const uint32_t f[4] = {un.f[u].x & 0xffffu, un.f[u].x >> 16, un.f[u].y & 0xffffu, un.f[u].y >> 16};
#pragma unroll
            for (int k = 0; k < 4; ++k) hits |= f[k] - lo <= hi - lo ? 1u << (4 * u + k) : 0u;  // lo > 0: a zero does not hit
        }
        if (__ballot(hits != 0) == 0) return;
        // queues the lane's values in h, layer pair by layer pair (neighbours in x
        // stay neighbours); returns the wave's count, queueing none beyond kQueue
        auto push = [&](uint32_t h) {
            int at[4], n = 0;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const uint32_t c = (uint32_t)__popc(h >> (4 * u) & 15u);
                const uint64_t c0 = __ballot(c & 1), c1 = __ballot(c & 2), c2 = __ballot(c & 4);
                auto below = [&](uint64_t m) { return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0)); };
                at[u] = n + below(c0) + 2 * below(c1) + 4 * below(c2);
                n += __popcll(c0) + 2 * __popcll(c1) + 4 * __popcll(c2);
            }
            if (n > kQueue) return n;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const uint32_t f[4] = {un.f[u].x & 0xffffu, un.f[u].x >> 16, un.f[u].y & 0xffffu, un.f[u].y >> 16};
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (h >> (4 * u + k) & 1) {
                        const int fi = (int)bin_of<true>(f[k], fm) - f0;
                        queue[at[u]++] = (uint32_t)fi << 10 | (uint32_t)(lz + 2 * u) << 7 | (uint32_t)ly << 4 | (uint32_t)(lx + k);
                    }
            }
            return n;
        };
        // all at once where the queue holds them, else one layer pair (256
        // values at most) at a time
        uint32_t left = hits, part = hits;
#pragma unroll 1
        for (int u = 0; __ballot(left != 0) != 0;) {
            const int n = push(part);
            if (n > kQueue) {
                part = left & 15u;
                u = 1;
                continue;
            }
            if (n > 0) drain(n, o);
            left &= ~part;
            part = left & (15u << (4 * u));
            ++u;
        }
    };

    for (int b0 = 0; b0 < g.bricks; b0 += kGroupThreads) {
        const int i = b0 + tid;
        if (i < g.bricks) {
            const uint32_t r = g.ranges[i], rlo = r >> 16, rhi = r & 0xffffu;
            // bricks go to the group's blocks by a hash of their number
            if (rlo <= hi && rhi >= lo && (((uint32_t)i * 2654435761u) >> 12) % parts == part)
                {
                const uint32_t y = (uint32_t)i / (uint32_t)g.nb[2];
                list[atomicAdd(&s_count, 1)] = (uint32_t)i % (uint32_t)g.nb[2] | y % (uint32_t)g.nb[1] << 11 | y / (uint32_t)g.nb[1] << 21;
            }
        }
        if (tid == 0) s_next = 0;
        __syncthreads();
        const int listed = s_count;
        const bool take = listed > kList - kGroupThreads || b0 + kGroupThreads >= g.bricks;  // uniform
        if (take) {
            // the next unit's values are on their way while one is counted
            auto next = [&](Unit &un) {
                int e = 0;
                if (lane == 0) e = atomicAdd(&s_next, 1);
                e = __builtin_amdgcn_readfirstlane(e);
                if (e >= listed << lunits) return false;
                fetch((uint32_t)__builtin_amdgcn_readfirstlane((int)list[e >> lunits]), e & ((1 << lunits) - 1), un);
                return true;
            };
            Unit a, b;
            bool more = next(a);
            while (more) {
                more = next(b);
                count(a);
                a = b;
            }
        }
        __syncthreads();
        if (take && tid == 0) s_count = 0;
        __syncthreads();
    }
    const int64_t rows = g.fb - f0 < g.G ? g.fb - f0 : g.G;
    flush_tables<true>(tab, rows, g.vb, f0, f0 + rows, bins);
}

// The general form.  Bricks of 32 x 32 x 64 voxels, walked by blocks that each
// take a contiguous range; pairs gather in an LDS hash table of kHashSlots
// keys (linear probing) that also counts its distinct keys.  The table
// reaches the bins, one atomic per distinct pair, when it holds more than
// kFlushAt keys after a step of kStepVoxels voxels, and at the end of the
// range; a step adds at most kStepVoxels keys, so the table is never more than
// half full and a free slot or the key itself is always found.
constexpr int kHashThreads = 128, kPerThread = 8;
constexpr int kStepVoxels = kHashThreads * kPerThread;
constexpr int kHashSlots = 8192;
constexpr int kHashShift = 19;  // 32 - log2(kHashSlots)
constexpr uint32_t kFlushAt = kHashSlots / 2 - kStepVoxels;
constexpr unsigned kHashBlocks = 512;  // two 64 KB blocks per CU of a 256-CU device
constexpr int kBrickX = 64, kBrickY = 32, kBrickZ = 32;
constexpr int kBrickRowsPerStep = kStepVoxels / kBrickX;  // 16 brick rows of 64 voxels per step
constexpr uint32_t kEmpty = 0xffffffffu;
static_assert(kHashSlots == (1 << (32 - kHashShift)), "hash table size");
static_assert(kBrickX % kPerThread == 0 && (kBrickY * kBrickZ) % kBrickRowsPerStep == 0, "brick shape");

struct HashArgs {
    int64_t nZ, nY, nX, nz, ny, nx, vb;
    const int32_t *zmap, *ymap, *xmap;  // voxel coordinate -> field coordinate
    const uint32_t *visits;             // of the grouped form, which counted unless they exceed visits_max; or null
    uint32_t visits_max;
};

template <bool FAST>
__global__ __launch_bounds__(kHashThreads) void k_field_hash(const uint16_t *__restrict__ vox, const uint16_t *__restrict__ field,
                                                             HashArgs a, BinMap vm, BinMap fm,
                                                             unsigned long long *__restrict__ bins) {
    __shared__ uint32_t keys[kHashSlots];
    __shared__ uint32_t counts[kHashSlots];
    __shared__ uint32_t n_keys;
    if (a.visits != nullptr && *a.visits <= a.visits_max) return;
    for (int i = threadIdx.x; i < kHashSlots; i += kHashThreads) {
        keys[i] = kEmpty;
        counts[i] = 0;
    }
    if (threadIdx.x == 0) n_keys = 0;
    __syncthreads();
    const int64_t bx_n = (a.nX + kBrickX - 1) / kBrickX, by_n = (a.nY + kBrickY - 1) / kBrickY;
    const int64_t bricks = bx_n * by_n * ((a.nZ + kBrickZ - 1) / kBrickZ);
    const int64_t per = (bricks + gridDim.x - 1) / gridDim.x;
    const int64_t b0 = (int64_t)blockIdx.x * per, b1 = b0 + per < bricks ? b0 + per : bricks;
    const int xo = (threadIdx.x % (kBrickX / kPerThread)) * kPerThread;
    const int ro = threadIdx.x / (kBrickX / kPerThread);
    constexpr int kSteps = kBrickY * kBrickZ / kBrickRowsPerStep;
    for (int64_t b = b0; b < b1; ++b) {
        const int64_t bx = b % bx_n, by = (b / bx_n) % by_n, bz = b / (bx_n * by_n);
        const int64_t x0 = bx * kBrickX + xo;
        for (int step = 0; step < kSteps; ++step) {
            const int r = step * kBrickRowsPerStep + ro;
            const int64_t Y = by * kBrickY + r % kBrickY, Z = bz * kBrickZ + r / kBrickY;
            if (x0 < a.nX && Y < a.nY && Z < a.nZ) {
                const uint16_t *vrow = vox + (Z * a.nY + Y) * a.nX;
                const uint16_t *frow = field + ((int64_t)a.zmap[Z] * a.ny + a.ymap[Y]) * a.nx;
                uint16_t v[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) v[k] = x0 + k < a.nX ? vrow[x0 + k] : (uint16_t)0;
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    if (x0 + k >= a.nX) break;
                    const uint32_t vi = bin_of<FAST>(v[k], vm);
                    if (vi == kNoBin) continue;
                    const uint32_t fi = bin_of<FAST>(frow[a.xmap[x0 + k]], fm);
                    if (fi == kNoBin) continue;
                    const uint32_t key = fi * (uint32_t)a.vb + vi;
                    uint32_t slot = (key * 2654435761u) >> kHashShift;
                    while (true) {
                        const uint32_t prev = atomicCAS(&keys[slot], kEmpty, key);
                        if (prev == kEmpty || prev == key) {
                            atomicAdd(&counts[slot], 1u);
                            if (prev == kEmpty) atomicAdd(&n_keys, 1u);
                            break;
                        }
                        slot = (slot + 1) & (kHashSlots - 1);
                    }
                }
            }
            __syncthreads();
            const bool flush = n_keys > kFlushAt || (b + 1 == b1 && step + 1 == kSteps);  // uniform: between two barriers
            __syncthreads();
            if (flush) {
                for (int i = threadIdx.x; i < kHashSlots; i += kHashThreads) {
                    const uint32_t key = keys[i];
                    if (key != kEmpty) {
                        atomicAdd(&bins[key], (unsigned long long)counts[i]);
                        keys[i] = kEmpty;
                        counts[i] = 0;
                    }
                }
                if (threadIdx.x == 0) n_keys = 0;
                __syncthreads();
            }
        }
    }
}

// The least field value whose bin is at least b (65536: none).  Bins are
// monotone in the value: subtraction, division by a positive number,
// multiplication and floor all are, rounded or not.
uint32_t least_value(const BinMap &m, int64_t b) {
    uint32_t lo = 0, hi = 65536;  // the value 0 is not counted
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (std::floor(m.c * (((double)mid - m.lo) / m.d)) >= (double)b) hi = mid;
        else lo = mid;
    }
    return hi;
}

}  // namespace

hipError_t launch_field_histogram(const uint16_t *vox, int64_t nZ, int64_t nY, int64_t nX, const uint16_t *field,
                                  int64_t nz, int64_t ny, int64_t nx, uint64_t *bins, int64_t fb, int64_t vb,
                                  double vmin, double vmax, double fmin, double fmax, void *ws,
                                  std::vector<int32_t> &words, hipStream_t s) {
    const BinMap vm = make_bin_map(vmin, vmax, vb, true), fm = make_bin_map(fmin, fmax, fb, false);
    if (vm.vlo > vm.vhi) return hipSuccess;  // no voxel is counted
    const int64_t n[3] = {nZ, nY, nX}, nf[3] = {nz, ny, nx}, nmaps = nZ + nY + nX;
    FieldPlan p;
    make_field_plan(n, nf, fb, vb, vm.fast && fm.fast, p);
    if (4 * p.table_words() > field_workspace_bytes(nZ, nY, nX)) return hipErrorInvalidValue;
    words = std::move(p.words);
    int32_t *const d = static_cast<int32_t *>(ws);
    unsigned long long *const dst = reinterpret_cast<unsigned long long *>(bins);
    const bool grouped = p.grouped;
    const int64_t box = p.width[0] * p.width[1] * p.width[2], bricks = p.bricks;
    FieldGeom g{};
    if (grouped) {
        g.G = (int32_t)p.G;
        g.bricks = (int32_t)bricks;
        g.fb = fb;
        g.vb = vb;
        g.ng = (int32_t)p.ng;
        const int32_t *st = d + nmaps;
        bool even = true;
        for (int k = 0; k < 3; ++k) {
            g.n[k] = n[k];
            g.nf[k] = nf[k];
            g.nb[k] = (int32_t)p.nb[k];
            g.lb[k] = p.lb[k];
            g.width[k] = (int32_t)p.width[k];
            even = even && p.width[k] * nf[k] == n[k];
            g.starts[k] = st;
            st += p.ns[k] + 1;
        }
        auto magic = [](int64_t v) { return v <= 1 ? 0u : (uint32_t)(((uint64_t(1) << 32) + v - 1) / v); };
        g.box = (uint32_t)box;
        const int64_t values = nz * ny * nx, mean = std::max<int64_t>(1, (nZ * nY * nX + values / 2) / values);
        g.mean = (uint32_t)mean;
        g.m_y = magic(p.width[1]);
        g.m_xy = magic(p.width[1] * p.width[2]);
        g.m_x = magic(p.width[2]);
        // testing a field value costs about 1/64 of hashing a voxel (0.7 against
        // 50 ps at 1024^3), and a value stands for `mean` voxels
        g.visits_max = (uint32_t)std::min<int64_t>(0x7fffffff, 64 * mean * bricks);
        // voxels of few values: 13 times that (k_field_plan), less in volumes that do
        // not fill the device with hash blocks, 512 of 2^16 voxels
        g.few_weight = (uint32_t)std::max<int64_t>(16, std::min<int64_t>(208, 208 * (nZ * nY * nX) >> 25));
        g.bound = reinterpret_cast<const uint32_t *>(d) + words.size();
        for (int i = 0; i <= g.ng; ++i)
            words.push_back((int32_t)least_value(fm, i < g.ng ? (int64_t)i * g.G : fb));
        g.start = reinterpret_cast<uint32_t *>(d) + words.size();
        g.ranges = g.start + g.ng + 2;
        g.blocks_wanted = (int32_t)std::max<int64_t>(1, std::min<int64_t>(kGroupBlocks, nZ * nY * nX / kBlockVoxels));
        g.pairs = mean <= 8 ? 4 : 1;
        // 32-bit offsets within a unit
        even = even && box <= 64 && (box & (box - 1)) == 0 && 8 * p.width[0] * nY * nX < (int64_t(1) << 31);
        g.lbox = -1;
        for (int k = 0; even && k <= 6; ++k)
            if (box == int64_t(1) << k) g.lbox = k;
    }
    hipError_t e = hipMemcpyAsync(ws, words.data(), words.size() * 4, hipMemcpyHostToDevice, s);
    if (e != hipSuccess) return e;
    if (grouped) {
        auto *fn = &k_field_groups;
        if ((e = allow_lds(fn, kGroupLds)) != hipSuccess) return e;
        hipLaunchKernelGGL(k_field_ranges, dim3((unsigned)((bricks + 3) / 4)), dim3(256), 0, s, field, g);
        hipLaunchKernelGGL(k_field_plan, dim3(1), dim3(kGroupThreads), 0, s, vox, g, vm);
        hipLaunchKernelGGL(fn, dim3((unsigned)(g.blocks_wanted + g.ng + 7) / 8 * 8), dim3(kGroupThreads), kGroupLds, s, vox, field, g, vm, fm, dst);
    }
    HashArgs h{nZ, nY, nX, nz, ny, nx, vb, d, d + nZ, d + nZ + nY, grouped ? g.start + g.ng + 1 : nullptr, g.visits_max};
    const int64_t hb = ((nX + kBrickX - 1) / kBrickX) * ((nY + kBrickY - 1) / kBrickY) * ((nZ + kBrickZ - 1) / kBrickZ);
    const unsigned grid = (unsigned)std::min<int64_t>(hb, kHashBlocks);
    if (vm.fast && fm.fast) hipLaunchKernelGGL(k_field_hash<true>, dim3(grid), dim3(kHashThreads), 0, s, vox, field, h, vm, fm, dst);
    else hipLaunchKernelGGL(k_field_hash<false>, dim3(grid), dim3(kHashThreads), 0, s, vox, field, h, vm, fm, dst);
    return hipGetLastError();
}

}  // namespace mxb
