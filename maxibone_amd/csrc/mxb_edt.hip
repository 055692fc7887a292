// Euclidean distance transform of a binary volume (gfx950): the core of the
// implant EDT field (src/processing_steps/0950_generate_edt.py:44-66, which
// calls edt.edt of the external `edt` package).  C ABI in
// include/maxibone_edt.h.
//
// Squared distances separably, three passes over (z, y, x) volumes:
//   pass x: g1[i] = min over sites j of the row of (i - j)^2
//   pass y: g2[i] = min_j g1[j] + (i - j)^2 along y
//   pass z: g3[i] = min_j g2[j] + (i - j)^2 along z
// Pass x is a row scan (k_edt_rows).
//
// Passes y and z are the lower envelope of the parabolas g[j] + (i - j)^2.
// Since g[j] + (i - j)^2 = i^2 + (c_j - 2 i j) with c_j = g[j] + j^2, the
// minimum over j is attained at a vertex of the lower convex hull of the
// points (j, c_j), and the minimising vertex moves right as i grows.  With
// at most 4096 voxels per axis, positions are below 2^12 and c below 2^27:
// 32-bit values, with 64-bit cross products.  With lines enough, a lane walks
// one line (k_edt_lines); short lines that are few scan outward (k_edt_scan,
// along z); the rest have one wave per line (k_edt_pass: 64 lanes, a band of L
// positions per lane, 64 L >= n):
//   A. each lane builds the lower hull of its band (monotone chain; the
//      band's values preloaded into registers, the stack in LDS);
//   B. six rounds merge adjacent groups of bands: the lower bridge of two
//      x-separated hulls is found by walking the left end left and the right
//      end right until neither moves (the bands' emptiness from one ballot
//      per round); the merged hull is a prefix of the left hull and a suffix
//      of the right one (each band keeps a [lo, hi) range);
//   C. the surviving vertices are compacted (wave prefix sum);
//   D. vertex m + 1 beats vertex m from an integer switch position on, and
//      the switch positions grow with m: a table holding at each position the
//      largest m + 1 switching there, then a prefix max over the positions,
//      gives every position its vertex.
// The results stay in registers until the line is answered, then overwrite
// the line in LDS.
//
// A block has one wave per line and holds its lines in an LDS tile, loaded
// and stored with coalesced accesses (for the strided passes, consecutive x
// per position); the line count is the largest that keeps a block within
// kBlockBudget bytes of LDS.  Tiles are dealt to the 8 XCDs in contiguous
// ranges, so neighbouring tiles, which share cache lines, meet in one L2.
// Positions in a tile line are padded by one word per 16 (p + p / 16), and
// the band stacks are stored entry-major (entry k of band b at k * 64 + b),
// so that lanes hit different banks.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <string>

#include "maxibone_diffusion.h"
#include "maxibone_edt.h"
#include "mxb_hist.h"
#include "mxb_internal.h"

namespace mxb {

namespace {

constexpr uint32_t kNone = MXB_EDT_NONE;
// The wave's min and max into mm[0], mm[1]: one atomic per value, only when
// it improves the global one.
__device__ __forceinline__ void fold_minmax(uint32_t lo, uint32_t hi, uint32_t *mm) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        lo = min(lo, (uint32_t)__shfl_xor((int)lo, d, 64));
        hi = max(hi, (uint32_t)__shfl_xor((int)hi, d, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        if (lo < __hip_atomic_load(mm, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(mm, lo);
        if (hi > __hip_atomic_load(mm + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(mm + 1, hi);
    }
}

// The correctly rounded square root of a whole number below 2^26 (as float32):
// the reciprocal square root and one residual, in a third of sqrtf's
// instructions.  Equal to sqrtf for every such value if the instruction returns
// the rounded reciprocal root; if it returns a neighbour, which is its bound, for
// all but seven, and for those it does not.
__device__ __forceinline__ float root(uint32_t d2) {
    const float x = (float)d2, y = __builtin_amdgcn_rsqf(x);
    const float g = x * y;
    return d2 == 0 ? 0.0f : __builtin_fmaf(__builtin_fmaf(-g, g, x), 0.5f * y, g);
}

enum EdtOut { kSquared, kDistance, kField };  // what the last pass writes
constexpr int kMaxLines = 8;              // lines (= waves) per block
constexpr int kMetaInts = 3 * 64;         // per wave: band lo, hi and spare
constexpr int kBlockBudget = 80 * 1024;   // LDS bytes per block (two blocks per CU)

struct EdtPass {
    const void *in;        // uint8 (first pass) or uint32
    uint32_t *out;         // uint32, or float bits (last pass)
    int64_t n;             // positions per line
    int64_t pos_stride;    // elements between positions
    int64_t n_inner, inner_stride;
    int64_t n_outer, outer_stride;
    int lines;             // lines per block (power of two)
    int pitch;             // LDS words per tile line
    const uint8_t *cyl;    // last pass: cylinder mask indexed by the line, or null
    uint32_t *minmax;      // last pass: ordered-encoded min and max
};

__device__ __forceinline__ int tix(int p) { return p + (p >> 4); }

// LDS ordering between the lanes of one wave (each wave's LDS operations
// execute in order; this keeps the compiler from moving them across).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ uint32_t f2ord_d(float f) {
    const uint32_t b = __float_as_uint(f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float ord2f_d(uint32_t o) {
    return __uint_as_float((o & 0x80000000u) ? (o & 0x7fffffffu) : ~o);
}

// cross((x0,c0), (x1,c1), (x2,c2)) <= 0: the middle point is on or above the
// segment between the outer two (x0 < x1 < x2).  Positions are below 2^12
// and c = g + x^2 below 3 * 4096^2 < 2^26 + 2^24, so the operands are 32-bit
// and each product (below 2^39) comes from one 32 x 32 -> 64 multiply.
__device__ __forceinline__ bool not_below(int x0, int c0, int x1, int c1, int x2, int c2) {
    return (int64_t)(x1 - x0) * (c2 - c0) - (int64_t)(c1 - c0) * (x2 - x0) <= 0;
}

// Highest / lowest set bit of a nonzero 64-bit mask.
__device__ __forceinline__ int top_bit(uint64_t m) { return 63 - __builtin_clzll(m); }
__device__ __forceinline__ int low_bit(uint64_t m) { return __builtin_ctzll(m); }
__device__ __forceinline__ uint64_t bits_below(int k) { return k <= 0 ? 0ull : (k >= 64 ? ~0ull : (1ull << k) - 1); }

// Position from which hull vertex m + 1 beats vertex m (they tie at no
// integer before it): the least i with c1 - c0 < 2 i (x1 - x0), clamped to
// [0, n].
__device__ __forceinline__ int switch_pos(int x0, int c0, int x1, int c1, int n) {
    const int num = c1 - c0;
    if (num < 0) return 0;
    const int t = (int)((uint32_t)num / (uint32_t)(2 * (x1 - x0))) + 1;
    return t > n ? n : t;
}

// Envelope pass along y or z: uint32 -> uint32, or uint32 -> float
// distance x cylinder with the block's min and max folded into P.minmax.
// Lines per block that the LDS budget admits for a band length L (the host
// clamps to it): a line needs 4 (pitch + 64 L + kMetaInts) bytes, over 25 KB
// once L = 64 (n > 2048) and over 13 KB at L = 32.  The kernel's launch bound
// follows it, so the long-line instances may hold their per-lane arrays
// (64 values each at L = 64) in registers without spilling.
constexpr int edt_max_lines(int L) { return L >= 64 ? 2 : (L >= 32 ? 4 : kMaxLines); }

template <int L, EdtOut OUT>
__global__ __launch_bounds__(edt_max_lines(L) * 64) void k_edt_pass(EdtPass P) {
    extern __shared__ __attribute__((aligned(16))) uint32_t smem[];
    const int kThreads = P.lines * 64;  // one wave per line
    const int n = (int)P.n;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    uint32_t *const tile = smem;
    // per wave: stk (64 L uint16: the band stacks, entry k of band b at
    // k * 64 + b, later the switch table, position p at tpos(p)), env (64 L
    // uint16); lanes touch consecutive entries, so no bank conflicts
    uint16_t *const stk = reinterpret_cast<uint16_t *>(smem + P.lines * P.pitch) + wv * 128 * L;
    uint16_t *const env = stk + 64 * L;
    int *const blo = reinterpret_cast<int *>(smem + P.lines * P.pitch + P.lines * 64 * L) + wv * kMetaInts;
    auto tpos = [](int p) { return (p % L) * 64 + p / L; };
    int *const bhi = blo + 64;

    // tile of this block (XCD-aware order: block b runs on XCD b % 8)
    const int64_t chunks = (P.n_inner + P.lines - 1) / P.lines;
    const int64_t B = chunks * P.n_outer;
    const int64_t b = blockIdx.x, q = B / 8, rem = B % 8, xcd = b % 8;
    const int64_t t_id = xcd * q + (xcd < rem ? xcd : rem) + b / 8;
    const int64_t outer = t_id / chunks, inner0 = (t_id % chunks) * P.lines;
    const int nl = (int)(P.n_inner - inner0 < P.lines ? P.n_inner - inner0 : P.lines);
    const int64_t base = outer * P.outer_stride + inner0 * P.inner_stride;
    const bool lines_contig = P.inner_stride == 1 && P.pos_stride != 1;
    int lshift = 0;
    while ((1 << lshift) < P.lines) ++lshift;

    // ---- load
    if (lines_contig) {
        const int total = P.lines * n;
        for (int t = tid; t < total; t += kThreads) {
            const int l = t & (P.lines - 1), p = t >> lshift;
            if (l >= nl) continue;
            const int64_t o = base + l + (int64_t)p * P.pos_stride;
            tile[l * P.pitch + tix(p)] = static_cast<const uint32_t *>(P.in)[o];
        }
    } else {
        for (int l = 0; l < nl; ++l)
            for (int p = tid; p < n; p += kThreads) {
                const int64_t o = base + (int64_t)l * P.inner_stride + (int64_t)p * P.pos_stride;
                tile[l * P.pitch + tix(p)] = static_cast<const uint32_t *>(P.in)[o];
            }
    }
    __syncthreads();

    uint32_t omin = 0xffffffffu, omax = 0u;
    const int b0 = lane * L;
    for (int l = wv; l < nl; l += P.lines) {
        uint32_t *const g = tile + l * P.pitch;
        float cyl = 1.0f;
        if (OUT == kField && P.cyl != nullptr) cyl = P.cyl[inner0 + l] != 0 ? 1.0f : 0.0f;
        auto cval = [&](int x) -> int { return (int)g[tix(x)] + x * x; };

        // A. lower hull of the band's points (the band's values preloaded)
        uint32_t gv[L];
#pragma unroll
        for (int t = 0; t < L; ++t) gv[t] = b0 + t < n ? g[tix(b0 + t)] : kNone;
        int h = 0;
        int xa = 0, ca = 0, xb = 0, cb = 0;  // second and top of the stack
#pragma unroll
        for (int t = 0; t < L; ++t) {
            const int j = b0 + t;
            if (gv[t] != kNone) {
                const int cj = (int)gv[t] + j * j;
                while (h >= 2 && not_below(xa, ca, xb, cb, j, cj)) {
                    --h;
                    xb = xa;
                    cb = ca;
                    if (h >= 2) {
                        xa = stk[(h - 2) * 64 + lane];
                        ca = cval(xa);
                    }
                }
                stk[h * 64 + lane] = (uint16_t)j;
                if (h >= 1) {
                    xa = xb;
                    ca = cb;
                }
                xb = j;
                cb = cj;
                ++h;
            }
        }
        int my_lo = 0, my_hi = h;
        blo[lane] = 0;
        bhi[lane] = h;
        wave_sync();

        // B. merge groups of bands [l0, mid) and [mid, l0 + gs); the bands'
        // emptiness at the start of a round comes from one ballot
        for (int gs = 2; gs <= 64; gs <<= 1) {
            const uint64_t ne = __ballot(my_hi > my_lo);
            if ((lane & (gs - 1)) == 0) {
                const int l0 = lane, mid = lane + gs / 2, r = lane + gs;
                const uint64_t left = ne & bits_below(mid) & ~bits_below(l0);
                const uint64_t right = ne & bits_below(r) & ~bits_below(mid);
                if (left != 0 && right != 0) {
                    int ba = top_bit(left), bb = low_bit(right);
                    int ia = bhi[ba] - 1, ib = blo[bb];
                    int ax = stk[ia * 64 + ba], bx = stk[ib * 64 + bb];
                    int ac = cval(ax), bc = cval(bx);
                    int lo_a = blo[ba], hi_b = bhi[bb];  // range ends of the current bands
                    for (;;) {
                        bool moved = false;
                        for (;;) {  // left end moves left while it is not below (prev, b)
                            int pa = ba, pi = ia - 1, plo = lo_a;
                            if (pi < lo_a) {
                                const uint64_t before = left & bits_below(ba);
                                if (before == 0) break;
                                pa = top_bit(before);
                                plo = blo[pa];
                                pi = bhi[pa] - 1;
                            }
                            const int px = stk[pi * 64 + pa], pc = cval(px);
                            if (!not_below(px, pc, ax, ac, bx, bc)) break;
                            ba = pa; ia = pi; ax = px; ac = pc; lo_a = plo;
                            moved = true;
                        }
                        for (;;) {  // right end moves right while it is not below (a, next)
                            int na = bb, ni = ib + 1, nhi = hi_b;
                            if (ni >= hi_b) {
                                const uint64_t after = right & ~bits_below(bb + 1);
                                if (after == 0) break;
                                na = low_bit(after);
                                ni = blo[na];
                                nhi = bhi[na];
                            }
                            const int qx = stk[ni * 64 + na], qc = cval(qx);
                            if (!not_below(ax, ac, bx, bc, qx, qc)) break;
                            bb = na; ib = ni; bx = qx; bc = qc; hi_b = nhi;
                            moved = true;
                        }
                        if (!moved) break;
                    }
                    bhi[ba] = ia + 1;
                    for (int k = ba + 1; k < mid; ++k) bhi[k] = blo[k];
                    blo[bb] = ib;
                    for (int k = mid; k < bb; ++k) blo[k] = bhi[k];
                }
            }
            wave_sync();
            my_lo = blo[lane];
            my_hi = bhi[lane];
        }

        // C. compact the hull into env
        const int cnt = my_hi - my_lo;
        int incl = cnt;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int v = __shfl_up(incl, d, 64);
            if (lane >= d) incl += v;
        }
        const int H = __shfl(incl, 63, 64);
        const int off = incl - cnt;
        for (int k = 0; k < cnt; ++k) env[off + k] = stk[(my_lo + k) * 64 + lane];
        wave_sync();

        // D. minimising vertex of every position: vertex m + 1 takes over from
        // m at switch_pos(m); the switch table (in the stack's place) holds at
        // each position the largest m + 1 switching there, and a prefix max
        // over positions gives each position its vertex
        uint32_t res[L];
        if (H == 0) {
#pragma unroll
            for (int t = 0; t < L; ++t) res[t] = kNone;
        } else {
#pragma unroll
            for (int t = 0; t < L; ++t) stk[t * 64 + lane] = 0;
            wave_sync();
            // edge m = 64 k + lane; edge m + 1 is the next lane's (lane 63:
            // lane 0's of the next chunk); a sentinel n + 1 follows the last edge
            auto edge_switch = [&](int m) -> int {
                if (m >= H - 1) return n + 1;
                const int x0 = env[m], x1 = env[m + 1];
                return switch_pos(x0, cval(x0), x1, cval(x1), n);
            };
            int s_cur = edge_switch(lane);
            for (int m0 = 0; m0 < H - 1; m0 += 64) {
                const int s_nxt = edge_switch(m0 + 64 + lane);
                const int s_dn = __shfl_down(s_cur, 1, 64);
                const int s_first = __shfl(s_nxt, 0, 64);
                const int s_next = lane < 63 ? s_dn : s_first;
                const int m = m0 + lane;
                if (m < H - 1 && s_next > s_cur && s_cur < n) stk[tpos(s_cur)] = (uint16_t)(m + 1);
                s_cur = s_nxt;
            }
            wave_sync();
            // the lane's own maximum first; the running maximum is read again
            // below rather than held, so only res[] stays live (L = 64 would
            // otherwise need 2 x 64 VGPRs and spill)
            int run = 0;
#pragma unroll
            for (int t = 0; t < L; ++t) run = max(run, (int)stk[t * 64 + lane]);
            int carry = run;  // exclusive prefix max over lanes
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int v = __shfl_up(carry, d, 64);
                if (lane >= d) carry = max(carry, v);
            }
            carry = __shfl_up(carry, 1, 64);
            if (lane == 0) carry = 0;
            run = carry;
#pragma unroll
            for (int t = 0; t < L; ++t) {
                const int i = b0 + t;
                run = max(run, (int)stk[t * 64 + lane]);
                const int xm = env[run];
                res[t] = g[tix(xm)] + (uint32_t)((i - xm) * (i - xm));
            }
        }
        wave_sync();
#pragma unroll
        for (int t = 0; t < L; ++t) {
            const int i = b0 + t;
            if (i < n) {
                if (OUT != kSquared) {
                    const float d = res[t] == kNone ? INFINITY : sqrtf((float)res[t]);
                    const float f = d * cyl;
                    if (OUT == kField) {
                        const uint32_t o = f2ord_d(f);
                        omin = min(omin, o);
                        omax = max(omax, o);
                    }
                    g[tix(i)] = __float_as_uint(f);
                } else {
                    g[tix(i)] = res[t];
                }
            }
        }
        wave_sync();
    }
    __syncthreads();

    // ---- store
    if (lines_contig) {
        const int total = P.lines * n;
        for (int t = tid; t < total; t += kThreads) {
            const int l = t & (P.lines - 1), p = t >> lshift;
            if (l >= nl) continue;
            P.out[base + l + (int64_t)p * P.pos_stride] = tile[l * P.pitch + tix(p)];
        }
    } else {
        for (int l = 0; l < nl; ++l)
            for (int p = tid; p < n; p += kThreads)
                P.out[base + (int64_t)l * P.inner_stride + (int64_t)p * P.pos_stride] = tile[l * P.pitch + tix(p)];
    }
    if (OUT == kField) {
        // block min / max (in the tile's first words, free after the store),
        // then one atomic per value, only when it improves the global one
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) {
            omin = min(omin, (uint32_t)__shfl_xor((int)omin, d, 64));
            omax = max(omax, (uint32_t)__shfl_xor((int)omax, d, 64));
        }
        __syncthreads();
        if (lane == 0) {
            tile[2 * wv] = omin;
            tile[2 * wv + 1] = omax;
        }
        __syncthreads();
        if (tid == 0) {
            for (int w = 1; w < P.lines; ++w) {
                omin = min(omin, tile[2 * w]);
                omax = max(omax, tile[2 * w + 1]);
            }
            if (omin < __hip_atomic_load(P.minmax, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                atomicMin(P.minmax, omin);
            if (omax > __hip_atomic_load(P.minmax + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                atomicMax(P.minmax + 1, omax);
        }
    }
}

__global__ void k_edt_minmax_init(uint32_t *mm) {
    if (threadIdx.x == 0) {
        mm[0] = 0xffffffffu;
        mm[1] = 0u;
    }
}

// Pass x: the distance to the nearest site of the row (sites: data == 0, or
// data != 0 when INVERT), as uint16 (0xffff: none) for the lane-per-line pass
// or squared as uint32 (kNone) for k_edt_pass.  `group` lanes (a power of two)
// share a row, 16 C voxels each, read and written in 16-byte pieces at any
// alignment; the nearest site in the lanes before and after comes from a
// prefix max and a suffix min over the group.  1024^3: 2.15 -> 1.13 ms (2.8
// TB/s) against one voxel per lane and chunk; half its time is the 20
// instructions per voxel (four rows per lane with their loads together: the
// same, and slower for small volumes).
template <bool INVERT, int C, typename OUT>
__global__ __launch_bounds__(256) void k_edt_rows(const uint8_t *__restrict__ data, int64_t rows, int nx, int group,
                                                  OUT *__restrict__ out) {
    constexpr int kSpan = 16 * C;
    constexpr int kFar = 20000;  // beyond any distance, and a difference of two still fits 16 bits
    const int lane = threadIdx.x & 63, gl = lane & (group - 1);
    const int64_t r = ((int64_t)blockIdx.x * 256 + threadIdx.x) / group;
    const int x0 = gl * kSpan;
    const uint8_t *const p = data + r * nx + x0;
    uint64_t m = 0;  // the lane's sites
    const int left = r < rows ? nx - x0 : 0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        uint32_t bits = 0;  // nonzero bytes of 16
        if (left >= 16 * c + 16) {
            uint32_t w[4];
            __builtin_memcpy(w, p + 16 * c, 16);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t t = (((w[k] & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w[k]) & 0x80808080u;
                bits |= ((t * 0x00204081u) >> 28) << (4 * k);  // bits 7, 15, 23, 31 to 28 .. 31
            }
            bits = INVERT ? bits : ~bits & 0xffffu;
        } else {
#pragma unroll
            for (int k = 0; k < 16; ++k)
                if (16 * c + k < left && ((p[16 * c + k] != 0) == INVERT)) bits |= 1u << k;
        }
        m |= (uint64_t)bits << (16 * c);
    }
    int last = m != 0 ? x0 + top_bit(m) : -kFar, first = m != 0 ? x0 + low_bit(m) : kFar;
    for (int d = 1; d < group; d <<= 1) {
        const int a = __shfl_up(last, d, group), b = __shfl_down(first, d, group);
        if (gl >= d) last = max(last, a);
        if (gl + d < group) first = min(first, b);
    }
    int before = __shfl_up(last, 1, group), after = __shfl_down(first, 1, group);
    if (gl == 0) before = -kFar;
    if (gl == group - 1) after = kFar;
    if (left <= 0) return;
    uint16_t d[kSpan];
#pragma unroll
    for (int k = 0; k < kSpan; ++k) {
        if (m >> k & 1) before = x0 + k;
        d[k] = (uint16_t)(x0 + k - before);
    }
#pragma unroll
    for (int k = kSpan - 1; k >= 0; --k) {
        if (m >> k & 1) after = x0 + k;
        const int e = min((int)d[k], after - x0 - k);
        d[k] = e > 4095 ? (uint16_t)0xffffu : (uint16_t)e;
    }
    OUT *const o = out + r * nx + x0;
    constexpr int kPer = 16 / (int)sizeof(OUT);
#pragma unroll
    for (int k = 0; k < kSpan; k += kPer) {
        OUT v[kPer];
#pragma unroll
        for (int t = 0; t < kPer; ++t) {
            if constexpr (sizeof(OUT) == 2) v[t] = d[k + t];
            else v[t] = d[k + t] == 0xffffu ? kNone : (uint32_t)d[k + t] * d[k + t];
        }
        if (left >= k + kPer) {
            __builtin_memcpy(o + k, v, 16);
        } else {
#pragma unroll
            for (int t = 0; t < kPer; ++t)
                if (k + t < left) o[k + t] = v[t];
        }
    }
}

// ---- one lane per line
// With lines enough to fill the device, a lane walks one line serially: the
// lower hull by a stack (each point is pushed once and popped at most once),
// then the answers from the far end, the stack shrinking as earlier vertices
// take over.  64 neighbouring lines are consecutive in memory, so all loads
// and stores are whole cache lines, and neighbours' stacks move alike.  The
// two uppermost entries live in registers, the next kRing in an LDS ring, and
// deeper ones in memory (`stack`), reached by evictions and by refills that
// the whole wave makes together; each is one 32-bit word:
//   Y: input uint16 distances; memory entries hold the position as uint16 in
//      the half of the workspace that the input leaves free, the value is
//      read again from the input;
//   Z: input uint32 squared distances; entries hold position << gbits | value
//      and are stored over the input (entry m <= positions read so far).
// The turn test is done in float64, where products below 2^39 are exact.
// 1024^3 implant field: y 10.1 -> 1.98 ms, z 14.8 -> 3.73 ms against one wave
// per line (k_edt_pass: 7100 instructions per 1024-voxel line and one min/max
// atomic per block).  z is bound by its vector instructions, 113 per 64 voxels
// (93 % of the SIMDs' cycles); y, 35 per 64 voxels and 55 %, by its serial loads
// beside them.
struct EdtLines {
    const void *in;
    void *stack;
    uint32_t *out;
    int n;                       // positions per line
    int64_t pos_stride;          // elements between positions
    int64_t lines, inner;        // lines; consecutive ones
    int64_t outer_stride;        // elements between runs of `inner` lines
    int gbits;                   // Z: bits of a value
    const uint8_t *cyl;          // kField: cylinder mask per line, or null
    uint32_t *minmax;            // kField: ordered-encoded min and max
};

constexpr int kLineThreads = 256;
constexpr int kRing = 16;    // entries per line in LDS (16 KB per block: eight blocks per CU)
constexpr int kRefill = 8;

template <bool Y, EdtOut OUT>
__global__ __launch_bounds__(kLineThreads) void k_edt_lines(EdtLines P) {
    __shared__ uint32_t ring[kRing][kLineThreads];
    const int tid = threadIdx.x;
    const int64_t line = (int64_t)blockIdx.x * kLineThreads + tid;
    bool live = line < P.lines;
    const int64_t run = live ? line / P.inner : 0;
    const int64_t base = live ? run * P.outer_stride + (line - run * P.inner) : 0;
    const int64_t ps = P.pos_stride;
    const int n = P.n;
    const uint16_t *const in16 = static_cast<const uint16_t *>(P.in) + base;
    const uint32_t *const in32 = static_cast<const uint32_t *>(P.in) + base;
    uint16_t *const st16 = static_cast<uint16_t *>(P.stack) + base;
    uint32_t *const st32 = static_cast<uint32_t *>(P.stack) + base;
    const int gbits = P.gbits;
    const uint32_t gmask = (1u << gbits) - 1;

    auto load = [&](int j) -> uint32_t {
        if constexpr (Y) return in16[j * ps];
        else return in32[j * ps];
    };
    auto none = [&](uint32_t g) { return Y ? g == 0xffffu : g == kNone; };
    auto entry = [&](int j, uint32_t g) { return Y ? (uint32_t)j << 16 | g : (uint32_t)j << gbits | g; };
    auto pos_of = [&](uint32_t e) { return (int)(Y ? e >> 16 : e >> gbits); };
    auto val_of = [&](uint32_t e) { return (int)(Y ? (e & 0xffffu) * (e & 0xffffu) : e & gmask); };

    uint32_t *const out = P.out + base;
    uint32_t lo = 0xffffffffu, hi = 0;
    float cyl = 1.0f;
    if (OUT == kField && P.cyl != nullptr && live) cyl = P.cyl[line] != 0 ? 1.0f : 0.0f;
    auto put = [&](uint32_t *o, uint32_t d2) {
        if (!live) return;
        if constexpr (OUT == kSquared) {
            *o = d2;
        } else {
            const float f = (d2 == kNone ? INFINITY : root(d2)) * cyl;
            *o = __float_as_uint(f);
            if constexpr (OUT == kField) {
                const uint32_t o = f2ord_d(f);
                lo = min(lo, o);
                hi = max(hi, o);
            }
        }
    };

    // A wave whose sites are near everywhere needs no hull: a least value of at
    // most kNear^2 among the positions nearer than kNear is the line's.  The
    // hull's chains are longest there (a whole line of zeros stays on the
    // stack; in noise some lane of 64 pops at every step).  From the first run of
    // 8 that holds a position without such a value a wave goes on with the
    // hull: the best vertex moves right as the position does, so vertices more
    // than kNear - 1 before that run are not needed.
    // Dense noise at 512^3, whole call: 3.12 -> 0.54 ms (one wave per line, 2.62);
    // one plane of sites in 100x700x701, whose line of zeros along y is a chain
    // of 700 memory accesses to the hull: 1.03 -> 0.45 ms (0.82).
    constexpr int kNear = 5, kAhead = 8;
    constexpr uint32_t kFarValue = 1u << 29;
    const uint32_t nothing = Y ? 0xffffu : kNone;
    auto fetch = [&](int j) { return live && j < n ? load(j) : nothing; };
    auto value = [&](uint32_t g) { return none(g) ? kFarValue : (Y ? g * g : g); };
    uint32_t cur[kAhead], nxt[kAhead];  // the next positions' input
#pragma unroll
    for (int k = 0; k < kAhead; ++k) cur[k] = fetch(k);
    uint32_t v[2 * kNear + 6];  // positions i0 - 4 .. i0 + 11
    auto nearest = [&](int k) {  // the least of position i0 + k
        const uint32_t *const c = v + k + kNear - 1;
        uint32_t d2 = c[0];
#pragma unroll
        for (int t = 1; t < kNear; ++t) d2 = min(d2, min(c[-t], c[t]) + (uint32_t)(t * t));
        return d2;
    };
#pragma unroll
    for (int k = 0; k < kNear - 1; ++k) v[k] = kFarValue;
#pragma unroll
    for (int k = 0; k < kAhead; ++k) v[kNear - 1 + k] = value(cur[k]);
    // lanes that hold nothing at the line's start are left to the hull, where an
    // empty line costs little; the first of the others to fail ends the walk
    const uint32_t start = nearest(0);
    const bool far = start >= kFarValue;
    int i0 = 0;  // uniform
    if (__ballot(live && !far) != 0 && __ballot(live && !far && start > (uint32_t)(kNear * kNear)) == 0) {
#pragma unroll
        for (int k = kAhead; k < kNear + 7; ++k) v[kNear - 1 + k] = value(fetch(k));
        for (; i0 < n; i0 += 8) {
            uint32_t more[8], d2[8], worst = 0;
#pragma unroll
            for (int k = 0; k < 8; ++k) more[k] = fetch(i0 + kNear + 7 + k);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                d2[k] = nearest(k);
                if (i0 + k < n) worst = max(worst, d2[k]);
            }
            if (__ballot(live && !far && worst > (uint32_t)(kNear * kNear)) != 0) break;
            if (!far)
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    if (i0 + k < n) put(out + (i0 + k) * ps, d2[k]);
#pragma unroll
            for (int k = 0; k < 2 * kNear - 2; ++k) v[k] = v[k + 8];
#pragma unroll
            for (int k = 0; k < 8; ++k) v[2 * kNear - 2 + k] = value(more[k]);
        }
    }
    const bool some_far = __ballot(live && far) != 0;
    if (i0 >= n) {
        if (!some_far) {
            if constexpr (OUT == kField) fold_minmax(lo, hi, P.minmax);
            return;
        }
        if (!far) live = false;  // this lane is done
    }
    if (some_far) i0 = 0;
    const int begin = i0 > kNear ? i0 - kNear : 0;  // the hull's first position
    if (begin > 0 || !live)
#pragma unroll
        for (int k = 0; k < kAhead; ++k) cur[k] = fetch(begin + k);

    // entries [0, vlo) are in memory, [vlo, h - 2) in the ring, h - 2 and
    // h - 1 (the top) in registers
    int h = 0, vlo = 0;
    auto evict = [&]() {  // the ring's lowest entry to memory
        const uint32_t e = ring[vlo & (kRing - 1)][tid];
        if constexpr (Y) st16[vlo * ps] = (uint16_t)(e >> 16);
        else st32[vlo * ps] = e;
        ++vlo;
    };
    auto refill = [&]() {  // up to kRefill entries from memory, below the ring's
        const int c = vlo < kRefill ? vlo : kRefill;
        uint32_t e[kRefill];
#pragma unroll
        for (int k = 0; k < kRefill; ++k) {
            e[k] = 0;
            if (k < c) e[k] = Y ? (uint32_t)st16[(vlo - 1 - k) * ps] : st32[(vlo - 1 - k) * ps];
        }
        if constexpr (Y) {
#pragma unroll
            for (int k = 0; k < kRefill; ++k)
                if (k < c) e[k] = e[k] << 16 | in16[e[k] * ps];
        }
#pragma unroll
        for (int k = 0; k < kRefill; ++k)
            if (k < c) ring[(vlo - 1 - k) & (kRing - 1)][tid] = e[k];
        vlo -= c;
    };

    // forward: the hull
    uint32_t pa = 0, pb = 0;                     // second and top entry
    double xa = 0, ca = 0, xb = 0, cb = 0;       // their points (j, g + j^2)
    auto open = [&](uint32_t e, double &x, double &c) {
        const int j = pos_of(e);
        x = (double)j;
        c = (double)(val_of(e) + __mul24(j, j));
    };
    for (int j0 = begin; j0 < n; j0 += kAhead) {
#pragma unroll
        for (int k = 0; k < kAhead; ++k) nxt[k] = fetch(j0 + kAhead + k);
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
            const int j = j0 + k;
            if (!none(cur[k])) {
                const uint32_t e = entry(j, cur[k]);
                const double x = (double)j;
                const double c = (double)((int)(Y ? cur[k] * cur[k] : cur[k]) + j * j);
                while (h >= 2 && __builtin_fma(xb - xa, c - ca, -((cb - ca) * (x - xa))) <= 0.0) {
                    --h;  // the top is on or above the segment between its neighbours
                    pb = pa; xb = xa; cb = ca;
                    if (h >= 2) {
                        if (h - 2 < vlo) refill();
                        pa = ring[(h - 2) & (kRing - 1)][tid];
                        open(pa, xa, ca);
                    }
                }
                if (h >= 2) {  // the second goes to the ring
                    if (h - 2 - vlo == kRing) evict();
                    ring[(h - 2) & (kRing - 1)][tid] = pa;
                }
                pa = pb; xa = xb; ca = cb;
                pb = e; xb = x; cb = c;
                ++h;
            }
        }
#pragma unroll
        for (int k = 0; k < kAhead; ++k) cur[k] = nxt[k];
    }

    // backward: position i belongs to the top until the vertex below ties or wins
    int xt = pos_of(pb), gt = val_of(pb), xs = pos_of(pa), gs = val_of(pa);
    uint32_t *o = out + (n - 1) * ps;
    for (int i = n - 1; i >= i0; --i, o -= ps) {
        // keep four entries at hand: all lanes with room refill together
        if (__ballot(vlo > 0 && h - 2 - vlo < 4) != 0 && vlo > 0 && h - 2 - vlo <= kRing - kRefill) refill();
        while (h >= 2 && gs + __mul24(i - xs, i - xs) <= gt + __mul24(i - xt, i - xt)) {
            --h;
            xt = xs; gt = gs;
            if (h >= 2) {
                if (h - 2 < vlo) refill();
                const uint32_t e = ring[(h - 2) & (kRing - 1)][tid];
                xs = pos_of(e);
                gs = val_of(e);
            }
        }
        const uint32_t d2 = h > 0 ? (uint32_t)(gt + __mul24(i - xt, i - xt)) : kNone;
        put(o, d2);
    }
    if constexpr (OUT == kField) fold_minmax(lo, hi, P.minmax);
}

// ---- outward scan
// With too few lines for a lane each, and short ones, every position looks
// outward for its minimum: g[j] + (i - j)^2 cannot win once (i - j)^2 and the
// line's least g reach the best value found.  A block holds 64 neighbouring
// lines in LDS (a lane's line in its own bank); a thread answers 8 consecutive
// positions of a line together, so a value read serves 8 of them with an addition and a minimum
// each, the squares being uniform: from the left, at distance t from the
// first position, g + t^2 + 2 t k + k^2 for position k, and mirrored from the
// right.
//
// Where values are far apart (one plane of sites in a deep volume) an outward
// look would cross the whole line value by value.  Beyond the nearest 16 or 32
// positions, or at once where a run of 8 itself holds nothing, it goes by runs
// of 16 and passes over those whose least value, from where they are, improves
// nothing.  One plane of sites, whole call: 256^3 501 -> 190 us (k_edt_pass 220),
// 500x250x250 1.19 -> 0.44 ms (0.36); a rod with specks at 129x300x257 259 -> 243
// us, dense noise there 212 -> 209.
constexpr int kScanLines = 64, kScanMax = 512;  // 132 KB of LDS at most
constexpr int kRunBits = 4;
constexpr int kRun = 1 << kRunBits;             // positions per run

// LDS of a block: the values, and per run and line the high half of its least
// value as a float.
__host__ __device__ inline size_t scan_smem(int n) {
    return (size_t)n * kScanLines * 4 + (size_t)((n + kRun - 1) / kRun) * kScanLines * 2;
}

template <EdtOut OUT>
__global__ __launch_bounds__(512) void k_edt_scan(EdtLines P) {
    extern __shared__ int32_t vals[];  // [n][kScanLines]
    __shared__ int32_t least[kScanLines];
    constexpr int kFarValue = 1 << 29;
    const int n = P.n, lane = threadIdx.x & 63, wv = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const int look_out = n <= 128 ? 2 * kRun : kRun;  // positions looked at one by one
    const int64_t line = (int64_t)blockIdx.x * kScanLines + lane;
    const bool live = line < P.lines;
    const int64_t run = live ? line / P.inner : 0;
    const int64_t base = live ? run * P.outer_stride + (line - run * P.inner) : 0;
    const uint32_t *const in = static_cast<const uint32_t *>(P.in) + base;
    if (threadIdx.x < kScanLines) least[lane] = kFarValue;
    __syncthreads();
    int gmin = kFarValue;
    for (int j = wv; j < n; j += waves) {
        const uint32_t g = live ? in[j * P.pos_stride] : kNone;
        const int v = g == kNone ? kFarValue : (int)g;
        vals[j * kScanLines + lane] = v;
        gmin = min(gmin, v);
    }
    atomicMin(&least[lane], gmin);
    __syncthreads();
    gmin = least[lane];
    float cyl = 1.0f;
    if (OUT == kField && P.cyl != nullptr && live) cyl = P.cyl[line] != 0 ? 1.0f : 0.0f;
    uint32_t lo = 0xffffffffu, hi = 0;
    // b[k] holds the best of position i0 + k found so far, less k^2
    auto put8 = [&](const int (&b)[8], int i0) {
        if (!live) return;
        uint32_t *o = P.out + base + i0 * P.pos_stride;
#pragma unroll
        for (int k = 0; k < 8; ++k, o += P.pos_stride) {
            if (i0 + k >= n) break;
            const int best = b[k] + k * k;
            const uint32_t d2 = best < kFarValue / 2 ? (uint32_t)best : kNone;
            if constexpr (OUT == kSquared) {
                *o = d2;
            } else {
                const float f = (d2 == kNone ? INFINITY : root(d2)) * cyl;
                *o = __float_as_uint(f);
                if constexpr (OUT == kField) {
                    lo = min(lo, f2ord_d(f));
                    hi = max(hi, f2ord_d(f));
                }
            }
        }
    };
    auto take = [&](int (&b)[8], int i0, int from, int to) {  // the values from .. to
#pragma unroll 1
        for (int j = from; j <= to; j += 4) {
            int g[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) g[u] = vals[min(j + u, to) * kScanLines + lane];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int d = i0 - min(j + u, to), c = g[u] + d * d;
#pragma unroll
                for (int k = 0; k < 8; ++k) b[k] = min(b[k], c + 2 * d * k);
            }
        }
    };
    // The rest of the line, beyond `seen` positions either way, by runs.  A wave
    // works out the runs' least values when it first needs them (all waves that
    // do write the same).
    const int runs = (n + kRun - 1) / kRun;
    uint16_t *const low = reinterpret_cast<uint16_t *>(vals + n * kScanLines) + lane;
    bool have_low = false;
    auto by_runs = [&](int (&b)[8], int i0, int seen) {
        if (!have_low) {
#pragma unroll 1
            for (int q = 0; q < runs; ++q) {
                int v = kFarValue;
#pragma unroll 8
                for (int u = 0; u < kRun; ++u) v = min(v, vals[min(kRun * q + u, n - 1) * kScanLines + lane]);
                low[q * kScanLines] = (uint16_t)(__float_as_uint((float)(v & ~7)) >> 16);  // rounded down: below 2^27, or 2^29
            }
            wave_sync();
            have_low = true;
        }
        int worst = 0;
        auto look = [&]() {
            worst = 0;
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (i0 + k < n) worst = max(worst, b[k] + k * k);
        };
        look();
#pragma unroll 1
        for (int side = -1; side <= 1; side += 2) {
            int q = side < 0 ? (i0 - 1 - seen) >> kRunBits : (i0 + 8 + seen) >> kRunBits;
#pragma unroll 1
            for (; q >= 0 && q < runs; q += side) {
                const int d = max(0, side < 0 ? i0 - (kRun * q + kRun - 1) : kRun * q - (i0 + 7));  // at the nearest
                if (__ballot(worst > gmin + d * d) == 0) break;
                if (__ballot(worst > (int)__uint_as_float((uint32_t)low[q * kScanLines] << 16) + d * d) == 0) continue;
                take(b, i0, kRun * q, min(kRun * q + kRun - 1, n - 1));
                look();
            }
        }
    };
    for (int i0 = 8 * wv; i0 < n; i0 += 8 * waves) {
        // l[k]: best from the left and within, less k^2; r[k]: from the right, less (7 - k)^2
        int l[8], rt[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) l[k] = rt[k] = kFarValue;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int g = i0 + j < n ? vals[(i0 + j) * kScanLines + lane] : kFarValue;
#pragma unroll
            for (int k = 0; k < 8; ++k) l[k] = min(l[k], g + (j - k) * (j - k) - k * k);
        }
        const int reach = max(i0, n - 8 - i0);
        int seen = -1;  // positions looked at on either side, where that is not enough (uniform)
        if (__ballot(l[0] >= kFarValue / 2 && gmin < kFarValue / 2) != 0) seen = 0;
        for (int t0 = 1; t0 <= reach && seen < 0; t0 += 4) {
            int worst = 0;
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (i0 + k < n) worst = max(worst, min(l[k] + k * k, rt[k] + (7 - k) * (7 - k)));
            if (__ballot(worst > gmin + t0 * t0) == 0) break;
            if (t0 > look_out) {
                seen = t0 - 1;
                break;
            }
            int a[4], b[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int t = t0 + u, jl = i0 - t, jr = i0 + 7 + t;
                a[u] = jl >= 0 ? vals[jl * kScanLines + lane] : kFarValue;
                b[u] = jr < n ? vals[jr * kScanLines + lane] : kFarValue;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int t = t0 + u, ca = a[u] + t * t, cb = b[u] + t * t;
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    l[k] = min(l[k], ca + 2 * t * k);
                    rt[k] = min(rt[k], cb + 2 * t * (7 - k));
                }
            }
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) l[k] = min(l[k], rt[k] + (7 - k) * (7 - k) - k * k);
        if (seen >= 0) by_runs(l, i0, seen);
        put8(l, i0);
    }
    if constexpr (OUT == kField) fold_minmax(lo, hi, P.minmax);
}

// general.hh:96-118 on the float field: (uint16)((f - vmin) / (vmax - vmin) *
// 65535) with vmax starting at FLT_MIN (general.hh:78), then x cylinder.  A
// thread takes 8 neighbours of a plane (the cylinder mask is one plane), at
// any alignment.  The division is by a value all threads share, done with its
// reciprocal and a residual (SharedDiv in mxb_hist.h); 1024^3: 1.8 -> 1.2 ms, where
// rows, a 64-bit division per item and IEEE division sequences held the loads
// back.
__global__ __launch_bounds__(256) void k_edt_to_u16(const float *__restrict__ f, int64_t nz, int64_t plane,
                                                    const uint8_t *__restrict__ cyl,
                                                    const uint32_t *__restrict__ mm,
                                                    uint16_t *__restrict__ out) {
    const float vmin = ord2f_d(mm[0]);
    const float vmax = fmaxf(ord2f_d(mm[1]), FLT_MIN);
    const SharedDiv div(vmax - vmin);
    const int64_t e0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
    if (e0 >= plane) return;
    const int left = plane - e0 < 8 ? (int)(plane - e0) : 8;
    uint8_t c[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) c[k] = 1;
    if (cyl != nullptr) {
        if (left == 8) __builtin_memcpy(c, cyl + e0, 8);
        else
            for (int k = 0; k < left; ++k) c[k] = cyl[e0 + k];
    }
    auto convert = [&](auto by) {
        for (int64_t z = blockIdx.y; z < nz; z += gridDim.y) {
            const float *const src = f + z * plane + e0;
            uint16_t *const dst = out + z * plane + e0;
            float v[8];
            if (left == 8) __builtin_memcpy(v, src, 32);
            else
                for (int k = 0; k < 8; ++k) v[k] = k < left ? src[k] : 0.0f;
            uint16_t o[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                o[k] = (uint16_t)(by(v[k] - vmin) * 65535.0f);
                if (c[k] == 0) o[k] = 0;
            }
            if (left == 8) __builtin_memcpy(dst, o, 16);
            else
                for (int k = 0; k < left; ++k) dst[k] = o[k];
        }
    };
    if (div.exact) convert([&](float x) { return div.quick(x); });
    else convert([&](float x) { return x / div.d; });
}

// Band length per lane: the least power of two with 64 L >= n.
int64_t band_of(int64_t n) {
    int64_t L = 1;
    while (64 * L < n) L <<= 1;
    return L;
}

size_t pass_smem(const EdtPass &P) {
    const int64_t L = band_of(P.n);
    return (size_t)4 * P.lines * ((size_t)P.pitch + (size_t)(64 * L) + kMetaInts);
}

template <int L, EdtOut OUT>
hipError_t launch_l(const EdtPass &P, hipStream_t s) {
    if (P.lines > edt_max_lines(L)) return hipErrorInvalidValue;  // beyond the launch bound
    const size_t smem = pass_smem(P);
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_edt_pass<L, OUT>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) return e;
    const int64_t blocks = ((P.n_inner + P.lines - 1) / P.lines) * P.n_outer;
    hipLaunchKernelGGL((k_edt_pass<L, OUT>), dim3((unsigned)blocks), dim3(P.lines * 64), smem, s, P);
    return hipGetLastError();
}

template <EdtOut OUT>
hipError_t launch_mode(const EdtPass &P, hipStream_t s) {
    const int64_t need = (P.n + 63) / 64;
    if (need <= 1) return launch_l<1, OUT>(P, s);
    if (need <= 2) return launch_l<2, OUT>(P, s);
    if (need <= 4) return launch_l<4, OUT>(P, s);
    if (need <= 8) return launch_l<8, OUT>(P, s);
    if (need <= 16) return launch_l<16, OUT>(P, s);
    if (need <= 32) return launch_l<32, OUT>(P, s);
    return launch_l<64, OUT>(P, s);
}

// Geometry of the pass along axis a (0 z, 1 y, 2 x) of an (nz, ny, nx) volume.
EdtPass pass_geom(int a, int64_t nz, int64_t ny, int64_t nx) {
    EdtPass P{};
    if (a == 2) {
        P.n = nx; P.pos_stride = 1;
        P.n_inner = nz * ny; P.inner_stride = nx; P.n_outer = 1; P.outer_stride = 0;
    } else if (a == 1) {
        P.n = ny; P.pos_stride = nx;
        P.n_inner = nx; P.inner_stride = 1; P.n_outer = nz; P.outer_stride = ny * nx;
    } else {
        P.n = nz; P.pos_stride = ny * nx;
        P.n_inner = ny * nx; P.inner_stride = 1; P.n_outer = 1; P.outer_stride = 0;
    }
    P.pitch = (int)(P.n + P.n / 16 + 1);
    // one wave per line; the largest count within the block budget
    int lines = edt_max_lines((int)band_of(P.n));
    while (lines > 1 && (int64_t)4 * lines * (P.pitch + 64 * band_of(P.n) + kMetaInts) > kBlockBudget)
        lines >>= 1;
    P.lines = lines;
    return P;
}

hipError_t run_pass(EdtOut mode, EdtPass P, hipStream_t s) {
    if (P.n_inner * P.n_outer == 0 || P.n == 0) return hipSuccess;
    if (mode == kSquared) return launch_mode<kSquared>(P, s);
    return mode == kDistance ? launch_mode<kDistance>(P, s) : launch_mode<kField>(P, s);
}

template <bool INVERT, typename OUT>
hipError_t launch_rows(const uint8_t *data, int64_t rows, int64_t nx, OUT *out, hipStream_t s) {
    const int c = (int)((nx + 1023) / 1024);  // 1 .. 4 (at most 4096 voxels)
    int group = 1;
    while (group < 64 && group * 16 * c < nx) group <<= 1;
    const unsigned blocks = (unsigned)((rows * group + 255) / 256);
    if (c == 1) hipLaunchKernelGGL((k_edt_rows<INVERT, 1, OUT>), dim3(blocks), dim3(256), 0, s, data, rows, (int)nx, group, out);
    else if (c == 2) hipLaunchKernelGGL((k_edt_rows<INVERT, 2, OUT>), dim3(blocks), dim3(256), 0, s, data, rows, (int)nx, group, out);
    else hipLaunchKernelGGL((k_edt_rows<INVERT, 4, OUT>), dim3(blocks), dim3(256), 0, s, data, rows, (int)nx, group, out);
    return hipGetLastError();
}

template <typename OUT>
hipError_t run_rows(const uint8_t *data, bool invert, int64_t rows, int64_t nx, OUT *out, hipStream_t s) {
    if (rows == 0 || nx == 0) return hipSuccess;
    return invert ? launch_rows<true>(data, rows, nx, out, s) : launch_rows<false>(data, rows, nx, out, s);
}

template <EdtOut OUT>
hipError_t launch_scan(const EdtLines &P, hipStream_t s) {
    const size_t smem = scan_smem(P.n);
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_edt_scan<OUT>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) return e;
    const unsigned waves = P.n > 128 ? 8 : 4;
    hipLaunchKernelGGL(k_edt_scan<OUT>, dim3((unsigned)((P.lines + kScanLines - 1) / kScanLines)), dim3(64 * waves), smem, s, P);
    return hipGetLastError();
}

hipError_t run_scan(const EdtLines &P, EdtOut mode, hipStream_t s) {
    if (mode == kSquared) return launch_scan<kSquared>(P, s);
    return mode == kDistance ? launch_scan<kDistance>(P, s) : launch_scan<kField>(P, s);
}

int bits_of(int64_t v) {
    int b = 0;
    while (v >> b) ++b;
    return b;
}

template <bool Y>
hipError_t run_lines(const EdtLines &P, EdtOut mode, hipStream_t s) {
    const dim3 grid((unsigned)((P.lines + kLineThreads - 1) / kLineThreads)), block(kLineThreads);
    if constexpr (Y) {
        hipLaunchKernelGGL((k_edt_lines<true, kSquared>), grid, block, 0, s, P);
    } else {
        if (mode == kSquared) hipLaunchKernelGGL((k_edt_lines<false, kSquared>), grid, block, 0, s, P);
        else if (mode == kDistance) hipLaunchKernelGGL((k_edt_lines<false, kDistance>), grid, block, 0, s, P);
        else hipLaunchKernelGGL((k_edt_lines<false, kField>), grid, block, 0, s, P);
    }
    return hipGetLastError();
}

int64_t vol_words_bytes(int64_t n) { return (n * 4 + 255) / 256 * 256; }

#define MXB_EHIP(expr)                                                          \
    do {                                                                        \
        hipError_t _e = (expr);                                                 \
        if (_e != hipSuccess) {                                                 \
            set_error(std::string(#expr) + ": " + hipGetErrorString(_e));       \
            return _e == hipErrorOutOfMemory ? ENOMEM_ : EDEVICE;               \
        }                                                                       \
    } while (0)

int check_extents(const char *who, int64_t nz, int64_t ny, int64_t nx) {
    if (nz < 0 || ny < 0 || nx < 0) {
        set_error(std::string(who) + ": negative extent");
        return EINVAL_;
    }
    if (nz > MXB_EDT_MAX_AXIS || ny > MXB_EDT_MAX_AXIS || nx > MXB_EDT_MAX_AXIS) {
        set_error(std::string(who) + ": at most " + std::to_string(MXB_EDT_MAX_AXIS) + " voxels per axis");
        return EINVAL_;
    }
    return OK;
}

// The three passes; the first reads `data` (sites: data == 0, or != 0 when
// `invert`), the last writes `last_out` in `mode` (kField: x cylinder, and
// min/max into mm).
int device_edt_core(const uint8_t *data, int64_t nz, int64_t ny, int64_t nx, bool invert, uint32_t *a,
                    uint32_t *b, uint32_t *last_out, EdtOut mode, const uint8_t *cyl, uint32_t *mm,
                    hipStream_t s) {
    if (mode == kField) {
        hipLaunchKernelGGL(k_edt_minmax_init, dim3(1), dim3(64), 0, s, mm);
        MXB_EHIP(hipGetLastError());
    }
    // A lane per line needs lines enough for the device, and is bound by the
    // latency of its serial steps below that (129x300x257: along y, 33 K lines,
    // 140 us against 95 for k_edt_pass; 400x333x417, 139 K lines along z, 793
    // us for the whole field against 1044 scanning outward and 1316 for
    // k_edt_pass).  Along z, where
    // after the y pass every plane with a site has values throughout, short
    // lines that are not plenty scan outward (whole field of 200^3: 211 us, k_edt_pass 391;
    // 256^3: 302, lanes 454; 500x250x250: 599, k_edt_pass 733, lanes 780);
    // along y, where most values are none, scanning is no faster.
    constexpr int64_t kLinesWanted = 65536, kLinesPlenty = 131072;
    if (nz * nx >= kLinesWanted) {
        // distances in the first half of `a`, the stacks in the second
        uint16_t *const d = reinterpret_cast<uint16_t *>(a);
        MXB_EHIP(run_rows(data, invert, nz * ny, nx, d, s));
        const EdtLines P{d, d + nz * ny * nx, b, (int)ny, nx, nz * nx, nx, ny * nx, 0, nullptr, nullptr};
        MXB_EHIP(run_lines<true>(P, kSquared, s));
    } else {
        EdtPass py = pass_geom(1, nz, ny, nx);
        py.in = a; py.out = b;
        MXB_EHIP(run_rows(data, invert, nz * ny, nx, a, s));
        MXB_EHIP(run_pass(kSquared, py, s));
    }
    // a value and a position share 32 bits up to 1024-voxel axes
    const int gbits = bits_of((nx - 1) * (nx - 1) + (ny - 1) * (ny - 1));
    const bool scan = nz <= kScanMax && ny * nx < kLinesPlenty;
    if (!scan && ny * nx >= kLinesWanted && gbits + bits_of(nz - 1) <= 32) {
        const EdtLines P{b, b, last_out, (int)nz, ny * nx, ny * nx, ny * nx, 0, gbits, cyl, mm};
        MXB_EHIP(run_lines<false>(P, mode, s));
    } else if (scan) {
        const EdtLines P{b, nullptr, last_out, (int)nz, ny * nx, ny * nx, ny * nx, 0, 0, cyl, mm};
        MXB_EHIP(run_scan(P, mode, s));
    } else {
        EdtPass pz = pass_geom(0, nz, ny, nx);
        pz.in = b; pz.out = last_out; pz.cyl = cyl; pz.minmax = mm;
        MXB_EHIP(run_pass(mode, pz, s));
    }
    return OK;
}

struct EBuf {
    void *p = nullptr;
    ~EBuf() {
        if (p) (void)hipFree(p);
    }
    int alloc(size_t n) {
        hipError_t e = hipMalloc(&p, n > 0 ? n : 1);
        if (e != hipSuccess) {
            set_error(std::string("hipMalloc: ") + hipGetErrorString(e));
            return e == hipErrorOutOfMemory ? ENOMEM_ : EDEVICE;
        }
        return OK;
    }
};

}  // namespace

}  // namespace mxb

using namespace mxb;

extern "C" {

int64_t mxb_edt_workspace_bytes(int64_t nz, int64_t ny, int64_t nx) {
    if (nz < 0 || ny < 0 || nx < 0) return -1;
    return 2 * vol_words_bytes(nz * ny * nx) + 256;
}

int mxb_device_edt(const uint8_t *dev_data, int64_t nz, int64_t ny, int64_t nx, uint32_t *dev_sq_out,
                   float *dev_out, void *dev_workspace, void *stream) {
    int rc = check_extents("edt", nz, ny, nx);
    if (rc != OK) return rc;
    const int64_t n = nz * ny * nx;
    if (n == 0) return OK;
    if (dev_data == nullptr || dev_workspace == nullptr || (dev_sq_out == nullptr && dev_out == nullptr)) {
        set_error("edt: null buffer");
        return EINVAL_;
    }
    hipStream_t s = (hipStream_t)stream;
    uint32_t *a = (uint32_t *)dev_workspace;
    uint32_t *b = (uint32_t *)((char *)dev_workspace + vol_words_bytes(n));
    uint32_t *mm = (uint32_t *)((char *)dev_workspace + 2 * vol_words_bytes(n));
    if (dev_sq_out != nullptr && (rc = device_edt_core(dev_data, nz, ny, nx, false, a, b, dev_sq_out, kSquared,
                                                       nullptr, mm, s)) != OK)
        return rc;
    if (dev_out != nullptr && (rc = device_edt_core(dev_data, nz, ny, nx, false, a, b, (uint32_t *)dev_out, kDistance,
                                                    nullptr, mm, s)) != OK)
        return rc;
    return OK;
}

int mxb_device_edt_field(const uint8_t *dev_implant_solid, int64_t nz, int64_t ny, int64_t nx,
                         const uint8_t *dev_cylinder, uint16_t *dev_out, void *dev_workspace, void *stream) {
    int rc = check_extents("edt_field", nz, ny, nx);
    if (rc != OK) return rc;
    const int64_t n = nz * ny * nx;
    if (n == 0) return OK;
    if (dev_implant_solid == nullptr || dev_out == nullptr || dev_workspace == nullptr) {
        set_error("edt_field: null buffer");
        return EINVAL_;
    }
    hipStream_t s = (hipStream_t)stream;
    uint32_t *a = (uint32_t *)dev_workspace;
    uint32_t *b = (uint32_t *)((char *)dev_workspace + vol_words_bytes(n));
    uint32_t *mm = (uint32_t *)((char *)dev_workspace + 2 * vol_words_bytes(n));
    // 0950:41 negates the implant mask: the sites are the implant voxels
    if ((rc = device_edt_core(dev_implant_solid, nz, ny, nx, true, a, b, a, kField, dev_cylinder, mm, s)) != OK)
        return rc;
    const dim3 grid((unsigned)((ny * nx + 2047) / 2048), (unsigned)std::min<int64_t>(nz, 65535));
    hipLaunchKernelGGL(k_edt_to_u16, grid, dim3(256), 0, s, (const float *)a, nz, ny * nx, dev_cylinder, mm, dev_out);
    MXB_EHIP(hipGetLastError());
    return OK;
}

int mxb_edt(const uint8_t *data, int64_t nz, int64_t ny, int64_t nx, uint32_t *sq_out, float *out,
            int verbose) {
    (void)verbose;
    int rc = check_extents("edt", nz, ny, nx);
    if (rc != OK) return rc;
    const int64_t n = nz * ny * nx;
    if (n == 0) return OK;
    if (data == nullptr || (sq_out == nullptr && out == nullptr)) {
        set_error("edt: null buffer");
        return EINVAL_;
    }
    EBuf d, ws, o2, of;
    if ((rc = d.alloc(n)) || (rc = ws.alloc(mxb_edt_workspace_bytes(nz, ny, nx)))) return rc;
    if (sq_out != nullptr && (rc = o2.alloc(n * 4))) return rc;
    if (out != nullptr && (rc = of.alloc(n * 4))) return rc;
    MXB_EHIP(staged_copy(d.p, data, n, true, nullptr));
    rc = mxb_device_edt((const uint8_t *)d.p, nz, ny, nx, (uint32_t *)o2.p, (float *)of.p, ws.p, nullptr);
    if (rc != OK) return rc;
    if (sq_out != nullptr) MXB_EHIP(staged_copy(sq_out, o2.p, n * 4, false, nullptr));
    if (out != nullptr) MXB_EHIP(staged_copy(out, of.p, n * 4, false, nullptr));
    return OK;
}

int mxb_edt_field(const uint8_t *implant_solid, int64_t nz, int64_t ny, int64_t nx, const uint8_t *cylinder,
                  uint16_t *out, int verbose) {
    (void)verbose;
    int rc = check_extents("edt_field", nz, ny, nx);
    if (rc != OK) return rc;
    const int64_t n = nz * ny * nx;
    if (n == 0) return OK;
    if (implant_solid == nullptr || out == nullptr) {
        set_error("edt_field: null buffer");
        return EINVAL_;
    }
    EBuf d, ws, o, c;
    if ((rc = d.alloc(n)) || (rc = ws.alloc(mxb_edt_workspace_bytes(nz, ny, nx))) || (rc = o.alloc(n * 2)))
        return rc;
    if (cylinder != nullptr && (rc = c.alloc(ny * nx))) return rc;
    MXB_EHIP(staged_copy(d.p, implant_solid, n, true, nullptr));
    if (cylinder != nullptr) MXB_EHIP(hipMemcpy(c.p, cylinder, ny * nx, hipMemcpyHostToDevice));
    rc = mxb_device_edt_field((const uint8_t *)d.p, nz, ny, nx, (const uint8_t *)c.p, (uint16_t *)o.p, ws.p,
                              nullptr);
    if (rc != OK) return rc;
    MXB_EHIP(staged_copy(out, o.p, n * 2, false, nullptr));
    return OK;
}

}  // extern "C"
