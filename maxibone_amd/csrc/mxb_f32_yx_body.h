// Fused y -> x pass of the masked 3D diffusion (gfx950), FP32 MFMA form.
//
// A repetition of the FP32 form runs as two kernels: the z-pass (A -> B) and
// this one (B -> A), which applies the y-pass to a strip of rows and the x-pass
// to its result in LDS, illuminating (src/lib/cpp/cpu/diffusion.cc:295-302,
// :314-320), so the (z, x, y) round trip through memory between the two
// disappears.  The body is shared by the single-volume kernel (mxb_f32_yx.hip)
// and the batched one (mxb_batched.hip).  Order, taps and accumulation chains are the separate passes'
// (mxb_f32_dma_body.h): the values are the same bit for bit.
//
// Block (the body below) = 512 threads (8 waves) on plane z, output rows [ya, ya + 64) and
// columns [xa, xb).  It marches along x in groups of 32 columns; iteration i:
//   A. waits until group i's columns, rows ya - RT .. ya + 64 + RT, have landed
//      in staging, barrier;
//   B. issues group i + 1 into the buffer consumed at iteration i - 1, and the
//      mask words of the pair that iteration i + 1 completes;
//   C. y-pass of group i and x-pass of pair p = i - L - 1 side by side, two
//      independent MFMA chains per wave: wave w takes rows 16 (w % 4) .. +15
//      and columns 16 (w / 4) .. +15 of the group (of the pair);
//   D. the y results go to the ring of G groups as rows of 64 y for the x-pass
//      of later iterations; the x results are illuminated and stored from the
//      registers, four columns of a row per lane.
// The x-pass of pair p reads groups p .. p + L, written by iteration p + L, so
// one barrier an iteration orders everything.
//
// LDS layouts, free of bank conflicts for each half of a wave: a staged row is
// 32 columns whose two halves are swapped in odd rows (an operand read takes 16
// columns of 4 consecutive rows).  A ring slot of 16 x by 64 y holds, for each
// x % 4 and y, the four values x / 4 = 0 .. 3 next to each other, so one
// 16-byte read serves four chunks of the x-pass; y ^ (x % 4) is stored in y's
// place, so a y-pass result's writes fall in distinct banks.
//
// Bound: the FP32 matrix cores from R = 40 on (busy 74 % of the cycles at 512^3, R =
// 40: 0.52 ms a launch; 56 % at R = 12), below that the chain of an iteration (barrier, operand reads,
// products, ring writes) beside 3.7 TB/s of memory traffic (512^3, R = 12: 0.28
// ms).  Two blocks share a CU up to R = 40 and three up to R = 16, which hides
// more than a second or third group in flight would (256^3, sigma 5: 805 us
// against 795).  Against the separate y- and x-passes: 257x331x403 sigma 4, ten
// repetitions 2.55 -> 1.69 ms, 256^3 sigma 5 921 -> 794 us, 512^3 sigma 3, four
// repetitions 2.85 -> 2.06 ms, 24x40x72 sigma 2, three repetitions 43 -> 29 us.
#pragma once
#include "mxb_dma.h"
#include "mxb_internal.h"
#include "mxb_lds_body.h"

namespace mxb {

struct YXGeom {
    int64_t ny, nx;                 // extents of a plane, of which (ny + 512) * pitch < 2^28
    int64_t pitch, plane;           // strides of rows and planes
    int64_t mask_plane, mask_word;  // mask-word strides: planes, 32 columns
};

template <int RT>
struct YXShape {
    static constexpr int NW = 8;
    static constexpr int C = LdsShape<RT>::C;
    static constexpr int W = LdsShape<RT>::W;
    static constexpr int L = W / 2;          // groups the x-pass needs after its own
    static constexpr int G = L + 2;          // ring groups
    static constexpr int NR = 64 + 2 * RT;   // staged rows
    static constexpr int SBUF = NR * 32;     // floats per staged group
    static constexpr int GRP = 2 * 16 * 64;  // floats per ring group
    static constexpr int TAPS = 4 * C + 32;
    static constexpr int BYTES = (G * GRP + 2 * (SBUF + 64) + TAPS) * 4;
    static constexpr int BLOCKS = 160 * 1024 / BYTES < 3 ? 160 * 1024 / BYTES : 3;  // on a CU
    static_assert(BLOCKS > 0 && RT % 4 == 0 && NR % 8 == 0, "whole loads of 8 rows");
};

// An 8-byte store to an address aligned to 2 bytes.
typedef uint32_t v2u32 __attribute__((ext_vector_type(2)));
typedef v2u32 __attribute__((aligned(2))) v2u32_a2;

// One block's share: rows [ya, ya + 64) and columns [xa, xb) of plane z, xa a
// multiple of 32; `taps` holds the 2 RT + 1 centred taps (any address space),
// `smem` YXShape<RT>::BYTES of LDS.  ANY: rows of any 4-byte alignment (4-byte
// loads), else rows of whole 16-byte pieces (a piece may pass the row's end
// where the pitch does).
template <int RT, bool OUTF, bool OUTU, bool ANY, typename TapSrc>
__device__ __forceinline__ void f32_yx_body(const float *__restrict__ in, float *__restrict__ out_f32,
                                            uint16_t *__restrict__ out_u16, const uint32_t *__restrict__ bits,
                                            const YXGeom &g, int64_t z, int ya, int xa, int xb, const TapSrc &taps,
                                            float *__restrict__ smem) {
    using S = YXShape<RT>;
    constexpr int C = S::C, W = S::W, L = S::L, G = S::G, NW = S::NW;
    static_assert(OUTF || OUTU, "at least one output");
    float *const ring = smem;
    float *const staging = ring + G * S::GRP;
    uint32_t *const mring = reinterpret_cast<uint32_t *>(staging + 2 * S::SBUF);
    float *const tap_lds = staging + 2 * (S::SBUF + 64);

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, kg = lane >> 4;

    const int ny = (int)g.ny, nx = (int)g.nx, pitch = (int)g.pitch;
    const int npairs = (xb - xa + 31) / 32;
    const int ngroups = npairs + L, nit = npairs + L + 1;

    for (int i = tid; i < S::TAPS; i += 512) {
        const int t = i - 16;
        tap_lds[i] = (t >= 0 && t <= 2 * RT) ? taps[t >= 0 && t <= 2 * RT ? t : 0] : 0.0f;
    }

    // ---- group loads: load q of a group is rows RPL q .. of staging, one wave
    // each; wave w issues loads w, w + 8, ...  Offsets are bytes from the plane's
    // start: rows outside the plane pass its end (or wrap past it), columns
    // outside a row are sent there, and read zeros.
    constexpr int RPL = ANY ? 2 : 8;              // rows per load
    constexpr int NLOADS = S::NR / RPL;           // per group, over the waves
    constexpr int NI = (NLOADS + NW - 1) / NW;    // per wave, at most
    constexpr uint32_t kOutside = 0x80000000u;
    const v4u32 buf = raw_buffer(in + z * g.plane, 4u * (uint32_t)(ny * pitch));
    const uint32_t stage_lds = lds_addr(staging);
    const int lrow = ANY ? lane >> 5 : lane >> 3;
    const int lcol = ANY ? (lane & 31) ^ (16 * (lane >> 5)) : 4 * ((lane & 7) ^ (4 * ((lane >> 3) & 1)));
    uint32_t loff = 4u * (uint32_t)((ya - RT + RPL * wv + lrow) * pitch + xa - RT + lcol);
    const uint32_t lstep = 4u * (uint32_t)(RPL * NW) * (uint32_t)pitch;
    int lx = xa - RT + lcol;
    // mask words of the 64 rows, by the last wave
    const uint32_t *const msrc = bits + z * g.mask_plane + (xa / 32) * g.mask_word + ya + lane;
    const bool mrow_ok = ya + lane < ny;
    auto issue_group = [&](int i) {
        const uint32_t dst = stage_lds + (uint32_t)((i & 1) * S::SBUF * 4);
        const bool ok = i < ngroups && (uint32_t)lx < (uint32_t)nx;
        uint32_t off = ok ? loff : kOutside;
        const uint32_t step = ok ? lstep : 0u;
#pragma unroll
        for (int n = 0; n < NI; ++n) {
            if (n * NW + NW > NLOADS && n * NW + wv >= NLOADS) break;  // uniform
            const uint32_t to = dst + (uint32_t)((n * NW + wv) * RPL * 128);
            if constexpr (ANY) dma4_buf(to, buf, off);
            else dma16_buf(to, buf, off);
            off += step;
        }
        if (wv == NW - 1) {
            const int p = i - L - 1;
            const bool mok = mrow_ok && p >= 0 && p < npairs;
            const void *src = mok ? static_cast<const void *>(msrc + p * g.mask_word) : static_cast<const void *>(g_dma_zero);
            dma4(lds_addr(mring) + (uint32_t)((i & 1) * 256), src);
        }
        loff += 128;
        lx += 32;
    };
    issue_group(0);
    __syncthreads();  // tap table
    float tv[C];
#pragma unroll
    for (int c = 0; c < C; ++c) tv[c] = tap_lds[4 * c + kg - col + 16];

    // this wave's 16 rows and, in the group and in the pair, 16 columns
    const int rt = wv & 3, u = wv >> 2;
    const int yo = (16 * rt + kg) * 32 + 16 * (u ^ (kg & 1)) + col;
    int yw[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
        yw[e] = u * 1024 + ((col & 3) * 64 + ((16 * rt + 4 * kg + e) ^ (col & 3))) * 4 + (col >> 2);
    const int xo = (kg * 64 + ((16 * rt + col) ^ kg)) * 4;
    const int y = ya + 16 * rt + col;
    const bool y_ok = y < ny;
    int64_t off = z * g.plane + (int64_t)y * pitch + xa + 16 * u + 4 * kg;
    float *const sinkf = reinterpret_cast<float *>(g_dma_sink + lane);
    uint16_t *const sinku = reinterpret_cast<uint16_t *>(g_dma_sink + lane);

    constexpr int ST = (OUTF ? 1 : 0) + (OUTU ? 1 : 0);
    int wgrp = 0;  // i % G
    for (int i = 0; i < nit; ++i) {
        // group i's loads are followed only by the stores of iteration i - 1
        if (i >= L + 2) vm_wait<ST>();
        else vm_wait<0>();
        __syncthreads();
        if (i + 1 < nit) issue_group(i + 1);
        const int p = i - L - 1;
        const float *const st = staging + (i & 1) * S::SBUF + yo;
        float ys[C];
        v4f xs[W];
        v4f accy = {0.0f, 0.0f, 0.0f, 0.0f}, accx = {0.0f, 0.0f, 0.0f, 0.0f};
        // slot 2 p + u + q is half (u + q) % 2 of group p + (u + q) / 2; group p
        // is the oldest, wgrp + 1
        int sb[W];
#pragma unroll
        for (int q = 0; q < W; ++q) {
            int gi = wgrp + 1 + ((u + q) >> 1);
            gi = gi >= G ? gi - G : gi;
            sb[q] = gi * S::GRP + ((u + q) & 1) * 1024;
        }
        // columns outside the volume hold zeros, and so do their y results
        const int xs0 = xa - RT + 32 * i + 16 * u;
        const bool do_y = i < ngroups && xs0 + 15 >= 0 && xs0 < nx, do_x = p >= 0;
        if (do_y && do_x) {
#pragma unroll
            for (int c = 0; c < C; ++c) ys[c] = st[128 * c];
#pragma unroll
            for (int q = 0; q < W; ++q) xs[q] = *reinterpret_cast<const v4f *>(&ring[sb[q] + xo]);
#pragma unroll
            for (int c = 0; c < C; ++c) {
                accy = __builtin_amdgcn_mfma_f32_16x16x4f32(tv[c], ys[c], accy, 0, 0, 0);
                accx = __builtin_amdgcn_mfma_f32_16x16x4f32(tv[c], xs[c / 4][c % 4], accx, 0, 0, 0);
            }
        } else if (do_y) {
#pragma unroll
            for (int c = 0; c < C; ++c) ys[c] = st[128 * c];
#pragma unroll
            for (int c = 0; c < C; ++c) accy = __builtin_amdgcn_mfma_f32_16x16x4f32(tv[c], ys[c], accy, 0, 0, 0);
        } else if (do_x) {
#pragma unroll
            for (int q = 0; q < W; ++q) xs[q] = *reinterpret_cast<const v4f *>(&ring[sb[q] + xo]);
#pragma unroll
            for (int c = 0; c < C; ++c) accx = __builtin_amdgcn_mfma_f32_16x16x4f32(tv[c], xs[c / 4][c % 4], accx, 0, 0, 0);
        }
        // a piece of a pitched row may hold columns beyond the row
        if (xs0 + 15 >= nx && xs0 + col >= nx) accy = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int e = 0; e < 4; ++e) ring[wgrp * S::GRP + yw[e]] = accy[e];
        if (p >= 0) {
            const uint32_t m = mring[(i & 1) * 64 + 16 * rt + col] >> (16 * u + 4 * kg);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if ((m >> e) & 1u) accx[e] = 1.0f;
            const int xp = xa + 32 * p;
            if (xp + 32 <= xb) {  // uniform; only a row's last pair is partial
                if constexpr (OUTF) store16_any(y_ok ? out_f32 + off : sinkf, accx);
                if constexpr (OUTU) {
                    const v2u32 w = {(uint32_t)quantise_u16_l(accx[0]) | ((uint32_t)quantise_u16_l(accx[1]) << 16),
                                     (uint32_t)quantise_u16_l(accx[2]) | ((uint32_t)quantise_u16_l(accx[3]) << 16)};
                    *(__attribute__((address_space(1))) v2u32_a2 *)(y_ok ? out_u16 + off : sinku) = w;
                }
            } else if (y_ok) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (xp + 16 * u + 4 * kg + e >= xb) break;
                    if constexpr (OUTF) gmem(out_f32)[off + e] = accx[e];
                    if constexpr (OUTU) gmem(out_u16)[off + e] = quantise_u16_l(accx[e]);
                }
            }
            off += 32;
        }
        wgrp = wgrp == G - 1 ? 0 : wgrp + 1;
    }
    vm_wait<0>();
}

}  // namespace mxb
