// FP32 line pass, LDS-staged forms: single-volume kernels and launcher (the
// per-block bodies live in mxb_lds_body.h and mxb_f32_dma_body.h).
#include <algorithm>

#include "mxb_f32_dma_body.h"

namespace mxb {

template <int RT>
__global__ __launch_bounds__(256) void k_line_mfma_lds(const float *__restrict__ in, LineGeom g,
                                                       Epilogue e, TapsF<2 * RT + 1> taps) {
    __shared__ float smem[LdsSmem<RT>::TOTAL];
    lds_fill_taps<RT>(smem, taps.k);
    int64_t bid = blockIdx.x;
    const int64_t seg_id = bid % g.nseg;
    bid /= g.nseg;
    const int64_t nlb = (g.n_lane + 63) >> 6;
    const int64_t lb = bid % nlb;
    const int64_t outer = bid / nlb;
    lds_line_body<RT>(in, g, e, outer, lb, seg_id, smem);
}

template <int RT, int D, bool MASK, bool OUTF, bool OUTU, bool ZSTAGE, bool ANY>
__global__ __launch_bounds__(256) void k_line_f32_dma(const float *__restrict__ in, LineGeom g,
                                                      Epilogue e, TapsF<2 * RT + 1> taps) {
    __shared__ __attribute__((aligned(16))) unsigned char smem[F32DmaForm<RT, D, MASK, ZSTAGE>::BYTES];
    int64_t bid = xcd_tile(blockIdx.x, gridDim.x);
    const int64_t seg_id = bid % g.nseg;
    bid /= g.nseg;
    const int64_t nlb = (g.n_lane + 63) >> 6;
    const int64_t lb = bid % nlb;
    const int64_t outer = bid / nlb;
    f32_dma_pass<RT, D, MASK, OUTF, OUTU, ZSTAGE, ANY>(in, g, e, outer, lb, seg_id, taps.k, smem);
}

// Which direct-load epilogue serves (g, e): 0 none, else a code for the
// template below.  `any`: the form with 4-byte loads, which takes any rows and
// any number of lines from 64 on; else 16-byte loads and stores.
static int f32_dma_form(const float *in, const LineGeom &g, const Epilogue &e, bool any) {
    if (any) {
        const bool f = e.out_f32 != nullptr, u = e.out_u16 != nullptr, m = e.mask != nullptr;
        if (g.n_lane < 64) return 0;
        if (g.out_lane == 1 && !m && !u && f) return 1;
        if (g.out_ax != 1 || (m && e.bits.w == nullptr)) return 0;
        return 2 + (m ? 4 : 0) + (f ? 1 : 0) + (u ? 2 : 0);
    }
    if (g.in_outer % 4 != 0 || g.in_ax % 4 != 0 || reinterpret_cast<uintptr_t>(in) % 16 != 0) return 0;
    if (g.n_lane % 4 != 0) return 0;
    const bool f = e.out_f32 != nullptr, u = e.out_u16 != nullptr, m = e.mask != nullptr;
    if (f && reinterpret_cast<uintptr_t>(e.out_f32) % 16 != 0) return 0;
    if (u && reinterpret_cast<uintptr_t>(e.out_u16) % 16 != 0) return 0;
    if (g.out_lane == 1 && !m && !u && f && g.out_outer % 4 == 0 && g.out_ax % 4 == 0) return 1;
    if (g.out_ax != 1 || g.out_lane % 8 != 0 || g.out_outer % 8 != 0) return 0;
    if (m && e.bits.w == nullptr) return 0;  // the direct-load illuminating pass reads mask bits
    return 2 + (m ? 4 : 0) + (f ? 1 : 0) + (u ? 2 : 0);
}

template <int RT, bool ANY>
static hipError_t launch_f32_dma_rt(int form, const float *in, LineGeom g, const Epilogue &e,
                                    const TapsF<2 * RT + 1> &t, hipStream_t s) {
    constexpr int D = MXB_F32_DMA_DEPTH;
    const dim3 grid((unsigned)(g.nseg * ((g.n_lane + 63) / 64) * g.n_outer)), block(256);
    switch (form) {
    case 1: hipLaunchKernelGGL((k_line_f32_dma<RT, D, false, true, false, true, ANY>), grid, block, 0, s, in, g, e, t); break;
    case 3: hipLaunchKernelGGL((k_line_f32_dma<RT, D, false, true, false, false, ANY>), grid, block, 0, s, in, g, e, t); break;
    case 4: hipLaunchKernelGGL((k_line_f32_dma<RT, D, false, false, true, false, ANY>), grid, block, 0, s, in, g, e, t); break;
    case 5: hipLaunchKernelGGL((k_line_f32_dma<RT, D, false, true, true, false, ANY>), grid, block, 0, s, in, g, e, t); break;
    case 7: hipLaunchKernelGGL((k_line_f32_dma<RT, D, true, true, false, false, ANY>), grid, block, 0, s, in, g, e, t); break;
    case 8: hipLaunchKernelGGL((k_line_f32_dma<RT, D, true, false, true, false, ANY>), grid, block, 0, s, in, g, e, t); break;
    case 9: hipLaunchKernelGGL((k_line_f32_dma<RT, D, true, true, true, false, ANY>), grid, block, 0, s, in, g, e, t); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

static bool rows_aligned(const float *in, const LineGeom &g) {
    return g.in_outer % 4 == 0 && g.in_ax % 4 == 0 && reinterpret_cast<uintptr_t>(in) % 16 == 0;
}

template <int RT>
static TapsF<2 * RT + 1> centred_taps_l(const float *k, int R) {
    TapsF<2 * RT + 1> t;
    for (int i = 0; i < 2 * RT + 1; ++i) {
        const int r = i - RT;
        t.k[i] = (r >= -R && r <= R) ? k[R + r] : 0.0f;
    }
    return t;
}

template <int RT>
static hipError_t launch_lds_rt(const float *in, LineGeom g, const Epilogue &e, const float *k,
                                int R, hipStream_t s) {
    // one block per (segment, 64 lines, outer); segments keep >= ~16 waves/CU
    const int64_t groups = ((g.n_lane + 63) / 64) * g.n_outer;
    const int64_t target = 256LL * 6;
    int64_t nseg = groups > 0 ? (target + groups - 1) / groups : 1;
    const int64_t q = e.mask != nullptr ? 32 : 16;  // the illuminating pass: whole mask-bit words
    // Segments of at least 64 positions, whose halo costs little; where single
    // tiles leave fewer than four blocks a CU, and no more than its LDS holds at
    // once, a pass is its blocks' own latency, and the shortest segments win
    // (64^3, sigma 3 / 10, ten repetitions: 140 -> 125 / 176 -> 130 us, 96^3
    // sigma 3 186 -> 176; at 128^3, four blocks a CU, 244 -> 246; 100x24x300
    // sigma 16, four blocks a CU of which two fit, 195 -> 237).
    constexpr int D = MXB_F32_DMA_DEPTH;
    const int bytes = e.mask != nullptr ? F32DmaForm<RT, D, true, false>::BYTES
                      : g.out_lane == 1 ? F32DmaForm<RT, D, false, true>::BYTES
                                        : F32DmaForm<RT, D, false, false>::BYTES;
    const int64_t max_tiles = (g.n_ax + q - 1) / q, at_once = 256 * std::min(4, 160 * 1024 / bytes);
    const int64_t max_seg = groups * max_tiles < at_once ? max_tiles : (g.n_ax + 63) / 64;
    if (nseg > max_seg) nseg = max_seg;
    if (nseg < 1) nseg = 1;
    int64_t seg = (g.n_ax + nseg - 1) / nseg;
    seg = ((seg + q - 1) / q) * q;
    g.seg = seg;
    g.nseg = (g.n_ax + seg - 1) / seg;
    g.vec_out = (g.out_ax == 1 && g.out_lane % 4 == 0 && g.out_outer % 4 == 0 &&
                 (e.out_f32 == nullptr || reinterpret_cast<uintptr_t>(e.out_f32) % 16 == 0) &&
                 (e.out_u16 == nullptr || reinterpret_cast<uintptr_t>(e.out_u16) % 8 == 0) &&
                 (e.mask == nullptr || reinterpret_cast<uintptr_t>(e.mask) % 4 == 0)) ? 1 : 0;
    g.stage_out = (g.out_lane == 1 && g.out_outer % 4 == 0 && g.out_ax % 4 == 0 &&
                   e.mask == nullptr && e.out_u16 == nullptr && e.out_f32 != nullptr &&
                   reinterpret_cast<uintptr_t>(e.out_f32) % 16 == 0) ? 1 : 0;
    const int64_t blocks = g.nseg * groups;
    if (blocks == 0) return hipSuccess;
    const TapsF<2 * RT + 1> t = centred_taps_l<RT>(k, R);
    if (!force_vgpr_staging()) {
        if (const int form = f32_dma_form(in, g, e, false)) return launch_f32_dma_rt<RT, false>(form, in, g, e, t, s);
        // lines too short for the loads to matter take the VGPR-staged form where
        // their rows allow it (y-pass of 1000x4x600 sigma 16 122 -> 73 us, ten
        // passes of 400x44x404 2 to 8 % faster; 400x76x404 2 to 14 % slower)
        const bool staged = rows_aligned(in, g) && g.n_ax < 64;
        if (const int form = staged ? 0 : f32_dma_form(in, g, e, true))
            return launch_f32_dma_rt<RT, true>(form, in, g, e, t, s);
    }
    if (!rows_aligned(in, g)) return hipErrorNotSupported;
    hipLaunchKernelGGL((k_line_mfma_lds<RT>), dim3((unsigned)blocks), dim3(256), 0, s, in, g, e, t);
    return hipGetLastError();
}

// Usable when the radius is compiled and either every input row is 16-byte
// aligned or the direct-load form with 4-byte loads serves.
bool lds_pass_supported(const float *in, const LineGeom &g, const Epilogue &e, int R) {
    return R <= 64 && (rows_aligned(in, g) || (!force_vgpr_staging() && f32_dma_form(in, g, e, true) != 0));
}

hipError_t launch_line_pass_f32_lds(const float *in, const LineGeom &g, const Epilogue &e,
                                    const float *taps, int R, hipStream_t s) {
#define MXB_LDS_CASE(rt) \
    if (R <= rt) return launch_lds_rt<rt>(in, g, e, taps, R, s);
    MXB_LDS_CASE(4)
    MXB_LDS_CASE(8)
    MXB_LDS_CASE(12)
    MXB_LDS_CASE(16)
    MXB_LDS_CASE(20)
    MXB_LDS_CASE(24)
    MXB_LDS_CASE(32)
    MXB_LDS_CASE(40)
    MXB_LDS_CASE(48)
    MXB_LDS_CASE(56)
    MXB_LDS_CASE(64)
#undef MXB_LDS_CASE
    return hipErrorInvalidValue;
}

}  // namespace mxb
