// Fused y -> x pass of the FP32 form on one volume (gfx950): the kernel around
// f32_yx_body (mxb_f32_yx_body.h) and its launch.
#include "mxb_f32_yx_body.h"

namespace mxb {

struct YXTiles {
    int64_t nyt;        // row tiles of 64
    int64_t seg, nseg;  // columns per block (a multiple of 32), blocks along x
};

template <int RT, bool OUTF, bool OUTU, bool ANY>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2 * YXShape<RT>::BLOCKS))) void k_yx_f32(
    const float *__restrict__ in, float *__restrict__ out_f32, uint16_t *__restrict__ out_u16,
    const uint32_t *__restrict__ bits, YXGeom g, YXTiles t, TapsF<2 * RT + 1> taps) {
    __shared__ __attribute__((aligned(16))) float smem[YXShape<RT>::BYTES / 4];
    int64_t tile = xcd_tile(blockIdx.x, gridDim.x);
    const int64_t yt = tile % t.nyt;
    tile /= t.nyt;
    const int xa = (int)(tile % t.nseg * t.seg);
    const int xb = xa + t.seg < g.nx ? xa + (int)t.seg : (int)g.nx;
    f32_yx_body<RT, OUTF, OUTU, ANY>(in, out_f32, out_u16, bits, g, tile / t.nseg, 64 * (int)yt, xa, xb, taps.k, smem);
}

// ---------------------------------------------------------------- host side
static bool yx_any(const float *in, int64_t nx) { return nx % 4 != 0 || reinterpret_cast<uintptr_t>(in) % 16 != 0; }

// Whole rows per block unless that leaves CUs idle (each segment repeats the
// y-pass of L groups), down to single pairs where every block has a CU of its own.
static YXTiles yx_tiles(int64_t nz, int64_t ny, int64_t nx) {
    YXTiles t;
    t.nyt = (ny + 63) / 64;
    const int64_t rows = nz * t.nyt;
    int64_t nseg = (256 * 2 + rows - 1) / rows;
    const int64_t max_pairs = (nx + 31) / 32;
    const int64_t max_seg = rows * max_pairs <= 256 ? max_pairs : (nx + 127) / 128;
    if (nseg > max_seg) nseg = max_seg;
    if (nseg < 1) nseg = 1;
    t.seg = ((nx + nseg - 1) / nseg + 31) / 32 * 32;
    t.nseg = (nx + t.seg - 1) / t.seg;
    return t;
}

// Whether the fused pass serves, and is the faster form: always up to R = 40.
// Above, one block fills a CU's LDS and the halo costs more, so volumes whose
// separate passes have whole 16-byte rows take it only while they are few
// blocks (sigma 12 / 15, four repetitions: 256^3 569 -> 535 / 637 -> 608 us, but
// 512^3 3536 -> 3710 / 4457 -> 4551) and little is idle: of the last round of
// blocks, one to a CU, and of the tiles' 64 rows (five repetitions of sigma 12:
// 257x4x600 314 us apart, 421 fused, 400x96x400 968 and 1081); narrow volumes,
// where the separate passes idle too, bear more (257x100x96 sigma 16 344 and
// 281).  Other rows always (301x401x501 2264 -> 2158 / 2567 -> 2429).
bool yx_f32_supported(const float *in, const MaskBits &bits, int64_t nz, int64_t ny, int64_t nx, int R) {
    if (R > 64 || nz * ny * nx == 0) return false;
    // bits as packed for whole volumes (a plane's words interleaved across y)
    if (bits.w == nullptr || bits.lane != 1) return false;
    // byte offsets of rows up to 512 before or after a plane stay below the
    // offset that means "outside"
    if ((ny + 512) * nx >= (int64_t(1) << 28) || reinterpret_cast<uintptr_t>(in) % 4 != 0) return false;
    if (R <= 40 || yx_any(in, nx)) return true;
    const YXTiles t = yx_tiles(nz, ny, nx);
    if (nz * t.nyt > 4 * 256) return false;
    const int64_t blocks = nz * t.nyt * t.nseg, rounds = (blocks + 255) / 256;
    const double busy = (double)blocks / (double)(256 * rounds) * (double)ny / (double)(64 * t.nyt);
    return busy * (1.0 + 300.0 / (double)nx) >= 0.6;
}

template <int RT, bool ANY>
static hipError_t launch_yx_rt(const float *in, float *out_f32, uint16_t *out_u16, const MaskBits &bits, int64_t nz,
                               int64_t ny, int64_t nx, const float *k, int R, hipStream_t s) {
    TapsF<2 * RT + 1> t;
    for (int i = 0; i < 2 * RT + 1; ++i) {
        const int r = i - RT;
        t.k[i] = (r >= -R && r <= R) ? k[R + r] : 0.0f;
    }
    const YXGeom g{ny, nx, nx, ny * nx, bits.outer, bits.word};
    const YXTiles tiles = yx_tiles(nz, ny, nx);
    const dim3 grid((unsigned)(nz * tiles.nyt * tiles.nseg)), block(512);
    if (out_f32 != nullptr && out_u16 != nullptr)
        hipLaunchKernelGGL((k_yx_f32<RT, true, true, ANY>), grid, block, 0, s, in, out_f32, out_u16, bits.w, g, tiles, t);
    else if (out_f32 != nullptr)
        hipLaunchKernelGGL((k_yx_f32<RT, true, false, ANY>), grid, block, 0, s, in, out_f32, out_u16, bits.w, g, tiles, t);
    else if (out_u16 != nullptr)
        hipLaunchKernelGGL((k_yx_f32<RT, false, true, ANY>), grid, block, 0, s, in, out_f32, out_u16, bits.w, g, tiles, t);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_yx_f32(const float *in, float *out_f32, uint16_t *out_u16, const MaskBits &bits, int64_t nz,
                         int64_t ny, int64_t nx, const float *taps, int R, hipStream_t s) {
    if (!yx_f32_supported(in, bits, nz, ny, nx, R)) return hipErrorInvalidValue;
    const bool any = yx_any(in, nx);
#define MXB_YX_CASE(rt)                                                                              \
    if (R <= rt)                                                                                     \
        return any ? launch_yx_rt<rt, true>(in, out_f32, out_u16, bits, nz, ny, nx, taps, R, s)      \
                   : launch_yx_rt<rt, false>(in, out_f32, out_u16, bits, nz, ny, nx, taps, R, s);
    MXB_YX_CASE(4)
    MXB_YX_CASE(8)
    MXB_YX_CASE(12)
    MXB_YX_CASE(16)
    MXB_YX_CASE(20)
    MXB_YX_CASE(24)
    MXB_YX_CASE(32)
    MXB_YX_CASE(40)
    MXB_YX_CASE(48)
    MXB_YX_CASE(56)
    MXB_YX_CASE(64)
#undef MXB_YX_CASE
    return hipErrorInvalidValue;
}

}  // namespace mxb
