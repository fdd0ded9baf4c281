// Launchers of the fast FP8 GEMM kernel for the recipes whose scales need no per-group fold: per-tensor scales and
// E8M0 block scales. Included by the one file that instantiates each.
#pragma once
#include "gemm_fast_kernel.hpp"

namespace viola {

// Per-tensor scales (TENSOR: args.sa / args.sb point at one float each) or E8M0 block scales (MX: they point at
// bytes; ldsa / ldsb = bytes per scale row). grid: (n tiles, m tiles of 128); n tiles are 128 wide, 64 for gated forward.
// KSPLIT: the k range of a 128 x 64 tile split over two teams of waves in a 512-thread block (plain mode)
template <int MODE, typename TO, int TN, bool TENSOR, bool MX, bool KSPLIT = false>
static void launch_scaled_formats(const GemmArgs& p, int a_dtype, int b_dtype, int bias_dtype, dim3 grid, hipStream_t stream) {
    const bool a5 = a_dtype == VIOLA_E5M2, b5 = b_dtype == VIOLA_E5M2;
    const dim3 block(KSPLIT ? 2 * FTHREADS : FTHREADS);
    if (!a5 && !b5) VIOLA_LAUNCH((group_gemm_fast<MODE, false, false, false, TO, TN, TENSOR, MX, KSPLIT>), grid, block, 0, stream, p, bias_dtype);
    else if (a5 && !b5) VIOLA_LAUNCH((group_gemm_fast<MODE, true, false, false, TO, TN, TENSOR, MX, KSPLIT>), grid, block, 0, stream, p, bias_dtype);
    else if (!a5 && b5) VIOLA_LAUNCH((group_gemm_fast<MODE, false, true, false, TO, TN, TENSOR, MX, KSPLIT>), grid, block, 0, stream, p, bias_dtype);
    else VIOLA_LAUNCH((group_gemm_fast<MODE, true, true, false, TO, TN, TENSOR, MX, KSPLIT>), grid, block, 0, stream, p, bias_dtype);
}

// shortest k range that the narrow tiles split
constexpr int64_t SCALED_SPLIT_MIN_K = 2048;

template <bool TENSOR, bool MX>
static int launch_scaled_gemm_fast(const GemmArgs& args, int mode, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, dim3 grid,
                                   hipStream_t stream) {
    GemmArgs p = args;
    {
        // MX: the scale arrays hold bytes; per-tensor scales are read directly, not through these descriptors
        const int64_t b_rows = mode == MODE_GATED_FWD ? 2 * p.n : p.n;
        p.sa_bytes = (p.m + p.ar - 1) / p.ar * p.ldsa;
        p.sb_bytes = (b_rows + p.br - 1) / p.br * p.ldsb;
    }
    // a gated forward that keeps no [g | u] takes the large tile where the plain product would (with [g | u] kept it is that product
    // and a pass over it)
    const ScaledTile tile = mode == MODE_PLAIN ? choose_scaled_tile(p.m, p.n, p.k)
                            : mode == MODE_GATED_FWD && !p.aux && !p.enc ? choose_scaled_tile(p.m, 2 * p.n, p.k, false) : SCALED_TILE_FAST;
    if (mode == MODE_PLAIN ? tile != SCALED_TILE_FAST : tile == SCALED_TILE_L)
        return (MX ? launch_mx_pingpong : launch_tensor_pingpong)(p, tile, mode != MODE_PLAIN, a_dtype, b_dtype, bias_dtype, out_dtype, stream);
    // fewer than 128 tiles of 128 x 128 (from 128 up choose_scaled_tile finds an alternating-phase tile): halve the tile in n to
    // keep more CUs busy, and over a long k split its k range inside the block (the grouped recipe's rule)
    const bool narrow = mode == MODE_PLAIN && (int64_t)grid.x * grid.y < 128 && p.n > 64;
    const bool split = narrow && p.k >= SCALED_SPLIT_MIN_K;
    if (narrow) grid.x = (unsigned)((p.n + 63) / 64);
    if ((int64_t)grid.x * grid.y < (1 << 30)) {
        p.tiles_n = (int)grid.x;
        p.tiles_m = (int)grid.y;
        grid = dim3((grid.x * grid.y + 7) / 8 * 8, 1, 1);
    }
#define VIOLA_SCALED(TO)                                                                                                        \
    if (split) launch_scaled_formats<MODE_PLAIN, TO, 1, TENSOR, MX, true>(p, a_dtype, b_dtype, bias_dtype, grid, stream);        \
    else if (narrow) launch_scaled_formats<MODE_PLAIN, TO, 1, TENSOR, MX>(p, a_dtype, b_dtype, bias_dtype, grid, stream);        \
    else if (mode == MODE_PLAIN) launch_scaled_formats<MODE_PLAIN, TO, 2, TENSOR, MX>(p, a_dtype, b_dtype, bias_dtype, grid, stream); \
    else if (mode == MODE_GATED_FWD) launch_scaled_formats<MODE_GATED_FWD, TO, 2, TENSOR, MX>(p, a_dtype, b_dtype, bias_dtype, grid, stream); \
    else launch_scaled_formats<MODE_GATED_BWD, TO, 2, TENSOR, MX>(p, a_dtype, b_dtype, bias_dtype, grid, stream);
    switch (out_dtype) {
        case VIOLA_F32: VIOLA_SCALED(float) break;
        case VIOLA_BF16: VIOLA_SCALED(bf16_t) break;
        case VIOLA_F16: VIOLA_SCALED(f16_t) break;
        default: return VIOLA_EINVAL;
    }
#undef VIOLA_SCALED
    return viola_launch_status();
}

}  // namespace viola
