// Grouped FP32-scale instances of the large-tile FP8 GEMM kernel.
#include "gemm_pingpong_grouped.hpp"

namespace viola {

template <bool ROWS>
static int launch(const GemmArgs& args, int row_tiles, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, unsigned groups, hipStream_t stream) {
    using S = std::conditional_t<ROWS, GroupedRows, GroupedWide>;
    GemmArgs p = args;
    p.tiles_m = row_tiles;
    p.tiles_n = (int)((p.n + S::COLS - 1) / S::COLS);
    const dim3 grid((unsigned)(((int64_t)p.tiles_m * p.tiles_n + 7) / 8 * 8), 1, groups), block(512);
    const bool a5 = a_dtype == VIOLA_E5M2, b5 = b_dtype == VIOLA_E5M2;
    if (!a5 && !b5) VIOLA_LAUNCH((gemm_pingpong_grouped<false, false, ROWS>), grid, block, 0, stream, p, bias_dtype, out_dtype);
    else if (a5 && !b5) VIOLA_LAUNCH((gemm_pingpong_grouped<true, false, ROWS>), grid, block, 0, stream, p, bias_dtype, out_dtype);
    else if (!a5 && b5) VIOLA_LAUNCH((gemm_pingpong_grouped<false, true, ROWS>), grid, block, 0, stream, p, bias_dtype, out_dtype);
    else VIOLA_LAUNCH((gemm_pingpong_grouped<true, true, ROWS>), grid, block, 0, stream, p, bias_dtype, out_dtype);
    return viola_launch_status();
}

int launch_group_pingpong(const GemmArgs& p, int row_tiles, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, bool rowscale,
                          unsigned groups, hipStream_t stream) {
    return rowscale ? launch<true>(p, row_tiles, a_dtype, b_dtype, bias_dtype, out_dtype, groups, stream)
                    : launch<false>(p, row_tiles, a_dtype, b_dtype, bias_dtype, out_dtype, groups, stream);
}

}  // namespace viola
