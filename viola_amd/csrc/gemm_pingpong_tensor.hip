// Per-tensor-scale instances of the large-tile FP8 GEMM kernel.
#include "gemm_pingpong.hpp"

namespace viola {

int launch_tensor_pingpong(const GemmArgs& p, ScaledTile tile, bool gated, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, hipStream_t stream) {
    return launch_pingpong_tile<false>(p, tile, gated, a_dtype, b_dtype, bias_dtype, out_dtype, stream);
}

}  // namespace viola
