// Grouped FP32-scale instances of the large-tile FP8 GEMM kernel.
#include "gemm_pingpong_grouped.hpp"

namespace viola {

template <typename S, bool ROWS>
static int launch(const GemmArgs& args, int row_tiles, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, unsigned groups, hipStream_t stream) {
    GemmArgs p = args;
    p.tiles_m = row_tiles;
    p.tiles_n = (int)((p.n + S::COLS - 1) / S::COLS);
    const int64_t blocks = (int64_t)p.tiles_m * p.tiles_n * (p.k_split ? p.parts : 1);
    const dim3 grid((unsigned)((blocks + 7) / 8 * 8), 1, groups), block(512);
    const bool a5 = a_dtype == VIOLA_E5M2, b5 = b_dtype == VIOLA_E5M2;
    if (!a5 && !b5) VIOLA_LAUNCH((gemm_pingpong_grouped<false, false, S, ROWS>), grid, block, 0, stream, p, bias_dtype, out_dtype);
    else if (a5 && !b5) VIOLA_LAUNCH((gemm_pingpong_grouped<true, false, S, ROWS>), grid, block, 0, stream, p, bias_dtype, out_dtype);
    else if (!a5 && b5) VIOLA_LAUNCH((gemm_pingpong_grouped<false, true, S, ROWS>), grid, block, 0, stream, p, bias_dtype, out_dtype);
    else VIOLA_LAUNCH((gemm_pingpong_grouped<true, true, S, ROWS>), grid, block, 0, stream, p, bias_dtype, out_dtype);
    return viola_launch_status();
}

static int launch_rounds(const GemmArgs& args, int row_tiles, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, hipStream_t stream) {
    GemmArgs p = args;
    p.tiles_m = row_tiles;
    p.tiles_n = (int)((p.n + GroupedWide::COLS - 1) / GroupedWide::COLS);
    // (variable groups: row_tiles is a bound; whatever the number of tiles turns out to be, their blocks are among these)
    const int64_t blocks = (int64_t)p.tiles_m * p.tiles_n + 256;
    const dim3 grid((unsigned)((blocks + 7) / 8 * 8)), block(512);
    const bool a5 = a_dtype == VIOLA_E5M2, b5 = b_dtype == VIOLA_E5M2;
    if (!a5 && !b5) VIOLA_LAUNCH((gemm_pingpong_grouped_rounds<false, false, GroupedWide, GroupedTall, GroupedQuarter>), grid, block, 0, stream, p, bias_dtype, out_dtype);
    else if (a5 && !b5) VIOLA_LAUNCH((gemm_pingpong_grouped_rounds<true, false, GroupedWide, GroupedTall, GroupedQuarter>), grid, block, 0, stream, p, bias_dtype, out_dtype);
    else if (!a5 && b5) VIOLA_LAUNCH((gemm_pingpong_grouped_rounds<false, true, GroupedWide, GroupedTall, GroupedQuarter>), grid, block, 0, stream, p, bias_dtype, out_dtype);
    else VIOLA_LAUNCH((gemm_pingpong_grouped_rounds<true, true, GroupedWide, GroupedTall, GroupedQuarter>), grid, block, 0, stream, p, bias_dtype, out_dtype);
    return viola_launch_status();
}

// out = sum of the parts, in ascending order. A thread owns eight consecutive values: 32 bytes of every part in flight at once.
// Bound by the read of the partial products, which the kernel before has just written: most of them are still in the last-level
// cache (3072 x 768 in three parts: 7.1 us for 33 MB).
template <typename TO>
__global__ __launch_bounds__(256) void sum_parts(const float* partial, int parts, int64_t stride, int64_t count, TO* out) {
    const int64_t at = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
    if (at >= count) return;
    if (at + 8 > count) {
        for (int64_t e = at; e < count; ++e) {
            float v = partial[e];
            for (int s = 1; s < parts; ++s) v += partial[s * stride + e];
            out[e] = from_f32<TO>(v);
        }
        return;
    }
    float v[8] = {};
#pragma unroll 4
    for (int s = 0; s < parts; ++s) {
        const float4 x = *reinterpret_cast<const float4*>(partial + s * stride + at), y = *reinterpret_cast<const float4*>(partial + s * stride + at + 4);
        v[0] += x.x; v[1] += x.y; v[2] += x.z; v[3] += x.w;
        v[4] += y.x; v[5] += y.y; v[6] += y.z; v[7] += y.w;
    }
    if ((reinterpret_cast<uintptr_t>(out) & 15) == 0) {
        Quad<TO>::store(out + at, {v[0], v[1], v[2], v[3]});
        Quad<TO>::store(out + at + 4, {v[4], v[5], v[6], v[7]});
    } else {
        for (int e = 0; e < 8; ++e) out[at + e] = from_f32<TO>(v[e]);
    }
}

int launch_group_parts(const GemmArgs& args, int parts, int a_dtype, int b_dtype, int out_dtype, float* workspace, hipStream_t stream) {
    GemmArgs p = args;
    const int64_t count = p.m * p.n;
    p.out = workspace;
    p.out_group_stride = (count + 3) / 4 * 4;
    // Whole chunks; the last part may be shorter. Cut as the k range padded to whole 128 is, which the native host path gives its
    // operands, so that the same values without the padding (the Python operators') are added in the same order.
    p.k_split = ((p.k + 127) / 128 * 128 + parts - 1) / parts;
    p.k_split = (p.k_split + FBK - 1) / FBK * FBK;
    p.parts = parts = (int)((p.k + p.k_split - 1) / p.k_split);
    const int status = launch<GroupedRows, true>(p, (int)((p.m + GroupedRows::ROWS - 1) / GroupedRows::ROWS), a_dtype, b_dtype, VIOLA_F32, VIOLA_F32, 1, stream);
    if (status) return status;
    const dim3 grid((unsigned)((count + 2047) / 2048)), block(256);
    if (out_dtype == VIOLA_F32) VIOLA_LAUNCH(sum_parts<float>, grid, block, 0, stream, workspace, parts, p.out_group_stride, count, static_cast<float*>(args.out));
    else if (out_dtype == VIOLA_BF16) VIOLA_LAUNCH(sum_parts<bf16_t>, grid, block, 0, stream, workspace, parts, p.out_group_stride, count, static_cast<bf16_t*>(args.out));
    else VIOLA_LAUNCH(sum_parts<f16_t>, grid, block, 0, stream, workspace, parts, p.out_group_stride, count, static_cast<f16_t*>(args.out));
    return viola_launch_status();
}

int launch_group_pingpong(const GemmArgs& p, int row_tiles, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, bool rowscale,
                          unsigned groups, hipStream_t stream) {
    return rowscale ? launch<GroupedRows, true>(p, row_tiles, a_dtype, b_dtype, bias_dtype, out_dtype, groups, stream)
                    : launch_rounds(p, row_tiles, a_dtype, b_dtype, bias_dtype, out_dtype, stream);
}

int launch_group_tall(const GemmArgs& p, int row_tiles, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, hipStream_t stream) {
    return launch<GroupedTall, false>(p, row_tiles, a_dtype, b_dtype, bias_dtype, out_dtype, 1, stream);
}

int launch_group_teams(const GemmArgs& p, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, hipStream_t stream) {
    return launch<GroupedTeams, true>(p, (int)((p.m + GroupedTeams::ROWS - 1) / GroupedTeams::ROWS), a_dtype, b_dtype, bias_dtype, out_dtype, 1, stream);
}

}  // namespace viola
