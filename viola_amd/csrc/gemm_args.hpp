// Shared between the generic and the fast grouped-scale FP8 GEMM translation units.
#pragma once
#include "common.hpp"

namespace viola {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int BM = 128, BN = 128;                                 // output tile of both kernels
enum { MODE_PLAIN = 0, MODE_GATED_FWD = 1, MODE_GATED_BWD = 2 };

struct GemmArgs {
    const uint8_t* a; const uint8_t* b; const float* sa; const float* sb;
    const void* bias; void* out; void* aux;
    int64_t m, n, k;              // n: rows of one b panel (h for the gated modes)
    int64_t lda, ldb;             // bytes between rows of a / b
    int64_t ldsa, ldsb;           // floats between rows of sa / sb
    int64_t ldo;                  // elements between rows of out
    int ar, br, ak_shift, bk_shift;
    int activation;
    // variable-group row ranges (grid.y walks the tiles of all groups)
    const int64_t* offsets; int groups; int64_t b_group_stride, sb_group_stride;
    // variable-group K ranges (grid.z = group): k range [koffsets[g], koffsets[g+1])
    const int64_t* koffsets; int64_t out_group_stride;
    // the same with `parts` equal ranges of k_split (0: none; large tiles only), the parts' tiles one after the other in grid.x
    int64_t k_split; int parts;
    // fast kernel only: 1-D grid of tiles_m * tiles_n output tiles (rounded up to a multiple of 8) walked in an
    // XCD-aware order; tiles_m == 0 keeps the plain (blockIdx.x, blockIdx.y) = (n tile, m tile) mapping
    int tiles_m, tiles_n;
    // fast kernel only, filled in by its launchers: bytes of the two scale arrays (a 16-byte piece may reach past the
    // last scale row and must then read zero, so their buffer descriptors carry the true size)
    int64_t sa_bytes, sb_bytes;
    // MX gated forward only: when enc is set, h is not written to out but quantized in the epilogue with E8M0
    // scales per 32 values, along its rows (enc [m, n], enc_scale [m, n / 32]) and along its columns
    // (enc_t [n, m], enc_t_scale [n, m / 32]; enc_t may be null); m and n are multiples of 32
    uint8_t* enc; uint8_t* enc_scale; uint8_t* enc_t; uint8_t* enc_t_scale; float enc_limit; int enc_bf8;
    // FP16-accumulator model of the generic kernel (HALF != 0): k covered by one FP16 partial sum before it is added to
    // the running total (0: the whole k range, no separate total), and whether that total is kept in bf16
    int half_period; int reduce_bf16;
};


// Any alignment and size; the FP16-accumulator model (per_tensor: scales applied to the finished total). gemm_generic.hip.
int launch_group_gemm_generic(const GemmArgs& p, int mode, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, bool rowscale, dim3 grid,
                              hipStream_t stream);
int launch_group_gemm_half(const GemmArgs& p, bool per_tensor, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, bool rowscale, dim3 grid,
                           hipStream_t stream);

// Fast path (16-byte aligned operands, k ranges multiples of 16). Defined in gemm_fast.hip.
int launch_group_gemm_fast(const GemmArgs& p, int mode, int a_dtype, int b_dtype, int bias_dtype, int out_dtype,
                           bool rowscale, dim3 grid, hipStream_t stream);

// Which form a plain product under the grouped recipe runs in (the values are viola_group_gemm_form's): the blocks of group_gemm_fast
// of 128 x 128 or 128 x 64, their k range split over two teams or not, or one of the three forms below. gemm_fast.hip.
enum GroupForm { GROUP_BLOCKS = 0, GROUP_BLOCKS_SPLIT, GROUP_NARROW, GROUP_NARROW_SPLIT, GROUP_LARGE, GROUP_TALL, GROUP_TEAMS };
GroupForm group_form(const GemmArgs& p, bool rowscale, dim3 grid);

// The grouped recipe on tiles of 256 x 256, a last round of few on narrower ones (row-wise b scales: 256 x 128); row_tiles: tiles of 256 rows (variable groups: a bound on
// them), groups: k ranges (row-wise b scales only). gemm_pingpong_grouped.hip.
int launch_group_pingpong(const GemmArgs& p, int row_tiles, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, bool rowscale, unsigned groups,
                          hipStream_t stream);

// Uniform b scales on one round of 256 x 128 tiles. gemm_pingpong_grouped.hip.
int launch_group_tall(const GemmArgs& p, int row_tiles, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, hipStream_t stream);

// Row-wise b scales on tiles of 128 x 128, the k range split over two teams of waves that take turns. gemm_pingpong_grouped.hip.
int launch_group_teams(const GemmArgs& p, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, hipStream_t stream);

// How many parts of k a row-wise scaled product is computed in (1: whole), and the product in that many: FP32 partial products
// [parts][m * n rounded up to 4] in workspace, then their sum in ascending order. gemm_fast.hip, gemm_pingpong_grouped.hip.
int plan_k_parts(int64_t m, int64_t n, int64_t k);
int launch_group_parts(const GemmArgs& p, int parts, int a_dtype, int b_dtype, int out_dtype, float* workspace, hipStream_t stream);

// Per-tensor scales on the same fast kernel (one v_mfma_f32_32x32x64_f8f6f4 per sub-tile and 64 k); mode = MODE_PLAIN or a
// gated mode (grid.x then counts the gated tile width). Defined in gemm_fast.hip.
int launch_tensor_gemm_fast(const GemmArgs& p, int mode, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, dim3 grid,
                            hipStream_t stream);

// E8M0 block scales applied by v_mfma_scale_f32_32x32x64_f8f6f4 (k a multiple of 128). Defined in gemm_fast.hip.
int launch_mx_gemm_fast(const GemmArgs& p, int mode, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, dim3 grid,
                        hipStream_t stream);

// misc.hip: the gated activation as a pass of its own, in 16-byte pieces (false: alignment does not allow them);
// epilogue_form: forward silu in the gated GEMM epilogue's expression instead of the stand-alone operator's
bool launch_gated_pieces(const void* z, const void* dy, int64_t dy_stride, void* out, int64_t rows, int64_t h, int dtype,
                         int activation, bool backward, bool epilogue_form, hipStream_t stream);

// Which kernel a plain per-tensor or block-scaled product runs on: gemm_pingpong with tiles of 256 x 256 (L), 256 x 128 (M) or
// 128 x 128 (S), or group_gemm_fast (from 512 tiles of 128 x 128 up with several blocks per CU, below 128 with halved tiles).
// The choice is the least of four estimates in microseconds, fitted to the measured times of 38 shapes (bf16 outputs, both recipes;
// within 15 % of nearly all). A round of one tile per CU takes a fixed part (first loads, stores of the tile) and a time per chunk of 64 k
// that grows with the share of CUs at work, because the clock falls as the matrix pipes fill (2.4 to 1.7 GHz):
//   L 0.40 .. 0.71 + 8.5    M 0.22 .. 0.39 + 5.3    S 0.235 alone + 4; two blocks per CU 0.57 for the pair + 4
// group_gemm_fast has no rounds to speak of (three small blocks per CU, their stores under each other's math): 0.31 per tile
// and chunk of a CU's share + 0.7 per tile. What that comes to: 8192 x 1024 x 4096 M (30 us), 4096 x 1152 x 4608 M (26),
// 4096 x 4096 x 4096 L (55), 4096 x 4608 x 1152 stays (30), 2048 x 1152 x 4608 S (19).
enum ScaledTile { SCALED_TILE_FAST = 0, SCALED_TILE_L, SCALED_TILE_M, SCALED_TILE_S, SCALED_TILE_L_THEN_S };
// L_THEN_S: full rounds of L, and the last up to 64 tiles as four S each (`last`; gated products do not run that way), which take
// 0.22 .. 0.40 a chunk, as the share of CUs, + 4.
inline ScaledTile choose_scaled_tile(int64_t m, int64_t n, int64_t k, bool last = true) {
    constexpr int64_t CUS = 256;
    auto tiles = [&](int64_t rows, int64_t cols) { return ((m + rows - 1) / rows) * ((n + cols - 1) / cols); };
    const int64_t small = tiles(128, 128);
    if (small < 128 || small >= (1 << 28) || 256 * k >= (1ll << 31)) return SCALED_TILE_FAST;
    const double chunks = (double)((k + 63) / 64);
    auto rounds = [&](int64_t count, double idle, double busy, double fixed) {
        const double full = (double)(count / CUS), rest = (double)(count % CUS) / CUS;
        return full * (chunks * busy + fixed) + (rest > 0 ? chunks * (idle + (busy - idle) * rest) + fixed : 0.0);
    };
    const double large = rounds(tiles(256, 256), 0.40, 0.71, 8.5), medium = rounds(tiles(256, 128), 0.22, 0.39, 5.3);
    const double pairs = small <= CUS ? chunks * 0.235 + 4.0 : (double)((small + 2 * CUS - 1) / (2 * CUS)) * (chunks * 0.57 + 4.0);
    const double fast = small >= 2 * CUS ? (double)small / CUS * (chunks * 0.31 + 0.7) + 4.0 : 1e30;
    ScaledTile best = SCALED_TILE_FAST;
    double least = fast;
    if (pairs < least) { least = pairs; best = SCALED_TILE_S; }
    if (medium < least) { least = medium; best = SCALED_TILE_M; }
    if (large < least) { least = large; best = SCALED_TILE_L; }
    const int64_t whole = tiles(256, 256) / CUS, rest = tiles(256, 256) % CUS;
    if (last && whole > 0 && rest > 0 && rest <= CUS / 4 &&
        (double)whole * (chunks * 0.71 + 8.5) + chunks * (0.22 + 0.18 * (double)rest / (CUS / 4)) + 4.0 < least)
        best = SCALED_TILE_L_THEN_S;
    return best;
}

// gemm_pingpong_tensor.hip, gemm_pingpong_mx.hip; gated: forward without [g | u], on the large tile
int launch_tensor_pingpong(const GemmArgs& p, ScaledTile tile, bool gated, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, hipStream_t stream);
int launch_mx_pingpong(const GemmArgs& p, ScaledTile tile, bool gated, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, hipStream_t stream);

}  // namespace viola
