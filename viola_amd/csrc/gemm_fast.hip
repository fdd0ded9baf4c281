// Grouped FP32-scale instances of the fast FP8 GEMM kernel (plain, gated forward, gated backward; uniform or
// row-wise b scales).
#include <math.h>

#include "gemm_fast_kernel.hpp"

namespace viola {

template <int MODE, bool B_ROWSCALE, typename TO, int TN, bool KSPLIT = false>
static void launch_formats(const GemmArgs& p, int a_dtype, int b_dtype, int bias_dtype, dim3 grid, hipStream_t stream) {
    const bool a5 = a_dtype == VIOLA_E5M2, b5 = b_dtype == VIOLA_E5M2;
    const dim3 block(KSPLIT ? 2 * FTHREADS : FTHREADS);
    if (!a5 && !b5) VIOLA_LAUNCH((group_gemm_fast<MODE, false, false, B_ROWSCALE, TO, TN, false, false, KSPLIT>), grid, block, 0, stream, p, bias_dtype);
    else if (a5 && !b5) VIOLA_LAUNCH((group_gemm_fast<MODE, true, false, B_ROWSCALE, TO, TN, false, false, KSPLIT>), grid, block, 0, stream, p, bias_dtype);
    else if (!a5 && b5) VIOLA_LAUNCH((group_gemm_fast<MODE, false, true, B_ROWSCALE, TO, TN, false, false, KSPLIT>), grid, block, 0, stream, p, bias_dtype);
    else VIOLA_LAUNCH((group_gemm_fast<MODE, true, true, B_ROWSCALE, TO, TN, false, false, KSPLIT>), grid, block, 0, stream, p, bias_dtype);
}

// plain mode, the k range of a tile split over two teams of waves
template <int TN, bool ROWSCALE>
static int launch_split(const GemmArgs& p, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, dim3 grid, hipStream_t stream) {
    switch (out_dtype) {
        case VIOLA_F32: launch_formats<MODE_PLAIN, ROWSCALE, float, TN, true>(p, a_dtype, b_dtype, bias_dtype, grid, stream); break;
        case VIOLA_BF16: launch_formats<MODE_PLAIN, ROWSCALE, bf16_t, TN, true>(p, a_dtype, b_dtype, bias_dtype, grid, stream); break;
        case VIOLA_F16: launch_formats<MODE_PLAIN, ROWSCALE, f16_t, TN, true>(p, a_dtype, b_dtype, bias_dtype, grid, stream); break;
        default: return VIOLA_EINVAL;
    }
    return viola_launch_status();
}

template <int MODE, int TN>
static int launch_mode(const GemmArgs& p, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, bool rowscale, dim3 grid,
                       hipStream_t stream) {
#define VIOLA_FAST(TO)                                                                           \
    if (rowscale) launch_formats<MODE, true, TO, TN>(p, a_dtype, b_dtype, bias_dtype, grid, stream); \
    else launch_formats<MODE, false, TO, TN>(p, a_dtype, b_dtype, bias_dtype, grid, stream);
    switch (out_dtype) {
        case VIOLA_F32: VIOLA_FAST(float) break;
        case VIOLA_BF16: VIOLA_FAST(bf16_t) break;
        case VIOLA_F16: VIOLA_FAST(f16_t) break;
        default: return VIOLA_EINVAL;
    }
#undef VIOLA_FAST
    return viola_launch_status();
}

// shortest k ranges worth splitting (4096 x 1024 tiles of 128 x 128: k = 1024 14.4 -> 15.1 us, k = 1536 17.7 -> 17.1 us; 1024 x 1024
// on 128 x 64 tiles: k = 512 slower, k = 1024 9.8 -> 9.1 us, k = 1536 12.6 -> 11.1 us)
constexpr int64_t SPLIT_MIN_K = 1536, NARROW_SPLIT_MIN_K = 1024;

// Whether a plain product runs on gemm_pingpong_grouped: the lesser of two estimates in microseconds, fitted to the measured times
// of 42 shapes (bf16 outputs, within 8 % of nearly all). Two blocks of 128 x 128 of group_gemm_fast share a CU and cover each
// other's first loads and stores, so a round of 512 costs little beside its chunks of 64 k, and a last one of up to 256 goes
// faster; the large tiles take a CU each, whole rounds of 256, with nothing to cover their ends. So they win from about k = 1024
// (8192 x 4096 x 1024 75 -> 67 us, 16384 x 4096 x 256 55 -> 56) where they fill the chip (4096 x 4096 x 2048, 256 of them, 68 -> 61;
// 6000 x 4096 x 1024, 384, 55 -> 60; row-wise 4096 x 3072 x 8192, 384, 245 -> 251). At 256 tiles of 128 x 128 and fewer the split
// forms have more of the chip at work (8192 x 4096 x 1024 transposed, 88 -> 115 us). Groups of rows fill half of their last tile
// on average; groups of k have each the average length. With uniform b scales a last round of up to 128 large tiles runs on halves or
// quarters of them (gemm_pingpong_grouped_rounds), so that one round and a quarter pays too (4352 x 4096 x 4096, 272 tiles,
// 154 -> 145; one and a half does not, 6000 x 4096 x 1024).
static bool prefer_pingpong(const GemmArgs& p, bool rowscale, unsigned k_groups) {
    constexpr double CUS = 256.0;
    if (p.k < 256 || 256 * p.lda >= (1ll << 31)) return false;
    auto tiles = [&](int64_t rows, int64_t cols) {
        const double row_tiles = p.offsets ? (double)p.m / rows + 0.5 * p.groups : (double)((p.m + rows - 1) / rows);
        return row_tiles * (double)((p.n + cols - 1) / cols) * k_groups;
    };
    const double chunks = (double)p.k / 64.0 / k_groups, small = tiles(128, 128), large = tiles(256, rowscale ? 128 : 256);
    if (small <= CUS) return false;
    const double pair = rowscale ? 1.2 : 0.97, idle = rowscale ? 0.82 : 1.2, busy = rowscale ? 1.04 : 1.61, ends = rowscale ? 6.0 : 7.5;
    const double pairs = floor(small / (2 * CUS)), left = small - pairs * 2 * CUS;
    const double now = pairs * (chunks * pair + 3.3) + (left > 0 ? chunks * pair * (left <= CUS ? 0.52 : 1.0) + 3.3 : 0.0);
    const double rounds = floor(large / CUS), rest = large / CUS - rounds;
    double last = rest > 0 ? chunks * (idle + (busy - idle) * rest) + ends : 0.0;
    if (!rowscale && rounds > 0 && rest > 0 && rest <= 0.25) last = chunks * (0.42 + 0.4 * rest) + 6.0;
    else if (!rowscale && rounds > 1 && rest > 0 && rest <= 0.5) last = chunks * (0.45 + rest) + 5.0;
    return rounds * (chunks * busy + ends) + last < now;
}

// Whether a product with uniform b scales that is too small for 256 x 256 tiles runs on tiles of 256 x 128, one round of them: where two
// blocks of 128 x 128 would share a CU. Measured over 129 to 256 such tiles (0 % to 20 % of them padding), both times are linear in the
// share of the chip at work: 8192 x 1024 x 4096 70 -> 66 us, 9850 x 768 x 3072 51 -> 49, 16384 x 512 x 8192 136 -> 126, 5000 x 1024 x 4096
// 58 -> 55; up to k = 1024 the small blocks, which cover each other's ends, are as fast (8192 x 1024 x 1024 20.7 us, x 512 12.6 against
// 13.3). Two rounds always lose (12000 x 768 x 2048, 282 tiles, 48 -> 62).
static bool prefer_tall(const GemmArgs& p) {
    if (p.koffsets || 256 * p.lda >= (1ll << 31)) return false;
    const int64_t columns = (p.n + 127) / 128, rows = p.offsets ? p.m / 256 + p.groups : (p.m + 255) / 256;
    const double tall = (double)(rows * columns), small = (double)columns * (p.offsets ? (double)p.m / 128 + 0.5 * p.groups : (double)((p.m + 127) / 128));
    if (small <= 256.0 || tall > 256.0) return false;
    const double chunks = (double)p.k / 64.0;
    return chunks * (0.45 + 0.5 * tall / 256.0) + 5.0 < chunks * (0.53 + 0.51 * small / 512.0) + 3.3;
}

// In how many parts of k a weight gradient runs, which has few tiles and a long k. Whole, 129 to 256 tiles of 128 x 128 leave CUs
// without a tile, and fewer run as narrow tiles, which read more per product; in parts, tiles of 256 x 128 fill the chip and a second
// launch adds the partial products, a few hundred cycles per part on top of their bytes. The least of the estimates in microseconds
// decides, and only where it saves a twentieth. Fitted to 56 shapes, whole and in up to 20 counts of parts (whole within 7 %, the counts
// that come near the best within 5 % on average); what it takes is within 8 % of the fastest count of each:
//   3072 x 768 x 9856 82 -> 64 us in three    1024 x 1024 x 16384 89 -> 50 in eight    512 x 512 x 16384 88 -> 28 in 20
//   256 x 256 x 16384 83 -> 24 in 32          1000 x 332 x 3200 22.5 -> 20.5 in ten    1152 x 1152 x 16384 90 -> 66 in five
// It stays whole where parts gain nothing, 4096 x 1024 x 8192 (75 us, 84 in two) and 1024 x 1024 x 4096 (26.7 us, 28.6 in seven), and where
// they gain less than the estimate can tell, 2048 x 1024 x 8192 (52.7 us, 50.3 in four).
// The partial products are scratch that a whole product does not need, in a pass that may be short of memory: at most PARTS_SCRATCH
// bytes. Up to 256 tiles of 128 x 128 and 16384 tokens no count that is taken needs more than 34 MB. Beyond, whole products fill the
// chip, and the 140 to 230 MB of larger ones, which gained 6 to 8 %, are not spent (4352 x 4224 x 16128 734 -> 681 us in two, 147 MB;
// 3072 x 3072 x 16384 455 -> 375 in four, 151 MB, but 400 in two, 75 MB, which it takes).
constexpr int64_t PARTS_SCRATCH = 96ll << 20;
int plan_k_parts(int64_t m, int64_t n, int64_t k) {
    constexpr double CUS = 256.0;
    if (k < 1024 || m < 64 || n < 64 || n % 4 != 0) return 1;               // (rows of the partial products in whole 16-byte pieces)
    const int64_t all = (k + 127) / 128 * (128 / FBK);                       // of the host path's pitch: see launch_group_parts
    const double chunks = (double)all, small = (double)((m + 127) / 128) * (double)((n + 127) / 128), large = (double)((m + 255) / 256) * (double)((n + 127) / 128);
    auto tiles_of = [&](double count, double length) {
        const double rounds = floor(count / CUS), rest = count / CUS - rounds;
        return rounds * (length * 0.95 + 4.3) + (rest > 0 ? length * (0.77 + 0.18 * rest) + 4.3 : 0.0);
    };
    // whole, as launch_group_gemm_fast runs it
    double least;
    if (small <= CUS / 2) least = chunks * (0.32 + 0.05 * small / 128.0) + 4.5;
    else if (small <= CUS) least = chunks * (0.35 + 0.18 * small / CUS) + 7.0;
    else {
        const double pairs = floor(small / (2 * CUS)), left = small - pairs * 2 * CUS, wide = tiles_of(large, chunks);
        least = pairs * (chunks * 1.15 + 3.3) + (left > 0 ? chunks * 1.15 * (left <= CUS ? 0.52 : 1.0) + 3.3 : 0.0);
        if (wide < least) least = wide;
    }
    least *= 0.95;
    int best = 1;
    for (int64_t parts = 2; parts <= 64 && all / parts >= 4 && parts * ((m * n + 3) / 4 * 16) <= PARTS_SCRATCH; ++parts) {
        const int64_t length = (all + parts - 1) / parts;
        if ((all + length - 1) / length != parts) continue;                  // the last ones would be empty: the same as fewer
        const double time = tiles_of(large * parts, (double)length) + 5.6 + 0.155 * parts + (double)m * n * (4.0 * parts + 2.0) / 4.1e6;
        if (time < least) { least = time; best = (int)parts; }
    }
    return best;
}

// The kernel of a product: plain ones on the large tiles where those win, else the blocks of group_gemm_fast. Two blocks of 128 x 128
// fit a CU, so from 257 tiles up every CU has work and the full tile, which reads the least, is the fastest form (4096 x 1152 x 4608:
// 75.6 -> 59.7 us against the split one, 6000 x 1000 x 1024: 27.0 -> 19.6 us against tiles halved in n). From 129 to 256 tiles a CU gets
// one: over a long k keep the tile and split its k range over twice the waves inside the block (7-12 % faster at 256 tiles, k >= 2048;
// with row-wise b scales the teams take turns, 4096 x 1024 x 8192 86 -> 74 us, 1536 x 1536 x 4096 43 -> 35, with uniform ones they do not
// gain by it, 68 against 77), else halve the tile in n for a second block per CU. With 128 tiles or fewer the narrow tiles keep more
// CUs busy and their k range is split: a CU then holds eight waves instead of four (1024 x 1024 x 16384: 98 -> 76 us, 512 x 512 x 4096:
// 27.5 -> 22.3 us). Narrow split tiles are one per CU: past 256 of them the second round costs more than the split gives
// (600 x 4096 x 1024: 17.2 us, unsplit 12.5 us).
GroupForm group_form(const GemmArgs& p, bool rowscale, dim3 grid) {
    if (prefer_pingpong(p, rowscale, grid.z)) return GROUP_LARGE;
    if (!rowscale && prefer_tall(p)) return GROUP_TALL;
    const int64_t tiles = (int64_t)grid.x * grid.y * grid.z;
    if (tiles > 256) return GROUP_BLOCKS;
    const bool fixed_k = !p.offsets && !p.koffsets;
    if (tiles > 128 && fixed_k && p.k >= SPLIT_MIN_K) return rowscale ? GROUP_TEAMS : GROUP_BLOCKS_SPLIT;
    if (p.n <= 64) return GROUP_BLOCKS;
    return tiles <= 128 && fixed_k && p.k >= NARROW_SPLIT_MIN_K ? GROUP_NARROW_SPLIT : GROUP_NARROW;
}

int launch_group_gemm_fast(const GemmArgs& args, int mode, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, bool rowscale,
                           dim3 grid, hipStream_t stream) {
    GemmArgs p = args;
    const int64_t b_rows = mode == MODE_GATED_FWD ? 2 * p.n : p.n;
    p.sa_bytes = (p.m + p.ar - 1) / p.ar * p.ldsa * 4;
    p.sb_bytes = (b_rows + p.br - 1) / p.br * p.ldsb * 4;
    const GroupForm form = mode == MODE_PLAIN ? group_form(p, rowscale, grid) : GROUP_BLOCKS;
    const int64_t row_tiles = p.offsets ? p.m / 256 + p.groups : (p.m + 255) / 256;
    if (form == GROUP_LARGE) return launch_group_pingpong(p, (int)row_tiles, a_dtype, b_dtype, bias_dtype, out_dtype, rowscale, grid.z, stream);
    if (form == GROUP_TALL) return launch_group_tall(p, (int)row_tiles, a_dtype, b_dtype, bias_dtype, out_dtype, stream);
    if (form == GROUP_TEAMS) return launch_group_teams(p, a_dtype, b_dtype, bias_dtype, out_dtype, stream);
    const bool narrow = form == GROUP_NARROW || form == GROUP_NARROW_SPLIT;
    if (narrow) grid.x = (unsigned)((p.n + 63) / 64);
    if ((int64_t)grid.x * grid.y < (1 << 30)) {
        p.tiles_n = (int)grid.x;
        p.tiles_m = (int)grid.y;
        grid = dim3((grid.x * grid.y + 7) / 8 * 8, 1, grid.z);
    }
    if (form == GROUP_BLOCKS_SPLIT) return launch_split<2, false>(p, a_dtype, b_dtype, bias_dtype, out_dtype, grid, stream);
    if (form == GROUP_NARROW_SPLIT)
        return rowscale ? launch_split<1, true>(p, a_dtype, b_dtype, bias_dtype, out_dtype, grid, stream)
                        : launch_split<1, false>(p, a_dtype, b_dtype, bias_dtype, out_dtype, grid, stream);
    if (narrow) return launch_mode<MODE_PLAIN, 1>(p, a_dtype, b_dtype, bias_dtype, out_dtype, rowscale, grid, stream);
    if (mode == MODE_PLAIN) return launch_mode<MODE_PLAIN, 2>(p, a_dtype, b_dtype, bias_dtype, out_dtype, rowscale, grid, stream);
    if (mode == MODE_GATED_FWD) return launch_mode<MODE_GATED_FWD, 2>(p, a_dtype, b_dtype, bias_dtype, out_dtype, rowscale, grid, stream);
    return launch_mode<MODE_GATED_BWD, 2>(p, a_dtype, b_dtype, bias_dtype, out_dtype, rowscale, grid, stream);
}

}  // namespace viola
