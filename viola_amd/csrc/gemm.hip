// Entry points of the FP8 GEMMs: argument checks and the choice of kernel (gemm_generic.hip, gemm_fast*.hip, gemm_pingpong*.hip).
#include "gemm_args.hpp"

namespace viola {

static int shift_of(int v) {
    int s = 0;
    while ((1 << s) < v) ++s;
    return s;
}

// the fast kernels address operands and scales with 31-bit byte offsets and stage the scales of 8 consecutive 32-wide K groups at once
static bool fast_sizes(const GemmArgs& p, int64_t b_rows) {
    return b_rows * p.ldb < (1ll << 31) && (int64_t)BM * p.lda < (1ll << 31) && (p.m + p.ar - 1) / p.ar * p.ldsa * 4 < (1ll << 31) &&
           (b_rows + p.br - 1) / p.br * p.ldsb * 4 < (1ll << 31) && p.ak_shift == 5 && p.bk_shift == 5;
}

template <int MODE>
static int launch_out(const GemmArgs& p, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, bool rowscale, bool vec,
                      dim3 grid, hipStream_t stream) {
    if (vec && fast_sizes(p, MODE == MODE_GATED_FWD ? 2 * p.n : p.n))
        return launch_group_gemm_fast(p, MODE, a_dtype, b_dtype, bias_dtype, out_dtype, rowscale, grid, stream);
    return launch_group_gemm_generic(p, MODE, a_dtype, b_dtype, bias_dtype, out_dtype, rowscale, grid, stream);
}

static bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }
static bool pow2(int v) { return v > 0 && (v & (v - 1)) == 0; }

}  // namespace viola

using namespace viola;

extern "C" int viola_group_gemm(const void* a, int a_dtype, const void* b, int b_dtype, const float* sa, const float* sb,
                                int64_t m, int64_t n, int64_t k, int ar, int ak, int br, int bk, const void* bias,
                                int bias_dtype, void* out, int out_dtype, viola_stream_t stream_) {
    hipStream_t stream = viola_enter(stream_);
    VIOLA_CHECK_ARG(viola_is_fp8(a_dtype) && viola_is_fp8(b_dtype) && viola_is_float(out_dtype));
    VIOLA_CHECK_ARG(m >= 0 && n >= 0 && k >= 0 && ar > 0 && br > 0 && pow2(ak) && pow2(bk) && ak >= 32 && bk >= 32);
    VIOLA_CHECK_ARG(!bias || viola_is_float(bias_dtype));
    if (m == 0 || n == 0) return 0;
    VIOLA_CHECK_ARG(out && (k == 0 || (a && b && sa && sb)));
    const int64_t gy = (m + BM - 1) / BM, gx = (n + BN - 1) / BN;
    VIOLA_CHECK_ARG(gy <= 65535);
    GemmArgs p = {};
    p.a = static_cast<const uint8_t*>(a); p.b = static_cast<const uint8_t*>(b); p.sa = sa; p.sb = sb;
    p.bias = bias; p.out = out; p.m = m; p.n = n; p.k = k; p.lda = k; p.ldb = k;
    p.ldsa = (k + ak - 1) / ak; p.ldsb = (k + bk - 1) / bk; p.ldo = n;
    p.ar = ar; p.br = br; p.ak_shift = shift_of(ak); p.bk_shift = shift_of(bk);
    const bool vec = k % 16 == 0 && aligned16(a) && aligned16(b);
    const bool rowscale = br % 32 != 0;
    return launch_out<MODE_PLAIN>(p, a_dtype, b_dtype, bias_dtype, out_dtype, rowscale, vec, dim3((unsigned)gx, (unsigned)gy), stream);
}

extern "C" int viola_scaled_gemm_form(int64_t m, int64_t n, int64_t k) {
    constexpr int64_t LARGEST = 1ll << 31;
    VIOLA_CHECK_ARG(m > 0 && n > 0 && k > 0 && m < LARGEST && n < LARGEST && k < LARGEST);
    return choose_scaled_tile(m, n, k);
}

extern "C" int viola_group_gemm_form(int64_t m, int64_t n, int64_t k, int row_scaled_b, int row_groups, int k_groups) {
    constexpr int64_t LARGEST = 1ll << 31;
    VIOLA_CHECK_ARG(m > 0 && n > 0 && k > 0 && m < LARGEST && n < LARGEST && k < LARGEST && k % 16 == 0);
    VIOLA_CHECK_ARG(row_groups >= 0 && k_groups >= 0 && k_groups <= 65535 && (!k_groups || (row_scaled_b && !row_groups)));
    const int64_t gy = (m + BM - 1) / BM + row_groups;
    VIOLA_CHECK_ARG(gy <= 65535);
    static const int64_t there = 0;                                          // (the rule asks only whether there are offsets)
    GemmArgs p = {};
    p.m = m; p.n = n; p.k = k; p.lda = k; p.ldb = k; p.groups = row_groups;
    p.ar = 1; p.br = row_scaled_b ? 1 : 32; p.ldsa = p.ldsb = (k + 31) / 32; p.ak_shift = p.bk_shift = 5;
    p.offsets = row_groups ? &there : nullptr;
    p.koffsets = k_groups ? &there : nullptr;
    VIOLA_CHECK_ARG(fast_sizes(p, n));
    return group_form(p, row_scaled_b != 0, dim3((unsigned)((n + BN - 1) / BN), (unsigned)gy, k_groups ? (unsigned)k_groups : 1));
}

// (what the fast kernel asks of a product with a scale per row and 32 k on both sides, plus what 256 rows of a large tile do)
static bool parts_fit(int64_t m, int64_t n, int64_t k) {
    const int64_t rows = m > n ? m : n;
    return rows * k < (1ll << 31) && 256 * k < (1ll << 31) && rows * ((k + 31) / 32) * 4 < (1ll << 31) && m * n < (1ll << 31);
}

extern "C" int viola_group_gemm_parts(int64_t m, int64_t n, int64_t k) {
    constexpr int64_t LARGEST = 1ll << 31;
    if (m <= 0 || n <= 0 || k <= 0 || m >= LARGEST || n >= LARGEST || k >= LARGEST || !parts_fit(m, n, k)) return 1;
    return plan_k_parts(m, n, k);
}

extern "C" int viola_group_gemm_in_parts(const void* a, int a_dtype, const void* b, int b_dtype, const float* sa, const float* sb, int64_t m, int64_t n,
                                         int64_t k, void* out, int out_dtype, int parts, float* workspace, int64_t workspace_floats, viola_stream_t stream_) {
    hipStream_t stream = viola_enter(stream_);
    VIOLA_CHECK_ARG(viola_is_fp8(a_dtype) && viola_is_fp8(b_dtype) && viola_is_float(out_dtype));
    VIOLA_CHECK_ARG(m >= 0 && n >= 0 && k > 0 && parts >= 2 && parts <= 64 && workspace && aligned16(workspace));
    if (m == 0 || n == 0) return 0;
    VIOLA_CHECK_ARG(a && b && sa && sb && out);
    if (k % 16 != 0 || !aligned16(a) || !aligned16(b) || !parts_fit(m, n, k)) return VIOLA_EUNSUPPORTED;
    VIOLA_CHECK_ARG(workspace_floats >= parts * ((m * n + 3) / 4 * 4));
    GemmArgs p = {};
    p.a = static_cast<const uint8_t*>(a); p.b = static_cast<const uint8_t*>(b); p.sa = sa; p.sb = sb;
    p.out = out; p.m = m; p.n = n; p.k = k; p.lda = k; p.ldb = k;
    p.ldsa = (k + 31) / 32; p.ldsb = (k + 31) / 32; p.ldo = n;
    p.sa_bytes = m * p.ldsa * 4; p.sb_bytes = n * p.ldsb * 4;
    p.ar = 1; p.br = 1; p.ak_shift = 5; p.bk_shift = 5;
    return launch_group_parts(p, parts, a_dtype, b_dtype, out_dtype, workspace, stream);
}

static int gcd_of(int a, int b) { while (b) { const int t = a % b; a = b; b = t; } return a; }

extern "C" int viola_group_gemm_half(const void* a, int a_dtype, const void* b, int b_dtype, const float* sa, const float* sb,
                                     int64_t m, int64_t n, int64_t k, int ar, int ak, int br, int bk, const void* bias,
                                     int bias_dtype, void* out, int out_dtype, int accum_block, int reduce_dtype,
                                     viola_stream_t stream_) {
    hipStream_t stream = viola_enter(stream_);
    VIOLA_CHECK_ARG(viola_is_fp8(a_dtype) && viola_is_fp8(b_dtype) && viola_is_float(out_dtype));
    VIOLA_CHECK_ARG(m >= 0 && n >= 0 && k >= 0 && ar > 0 && br > 0 && pow2(ak) && pow2(bk) && ak >= 32 && bk >= 32);
    VIOLA_CHECK_ARG((!bias || viola_is_float(bias_dtype)) && accum_block >= 0 && accum_block % 32 == 0);
    VIOLA_CHECK_ARG(reduce_dtype == VIOLA_F32 || reduce_dtype == VIOLA_BF16);
    if (m == 0 || n == 0) return 0;
    VIOLA_CHECK_ARG(out && (k == 0 || (a && b && sa && sb)));
    const int64_t gy = (m + BM - 1) / BM, gx = (n + BN - 1) / BN;
    VIOLA_CHECK_ARG(gy <= 65535);
    GemmArgs p = {};
    p.a = static_cast<const uint8_t*>(a); p.b = static_cast<const uint8_t*>(b); p.sa = sa; p.sb = sb;
    p.bias = bias; p.out = out; p.m = m; p.n = n; p.k = k; p.lda = k; p.ldb = k;
    p.ldsa = (k + ak - 1) / ak; p.ldsb = (k + bk - 1) / bk; p.ldo = n;
    p.ar = ar; p.br = br; p.ak_shift = shift_of(ak); p.bk_shift = shift_of(bk);
    // the partial is cleared where the reference clears it: every gcd(a's K group, b's K group, accum_block) k
    p.half_period = accum_block ? gcd_of(gcd_of(ak, bk), accum_block) : gcd_of(ak, bk);
    p.reduce_bf16 = reduce_dtype == VIOLA_BF16;
    return launch_group_gemm_half(p, false, a_dtype, b_dtype, bias_dtype, out_dtype, br % 32 != 0, dim3((unsigned)gx, (unsigned)gy), stream);
}

extern "C" int viola_tensor_gemm_half(const void* a, int a_dtype, const void* b, int b_dtype, const float* sa, const float* sb,
                                      int64_t m, int64_t n, int64_t k, const void* bias, int bias_dtype, void* out, int out_dtype,
                                      int accum_block, int reduce_dtype, viola_stream_t stream_) {
    hipStream_t stream = viola_enter(stream_);
    VIOLA_CHECK_ARG(viola_is_fp8(a_dtype) && viola_is_fp8(b_dtype) && viola_is_float(out_dtype));
    VIOLA_CHECK_ARG(m >= 0 && n >= 0 && k >= 0 && k < (1ll << 30) && (!bias || viola_is_float(bias_dtype)));
    VIOLA_CHECK_ARG(accum_block >= 0 && accum_block % 32 == 0 && (reduce_dtype == VIOLA_F32 || reduce_dtype == VIOLA_BF16));
    if (m == 0 || n == 0) return 0;
    VIOLA_CHECK_ARG(out && sa && sb && (k == 0 || (a && b)));
    const int64_t gy = (m + BM - 1) / BM, gx = (n + BN - 1) / BN;
    VIOLA_CHECK_ARG(gy <= 65535);
    GemmArgs p = {};
    p.a = static_cast<const uint8_t*>(a); p.b = static_cast<const uint8_t*>(b); p.sa = sa; p.sb = sb;
    p.bias = bias; p.out = out; p.m = m; p.n = n; p.k = k; p.lda = k; p.ldb = k; p.ldo = n;
    p.ldsa = 0; p.ldsb = 0; p.ar = 1 << 30; p.br = 1 << 30; p.ak_shift = 30; p.bk_shift = 30;
    // the reference's loop adds the partial to the total after whole chunks of 64 k (of accum_block k below that):
    // viola/nn/_linear_kernels.py:150-153, :272-273
    p.half_period = accum_block < 64 ? accum_block : accum_block / 64 * 64;
    p.reduce_bf16 = reduce_dtype == VIOLA_BF16;
    return launch_group_gemm_half(p, true, a_dtype, b_dtype, bias_dtype, out_dtype, false, dim3((unsigned)gx, (unsigned)gy), stream);
}

// Large gated products run as the plain GEMM on the tile that suits it plus one elementwise pass over its output: with one block
// per CU nothing covers a block's gated epilogue, and the pass costs less than that (MLP step at 16384 x 4096 -> 11008: 7.55 ms
// against 7.90 ms under per-tensor scales, 8.41 ms against 9.06 ms under MXFP8). Backward the epilogue also reads [g | u] in
// place, so the pass wins on every tile (4096 x 4608 x 1152 106 -> 78 us, 1024 x 1024 x 1024 19.2 -> 10.3 us) down to where a
// second launch is what counts. No extra memory: forward the plain product is the [g | u] the caller keeps anyway, backward it
// lands in the up half of dz and is replaced there.
static bool gated_in_two_passes(int64_t m, int64_t k, int64_t h, const void* aux, const void* out, int out_dtype, bool backward) {
    const int64_t piece = out_dtype == VIOLA_F32 ? 4 : 8;
    if (!aux || h % piece != 0 || !aligned16(aux) || !aligned16(out) || m * (h / piece) / 256 >= 0x7fffffff) return false;   // the pass is one launch of 256-thread blocks
    if (backward) return m * h >= (1 << 17);
    const ScaledTile tile = choose_scaled_tile(m, 2 * h, k, false);
    return tile == SCALED_TILE_L || tile == SCALED_TILE_M;
}

static int tensor_gemm(const void* a, int a_dtype, const void* b, int b_dtype, const float* sa, const float* sb, int64_t m,
                       int64_t n, int64_t k, const void* bias, int bias_dtype, void* out, int64_t ldo, int out_dtype,
                       hipStream_t stream) {
    VIOLA_CHECK_ARG(viola_is_fp8(a_dtype) && viola_is_fp8(b_dtype) && viola_is_float(out_dtype));
    VIOLA_CHECK_ARG(m >= 0 && n >= 0 && k >= 0 && k < (1ll << 30) && (!bias || viola_is_float(bias_dtype)));
    if (m == 0 || n == 0) return 0;
    VIOLA_CHECK_ARG(out && sa && sb && (k == 0 || (a && b)));
    const int64_t gy = (m + BM - 1) / BM, gx = (n + BN - 1) / BN;
    VIOLA_CHECK_ARG(gy <= 65535);
    GemmArgs p = {};
    p.a = static_cast<const uint8_t*>(a); p.b = static_cast<const uint8_t*>(b); p.sa = sa; p.sb = sb;
    p.bias = bias; p.out = out; p.m = m; p.n = n; p.k = k; p.lda = k; p.ldb = k; p.ldo = ldo;
    // one scale group per operand: every (row, k) lands on scale index 0
    p.ldsa = 0; p.ldsb = 0; p.ar = 1 << 30; p.br = 1 << 30; p.ak_shift = 30; p.bk_shift = 30;
    const dim3 grid((unsigned)gx, (unsigned)gy);
    const bool vec = k % 16 == 0 && k > 0 && aligned16(a) && aligned16(b);
    if (vec && n * k < (1ll << 31) && (int64_t)BM * k < (1ll << 31))
        return launch_tensor_gemm_fast(p, MODE_PLAIN, a_dtype, b_dtype, bias_dtype, out_dtype, grid, stream);
    // odd alignment: the generic kernel, which multiplies each 32-wide K group's sum by sa * sb as it goes
    return launch_out<MODE_PLAIN>(p, a_dtype, b_dtype, bias_dtype, out_dtype, false, false, grid, stream);
}

extern "C" int viola_tensor_gemm(const void* a, int a_dtype, const void* b, int b_dtype, const float* sa, const float* sb,
                                 int64_t m, int64_t n, int64_t k, const void* bias, int bias_dtype, void* out, int out_dtype,
                                 viola_stream_t stream) {
    return tensor_gemm(a, a_dtype, b, b_dtype, sa, sb, m, n, k, bias, bias_dtype, out, n, out_dtype, static_cast<hipStream_t>(stream));
}

static int mx_gemm(const void* a, int a_dtype, const void* b, int b_dtype, const uint8_t* sa, const uint8_t* sb, int64_t m,
                   int64_t n, int64_t k, int ar, int br, const void* bias, int bias_dtype, void* out, int64_t ldo, int out_dtype,
                   hipStream_t stream) {
    VIOLA_CHECK_ARG(viola_is_fp8(a_dtype) && viola_is_fp8(b_dtype) && viola_is_float(out_dtype));
    VIOLA_CHECK_ARG(m >= 0 && n >= 0 && k >= 0 && ar > 0 && br > 0 && (!bias || viola_is_float(bias_dtype)));
    if (m == 0 || n == 0) return 0;
    VIOLA_CHECK_ARG(out && (k == 0 || (a && b && sa && sb)));
    const int64_t gy = (m + BM - 1) / BM, gx = (n + BN - 1) / BN;
    VIOLA_CHECK_ARG(gy <= 65535);
    // the block-scaled MFMA path only: whole 128-k scale pieces, 16-byte aligned codes, 4-byte aligned scale rows
    if (k == 0 || k % 128 != 0 || !aligned16(a) || !aligned16(b) || reinterpret_cast<uintptr_t>(sa) % 4 != 0 ||
        reinterpret_cast<uintptr_t>(sb) % 4 != 0 || n * k >= (1ll << 31) || (int64_t)BM * k >= (1ll << 31) ||
        (br != 1 && br % 32 != 0))
        return VIOLA_EUNSUPPORTED;
    GemmArgs p = {};
    p.a = static_cast<const uint8_t*>(a); p.b = static_cast<const uint8_t*>(b);
    p.sa = reinterpret_cast<const float*>(sa); p.sb = reinterpret_cast<const float*>(sb);
    p.bias = bias; p.out = out; p.m = m; p.n = n; p.k = k; p.lda = k; p.ldb = k; p.ldo = ldo;
    p.ldsa = k / 32; p.ldsb = k / 32; p.ar = ar; p.br = br; p.ak_shift = 5; p.bk_shift = 5;
    return launch_mx_gemm_fast(p, MODE_PLAIN, a_dtype, b_dtype, bias_dtype, out_dtype, dim3((unsigned)gx, (unsigned)gy), stream);
}

extern "C" int viola_mx_gemm(const void* a, int a_dtype, const void* b, int b_dtype, const uint8_t* sa, const uint8_t* sb,
                             int64_t m, int64_t n, int64_t k, int ar, int br, const void* bias, int bias_dtype, void* out,
                             int out_dtype, viola_stream_t stream) {
    return mx_gemm(a, a_dtype, b, b_dtype, sa, sb, m, n, k, ar, br, bias, bias_dtype, out, n, out_dtype, static_cast<hipStream_t>(stream));
}

// The two-pass form of a gated product; `plain(n, bias, out, ldo)` launches the plain GEMM of the recipe.
template <typename Plain>
static int gated_two_passes(Plain&& plain, int64_t m, int64_t h, const void* bias, void* aux, void* out, int out_dtype,
                            int activation, int backward, hipStream_t stream) {
    if (!backward) {
        const int status = plain(2 * h, bias, aux, 2 * h);                  // [g | u], biased
        if (status) return status;
        launch_gated_pieces(aux, nullptr, 0, out, m, h, out_dtype, activation, false, true, stream);
        return viola_launch_status();
    }
    uint8_t* up_half = static_cast<uint8_t*>(out) + h * (out_dtype == VIOLA_F32 ? 4 : 2);
    const int status = plain(h, nullptr, up_half, 2 * h);                   // dh, where d u will stand
    if (status) return status;
    launch_gated_pieces(aux, up_half, 2 * h, out, m, h, out_dtype, activation, true, true, stream);
    return viola_launch_status();
}

// The gated projections of an MLP under the per-tensor recipes: viola_gated_gemm's epilogues behind
// (acc * sa[0]) * sb[0].
extern "C" int viola_tensor_gated_gemm(const void* a, int a_dtype, const void* b, int b_dtype, const float* sa, const float* sb,
                                       int64_t m, int64_t h, int64_t k, const void* bias, int bias_dtype, void* aux, void* out,
                                       int out_dtype, int activation, int backward, viola_stream_t stream_) {
    hipStream_t stream = viola_enter(stream_);
    VIOLA_CHECK_ARG(viola_is_fp8(a_dtype) && viola_is_fp8(b_dtype) && viola_is_float(out_dtype));
    VIOLA_CHECK_ARG(m >= 0 && h >= 0 && k >= 0 && k < (1ll << 30));
    VIOLA_CHECK_ARG(activation >= VIOLA_SILU && activation <= VIOLA_RELU && (!bias || viola_is_float(bias_dtype)));
    if (m == 0 || h == 0) return 0;
    VIOLA_CHECK_ARG(out && sa && sb && (k == 0 || (a && b)) && (!backward || aux));
    GemmArgs p = {};
    p.a = static_cast<const uint8_t*>(a); p.b = static_cast<const uint8_t*>(b); p.sa = sa; p.sb = sb;
    p.bias = backward ? nullptr : bias; p.out = out; p.aux = aux; p.m = m; p.n = h; p.k = k; p.lda = k; p.ldb = k;
    p.ldo = backward ? 2 * h : h; p.activation = activation;
    p.ldsa = 0; p.ldsb = 0; p.ar = 1 << 30; p.br = 1 << 30; p.ak_shift = 30; p.bk_shift = 30;
    const int64_t gy = (m + BM - 1) / BM;
    VIOLA_CHECK_ARG(gy <= 65535);
    const int mode = backward ? MODE_GATED_BWD : MODE_GATED_FWD;
    const int64_t width = backward ? BN : BN / 2;
    const dim3 grid((unsigned)((h + width - 1) / width), (unsigned)gy);
    const bool vec = k % 16 == 0 && k > 0 && aligned16(a) && aligned16(b);
    if (vec && 2 * h * k < (1ll << 31) && (int64_t)BM * k < (1ll << 31)) {
        if (gated_in_two_passes(m, k, h, aux, out, out_dtype, backward)) {
            auto plain = [&](int64_t n, const void* n_bias, void* to, int64_t ldo) {
                return tensor_gemm(a, a_dtype, b, b_dtype, sa, sb, m, n, k, n_bias, bias_dtype, to, ldo, out_dtype, stream);
            };
            return gated_two_passes(plain, m, h, bias, aux, out, out_dtype, activation, backward, stream);
        }
        return launch_tensor_gemm_fast(p, mode, a_dtype, b_dtype, bias_dtype, out_dtype, grid, stream);
    }
    if (backward) return launch_out<MODE_GATED_BWD>(p, a_dtype, b_dtype, bias_dtype, out_dtype, false, false, grid, stream);
    return launch_out<MODE_GATED_FWD>(p, a_dtype, b_dtype, bias_dtype, out_dtype, false, false, grid, stream);
}

// The same under E8M0 block scales; VIOLA_EUNSUPPORTED where viola_mx_gemm returns it, and when the up rows of b do
// not start on a scale-row boundary (h not a multiple of br).
extern "C" int viola_mx_gated_gemm(const void* a, int a_dtype, const void* b, int b_dtype, const uint8_t* sa, const uint8_t* sb,
                                   int64_t m, int64_t h, int64_t k, int ar, int br, const void* bias, int bias_dtype, void* aux,
                                   void* out, int out_dtype, int activation, int backward, viola_stream_t stream_) {
    hipStream_t stream = viola_enter(stream_);
    VIOLA_CHECK_ARG(viola_is_fp8(a_dtype) && viola_is_fp8(b_dtype) && viola_is_float(out_dtype));
    VIOLA_CHECK_ARG(m >= 0 && h >= 0 && k >= 0 && ar > 0 && br > 0);
    VIOLA_CHECK_ARG(activation >= VIOLA_SILU && activation <= VIOLA_RELU && (!bias || viola_is_float(bias_dtype)));
    if (m == 0 || h == 0) return 0;
    VIOLA_CHECK_ARG(out && (k == 0 || (a && b && sa && sb)) && (!backward || aux));
    const int64_t gy = (m + BM - 1) / BM;
    VIOLA_CHECK_ARG(gy <= 65535);
    if (k == 0 || k % 128 != 0 || !aligned16(a) || !aligned16(b) || reinterpret_cast<uintptr_t>(sa) % 4 != 0 ||
        reinterpret_cast<uintptr_t>(sb) % 4 != 0 || 2 * h * k >= (1ll << 31) || (int64_t)BM * k >= (1ll << 31) ||
        (br != 1 && br % 32 != 0) || (!backward && h % br != 0))
        return VIOLA_EUNSUPPORTED;
    if (gated_in_two_passes(m, k, h, aux, out, out_dtype, backward)) {
        auto plain = [&](int64_t n, const void* n_bias, void* to, int64_t ldo) {
            return mx_gemm(a, a_dtype, b, b_dtype, sa, sb, m, n, k, ar, br, n_bias, bias_dtype, to, ldo, out_dtype, stream);
        };
        return gated_two_passes(plain, m, h, bias, aux, out, out_dtype, activation, backward, stream);
    }
    GemmArgs p = {};
    p.a = static_cast<const uint8_t*>(a); p.b = static_cast<const uint8_t*>(b);
    p.sa = reinterpret_cast<const float*>(sa); p.sb = reinterpret_cast<const float*>(sb);
    p.bias = backward ? nullptr : bias; p.out = out; p.aux = aux; p.m = m; p.n = h; p.k = k; p.lda = k; p.ldb = k;
    p.ldo = backward ? 2 * h : h; p.activation = activation;
    p.ldsa = k / 32; p.ldsb = k / 32; p.ar = ar; p.br = br; p.ak_shift = 5; p.bk_shift = 5;
    const int64_t width = backward ? BN : BN / 2;
    return launch_mx_gemm_fast(p, backward ? MODE_GATED_BWD : MODE_GATED_FWD, a_dtype, b_dtype, bias_dtype, out_dtype,
                               dim3((unsigned)((h + width - 1) / width), (unsigned)gy), stream);
}

extern "C" int viola_gated_gemm(const void* a, int a_dtype, const void* b, int b_dtype, const float* sa, const float* sb,
                                int64_t m, int64_t h, int64_t k, int ar, int ak, int br, int bk, const void* bias,
                                int bias_dtype, void* aux, void* out, int out_dtype, int activation, int backward,
                                viola_stream_t stream_) {
    hipStream_t stream = viola_enter(stream_);
    VIOLA_CHECK_ARG(viola_is_fp8(a_dtype) && viola_is_fp8(b_dtype) && viola_is_float(out_dtype));
    VIOLA_CHECK_ARG(m >= 0 && h >= 0 && k >= 0 && ar > 0 && br > 0 && pow2(ak) && pow2(bk) && ak >= 32 && bk >= 32);
    VIOLA_CHECK_ARG(activation >= VIOLA_SILU && activation <= VIOLA_RELU && (!bias || viola_is_float(bias_dtype)));
    if (m == 0 || h == 0) return 0;
    VIOLA_CHECK_ARG(out && (k == 0 || (a && b && sa && sb)) && (!backward || aux));
    GemmArgs p = {};
    p.a = static_cast<const uint8_t*>(a); p.b = static_cast<const uint8_t*>(b); p.sa = sa; p.sb = sb;
    p.bias = backward ? nullptr : bias; p.out = out; p.aux = aux; p.m = m; p.n = h; p.k = k; p.lda = k; p.ldb = k;
    p.ldsa = (k + ak - 1) / ak; p.ldsb = (k + bk - 1) / bk; p.ldo = backward ? 2 * h : h;
    p.ar = ar; p.br = br; p.ak_shift = shift_of(ak); p.bk_shift = shift_of(bk); p.activation = activation;
    const bool vec = k % 16 == 0 && aligned16(a) && aligned16(b);
    const int64_t gy = (m + BM - 1) / BM;
    VIOLA_CHECK_ARG(gy <= 65535);
    if (backward) {
        const bool rowscale = br % 32 != 0;
        return launch_out<MODE_GATED_BWD>(p, a_dtype, b_dtype, bias_dtype, out_dtype, rowscale, vec,
                                          dim3((unsigned)((h + BN - 1) / BN), (unsigned)gy), stream);
    }
    const bool rowscale = br % 32 != 0 || h % 32 != 0;
    return launch_out<MODE_GATED_FWD>(p, a_dtype, b_dtype, bias_dtype, out_dtype, rowscale, vec,
                                      dim3((unsigned)((h + BN / 2 - 1) / (BN / 2)), (unsigned)gy), stream);
}

// viola_mx_gated_gemm forward whose h leaves the kernel as FP8 codes with E8M0 scales in both layouts.
extern "C" int viola_mx_gated_gemm_encode(const void* a, int a_dtype, const void* b, int b_dtype, const uint8_t* sa, const uint8_t* sb,
                                          int64_t m, int64_t h, int64_t k, int ar, int br, const void* bias, int bias_dtype,
                                          void* aux, int aux_dtype, void* enc, uint8_t* enc_scale, void* enc_t,
                                          uint8_t* enc_t_scale, int enc_dtype, float limit, int activation,
                                          viola_stream_t stream_) {
    hipStream_t stream = viola_enter(stream_);
    VIOLA_CHECK_ARG(viola_is_fp8(a_dtype) && viola_is_fp8(b_dtype) && viola_is_float(aux_dtype) && viola_is_fp8(enc_dtype));
    VIOLA_CHECK_ARG(m >= 0 && h >= 0 && k >= 0 && ar > 0 && br > 0 && limit > 0.0f);
    VIOLA_CHECK_ARG(activation >= VIOLA_SILU && activation <= VIOLA_RELU && (!bias || viola_is_float(bias_dtype)));
    if (m == 0 || h == 0) return 0;
    VIOLA_CHECK_ARG(enc && enc_scale && (!enc_t || enc_t_scale) && (k == 0 || (a && b && sa && sb)));
    const int64_t gy = (m + BM - 1) / BM;
    VIOLA_CHECK_ARG(gy <= 65535);
    if (k == 0 || k % 128 != 0 || !aligned16(a) || !aligned16(b) || reinterpret_cast<uintptr_t>(sa) % 4 != 0 ||
        reinterpret_cast<uintptr_t>(sb) % 4 != 0 || 2 * h * k >= (1ll << 31) || (int64_t)BM * k >= (1ll << 31) ||
        (br != 1 && br % 32 != 0) || h % br != 0 || h % 32 != 0 || m % 32 != 0 || !aligned16(aux) || !aligned16(enc) ||
        !aligned16(enc_t))
        return VIOLA_EUNSUPPORTED;
    if (aux && enc_t && aux_dtype != VIOLA_F32 && choose_scaled_tile(m, 2 * h, k, false) != SCALED_TILE_FAST) {
        // the plain GEMM on the tile that suits it writes [g | u], one pass over it writes the codes of h in both layouts
        // (the encoding epilogue does not fit the large tiles' registers; 2.0 ms against 2.5 ms at 16384 x 4096 -> 11008)
        const int status = mx_gemm(a, a_dtype, b, b_dtype, sa, sb, m, 2 * h, k, ar, br, bias, bias_dtype, aux, 2 * h, aux_dtype, stream);
        if (status) return status;
        return viola_gated_quantize_dual(aux, aux_dtype, m, h, activation, enc, enc_scale, enc_t, enc_t_scale, enc_dtype, 32, limit,
                                         VIOLA_SCALE_E8M0, stream_);
    }
    GemmArgs p = {};
    p.a = static_cast<const uint8_t*>(a); p.b = static_cast<const uint8_t*>(b);
    p.sa = reinterpret_cast<const float*>(sa); p.sb = reinterpret_cast<const float*>(sb);
    p.bias = bias; p.out = nullptr; p.aux = aux; p.m = m; p.n = h; p.k = k; p.lda = k; p.ldb = k; p.ldo = h;
    p.activation = activation;
    p.ldsa = k / 32; p.ldsb = k / 32; p.ar = ar; p.br = br; p.ak_shift = 5; p.bk_shift = 5;
    p.enc = static_cast<uint8_t*>(enc); p.enc_scale = enc_scale; p.enc_t = static_cast<uint8_t*>(enc_t); p.enc_t_scale = enc_t_scale;
    p.enc_limit = limit; p.enc_bf8 = enc_dtype == VIOLA_E5M2;
    return launch_mx_gemm_fast(p, MODE_GATED_FWD, a_dtype, b_dtype, bias_dtype, aux_dtype,
                               dim3((unsigned)((h + BN / 2 - 1) / (BN / 2)), (unsigned)gy), stream);
}

extern "C" int viola_varlen_group_gemm(const void* a, int a_dtype, const void* b, int b_dtype, const float* sa,
                                       const float* sb, const int64_t* offsets, int groups, int64_t m_total, int64_t n,
                                       int64_t k, int ar, int ak, int br, int bk, int64_t b_group_stride,
                                       int64_t sb_group_stride, void* out, int out_dtype, viola_stream_t stream_) {
    hipStream_t stream = viola_enter(stream_);
    VIOLA_CHECK_ARG(viola_is_fp8(a_dtype) && viola_is_fp8(b_dtype) && viola_is_float(out_dtype));
    VIOLA_CHECK_ARG(m_total >= 0 && n >= 0 && k >= 0 && groups > 0 && ar == 1 && br > 0 && pow2(ak) && pow2(bk) && ak >= 32 && bk >= 32);
    if (m_total == 0 || n == 0) return 0;
    VIOLA_CHECK_ARG(out && offsets && (k == 0 || (a && b && sa && sb)));
    const int64_t gy = (m_total + BM - 1) / BM + groups;
    VIOLA_CHECK_ARG(gy <= 65535);
    GemmArgs p = {};
    p.a = static_cast<const uint8_t*>(a); p.b = static_cast<const uint8_t*>(b); p.sa = sa; p.sb = sb;
    p.out = out; p.m = m_total; p.n = n; p.k = k; p.lda = k; p.ldb = k;
    p.ldsa = (k + ak - 1) / ak; p.ldsb = (k + bk - 1) / bk; p.ldo = n;
    p.ar = ar; p.br = br; p.ak_shift = shift_of(ak); p.bk_shift = shift_of(bk);
    p.offsets = offsets; p.groups = groups; p.b_group_stride = b_group_stride; p.sb_group_stride = sb_group_stride;
    const bool vec = k % 16 == 0 && aligned16(a) && aligned16(b) && b_group_stride % 16 == 0;
    const bool rowscale = br % 32 != 0;
    return launch_out<MODE_PLAIN>(p, a_dtype, b_dtype, VIOLA_F32, out_dtype, rowscale, vec,
                                  dim3((unsigned)((n + BN - 1) / BN), (unsigned)gy), stream);
}

extern "C" int viola_varlen_wgrad_gemm(const void* at, int a_dtype, const void* bt, int b_dtype, const float* sat,
                                       const float* sbt, const int64_t* poffsets, int groups, int64_t t_total, int64_t n,
                                       int64_t kout, void* out, int out_dtype, viola_stream_t stream_) {
    hipStream_t stream = viola_enter(stream_);
    VIOLA_CHECK_ARG(viola_is_fp8(a_dtype) && viola_is_fp8(b_dtype) && viola_is_float(out_dtype));
    VIOLA_CHECK_ARG(t_total >= 0 && t_total % 32 == 0 && n >= 0 && kout >= 0 && groups > 0 && groups <= 65535);
    if (n == 0 || kout == 0) return 0;
    VIOLA_CHECK_ARG(out && poffsets && (t_total == 0 || (at && bt && sat && sbt)));
    const int64_t gy = (n + BM - 1) / BM;
    VIOLA_CHECK_ARG(gy <= 65535);
    GemmArgs p = {};
    p.a = static_cast<const uint8_t*>(at); p.b = static_cast<const uint8_t*>(bt); p.sa = sat; p.sb = sbt;
    p.out = out; p.m = n; p.n = kout; p.k = t_total; p.lda = t_total; p.ldb = t_total;
    p.ldsa = t_total / 32; p.ldsb = t_total / 32; p.ldo = kout;
    p.ar = 1; p.br = 1; p.ak_shift = 5; p.bk_shift = 5;
    p.koffsets = poffsets; p.out_group_stride = n * kout;
    const bool vec = t_total % 16 == 0 && aligned16(at) && aligned16(bt);
    return launch_out<MODE_PLAIN>(p, a_dtype, b_dtype, VIOLA_F32, out_dtype, true, vec,
                                  dim3((unsigned)((kout + BN - 1) / BN), (unsigned)gy, (unsigned)groups), stream);
}
