// Linear products too small to fill the chip with tiles of 128 x 64 (decoding, short sequences, narrow layers): out [m, n] = x W^T +
// bias on tiles of 16 or 32 a side whose k range all waves of a block share, x quantized on the way in where that pays.
#include "common.hpp"

namespace viola {

// Most waves of a block: with two tiles of either kind a lane needs more than a quarter of the registers.
constexpr int skinny_waves(int mt, int nt) { return mt * nt == 1 ? 16 : 8; }

struct SkinnyArgs {
    const void* x; const uint8_t* w; const void* sw; const float* sx;
    const void* bias; void* out;
    int64_t n, k, ldsw;
    int m, bias_dtype, out_dtype, e8m0;
    float limit;
    float* history; int64_t slot; float* scale;    // per-tensor scale formed here: where the maximum and the scale go
};

// The lanes of the two halves (or, ROW: of the even and odd rows of 16 lanes) exchanged: a gets b's first part behind its own,
// b gets a's second part before its own.
template <bool ROW>
__device__ __forceinline__ void swap_lanes(uint32_t& a, uint32_t& b) {
    const auto r = ROW ? __builtin_amdgcn_permlane16_swap(a, b, false, false) : __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
__device__ __forceinline__ uint32_t max_of_rows(uint32_t v) {               // over lanes l and l ^ 16
    uint32_t w = v;
    swap_lanes<true>(v, w);
    return v > w ? v : w;
}

// The scales of the two groups of step `step` of one row of `count` scales (an odd row's last step has one).
__device__ __forceinline__ void two_scales(const void* scales, int64_t row, int64_t step, int64_t count, int e8m0, float (&s)[2]) {
    const int64_t at = row * count + 2 * step;
    if (count % 2 == 0) {
        if (e8m0) {
            const uint32_t pair = reinterpret_cast<const uint16_t*>(scales)[at / 2];
            s[0] = __uint_as_float((pair & 0xffu) << 23);
            s[1] = __uint_as_float((pair >> 8) << 23);
        } else {
            const float2 pair = reinterpret_cast<const float2*>(scales)[at / 2];
            s[0] = pair.x;
            s[1] = pair.y;
        }
    } else {
        s[0] = get_scale(static_cast<const float*>(scales), at, e8m0);
        s[1] = get_scale(static_cast<const float*>(scales), 2 * step + 1 < count ? at + 1 : at, e8m0);
    }
}

template <typename TW, typename TX>
__device__ __forceinline__ f32x4_t skinny_mfma(uint2 w, uint2 x, f32x4_t c) {
    constexpr bool W5 = std::is_same<TW, e5m2_t>::value, X5 = std::is_same<TX, e5m2_t>::value;
    const long a = __builtin_bit_cast(long, w), b = __builtin_bit_cast(long, x);
    if constexpr (W5 && X5) return __builtin_amdgcn_mfma_f32_16x16x32_bf8_bf8(a, b, c, 0, 0, 0);
    else if constexpr (W5) return __builtin_amdgcn_mfma_f32_16x16x32_bf8_fp8(a, b, c, 0, 0, 0);
    else if constexpr (X5) return __builtin_amdgcn_mfma_f32_16x16x32_fp8_bf8(a, b, c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(a, b, c, 0, 0, 0);
}

// Sixteen 16-bit values -> codes, for a group (or tensor) whose scale is s.
template <typename TIn>
__device__ __forceinline__ void skinny_widen(const uint32_t (&words)[4], float (&v)[8]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = widen16<TIn>(words[i] & 0xffffu);
        v[2 * i + 1] = widen16<TIn>(words[i] >> 16);
    }
}
template <typename TIn, typename TOut>
__device__ __noinline__ uint2 skinny_encode_exact(uint32_t x, uint32_t y, uint32_t z, uint32_t w, float s, float limit) {
    float v[8];
    const uint32_t words[4] = {x, y, z, w};
    skinny_widen<TIn>(words, v);
    return encode8<TOut>(v, s, limit, SharedDivisor(s, __uint_as_float(0x7fc00000u)));
}
template <typename TIn, typename TOut>
__device__ __forceinline__ void skinny_encode(const uint4 (&raw)[2], float s, float limit, bool e8m0, bool nonfinite, uint2 (&codes)[2]) {
    const SharedDivisor d(s, nonfinite ? __uint_as_float(0x7fc00000u) : 0.0f);
    const bool exact = __builtin_amdgcn_ballot_w64(!d.fast) != 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t words[4] = {raw[h].x, raw[h].y, raw[h].z, raw[h].w};
        float v[8];
        skinny_widen<TIn>(words, v);
        if (exact) {
            codes[h] = skinny_encode_exact<TIn, TOut>(words[0], words[1], words[2], words[3], s, limit);
        } else if (e8m0) {
            const PowerDivisor p{d.r};
            codes[h] = make_uint2(fast_encode4<TOut>(p, limit, v[0], v[1], v[2], v[3]), fast_encode4<TOut>(p, limit, v[4], v[5], v[6], v[7]));
        } else {
            codes[h] = make_uint2(fast_encode4<TOut>(d, limit, v[0], v[1], v[2], v[3]), fast_encode4<TOut>(d, limit, v[4], v[5], v[6], v[7]));
        }
    }
}

// What bounds it: one read of W, and below about 16 MB of W the latency of a launch that reads anything at all. So nothing is
// staged: a block owns a tile of 16 MT x 16 NT, its waves a share of k each, and a lane loads its 16-byte pieces of W and its 16 values of
// x straight into registers, the next step's loads in flight under the arithmetic of this one. A step is 64 k: lane l has row
// l % 16, k 16 (l / 16) .. + 15 of both operands, so one exchange between the half waves puts the first scale group into one
// v_mfma_f32_16x16x32 and the second into another (k in the same new order on both sides). Every block quantizes its rows
// of x for itself, which is why it has few of them. A lane quantizes the row of x whose column of the result it
// accumulates, so scales stay in their lanes. The waves' sums meet in LDS.
//   GROUPED: a scale per row and 32 k of x and per 32 x 32 block of W (FP32 or E8M0), applied as acc * (sx sw) per group.
//   else one scale per tensor: acc runs through, (sum * sx) * sw at the end. CODED: x arrives as codes with its scale; otherwise
//   every block takes the maximum of x (the launcher bounds its size) and block 0 records it.
// 8 x 1024 -> 4096, grouped: 2.3 (quantizer) + 9.9 -> 5.3 us. As codes, against 128 x 64 tiles with their k split in two:
// 256 x 4096 -> 256 grouped 22.2 -> 8.9 us, per-tensor 11.9 -> 6.9; 64 x 1024 -> 1024 9.2 -> 4.4 and 6.2 -> 4.1; 128 x 4096 -> 2048 22.5 ->
// 15.3 and 11.9 -> 10.5.
// TIn: type of x's values (CODED: its format, TX); TX, TW: formats of the two operands.
template <typename TIn, typename TX, typename TW, bool GROUPED, int MT, int NT>
__global__ __launch_bounds__(64 * skinny_waves(MT, NT)) void skinny_linear(const SkinnyArgs p) {
    constexpr int U = 2;                                                     // steps loaded ahead
    constexpr bool CODED = std::is_same<TIn, TX>::value;
    constexpr uint32_t MAGNITUDE = 0x7fff7fffu, INF16 = std::is_same<TIn, bf16_t>::value ? 0x7f80u : 0x7c00u;   // 16-bit x
    extern __shared__ __attribute__((aligned(16))) char shared[];
    f32x4_t* sums = reinterpret_cast<f32x4_t*>(shared);                      // [wave][tile][lane]
    const int lane = threadIdx.x % WAVE, waves = blockDim.x / WAVE;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int l16 = lane & 15, quarter = lane >> 4;
    const int64_t n0 = (int64_t)blockIdx.x * 16 * NT;
    const int m0 = (int)blockIdx.y * 16 * MT;
    const int64_t steps = (p.k + 63) / 64, begin = steps * wave / waves, end = steps * (wave + 1) / waves;

    const uint8_t* wrow[NT];
    int64_t wscale[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int64_t row = n0 + 16 * t + l16, first = n0 + 16 * t;
        wrow[t] = p.w + (row < p.n ? row : p.n - 1) * p.k;
        wscale[t] = (first < p.n ? first : p.n - 1) / 32;
    }
    constexpr int XB = CODED ? 1 : 2;                                        // bytes per value of x
    const uint8_t* xrow[MT];
    int64_t xscale[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int64_t row = m0 + 16 * t + l16 < p.m ? m0 + 16 * t + l16 : p.m - 1;
        xrow[t] = static_cast<const uint8_t*>(p.x) + row * p.k * XB;
        xscale[t] = row;
    }

    struct Batch { uint4 w[NT][U], x[MT][U][XB]; float sw[NT][U][2], sx[MT][U][2]; };
    auto load = [&](Batch& b, int64_t g) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t step = g + u < end ? g + u : end - 1;
            const int64_t at = step * 64 + quarter * 16;
            const bool inside = at < p.k;                                    // k % 16 == 0: pieces are whole
            const int64_t from = inside ? at : 0;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                b.w[t][u] = *reinterpret_cast<const uint4*>(wrow[t] + from);
                if (!inside) b.w[t][u] = make_uint4(0, 0, 0, 0);
                if constexpr (GROUPED) two_scales(p.sw, wscale[t], step, p.ldsw, p.e8m0, b.sw[t][u]);
            }
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int h = 0; h < XB; ++h) {
                    b.x[t][u][h] = *reinterpret_cast<const uint4*>(xrow[t] + from * XB + 16 * h);
                    if (!inside) b.x[t][u][h] = make_uint4(0, 0, 0, 0);
                }
            if constexpr (GROUPED && CODED)
#pragma unroll
                for (int t = 0; t < MT; ++t) two_scales(p.sx, xscale[t], step, p.ldsw, p.e8m0, b.sx[t][u]);
        }
    };
    Batch now;
    if (begin < end) load(now, begin);

    float s_tensor = 0.0f;
    if constexpr (!GROUPED && !CODED) {
        // the whole tensor's maximum, by every block (m k is at most a few loads per thread)
        float amax = 0.0f;
        for (int64_t i = threadIdx.x; i < p.m * p.k / 8; i += blockDim.x) {
            const uint4 raw = reinterpret_cast<const uint4*>(p.x)[i];
            const uint32_t words[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) amax = fmaxf(amax, fmaxf(fabsf(widen16<TIn>(words[e] & 0xffffu)), fabsf(widen16<TIn>(words[e] >> 16))));
        }
        amax = wave_max(amax);
        float* part = reinterpret_cast<float*>(shared);
        if (lane == 0) part[wave] = amax;
        __syncthreads();
        for (int i = 0; i < waves; ++i) amax = fmaxf(amax, part[i]);
        s_tensor = scale_of(amax, p.limit);
        if (blockIdx.x + blockIdx.y == 0 && threadIdx.x == 0) {
            if (p.scale) p.scale[0] = s_tensor;
            p.history[p.slot] = amax;
        }
        __syncthreads();                                                     // part becomes sums
    } else if constexpr (!GROUPED) {
        s_tensor = p.sx[0];
    }

    f32x4_t total[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) total[i][j] = f32x4_t{0, 0, 0, 0};
    for (int64_t g = begin; g < end; g += U) {
        Batch next;
        if (g + U < end) load(next, g + U);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (g + u >= end) break;
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                uint4& w = now.w[j][u];
                if constexpr (GROUPED) {
                    swap_lanes<false>(w.x, w.z);
                    swap_lanes<false>(w.y, w.w);
                }
            }
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                uint2 codes[2];
                float sx[2] = {0.0f, 0.0f};
                if constexpr (CODED) {
                    codes[0] = make_uint2(now.x[i][u][0].x, now.x[i][u][0].y);
                    codes[1] = make_uint2(now.x[i][u][0].z, now.x[i][u][0].w);
                    sx[0] = now.sx[i][u][0];
                    sx[1] = now.sx[i][u][1];
                } else {
                    const uint4 raw[2] = {now.x[i][u][0], now.x[i][u][1]};
                    uint32_t top = 0;
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        top = pk_max_u16(top, pk_max_u16(pk_max_u16(raw[h].x & MAGNITUDE, raw[h].y & MAGNITUDE), pk_max_u16(raw[h].z & MAGNITUDE, raw[h].w & MAGNITUDE)));
                    top = (top & 0xffffu) > (top >> 16) ? (top & 0xffffu) : (top >> 16);
                    float s = s_tensor;
                    if constexpr (GROUPED) {
                        top = max_of_rows(top);                              // a group is 16 values of two lanes
                        float amax = widen16<TIn>(top);
                        if (__builtin_amdgcn_ballot_w64(top >= INF16) != 0) {   // an Inf or a NaN in some group: the maximum ignores NaN
                            float own = 0.0f;
#pragma unroll
                            for (int h = 0; h < 2; ++h) {
                                const uint32_t words[4] = {raw[h].x, raw[h].y, raw[h].z, raw[h].w};
                                float v[8];
                                skinny_widen<TIn>(words, v);
#pragma unroll
                                for (int e = 0; e < 8; ++e) own = fmaxf(own, fabsf(v[e]));
                            }
                            amax = __uint_as_float(max_of_rows(__float_as_uint(own)));
                        }
                        s = group_scale(amax, p.limit, p.e8m0);
                        uint32_t first = __float_as_uint(s), second = first;
                        swap_lanes<false>(first, second);                    // the lower half's group everywhere, the upper half's
                        sx[0] = __uint_as_float(first);
                        sx[1] = __uint_as_float(second);
                    }
                    skinny_encode<TIn, TX>(raw, s, p.limit, GROUPED && p.e8m0, top >= INF16, codes);
                }
                if constexpr (GROUPED) {
                    swap_lanes<false>(codes[0].x, codes[1].x);
                    swap_lanes<false>(codes[0].y, codes[1].y);
                }
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const uint4 w = now.w[j][u];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const uint2 piece = h ? make_uint2(w.z, w.w) : make_uint2(w.x, w.y);
                        if constexpr (GROUPED) {
                            const f32x4_t part = skinny_mfma<TW, TX>(piece, codes[h], f32x4_t{0, 0, 0, 0});
                            const float s = sx[h] * now.sw[j][u][h];
#pragma unroll
                            for (int r = 0; r < 4; ++r) total[i][j][r] = fmaf(part[r], s, total[i][j][r]);
                        } else {
                            total[i][j] = skinny_mfma<TW, TX>(piece, codes[h], total[i][j]);
                        }
                    }
                }
            }
        }
        now = next;
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) sums[(wave * MT * NT + i * NT + j) * WAVE + lane] = total[i][j];
    __syncthreads();
    for (int tile = wave; tile < MT * NT; tile += waves) {
        f32x4_t v = {0, 0, 0, 0};
        for (int i = 0; i < waves; ++i) v += sums[(i * MT * NT + tile) * WAVE + lane];
        // lane l: row l % 16 of x, columns 4 (l / 16) .. + 3 of the tile
        const int row = m0 + tile / NT * 16 + l16;
        const int64_t col = n0 + tile % NT * 16 + quarter * 4;
        if (row >= p.m || col >= p.n) continue;
        float f[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            f[r] = v[r];
            if constexpr (!GROUPED) f[r] = (f[r] * s_tensor) * static_cast<const float*>(p.sw)[0];
            if (p.bias && col + r < p.n) f[r] += load_float(p.bias, col + r, p.bias_dtype);
        }
        const int64_t at = (int64_t)row * p.n + col;
        if (p.n % 4 == 0 && p.out_dtype == VIOLA_BF16) *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p.out) + at) = make_uint2(f32_to_bf16x2_bits(f[0], f[1]), f32_to_bf16x2_bits(f[2], f[3]));
        else if (p.n % 4 == 0 && p.out_dtype == VIOLA_F16) *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p.out) + at) = make_uint2(narrow16<f16_t>(f[0]) | narrow16<f16_t>(f[1]) << 16, narrow16<f16_t>(f[2]) | narrow16<f16_t>(f[3]) << 16);
        else for (int r = 0; r < 4 && col + r < p.n; ++r) store_float(p.out, at + r, p.out_dtype, f[r]);
    }
}

// The tile: the smallest that leaves one block per CU (256). Past that a second round of blocks reads W and x again and larger
// tiles from LDS win (256 x 4096 -> 1024: 32 x 32 tiles 28 us per round pair, 128 x 64 tiles 22 us), except for up to 32 rows,
// where those would be mostly padding. False: not this kernel.
static bool skinny_tile(int64_t m, int64_t n, int& mt, int& nt) {
    auto fits = [&](int rows, int cols) { return ((m + 16 * rows - 1) / (16 * rows)) * ((n + 16 * cols - 1) / (16 * cols)) <= 256; };
    mt = nt = 1;
    if (fits(1, 1)) return true;
    nt = 2;
    if (fits(1, 2)) return true;
    mt = m > 16 ? 2 : 1;
    return fits(2, 2) || m <= 32;
}

template <typename TIn, typename TX, typename TW, bool GROUPED>
static int launch_skinny(const SkinnyArgs& p, int mt, int nt, hipStream_t stream) {
    // waves: two steps of k for each (one while there are few blocks)
    const int64_t blocks_n = (p.n + 16 * nt - 1) / (16 * nt), blocks_m = (p.m + 16 * mt - 1) / (16 * mt), steps = (p.k + 63) / 64;
    int waves = skinny_waves(mt, nt);
    while (waves > 1 && steps < waves * (blocks_n * blocks_m < 128 ? 1 : 2)) waves /= 2;
    const dim3 grid((unsigned)blocks_n, (unsigned)blocks_m), block((unsigned)(64 * waves));
    const size_t lds = (size_t)waves * mt * nt * 1024;
#define VIOLA_SKINNY(MT, NT) VIOLA_LAUNCH((skinny_linear<TIn, TX, TW, GROUPED, MT, NT>), grid, block, lds, stream, p)
    if (mt == 1 && nt == 1) VIOLA_SKINNY(1, 1);
    else if (mt == 1) VIOLA_SKINNY(1, 2);
    else VIOLA_SKINNY(2, 2);
#undef VIOLA_SKINNY
    return viola_launch_status();
}

}  // namespace viola

using namespace viola;

extern "C" int viola_skinny_linear(const void* x, int x_dtype, const float* sx, int64_t m, int64_t k, const void* w, int w_dtype, const void* sw,
                                   int grouped, int64_t n, float limit, int scale_format, float* history, int64_t slot, float* scale, const void* bias,
                                   int bias_dtype, void* out, int out_dtype, viola_stream_t stream_) {
    hipStream_t stream = viola_enter(stream_);
    const bool coded = viola_is_fp8(x_dtype);
    VIOLA_CHECK_ARG((coded || viola_is_float(x_dtype)) && viola_is_fp8(w_dtype) && viola_is_float(out_dtype) && (!bias || viola_is_float(bias_dtype)));
    VIOLA_CHECK_ARG(m >= 0 && n >= 0 && k >= 0 && limit > 0.0f && (scale_format == VIOLA_SCALE_F32 || scale_format == VIOLA_SCALE_E8M0));
    if (m == 0 || n == 0) return 0;
    VIOLA_CHECK_ARG(out && sw && (k == 0 || (x && w)));
    int mt, nt;
    if (m > 4096 || !skinny_tile(m, n, mt, nt) || (!coded && m > 32 && mt > 1) || k == 0 || k % 16 != 0 || k >= (1 << 30) || n >= (1ll << 31) || x_dtype == VIOLA_F32 ||
        reinterpret_cast<uintptr_t>(x) % 16 != 0 || reinterpret_cast<uintptr_t>(w) % 16 != 0 || reinterpret_cast<uintptr_t>(out) % 8 != 0 ||
        (grouped && (reinterpret_cast<uintptr_t>(sw) % 8 != 0 || reinterpret_cast<uintptr_t>(sx) % 8 != 0)))
        return VIOLA_EUNSUPPORTED;
    if (coded) VIOLA_CHECK_ARG(sx);
    else if (!grouped) VIOLA_CHECK_ARG(history && slot >= 0);
    SkinnyArgs p = {};
    p.x = x; p.w = static_cast<const uint8_t*>(w); p.sw = sw; p.sx = sx; p.bias = bias; p.out = out;
    p.n = n; p.k = k; p.ldsw = (k + 31) / 32; p.m = (int)m; p.bias_dtype = bias_dtype; p.out_dtype = out_dtype;
    p.e8m0 = scale_format == VIOLA_SCALE_E8M0; p.limit = limit; p.history = history; p.slot = slot; p.scale = scale;
    auto launch = [&](auto in, auto x_format, auto w_format) {
        using TIn = decltype(in);
        using TX = decltype(x_format);
        using TW = decltype(w_format);
        return grouped ? launch_skinny<TIn, TX, TW, true>(p, mt, nt, stream) : launch_skinny<TIn, TX, TW, false>(p, mt, nt, stream);
    };
    auto by_weight = [&](auto x_format) { return w_dtype == VIOLA_E4M3 ? launch(x_format, x_format, e4m3_t{}) : launch(x_format, x_format, e5m2_t{}); };
    auto by_format = [&](auto in) { return w_dtype == VIOLA_E4M3 ? launch(in, e4m3_t{}, e4m3_t{}) : launch(in, e5m2_t{}, e5m2_t{}); };
    if (coded) return x_dtype == VIOLA_E4M3 ? by_weight(e4m3_t{}) : by_weight(e5m2_t{});
    return x_dtype == VIOLA_F16 ? by_format(f16_t{}) : by_format(bf16_t{});
}
