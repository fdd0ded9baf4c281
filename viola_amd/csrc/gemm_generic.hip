// Grouped-scale FP8 GEMM for gfx950 ("NT": out[m, n] = sum_k a[m, k] * b[n, k]) with FP32 scales
// per (row group, 32-wide K group) on both operands.
//
// Per 32-wide K group the raw code product is formed on the matrix cores
// (v_mfma_f32_32x32x16_fp8_fp8 twice) and folded into an FP32 total with one VALU FMA per output
// element: total += acc * (sa * sb). The FP32 scales cannot be applied inside a wider MFMA, so the
// K = 32 instructions are the ones that fit this contract.
//
// Orientation: the B matrix (rows n) is fed as the MFMA "A" operand and the A matrix (rows m) as
// the MFMA "B" operand, so a lane's 16 accumulators of a 32 x 32 tile share one m and cover 16
// values of n inside one 32-row block of b. With 2-D weight blocks (br a multiple of 32) the scale
// product sa[m] * sb[block] is then a single per-lane scalar per K group.
//
// Block: 256 threads = 2 x 2 wavefronts, tile 128 (m) x 128 (b rows) x 64 (k), two LDS stages,
// global loads for chunk i+1 issued before the math of chunk i.
//
// One kernel template serves: the plain GEMM, the gated-MLP forward (two 64-row panels of b, gate
// and up, sharing a; epilogue act(g)*u), the gated-MLP backward (epilogue reads g,u and writes
// [d*u*act'(g), d*act(g)]), the variable-group row-range GEMM and the variable-group wgrad.
#include "gemm_args.hpp"

namespace viola {

constexpr int BK = 64, LDK = BK + 8, KG = BK / 32;

template <bool A_BF8, bool B_BF8>
__device__ __forceinline__ f32x16 mfma32(long x, long y, f32x16 c) {
    // x: 8 codes of the b matrix (MFMA srcA), y: 8 codes of the a matrix (MFMA srcB)
    if constexpr (!B_BF8 && !A_BF8) return __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(x, y, c, 0, 0, 0);
    else if constexpr (!B_BF8 && A_BF8) return __builtin_amdgcn_mfma_f32_32x32x16_fp8_bf8(x, y, c, 0, 0, 0);
    else if constexpr (B_BF8 && !A_BF8) return __builtin_amdgcn_mfma_f32_32x32x16_bf8_fp8(x, y, c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_32x32x16_bf8_bf8(x, y, c, 0, 0, 0);
}

template <typename TO> __device__ __forceinline__ float round_through(float v) { return to_f32(from_f32<TO>(v)); }

// A_BF8/B_BF8: operand formats (false = e4m3, true = e5m2). B_ROWSCALE: b scales vary inside a 32-row block.
// VEC: 16-byte global loads are legal (k ranges and row strides multiples of 16, aligned bases).
//
// HALF models the reference's accum_dtype="fp16" (viola/nn/_grouped_kernels.py:268-292, _linear_kernels.py:139-155,
// :198-211): its FP8 tensor-core instruction covers 32 k and, with an FP16 accumulator, returns
// fp16(accumulator + the 32 products); the accumulator is cleared after `half_period` k, when it is added to a
// running total held in FP32 or bf16 (rounded after every addition). HALF == 1 is the grouped recipe (a period is one
// scale group: the partial is scaled by sa * sb as it is added, (partial * sa) * sb), HALF == 2 the per-tensor recipe
// (scales applied to the finished total; half_period == 0: one partial over the whole k range and no total). Here the
// 32 products are summed in FP32 by the MFMA and rounded once, which is that instruction's best case; where the
// hardware's own sum is coarser the reference's results differ, inside the bound its checks allow (.01).
template <int MODE, bool A_BF8, bool B_BF8, bool B_ROWSCALE, bool VEC, typename TO, int HALF = 0>
__global__ __launch_bounds__(256, 2) void group_gemm_kernel(GemmArgs p, int bias_dtype) {
    static_assert(HALF == 0 || MODE == MODE_PLAIN, "the FP16-accumulator model is built for the plain product");
    __shared__ __attribute__((aligned(16))) uint8_t lds_a[2][BM * LDK];
    __shared__ __attribute__((aligned(16))) uint8_t lds_b[2][BN * LDK];
    __shared__ __attribute__((aligned(16))) float lds_sa[2][KG][BM];
    __shared__ __attribute__((aligned(16))) float lds_sb[2][KG][BN];

    constexpr int PANEL = MODE == MODE_GATED_FWD ? BN / 2 : BN;       // b rows per panel in the tile
    const int tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
    const int wm = wave / 2, wn = wave % 2;
    const int l32 = lane % 32, lhi = lane / 32;

    // ---- which problem / tile
    int64_t m_begin = (int64_t)blockIdx.y * BM, m_end = p.m;
    int64_t k_begin = 0, k_end = p.k;
    const uint8_t* bptr = p.b;
    const float* sbptr = p.sb;
    uint8_t* outptr = static_cast<uint8_t*>(p.out);
    if (p.offsets) {
        int64_t tile = blockIdx.y;
        int g = 0;
        bool found = false;
        for (; g < p.groups; ++g) {
            const int64_t lo = p.offsets[g], hi = p.offsets[g + 1];
            const int64_t tiles = (hi - lo + BM - 1) / BM;
            if (tile < tiles) { m_begin = lo + tile * BM; m_end = hi; found = true; break; }
            tile -= tiles;
        }
        if (!found) return;
        bptr += (int64_t)g * p.b_group_stride;
        sbptr += (int64_t)g * p.sb_group_stride;
    }
    if (p.koffsets) {
        const int g = blockIdx.z;
        k_begin = p.koffsets[g];
        k_end = p.koffsets[g + 1];
        outptr += (int64_t)g * p.out_group_stride * (int64_t)sizeof(TO);
    }
    if (m_begin >= m_end) return;
    const int64_t n_begin = (int64_t)blockIdx.x * PANEL;

    // global row of tile-local b row `lr`
    auto b_row = [&](int lr) -> int64_t {
        if constexpr (MODE == MODE_GATED_FWD) return (int64_t)(lr / PANEL) * p.n + n_begin + lr % PANEL;
        else return n_begin + lr;
    };
    const int64_t b_rows_total = MODE == MODE_GATED_FWD ? 2 * p.n : p.n;
    auto b_row_valid = [&](int lr) -> bool {
        if constexpr (MODE == MODE_GATED_FWD) return n_begin + lr % PANEL < p.n;
        else return n_begin + lr < p.n;
    };

    // ---- staging registers for the next chunk
    uint4 ra[2], rb[2];
    float rsa, rsb;
    auto fetch = [&](int64_t k0) {
#pragma unroll
        for (int it = 0; it < 2; ++it) {
            const int id = it * 256 + tid;
            const int lr = id / 4, c = id % 4;
            const int64_t kk = k0 + c * 16;
            int64_t am = m_begin + lr;
            am = am < m_end ? am : m_end - 1;
            int64_t bn = b_row(lr);
            bn = bn < b_rows_total ? bn : b_rows_total - 1;
            if constexpr (VEC) {
                ra[it] = kk < k_end ? *reinterpret_cast<const uint4*>(p.a + am * p.lda + kk) : make_uint4(0, 0, 0, 0);
                rb[it] = kk < k_end ? *reinterpret_cast<const uint4*>(bptr + bn * p.ldb + kk) : make_uint4(0, 0, 0, 0);
            } else {
                uint32_t wa[4] = {0, 0, 0, 0}, wb[4] = {0, 0, 0, 0};
                for (int i = 0; i < 16; ++i) {
                    if (kk + i < k_end) {
                        wa[i / 4] |= (uint32_t)p.a[am * p.lda + kk + i] << (8 * (i % 4));
                        wb[i / 4] |= (uint32_t)bptr[bn * p.ldb + kk + i] << (8 * (i % 4));
                    }
                }
                ra[it] = make_uint4(wa[0], wa[1], wa[2], wa[3]);
                rb[it] = make_uint4(wb[0], wb[1], wb[2], wb[3]);
            }
        }
        {
            const int kg = tid / BM, lr = tid % BM;                    // KG * 128 == 256 entries each
            const int64_t kk = k0 + kg * 32;
            int64_t am = m_begin + lr;
            am = am < m_end ? am : m_end - 1;
            int64_t bn = b_row(lr);
            bn = bn < b_rows_total ? bn : b_rows_total - 1;
            rsa = kk < k_end ? p.sa[am / p.ar * p.ldsa + (kk >> p.ak_shift)] : 0.0f;
            rsb = kk < k_end ? sbptr[bn / p.br * p.ldsb + (kk >> p.bk_shift)] : 0.0f;
        }
    };
    auto stash = [&](int s) {
#pragma unroll
        for (int it = 0; it < 2; ++it) {
            const int id = it * 256 + tid;
            const int lr = id / 4, c = id % 4;
            uint2* da = reinterpret_cast<uint2*>(&lds_a[s][lr * LDK + c * 16]);
            da[0] = make_uint2(ra[it].x, ra[it].y);
            da[1] = make_uint2(ra[it].z, ra[it].w);
            uint2* db = reinterpret_cast<uint2*>(&lds_b[s][lr * LDK + c * 16]);
            db[0] = make_uint2(rb[it].x, rb[it].y);
            db[1] = make_uint2(rb[it].z, rb[it].w);
        }
        lds_sa[s][tid / BM][tid % BM] = rsa;
        lds_sb[s][tid / BM][tid % BM] = rsb;
    };

    // tile-local b row of this wavefront's sub-tile i (32 rows each)
    auto b_sub = [&](int i) -> int {
        if constexpr (MODE == MODE_GATED_FWD) return i * PANEL + wn * 32;   // i = 0 gate, 1 up
        else return wn * 64 + i * 32;
    };

    f32x16 total[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) total[i][j][r] = 0.0f;

    // HALF: the FP16 partial sums (kept as the floats they round to)
    f32x16 partial[HALF ? 2 : 1][HALF ? 2 : 1];
    if constexpr (HALF != 0) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) partial[i][j][r] = 0.0f;
    }
    auto to_half = [](float v) -> float { return (float)(_Float16)v; };
    auto reduced = [&](float v) -> float { return p.reduce_bf16 ? bf16_bits_to_f32(f32_to_bf16_bits(v)) : v; };

    const int64_t chunks = (k_end - k_begin + BK - 1) / BK;
    if (chunks > 0) {
        fetch(k_begin);
        stash(0);
    }
    __syncthreads();
    for (int64_t chunk = 0; chunk < chunks; ++chunk) {
        const int s = (int)(chunk & 1);
        if (chunk + 1 < chunks) fetch(k_begin + (chunk + 1) * BK);
#pragma unroll
        for (int kg = 0; kg < KG; ++kg) {
            f32x16 acc[2][2];
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                const int koff = kg * 32 + ks * 16 + lhi * 8;
                long opb[2], opa[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) opb[i] = *reinterpret_cast<const long*>(&lds_b[s][(b_sub(i) + l32) * LDK + koff]);
#pragma unroll
                for (int j = 0; j < 2; ++j) opa[j] = *reinterpret_cast<const long*>(&lds_a[s][(wm * 64 + j * 32 + l32) * LDK + koff]);
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        if (ks == 0) {
                            f32x16 zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
                            acc[i][j] = mfma32<A_BF8, B_BF8>(opb[i], opa[j], zero);
                        } else {
                            acc[i][j] = mfma32<A_BF8, B_BF8>(opb[i], opa[j], acc[i][j]);
                        }
                    }
            }
            if constexpr (HALF != 0) {
                // this 32-k step joins the FP16 partial; at the end of a period (and of the k range) the partial joins the total
                const int64_t done = chunk * BK + kg * 32 + 32;                  // k covered so far, relative to k_begin
                const bool last = done >= k_end - k_begin;
                const bool flush = p.half_period ? (done % p.half_period == 0 || last) : false;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const float sa_l = lds_sa[s][kg][wm * 64 + j * 32 + l32];
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const float h = to_half(partial[i][j][r] + acc[i][j][r]);
                            partial[i][j][r] = h;
                            if (flush) {
                                float term = h;
                                if constexpr (HALF == 1) {
                                    const float sb_l = B_ROWSCALE ? lds_sb[s][kg][b_sub(i) + (r / 4) * 8 + lhi * 4 + r % 4] : lds_sb[s][kg][b_sub(i)];
                                    term = (h * sa_l) * sb_l;
                                }
                                total[i][j][r] = reduced(total[i][j][r] + term);
                                partial[i][j][r] = 0.0f;
                            }
                        }
                    }
                }
                continue;
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float sa_l = lds_sa[s][kg][wm * 64 + j * 32 + l32];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    if constexpr (!B_ROWSCALE) {
                        const float sc = sa_l * lds_sb[s][kg][b_sub(i)];
#pragma unroll
                        for (int r = 0; r < 16; ++r) total[i][j][r] = fmaf(acc[i][j][r], sc, total[i][j][r]);
                    } else {
#pragma unroll
                        for (int r4 = 0; r4 < 4; ++r4) {
                            const float4 sb4 = *reinterpret_cast<const float4*>(&lds_sb[s][kg][b_sub(i) + r4 * 8 + lhi * 4]);
                            total[i][j][r4 * 4 + 0] = fmaf(acc[i][j][r4 * 4 + 0], sa_l * sb4.x, total[i][j][r4 * 4 + 0]);
                            total[i][j][r4 * 4 + 1] = fmaf(acc[i][j][r4 * 4 + 1], sa_l * sb4.y, total[i][j][r4 * 4 + 1]);
                            total[i][j][r4 * 4 + 2] = fmaf(acc[i][j][r4 * 4 + 2], sa_l * sb4.z, total[i][j][r4 * 4 + 2]);
                            total[i][j][r4 * 4 + 3] = fmaf(acc[i][j][r4 * 4 + 3], sa_l * sb4.w, total[i][j][r4 * 4 + 3]);
                        }
                    }
                }
            }
        }
        if (chunk + 1 < chunks) stash(s ^ 1);
        __syncthreads();
    }

    // ---- epilogue: lane holds m = l32 of sub-tile j, n = (r/4)*8 + lhi*4 + r%4 of sub-tile i
    TO* out = reinterpret_cast<TO*>(outptr);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int64_t mrow = m_begin + wm * 64 + j * 32 + l32;
        if (mrow >= m_end) continue;
        if constexpr (MODE == MODE_GATED_FWD) {
            TO* aux = static_cast<TO*>(p.aux);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int64_t ncol = n_begin + wn * 32 + (r / 4) * 8 + lhi * 4 + r % 4;
                if (ncol >= p.n) continue;
                float gv = total[0][j][r], uv = total[1][j][r];
                if (p.bias) {
                    gv += load_float(p.bias, ncol, bias_dtype);
                    uv += load_float(p.bias, p.n + ncol, bias_dtype);
                }
                const TO gq = from_f32<TO>(gv), uq = from_f32<TO>(uv);
                if (aux) {
                    aux[mrow * 2 * p.n + ncol] = gq;
                    aux[mrow * 2 * p.n + p.n + ncol] = uq;
                }
                float act, derivative;
                gate_math(p.activation, to_f32(gq), act, derivative);
                out[mrow * p.ldo + ncol] = from_f32<TO>(act * to_f32(uq));
            }
        } else {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int64_t ncol = n_begin + wn * 64 + i * 32 + (r / 4) * 8 + lhi * 4 + r % 4;
                    if (ncol >= p.n) continue;
                    float v = total[i][j][r];
                    if constexpr (HALF == 2) {
                        v = p.half_period ? v : partial[i][j][r];
                        v = (v * p.sa[0]) * p.sb[0];
                    }
                    if constexpr (MODE == MODE_PLAIN) {
                        if (p.bias) v += load_float(p.bias, ncol, bias_dtype);
                        out[mrow * p.ldo + ncol] = from_f32<TO>(v);
                    } else {
                        const TO* aux = static_cast<const TO*>(p.aux);
                        const float d = round_through<TO>(v);
                        const float g = to_f32(aux[mrow * 2 * p.n + ncol]);
                        const float u = to_f32(aux[mrow * 2 * p.n + p.n + ncol]);
                        float act, derivative;
                        gate_math(p.activation, g, act, derivative);
                        out[mrow * p.ldo + ncol] = from_f32<TO>(d * u * derivative);
                        out[mrow * p.ldo + p.n + ncol] = from_f32<TO>(d * act);
                    }
                }
            }
        }
    }
}

template <int MODE, bool B_ROWSCALE, bool VEC, typename TO>
static void launch_formats(const GemmArgs& p, int a_dtype, int b_dtype, int bias_dtype, dim3 grid, hipStream_t stream) {
    const bool a5 = a_dtype == VIOLA_E5M2, b5 = b_dtype == VIOLA_E5M2;
    if (!a5 && !b5) VIOLA_LAUNCH((group_gemm_kernel<MODE, false, false, B_ROWSCALE, VEC, TO>), grid, dim3(256), 0, stream, p, bias_dtype);
    else if (a5 && !b5) VIOLA_LAUNCH((group_gemm_kernel<MODE, true, false, B_ROWSCALE, VEC, TO>), grid, dim3(256), 0, stream, p, bias_dtype);
    else if (!a5 && b5) VIOLA_LAUNCH((group_gemm_kernel<MODE, false, true, B_ROWSCALE, VEC, TO>), grid, dim3(256), 0, stream, p, bias_dtype);
    else VIOLA_LAUNCH((group_gemm_kernel<MODE, true, true, B_ROWSCALE, VEC, TO>), grid, dim3(256), 0, stream, p, bias_dtype);
}

template <int MODE, typename TO>
static void launch_paths(const GemmArgs& p, int a_dtype, int b_dtype, int bias_dtype, bool rowscale, dim3 grid, hipStream_t stream) {
    // the generic kernel is only built with guarded byte loads; aligned problems take the fast kernel
    if (rowscale) launch_formats<MODE, true, false, TO>(p, a_dtype, b_dtype, bias_dtype, grid, stream);
    else launch_formats<MODE, false, false, TO>(p, a_dtype, b_dtype, bias_dtype, grid, stream);
}

template <int MODE>
static int launch_mode(const GemmArgs& p, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, bool rowscale, dim3 grid, hipStream_t stream) {
    switch (out_dtype) {
        case VIOLA_F32: launch_paths<MODE, float>(p, a_dtype, b_dtype, bias_dtype, rowscale, grid, stream); break;
        case VIOLA_BF16: launch_paths<MODE, bf16_t>(p, a_dtype, b_dtype, bias_dtype, rowscale, grid, stream); break;
        case VIOLA_F16: launch_paths<MODE, f16_t>(p, a_dtype, b_dtype, bias_dtype, rowscale, grid, stream); break;
        default: return VIOLA_EINVAL;
    }
    return viola_launch_status();
}

int launch_group_gemm_generic(const GemmArgs& p, int mode, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, bool rowscale, dim3 grid,
                              hipStream_t stream) {
    if (mode == MODE_PLAIN) return launch_mode<MODE_PLAIN>(p, a_dtype, b_dtype, bias_dtype, out_dtype, rowscale, grid, stream);
    if (mode == MODE_GATED_FWD) return launch_mode<MODE_GATED_FWD>(p, a_dtype, b_dtype, bias_dtype, out_dtype, rowscale, grid, stream);
    return launch_mode<MODE_GATED_BWD>(p, a_dtype, b_dtype, bias_dtype, out_dtype, rowscale, grid, stream);
}

// The FP16-accumulator model: always the generic kernel (an ablation option of the reference, not a fast path).
template <int HALF, bool B_ROWSCALE, typename TO>
static void launch_half_formats(const GemmArgs& p, int a_dtype, int b_dtype, int bias_dtype, dim3 grid, hipStream_t stream) {
    const bool a5 = a_dtype == VIOLA_E5M2, b5 = b_dtype == VIOLA_E5M2;
    if (!a5 && !b5) VIOLA_LAUNCH((group_gemm_kernel<MODE_PLAIN, false, false, B_ROWSCALE, false, TO, HALF>), grid, dim3(256), 0, stream, p, bias_dtype);
    else if (a5 && !b5) VIOLA_LAUNCH((group_gemm_kernel<MODE_PLAIN, true, false, B_ROWSCALE, false, TO, HALF>), grid, dim3(256), 0, stream, p, bias_dtype);
    else if (!a5 && b5) VIOLA_LAUNCH((group_gemm_kernel<MODE_PLAIN, false, true, B_ROWSCALE, false, TO, HALF>), grid, dim3(256), 0, stream, p, bias_dtype);
    else VIOLA_LAUNCH((group_gemm_kernel<MODE_PLAIN, true, true, B_ROWSCALE, false, TO, HALF>), grid, dim3(256), 0, stream, p, bias_dtype);
}

template <int HALF>
static int launch_half(const GemmArgs& p, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, bool rowscale, dim3 grid,
                       hipStream_t stream) {
#define VIOLA_HALF(TO)                                                                                        \
    if (HALF == 1 && rowscale) launch_half_formats<HALF, HALF == 1, TO>(p, a_dtype, b_dtype, bias_dtype, grid, stream); \
    else launch_half_formats<HALF, false, TO>(p, a_dtype, b_dtype, bias_dtype, grid, stream);
    switch (out_dtype) {
        case VIOLA_F32: VIOLA_HALF(float) break;
        case VIOLA_BF16: VIOLA_HALF(bf16_t) break;
        case VIOLA_F16: VIOLA_HALF(f16_t) break;
        default: return VIOLA_EINVAL;
    }
#undef VIOLA_HALF
    return viola_launch_status();
}

int launch_group_gemm_half(const GemmArgs& p, bool per_tensor, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, bool rowscale, dim3 grid,
                           hipStream_t stream) {
    if (per_tensor) return launch_half<2>(p, a_dtype, b_dtype, bias_dtype, out_dtype, rowscale, grid, stream);
    return launch_half<1>(p, a_dtype, b_dtype, bias_dtype, out_dtype, rowscale, grid, stream);
}

}  // namespace viola
