// FP8 products without a per-group fold (per-tensor scales, E8M0 block scales) for gfx950: the kernel for shapes that
// give every CU a tile of its own. Same operand layout, MFMA orientation and stage format as gemm_fast_kernel.hpp.
//
// Eight waves (two per SIMD) own one tile. Their memory work and their math alternate in phases a barrier apart, the two
// halves of the block half a turn out of step: while waves 0-3 run the MFMAs of chunk c (at raised priority), waves 4-7 read
// their operands of chunk c from LDS into registers and issue the global -> LDS loads of chunk c + STAGES - 1, then they swap.
// So each SIMD always has one wave in either role, the LDS port serves four waves at a time instead of eight in a burst, and
// one operand register set per wave is enough (the 128 x 128 kernel reads the next chunk's operands in a burst ahead of its
// MFMAs, which then wait for that burst to issue).
#pragma once
#include <type_traits>

#include "gemm_fast_kernel.hpp"

namespace viola {

// WM x WN waves of TM x TN sub-tiles of 32 x 32; STAGES chunks of CHUNK k (bytes per operand row) in the ring
template <int WM_, int WN_, int TM_, int TN_, int STAGES_, int CHUNK_ = FBK>
struct PingPongShape {
    static constexpr int CHUNK = CHUNK_, PIECES = CHUNK / 16, HALVES = CHUNK / 64;   // 16-byte pieces of a row; 64 k per MFMA
    static constexpr int WM = WM_, WN = WN_, TM = TM_, TN = TN_, STAGES = STAGES_;
    static constexpr int TEAMS = 8 / (WM * WN), THREADS = 512 / TEAMS;       // two teams of four waves: gemm_pingpong_grouped.hpp
    static constexpr int ROWS = WM * TM * 32, COLS = WN * TN * 32;
    static constexpr int LOAD_ROWS = THREADS / PIECES;                       // a load instruction of all threads: 16 bytes each
    static constexpr int A_LOADS = ROWS / LOAD_ROWS, B_LOADS = COLS / LOAD_ROWS, LOADS = A_LOADS + B_LOADS;
    static constexpr int A_BYTES = ROWS * CHUNK, B_BYTES = COLS * CHUNK, STAGE = A_BYTES + B_BYTES;
    static_assert(WM * WN * TEAMS == 8 && ROWS % LOAD_ROWS == 0 && COLS % LOAD_ROWS == 0);
};

// Epilogue. The tile's bias as fp32 in LDS (COLS floats), -0 where there is none: adding that changes nothing, not even a sign.
template <typename S, bool GATED = false>
__device__ __forceinline__ void stage_bias(const GemmArgs& p, int64_t n_begin, float* bias_lds, int bias_dtype) {
    constexpr int PANEL = GATED ? S::COLS / 2 : S::COLS;
    const int tid = threadIdx.x;
    if (tid < S::COLS) {
        const int64_t col = n_begin + tid % PANEL;
        bias_lds[tid] = p.bias && col < p.n ? load_float(p.bias, (GATED ? tid / PANEL * p.n : 0) + col, bias_dtype) : -0.0f;
    }
    __syncthreads();
}

// A wave parks its first SUBS sub-tile columns, 32 rows at a time, in its own part of the ring (which every wave has left) and
// stores them as 16-byte pieces along the rows. The bias (nullptr: added before) is added on the way: before it, on all totals
// at once, the 256 x 256 tiles have no registers to spare (48 spilled; 70 instead of 68 us at 8192 x 4096 x 1024, grouped).
template <typename S, int SUBS, bool BIAS, typename TO>
__device__ __forceinline__ void store_tile(const f32x16 (&total)[S::TN][S::TM], const GemmArgs& p, TO* out, int64_t m_begin, int64_t m_end,
                                           int64_t n_begin, uint8_t* ring, const float* bias_lds) {
    const int lane = threadIdx.x % WAVE, l32 = lane % 32, lhi = lane / 32;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / WAVE), wm = wave % (S::WM * S::WN) / S::WN, wn = wave % S::WN;
    const bool pieces_out = (p.ldo * sizeof(TO)) % 16 == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
    constexpr int PER = 16 / (int)sizeof(TO), COLS_W = 32 * SUBS, PLD = COLS_W + PER, PIECES = COLS_W / PER;
    static_assert(8 * 32 * PLD * (int)sizeof(TO) <= S::TEAMS * S::STAGES * S::STAGE);
    TO* park = reinterpret_cast<TO*>(ring) + wave * 32 * PLD;
    const int64_t ncol0 = n_begin + wn * COLS_W;
#pragma unroll
    for (int j = 0; j < (S::TEAMS > 1 ? 1 : S::TM); ++j) {
        // (two teams: either stores one row of sub-tiles, team t the t-th, which it holds in the first one's place)
        const int64_t row0 = m_begin + (wm * S::TM + j + wave / (S::WM * S::WN)) * 32;
#pragma unroll
        for (int i = 0; i < SUBS; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float v[4] = {total[i][j][4 * q], total[i][j][4 * q + 1], total[i][j][4 * q + 2], total[i][j][4 * q + 3]};
                if constexpr (BIAS) {
                    const float4 bq = *reinterpret_cast<const float4*>(&bias_lds[(wn * SUBS + i) * 32 + q * 8 + lhi * 4]);
                    v[0] += bq.x; v[1] += bq.y; v[2] += bq.z; v[3] += bq.w;
                }
                Quad<TO>::store(&park[l32 * PLD + i * 32 + q * 8 + lhi * 4], v);
            }
#pragma unroll
        for (int it = 0; it < 32 * PIECES / WAVE; ++it) {
            const int id = it * WAVE + lane, pr = id / PIECES, pc = id % PIECES;
            const int64_t mrow = row0 + pr, ncol = ncol0 + pc * PER;
            const uint4 value = *reinterpret_cast<const uint4*>(&park[pr * PLD + pc * PER]);
            if (mrow >= m_end || ncol >= p.n) continue;
            if (pieces_out && ncol + PER <= p.n) {
                store_streaming(out + mrow * p.ldo + ncol, value);
            } else {
                const TO* values = reinterpret_cast<const TO*>(&value);
                for (int e = 0; e < PER; ++e)
                    if (ncol + e < p.n) out[mrow * p.ldo + ncol + e] = values[e];
            }
        }
    }
}

// Bytes of LDS a tile takes: the ring, and behind it two scale blocks of 16 K groups (a rows, then b rows), later the bias row.
template <bool MX, typename S>
constexpr int pingpong_lds() {
    return S::STAGES * S::STAGE + (MX ? 2 * (S::ROWS + S::COLS) * MX_GROUPS : S::COLS * 4);
}

// One tile. GATED: the tile's b rows are COLS / 2 gate rows, then the up rows of the same columns of h (sub-tiles 0 and 1 of a wave);
// out = act(g) * u, [g | u] itself is not kept.
template <bool A_BF8, bool B_BF8, bool MX, typename S, bool GATED>
__device__ __forceinline__ void pingpong_tile(const GemmArgs& p, int64_t m_begin, int64_t n_begin, uint8_t* lds, int bias_dtype, int out_dtype) {
    constexpr int TM = S::TM, TN = S::TN, STAGES = S::STAGES;
    static_assert(!GATED || TN == 2, "a gate and an up sub-tile per wave");
    constexpr int PANEL = GATED ? S::COLS / 2 : S::COLS;                     // columns of the output per tile
    constexpr int RING = STAGES * S::STAGE;
    constexpr int SCALE_BLOCK = (S::ROWS + S::COLS) * MX_GROUPS;             // scale bytes of 16 K groups, a rows then b rows
    static_assert(!MX || 2 * SCALE_BLOCK >= S::COLS * 4);
    const int tid = threadIdx.x, lane = tid % WAVE, l32 = lane % 32, lhi = lane / 32;
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int wm = wave / S::WN, wn = wave % S::WN;

    // ---- load plan: instruction `it` brings LOAD_ROWS rows of an operand, unit U = PIECES row + slot holds piece slot ^ swizzle(row)
    const i32x4 res_a = raw_resource(p.a + m_begin * p.lda), res_b = raw_resource(p.b);
    constexpr uint32_t OUTSIDE = 0x80000000u;
    const int chunks = (int)((p.k + S::CHUNK - 1) / S::CHUNK), full_chunks = (int)(p.k / S::CHUNK), groups_total = (int)((p.k + 31) / 32);
    // 16 consecutive rows reading the same piece then cover all banks
    auto swizzle = [](int row) -> int { return S::PIECES == 4 ? (row >> 2) & 3 : (row >> 1) & 7; };
    const int piece = tid % S::PIECES ^ swizzle(tid / S::PIECES);
    const bool inside_tail = (int64_t)full_chunks * S::CHUNK + piece * 16 < p.k;
    auto row_in = [](int64_t row, int64_t rows) -> uint32_t { return (uint32_t)(row < rows ? row : rows - 1); };
    auto b_row = [&](int r) -> uint32_t {                                    // tile-local b row -> row of b
        if constexpr (GATED) return (uint32_t)(r / PANEL) * (uint32_t)p.n + row_in(n_begin + r % PANEL, p.n);
        else return row_in(n_begin + r, p.n);
    };
    uint32_t cur[S::LOADS];
#pragma unroll
    for (int it = 0; it < S::LOADS; ++it) {
        const int r = (it < S::A_LOADS ? it : it - S::A_LOADS) * S::LOAD_ROWS + tid / S::PIECES;
        if (it < S::A_LOADS) cur[it] = (uint32_t)(row_in(m_begin + r, p.m) - m_begin) * (uint32_t)p.lda + piece * 16;
        else cur[it] = b_row(r) * (uint32_t)p.ldb + piece * 16;
    }
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
    auto issue = [&](int c, int stage) {
        if (__builtin_expect(c >= full_chunks, 0)) {                         // the chunk that straddles the end of k, and those past it
            asm volatile("; end of the k range");
            const bool here = c == full_chunks && inside_tail;
#pragma unroll
            for (int it = 0; it < S::LOADS; ++it) {
                const uint32_t at = here ? cur[it] : OUTSIDE;
                load16_to_lds(it < S::A_LOADS ? res_a : res_b, lds_base + (uint32_t)stage * S::STAGE + it * 8192 + (uint32_t)wave * 1024, at, (uint32_t)c * S::CHUNK);
            }
            return;
        }
#pragma unroll
        for (int it = 0; it < S::LOADS; ++it)
            load16_to_lds(it < S::A_LOADS ? res_a : res_b, lds_base + (uint32_t)stage * S::STAGE + it * 8192 + (uint32_t)wave * 1024, cur[it], (uint32_t)c * S::CHUNK);
    };
    // E8M0 scales: one 16-byte piece (16 K groups) per tile row, block `b` in buffer b & 1
    const i32x4 res_sa = raw_resource(p.sa, p.sa_bytes), res_sb = raw_resource(p.sb, p.sb_bytes);
    uint32_t scale_at = 0;
    if constexpr (MX) {
        scale_at = tid < S::ROWS ? row_in(m_begin + tid, p.m) / (uint32_t)p.ar * (uint32_t)p.ldsa : b_row(tid - S::ROWS) / (uint32_t)p.br * (uint32_t)p.ldsb;
    }
    const bool scale_wave = wave * 64 < S::ROWS + S::COLS;
    auto issue_scales = [&](int block) {
        if (!scale_wave) return;
        const uint32_t to = lds_base + RING + (uint32_t)(block & 1) * SCALE_BLOCK + (uint32_t)wave * 1024;
        load16_to_lds(wave * 64 < S::ROWS ? res_sa : res_sb, to, block * MX_GROUPS < groups_total ? scale_at : OUTSIDE, (uint32_t)(block * MX_GROUPS));
    };

    // ---- operand reads
    const int sw = swizzle(l32);
    const int rd_a0 = (wm * TM * 32 + l32) * S::CHUNK + ((lhi ^ sw) * 16), rd_b0 = S::A_BYTES + ((GATED ? wn : wn * TN) * 32 + l32) * S::CHUNK + ((lhi ^ sw) * 16);
    constexpr int NEXT_B = GATED ? PANEL : 32;                               // b rows from one sub-tile of a wave to the next
    f32x16 total[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) total[i][j][r] = 0.0f;
    constexpr int HALVES = S::HALVES;                                        // of a chunk: 64 k, one MFMA per sub-tile
    constexpr int SCALE_CHUNKS = MX_CHUNKS / HALVES;                         // chunks per scale block
    i32x8 oa[HALVES][TM], ob[HALVES][TN];
    // scale words of the 128 k at hand: byte 0 = this lane's K group of the first 64 k, byte 2 = of the second
    uint32_t wa[TM], wb[TN];
#pragma unroll
    for (int j = 0; j < TM; ++j) wa[j] = 0;
#pragma unroll
    for (int i = 0; i < TN; ++i) wb[i] = 0;
    auto read = [&](int stage, int c) {
        const uint8_t* base = lds + stage * S::STAGE;
        int rd_a = rd_a0, rd_b = rd_b0;
        asm volatile("" : "+v"(rd_a), "+v"(rd_b));                           // the addresses below: formed anew, 256 x 256 has no registers to keep them
        auto operand = [&](int offset, int half) -> i32x8 {                  // pieces 4 half + lhi and 4 half + lhi + 2
            const i32x4 lo = *reinterpret_cast<const i32x4*>(base + (offset ^ (half * 64))), hi = *reinterpret_cast<const i32x4*>(base + (offset ^ (half * 64 + 32)));
            return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        };
#pragma unroll
        for (int h = 0; h < HALVES; ++h) {
#pragma unroll
            for (int i = 0; i < TN; ++i) ob[h][i] = operand(rd_b + i * NEXT_B * S::CHUNK, h);
#pragma unroll
            for (int j = 0; j < TM; ++j) oa[h][j] = operand(rd_a + j * 32 * S::CHUNK, h);
        }
        if constexpr (MX) {
            if (HALVES == 2 || (c & 1) == 0) {
                const uint8_t* block = lds + RING + ((c / SCALE_CHUNKS) & 1) * SCALE_BLOCK + (c % SCALE_CHUNKS) * FKG * HALVES;
#pragma unroll
                for (int j = 0; j < TM; ++j) wa[j] = *reinterpret_cast<const uint32_t*>(block + (wm * TM * 32 + j * 32 + l32) * MX_GROUPS) >> (8 * lhi);
#pragma unroll
                for (int i = 0; i < TN; ++i) wb[i] = *reinterpret_cast<const uint32_t*>(block + (S::ROWS + (GATED ? wn : wn * TN) * 32 + i * NEXT_B + l32) * MX_GROUPS) >> (8 * lhi);
            }
        }
    };
    auto math = [&](auto odd) {
        constexpr int FB = B_BF8 ? 1 : 0, FA = A_BF8 ? 1 : 0, BYTE = MX && HALVES == 1 && decltype(odd)::value ? 2 : 0;
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
            for (int j = 0; j < TM; ++j)
                total[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(ob[0][i], oa[0][j], total[i][j], FB, FA, BYTE, MX ? (int)wb[i] : 0, BYTE, MX ? (int)wa[j] : 0);
        if constexpr (HALVES == 2) {
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j)
                    total[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(ob[HALVES - 1][i], oa[HALVES - 1][j], total[i][j], FB, FA, MX ? 2 : 0, MX ? (int)wb[i] : 0,
                                                                                  MX ? 2 : 0, MX ? (int)wa[j] : 0);
        }
        // (the compiler sinks MFMAs into the following read phase otherwise: intrinsics without side effects cross a barrier)
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
            for (int j = 0; j < TM; ++j) asm volatile("" : "+v"(total[i][j]));
        __builtin_amdgcn_s_setprio(0);
    };
    auto pin_operands = [&] {                                                // in registers before the barrier, scale bytes in place
#pragma unroll
        for (int h = 0; h < HALVES; ++h) {
#pragma unroll
            for (int j = 0; j < TM; ++j) asm volatile("" : "+v"(oa[h][j]), "+v"(wa[j]));
#pragma unroll
            for (int i = 0; i < TN; ++i) asm volatile("" : "+v"(ob[h][i]), "+v"(wb[i]));
        }
    };
    auto barrier = [] {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };

    // Phases. Waves 0-3 read chunk c in phase 2c and multiply in phase 2c + 1, waves 4-7 one phase later. The loads of chunk
    // c + STAGES - 1 go out in the read phase of chunk c, into the stage of chunk c - 1: its last readers (waves 4-7, phase
    // 2c - 1) had their operands in registers before the barrier that ended that phase. Every wave ends its read phase of
    // chunk c with its own loads of chunk c + 1 landed (at most those of the STAGES - 2 chunks after it in flight, and a
    // scale block issued in this phase: waiting for that as well, 4096 x 1152 x 9216 and x 4608 took 105.9 us
    // behind the quantizers of a step where they take 103.1), and chunk c + 1 is first read two barriers later.
    // Two stages: chunk c + 1 goes out in phase 2c, once waves 4-7 have read chunk c - 1 (waves 0-3 issue it in their read phase of
    // chunk c, waves 4-7 in their math phase of chunk c - 1), and every wave waits for its part before the barrier that ends phase
    // 2c + 1 (waves 0-3 behind their math, waves 4-7 behind their reads of chunk c).
    constexpr bool TWO = STAGES == 2;
    constexpr int AHEAD = TWO ? 0 : (STAGES - 2) * S::LOADS;
    static_assert((STAGES - 1) * S::LOADS < 16);
    if constexpr (MX) issue_scales(0);
#pragma unroll
    for (int s = 0; s < (TWO ? 2 : STAGES - 1); ++s) issue(s, s);
    __builtin_amdgcn_s_waitcnt(0x0F70 | (TWO ? S::LOADS : AHEAD));           // chunk 0 and scale block 0
    barrier();
    const bool late = wave >= 4;
    if (late) barrier();
    int stage = 0, fill = TWO && late ? 0 : STAGES - 1;
    auto step = [&](int c, auto odd) {
        read(stage, c);
        auto issue_next = [&](int next) {
            if constexpr (MX) {
                if (c % SCALE_CHUNKS == 0) issue_scales(c / SCALE_CHUNKS + 1);
            }
            if (!TWO || next > 1) issue(next, fill);                         // (two stages: chunk 1 went out with chunk 0)
            fill = fill == STAGES - 1 ? 0 : fill + 1;
        };
        if (!TWO || !late) issue_next(c + STAGES - 1);
        stage = stage == STAGES - 1 ? 0 : stage + 1;
        __builtin_amdgcn_sched_barrier(0);
        if (MX && !TWO && c % SCALE_CHUNKS == 0 && scale_wave) __builtin_amdgcn_s_waitcnt(0x0070 | (AHEAD + 1));
        else if (!TWO || late) __builtin_amdgcn_s_waitcnt(0x0070 | AHEAD);
        else __builtin_amdgcn_s_waitcnt(0xC07F);                             // the LDS reads alone
        pin_operands();
        barrier();
        if (TWO && late) issue_next(c + 2);
        math(odd);
        if (TWO && !late) __builtin_amdgcn_s_waitcnt(0x0F70);
        barrier();
    };
    int c = 0;
    for (; c + 1 < chunks; c += 2) {
        step(c, std::false_type{});
        step(c + 1, std::true_type{});
    }
    if (c < chunks) step(c, std::false_type{});
    if (!late) barrier();
    __builtin_amdgcn_s_waitcnt(0x0F70);                                      // the trailing loads must not land in what follows

    // ---- epilogue
    if constexpr (!MX) {
        const float sa = p.sa[0], sb = p.sb[0];
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
            for (int j = 0; j < TM; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) { const float v = total[i][j][r] * sa; total[i][j][r] = v * sb; }
    }
    barrier();                                                               // every wave has left the ring
    float* bias_lds = reinterpret_cast<float*>(lds + RING);
    stage_bias<S, GATED>(p, n_begin, bias_lds, bias_dtype);
    // (one kernel for the three output types: they differ from here on only)
    auto finish = [&](auto type) {
        using TO = decltype(type);
        if constexpr (GATED) {
            float4 bias_g[4], bias_u[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                bias_g[q] = *reinterpret_cast<const float4*>(&bias_lds[wn * 32 + q * 8 + lhi * 4]);
                bias_u[q] = *reinterpret_cast<const float4*>(&bias_lds[PANEL + wn * 32 + q * 8 + lhi * 4]);
            }
#pragma unroll
            for (int j = 0; j < TM; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    total[0][j][r] += (&bias_g[r / 4].x)[r % 4];
                    total[TN - 1][j][r] += (&bias_u[r / 4].x)[r % 4];
                    float act, derivative, h;
                    gate_math(p.activation, rounded<TO>(total[0][j][r]), act, derivative);
                    h = act * rounded<TO>(total[TN - 1][j][r]);
                    asm volatile("" : "+v"(h));                                 // an FP32 value of its own (see group_gemm_fast)
                    total[0][j][r] = h;
                }
        }
        store_tile<S, GATED ? 1 : TN, !GATED>(total, p, static_cast<TO*>(p.out), m_begin, p.m, n_begin, lds, bias_lds);
    };
    if (out_dtype == VIOLA_F32) finish(float{});
    else if (out_dtype == VIOLA_BF16) finish(bf16_t{});
    else finish(f16_t{});
}

// Tile `t` in the order of the walk: groups of 8 m tiles (see group_gemm_fast).
__device__ __forceinline__ void pingpong_place(const GemmArgs& p, int t, int rows, int cols, int64_t& m_begin, int64_t& n_begin) {
    const int group = 8 * p.tiles_n, first_m = t / group * 8;
    const int rows_here = p.tiles_m - first_m < 8 ? p.tiles_m - first_m : 8;
    m_begin = (int64_t)(first_m + t % group % rows_here) * rows;
    n_begin = (int64_t)(t % group / rows_here) * cols;
}

template <bool A_BF8, bool B_BF8, bool MX, typename S, int WAVES_PER_SIMD, bool GATED = false>
__global__ __launch_bounds__(512, WAVES_PER_SIMD) void gemm_pingpong(GemmArgs p, int bias_dtype, int out_dtype) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[pingpong_lds<MX, S>()];
    const int t = (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;       // contiguous ranges per XCD
    if (t >= p.tiles_m * p.tiles_n) return;
    int64_t m_begin, n_begin;
    pingpong_place(p, t, S::ROWS, GATED ? S::COLS / 2 : S::COLS, m_begin, n_begin);
    pingpong_tile<A_BF8, B_BF8, MX, S, GATED>(p, m_begin, n_begin, lds, bias_dtype, out_dtype);
}

// The first `whole` tiles (a multiple of 8) as they are, each of the others as tiles of the smaller shape T: a last round of few tiles, which
// takes as long as a full one and leaves most CUs without a tile, is shared among four times as many. 256 x 256, then 128 x 128 (E8M0
// scales, us): 4096 x 9216 x 1152 (two rounds and 64 tiles) 60.4 -> 53.8, 2891 x 5760 x 3072 (one and 20) 77 -> 60.5, 16384 x 1280 x 4096 (one and 64)
// 100 -> 84, 4096 x 8704 x 8192 279 -> 247, 8192 x 8448 x 1024 (four and 32) 87.5 -> 81.8. (A last round on 256 x 128 takes 1 to 4 us
// longer, rounds of 256 x 128 with a last one of 128 x 128 as long as 256 x 256 without: neither is built.)
template <bool A_BF8, bool B_BF8, bool MX, typename S, typename T>
__global__ __launch_bounds__(512, 2) void gemm_pingpong_tail(GemmArgs p, int whole, int bias_dtype, int out_dtype) {
    constexpr int ACROSS = S::COLS / T::COLS, EACH = S::ROWS / T::ROWS * ACROSS;
    static_assert(S::ROWS % T::ROWS == 0 && S::COLS % T::COLS == 0);
    constexpr int LDS_S = pingpong_lds<MX, S>(), LDS_T = pingpong_lds<MX, T>();
    __shared__ __attribute__((aligned(1024))) uint8_t lds[LDS_S > LDS_T ? LDS_S : LDS_T];
    int64_t m_begin, n_begin;
    const int block = blockIdx.x;
    if (block < whole) {
        pingpong_place(p, block % 8 * (whole / 8) + block / 8, S::ROWS, S::COLS, m_begin, n_begin);
        pingpong_tile<A_BF8, B_BF8, MX, S, false>(p, m_begin, n_begin, lds, bias_dtype, out_dtype);
        return;
    }
    const int rest = block - whole, u = rest % 8 * (((int)gridDim.x - whole) / 8) + rest / 8, t = whole + u / EACH, part = u % EACH;
    if (t >= p.tiles_m * p.tiles_n) return;
    pingpong_place(p, t, S::ROWS, S::COLS, m_begin, n_begin);
    m_begin += part / ACROSS * T::ROWS;
    n_begin += part % ACROSS * T::COLS;
    if (m_begin >= p.m || n_begin >= p.n) return;                            // a tile across the edge: nothing of it here
    pingpong_tile<A_BF8, B_BF8, MX, T, false>(p, m_begin, n_begin, lds, bias_dtype, out_dtype);
}

// The three tiles: 256 x 256 and 256 x 128 with one block per CU, 128 x 128 with one or two. A turn of the two halves costs some 200
// cycles beside the math (barriers, the first LDS reads), which is a lot next to the 256 or 512 cycles of a wave's four or eight
// MFMAs: where registers and LDS allow it a chunk is 128 k (whole cache lines of the operands, too). 256 x 256, in two stages for
// want of LDS: 4096 x 4096 x 4096 61 -> 55 us (E8M0 64 -> 57), 16384 x 4096 x 11008 547 -> 509, 8192 x 8192 x 8192 394 -> 387 (the
// power limit), even up to k = 1024. (Four stages of
// 64 k are on their way for longer, and faster at 180 tiles on warm operands, 9216 x 1152 x 4096 54 -> 48 us, but not behind the
// quantizers of a step: 54.8 against 55.3.) 256 x 128: 4096 x 1152 x 9216 61 -> 47 us,
// 8192 x 1024 x 4096 36 -> 30, 4096 x 1152 x 4608 33 -> 26 (E8M0 35 -> 30); 128 x 128 alone on its CU: 2048 x 1152 x 4608 22 -> 19.
// (96- and 192-column tiles, which leave fewer CUs idle at widths like 1152, gain nothing: a smaller tile's turn takes as long.)
using PingPongL = PingPongShape<2, 4, 4, 2, 2, 128>;
using PingPongM = PingPongShape<4, 2, 2, 2, 3, 128>;
using PingPongS = PingPongShape<2, 4, 2, 1, 3, 128>;
using PingPongPairs = PingPongShape<2, 4, 2, 1, 4>;

template <bool MX, typename S, int WAVES_PER_SIMD, bool GATED = false>
static int launch_pingpong(const GemmArgs& args, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, hipStream_t stream) {
    GemmArgs p = args;
    constexpr int PANEL = GATED ? S::COLS / 2 : S::COLS;
    p.tiles_m = (int)((p.m + S::ROWS - 1) / S::ROWS);
    p.tiles_n = (int)((p.n + PANEL - 1) / PANEL);
    if (!viola_is_float(out_dtype)) return VIOLA_EINVAL;
    const bool a5 = a_dtype == VIOLA_E5M2, b5 = b_dtype == VIOLA_E5M2;
    const dim3 grid((unsigned)(((int64_t)p.tiles_m * p.tiles_n + 7) / 8 * 8)), block(512);
    if (!a5 && !b5) VIOLA_LAUNCH((gemm_pingpong<false, false, MX, S, WAVES_PER_SIMD, GATED>), grid, block, 0, stream, p, bias_dtype, out_dtype);
    else if (a5 && !b5) VIOLA_LAUNCH((gemm_pingpong<true, false, MX, S, WAVES_PER_SIMD, GATED>), grid, block, 0, stream, p, bias_dtype, out_dtype);
    else if (!a5 && b5) VIOLA_LAUNCH((gemm_pingpong<false, true, MX, S, WAVES_PER_SIMD, GATED>), grid, block, 0, stream, p, bias_dtype, out_dtype);
    else VIOLA_LAUNCH((gemm_pingpong<true, true, MX, S, WAVES_PER_SIMD, GATED>), grid, block, 0, stream, p, bias_dtype, out_dtype);
    return viola_launch_status();
}

template <bool MX, typename S, typename T>
static int launch_pingpong_tail(const GemmArgs& args, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, hipStream_t stream) {
    GemmArgs p = args;
    p.tiles_m = (int)((p.m + S::ROWS - 1) / S::ROWS);
    p.tiles_n = (int)((p.n + S::COLS - 1) / S::COLS);
    if (!viola_is_float(out_dtype)) return VIOLA_EINVAL;
    const bool a5 = a_dtype == VIOLA_E5M2, b5 = b_dtype == VIOLA_E5M2;
    const int tiles = p.tiles_m * p.tiles_n, whole = tiles / 256 * 256, each = S::ROWS / T::ROWS * (S::COLS / T::COLS);
    const dim3 grid((unsigned)(whole + ((int64_t)(tiles - whole) * each + 7) / 8 * 8)), block(512);
    if (!a5 && !b5) VIOLA_LAUNCH((gemm_pingpong_tail<false, false, MX, S, T>), grid, block, 0, stream, p, whole, bias_dtype, out_dtype);
    else if (a5 && !b5) VIOLA_LAUNCH((gemm_pingpong_tail<true, false, MX, S, T>), grid, block, 0, stream, p, whole, bias_dtype, out_dtype);
    else if (!a5 && b5) VIOLA_LAUNCH((gemm_pingpong_tail<false, true, MX, S, T>), grid, block, 0, stream, p, whole, bias_dtype, out_dtype);
    else VIOLA_LAUNCH((gemm_pingpong_tail<true, true, MX, S, T>), grid, block, 0, stream, p, whole, bias_dtype, out_dtype);
    return viola_launch_status();
}

template <bool MX>
static int launch_pingpong_tile(const GemmArgs& p, ScaledTile tile, bool gated, int a_dtype, int b_dtype, int bias_dtype, int out_dtype, hipStream_t stream) {
    if (gated) return launch_pingpong<MX, PingPongL, 2, true>(p, a_dtype, b_dtype, bias_dtype, out_dtype, stream);
    switch (tile) {
        case SCALED_TILE_L: return launch_pingpong<MX, PingPongL, 2>(p, a_dtype, b_dtype, bias_dtype, out_dtype, stream);
        case SCALED_TILE_L_THEN_S: return launch_pingpong_tail<MX, PingPongL, PingPongS>(p, a_dtype, b_dtype, bias_dtype, out_dtype, stream);
        case SCALED_TILE_M: return launch_pingpong<MX, PingPongM, 2>(p, a_dtype, b_dtype, bias_dtype, out_dtype, stream);
        default: break;
    }
    if ((p.m + 127) / 128 * ((p.n + 127) / 128) <= 256) return launch_pingpong<MX, PingPongS, 2>(p, a_dtype, b_dtype, bias_dtype, out_dtype, stream);
    return launch_pingpong<MX, PingPongPairs, 4>(p, a_dtype, b_dtype, bias_dtype, out_dtype, stream);
}

}  // namespace viola
