// Plain products with FP32 scales per 32 k (the grouped recipe) on large tiles: the phases of gemm_pingpong.hpp with the fold of
// gemm_fast_kernel.hpp. A block of eight waves owns one tile; waves 0-3 and 4-7 alternate between reading operands and multiplying.
//
// What bounds it. A unit (32 x 32 outputs, one K group) is two K = 16 MFMAs, 64 cycles of the matrix pipe, and 16 FMAs that fold
// the group's sums into the totals under sa * sb. A wave issues an FMA every 4.3 cycles, an MFMA every 6 or so, 82 to 87 cycles
// for the unit; and under that load on random data the card is at its power limit (1.8 - 1.9 GHz), so what counts next is the
// energy spent beside the arithmetic. Hence the tiles: 256 x 256 with 64 x 128 outputs per wave reads 768 bytes of operands from
// LDS per unit where 64 x 64 per wave read 1024, and fetches half of what two tiles of 128 x 128 fetch.
//
// Uniform b scales (forward, data gradient; ROWS false, 256 x 256). Three accumulators rotate: the FMAs among the MFMAs of unit u fold unit
// u - 2, whose sums are there without a wait (two accumulators, folding unit u - 1, cost nine wait states a unit: 500 against
// 432 us at 16384 x 4096 x 4096). The last two units of a chunk are folded in the wave's next read phase, under the other half's
// MFMAs, so that the accumulators' numbering starts over with each chunk; all 256 registers are in use.
//   16384 x 4096 x 4096   505 -> 440 us    16384 x 22016 x 4096   2700 -> 2380    8192 x 4096 x 1024   75 -> 67
// Products too small for those take tiles of 256 x 128 (GroupedTall, 64 x 64 per wave) in chunks of 128 k, so that a turn has as much
// math. Its registers allow more accumulators, but folding more units in the read phase gains nothing (16384 x 4096 x 4096 on these
// tiles: 487 us with a lag of two, 505, 505 and 506 with three, four and five; 8192 x 1024 x 4096 61.6, 64.8 to 65.3); nor does issuing
// the loads ahead of the LDS reads (521 against 513, in an earlier form).   8192 x 1024 x 4096  70 -> 62 to 66 us
// Row-wise b scales (weight gradient; ROWS true, 256 x 128). The products sa * sb of a pair of units come from one
// v_mfma_f32_32x32x1_2b (see group_gemm_fast), which occupies the FMA units for its 64 cycles as well; the pair of units before
// is folded meanwhile, across chunks too, out of two sets of accumulators and products.
//   22016 x 4096 x 16384  3450 -> 3080 us    4096 x 11008 x 16384   1660 -> 1560    4096 x 4096 x 4096   160 -> 142 to 149
// With few tiles (GroupedTeams, 128 x 128) the halves of the block are two teams with rings of their own that share the k range, as
// in group_gemm_fast's split form: the same sums, added in the same order.   4096 x 1024 x 8192  86 -> 74 to 77 us
#pragma once
#include "gemm_pingpong.hpp"

namespace viola {

using GroupedWide = PingPongShape<2, 4, 4, 2, 4>;                            // uniform b scales: 64 x 128 outputs (a x b) per wave, transposed
using GroupedRows = PingPongShape<4, 2, 2, 2, 4>;                            // row-wise b scales: 64 x 64
using GroupedTall = PingPongShape<4, 2, 2, 2, 3, 128>;                       // uniform b scales, half as wide: 64 x 64 per wave

using GroupedQuarter = PingPongShape<4, 2, 2, 1, 3, 128>;                    // uniform b scales, 256 x 64: 64 x 32

using GroupedTeams = PingPongShape<2, 2, 2, 2, 4>;                           // row-wise, 128 x 128, two teams that share the k range

typedef float f32x32 __attribute__((ext_vector_type(32)));

// Row tiles (of ROWS rows) of group base + lane, and of all groups base .. base + lane together.
template <int ROWS>
__device__ __forceinline__ void group_row_tiles(const GemmArgs& p, int base, int& tiles, int& end) {
    const int lane = threadIdx.x % WAVE, g = base + lane;
    tiles = g < p.groups ? (int)((p.offsets[g + 1] - p.offsets[g] + ROWS - 1) / ROWS) : 0;
    end = tiles;
#pragma unroll
    for (int step = 1; step < WAVE; step *= 2) {
        const int below = __shfl_up(end, step, WAVE);
        if (lane >= step) end += below;
    }
}

// A scale block is 8 K groups in 16-byte pieces of 4: [half][row of a], then [half][row of b], or with uniform b scales
// [half][sub-tile of b] (what 64 lanes of one load instruction bring); two buffers.
// Chunks of 128 k (OWN) bring their 4 K groups themselves: a block of [row of a], then [sub-tile of b] per stage.
template <typename S, bool ROWS>
struct GroupedLds {
    static constexpr bool OWN = S::CHUNK == 128;
    static constexpr int B_ENTRIES = ROWS ? S::COLS : S::COLS / 32;
    static constexpr int A_SCALES = (OWN ? 1 : 2) * S::ROWS * 16, B_SCALES = ROWS ? 2 * B_ENTRIES * 16 : 1024, SCALE_BLOCK = A_SCALES + B_SCALES;
    static constexpr int RING = S::STAGES * S::STAGE, SCALE_BUFFERS = OWN ? S::STAGES : 2, TEAM = RING + SCALE_BUFFERS * SCALE_BLOCK;
    static constexpr int BYTES = S::TEAMS * TEAM;
};

// Where a tile lies: its rows and first column, its k range, the b matrix of its group.
struct GroupedPlace {
    int64_t m_begin, m_end, n_begin, k_begin, k_end, out_shift;
    const uint8_t* b;
    const float* sb;
};

template <bool A_BF8, bool B_BF8, typename S, bool ROWS>
__device__ __forceinline__ void grouped_tile(const GemmArgs& p, const GroupedPlace& at, uint8_t* lds_all, int bias_dtype, int out_dtype) {
    constexpr int TM = S::TM, TN = S::TN, STAGES = S::STAGES, RING = STAGES * S::STAGE;
    using L = GroupedLds<S, ROWS>;
    constexpr int KG = S::CHUNK / 32, B_ENTRIES = L::B_ENTRIES, A_SCALES = L::A_SCALES, B_SCALES = L::B_SCALES, SCALE_BLOCK = L::SCALE_BLOCK;
    constexpr int SCALE_BUFFERS = L::SCALE_BUFFERS, TEAM_LDS = L::TEAM;
    constexpr bool OWN = L::OWN;
    static_assert(2 * S::ROWS == S::THREADS && (ROWS || 2 * B_ENTRIES <= 64) && SCALE_BUFFERS * SCALE_BLOCK >= S::COLS * 4);
    static_assert(KG == 2 || (OWN && !ROWS && S::TEAMS == 1));
    // tid, wave and lds are the team's own
    const int team = S::TEAMS > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / S::THREADS) : 0;
    const int tid = threadIdx.x % S::THREADS, lane = tid % WAVE, l32 = lane % 32, lhi = lane / 32;
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    uint8_t* const lds = lds_all + team * TEAM_LDS;
    const int wm = wave / S::WN, wn = wave % S::WN;

    const int64_t m_begin = at.m_begin, m_end = at.m_end, n_begin = at.n_begin, out_shift = at.out_shift;
    int64_t k_begin = at.k_begin, k_end = at.k_end;
    const uint8_t* bptr = at.b;
    const float* sbptr = at.sb;
    int split_chunks = 0;                                                    // of the longer (first) half of two teams
    if constexpr (S::TEAMS > 1) {
        constexpr int64_t CUT = F_SGROUPS * 32;                              // a scale block belongs to one team
        const int64_t len = k_end - k_begin, half = ((len + CUT - 1) / CUT + 1) / 2 * CUT, first = half < len ? half : len;
        split_chunks = (int)((first + S::CHUNK - 1) / S::CHUNK);
        if (team == 0) k_end = k_begin + first;
        else k_begin += first;
    }
    const int64_t k_len = k_end - k_begin;

    // ---- load plan: as in gemm_pingpong
    const i32x4 res_a = raw_resource(p.a + m_begin * p.lda + k_begin), res_b = raw_resource(bptr + k_begin);
    constexpr uint32_t OUTSIDE = 0x80000000u;
    // (both teams walk the first half's chunks, they share the barriers: past its own range a team loads zero codes)
    const int chunks = S::TEAMS > 1 ? split_chunks : (int)((k_len + S::CHUNK - 1) / S::CHUNK), full_chunks = (int)(k_len / S::CHUNK), groups_total = (int)((k_len + 31) / 32);
    auto swizzle = [](int row) -> int { return S::PIECES == 4 ? (row >> 2) & 3 : (row >> 1) & 7; };
    const int piece = tid % S::PIECES ^ swizzle(tid / S::PIECES);
    const bool inside_tail = (int64_t)full_chunks * S::CHUNK + piece * 16 < k_len;
    auto row_in = [](int64_t row, int64_t rows) -> uint32_t { return (uint32_t)(row < rows ? row : rows - 1); };
    uint32_t cur[S::LOADS];
#pragma unroll
    for (int it = 0; it < S::LOADS; ++it) {
        const int r = (it < S::A_LOADS ? it : it - S::A_LOADS) * S::LOAD_ROWS + tid / S::PIECES;
        if (it < S::A_LOADS) cur[it] = (uint32_t)(row_in(m_begin + r, m_end) - m_begin) * (uint32_t)p.lda;
        else cur[it] = row_in(n_begin + r, p.n) * (uint32_t)p.ldb;
        asm volatile("" : "+v"(cur[it]));                                    // (as one 64-bit multiply-add it would hold a register pair all along)
        cur[it] += piece * 16;
    }
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
    auto issue = [&](int c, int stage) {
        if (__builtin_expect(c >= full_chunks, 0)) {                         // the chunk that straddles the end of k, and those past it
            asm volatile("; end of the k range");
            const bool here = c == full_chunks && inside_tail;
#pragma unroll
            for (int it = 0; it < S::LOADS; ++it) {
                const uint32_t at = here ? cur[it] : OUTSIDE;
                load16_to_lds(it < S::A_LOADS ? res_a : res_b, lds_base + (uint32_t)stage * S::STAGE + it * S::THREADS * 16 + (uint32_t)wave * 1024, at, (uint32_t)c * S::CHUNK);
            }
            return;
        }
#pragma unroll
        for (int it = 0; it < S::LOADS; ++it)
            load16_to_lds(it < S::A_LOADS ? res_a : res_b, lds_base + (uint32_t)stage * S::STAGE + it * S::THREADS * 16 + (uint32_t)wave * 1024, cur[it], (uint32_t)c * S::CHUNK);
    };
    // Scale block `block` -> buffer block & 1: every thread one piece of the a rows, the first waves one of b (lanes past b's last
    // entry read zero). Entries past the end of the k range, which hold whatever follows in memory (see group_gemm_fast), are
    // cleared once in LDS.
    const i32x4 res_sa = raw_resource(p.sa, p.sa_bytes), res_sb = raw_resource(sbptr, p.sb_bytes);
    const int a_half = OWN ? 0 : wave * WAVE / S::ROWS, b_half = ROWS ? wave * WAVE / B_ENTRIES : lane / B_ENTRIES;
    const uint32_t group0 = (uint32_t)(k_begin >> 5) * 4;
    uint32_t sa_at = row_in(m_begin + tid % S::ROWS, m_end) / (uint32_t)p.ar * (uint32_t)p.ldsa * 4 + group0 + a_half * 16;
    uint32_t sb_at = row_in(n_begin + tid % B_ENTRIES * (ROWS ? 1 : 32), p.n) / (uint32_t)p.br * (uint32_t)p.ldsb * 4 + group0 + b_half * 16;
    if (b_half >= (OWN ? 1 : 2)) sb_at = OUTSIDE;
    asm volatile("" : "+v"(sa_at), "+v"(sb_at));
    const int last_block = (groups_total - 1) / F_SGROUPS;
    // (past the last block: that one again, to keep the load counts uniform; a team that walks on past its own range reads zeros)
    auto issue_scales = [&](int block) {
        if constexpr (OWN) {                                                 // waves 0-3: a; each of the others b, so that all have the same count
            const bool first = wave * WAVE < S::ROWS;
            const uint32_t to = lds_base + RING + (uint32_t)(block % STAGES) * SCALE_BLOCK + (first ? (uint32_t)wave * 1024 : A_SCALES);
            const uint32_t at = first ? sa_at : sb_at;
            load16_to_lds(first ? res_sa : res_sb, to, block < chunks ? at : OUTSIDE, (uint32_t)block * 16);
            return;
        }
        const uint32_t to = lds_base + RING + (uint32_t)(block & 1) * SCALE_BLOCK + (uint32_t)wave * 1024;
        const uint32_t first = (uint32_t)(block < last_block ? block : last_block) * F_SGROUPS * 4;
        const bool past = S::TEAMS > 1 && block > last_block;
        if (wave < B_SCALES / 1024) load16_to_lds(res_sb, to + A_SCALES, past ? OUTSIDE : sb_at, first);
        load16_to_lds(res_sa, to, past ? OUTSIDE : sa_at, first);
    };
    const bool straddles = groups_total % F_SGROUPS != 0 || groups_total == 0;
    auto clear_past_the_end = [&] {
        const int left_a = groups_total - (last_block * F_SGROUPS + a_half * 4), left_b = groups_total - (last_block * F_SGROUPS + b_half * 4);
        float* mine = reinterpret_cast<float*>(lds + RING + (last_block & 1) * SCALE_BLOCK + tid * 16);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (q >= left_a) mine[q] = 0.0f;
            if (q >= left_b && wave < B_SCALES / 1024) mine[A_SCALES / 4 + q] = 0.0f;
        }
    };

    // ---- operands: a lane's 16 bytes of K group kg of its row in every sub-tile, and the scales
    const int sw = swizzle(l32);
    const int rd_a = (wm * TM * 32 + l32) * S::CHUNK + ((lhi ^ sw) * 16), rd_b = S::A_BYTES + (wn * TN * 32 + l32) * S::CHUNK + ((lhi ^ sw) * 16);
    f32x16 total[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) total[i][j][r] = 0.0f;
    i32x4 oa[KG][TM], ob[KG][TN];
    // sa[j]: of the lane's row in sub-tile j; ROWS: sa[0] of row `lane` of the wave's 64, the operand of the scale products
    constexpr int SA = ROWS ? 1 : TM;
    float sa[SA][KG], sb[TN][KG];
    float4 va[SA], vb[TN];
    auto read = [&](int stage, int c) {
        // (addresses of K group 1 made here from those of K group 0: kept over the loop they would take two registers too many)
        int at_a = stage * S::STAGE + rd_a, at_b = stage * S::STAGE + rd_b;
        asm volatile("" : "+v"(at_a), "+v"(at_b));
#pragma unroll
        for (int kg = 0; kg < KG; ++kg) {
#pragma unroll
            for (int i = 0; i < TN; ++i) ob[kg][i] = *reinterpret_cast<const i32x4*>(lds + (at_b ^ (kg * 32)) + i * 32 * S::CHUNK);
#pragma unroll
            for (int j = 0; j < TM; ++j) oa[kg][j] = *reinterpret_cast<const i32x4*>(lds + (at_a ^ (kg * 32)) + j * 32 * S::CHUNK);
        }
        if constexpr (OWN) {
            const float* block = reinterpret_cast<const float*>(lds + RING + stage * SCALE_BLOCK);
#pragma unroll
            for (int j = 0; j < SA; ++j) va[j] = *reinterpret_cast<const float4*>(&block[(wm * TM * 32 + j * 32 + l32) * 4]);
#pragma unroll
            for (int i = 0; i < TN; ++i) vb[i] = *reinterpret_cast<const float4*>(&block[A_SCALES / 4 + (wn * TN + i) * 4]);
            return;
        }
        const int g8 = c % F_SCHUNKS * KG;                                  // group of the block (even: both groups of the chunk in one read)
        const float* block = reinterpret_cast<const float*>(lds + RING + ((c / F_SCHUNKS) & 1) * SCALE_BLOCK);
#pragma unroll
        for (int j = 0; j < SA; ++j) {
            const float2 v = *reinterpret_cast<const float2*>(&block[((g8 >> 2) * S::ROWS + wm * TM * 32 + j * 32 + (ROWS ? lane : l32)) * 4 + (g8 & 3)]);
            sa[j][0] = v.x; sa[j][1] = v.y;
        }
#pragma unroll
        for (int i = 0; i < TN; ++i) {
            const int entry = ROWS ? (wn * TN + i) * 32 + l32 : wn * TN + i;
            const float2 v = *reinterpret_cast<const float2*>(&block[A_SCALES / 4 + ((g8 >> 2) * B_ENTRIES + entry) * 4 + (g8 & 3)]);
            // (uniform: into scalar registers)
            sb[i][0] = ROWS ? v.x : __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v.x)));
            sb[i][1] = ROWS ? v.y : __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v.y)));
        }
    };
    // OWN: the scales of the chunk out of the pieces read. Past the end of k these hold whatever follows in memory, and the codes are zero.
    auto take_scales = [&](int c) {
        const int left = groups_total - c * KG;
#pragma unroll
        for (int j = 0; j < SA; ++j) asm volatile("" : "+v"(va[j].x), "+v"(va[j].y), "+v"(va[j].z), "+v"(va[j].w));
#pragma unroll
        for (int i = 0; i < TN; ++i) asm volatile("" : "+v"(vb[i].x), "+v"(vb[i].y), "+v"(vb[i].z), "+v"(vb[i].w));
#pragma unroll
        for (int kg = 0; kg < KG; ++kg) {
            const bool in = kg < left;
#pragma unroll
            for (int j = 0; j < SA; ++j) sa[j][kg] = in ? (&va[j].x)[kg] : 0.0f;
#pragma unroll
            for (int i = 0; i < TN; ++i) {
                const float v = in ? (&vb[i].x)[kg] : 0.0f;
                sb[i][kg] = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v)));
            }
        }
    };
    auto pin_operands = [&] {                                                // in registers before the barrier
#pragma unroll
        for (int kg = 0; kg < KG; ++kg) {
#pragma unroll
            for (int j = 0; j < TM; ++j) asm volatile("" : "+v"(oa[kg][j]));
#pragma unroll
            for (int j = 0; j < SA; ++j) asm volatile("" : "+v"(sa[j][kg]));
#pragma unroll
            for (int i = 0; i < TN; ++i) {
                asm volatile("" : "+v"(ob[kg][i]));
                if constexpr (ROWS) asm volatile("" : "+v"(sb[i][kg]));
                else asm volatile("" : "+s"(sb[i][kg]));
            }
        }
    };

    // ---- math
    const f32x16 zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    auto product = [&](int kg, int i, int j, int half, const f32x16& onto) -> f32x16 {
        auto codes = [&](const i32x4& v) -> long { return (long)(((uint64_t)(uint32_t)v[2 * half + 1] << 32) | (uint32_t)v[2 * half]); };
        return mfma32<A_BF8, B_BF8>(codes(ob[kg][i]), codes(oa[kg][j]), onto);
    };
    constexpr int ACCS = ROWS ? 4 : 3;
    f32x16 acc[ACCS];
#pragma unroll
    for (int x = 0; x < ACCS; ++x)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[x][r] = 0.0f;
    // uniform b scales: units in the order (kg, i, j), unit u in accumulator u % 3
    constexpr int UNITS = KG * TN * TM, LAG = 2;
    float scale[ACCS] = {};
    auto fold_unit = [&](int u, int first, int count) {
        const int i = u / TM % TN, j = u % TM, x = u % ACCS;
#pragma unroll
        for (int r = first; r < first + count; ++r) total[i][j][r] = fmaf(acc[x][r], scale[x], total[i][j][r]);
    };
    // row-wise: pairs of units (kg, i, j = 0 and 1), pair q in accumulators 2 (q & 1) + j, its scale products in prod[q & 1]
    constexpr int PAIRS = KG * TN;
    f32x32 prod[ROWS ? 2 : 1];
    if constexpr (ROWS) {
#pragma unroll
        for (int r = 0; r < 32; ++r) prod[0][r] = prod[1][r] = 0.0f;
    }
    auto fold_pair = [&](int q, int first, int count) {                      // elements first .. of the pair's 32
        const int set = q & 1;
#pragma unroll
        for (int e = first; e < first + count; ++e) {
            const int j = e / 16, r = e % 16;
            total[q % TN][j][r] = fmaf(acc[2 * set + j][r], prod[set][e], total[q % TN][j][r]);
        }
    };
    auto math = [&] {
        __builtin_amdgcn_s_setprio(1);
        if constexpr (!ROWS) {
#pragma unroll
            for (int u = 0; u < UNITS; ++u) {
                const int kg = u / (TN * TM), i = u / TM % TN, j = u % TM, x = u % ACCS;
                acc[x] = product(kg, i, j, 0, zero);
                if (u >= LAG) fold_unit(u - LAG, 0, 8);
                __builtin_amdgcn_sched_barrier(0);
                acc[x] = product(kg, i, j, 1, acc[x]);
                if (u >= LAG) fold_unit(u - LAG, 8, 8);
                __builtin_amdgcn_sched_barrier(0);
                scale[x] = sa[j][kg] * sb[i][kg];
            }
#pragma unroll
            for (int u = UNITS - LAG; u < UNITS; ++u) asm volatile("" : "+v"(acc[u % ACCS]), "+v"(scale[u % ACCS]));
        } else {
            static_assert(!ROWS || (TM == 2 && PAIRS % 2 == 0));
            const f32x32 zero32 = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
            for (int q = 0; q < PAIRS; ++q) {
                const int kg = q / TN, i = q % TN, set = q & 1, before = (q + PAIRS - 1) % PAIRS;
                prod[set] = __builtin_amdgcn_mfma_f32_32x32x1f32(sb[i][kg], sa[0][kg], zero32, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                fold_pair(before, 0, 8);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    const int j = x & 1;
                    acc[2 * set + j] = product(kg, i, j, x / 2, x < 2 ? zero : acc[2 * set + j]);
                    __builtin_amdgcn_sched_barrier(0);
                    fold_pair(before, 8 + x * 6, 6);
                    __builtin_amdgcn_sched_barrier(0);
                }
                asm volatile("" : "+v"(total[before % TN][0]), "+v"(total[before % TN][1]));
            }
            asm volatile("" : "+v"(acc[2]), "+v"(acc[3]), "+v"(prod[ROWS ? 1 : 0]));
        }
        __builtin_amdgcn_s_setprio(0);
    };
    auto drain = [&] {                                                       // the units of the last chunk that are not folded yet
        if constexpr (!ROWS) {
#pragma unroll
            for (int u = UNITS - LAG; u < UNITS; ++u) fold_unit(u, 0, 16);
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) asm volatile("" : "+v"(total[i][j]));
        } else {
            fold_pair(PAIRS - 1, 0, 32);
        }
    };
    auto barrier = [] {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };

    // ---- phases, stages and waits: as in gemm_pingpong. Scale block b + 1 is fetched in the read phase of chunk 4 b, into the
    // buffer that block b - 1 left a chunk ago (its last readers, waves 4-7, had it in registers before the barrier that ended
    // their read phase); it has landed when the read phase of chunk 4 b + 1 ends and is first read in chunk 4 b + 4, with the
    // straddling piece cleared in chunk 4 b + 2.
    // (Chunks with scales of their own: these are one load more of the chunk.)
    constexpr int AHEAD = (STAGES - 2) * (S::LOADS + (OWN ? 1 : 0));
    static_assert(AHEAD + 1 < 16 && STAGES >= 3);
    if (!OWN) issue_scales(0);
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s) {
        if (OWN) issue_scales(s);
        issue(s, s);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70 | AHEAD);                              // chunk 0 and scale block 0
    barrier();
    if (S::TEAMS > 1) {                                                      // the condition differs between the teams, the barrier must not
        if (last_block == 0 && straddles) clear_past_the_end();
        __syncthreads();
    } else if (!OWN && last_block == 0 && straddles) {
        clear_past_the_end();
        __syncthreads();
    }
    const bool late = S::TEAMS > 1 ? team == 1 : wave >= 4;
    if (late) barrier();
    int stage = 0, fill = STAGES - 1;
    for (int c = 0; c < chunks; ++c) {
        read(stage, c);
        const bool scales_now = !OWN && c % F_SCHUNKS == 0;
        if (scales_now) issue_scales(c / F_SCHUNKS + 1);
        if (!OWN && c % F_SCHUNKS == 2 && c / F_SCHUNKS + 1 == last_block && straddles) clear_past_the_end();
        if (OWN) issue_scales(c + STAGES - 1);
        issue(c + STAGES - 1, fill);
        stage = stage == STAGES - 1 ? 0 : stage + 1;
        fill = fill == STAGES - 1 ? 0 : fill + 1;
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!ROWS) {
            drain();
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (OWN) take_scales(c);
        }
        if (scales_now) __builtin_amdgcn_s_waitcnt(0x0070 | (AHEAD + 1));   // (the scale block just issued is among the newest)
        else __builtin_amdgcn_s_waitcnt(0x0070 | AHEAD);
        pin_operands();
        barrier();
        math();
        barrier();
    }
    if (!late) barrier();
    drain();
    __builtin_amdgcn_s_waitcnt(0x0F70);                                      // the trailing loads must not land in what follows
    barrier();
    if constexpr (S::TEAMS > 1) {
        // team 0's sums of the second row of sub-tiles go to team 1, team 1's of the first to team 0 (the rings are idle now):
        // [register quad][thread]. Either adds and stores half of the tile; x + y is y + x, so a launch is reproducible bit for bit.
        static_assert(TM == 2);
        float4* exchange = reinterpret_cast<float4*>(lds_all);
        constexpr int QUADS = TN * 4;
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                auto give = [&](int e) -> float {
                    const float first = total[i][0][4 * q + e], second = total[i][TM - 1][4 * q + e];
                    return team == 0 ? second : first;
                };
                exchange[(team * QUADS + i * 4 + q) * S::THREADS + tid] = make_float4(give(0), give(1), give(2), give(3));
            }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 t = exchange[((1 - team) * QUADS + i * 4 + q) * S::THREADS + tid];
                const float add[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {                                // (the half it stores goes to the first row of sub-tiles' place)
                    const float first = total[i][0][4 * q + e], second = total[i][TM - 1][4 * q + e];
                    total[i][0][4 * q + e] = (team == 0 ? first : second) + add[e];
                }
            }
        __syncthreads();
    }
    float* bias_lds = reinterpret_cast<float*>(lds_all + S::TEAMS * TEAM_LDS - SCALE_BUFFERS * SCALE_BLOCK);
    stage_bias<S>(p, n_begin, bias_lds, bias_dtype);
    auto finish = [&](auto type) {
        using TO = decltype(type);
        store_tile<S, TN, true>(total, p, static_cast<TO*>(p.out) + out_shift, m_begin, m_end, n_begin, lds_all, bias_lds);
    };
    if (out_dtype == VIOLA_F32) finish(float{});
    else if (out_dtype == VIOLA_BF16) finish(bf16_t{});
    else finish(f16_t{});
}

// Row tiles of all groups together; of the first 64 groups' those of each and up to it (see group_row_tiles).
template <int ROWS>
__device__ __forceinline__ int count_row_tiles(const GemmArgs& p, int& group_tiles, int& group_end) {
    if (!p.offsets) return p.tiles_m;
    int tiles_m = 0;
    for (int base = 0; base < p.groups; base += WAVE) {
        int count, end;
        group_row_tiles<ROWS>(p, base, count, end);
        if (base == 0) { group_tiles = count; group_end = end; }
        tiles_m += __builtin_amdgcn_readlane(end, WAVE - 1);
    }
    return tiles_m;
}

// Tile t of tiles_m x p.tiles_n, walked in groups of 4 m tiles, so that the 32 tiles at work on an XCD are 4 x 8
// (8 x 4: 70 instead of 67 us at 8192 x 4096 x 1024). Variable groups: see group_gemm_fast.
template <typename S>
__device__ __forceinline__ GroupedPlace grouped_place(const GemmArgs& p, int t, int tiles_m, int group_tiles, int group_end) {
    constexpr int WALK = 4;
    const int walk = WALK * p.tiles_n, first_m = t / walk * WALK;
    const int rows_here = tiles_m - first_m < WALK ? tiles_m - first_m : WALK;
    const int tile_m = first_m + t % walk % rows_here;
    GroupedPlace at = {(int64_t)tile_m * S::ROWS, p.m, (int64_t)(t % walk / rows_here) * S::COLS, 0, p.k, 0, p.b, p.sb};
    if (p.offsets) {
        int tile = tile_m, g = 0;
        for (int base = 0;; base += WAVE) {                                  // ends: tile_m is one of the tiles counted above
            if (base) group_row_tiles<S::ROWS>(p, base, group_tiles, group_end);
            const uint64_t past = __builtin_amdgcn_ballot_w64(tile < group_end);
            if (past) {
                const int lane = __builtin_ctzll(past);
                tile -= __builtin_amdgcn_readlane(group_end - group_tiles, lane);
                g = base + lane;
                break;
            }
            tile -= __builtin_amdgcn_readlane(group_end, WAVE - 1);
        }
        at.m_begin = p.offsets[g] + (int64_t)tile * S::ROWS;
        at.m_end = p.offsets[g + 1];
        at.b += (int64_t)g * p.b_group_stride;
        at.sb += (int64_t)g * p.sb_group_stride;
    }
    return at;
}

// Contiguous ranges of the tiles per XCD.
template <bool A_BF8, bool B_BF8, typename S, bool ROWS>
__global__ __launch_bounds__(512, 2) void gemm_pingpong_grouped(GemmArgs p, int bias_dtype, int out_dtype) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[GroupedLds<S, ROWS>::BYTES];
    int group_tiles = 0, group_end = 0;
    const int tiles_m = count_row_tiles<S::ROWS>(p, group_tiles, group_end), tiles = tiles_m * p.tiles_n;
    const int per_xcd = p.offsets ? (int)(((int64_t)tiles + 7) / 8) : (int)(gridDim.x / 8);
    const int seq = blockIdx.x / 8, place = (blockIdx.x % 8) * per_xcd + seq;
    const int part = p.k_split ? place / tiles : 0, t = place - part * tiles;
    if (seq >= per_xcd || (p.k_split ? part >= p.parts : t >= tiles)) return;
    GroupedPlace at = grouped_place<S>(p, t, tiles_m, group_tiles, group_end);
    if (p.koffsets) {
        at.k_begin = p.koffsets[blockIdx.z];
        at.k_end = p.koffsets[blockIdx.z + 1];
        at.out_shift = (int64_t)blockIdx.z * p.out_group_stride;
    }
    if (p.k_split) {
        at.k_begin = part * p.k_split;
        at.k_end = at.k_begin + p.k_split < p.k ? at.k_begin + p.k_split : p.k;
        at.out_shift = part * p.out_group_stride;
    }
    grouped_tile<A_BF8, B_BF8, S, ROWS>(p, at, lds, bias_dtype, out_dtype);
}

// Uniform b scales: rounds of S tiles, a CU each. A last round of few, which would take as long as a full one and leave CUs without a tile, runs
// on tiles of the same rows and fewer columns: up to 128 tiles as two of HALF each, up to 64 as four of QUARTER. Here and not on the host,
// because how many tiles variable groups make shows here only. Before, on blocks of 128 x 128 or tiles of 256 x 256 alone, and now (us):
// 8192 x 4608 x 4096 (two rounds and 64) 286, 312 -> 264; 4352 x 4096 x 4096 (one and 16) 154, 200 -> 145; 16384 x 8704 x 1024 (eight and 128)
// 326, 295 -> 275; 4096 x 10240 x 2048 (two and 128) 166, 169 -> 151; 4096 x 9216 x 1152 (two and 64) 95, 105 -> 87.5.
template <bool A_BF8, bool B_BF8, typename S, typename HALF, typename QUARTER>
__global__ __launch_bounds__(512, 2) void gemm_pingpong_grouped_rounds(GemmArgs p, int bias_dtype, int out_dtype) {
    constexpr int ROUND = 256;
    static_assert(S::ROWS == HALF::ROWS && S::ROWS == QUARTER::ROWS && S::COLS == 2 * HALF::COLS && S::COLS == 4 * QUARTER::COLS);
    constexpr int LDS_S = GroupedLds<S, false>::BYTES, LDS_H = GroupedLds<HALF, false>::BYTES;
    static_assert(GroupedLds<QUARTER, false>::BYTES <= LDS_H);
    __shared__ __attribute__((aligned(1024))) uint8_t lds[LDS_S > LDS_H ? LDS_S : LDS_H];
    int group_tiles = 0, group_end = 0;
    const int tiles_m = count_row_tiles<S::ROWS>(p, group_tiles, group_end), tiles = tiles_m * p.tiles_n;
    const int rest = tiles % ROUND, each = tiles < ROUND || rest * 2 > ROUND ? 1 : rest * 4 > ROUND ? 2 : 4;
    const int whole = each > 1 ? tiles - rest : (tiles + 7) / 8 * 8;
    const int block = blockIdx.x;
    if (block < whole) {                                                     // contiguous ranges per XCD
        const int t = block % 8 * (whole / 8) + block / 8;
        if (t >= tiles) return;
        grouped_tile<A_BF8, B_BF8, S, false>(p, grouped_place<S>(p, t, tiles_m, group_tiles, group_end), lds, bias_dtype, out_dtype);
        return;
    }
    if (each == 1) return;
    const int per_xcd = (rest * each + 7) / 8, seq = (block - whole) / 8, u = (block - whole) % 8 * per_xcd + seq, t = whole + u / each;
    if (seq >= per_xcd || t >= tiles) return;
    GroupedPlace at = grouped_place<S>(p, t, tiles_m, group_tiles, group_end);
    at.n_begin += u % each * (S::COLS / each);
    if (at.n_begin >= p.n) return;
    if (each == 2) grouped_tile<A_BF8, B_BF8, HALF, false>(p, at, lds, bias_dtype, out_dtype);
    else grouped_tile<A_BF8, B_BF8, QUARTER, false>(p, at, lds, bias_dtype, out_dtype);
}

}  // namespace viola
