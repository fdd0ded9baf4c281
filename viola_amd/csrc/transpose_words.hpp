// A 64 x 64 tile of bytes turned by a block of 256 threads, whose rows, cols and pitch are multiples of 4 and whose pointers lie on 4 bytes.
#pragma once

#include "common.hpp"

namespace viola {

// Tile (r0, c0) of x [rows, cols] -> out [cols, out_pitch]; what lies past the matrix is zeros. A thread owns a 4 x 4 byte block: four
// 4-byte loads (16 lanes cover 64 contiguous bytes of a row), a 4 x 4 transpose with byte permutes, the four words
// handed over through LDS so that the stores are again 64 contiguous bytes per 16 lanes.
__device__ __forceinline__ void transpose_words(const uint8_t* __restrict__ x, uint8_t* __restrict__ out, int64_t rows, int64_t cols, int64_t out_pitch,
                                                int64_t r0, int64_t c0, uint32_t (*tile)[17]) {
    const int b = threadIdx.x % 16, a = threadIdx.x / 16;               // block of rows 4a.., cols 4b..
    uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (r0 + 4 * a + i < rows && c0 + 4 * b < cols) w[i] = *reinterpret_cast<const uint32_t*>(x + (r0 + 4 * a + i) * cols + c0 + 4 * b);
    // t[j] = byte j of w[0..3]
    const uint32_t lo01 = __builtin_amdgcn_perm(w[1], w[0], 0x05010400u);   // w0.b0 w1.b0 w0.b1 w1.b1
    const uint32_t hi01 = __builtin_amdgcn_perm(w[1], w[0], 0x07030602u);   // w0.b2 w1.b2 w0.b3 w1.b3
    const uint32_t lo23 = __builtin_amdgcn_perm(w[3], w[2], 0x05010400u);
    const uint32_t hi23 = __builtin_amdgcn_perm(w[3], w[2], 0x07030602u);
    tile[4 * b + 0][a] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u);    // bytes 0,1 of lo01 then of lo23
    tile[4 * b + 1][a] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
    tile[4 * b + 2][a] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
    tile[4 * b + 3][a] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = threadIdx.x / 16 + 16 * i, ra = threadIdx.x % 16;
        if (c0 + c < cols && r0 + 4 * ra < out_pitch) *reinterpret_cast<uint32_t*>(out + (c0 + c) * out_pitch + r0 + 4 * ra) = tile[c][ra];
    }
}

}  // namespace viola
