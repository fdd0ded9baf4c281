// Sums of squares of a matrix, which Newton-Schulz starts from, in one order wherever they are formed: by a pass over the matrix (ns.hip) and
// beside the momentum that makes it (optim.hip, tiles of any size), alone or with others in one launch. The norm is rounded to 16 bits, so that two
// orders would now and then scale a whole matrix differently.
#pragma once

#include "common.hpp"

namespace viola {

// A matrix is walked in units of 4096 elements; unit u goes to slot u % 256 of its 256 partial sums. A chunk of 256 of a unit's elements is a
// wavefront's, four consecutive ones per lane, and a lane adds what it gets in order, over the units of its slot. A slot is the sum, in order, of the
// wave_sums of its 16 chunks.
constexpr int NS_PARTS = 256, NS_UNIT = 4096, NS_CHUNK = 256, NS_CHUNKS = NS_UNIT / NS_CHUNK;

// blocks per matrix: its slots that are not zero from the start
inline dim3 ns_sum_blocks(int64_t count, int64_t matrices) {
    const int64_t units = (count + NS_UNIT - 1) / NS_UNIT;
    return dim3((unsigned)(units < 1 ? 1 : units > NS_PARTS ? NS_PARTS : units), (unsigned)matrices);
}

__device__ __forceinline__ void ns_add_squares(float& sum, const float (&v)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) sum += v[e] * v[e];
}

// wave_sum of four values at once, 7 exchanges instead of 24: lane 16 i has that of v[i].
__device__ __forceinline__ float wave_sum4(const float (&v)[4]) {
    const bool high = threadIdx.x & 32, odd = threadIdx.x & 16;
    float a = high ? v[2] : v[0], b = high ? v[3] : v[1];
    a += __shfl_xor(high ? v[0] : v[2], 32, WAVE);
    b += __shfl_xor(high ? v[1] : v[3], 32, WAVE);
    float sum = odd ? b : a;
    sum += __shfl_xor(odd ? a : b, 16, WAVE);
#pragma unroll
    for (int offset = 8; offset > 0; offset >>= 1) sum += __shfl_xor(sum, offset, WAVE);
    return sum;
}

// The block's slot from its lanes' sums, KEPT neighbouring chunks a wavefront: a block has 1024 / KEPT threads. Slots that no block has are zero.
template <int KEPT>
__device__ __forceinline__ void ns_store_slot(const float (&sums)[KEPT], float* __restrict__ slots) {
    __shared__ __attribute__((aligned(16))) float partial[NS_CHUNKS];
    const int wave = threadIdx.x / WAVE;
    if constexpr (KEPT == 4) {
        const float sum = wave_sum4(sums);
        if (threadIdx.x % 16 == 0) partial[threadIdx.x / 16] = sum;
    } else {
#pragma unroll
        for (int k = 0; k < KEPT; ++k) {
            const float sum = wave_sum(sums[k]);
            if (threadIdx.x % WAVE == 0) partial[wave * KEPT + k] = sum;
        }
    }
    __syncthreads();
    if (threadIdx.x >= WAVE) return;
    float sum = 0.0f;
#pragma unroll
    for (int chunk = 0; chunk < NS_CHUNKS; ++chunk) sum += partial[chunk];
    for (unsigned slot = blockIdx.x + threadIdx.x * gridDim.x; slot < NS_PARTS; slot += gridDim.x * WAVE) slots[slot] = slot == blockIdx.x ? sum : 0.0f;
}

}  // namespace viola
