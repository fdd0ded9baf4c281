// Arguments of the tiled Newton-Schulz GEMM (ns_fast.hip), shared with the entry point in ns.hip.
#pragma once
#include "common.hpp"

namespace viola {

struct NsArgs {
    const uint16_t* a;          // [batch, m, k]
    const uint16_t* b;          // [batch, n, k], or [batch, k, n] when b_kn
    const uint16_t* residual;   // [batch, m, n] or null
    uint16_t* out;              // [batch, m, n]
    uint16_t* out_diag;         // second copy with add_diag on the diagonal, or null
    int64_t batch, m, n, k;
    float add_diag;
    int transpose_out;          // store out (and out_diag) as [batch, n, m]
    int symmetric;              // b == a, m == n: compute tiles with tn >= tm only and mirror them
    int tiles_m, tiles_n;
    int group_m;                // tile rows per band of the work order (ns_fast.hip)
    int64_t tiles;              // batch * tiles_m * tiles_n
    int b_kn, epilogue;         // read where products of several kinds share a launch
    const int64_t* weights;     // such launches: not null, weights[batch] -> FP32 [m, n] (transpose_out: [n, m]) = weight * keep - rate * result,
    float keep, rate;           // and the result itself is not stored
};

// Products of one launch (by value in the kernel's arguments).
constexpr int NS_MANY = 8;
struct NsMany {
    NsArgs product[NS_MANY];
    int rounds[NS_MANY];        // blocks of a product per XCD
    int count;
};

// Tile shapes of the tiled kernel (rows x columns of output per block); NS_TILE_GENERIC is the kernel in ns.hip that
// takes every shape the tiled one refuses.
enum NsTile { NS_TILE_GENERIC = 0, NS_TILE_64x64 = 1, NS_TILE_128x64 = 2, NS_TILE_128x128 = 3, NS_TILE_192x192 = 4, NS_TILE_384x192 = 5 };
NsTile ns_choose_tile(int64_t batch, int64_t m, int64_t n, bool symmetric);
bool ns_fast_takes(const NsArgs& args);
NsTile ns_choose_tile_many(const NsMany& many);
bool ns_many_takes(const NsMany& many);

// Launches the tiled kernel when the shape qualifies (16-byte aligned rows, k and n multiples of 8,
// one matrix below 2 GiB); returns false without launching otherwise. `many`: unless every product qualifies.
bool launch_ns_gemm_many(const NsMany& many, bool is_bf16, hipStream_t stream);
bool launch_ns_gemm_fast(const NsArgs& args, bool is_bf16, bool b_kn, int epilogue, hipStream_t stream);

}  // namespace viola
