// gemm_rule.hpp — which tile size a projection GEMM runs in: 256 (gemm_tile.hpp), 128 or 64
// (gemm_small.hip). Plain C++ with no HIP types, shared with tests/gemm_rule_query.cpp.
#pragma once

#include <initializer_list>

namespace slime {
namespace gemm_rule {

// The shape of a launch: GemmArgs's sizes and the storage type (0 fp32, 1 bf16).
struct Dims {
    int dtype;
    int M, N, K, ncol, rows_per_batch;
};

// The 256 x 256 kernel's shapes: whole tiles in M, N, the planes and the batches, and K in
// whole groups of 4 slabs (4 x 64 bytes: 128 bf16 or 64 fp32).
inline bool fits256(const Dims& d) {
    const int k_group = d.dtype == 1 ? 128 : 64;
    return d.M % 256 == 0 && d.N % 256 == 0 && d.ncol % 256 == 0 && d.K % k_group == 0 && d.rows_per_batch % 256 == 0;
}

// The smaller ones': whole tiles of columns inside a plane, at least one tile of rows per
// batch, whole slabs (64 or 128 bytes) of K.
inline bool fits_small(int tile, const Dims& d) {
    const int slab = (tile == 128 ? 64 : 128) / (d.dtype == 1 ? 2 : 4);
    return d.N % tile == 0 && d.ncol % tile == 0 && d.rows_per_batch >= tile && d.M % d.rows_per_batch == 0 &&
           d.K % slab == 0;
}

// The tile whose rounds over the card take least time: ceil(tiles / CUs) rounds of
// tile^2 products each, at the rate the kernel reaches once it fills the card; 0 when none
// fits. Measured on K = 512 forward products (TFLOP/s, 256 / 128 / 64 wide): bf16 915 / 730 /
// 610 at 65,536 rows, fp32 139 / 137 / 131; so the 256-wide kernel keeps what it tiles and
// fills, and a batch that leaves its last round mostly empty goes to the smaller tiles:
// 16,384 x 1536 x 512 in fp32 (384 tiles of 256 on 256 CUs) 272 -> 192 us in 1536 tiles of
// 128; 8192 x 768 x 256 80 -> 31 us in tiles of 64. Shapes that 256 does not divide ran one
// thread per output before (0.55 TFLOP/s): 73,984 x 1536 x 512 bf16 211 ms -> 0.17 ms in
// tiles of 128, 0.13 ms in tiles of 256 over the four batch entries of one pod.
inline int pick(const Dims& d, int n_cu) {
    int best = 0;
    double best_t = 0.0;
    for (const int tile : {256, 128, 64}) {
        if (tile == 256 ? !fits256(d) : !fits_small(tile, d)) continue;
        const long long rows = (d.rows_per_batch + tile - 1) / tile;  // per batch
        const long long ntiles = d.M / d.rows_per_batch * rows * (d.N / tile);
        const long long rounds = (ntiles + n_cu - 1) / n_cu;
        const double rate = tile == 256 ? 1.0 : d.dtype == 1 ? (tile == 128 ? 0.8 : 0.66) : (tile == 128 ? 0.98 : 0.94);
        const double t = (double)rounds * tile * tile / rate;
        if (!best || t < best_t) best = tile, best_t = t;
    }
    return best;
}

}  // namespace gemm_rule
}  // namespace slime
