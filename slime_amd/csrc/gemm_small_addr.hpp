// gemm_small_addr.hpp — the address arithmetic of the 128- and 64-wide tile GEMM
// (gemm_small.hip): the tile walk with its overlapping last tile per batch, the direct
// loads, the operand fragment reads and the ring's waits. Plain C++ with no HIP types, shared
// with the host replay tests/gemm_small_replay.cpp, which checks every address of a launch
// against its buffer, every fragment read against the row and chunk its MFMA needs and
// every wait against the order in which the wave's loads complete.
#pragma once

#include "gemm_addr.hpp"

namespace slime {
namespace gemm_small {

constexpr int kThreads = 256, kWaves = 4;
constexpr int kStages = 3;  // LDS ring: slab ks in stage ks % kStages

// The slabs whose loads a wave has issued after slab ks's when it waits for that one: the
// prologue issues kStages - 1 slabs, step ks slab ks + kStages - 1 after its wait.
SLIME_HD constexpr int younger_slabs(int ks, int nk) {
    return nk - 1 - ks < kStages - 2 ? nk - 1 - ks : kStages - 2;
}

// BT x BT output tile (cells x output channels), K in slabs of SB bytes per row.
template <int BT, int SB>
struct Shape {
    static constexpr int kStageB = 2 * BT * SB;       // cell rows, then weight rows
    static constexpr int kRPI = 1024 / SB;            // rows one direct-load instruction fills
    static constexpr int kCPR = SB / 16;              // 16-byte chunks per row
    static constexpr int kGroups = 2 * BT / kRPI;     // direct-load instructions per slab
    static constexpr int kDps = kGroups / kWaves;     // ... per wave
    static constexpr int kBlk = BT / 64;              // 32-wide blocks per wave and operand
    static constexpr int kHalves = SB / 32;           // 32-byte K pieces per slab
    static_assert(BT / kRPI % kWaves == 0, "a load index covers one operand in every wave");

    // Physical chunk = logical chunk ^ swz(row): the 16 lanes of each pass of a 16-byte
    // LDS read (gemm_addr.hpp) fall in distinct bank groups. Rows of 64 bytes: as there;
    // rows of 128 bytes: the even (odd) rows of a pass take all eight chunks.
    SLIME_HD static constexpr int swz(int r) {
        return SB == 64 ? (r >> 2) & 3 : ((r >> 1) & 1) | (((r >> 3) & 3) << 1);
    }
    // Direct load j of wave w fills rows RPI g .. of the stage, g = 4 j + w; lane l takes
    // row l / CPR of those, physical chunk l % CPR.
    SLIME_HD static constexpr int group(int j, int wave) { return kWaves * j + wave; }
    SLIME_HD static constexpr bool is_cells(int j) { return kWaves * j < BT / kRPI; }
    SLIME_HD static long long src_row(int j, int wave) {  // first row of that operand's tile
        const int g = group(j, wave);
        return (long long)(is_cells(j) ? g : g - BT / kRPI) * kRPI;
    }
    SLIME_HD static unsigned lane_off(int wave, int lane, long long row_bytes) {
        const int r = lane / kCPR;
        // group % 4 = wave, so RPI * group has the row bits that swz reads from the wave
        const int chunk = (lane % kCPR) ^ swz(kRPI * wave + r);
        return (unsigned)(r * row_bytes + chunk * 16);
    }
    SLIME_HD static unsigned lds_off(int j, int wave) { return (unsigned)(group(j, wave) * 1024); }
    // Fragment read of 32-row block q of either operand, 32-byte piece kk: row lane % 32,
    // logical chunk 2 kk + lane / 32.
    SLIME_HD static unsigned frag_off(int wave_half, int lane, int kk, bool weights) {
        const int r = lane & 31, half = lane >> 5;
        return (unsigned)((wave_half * (BT / 2) + (weights ? BT : 0) + r) * SB +
                          (((2 * kk + half) ^ swz(r)) << 4));
    }
    SLIME_HD static constexpr unsigned block_off(int q) { return (unsigned)(q * 32 * SB); }
};

// Row tiles per batch: the last one is moved back to end with the batch, so its first
// rows repeat rows of the tile before (the same values, written twice) and no tile
// reads or writes outside the batch. Needs rows_per_batch >= BT.
SLIME_HD int tiles_per_batch(int BT, int rows_per_batch) { return (rows_per_batch + BT - 1) / BT; }
SLIME_HD long long tile_row0(int BT, int mt, int rows_per_batch, int* batch) {
    const int tpb = tiles_per_batch(BT, rows_per_batch);
    const int b = mt / tpb, i = mt - b * tpb;
    const int r = i * BT < rows_per_batch - BT ? i * BT : rows_per_batch - BT;
    *batch = b;
    return (long long)b * rows_per_batch + r;
}

// Tile of a workgroup: XCD x (workgroup % 8) takes the x-th eighth of the tiles, so
// neighbouring tiles share its L2; -1 past that eighth's end. Launch 8 * ceil(n / 8).
SLIME_HD int tile_of_block(int block, int ntiles) {
    const int span = (ntiles + 7) >> 3;
    const int t = (block & 7) * span + (block >> 3);
    return (block >> 3) < span && t < ntiles ? t : -1;
}

}  // namespace gemm_small
}  // namespace slime
