// Host replay of the 128- and 64-wide tile GEMM's addresses (slime_amd/csrc/gemm_small.hip)
// through the kernel's own address functions (gemm_small_addr.hpp). Test infrastructure:
// built with g++ by tests/test_gemm_small_addr.py.
//
// For every workgroup, wave and lane of one launch it checks that each direct load reads
// inside A or Bt and fills its own 16 bytes of a stage, that every fragment read finds the
// row and 16-byte chunk its MFMA needs, that each tile lies inside one batch and one output
// plane, that the tiles are visited once, and that they cover every output row and column;
// and, for one wave's walk over the K slabs, that each vmcnt wait covers its slab under
// in-order completion of the wave's direct loads (no looser, no stricter), that a step reads
// the stage which holds its slab, and that no load fills a stage still to be read.
//
// Usage: gemm_small_replay TILE SLAB M N K elem rows_per_batch bt_batch_stride bt_elems ncol [plant]
//   plant "past-end": model the last tile of a batch as starting at its grid position (a
//   planted mistake: it would read past a ragged batch's end)
//   plant "loose-wait": model every wait one slab looser than the kernel's
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "../slime_amd/csrc/gemm_small_addr.hpp"

using namespace slime::gemm_small;

namespace {

[[noreturn]] void fail(const char* what, long long a, long long b, long long c) {
    std::printf("FAIL %s (%lld, %lld, %lld)\n", what, a, b, c);
    std::exit(1);
}

// The kernel's K loop as one wave sees it: kDps direct loads per slab, a wait and a barrier
// at each step, then the next slab's loads and the reads of this one.
template <int BT, int SB>
void check_ring(int nk, bool loose) {
    using S = Shape<BT, SB>;
    std::vector<int> ops;  // the slab of each direct load, in issue order
    int stage[kStages];
    for (int& s : stage) s = -1;
    auto issue = [&](int ks, int step) {
        int& held = stage[ks % kStages];
        if (held >= step) fail("a load fills a stage still to be read", ks, held, step);
        held = ks;
        for (int j = 0; j < S::kDps; ++j) ops.push_back(ks);
    };
    for (int ks = 0; ks < kStages - 1 && ks < nk; ++ks) issue(ks, 0);
    for (int ks = 0; ks < nk; ++ks) {
        const int n = younger_slabs(ks, nk) * S::kDps + (loose ? S::kDps : 0);
        if (n > 63) fail("vmcnt immediate beyond the 6-bit counter", ks, n, 0);
        long long last = (long long)ops.size() - 1;
        while (last >= 0 && ops[last] != ks) --last;
        const long long younger = (long long)ops.size() - 1 - last;
        if (last < 0) fail("wait for a slab never loaded", ks, nk, n);
        if (n > younger) fail("wait too loose: slab may be incomplete", ks, n, younger);
        if (n < younger) fail("wait stricter than needed", ks, n, younger);
        if (ks + kStages - 1 < nk) issue(ks + kStages - 1, ks);
        if (stage[ks % kStages] != ks) fail("step reads a stage that holds another slab", ks, stage[ks % kStages], 0);
    }
}

template <int BT, int SB>
void run(long long M, long long N, long long K, int elem, int rpb, long long bt_stride, long long bt_elems,
         int ncol, const char* planted) {
    using S = Shape<BT, SB>;
    const long long row_bytes = K * elem;
    const int nN = (int)(N / BT), nk = (int)(row_bytes / SB);
    if (N % BT || ncol % BT || row_bytes % SB || rpb < BT || M % rpb) fail("shape", M, N, K);
    const int ntiles = (int)(M / rpb) * tiles_per_batch(BT, rpb) * nN;
    const bool plant = !std::strcmp(planted, "past-end");
    check_ring<BT, SB>(nk, !std::strcmp(planted, "loose-wait"));
    std::vector<int> seen(ntiles, 0);
    std::vector<char> rows(M, 0);
    const int grid = 8 * ((ntiles + 7) / 8);
    for (int blk = 0; blk < grid; ++blk) {
        const int t = tile_of_block(blk, ntiles);
        if (t < 0) continue;
        if (t >= ntiles || seen[t]++) fail("tile visited twice or out of range", blk, t, ntiles);
        int b;
        long long m0 = tile_row0(BT, t / nN, rpb, &b);
        if (plant) m0 = (long long)b * rpb + (t / nN - (long long)b * tiles_per_batch(BT, rpb)) * BT;
        const long long n0 = (long long)(t % nN) * BT;
        if (m0 / rpb != b || (m0 + BT - 1) / rpb != b) fail("tile outside its batch", t, m0, b);
        if (n0 / ncol != (n0 + BT - 1) / ncol) fail("tile over two planes", t, n0, ncol);
        for (int r = 0; r < BT; ++r) rows[m0 + r] = 1;
        // What each 16 bytes of a stage hold after slab ks: (row of the stage, logical chunk).
        std::vector<int> held(S::kStageB / 16, -1);
        for (int w = 0; w < kWaves; ++w)
            for (int j = 0; j < S::kDps; ++j)
                for (int l = 0; l < 64; ++l) {
                    const long long off = S::src_row(j, w) * row_bytes + S::lane_off(w, l, row_bytes);
                    const long long base = S::is_cells(j) ? m0 * row_bytes : (b * bt_stride + n0 * K) * elem;
                    const long long size = S::is_cells(j) ? M * row_bytes : bt_elems * elem;
                    for (int ks : {0, nk - 1}) {
                        const long long a = base + off + (long long)ks * SB;
                        if (a < 0 || a + 16 > size) fail("direct load out of range", t, a, size);
                    }
                    const unsigned dst = S::lds_off(j, w) + 16u * l;
                    if (dst + 16 > (unsigned)S::kStageB || held[dst / 16] != -1) fail("stage slot", j, w, l);
                    const long long srow = off / row_bytes, chunk = off % row_bytes / 16;
                    if (chunk >= S::kCPR) fail("chunk past the slab", j, l, chunk);
                    held[dst / 16] = (int)((srow + (S::is_cells(j) ? 0 : BT)) * S::kCPR + chunk);
                }
        for (int wh = 0; wh < 2; ++wh)
            for (int op = 0; op < 2; ++op)
                for (int kk = 0; kk < S::kHalves; ++kk)
                    for (int q = 0; q < S::kBlk; ++q)
                        for (int l = 0; l < 64; ++l) {
                            const unsigned a = S::frag_off(wh, l, kk, op) + S::block_off(q);
                            if (a % 16 || a + 16 > (unsigned)S::kStageB) fail("fragment read", a, kk, q);
                            const int row = (op ? BT : 0) + wh * (BT / 2) + 32 * q + (l & 31);
                            if (held[a / 16] != row * S::kCPR + 2 * kk + (l >> 5)) fail("fragment data", row, kk, l);
                        }
    }
    for (int t = 0; t < ntiles; ++t)
        if (!seen[t]) fail("tile missed", t, ntiles, 0);
    for (long long r = 0; r < M; ++r)
        if (!rows[r]) fail("row missed", r, M, 0);
    std::printf("OK %d tiles\n", ntiles);
}

}  // namespace

int main(int argc, char** argv) {
    if (argc < 11) return 2;
    const int tile = std::atoi(argv[1]), slab = std::atoi(argv[2]);
    long long v[8];
    for (int i = 0; i < 8; ++i) v[i] = std::atoll(argv[3 + i]);
    const char* plant = argc > 11 ? argv[11] : "";
    if (tile == 128 && slab == 64)
        run<128, 64>(v[0], v[1], v[2], (int)v[3], (int)v[4], v[5], v[6], (int)v[7], plant);
    else if (tile == 64 && slab == 128)
        run<64, 128>(v[0], v[1], v[2], (int)v[3], (int)v[4], v[5], v[6], (int)v[7], plant);
    else
        return 2;
    return 0;
}
