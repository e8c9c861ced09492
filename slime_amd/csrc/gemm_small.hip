// gemm_small.hip — the projection GEMM in 128- and 64-wide tiles, for the shapes that the
// 256 x 256 persistent kernel (gemm_tile.hpp) does not tile or does not fill the card on:
// grids whose cell count is no multiple of 256 (G an odd multiple of 8), narrow heads
// (C = 64 or 128) and small batches, forward, taped and with the dX GEMM's addend.
//
// Same operand roles, LDS swizzle idea and rounding as the 256-wide kernel; what differs
// is the balance: one tile per workgroup and two or more workgroups per CU, so one's
// epilogue and load latency run beside another's K loop, and a ragged row count ends in
// a tile moved back to the batch's end (gemm_small_addr.hpp) instead of a masked one.
//
// What bounds it: 128-wide bf16 tiles read 16 KiB of fragments from LDS per 128 cycles of
// MFMAs, the LDS rate, and reach 730 TFLOP/s at 65,536 x 1536 x 512; fp32 tiles are bound
// by the matrix cores (137 of 157 TFLOP/s); the smallest products (M <= 1024, K <= 192)
// take 4 us, a launch and two memory round trips. Three stages (48 KiB, three workgroups
// per CU) instead of four: 16,384 x 1536 x 512 fp32 197 -> 192 us, 65,536 x 384 x 128 bf16
// 20.5 -> 18.8 us, no shape slower. The choice of tile: gemm_rule.hpp.
#include "common.hpp"
#include "gemm_rule.hpp"
#include "gemm_small_addr.hpp"
#include "kernels.hpp"

namespace slime {
namespace {

using namespace gemm_small;

enum Mode { kPlain = 0, kAdd = 1, kTape = 2 };

__device__ __forceinline__ void lds_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // s_waitcnt lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// s_waitcnt vmcnt(n)
template <int n>
__device__ __forceinline__ void wait_vm() {
    static_assert(n < 64, "vmcnt has 6 bits");
    __builtin_amdgcn_s_waitcnt(((n & 15) | (((n >> 4) & 3) << 14)) | 0x0F70);
}

template <typename T>
__device__ __forceinline__ void mfma_block(f32x16& acc, const u32x4& w, const u32x4& x) {
    if constexpr (sizeof(T) == 2) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_v, w),
                                                      __builtin_bit_cast(bf16x8_v, x), acc, 0, 0, 0);
    } else {
        const f32x4 wv = __builtin_bit_cast(f32x4, w), xv = __builtin_bit_cast(f32x4, x);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(wv[e], xv[e], acc, 0, 0, 0);
    }
}

// One 32 x 32 block: lane l holds cell l % 32, channels 8 q + 4 (l / 32) + e in value
// 4 q + e. bf16: the two halves of the wave trade 4-channel pieces, so that a lane
// stores 8 consecutive channels; fp32: 4 channels are 16 bytes already.
template <typename T>
__device__ __forceinline__ void store_block(T* out, int ncol, int lane, float (&v)[16]) {
    const int cell = lane & 31, half = lane >> 5;
    if constexpr (sizeof(T) == 2) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const int q = 2 * p;
            const u32x2 a = __builtin_amdgcn_permlane32_swap(pack_bf16x2(v[4 * q], v[4 * q + 1]),
                                                             pack_bf16x2(v[4 * q + 4], v[4 * q + 5]), false, false);
            const u32x2 b = __builtin_amdgcn_permlane32_swap(pack_bf16x2(v[4 * q + 2], v[4 * q + 3]),
                                                             pack_bf16x2(v[4 * q + 6], v[4 * q + 7]), false, false);
            *reinterpret_cast<u32x4*>(out + (long long)cell * ncol + 8 * (q + half)) = u32x4{a[0], b[0], a[1], b[1]};
        }
    } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *reinterpret_cast<float4*>(out + (long long)cell * ncol + 8 * q + 4 * half) =
                make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
    }
}

template <typename T, int BT, int SB, Mode kMode>
__global__ __launch_bounds__(kThreads, 2) void gemm_small_kernel(GemmArgs g, void* aux) {
    using S = Shape<BT, SB>;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[kStages * S::kStageB];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 1, wn = wave >> 1;
    const int nN = g.N / BT, nk = g.K * (int)sizeof(T) / SB;
    const int ntiles = g.M / g.rows_per_batch * tiles_per_batch(BT, g.rows_per_batch) * nN;
    const int t = tile_of_block(blockIdx.x, ntiles);
    if (t < 0) return;
    int batch;
    const long long m0 = tile_row0(BT, t / nN, g.rows_per_batch, &batch);
    const int n0 = t % nN * BT;
    const long long row_bytes = (long long)g.K * (long long)sizeof(T);
    const char* xs = reinterpret_cast<const char*>(static_cast<const T*>(g.A)) + m0 * row_bytes;
    const char* ws = reinterpret_cast<const char*>(static_cast<const T*>(g.Bt) + batch * g.bt_batch_stride) +
                     n0 * row_bytes;
    const unsigned voff = S::lane_off(wave, lane, row_bytes);
    auto issue = [&](int ks, int stage) {
        const unsigned sb = lds_addr(lds) + stage * S::kStageB;
#pragma unroll
        for (int j = 0; j < S::kDps; ++j)
            dma16_lds((S::is_cells(j) ? xs : ws) + S::src_row(j, wave) * row_bytes + (long long)ks * SB, voff,
                      sb + S::lds_off(j, wave));
    };

    f32x16 acc[S::kBlk][S::kBlk];  // [channel block][cell block]
#pragma unroll
    for (int i = 0; i < S::kBlk; ++i)
#pragma unroll
        for (int j = 0; j < S::kBlk; ++j) acc[i][j] = f32x16{};

    for (int ks = 0; ks < kStages - 1 && ks < nk; ++ks) issue(ks, ks);
    int rd = 0, wr = kStages - 1;
    for (int ks = 0; ks < nk; ++ks) {
        static_assert(kStages == 3, "one slab is younger than the one waited for, none at the end");
        if (younger_slabs(ks, nk) > 0) wait_vm<S::kDps>();
        else wait_vm<0>();
        lds_barrier();  // slab ks is in LDS; every wave has read slab ks - 1, whose stage is free
        if (ks + kStages - 1 < nk) issue(ks + kStages - 1, wr);
        const unsigned char* st = lds + rd * S::kStageB;
#pragma unroll
        for (int kk = 0; kk < S::kHalves; ++kk) {
            u32x4 w[S::kBlk], x[S::kBlk];
            const unsigned ox = S::frag_off(wm, lane, kk, false), ow = S::frag_off(wn, lane, kk, true);
#pragma unroll
            for (int q = 0; q < S::kBlk; ++q) {
                x[q] = *reinterpret_cast<const u32x4*>(st + ox + S::block_off(q));
                w[q] = *reinterpret_cast<const u32x4*>(st + ow + S::block_off(q));
            }
#pragma unroll
            for (int i = 0; i < S::kBlk; ++i)
#pragma unroll
                for (int j = 0; j < S::kBlk; ++j) mfma_block<T>(acc[i][j], w[i], x[j]);
        }
        rd = rd + 1 == kStages ? 0 : rd + 1;
        wr = wr + 1 == kStages ? 0 : wr + 1;
    }

    // The tile lies in one output plane (ncol is a multiple of BT): uniform activation.
    const int plane = n0 / g.ncol;
    const long long o0 = (m0 + wm * (BT / 2)) * g.ncol + (n0 - plane * g.ncol + wn * (BT / 2));
    const int act = g.act[plane];
#pragma unroll
    for (int j = 0; j < S::kBlk; ++j)
#pragma unroll
        for (int i = 0; i < S::kBlk; ++i) {
            const long long o = o0 + (long long)j * 32 * g.ncol + i * 32;
            float v[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) v[e] = acc[i][j][e];
            if constexpr (kMode == kAdd) {
                const float* add = static_cast<const float*>(aux) + o;
                const int cell = lane & 31, half = lane >> 5;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 d = *reinterpret_cast<const float4*>(add + (long long)cell * g.ncol + 8 * q + 4 * half);
                    v[4 * q] += d.x, v[4 * q + 1] += d.y, v[4 * q + 2] += d.z, v[4 * q + 3] += d.w;
                }
                store_block<float>(static_cast<float*>(g.out[0]) + o, g.ncol, lane, v);
            } else {
                if (act == 2) {
                    if constexpr (kMode == kTape) store_block<T>(static_cast<T*>(aux) + o, g.ncol, lane, v);
                    gelu_tanh_n(v);
                } else if (act == 1) {
#pragma unroll
                    for (int e = 0; e < 16; ++e) v[e] = v[e] > 0.f ? v[e] : 0.f;
                }
                store_block<T>(static_cast<T*>(g.out[plane]) + o, g.ncol, lane, v);
            }
        }
}

template <typename T, Mode kMode>
hipError_t launch_mode(int tile, const GemmArgs& a, void* aux, hipStream_t s) {
    const int ntiles = a.M / a.rows_per_batch * tiles_per_batch(tile, a.rows_per_batch) * (a.N / tile);
    const dim3 grid(8 * ((ntiles + 7) / 8));
    if (tile == 128)
        hipLaunchKernelGGL((gemm_small_kernel<T, 128, 64, kMode>), grid, dim3(kThreads), 0, s, a, aux);
    else
        hipLaunchKernelGGL((gemm_small_kernel<T, 64, 128, kMode>), grid, dim3(kThreads), 0, s, a, aux);
    return hipGetLastError();
}

template <Mode kMode>
hipError_t launch_small(int dtype, int tile, const GemmArgs& a, void* aux, hipStream_t s) {
    if (!gemm_small_fits(dtype, tile, a)) return hipErrorInvalidValue;
    return dtype == 1 ? launch_mode<bf16_t, kMode>(tile, a, aux, s) : launch_mode<float, kMode>(tile, a, aux, s);
}

}  // namespace

bool gemm_small_fits(int dtype, int tile, const GemmArgs& a) {
    return gemm_rule::fits_small(tile, {dtype, a.M, a.N, a.K, a.ncol, a.rows_per_batch});
}

hipError_t launch_gemm_small(int dtype, int tile, const GemmArgs& a, hipStream_t s) {
    return launch_small<kPlain>(dtype, tile, a, nullptr, s);
}
hipError_t launch_gemm_small_tape(int dtype, int tile, const GemmArgs& a, void* pre, hipStream_t s) {
    return pre ? launch_small<kTape>(dtype, tile, a, pre, s) : hipErrorInvalidValue;
}
hipError_t launch_gemm_small_add(int dtype, int tile, const GemmArgs& a, const float* add, hipStream_t s) {
    if (!add || a.N != a.ncol || a.act[0] != 0 || add == a.out[0]) return hipErrorInvalidValue;
    return launch_small<kAdd>(dtype, tile, a, const_cast<float*>(add), s);
}

}  // namespace slime
