// fitness.hip — E1-E5: fitness = effective_rank x coherence per (batch, head).
//
// Reference:
//   E1 Gram      A_h = (1/N) sum_cells x_h x_h^T   failed_attempts/pseudopod.cu:366-384
//                (over the last state of the history; per head, not head-averaged)
//   E2 Jacobi    two-sided Jacobi, skip |a_pq| <= 1e-6, <= 30 sweeps, stop when
//                sum |a_pq| < 1e-6 * n              failed_attempts/pseudopod.cu:391-436,
//                                                   slime/kernels/warp_ca.cu:20,51-63
//                sigma_i = sqrt|lambda_i|           slime/kernels/warp_ca.cu:101-103
//   E3 rank      exp(-sum p log(p+1e-7)), p = sigma/(sum sigma + 1e-7)
//                                                   slime/kernels/warp_ca.cu:118-143
//   E4 coherence (mean_t Pearson(X_t, X_{t-1}) + 1) / 2, t = 1..T-1
//                                                   slime/core/organism.cu:256-257
//   E5 fitness   erank * coh                        slime/kernels/warp_ca.cu:219
//
// The reference launches SVD, rank and coherence as dynamic-parallelism children
// of one parent (slime/kernels/warp_ca.cu:178-226). Here two stream-ordered
// kernels do the work: a wide pass over the history that writes per-chunk fp64
// Gram and moment partials, then one workgroup per (batch, head) that reduces them in
// fixed order, runs the cyclic Jacobi on the fp64 matrix in LDS, and finishes
// rank, coherence and fitness.
#include <algorithm>
#include <cstring>
#include <mutex>

#include "common.hpp"
#include "fp64.hpp"
#include "jacobi_wave.hpp"
#include "kernels.hpp"

// Scratch of the allocation-free entry point slime_ca_fitness_static: the Gram and
// moment partials of one call. One copy per GPU, created when the code object loads
// on that device and held until the process ends; every call on a GPU shares it.
// Calls on different streams are ordered by launch_fitness_static (each waits for the
// previous call's event); calls under graph capture are not, and replays that overlap
// on one GPU race. Host code never takes the array's name as an address (on the host
// it is only a stand-in for the symbol): the device address is looked up once per
// device and kernels receive that pointer.
static __device__ __align__(256) unsigned char scratch[slime::kFitnessScratchBytes];

namespace slime {
namespace {

// State t of the history starts t * f.t_stride bytes after f.hist. The stride may be
// negative: two separately allocated states form a history of two.
template <typename T>
__device__ __forceinline__ const T* history_state(const FitnessArgs& f, int t) {
    return reinterpret_cast<const T*>(static_cast<const char*>(f.hist) + t * f.t_stride);
}

__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m, 64);
    return v;
}

// The partial pass has two kinds of workgroups in one launch, interleaved so that the
// matrix cores' work runs beside the other kind's streaming:
//   moments: per (batch, chunk of cells) and every state t of the history, each head's sums
//     S1 = sum x_t, S2 = sum x_t^2 and P = sum x_{t-1} x_t (P of state 0 is 0), which give
//     the lag-1 moments of each consecutive pair. A workgroup reads whole cells, all heads
//     (a state's rows are contiguous), and a thread's 16-byte pieces always belong to one
//     head. Bound by HBM.
//   Gram: per (batch, head, chunk) the D x D Gram partial of the last state on the fp64
//     matrix cores (v_mfma_f64_16x16x4), the blocks on and above the diagonal only.
// Products of the fp32 values are exact in fp64 and accumulate in fp64, so the partials
// carry no accumulation error that the Jacobi solve could amplify on a nearly singular
// Gram (small eigenvalues enter the rank through their square roots).
//
// Measured at 8 states of 16 x 128^2 x 512 bf16 (2.15 GB): 461 us = 4.66 TB/s (a copy reaches
// 4.84), 784 us with the Gram on the VALU in the same workgroups and one head's 128-byte row
// segments per workgroup; 2 states of 128^2 x 512 fp32: 27 us, 127 us with 128 workgroups
// and eight states' loads whatever T.
constexpr int kUnit = 64;  // cells per Gram step of a workgroup: 16 per wave

// Workgroup k of n_g Gram and n_m moment workgroups: groups of 8 (one per XCD), the kinds
// spread evenly over the launch. Returns its kind's index; -1 past the end.
__device__ __forceinline__ long long split_kinds(long long k, long long n_g, long long n_m, bool* gram) {
    const long long gg = (n_g + 7) / 8, gm = (n_m + 7) / 8, g = k >> 3;
    const long long before = g * gg / (gg + gm), after = (g + 1) * gg / (gg + gm);
    *gram = after > before;
    const long long idx = 8 * (*gram ? before : g - before) + (k & 7);
    return idx < (*gram ? n_g : n_m) ? idx : -1;
}

template <typename T>
__device__ __forceinline__ void unpack_piece(const uint4& v, float (&e)[16 / sizeof(T)]) {
    if constexpr (sizeof(T) == 2) {
        e[0] = bf16lo(v.x), e[1] = bf16hi(v.x), e[2] = bf16lo(v.y), e[3] = bf16hi(v.y);
        e[4] = bf16lo(v.z), e[5] = bf16hi(v.z), e[6] = bf16lo(v.w), e[7] = bf16hi(v.w);
    } else {
        e[0] = __builtin_bit_cast(float, v.x), e[1] = __builtin_bit_cast(float, v.y);
        e[2] = __builtin_bit_cast(float, v.z), e[3] = __builtin_bit_cast(float, v.w);
    }
}

// The geometry of a moment workgroup's reads.
template <typename T, int D>
struct Rows {
    static constexpr int kCE = 16 / (int)sizeof(T);             // elements per 16-byte piece
    static constexpr int kPPC = kHeads * D / kCE;                // pieces per cell, a power of two
    static constexpr int kPPH = D / kCE;                         // ... of one head
    static constexpr int kCells = 256 / kPPC;                    // cells the workgroup reads at once
    static constexpr int kPPT = 2;                               // pieces per thread and state in flight
    static constexpr int kStage = kCells * kPPT;                 // cells per stage; divides 64
    static constexpr int kHW = kPPC <= 64 ? kHeads : 64 / kPPH;  // heads in a wave
};

// Sum over the lanes of a wave that hold the same head: the kPPH lanes of a cell, then the
// wave's cells.
template <typename R>
__device__ __forceinline__ double head_sum(double v) {
    if constexpr (R::kPPH >= 2) v += dpp_f64<0xB1>(v);
    if constexpr (R::kPPH >= 4) v += dpp_f64<0x4E>(v);
    if constexpr (R::kPPH >= 8) v += dpp_f64<0x141>(v);
    if constexpr (R::kPPH >= 16) v += dpp_f64<0x140>(v);
#pragma unroll
    for (int m = R::kPPC; m < 64; m *= 2) v += __shfl_xor(v, m, 64);
    return v;
}

// Moments of up to kTB states per pass over the chunk; each pass reads states tb - 1 ..
// tb + kTB - 1 once, a stage's loads all in flight together.
template <typename T, int D, int kTB>
__device__ __forceinline__ void moments(const FitnessArgs& f, int b, int chunk, double* sred) {
    using R = Rows<T, D>;
    constexpr int kItems = 3 * kTB;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const long long cells = (long long)f.G * f.G, stages = cells / R::kStage;
    const long long st0 = stages * chunk / f.mom_chunks, st1 = stages * (chunk + 1) / f.mom_chunks;
    const int row_bytes = kHeads * D * (int)sizeof(T);
    const unsigned off = (unsigned)(tid * 16);  // cell tid / kPPC of the read, piece tid % kPPC
    for (int tb = 0; tb < f.T; tb += kTB) {
        const int tn = min(kTB, f.T - tb);  // states tb .. tb + tn - 1 in this pass
        double s1[kTB], s2[kTB], pr[kTB];
#pragma unroll
        for (int k = 0; k < kTB; ++k) s1[k] = s2[k] = pr[k] = 0.0;
        for (long long st = st0; st < st1; ++st) {
            const long long base = (b * cells + st * R::kStage) * row_bytes;
            uint4 x[kTB + 1][R::kPPT];  // states tb - 1 .. tb + kTB - 1
#pragma unroll
            for (int k = 0; k <= kTB; ++k)
#pragma unroll
                for (int j = 0; j < R::kPPT; ++j) x[k][j] = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
            for (int k = 0; k <= kTB; ++k) {
                const int t = tb + k - 1;
                if (t < 0 || t >= f.T) continue;  // uniform; those sums are unused
                const char* src = static_cast<const char*>(f.hist) + t * f.t_stride + base;
#pragma unroll
                for (int j = 0; j < R::kPPT; ++j)
                    x[k][j] = *reinterpret_cast<const uint4*>(src + j * 4096 + off);
            }
#pragma unroll
            for (int k = 0; k < kTB; ++k)
#pragma unroll
                for (int j = 0; j < R::kPPT; ++j) {
                    float a[R::kCE], e[R::kCE];
                    unpack_piece<T>(x[k][j], a);
                    unpack_piece<T>(x[k + 1][j], e);
#pragma unroll
                    for (int u = 0; u < R::kCE; ++u) {
                        const double va = a[u], vb = e[u];
                        s1[k] += vb;
                        s2[k] = __builtin_fma(vb, vb, s2[k]);
                        pr[k] = __builtin_fma(va, vb, pr[k]);
                    }
                    // one piece at a time: the converted values stay few
                    __builtin_amdgcn_sched_barrier(0);
                }
        }
        // Workgroup sums per head in a fixed order (lanes, then waves).
        const int h = (tid % R::kPPC) / R::kPPH;
        const bool first = (lane & (R::kPPH - 1)) == 0 && lane / R::kPPH < R::kHW;
#pragma unroll
        for (int k = 0; k < kTB; ++k) {
            const double v[3] = {head_sum<R>(s1[k]), head_sum<R>(s2[k]), head_sum<R>(pr[k])};
            if (first) {
#pragma unroll
                for (int u = 0; u < 3; ++u) sred[(wave * kHeads + h) * kItems + 3 * k + u] = v[u];
            }
        }
        __syncthreads();
        for (int i = tid; i < kHeads * 3 * tn; i += 256) {
            const int hh = i / (3 * tn), it = i - hh * (3 * tn);
            double sum = 0.0;
#pragma unroll
            for (int w = 0; w < 4; ++w)
                if (R::kHW == kHeads || (w * R::kHW) % kHeads == hh / R::kHW * R::kHW)
                    sum += sred[(w * kHeads + hh) * kItems + it];
            f.mom_part[((((long long)b * kHeads + hh) * f.mom_chunks + chunk) * f.T + tb) * 3 + it] =
                tb == 0 && it == 2 ? 0.0 : sum;
        }
        __syncthreads();
    }
}

typedef __attribute__((ext_vector_type(4))) double f64x4;

// Gram partial of the last state over one chunk of one head. Lane (i = lane % 16, k = lane /
// 16) reads channels NR i .. NR i + NR - 1 of cell k of a group of four; channel NR i + r is
// row (and column) i of 16-wide block r, so that one register is an operand of either side
// of v_mfma_f64_16x16x4 (row or column lane % 16, k = lane / 16; result value e of a lane:
// row lane / 16 + 4 e, column lane % 16).
template <typename T, int D>
__device__ __forceinline__ void gram(const FitnessArgs& f, int bh, int chunk, double* sred) {
    constexpr int NR = D >= 16 ? D / 16 : 1, kBlocks = NR * (NR + 1) / 2;
    constexpr int kBytes = NR * (int)sizeof(T);  // per lane and cell: 2 to 16
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int i = lane & 15, kq = lane >> 4;
    const long long cells = (long long)f.G * f.G, units = cells / kUnit;
    const long long u0 = units * chunk / f.chunks, u1 = units * (chunk + 1) / f.chunks;
    const int b = bh / kHeads, h = bh % kHeads;
    constexpr int C = kHeads * D;
    const bool on = D >= 16 || i < D;  // D = 8: half of the 16 rows
    const T* src = history_state<T>(f, f.T - 1) + (long long)b * cells * C + (long long)(16 * wave + kq) * C + h * D +
                   (on ? NR * i : 0);
    struct Raw {
        unsigned w[4][kBytes >= 4 ? kBytes / 4 : 1];  // four groups of four cells
    };
    auto load = [&](long long u, Raw& r) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const T* p = src + (u * kUnit + 4 * g) * C;
            if constexpr (kBytes == 16) {
                const uint4 v = *reinterpret_cast<const uint4*>(p);
                r.w[g][0] = v.x, r.w[g][1] = v.y, r.w[g][2] = v.z, r.w[g][3] = v.w;
            } else if constexpr (kBytes == 8) {
                const uint2 v = *reinterpret_cast<const uint2*>(p);
                r.w[g][0] = v.x, r.w[g][1] = v.y;
            } else if constexpr (kBytes == 4) {
                r.w[g][0] = *reinterpret_cast<const unsigned*>(p);
            } else {
                r.w[g][0] = *p;
            }
            if (!on) r.w[g][0] = 0u;
        }
    };
    f64x4 acc[kBlocks];
#pragma unroll
    for (int k = 0; k < kBlocks; ++k) acc[k] = f64x4{0.0, 0.0, 0.0, 0.0};
    Raw cur, nxt;
    if (u0 < u1) load(u0, cur);
    for (long long u = u0; u < u1; ++u) {
        load(u + 1 < u1 ? u + 1 : u, nxt);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            double x[NR];
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                if constexpr (sizeof(T) == 4) x[r] = __builtin_bit_cast(float, cur.w[g][r]);
                else x[r] = r & 1 ? bf16hi(cur.w[g][r / 2]) : bf16lo(cur.w[g][r / 2]);
            }
            int k = 0;
#pragma unroll
            for (int r1 = 0; r1 < NR; ++r1)
#pragma unroll
                for (int r2 = r1; r2 < NR; ++r2, ++k)
                    acc[k] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[r1], x[r2], acc[k], 0, 0, 0);
        }
        cur = nxt;
    }
    // Waves 1, 2, 3 added to wave 0 in turn, then the elements on and above the diagonal.
    for (int w = 1; w < 4; ++w) {
        if (wave == w) {
#pragma unroll
            for (int k = 0; k < kBlocks; ++k)
#pragma unroll
                for (int e = 0; e < 4; ++e) sred[(4 * k + e) * 64 + lane] = acc[k][e];
        }
        __syncthreads();
        if (wave == 0) {
#pragma unroll
            for (int k = 0; k < kBlocks; ++k)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[k][e] += sred[(4 * k + e) * 64 + lane];
        }
        __syncthreads();
    }
    if (wave != 0) return;
    double* gp = f.gram_part + ((long long)bh * f.chunks + chunk) * D * D;
    int k = 0;
#pragma unroll
    for (int r1 = 0; r1 < NR; ++r1)
#pragma unroll
        for (int r2 = r1; r2 < NR; ++r2, ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int ri = kq + 4 * e, c1 = NR * ri + r1, c2 = NR * i + r2;
                if (D < 16 && (ri >= D || i >= D)) continue;
                if (r1 != r2 || ri <= i) gp[c1 <= c2 ? c1 * D + c2 : c2 * D + c1] = acc[k][e];
            }
}

template <typename T, int D, int kTB>
__global__ __launch_bounds__(256, 2) void fitness_partial_kernel(FitnessArgs f) {
    constexpr int NR = D >= 16 ? D / 16 : 1;
    constexpr int kGramLds = NR * (NR + 1) / 2 * 4 * 64, kMomLds = 4 * kHeads * 3 * kTB;
    __shared__ double sred[kGramLds > kMomLds ? kGramLds : kMomLds];
    bool is_gram;
    const long long n_g = (long long)f.B * kHeads * f.chunks, n_m = (long long)f.B * f.mom_chunks;
    const long long idx = split_kinds(blockIdx.x, n_g, n_m, &is_gram);
    if (idx < 0) return;
    if (is_gram) gram<T, D>(f, (int)(idx / f.chunks), (int)(idx % f.chunks), sred);
    else moments<T, D, kTB>(f, (int)(idx / f.mom_chunks), (int)(idx % f.mom_chunks), sred);
}

// Keeps the compiler from moving LDS accesses across this point. The block is one
// wave and LDS executes a wave's accesses in issue order, so program order is all
// the ordering that one lane's write and another lane's later read need.
__device__ __forceinline__ void lds_order() { asm volatile("" ::: "memory"); }

// Workgroup barrier for LDS data.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // s_waitcnt lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// One workgroup per (batch, head): fixed-order reduction of the partials, the cyclic
// two-sided Jacobi solve in fp64, then rank, coherence and fitness.
//
// The solve rotates the pairs (p, q) in the reference's cyclic row order
// (failed_attempts/pseudopod.cu:391-436) and skips |a_pq| <= 1e-6. That absolute
// threshold makes the converged diagonal depend on the order when the Gram is nearly
// singular, so the order is kept. What bounds it is the chain of a rotation's fp64
// operations (two hardware estimates in a row with their refinements, ~450 cycles), so
// the solve runs the cyclic order as a wave front (jacobi_wave.hpp): the up to D / 2
// rotations of a step share no index, commute, and run in the lanes of one wave, D steps
// to a sweep instead of D (D - 1) / 2 rotations; every rotation sees the values that the
// serial order would give it, up to the fp64 rounding of commuted updates.
//
// Wave 0 computes the rotations, one step ahead: for step T + 1 it reads four elements
// of the matrix as it was before step T and applies step T's rotations to them itself,
// while the other waves apply step T to the whole upper triangle, from one LDS copy to
// the other; one barrier per step. The diagonal is wave 0's alone. A step without a
// rotation leaves the matrix alone.
//
// A sweep's last rotations run beside the first ones of the next sweep, so each index's
// diagonal is noted when its row of the sweep is done, and the result is the noted
// diagonal of the sweep that ends the solve: the one whose sum |a_pq| is below 1e-6 D,
// the one that rotated nothing (every later sweep would repeat it up to the limit, and
// 30 sweeps are reported, as the reference runs them), or the 30th.
//
// Measured on 128 Grams of 64 x 64 (16 pods x 8 heads, ~11.7k rotations each): 315 us,
// 2920 us as one rotation at a time. A step (~1300 cycles) is shared between the chain and
// the update's LDS traffic (48 KB of the CU's 128 B per cycle): halving the chain's hardware
// estimates took 5 %; two or four items per update thread take the whole fitness from 751 to
// 794 and 878 us.
constexpr int kFinUpdate = 512;                // threads that apply the rotations
constexpr int kFinThreads = 64 + kFinUpdate;   // wave 0 computes them

template <int D>
__global__ __launch_bounds__(kFinThreads) void fitness_finalize_kernel(FitnessArgs f) {
    using namespace jacobi_wave;
    constexpr int S = D / 2;  // pairs per step
    __shared__ double A[2][D * D];  // upper triangle
    __shared__ __attribute__((aligned(16))) double2 cs[2][D];  // new a_i = c a_i + s a_partner
    __shared__ int flag[2];  // a step's: 0 no rotation, 1 rotations, 2 the solve has ended
    __shared__ double dg[D];  // the diagonal (wave 0 only)
    __shared__ double msum[3 * 65];  // [state][S1, S2, P] over all chunks
    __shared__ double rho[64];
    __shared__ double sv[D], term[D];

    const int bh = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const double ncell = (double)f.G * f.G;
    const double tol = 1e-6;
    const int BH = gridDim.x;
    // Per-state factors of a rolled-out history (1 when the states are stored as they are).
    auto scale_of = [&](int t) { return f.scales ? f.scales[(long long)t * BH + bh] : 1.0; };
    const double s_last = scale_of(f.T - 1);
    const double gram_scale = s_last * s_last / ncell;

    // Fixed-order reduction of the Gram partials: an element sums chunks 0, 1, ... in turn.
    {
        const double* gp = f.gram_part + (long long)bh * f.chunks * D * D;
        for (int e = tid; e < D * D; e += kFinThreads) {
            if (e % D < e / D) continue;
            double s = 0.0;
#pragma unroll 8
            for (int c = 0; c < f.chunks; ++c) s += gp[(long long)c * D * D + e];
            A[0][e] = f.scales ? s * gram_scale : s / ncell;
        }
        if (tid < 2) flag[tid] = 0;
        // The moment sums: a wave per sum, its lanes striding over the chunks, then a
        // fixed tree.
        const double* mp = f.mom_part + (long long)bh * f.mom_chunks * f.T * 3;
        for (int it = tid >> 6; it < 3 * f.T; it += kFinThreads / 64) {
            double s = 0.0;
            for (int c = lane; c < f.mom_chunks; c += 64) s += mp[(long long)c * f.T * 3 + it];
            s = wave_sum_f64(s);
            if (lane == 0) msum[it] = s;
        }
    }
    __syncthreads();

    int cur = 0;
    if (tid >= 64) {
        // ---- apply step T to the matrix ----------------------------------------------------
        // One item (the block of slots d1 and d2) per thread, and in the first S threads the own
        // element of slot d1's pair.
        static_assert(S * S / 2 <= kFinUpdate, "one work item per thread");
        const int u = tid - 64;
        SLIME_JACOBI_ITEM(u, S, d1, d2, act);
        const bool pairs = u < S;
        for (int T = 0;; ++T) {
            const int sig = T & (D - 1);
            const double* M = A[cur];
            double* W = A[cur ^ 1];
            const double2* r = cs[T & 1];
            int i1, j1, i2, j2;
            slot(sig, d1, D, &i1, &j1);
            slot(sig, d2, D, &i2, &j2);
            const int ea = upper(i1, i2, D), eb = upper(i1, j2, D), ec = upper(j1, i2, D), ed = upper(j1, j2, D);
            const int ep = upper(i1, j1, D);
            // all reads at once, before the step is known to rotate anything
            const int fl = flag[T & 1];
            const double2 r1 = r[i1], r2 = r[i2];
            const double a = M[ea], b = M[eb], c = M[ec], d = M[ed];
            const double own = M[ep];
            if (fl == 2) return;
            if (fl) {
                if (act) {
                    const double ar = r1.x * a + r1.y * c, br = r1.x * b + r1.y * d;
                    const double cr = r1.x * c - r1.y * a, dr = r1.x * d - r1.y * b;
                    W[ea] = r2.x * ar + r2.y * br;
                    W[eb] = r2.x * br - r2.y * ar;
                    W[ec] = r2.x * cr + r2.y * dr;
                    W[ed] = r2.x * dr - r2.y * cr;
                }
                if (pairs) W[ep] = r1.y != 0.0 ? 0.0 : own;  // a rotated pair's element is zero now
                cur ^= 1;
            }
            lds_barrier();
        }
    }

    // ---- wave 0: the rotations of step T + 1 --------------------------------------------------
    const bool own = D == kWave || lane < D;
    double c = 1.0, s = 0.0;           // this lane's rotation of step T
    double off = 0.0, off_done = 0.0;  // this row's share of sum |a_pq|: running, and of its last whole sweep
    bool rot = false, rot_done = false;
    double diag = 0.0;                 // index `lane`'s diagonal at the end of that sweep
    int sweeps = 0;
    bool any = false;                  // step T rotates
    if (own) dg[lane] = A[0][lane * D + lane];
    // The four elements of a step, with m = q_partner_before(p): (p, m), (p, q), (q - 1, m)
    // and (q - 1, q), are at offsets linear in q (lanes without a pair read in range and
    // use nothing).
    const int lp = own ? lane : 0, m = q_partner_before(lp, D);
    const int at1 = upper(lp, m, D);
    const int at3_0 = lp > 0 ? m * D - 1 : m - D, at3_q = lp > 0 ? 1 : D;
    for (int T = 0;; ++T) {
        const int sig = (T + 1) & (D - 1);
        const Role ro = role(sig, lane, D);
        const bool pair = own && ro.pair, self = own && ro.self;
        const int q = ro.q > 0 ? ro.q : 1;
        const double* M = A[cur];
        lds_order();
        const double e1 = M[at1], e2 = M[lp * D + q], e3 = M[at3_0 + q * at3_q], e4 = M[q * (D + 1) - D];
        const double app = dg[lp];
        double aqq = dg[q];
        double2 rq = cs[T & 1][q];  // index q's rotation of step T, with index m
        asm volatile("" : "+v"(aqq));  // read here, not where it is first used
        if (!any) rq = make_double2(1.0, 0.0);
        const double x = c * e1 - s * e3, y = c * e2 - s * e4;
        const double apq = rq.y * x + rq.x * y;
        const bool real = pair && (T + 1 >= D || !ro.prev);  // sweep 0 has no sweep before it
        const double mag = real ? fabs(apq) : 0.0;
        const bool rotate = mag > tol;
        const bool any1 = __ballot(rotate) != 0;
        c = 1.0;
        s = 0.0;
        double app_now = app;
        if (any1) {
            double cr, sr;
            jacobi_rotation(app, aqq, rotate ? apq : 1.0, cr, sr);
            const double app_new = cr * cr * app + sr * sr * aqq - 2.0 * cr * sr * apq;
            const double aqq_new = sr * sr * app + cr * cr * aqq + 2.0 * cr * sr * apq;
            c = rotate ? cr : 1.0;
            s = rotate ? sr : 0.0;
            app_now = rotate ? app_new : app;
            double2* w = cs[(T + 1) & 1];
            if (own && !(ro.q < lane)) {  // a pair, or an index that rests: both writes are its own
                w[ro.q] = make_double2(c, s);
                w[lane] = make_double2(c, -s);
                dg[ro.q] = rotate ? aqq_new : aqq;
                dg[lane] = app_now;
            }
        }
        if (self) {
            off = 0.0;
            rot = false;
        }
        off += mag;
        rot = rot || rotate;
        if (own && ro.q == D - 1) {  // this row's sweep is done (index D - 1: with all others)
            diag = app_now;
            off_done = off;
            rot_done = rot;
        }
        bool end = false;
        if (sig == D - 2 && T + 1 >= 2 * D - 2) {
            sweeps = (T + 1) / D;
            const bool converged = wave_sum_f64(own ? off_done : 0.0) < tol * D;
            const bool idle = __ballot(own && rot_done) == 0;
            if (idle && !converged) sweeps = 30;
            end = converged || idle || sweeps == 30;
        }
        if (lane == 0) flag[(T + 1) & 1] = end ? 2 : (any1 ? 1 : 0);
        cur ^= any ? 1 : 0;
        any = any1;
        lds_barrier();
        if (end) break;
    }

    // Coherence from the per-state sums: pair t = (t - 1, t) has sum a = S1(t-1),
    // sum b = S1(t), sum ab = P(t), sum aa = S2(t-1), sum bb = S2(t).
    const int npair = f.T - 1;
    const double n = ncell * D;
    for (int t = lane + 1; t < f.T; t += 64) {
        double mo[5] = {msum[(t - 1) * 3], msum[t * 3], msum[t * 3 + 2], msum[(t - 1) * 3 + 1], msum[t * 3 + 1]};
        if (f.scales) {
            const double sa = scale_of(t - 1), sb = scale_of(t);
            mo[0] *= sa;
            mo[1] *= sb;
            mo[2] *= sa * sb;
            mo[3] *= sa * sa;
            mo[4] *= sb * sb;
        }
        const double cov = mo[2] - mo[0] * mo[1] / n;
        const double va = mo[3] - mo[0] * mo[0] / n;
        const double vb = mo[4] - mo[1] * mo[1] / n;
        const double den = sqrt(fmax(va, 0.0) * fmax(vb, 0.0));
        rho[t - 1] = den > 0.0 ? cov / den : 0.0;
    }
    // Singular values in descending order (each lane counts the ones before its own), then
    // the sums in that order.
    const double v = own ? sqrt(fabs(diag)) : 0.0;
    if (own) term[lane] = v;
    lds_order();
    if (own) {
        int rank = 0;
#pragma unroll 8
        for (int i = 0; i < D; ++i) {
            const double o = term[i];
            rank += o > v || (o == v && i < lane) ? 1 : 0;
        }
        sv[__ballot(v != v) ? lane : rank] = v;  // NaN has no rank, and every order gives NaN
    }
    lds_order();
    double sum = 0.0;
#pragma unroll 8
    for (int i = 0; i < D; ++i) sum += sv[i];
    if (own) {
        const double pr = div_rn(sv[lane], sum + 1e-7);
        term[lane] = -pr * log(pr + 1e-7);
    }
    lds_order();
    if (lane == 0) {
        double ent = 0.0;
#pragma unroll 8
        for (int i = 0; i < D; ++i) ent += term[i];
        const double er = exp(ent);
        double rs_ = 0.0;
        for (int t = 0; t < npair; ++t) rs_ += rho[t];
        const double coh = (rs_ / npair + 1.0) * 0.5;
        f.erank[bh] = (float)er;
        f.coh[bh] = (float)coh;
        f.fitness[bh] = (float)(er * coh);
        if (f.sweeps) f.sweeps[bh] = sweeps;
    }
}

template <typename T, int D>
hipError_t launch_td(const FitnessArgs& f, hipStream_t s) {
    const long long n_g = (long long)f.B * kHeads * f.chunks, n_m = (long long)f.B * f.mom_chunks;
    const dim3 grid((unsigned)(8 * ((n_g + 7) / 8 + (n_m + 7) / 8)));
    // States per pass: a short history needs no registers for eight.
    if (f.T <= 2)
        hipLaunchKernelGGL((fitness_partial_kernel<T, D, 2>), grid, dim3(256), 0, s, f);
    else if (f.T <= 4)
        hipLaunchKernelGGL((fitness_partial_kernel<T, D, 4>), grid, dim3(256), 0, s, f);
    else
        hipLaunchKernelGGL((fitness_partial_kernel<T, D, 8>), grid, dim3(256), 0, s, f);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(fitness_finalize_kernel<D>, dim3(f.B * kHeads), dim3(kFinThreads), 0, s, f);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_t(const FitnessArgs& f, hipStream_t s) {
    switch (f.D) {
        case 8: return launch_td<T, 8>(f, s);
        case 16: return launch_td<T, 16>(f, s);
        case 32: return launch_td<T, 32>(f, s);
        case 64: return launch_td<T, 64>(f, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

FitnessChunks fitness_chunks(int B, int G) {
    const long long units = (long long)G * G / kUnit;
    auto clamp = [&](long long v, long long lo, long long hi) { return v < lo ? lo : v > hi ? hi : v; };
    FitnessChunks c;
    // Gram: about four workgroups per CU, not more partials than the finalize reads in a few
    // microseconds. Moments: about eight per CU. Neither splits below 64 cells.
    c.gram = (int)std::min(units, clamp(1024 / (B * kHeads), 4, 32));
    c.mom = (int)std::min(units, clamp(2048 / B, 1, 512));
    return c;
}

hipError_t launch_fitness(int dtype, const FitnessArgs& f, hipStream_t s) {
    return dtype == 1 ? launch_t<bf16_t>(f, s) : launch_t<float>(f, s);
}

size_t fitness_partial_bytes(int B, int D, int T, FitnessChunks c) {
    return (size_t)B * kHeads * ((size_t)c.gram * D * D + (size_t)c.mom * 3 * T) * sizeof(double);
}

FitnessChunks fitness_static_chunks(int B, int G, int D, int T) {
    FitnessChunks c = fitness_chunks(B, G);
    while (fitness_partial_bytes(B, D, T, c) > kFitnessScratchBytes) {
        if (c.gram == 1 && c.mom == 1) return FitnessChunks{0, 0};
        c.gram = (c.gram + 1) / 2;
        c.mom = (c.mom + 1) / 2;
    }
    return c;
}

namespace {
// Per device: the scratch's device address, and the event and stream of the last
// call that launched outside graph capture.
struct StaticSlot {
    void* addr = nullptr;
    hipEvent_t done = nullptr;
    hipStream_t last = nullptr;
    bool recorded = false;
};
constexpr int kMaxDevices = 64;
std::mutex g_static_mu;
StaticSlot g_static[kMaxDevices];

hipError_t static_slot(StaticSlot** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    StaticSlot& s = g_static[dev];
    if (!s.addr) {
        hipDeviceProp_t prop;
        e = hipGetDeviceProperties(&prop, dev);
        if (e != hipSuccess) return e;
        if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) return hipErrorNoBinaryForGpu;
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (!p) return hipErrorInvalidSymbol;
        e = hipEventCreateWithFlags(&s.done, hipEventDisableTiming);
        if (e != hipSuccess) return e;
        s.addr = p;
    }
    *out = &s;
    return hipSuccess;
}
}  // namespace

hipError_t fitness_static_scratch(void** ptr) {
    std::lock_guard<std::mutex> lock(g_static_mu);
    StaticSlot* s = nullptr;
    const hipError_t e = static_slot(&s);
    if (e == hipSuccess) *ptr = s->addr;
    return e;
}

hipError_t launch_fitness_static(int dtype, FitnessArgs f, hipStream_t stream) {
    std::lock_guard<std::mutex> lock(g_static_mu);
    StaticSlot* s = nullptr;
    hipError_t e = static_slot(&s);
    if (e != hipSuccess) return e;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    e = hipStreamIsCapturing(stream, &cap);
    if (e != hipSuccess) return e;
    const bool ordered = cap == hipStreamCaptureStatusNone;
    // The previous call's kernels, if they ran on another stream, finish with the
    // scratch before this call's kernels write it.
    if (ordered && s->recorded && s->last != stream) {
        e = hipStreamWaitEvent(stream, s->done, 0);
        if (e != hipSuccess) return e;
    }
    f.gram_part = static_cast<double*>(s->addr);
    f.mom_part = f.gram_part + (size_t)f.B * kHeads * f.chunks * f.D * f.D;
    e = launch_fitness(dtype, f, stream);
    if (e != hipSuccess || !ordered) return e;
    e = hipEventRecord(s->done, stream);
    if (e == hipSuccess) {
        s->last = stream;
        s->recorded = true;
    }
    return e;
}

}  // namespace slime
