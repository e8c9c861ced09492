// organism.hip — the adapters around the CA step in the reference organism loop:
//   initialize_ca_from_field_kernel  X[y,x,c] = conc[y,x] * sin(0.1 c)
//                                    slime/core/organism.cu:691-720 (the else-branch
//                                    there is unreachable because NUM_HEADS*HEAD_DIM
//                                    == CHANNELS)
//   update_field_from_ca_kernel      conc[y,x] = mean_c X[y,x,c]
//                                    slime/core/organism.cu:723-743
// One wave per cell for the field update (a wave64 DPP sum over the channels).
// organism_report_kernel writes what neural_ca_update_kernel
// (slime/core/organism.cu:617-688) leaves behind per generation: the per-head mass
// buffer and one effective-rank entry of the history.
#include "common.hpp"
#include "kernels.hpp"

namespace slime {
namespace {

// Four consecutive channels per thread, whose sines it computes once for all its cells, and
// 16-byte (fp32) or 8-byte (bf16) stores: a workgroup writes 256 / (C / 4) whole cells at a
// time, kInitReps times (element by element where x is not aligned to that). Bound by the
// writes: 128^2 x 512 fp32 9.6 us, 17 us with a sine and a 4-byte store per thread.
constexpr int kInitReps = 8;

template <typename T>
__global__ __launch_bounds__(256) void init_from_field_kernel(const float* conc, T* X, long long cells, int C, bool vec) {
    const int quads = C / 4, step = 256 / quads;  // cells at a time (C <= 512)
    const int c0 = threadIdx.x % quads * 4, lane_cell = threadIdx.x / quads;
    float w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = sinf((float)(c0 + e) * 0.1f);
    const long long cell0 = (long long)blockIdx.x * step * kInitReps + lane_cell;
#pragma unroll
    for (int r = 0; r < kInitReps; ++r) {
        const long long cell = cell0 + r * step;
        if (cell >= cells) return;
        const float v = conc[cell];
        T* x = X + cell * C + c0;
        if (!vec) {
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = Store<T>::from_f32(v * w[e]);
        } else if constexpr (sizeof(T) == 2)
            *reinterpret_cast<uint2*>(x) = make_uint2(pack_bf16x2(v * w[0], v * w[1]), pack_bf16x2(v * w[2], v * w[3]));
        else
            *reinterpret_cast<float4*>(x) = make_float4(v * w[0], v * w[1], v * w[2], v * w[3]);
    }
}

template <typename T>
__global__ __launch_bounds__(256) void field_from_state_kernel(const T* X, float* conc, int G, int C) {
    const long long cell = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const bool valid = cell < (long long)G * G;
    float s = 0.f;
    if (valid)
        for (int c = lane; c < C; c += 64) s += Store<T>::to_f32(X[cell * C + c]);
    s = wave_sum(s);
    if (valid && lane == 0) conc[cell] = s / (float)C;
}

// After one organism generation: mass_buffer[h] = conserved mass of head h (may be
// null) and *erank_out = mean over heads of the effective rank, added in head order.
__global__ __launch_bounds__(64) void organism_report_kernel(const double* mass_out,
                                                             const float* erank, int H,
                                                             float* mass_buffer,
                                                             float* erank_out) {
    const int h = threadIdx.x;
    if (mass_buffer && h < H) mass_buffer[h] = (float)mass_out[h];
    if (h == 0) {
        float s = 0.f;
        for (int i = 0; i < H; ++i) s += erank[i];
        *erank_out = s / (float)H;
    }
}

}  // namespace

hipError_t launch_organism_report(const double* mass_out, const float* erank, int H,
                                  float* mass_buffer, float* erank_out, hipStream_t s) {
    hipLaunchKernelGGL(organism_report_kernel, dim3(1), dim3(64), 0, s, mass_out, erank, H,
                       mass_buffer, erank_out);
    return hipGetLastError();
}

hipError_t launch_init_from_field(int dtype, const float* conc, void* X, int G, int C, hipStream_t s) {
    const long long cells = (long long)G * G, per_wg = 256 / (C / 4) * kInitReps;
    const dim3 grid((unsigned)((cells + per_wg - 1) / per_wg));
    const bool vec = reinterpret_cast<uintptr_t>(X) % (dtype == 1 ? 8 : 16) == 0;
    if (dtype == 1)
        hipLaunchKernelGGL(init_from_field_kernel<bf16_t>, grid, dim3(256), 0, s, conc,
                           static_cast<bf16_t*>(X), cells, C, vec);
    else
        hipLaunchKernelGGL(init_from_field_kernel<float>, grid, dim3(256), 0, s, conc,
                           static_cast<float*>(X), cells, C, vec);
    return hipGetLastError();
}

hipError_t launch_field_from_state(int dtype, const void* X, float* conc, int G, int C, hipStream_t s) {
    const dim3 grid((unsigned)(((long long)G * G + 3) / 4));
    if (dtype == 1)
        hipLaunchKernelGGL(field_from_state_kernel<bf16_t>, grid, dim3(256), 0, s,
                           static_cast<const bf16_t*>(X), conc, G, C);
    else
        hipLaunchKernelGGL(field_from_state_kernel<float>, grid, dim3(256), 0, s,
                           static_cast<const float*>(X), conc, G, C);
    return hipGetLastError();
}

}  // namespace slime
