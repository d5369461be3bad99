// MFMA rate on constant and on random operands, the instruction mix of the prefill GEMM's main loop (csrc/mgemm.hip) with
// no copies, LDS reads or barriers: per 32x32 result four dependent v_mfma_f32_32x32x16_f16 and 16 scale FMAs, two
// results in flight, the FMAs of one behind the MFMAs of the next.  Output: mfma_rate_probe.md.
//   hipcc -O3 --offload-arch=gfx950 -Xclang -target-feature -Xclang -packed-fp32-ops mfma_rate_probe.hip -o probe && ./probe
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <vector>

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int kBlocks = 256, kThreads = 512, kFrags = 12;

__global__ __launch_bounds__(kThreads) void rate_kernel(const half8_t* in, float* out, int iters) {
    const int tid = blockIdx.x * kThreads + threadIdx.x;
    half8_t x[2][4], w[2][2];
    for (int i = 0; i < 8; ++i) x[i / 4][i % 4] = in[(size_t)i * kBlocks * kThreads + tid];
    for (int i = 0; i < 4; ++i) w[i / 2][i % 2] = in[(size_t)(8 + i) * kBlocks * kThreads + tid];
    f32x16_t acc[2] = {}, d[2] = {};
    const float sc = (float)x[0][0][0] * 1e-6f;
    for (int it = 0; it < iters; ++it) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            f32x16_t v = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[t][0], w[t][0], f32x16_t{}, 0, 0, 0);
            v = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[t][2], w[t][1], v, 0, 0, 0);
            v = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[t][1], w[t][0], v, 0, 0, 0);
            d[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[t][3], w[t][1], v, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[t ^ 1][i] = fmaf(sc, d[t ^ 1][i], acc[t ^ 1][i]);
            asm volatile("" : "+v"(acc[t ^ 1]), "+v"(x[t][0]), "+v"(w[t][0]));  // (each iteration's products are its own)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    float s = 0.0f;
    for (int i = 0; i < 16; ++i) s += acc[0][i] + acc[1][i] + d[0][i] + d[1][i];
    out[tid] = s;
}

#define CHECK(e) do { if ((e) != hipSuccess) { fprintf(stderr, "%s failed\n", #e); return 1; } } while (0)

int main() {
    const size_t n = (size_t)kFrags * kBlocks * kThreads;
    half8_t* in;
    float* out;
    CHECK(hipMalloc((void**)&in, n * sizeof(half8_t)));
    CHECK(hipMalloc((void**)&out, (size_t)kBlocks * kThreads * sizeof(float)));
    hipEvent_t e0, e1;
    CHECK(hipEventCreate(&e0));
    CHECK(hipEventCreate(&e1));
    std::vector<_Float16> h(n * 8);
    const int iters = 4000;
    for (int random = 0; random < 2; ++random) {
        srand(1);
        // fragments x[t][0..3]: hi, lo, hi, lo of a token row under its power of two; then w: quants
        for (size_t i = 0; i < h.size(); ++i) {
            const size_t f = i / 8 / ((size_t)kBlocks * kThreads);
            const float u = (rand() % 20001 - 10000) / 10000.0f;
            h[i] = !random ? (_Float16)1.0f : f >= 8 ? (_Float16)(float)(int)(127 * u) : (_Float16)(f % 2 ? 8 * u : 20000 * u);
        }
        CHECK(hipMemcpy(in, h.data(), n * sizeof(half8_t), hipMemcpyHostToDevice));
        float best = 1e30f, ms = 0.0f;
        for (int rep = 0; rep < 6; ++rep) {
            CHECK(hipEventRecord(e0, nullptr));
            hipLaunchKernelGGL(rate_kernel, dim3(kBlocks), dim3(kThreads), 0, nullptr, in, out, iters);
            CHECK(hipEventRecord(e1, nullptr));
            CHECK(hipEventSynchronize(e1));
            CHECK(hipEventElapsedTime(&ms, e0, e1));
            if (ms < best) best = ms;
        }
        const double flop = 2.0 * 32 * 32 * 16 * 8 * iters * (kBlocks * (kThreads / 64));
        printf("%s operands: %.3f ms, %.0f TFLOP/s\n", random ? "random" : "constant", best, flop / best * 1e-9);
        fflush(stdout);
    }
    return 0;
}
