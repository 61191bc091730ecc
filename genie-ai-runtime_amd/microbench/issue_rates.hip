// issue_rates.hip -- clocks that one wave instruction of each kind occupies a
// SIMD of gfx950 with, alone and next to matrix instructions: what the prefill
// attention's tile (about 8 VALU operations per MFMA) is bound by.
//
// 256 workgroups of 4 or 8 waves (1 or 2 per SIMD); each wave repeats ITER
// times 8 groups of 8 independent operations on registers, with or without one
// v_mfma_f32_32x32x16_f16 per group.  Reported: core clocks of a workgroup's
// slowest wave (the older wave of a SIMD is served first and ends early), mean
// over the workgroups, per operation and SIMD; with MFMAs their own issue is
// included.
//
// Build: hipcc --offload-arch=gfx950 -O3 -Xclang -target-feature -Xclang
//        -packed-fp32-ops -o issue_rates issue_rates.hip
// Run:   ./issue_rates
#include <hip/hip_runtime.h>
#include <cstdio>
#include <cstdint>

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));

constexpr int ITER = 512, GROUPS = 8, OPS = 8, BLOCKS = 256;

enum { ADD, AND, MAX, PERM, PK_F16, FMA, CVT, CVT_SDWA, MIX, EXP, DOT2, NONE };
static const char* const NAMES[] = {"v_add_f32", "v_and_b32", "v_max_f32", "v_perm_b32", "v_pk_add_f16", "v_fma_f32",
                                    "v_cvt_f16_f32", "v_cvt_f16_i16_sdwa", "v_fma_mix_f32", "v_exp_f32", "v_dot2_f32_f16",
                                    "(MFMA only)"};

template <int OP>
__device__ __forceinline__ void op(float& r, float c) {
    if (OP == ADD) asm volatile("v_add_f32 %0, %0, %1" : "+v"(r) : "v"(c));
    if (OP == AND) asm volatile("v_and_b32 %0, %0, %1" : "+v"(r) : "v"(c));
    if (OP == MAX) asm volatile("v_max_f32 %0, %0, %1" : "+v"(r) : "v"(c));
    if (OP == PERM) asm volatile("v_perm_b32 %0, %0, %1, %1" : "+v"(r) : "v"(c));
    if (OP == PK_F16) asm volatile("v_pk_add_f16 %0, %0, %1" : "+v"(r) : "v"(c));
    if (OP == FMA) asm volatile("v_fma_f32 %0, %0, %1, %1" : "+v"(r) : "v"(c));
    if (OP == CVT) asm volatile("v_cvt_f16_f32 %0, %0" : "+v"(r));
    if (OP == CVT_SDWA) asm volatile("v_cvt_f16_i16_sdwa %0, sext(%1) dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:BYTE_1" : "+v"(r) : "v"(c));
    if (OP == MIX) asm volatile("v_fma_mix_f32 %0, %1, -1.0, %0 op_sel_hi:[1,0,0]" : "+v"(r) : "v"(c));
    if (OP == EXP) asm volatile("v_exp_f32 %0, %0" : "+v"(r));
    if (OP == DOT2) asm volatile("v_dot2_f32_f16 %0, %1, %1, %0" : "+v"(r) : "v"(c));
}

template <int OP, bool MFMA>
__global__ __launch_bounds__(512) void rate_kernel(float* out, uint64_t* clk, float c) {
    float r[OPS];
    for (int i = 0; i < OPS; i++) r[i] = c * (float)(i + (int)threadIdx.x);
    h8 a, b;
    for (int i = 0; i < 8; i++) { a[i] = (_Float16)(float)threadIdx.x; b[i] = (_Float16)c; }
    f32x16 acc[2] = {f32x16{}, f32x16{}};
    __syncthreads();
    const uint64_t t0 = clock64();
#pragma unroll 1
    for (int it = 0; it < ITER; it++) {
#pragma unroll
        for (int g = 0; g < GROUPS; g++) {
            if (MFMA) acc[g & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, acc[g & 1], 0, 0, 0);
            if (OP != NONE) {
#pragma unroll
                for (int i = 0; i < OPS; i++) op<OP>(r[i], c);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    float s = 0.0f;
    for (int i = 0; i < 16; i++) s += acc[0][i] + acc[1][i];
    for (int i = 0; i < OPS; i++) s += r[i];
    const uint64_t t1 = clock64();
    const int w = (int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    if ((threadIdx.x & 63) == 0) clk[w] = t1 - t0;
    out[(size_t)blockIdx.x * blockDim.x + threadIdx.x] = s;
}

template <int OP, bool MFMA>
static double run(int wps, float* out, uint64_t* clk) {
    static uint64_t host[BLOCKS * 8];
    const int waves = 4 * wps;
    for (int i = 0; i < 2; i++) hipLaunchKernelGGL((rate_kernel<OP, MFMA>), dim3(BLOCKS), dim3(64 * waves), 0, 0, out, clk, 1.0f);
    if (hipMemcpy(host, clk, sizeof(uint64_t) * BLOCKS * waves, hipMemcpyDeviceToHost) != hipSuccess) return -1.0;
    double sum = 0;
    for (int b = 0; b < BLOCKS; b++) {
        uint64_t m = 0;
        for (int w = 0; w < waves; w++) m = host[b * waves + w] > m ? host[b * waves + w] : m;
        sum += (double)m;
    }
    return sum / BLOCKS / ((double)ITER * GROUPS * (OP == NONE ? 1 : OPS) * wps);
}

template <int OP>
static void row(float* out, uint64_t* clk) {
    if (OP == NONE) printf("| %s, clocks per MFMA | | | %.1f | %.1f |\n", NAMES[OP], run<OP, true>(1, out, clk), run<OP, true>(2, out, clk));
    else printf("| %s | %.1f | %.1f | %.1f | %.1f |\n", NAMES[OP], run<OP, false>(1, out, clk), run<OP, false>(2, out, clk),
                run<OP, true>(1, out, clk), run<OP, true>(2, out, clk));
    fflush(stdout);
}

int main() {
    float* out = nullptr;
    uint64_t* clk = nullptr;
    if (hipMalloc(&out, sizeof(float) * BLOCKS * 512) != hipSuccess || hipMalloc(&clk, sizeof(uint64_t) * BLOCKS * 8) != hipSuccess) return 1;
    printf("| operation | alone, 1 wave | alone, 2 waves | one MFMA per 8, 1 wave | one MFMA per 8, 2 waves |\n|---|---|---|---|---|\n");
    row<ADD>(out, clk);
    row<AND>(out, clk);
    row<MAX>(out, clk);
    row<PERM>(out, clk);
    row<PK_F16>(out, clk);
    row<FMA>(out, clk);
    row<CVT>(out, clk);
    row<CVT_SDWA>(out, clk);
    row<MIX>(out, clk);
    row<EXP>(out, clk);
    row<DOT2>(out, clk);
    row<NONE>(out, clk);
    (void)hipFree(out);
    (void)hipFree(clk);
    return 0;
}
