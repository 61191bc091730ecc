// mmq_tile.h -- the output tile of the prefill GEMM kernels (mmq.hip,
// gemm_q5k.hip): from the MFMA layout through LDS to y.
#pragma once
#include "kq_common.h"

namespace jllm_hip {

typedef float mt_f32x4 __attribute__((ext_vector_type(4)));
typedef float mt_f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t mt_u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t mt_u32x4 __attribute__((ext_vector_type(4)));
constexpr int MMQ_TILE_THREADS = 256;

// A GEMM workgroup's output tile through LDS, [token][128 rows] (rows padded so
// that both the token-wise writes and the row-wise reads spread over the
// banks), so that a token's rows leave as whole lines: the MFMA layout holds 4
// rows of a token per lane, and storing from it sent a 2- or 4-byte write per
// element, each to a line of its own -- the address unit and the L2's request
// rate were the bound of the kernels' end (us: Q4_K 9728 x 2560 at N = 1261
// 111.5 -> 92.6, at N = 33 21.3 -> 17.0; Q6_K 2560 x 9728 at N = 512 74.2 ->
// 61.1; Q5_K 9728 x 2560 at N = 300 49.5 -> 43.8; same bits).
template <bool F32>
constexpr int mmq_tile_bytes(int tokens) { return tokens * 132 * (F32 ? 4 : 2); }

// the 4 x 4 consecutive rows r0 + 8 m .. +3 of token tl held by a lane
template <bool F32>
__device__ __forceinline__ void mmq_put_tile(uint8_t* T, int tl, int r0, const mt_f32x16& acc) {
#pragma unroll
    for (int m = 0; m < 4; m++) {
        if (F32) {
            *(mt_f32x4*)((float*)T + tl * 132 + r0 + 8 * m) = mt_f32x4{acc[4 * m], acc[4 * m + 1], acc[4 * m + 2], acc[4 * m + 3]};
        } else {
            *(mt_u32x2*)((uint16_t*)T + tl * 132 + r0 + 8 * m) =
                mt_u32x2{(uint32_t)f32_to_f16_bits(acc[4 * m]) | ((uint32_t)f32_to_f16_bits(acc[4 * m + 1]) << 16),
                       (uint32_t)f32_to_f16_bits(acc[4 * m + 2]) | ((uint32_t)f32_to_f16_bits(acc[4 * m + 3]) << 16)};
        }
    }
}

// the tile's rows row0 .. row0 + 127 (< M) of tokens col0 .. (< N) to y [N][M]
// (fp32: to the partials of this range of K, blockIdx.y); 256 threads.  Where a
// 16-byte piece would not be aligned (M or y), consecutive lanes store
// consecutive elements.
template <bool F32>
__device__ __forceinline__ void mmq_store_tile(void* y, const uint8_t* T, int row0, int col0, int tokens, int M, int N) {
    constexpr int PR = F32 ? 4 : 8, NPR = 128 / PR;    // rows of a 16-byte piece, pieces per token
    const int64_t base = F32 ? (int64_t)blockIdx.y * N * M : 0;
    if (M % PR == 0 && ((uintptr_t)y & 15u) == 0) {
        for (int e = threadIdx.x; e < tokens * NPR; e += MMQ_TILE_THREADS) {
            const int tl = e / NPR, r = row0 + (e % NPR) * PR, tok = col0 + tl;
            if (tok >= N || r >= M) continue;
            const int64_t at = base + (int64_t)tok * M + r;
            if (F32) {
                *(mt_f32x4*)((float*)y + at) = *(const mt_f32x4*)((const float*)T + tl * 132 + (r - row0));
            } else {
                const uint16_t* t = (const uint16_t*)T + tl * 132 + (r - row0);
                const mt_u32x2 a = *(const mt_u32x2*)t, b = *(const mt_u32x2*)(t + 4);
                *(mt_u32x4*)((uint16_t*)y + at) = mt_u32x4{a.x, a.y, b.x, b.y};
            }
        }
        return;
    }
    const int r = threadIdx.x & 127;
    if (row0 + r >= M) return;
    for (int tl = threadIdx.x >> 7; tl < min(tokens, N - col0); tl += MMQ_TILE_THREADS / 128) {
        const int64_t at = base + (int64_t)(col0 + tl) * M + row0 + r;
        if (F32) ((float*)y)[at] = ((const float*)T)[tl * 132 + r];
        else     ((uint16_t*)y)[at] = ((const uint16_t*)T)[tl * 132 + r];
    }
}

}  // namespace jllm_hip
