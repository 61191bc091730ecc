// attn_common.h -- device helpers shared by the decode and prefill attention
// kernels (attention.hip, attention_prefill.hip).
#pragma once
#include "kq_common.h"

namespace jllm_hip {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4a __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2a __attribute__((ext_vector_type(2)));
typedef float f32x4a __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));

constexpr int AT_KEYS = 32;          // keys per tile (one MFMA column block)

// 4 signed int8 (one word) -> 4 exact fp16 values (two words): with u = b ^ 0x80
// in [1, 255], the half with bits 0x64 : u is 1024 + u (byte permutes against
// a word of 0x64 bytes), minus 1152 gives b.
__device__ __forceinline__ u32x2a i8x4_to_h4(uint32_t w) {
    const half2_t bias = {(_Float16)-1152.0f, (_Float16)-1152.0f};
    const uint32_t u = w ^ 0x80808080u;
    const uint32_t a = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u);
    const uint32_t b = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);
    return u32x2a{h2_bits(as_h2(a) + bias), h2_bits(as_h2(b) + bias)};
}

template <bool INT8>
__device__ __forceinline__ h8 kv8_to_h8(const uint8_t* p) {
    if (INT8) {
        const u32x2a w = *(const u32x2a*)p;
        const u32x2a lo = i8x4_to_h4(w.x), hi = i8x4_to_h4(w.y);
        return __builtin_bit_cast(h8, u32x4a{lo.x, lo.y, hi.x, hi.y});
    } else {
        return __builtin_bit_cast(h8, *(const u32x4a*)p);
    }
}

// identity operands of the V transpose.  int8: lane (col li, lg) holds
// B[16lg + i][li] = (16lg + i == li).  fp16: two K = 16 halves, lane
// (col li, lg) holds B_hh[8lg + e][li] = (16hh + 8lg + e == li).
__device__ __forceinline__ void eye_operands(int li, int lg, i32x4& eye8, h8 (&eyeh)[2]) {
    uint32_t w[4] = {0u, 0u, 0u, 0u};
    const int pos = li - 16 * lg;
    if (pos >= 0 && pos < 16) w[pos >> 2] = 1u << (8 * (pos & 3));
    eye8 = i32x4{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
#pragma unroll
    for (int hh = 0; hh < 2; hh++)
#pragma unroll
        for (int e = 0; e < 8; e++) eyeh[hh][e] = (_Float16)((16 * hh + 8 * lg + e == li) ? 1.0f : 0.0f);
}

}  // namespace jllm_hip
