// attention_prefill.hip -- causal attention of N query tokens over an INT8
// (or FP16) KV cache, gfx950.
//
// Token t (absolute position start + t) attends to keys [0, start + t] (the
// last `window` of them): flash_attention_prefill_batched_kernel,
// attention.cu:382-514.  Scores are (q . k) * ks[pos][kv_head] * scale,
// values v * vs[pos][kv_head]; an online softmax per (token, head).
#include <float.h>
#include "kq_common.h"
#include "attention.h"
#include "quant_chunk.h"
#include "attn_common.h"

namespace jllm_hip {

// One workgroup of AP_WAVES waves per (KV head, block of tq tokens).  Its columns
// are the (token, head) pairs of the block -- column c = token tok0 + c / G,
// head kvh * G + c % G -- in NG groups of 32, and every wave holds all of
// them; the waves deal the 32-key tiles among themselves, tile t to wave
// t % AP_WAVES, and their softmax states are combined in LDS in wave order.  The
// number of waves is the same in every form of the launch, so a token's result
// does not depend on how a prompt is cut into calls, bit for bit, as long as its
// window does not bind (where it does, the tiles start at the window start of the
// block's first token).  A value of V or a V scale that is not finite is the
// exception: masked keys enter the products with probability 0, so it reaches
// every token of its block, the earlier ones too.
//
// Everything a tile needs after its loads stays in a wave's registers.  Lane
// (li = lane & 31, lg = lane >> 5), MFMA elements v = 0..15 <-> index
// 8 (v / 4) + 4 lg + v % 4:
//   S^T = K.q^T     rows = keys, lane li = column li: the softmax runs along
//                   the lane's own 16 keys and one exchange with lane ^ 32,
//                   and corr / max / sum are one number per lane
//   P^T             the B operand of the second product is the lane's own 16
//                   probabilities (times vs), split into fp16 high and low
//                   parts (~22 bits) -- no trip through LDS
//   V^T             the A operand: the V rows turned by an identity MFMA
//                   (int8: v_mfma_i32_32x32x32_i8, exact), whose result layout
//                   delivers the keys in exactly the order P^T holds them
//   O^T += V^T.P^T  rows = d, lane li = column li: the rescale factor of a
//                   moved maximum is a lane constant
// The K rows of the wave's next tile are fetched as soon as Q.K^T has read the
// current ones, the V rows after P.V: one LDS buffer each.
// What bounds it: VALU issue.  With MFMAs in flight a SIMD issues one VALU
// operation per 5.3 clocks whatever its number of waves (exponentials 9.3:
// microbench/issue_rates.hip), and a 32-key x 64-column tile takes ~440 of them in
// the loop, ~2500 clocks against 1664 of MFMA; hence the one-operation conversions below, the scores
// formed relative to the reference (one fma), and two column groups per K / V
// conversion.  32 / 8 heads x 128, INT8 KV, 512 tokens: at start 0 17.1 -> 14.1
// us, at start 7680 167 -> 115 us (580 TFLOP/s of q.k and p.v products) against
// the form it replaces (P' through LDS, lane-per-row loads, exact maxima).
//
// A column's softmax reference is not its running maximum but a value at most
// AP_SLACK (in base 2) below it, so that the accumulators are rescaled only
// when the maximum has grown 2^6-fold since the last time, not whenever one of
// the 64 columns moves (64 fp32 multiplies per lane and group).  p <= 64, and
// p * vs must fit fp16: tiles with a larger vs than AP_VS_MAX (a V row beyond
// the fp16 range times 1/127) take the exact maximum.
constexpr float AP_SLACK = 6.0f, AP_VS_MAX = 1000.0f;
constexpr float LOG2E = 1.4426950408889634f;
constexpr int AP_WAVES = 8;

typedef __attribute__((address_space(3))) void ap_lds_void;

// x(r): row r of a tile with NP pieces a row keeps piece p at position p ^ x(r)
template <int NP>
__device__ __forceinline__ int ap_swz(int r) {
    return NP == 8 ? ((r ^ (r >> 3)) & 7) : NP == 16 ? (r & 15) : NP == 4 ? ((r >> 1) & 3) : 0;
}
// at most N of the wave's newest global loads are still in flight
template <int N>
__device__ __forceinline__ void ap_wait_vm() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
    __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void ap_wait_lds() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// 8 codes of two words -> 8 fp16 values: one SDWA conversion a code (signed
// byte in, half of a register out).  The closing s_nop covers the two wait
// states between a VALU write and the MFMA that reads it.
__device__ __forceinline__ h8 ap_i8x8_to_h8(uint32_t a, uint32_t b) {
    u32x4a r;
    asm("v_cvt_f16_i16_sdwa %0, sext(%4) dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:BYTE_0\n\t"
        "v_cvt_f16_i16_sdwa %1, sext(%4) dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:BYTE_2\n\t"
        "v_cvt_f16_i16_sdwa %2, sext(%5) dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:BYTE_0\n\t"
        "v_cvt_f16_i16_sdwa %3, sext(%5) dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:BYTE_2\n\t"
        "v_cvt_f16_i16_sdwa %0, sext(%4) dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:BYTE_1\n\t"
        "v_cvt_f16_i16_sdwa %1, sext(%4) dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:BYTE_3\n\t"
        "v_cvt_f16_i16_sdwa %2, sext(%5) dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:BYTE_1\n\t"
        "v_cvt_f16_i16_sdwa %3, sext(%5) dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:BYTE_3\n\t"
        "s_nop 1"
        : "=&v"(r.x), "=&v"(r.y), "=&v"(r.z), "=&v"(r.w)
        : "v"(a), "v"(b));
    return __builtin_bit_cast(h8, r);
}

// 8 int32 results of an MFMA (int8 values) -> 8 fp16 values.  The low halves
// are ordinary conversions, which the compiler holds until the MFMA is done;
// the high halves follow them (they need their registers), so the results they
// read are complete too.
__device__ __forceinline__ h8 ap_i32x8_to_h8(int c0, int c1, int c2, int c3, int c4, int c5, int c6, int c7) {
    u32x4a r = u32x4a{__builtin_bit_cast(uint16_t, (_Float16)(short)c0), __builtin_bit_cast(uint16_t, (_Float16)(short)c2),
                      __builtin_bit_cast(uint16_t, (_Float16)(short)c4), __builtin_bit_cast(uint16_t, (_Float16)(short)c6)};
    asm("v_cvt_f16_i16_sdwa %0, %4 dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:WORD_0\n\t"
        "v_cvt_f16_i16_sdwa %1, %5 dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:WORD_0\n\t"
        "v_cvt_f16_i16_sdwa %2, %6 dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:WORD_0\n\t"
        "v_cvt_f16_i16_sdwa %3, %7 dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:WORD_0\n\t"
        "s_nop 1"
        : "+v"(r.x), "+v"(r.y), "+v"(r.z), "+v"(r.w)
        : "v"(c1), "v"(c3), "v"(c5), "v"(c7));
    return __builtin_bit_cast(h8, r);
}

// the fp16 high parts h of (q0, q1) and the fp16 parts of what they leave:
// q - h is exact in fp32 (one mixed-precision fma reads the half in place)
__device__ __forceinline__ void ap_split(float q0, float q1, uint32_t& hi, uint32_t& lo) {
    typedef float f32x2a __attribute__((ext_vector_type(2)));
    hi = h2_bits(__builtin_convertvector((f32x2a{q0, q1}), half2_t));
    float l0, l1;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(l0) : "v"(hi), "v"(q0));
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(l1) : "v"(hi), "v"(q1));
    lo = h2_bits(__builtin_convertvector((f32x2a{l0, l1}), half2_t));
}

template <bool INT8, int HD, int NG>
__global__ __launch_bounds__(64 * AP_WAVES) __attribute__((amdgpu_waves_per_eu(2, 2)))
void attn_prefill_kernel(AttnArgs a) {
    constexpr int W = AP_WAVES;
    constexpr int EB = INT8 ? 1 : 2;
    constexpr int hd = HD, half = HD / 2;
    constexpr int NDT = HD / 32;                        // 32-wide d chunks
    constexpr int NST = half / 8;                       // Q.K^T MFMA steps
    constexpr int NP = HD * EB / 16;                    // 16-byte pieces of a K or V row
    constexpr int NI = NP / 2;                          // 1 KiB DMA instructions per tile of 32 rows
    constexpr int TILE_B = 32 * NP * 16;
    // q rows in LDS: 16-byte pieces of consecutive columns fall on distinct
    // bank groups (row stride an odd number of 16-byte pieces)
    constexpr int QLD = HD + 8;
    constexpr int OLD = HD + 4;                         // fp32 rows of the combination, the same way
    constexpr int Q_B = 32 * NG * QLD * 2, LOOP_B = Q_B + W * (2 * TILE_B + 256);
    constexpr int COMB_B = W * 32 * OLD * 4;
    constexpr int AREA_B = LOOP_B > COMB_B ? LOOP_B : COMB_B;
    __shared__ __attribute__((aligned(16))) uint8_t smem[AREA_B + (W * 2 + 1) * NG * 32 * 4];
    float (*sML)[NG][2][32] = (float (*)[NG][2][32])(smem + AREA_B);    // [wave]: m, l of its columns
    float (*sDen)[32] = (float (*)[32])(smem + AREA_B + W * 2 * NG * 32 * 4);

    const int t = (int)threadIdx.x;
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int l = t & 63, li = l & 31, lg = l >> 5;
    // the last token blocks (the most key tiles) are dispatched first
    const int kvh = blockIdx.x, tok0 = ((int)gridDim.z - 1 - (int)blockIdx.z) * a.tq;
    const int G = a.n_heads / a.n_kv;
    const int ntok = min(a.tq, a.tokens - tok0);
    const int GC = ntok * G;                            // live columns
    // this lane's columns: causal bound and window start
    int seq_c[NG], lo_c[NG];
#pragma unroll
    for (int g = 0; g < NG; g++) {
        const int c = 32 * g + li;
        seq_c[g] = a.seq + tok0 + (c < GC ? c / G : 0);
        lo_c[g] = a.window > 0 ? max(0, seq_c[g] - a.window) : 0;
    }
    // the key range covers every column's
    const int seq = a.seq + tok0 + ntok - 1;
    const int lo_pos = a.window > 0 ? max(0, a.seq + tok0 - a.window) : 0;
    const int kv_dim = a.n_kv * a.cache_head_dim, hoff = kvh * a.cache_head_dim;

    _Float16* sQ = (_Float16*)smem;                                 // [32 NG][QLD]
    uint8_t* sK = smem + Q_B + wv * (2 * TILE_B + 256);             // this wave's K rows | V rows
    uint8_t* sV = sK + TILE_B;
    float* sS = (float*)(sV + TILE_B);                              // ks[32] | vs[32]

    // The tile's rows go from global memory straight to the wave's LDS, NP
    // lanes per row (whole cache lines; a lane-per-row load into the operand
    // layout touches 32 lines per instruction and made the address unit the
    // bound).  Slot (row r, position p) holds piece p ^ x(r) (ap_swz), so that
    // the operand reads -- one piece of 8 consecutive rows -- hit distinct
    // banks.
    const int row_b = kv_dim * EB;
    auto load_rows = [&](const void* base, uint8_t* dst, int p0, int lane) {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            (void*)((const uint8_t*)base + (int64_t)p0 * row_b + hoff * EB), (short)0, 0x7FFFFFFF, 0x00020000);
        const int last = seq - 1 - p0;                              // rows past it repeat it
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int idx = 64 * i + lane, r = idx / NP, p = (idx % NP) ^ ap_swz<NP>(r);
            if (64 % NP == 0 && last >= 31) {
                // a whole tile: one lane offset (up to the swizzle), the row step in a scalar
                constexpr int RI = 64 / NP;
                const int r0 = lane / NP;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (ap_lds_void*)(dst + 1024 * i), 16, r0 * row_b + 16 * p,
                                                         RI * i * row_b, 0, 0);
            } else {
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (ap_lds_void*)(dst + 1024 * i), 16, min(r, last) * row_b + 16 * p,
                                                         0, 0, 0);
            }
        }
    };
    // byte offsets of this lane's operand pieces: K piece c of its half row,
    // V piece c + lg of its row (off_k / off_v of the two lane constants)
    constexpr bool SW = NP == 4 || NP == 8 || NP == 16;
    const int x16 = 16 * ap_swz<NP>(li);
    int kx = SW ? ((8 * NP * lg) ^ x16) : 8 * NP * lg, vx = SW ? ((16 * lg) ^ x16) : 16 * lg;
    auto off = [&](int x, int c) { return li * NP * 16 + (SW ? (x ^ (16 * c)) : x + 16 * c); };
    // one scale per lane: ks of key li (lg = 0), vs of key li (lg = 1); 1 where the
    // caller has none.  Such a lane loads as well (the first word of q, unused):
    // the waits below count the wave's loads, so every INT8 call issues exactly
    // one scale load per tile.
    const bool own_sc = (lg ? a.vs : a.ks) != nullptr;
    const float* sp = own_sc ? (lg ? a.vs : a.ks) + kvh : (const float*)a.q;
    const int sc_row = own_sc ? a.n_kv : 0;
    float scn = 1.0f;
    auto load_sc = [&](int p0) {
        if (INT8) scn = sp[(int64_t)min(p0 + li, seq - 1) * sc_row];
    };
    const int first = lo_pos + wv * AT_KEYS;
    constexpr int stride = W * AT_KEYS;
    if (first < seq) { load_rows(a.k, sK, first, l); load_sc(first); load_rows(a.v, sV, first, l); }

    // the columns' q rows, shared by the waves (zeros past the live columns)
    for (int e = t; e < 32 * NG * (HD / 8); e += 64 * W) {
        const int c = e / (HD / 8), d0 = (e % (HD / 8)) * 8;
        const int cc = c < GC ? c : 0;
        const u32x4a qv = *(const u32x4a*)(a.q + ((int64_t)(tok0 + cc / G) * a.n_heads + kvh * G + cc % G) * hd + d0);
        *(u32x4a*)&sQ[c * QLD + d0] = c < GC ? qv : u32x4a{0u, 0u, 0u, 0u};
    }

    i32x4 eye8;
    h8 eyeh[2];
    eye_operands(li, lg, eye8, eyeh);

    // softmax reference (base 2) and sum; none: 0 once the reference is set
    float run_m[NG], run_l[NG], none[NG];
    f32x16 acc[NG][NDT];
#pragma unroll
    for (int g = 0; g < NG; g++) {
        run_m[g] = 0.0f;
        none[g] = -FLT_MAX;
        run_l[g] = 0.0f;
#pragma unroll
        for (int i = 0; i < NDT; i++) acc[g][i] = f32x16{};
    }
    __syncthreads();

    int lane = l;
#pragma unroll 1
    for (int p0 = first; p0 < seq; p0 += stride) {
        const int n = min(AT_KEYS, seq - p0), pn = min(p0 + stride, seq - 1);
        // (opaque per tile: the addresses formed from these few lane constants
        // would otherwise be hoisted and spilled)
        asm volatile("" : "+v"(kx), "+v"(vx), "+v"(lane));
        const float scv = own_sc ? scn : 1.0f;
        // per-key scales through LDS to the lanes that hold a key's scores
        // (keys 8m + 4lg + [0,4))
        if (INT8) sS[32 * lg + li] = lg ? scv : scv * (a.scale * LOG2E);
        const uint32_t big_vs = INT8 ? (uint32_t)(__builtin_amdgcn_ballot_w64(lg && !(fabsf(scv) <= AP_VS_MAX)) >> 32) : 0u;
        // 1. transposed scores
        ap_wait_vm<NI>();                                // the K rows (the V rows may be in flight)
        // All K pieces first, the q pieces two steps ahead of their products,
        // the conversion of a step under the products of the one before.
        f32x16 sc[NG];
#pragma unroll
        for (int g = 0; g < NG; g++) sc[g] = f32x16{};
        u32x4a kr[NST * EB / 2];
        h8 qb[3][NG];
        auto read_q = [&](int st) {
#pragma unroll
            for (int g = 0; g < NG; g++) qb[st % 3][g] = *(const h8*)&sQ[(32 * g + li) * QLD + lg * half + 8 * st];
        };
#pragma unroll
        for (int c = 0; c < NST * EB / 2; c++) kr[c] = *(const u32x4a*)(sK + off(kx, c));
        read_q(0);
        if (NST > 1) read_q(1);
        __builtin_amdgcn_sched_barrier(0);
        auto conv_k = [&](int st) {
            const uint32_t* w = (const uint32_t*)&kr[0] + 2 * st * EB;
            return INT8 ? ap_i8x8_to_h8(w[0], w[1]) : __builtin_bit_cast(h8, kr[INT8 ? 0 : st]);
        };
        h8 kb = conv_k(0);
#pragma unroll
        for (int st = 0; st < NST; st++) {
            if (st + 2 < NST) read_q(st + 2);
#pragma unroll
            for (int g = 0; g < NG; g++) sc[g] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kb, qb[st % 3][g], sc[g], 0, 0, 0);
            if (st + 1 < NST) kb = conv_k(st + 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        ap_wait_lds();                                   // the K rows have been read
        load_rows(a.k, sK, pn, lane);
        load_sc(pn);
        // scores in base 2, relative to the column's reference so far
        float vscl[16];
        if (INT8) {
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int m4 = 0; m4 < 4; m4++) {
                const f32x4a k4 = *(const f32x4a*)&sS[8 * m4 + 4 * lg];
                const f32x4a v4 = *(const f32x4a*)&sS[32 + 8 * m4 + 4 * lg];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    vscl[4 * m4 + r] = v4[r];
#pragma unroll
                    for (int g = 0; g < NG; g++) sc[g][4 * m4 + r] = __builtin_fmaf(sc[g][4 * m4 + r], k4[r], -run_m[g]);
                }
            }
        } else {
#pragma unroll
            for (int g = 0; g < NG; g++)
#pragma unroll
                for (int v = 0; v < 16; v++) sc[g][v] = __builtin_fmaf(sc[g][v], a.scale * LOG2E, -run_m[g]);
        }
        // key masks only where a tile can hold dead keys (uniform branch): it
        // reaches past the first column's causal bound, below the last
        // column's window start, or has fewer than AT_KEYS keys
        const bool full = n == AT_KEYS && p0 + AT_KEYS <= a.seq + tok0 &&
                          (a.window <= 0 || p0 >= a.seq + tok0 + ntok - 1 - a.window);
        if (!full) {
#pragma unroll
            for (int g = 0; g < NG; g++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const int key = 8 * (v >> 2) + 4 * lg + (v & 3), pos = p0 + key;
                    sc[g][v] = key < n && pos < seq_c[g] && pos >= lo_c[g] ? sc[g][v] : -INFINITY;
                }
        }
        // 2. online softmax of the lane's column(s).  A column's reference moves
        // only when its maximum passes it by more than `slack`; its first live
        // key sets it.  (Keys past the column's causal bound have no say.)
        float slack[NG], up[NG];
#pragma unroll
        for (int g = 0; g < NG; g++) slack[g] = AP_SLACK;
        if (big_vs) {
#pragma unroll
            for (int g = 0; g < NG; g++)
                if (seq_c[g] > p0 && (big_vs << max(0, AT_KEYS - (seq_c[g] - p0))) != 0) slack[g] = 0.0f;
        }
        bool mv[NG], moved = false;
#pragma unroll
        for (int g = 0; g < NG; g++) {
            float mx = sc[g][0];
#pragma unroll
            for (int v = 1; v < 16; v++) mx = fmaxf(mx, sc[g][v]);
            float a0, a1;
            wave_halves(mx, a0, a1);
            mx = fmaxf(a0, a1);
            mv[g] = mx > none[g] + slack[g];
            up[g] = mv[g] ? mx : 0.0f;
            moved |= mv[g];
        }
        if (__builtin_amdgcn_ballot_w64(moved) != 0) {
#pragma unroll
            for (int g = 0; g < NG; g++) {
                const float corr = none[g] == 0.0f ? __builtin_amdgcn_exp2f(-up[g]) : 1.0f;
                run_m[g] += up[g];
                if (mv[g]) none[g] = 0.0f;
                run_l[g] *= corr;
#pragma unroll
                for (int v = 0; v < 16; v++) sc[g][v] -= up[g];
#pragma unroll
                for (int dt = 0; dt < NDT; dt++)
#pragma unroll
                    for (int v = 0; v < 16; v++) acc[g][dt][v] *= corr;
            }
        }
        // 3. P^T
        u32x4a phi[NG][2], plo[NG][2];
#pragma unroll
        for (int g = 0; g < NG; g++) {
            float ps = 0.0f;
#pragma unroll
            for (int v = 0; v < 16; v += 2) {
                const float p0v = __builtin_amdgcn_exp2f(sc[g][v]), p1v = __builtin_amdgcn_exp2f(sc[g][v + 1]);
                ps += p0v + p1v;
                uint32_t h, lo;
                ap_split(INT8 ? p0v * vscl[v] : p0v, INT8 ? p1v * vscl[v + 1] : p1v, h, lo);
                phi[g][v >> 3][(v & 7) / 2] = h;
                plo[g][v >> 3][(v & 7) / 2] = lo;
            }
            float a0, a1;
            wave_halves(ps, a0, a1);
            run_l[g] += a0 + a1;
        }
        ap_wait_vm<NI + (INT8 ? 1 : 0)>();               // the V rows (the next K rows may be in flight)
        // 4. O^T += V^T.P^T; V^T: the rows turned by the identity MFMA, a
        // 32-wide chunk ahead of the products that read it
        i32x16 ci = {};
        f32x16 cf = {};
        auto turn = [&](int dt) {
            if (INT8) {
                ci = __builtin_amdgcn_mfma_i32_32x32x32_i8(*(const i32x4*)(sV + off(vx, 2 * dt)), eye8, i32x16{}, 0, 0, 0);
            } else {
                cf = __builtin_amdgcn_mfma_f32_32x32x16_f16(*(const h8*)(sV + off(vx, 4 * dt)), eyeh[0], f32x16{}, 0, 0, 0);
                cf = __builtin_amdgcn_mfma_f32_32x32x16_f16(*(const h8*)(sV + off(vx, 4 * dt + 2)), eyeh[1], cf, 0, 0, 0);
            }
        };
        turn(0);
#pragma unroll
        for (int dt = 0; dt < NDT; dt++) {
            h8 vb[2];
#pragma unroll
            for (int st = 0; st < 2; st++) {                             // exact
                if (INT8) {
                    vb[st] = ap_i32x8_to_h8(ci[8 * st], ci[8 * st + 1], ci[8 * st + 2], ci[8 * st + 3], ci[8 * st + 4],
                                            ci[8 * st + 5], ci[8 * st + 6], ci[8 * st + 7]);
                } else {
#pragma unroll
                    for (int e = 0; e < 8; e++) vb[st][e] = (_Float16)cf[8 * st + e];
                }
            }
            if (dt + 1 < NDT) turn(dt + 1);
#pragma unroll
            for (int st = 0; st < 2; st++)
#pragma unroll
                for (int g = 0; g < NG; g++) {
                    acc[g][dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vb[st], __builtin_bit_cast(h8, phi[g][st]), acc[g][dt], 0, 0, 0);
                    acc[g][dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vb[st], __builtin_bit_cast(h8, plo[g][st]), acc[g][dt], 0, 0, 0);
                }
        }
        ap_wait_lds();                                   // the V rows have been read
        load_rows(a.v, sV, pn, lane);
    }
    ap_wait_vm<0>();                                     // the rows fetched past the last tile have landed

    // 5. the waves' states combined per column, waves in order:
    // out = sum_w acc_w 2^(m_w - M) / sum_w l_w 2^(m_w - M), M = max_w m_w
    if (lg == 0) {
#pragma unroll
        for (int g = 0; g < NG; g++) {
            sML[wv][g][0][li] = none[g] == 0.0f ? run_m[g] : -FLT_MAX;
            sML[wv][g][1][li] = run_l[g];
        }
    }
    __syncthreads();                                     // (every wave has read its last q rows, too)
    float* sO = (float*)smem;
    constexpr int nd8 = HD / 8;
    const bool vec = ((uintptr_t)a.out & 15u) == 0;
#pragma unroll
    for (int g = 0; g < NG; g++) {
        float M = sML[0][g][0][li];
#pragma unroll
        for (int u = 1; u < W; u++) M = fmaxf(M, sML[u][g][0][li]);
        const float f = __builtin_amdgcn_exp2f(sML[wv][g][0][li] - M);
        if (wv == 0 && lg == 0) {
            float den = 0.0f;
#pragma unroll
            for (int u = 0; u < W; u++) den += sML[u][g][1][li] * __builtin_amdgcn_exp2f(sML[u][g][0][li] - M);
            sDen[g][li] = den;
        }
#pragma unroll
        for (int dt = 0; dt < NDT; dt++)
#pragma unroll
            for (int m4 = 0; m4 < 4; m4++)
                *(f32x4a*)&sO[(wv * 32 + li) * OLD + 32 * dt + 8 * m4 + 4 * lg] =
                    f32x4a{acc[g][dt][4 * m4] * f, acc[g][dt][4 * m4 + 1] * f, acc[g][dt][4 * m4 + 2] * f, acc[g][dt][4 * m4 + 3] * f};
        __syncthreads();
        // each thread: 8 consecutive d of a column
        const int gc = min(32, GC - 32 * g);
        for (int e = t; e < gc * nd8; e += 64 * W) {
            const int cl = e / nd8, d0 = (e - cl * nd8) * 8, c = 32 * g + cl;
            f32x4a n0 = f32x4a{0.0f, 0.0f, 0.0f, 0.0f}, n1 = n0;
#pragma unroll
            for (int u = 0; u < W; u++) {
                const f32x4a h0 = *(const f32x4a*)&sO[(u * 32 + cl) * OLD + d0], h1 = *(const f32x4a*)&sO[(u * 32 + cl) * OLD + d0 + 4];
#pragma unroll
                for (int i = 0; i < 4; i++) { n0[i] += h0[i]; n1[i] += h1[i]; }
            }
            const float den = sDen[g][cl];
            uint32_t o[4];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                o[i] = (uint32_t)f32_to_f16_bits(den > 0.0f ? n0[2 * i] / den : 0.0f) |
                       ((uint32_t)f32_to_f16_bits(den > 0.0f ? n0[2 * i + 1] / den : 0.0f) << 16);
                o[2 + i] = (uint32_t)f32_to_f16_bits(den > 0.0f ? n1[2 * i] / den : 0.0f) |
                           ((uint32_t)f32_to_f16_bits(den > 0.0f ? n1[2 * i + 1] / den : 0.0f) << 16);
            }
            const int ct = c / G, ch = c - ct * G;
            uint16_t* ot = a.out + (int64_t)(tok0 + ct) * a.n_heads * hd + (int64_t)(kvh * G + ch) * hd + d0;
            if (vec) {
                *(u32x4a*)ot = u32x4a{o[0], o[1], o[2], o[3]};
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++) { ot[2 * i] = (uint16_t)(o[i] & 0xFFFFu); ot[2 * i + 1] = (uint16_t)(o[i] >> 16); }
            }
            if (a.qcodes) {
                // the 4 lanes of an aligned quad hold the 32 values of one
                // quantiser block (hd % 32 == 0, nd8 % 4 == 0)
                float v[8];
#pragma unroll
                for (int i = 0; i < 4; i++) { v[2 * i] = f16_bits_to_f32(o[i] & 0xFFFFu); v[2 * i + 1] = f16_bits_to_f32(o[i] >> 16); }
                const int kb32 = ((kvh * G + ch) * hd + d0) >> 5, sub = (d0 >> 3) & 3;
                if (a.q_i8) quant_chunk<true>(v, sub, kb32, tok0 + ct, a.q_npad, a.qcodes, a.qscl, true);
                else        quant_chunk<false>(v, sub, kb32, tok0 + ct, a.q_npad, a.qcodes, a.qscl, false);
            }
        }
        if (g + 1 < NG) __syncthreads();
    }
}

// Column groups of a workgroup, by the grid: one where 32-column blocks leave
// CUs idle, else two, with half the K / V conversions and reads per column (32 /
// 8 heads x 128, INT8 KV, us for 32 / 64 columns; N tokens at start: 33 at 0 6.2 /
// 9.4; 32 at 1000 13.0 / 19.7; 256 at 512 11.6 / 16.6; 300 at 724 21.7 / 19.7; 512
// at 0 14.8 / 14.1; 512 at 7680 142 / 115).  The same side is faster for FP16
// caches, head sizes 32 to 96, 1 to 16 heads on each of 1 to 32 KV heads and
// windows of 100 to 1500 keys (80 calls).
// Four waves of 32 columns, two workgroups on a CU, were faster below ~500 keys
// (512 at 0 11.6, at 256 15.5 against 17.2) and are not used: the bits would follow
// the form, and with it the cut of a prompt.  Four waves that form the eight
// states two each: 13.8 and 17.5.
template <bool INT8, int HD>
static void attn_prefill_go(AttnArgs& a, hipStream_t st) {
    const int tq1 = ATTN_MAX_COLUMNS / (a.n_heads / a.n_kv);
    const bool one = (int64_t)a.n_kv * ((a.tokens + tq1 - 1) / tq1) <= 256;
    a.tq = one ? tq1 : 2 * ATTN_MAX_COLUMNS / (a.n_heads / a.n_kv);
    const dim3 grid(a.n_kv, 1, (a.tokens + a.tq - 1) / a.tq);
    if (one) hipLaunchKernelGGL((attn_prefill_kernel<INT8, HD, 1>), grid, dim3(64 * AP_WAVES), 0, st, a);
    else     hipLaunchKernelGGL((attn_prefill_kernel<INT8, HD, 2>), grid, dim3(64 * AP_WAVES), 0, st, a);
}

hipError_t attn_prefill_launch(AttnArgs a, bool kv_int8, hipStream_t st) {
    if (a.tokens < 1 || a.n_kv < 1 || a.n_heads % a.n_kv) return hipErrorInvalidValue;
    const int G = a.n_heads / a.n_kv;
    if (G < 1 || G > ATTN_MAX_COLUMNS) return hipErrorInvalidValue;
    if (a.qcodes && (a.head_dim % 32 || !a.qscl || a.q_npad < a.tokens)) return hipErrorInvalidValue;
    switch (a.head_dim * 2 + (kv_int8 ? 1 : 0)) {
    case 64:  attn_prefill_go<false, 32>(a, st); break;
    case 65:  attn_prefill_go<true, 32>(a, st); break;
    case 128: attn_prefill_go<false, 64>(a, st); break;
    case 129: attn_prefill_go<true, 64>(a, st); break;
    case 192: attn_prefill_go<false, 96>(a, st); break;
    case 193: attn_prefill_go<true, 96>(a, st); break;
    case 256: attn_prefill_go<false, 128>(a, st); break;
    case 257: attn_prefill_go<true, 128>(a, st); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace jllm_hip
