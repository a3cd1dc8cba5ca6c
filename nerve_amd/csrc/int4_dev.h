// Shared pieces of the INT4 linears: code expansion, scale decoding, the
// kernel arguments and the finalizing store.
#pragma once

#include "common.h"

namespace nh {

struct Int4Args {
    const uint16_t* x;
    const uint32_t* qw;
    const uint16_t* scales;
    const uint32_t* qzeros;   // gptq only, may be null (zero = 8)
    const uint16_t* aux;      // bias [N] or residual [B, N]
    uint16_t* y;
    uint32_t B, K, N, G;
    int scale_bf16, finalize;
};

struct PpArgs {
    const uint32_t* q;          // int8 words [B, K/4], pair-packed
    const float* s;             // [B, K/32]
    const int32_t* sums;        // [B, K/32]
    Int4Args L;                 // qweight, scales, aux, y, shapes
};

}  // namespace nh

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

namespace {

using nh::Int4Args;
using nh::PpArgs;

__device__ __forceinline__ v4f mfma_bf16(v4i a, v4i b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
}

// 8 codes of one word (low nibble first along k) as bf16 (128 + q) pairs in
// k order (0,4),(1,5),(2,6),(3,7).
__device__ __forceinline__ v4i dequant_word(uint32_t w) {
    return v4i{(int)((w & 0x000F000Fu) | 0x43004300u), (int)(((w >> 4) & 0x000F000Fu) | 0x43004300u),
               (int)(((w >> 8) & 0x000F000Fu) | 0x43004300u), (int)(((w >> 12) & 0x000F000Fu) | 0x43004300u)};
}

// The same with the exponent bits in a vector register (pair_exponent()): mask
// and exponent are then one v_and_or_b32 (an instruction takes no literal there
// and one scalar operand at most), 7 instructions a word instead of 11.
__device__ __forceinline__ uint32_t pair_exponent() {
    uint32_t e;
    asm("v_mov_b32 %0, 0x43004300" : "=v"(e));
    return e;
}
__device__ __forceinline__ v4i dequant_word(uint32_t w, uint32_t e) {
    return v4i{(int)((w & 0x000F000Fu) | e), (int)(((w >> 4) & 0x000F000Fu) | e),
               (int)(((w >> 8) & 0x000F000Fu) | e), (int)(((w >> 12) & 0x000F000Fu) | e)};
}

// 8 contiguous bf16 activations reordered to the same (0,4),(1,5),(2,6),(3,7) order.
__device__ __forceinline__ v4i permute_act(v4i a) {
    uint32_t d0 = (uint32_t)a.x, d1 = (uint32_t)a.y, d2 = (uint32_t)a.z, d3 = (uint32_t)a.w;
    return v4i{(int)((d0 & 0xFFFFu) | (d2 << 16)), (int)((d0 >> 16) | (d2 & 0xFFFF0000u)),
               (int)((d1 & 0xFFFFu) | (d3 << 16)), (int)((d1 >> 16) | (d3 & 0xFFFF0000u))};
}

__device__ __forceinline__ float decode_scale(uint16_t v, bool bf16) {
    if (bf16) return bf16_to_f32(v);
    return (float)__builtin_bit_cast(_Float16, v);
}

__device__ __forceinline__ float load_scale(const uint16_t* p, bool bf16) { return decode_scale(*p, bf16); }

constexpr uint32_t ONES_BF16 = 0x3F803F80u;

// The matrix-core forms for INT8 rows add a segment's dots times their activation
// scales before the weight scale comes in.  A block's dot reaches 32 * 127 * 8 and
// a segment has up to four blocks, so with bf16 rows near the type's limit (scales
// up to 2^121) that sum passes the largest f32 although the result, fma(dot,
// s_x s_w, sum) in the shader, does not.  The activation scales are therefore
// taken 2^-11 times (130048 * 2^121 * 2^-11 < 2^128) and the sum 2^11 times at the
// end.  Both are exact for activation scales from 2^-115 on (rows whose block
// maximum is 2^-108 or more), and such results keep every bit; a smaller scale is
// rounded to a multiple of 2^-138, where the shader rounds s_x s_w to one of 2^-149.
// 48 rows of a 4096 / 14336 feed-forward 73.0 -> 74.6 us; up to 16 rows no change.
constexpr float I8_SCALE_DOWN = 0x1p-11f, I8_SCALE_UP = 0x1p11f;

__device__ __forceinline__ void finalize_store(const Int4Args& A, uint32_t t, uint32_t n, float sum) {
    // nerve/model_package_shader_selection.py:2504-2533
    float v = sum;
    if (A.finalize == 1) v = bf16_to_f32(A.aux[n]) + sum;
    else if (A.finalize == 2) v = bf16_to_f32(A.aux[(uint64_t)t * A.N + n]) + round_bf16(sum);
    A.y[(uint64_t)t * A.N + n] = (uint16_t)f32_to_bf16(v);
}

// J consecutive packed words of one qweight row (J = 1, 2 or 4).
template <int J>
__device__ __forceinline__ void load_words(const uint32_t* p, uint32_t (&w)[J]) {
    if constexpr (J == 4) {
        v4i v = *reinterpret_cast<const v4i*>(p);
        w[0] = (uint32_t)v.x; w[1] = (uint32_t)v.y; w[2] = (uint32_t)v.z; w[3] = (uint32_t)v.w;
    } else if constexpr (J == 2) {
        v2i v = *reinterpret_cast<const v2i*>(p);
        w[0] = (uint32_t)v.x; w[1] = (uint32_t)v.y;
    } else {
        w[0] = *p;
    }
}

typedef __bf16 v2bf __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float dot2_bf16(uint32_t a, uint32_t b, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2bf, a), __builtin_bit_cast(v2bf, b), c, false);
}

}  // namespace

namespace nh {

// Tiled split-K form, mostly for more than 16 rows (int4_gemm.hip): launches and
// returns true when the shape and alignment allow its loads, else false.
// `i8` is null for bf16 activations.
bool int4_gemm(const nerve_hip_ctx* ctx, const Int4Args& A, const PpArgs* i8, bool paired, bool ct, hipStream_t st);

// Adds the partial sums f32 [splits][B][N] in split order, finalizes and stores.
void int4_split_sum(const Int4Args& A, const float* part, uint32_t splits, hipStream_t st);

}  // namespace nh
