// rq_dequant.h -- packed codes to bf16 weights, ŵ = bf16(scale * code + bias),
// shared by the GEMMs.
#pragma once

#include "rq_common.h"

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

namespace {

// One run of 32 codes -> 16 dwords of bf16 pairs, ŵ = bf16(scale*code + bias).
template <int BITS>
RQ_DEV void dequant_run_bf16(const uint32_t* words, float s, float b, uint32_t* out) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const float lo = fmaf(s, (float)run_code<BITS>(words, 2 * i), b);
        const float hi = fmaf(s, (float)run_code<BITS>(words, 2 * i + 1), b);
        out[i] = pack_bf16x2(lo, hi);
    }
}

// Eight 4-bit codes of one word -> 4 dwords of bf16 pairs (codes 0,1 .. 6,7),
// ŵ = bf16(s*code + b).  gfx950's v_cvt_scalef32_pk_f32_fp8 turns two bytes
// into two fp32 values in one instruction: an e4m3 byte 0x0q is exactly
// q / 512 (its subnormals and first binade are evenly spaced, 2^-9 apart),
// and the conversion applies only the exponent of its scale (measured on
// the box), so a scale of 512 gives q exactly.  Per 8 codes: 3 mask ops, 4
// converts, 8 fmas, 4 packs (byte converts took 8 converts).
RQ_DEV void dequant_word4(uint32_t word, float s, float b, uint32_t* out) {
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
    const uint32_t lo = word & 0x0F0F0F0Fu;         // codes 0,2,4,6
    const uint32_t hi = (word >> 4) & 0x0F0F0F0Fu;  // codes 1,3,5,7
    const f32x2_t l0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(lo, 512.f, false);
    const f32x2_t l1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(lo, 512.f, true);
    const f32x2_t h0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(hi, 512.f, false);
    const f32x2_t h1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(hi, 512.f, true);
    out[0] = pack_bf16x2(fmaf(s, l0[0], b), fmaf(s, h0[0], b));
    out[1] = pack_bf16x2(fmaf(s, l0[1], b), fmaf(s, h0[1], b));
    out[2] = pack_bf16x2(fmaf(s, l1[0], b), fmaf(s, h1[0], b));
    out[3] = pack_bf16x2(fmaf(s, l1[1], b), fmaf(s, h1[1], b));
}

// One run of 32 codes -> 16 dwords of bf16 pairs, ŵ = bf16(scale*code + bias):
// 4-bit codes by dequant_word4, 8-bit ones by byte converts
// (v_cvt_f32_ubyte0..3; the bytes are hidden from the optimiser by an empty
// asm, otherwise it folds each byte select into a bit-field extract, a second
// VALU op per code in front of a v_cvt_f32_ubyte0).
template <int BITS>
RQ_DEV void dequant_run_fast(const uint32_t* words, float s, float b, uint32_t* out) {
    if constexpr (BITS == 4) {
#pragma unroll
        for (int w = 0; w < 4; ++w) dequant_word4(words[w], s, b, out + 4 * w);
    } else if constexpr (BITS == 8) {
#pragma unroll
        for (int w = 0; w < 8; ++w) {
            uint32_t v = words[w];
            asm("" : "+v"(v));
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const float c0 = (float)(uint8_t)(v >> (16 * i));
                const float c1 = (float)(uint8_t)(v >> (16 * i + 8));
                out[2 * w + i] = pack_bf16x2(fmaf(s, c0, b), fmaf(s, c1, b));
            }
        }
    } else {
        dequant_run_bf16<BITS>(words, s, b, out);
    }
}

// 16 codes (half a run) of an even bit width, BITS / 2 words -> 8 dwords of
// bf16 pairs.
template <int BITS>
RQ_DEV void dequant_half_run(const uint32_t* words, float s, float b, uint32_t* out) {
    static_assert(BITS % 2 == 0, "half a run is whole words at even widths");
    if constexpr (BITS == 4) {
        dequant_word4(words[0], s, b, out);
        dequant_word4(words[1], s, b, out + 4);
    } else if constexpr (BITS == 8) {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            uint32_t v = words[w];
            asm("" : "+v"(v));
#pragma unroll
            for (int i = 0; i < 2; ++i)
                out[2 * w + i] = pack_bf16x2(fmaf(s, (float)(uint8_t)(v >> (16 * i)), b),
                                             fmaf(s, (float)(uint8_t)(v >> (16 * i + 8)), b));
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            out[i] = pack_bf16x2(fmaf(s, (float)run_code<BITS>(words, 2 * i), b),
                                 fmaf(s, (float)run_code<BITS>(words, 2 * i + 1), b));
    }
}

// Two outputs of dtype dt (bf16 or f16) packed in one dword, RNE.
RQ_DEV uint32_t pack2_dt(int dt, float lo, float hi) {
    return dt == RQ_BF16 ? pack_bf16x2(lo, hi) : (f32_to_f16_bits(lo) | (f32_to_f16_bits(hi) << 16));
}

}  // namespace
