// rq_mid.hip -- GEMMs on group-affine packed weights for batches of activation
// rows that give the large-tile GEMMs (rq_qmm.hip) too few tiles to fill the
// chip: short prompts, batched decode beyond the GEMV, short QLoRA batches.
//
//   qmm_t_mid : y[m, r] = sum_k x[m, k] * ŵ[r, k]     (transpose=True)
//   qmm_n_mid : y[m, k] = sum_r x[m, r] * ŵ[r, k]     (transpose=False, dX = dY·W)
//
// (mx.quantized_matmul, rwkv_metal/lora/rwkvq_native.py:120-122, QuantizedLinear
// inside LoRALinear, rwkv_metal/lora/lora.py:58-59, and its VJP w.r.t. x,
// rwkv_metal/lora/finetune.py:141.)
//
// Such a product moves a few MB and does well under a microsecond of matrix
// work, so its time is memory round trips and the length of the longest serial
// chain.  A block is one tile of 16*TM activation rows x 16*TN weight rows; its
// waves (up to 16) each take a contiguous slice of the contraction, so that a
// wave walks one to a few 128-element spans however long K is, and add their
// fp32 tiles through LDS at the end, in wave order (deterministic).  Nothing is
// shared before that: no barrier precedes the MFMAs.
//  * A span is 128 codes of the 16 rows of an MFMA tile.  Lane L loads run L/16
//    (32 codes, whole words at every bit width) of row L%16; lane groups 0 and
//    1 load the span's scales and biases of row L%16 in one load and swaps hand
//    them to all four.  The MFMAs contract k = 64 h + 16 (L/16) + 8 j .. +7 (half
//    h, j = 0, 1): the packed words are spread over the lane groups with
//    v_permlane16_swap / v_permlane32_swap (two swaps per pair of words) and
//    dequantized there (ŵ = bf16(fma(scale, code, bias)), as the large GEMMs).
//  * Activations go through a wave-private LDS tile, half a span at a time.  A
//    load instruction whose neighbouring lanes read different rows costs one
//    address cycle per lane; eight lanes per 128-byte line cost a quarter of
//    it.  (Activations loaded straight in the MFMA operand's layout: [2048,
//    2048] at M = 77 9.4 us against 7.2, [16384, 4096] 56 against 40.)
//  * The weight fragment is the MFMA's A operand, so a lane ends with four
//    consecutive outputs of one activation row.
#include "rq_common.h"
#include "rq_dequant.h"
#include "rq_launch.h"
#include "rq_mid.h"

#ifndef RQ_BITS
#error "compile rq_mid.hip once per bit width with -DRQ_BITS=<bits>"
#endif

namespace {

typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef const __attribute__((address_space(1))) u32x4_t* gvec_t;
typedef const __attribute__((address_space(1))) uint32_t* gword_t;
typedef const __attribute__((address_space(1))) uint16_t* ghalf_t;
typedef const __attribute__((address_space(1))) uint8_t* gbyte_t;
// loads of less than their natural alignment
typedef uint32_t u32_a2_t __attribute__((aligned(2)));
typedef uint32_t u32x2_a2_t __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t u32x2_a4_t __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t u32x4_a4_t __attribute__((ext_vector_type(4), aligned(4)));
typedef const __attribute__((address_space(1))) u32_a2_t* gword_a2_t;
typedef const __attribute__((address_space(1))) u32x2_a2_t* gvec2_a2_t;
typedef const __attribute__((address_space(1))) u32x2_a4_t* gvec2_a4_t;
typedef const __attribute__((address_space(1))) u32x4_a4_t* gvec_a4_t;
typedef uint32_t u32x4_a2_t __attribute__((ext_vector_type(4), aligned(2)));
typedef const __attribute__((address_space(1))) u32x4_a2_t* gvec_a2_t;

struct MidArgs {
    const uint8_t* x;
    const uint32_t* wq;
    const void* scales;
    const void* biases;
    void* y;
    int64_t M, R, K;
    int gs_shift, sb_f16, x_f16, y_dt, y_vec;
    int tiles_m, tiles_n;
    int spw;  // spans per wave
    rq::LoraArgs lora;
};

// LDS bytes per wave
__host__ __device__ constexpr int mid_wave_bytes(int tm, int tn) {
    return (tn > 2 ? tm * tn : 2 * tm) * 1024;
}

// Swap of the odd lane groups of a with the even ones of b, then of lane
// groups 2, 3 of a with 0, 1 of b.  With a, b the lower and upper half of each
// lane group's piece list (group g: pieces 2g, 2g + 1), a ends with piece g and
// b with piece 4 + g.
RQ_DEV void spread_pieces(uint32_t& a, uint32_t& b) {
    const auto r0 = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    const auto r1 = __builtin_amdgcn_permlane32_swap(r0[0], r0[1], false, false);
    a = r1[0];
    b = r1[1];
}

// One 16-row weight tile's span: the lane's run of codes, and in lane groups
// 0 / 1 the raw scales / biases of the span's groups of row lr.
template <int BITS, bool SB32>
struct SpanRegs {
    static constexpr int NW = SB32 ? 4 : 2;  // words of one array: up to four groups
    uint32_t w[BITS];
    uint32_t sb[NW];

    RQ_DEV void load_codes(const uint8_t* wq, uint32_t off) {
        const gbyte_t p = (gbyte_t)wq + off;
        if constexpr (BITS == 4 || BITS == 8) {
#pragma unroll
            for (int i = 0; i < BITS / 4; ++i) {
                const u32x4_t v = ((gvec_t)p)[i];
#pragma unroll
                for (int e = 0; e < 4; ++e) w[4 * i + e] = v[e];
            }
        } else {
#pragma unroll
            for (int i = 0; i < BITS; ++i) w[i] = ((gword_t)p)[i];
        }
    }
    // ng: groups of this span in the row; 4 >> gsh unless the row ends in it.
    // One load of all of them (rows of an odd number of groups are 2-byte
    // aligned), element by element where the row ends.
    RQ_DEV void load_sb(gbyte_t p, int gsh, int ng) {
        if (ng == (4 >> gsh)) {
            if constexpr (SB32) {
                if (gsh == 0) {
                    const u32x4_t v = *(gvec_a4_t)p;
#pragma unroll
                    for (int e = 0; e < 4; ++e) sb[e] = v[e];
                } else if (gsh == 1) {
                    const u32x2_t v = *(gvec2_a4_t)p;
                    sb[0] = v[0];
                    sb[1] = v[1];
                } else {
                    sb[0] = *(gword_t)p;
                }
            } else {
                if (gsh == 0) {
                    const u32x2_t v = *(gvec2_a2_t)p;
                    sb[0] = v[0];
                    sb[1] = v[1];
                } else if (gsh == 1) {
                    sb[0] = *(gword_a2_t)p;
                } else {
                    sb[0] = *(ghalf_t)p;
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < NW; ++i) {
                sb[i] = 0;  // a weight past the row's end is 0
                if constexpr (SB32) {
                    if (i < ng) sb[i] = ((gword_t)p)[i];
                } else {
                    if (2 * i < ng) sb[i] = ((ghalf_t)p)[2 * i];
                    if (2 * i + 1 < ng) sb[i] |= (uint32_t)((ghalf_t)p)[2 * i + 1] << 16;
                }
            }
        }
    }
    // The scales to every lane group, and the biases.
    RQ_DEV void spread_sb(uint32_t* sv, uint32_t* bv) const {
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            const auto r0 = __builtin_amdgcn_permlane32_swap(sb[i], sb[i], false, false);
            const auto r1 = __builtin_amdgcn_permlane16_swap(r0[0], r0[0], false, false);
            sv[i] = r1[0];
            bv[i] = r1[1];
        }
    }
    // Value of the span's group g.
    RQ_DEV static float group_value(const uint32_t* v, int g, bool f16) {
        if constexpr (SB32) return __uint_as_float(v[g]);
        const uint32_t h = (v[g >> 1] >> (16 * (g & 1))) & 0xffffu;
        return f16 ? f16_bits_to_f32(h) : bf16_bits_to_f32(h);
    }
    // The weights as the fragments of four MFMAs: frag[2 h + j] holds, in lane
    // (lg, lr), k = 64 h + 16 lg + 8 j .. +7 of row lr.
    RQ_DEV void fragments(int gsh, int lg, bool f16, u32x4_t* frag) {
        uint32_t sv[NW], bv[NW];
        spread_sb(sv, bv);
        if constexpr (BITS % 2 == 0) {
            // 16 codes are BITS / 2 whole words: spread the packed words, then
            // dequantize; group of the lane's codes of half h: (2 h + lg / 2) >> gsh
            constexpr int HW = BITS / 2;
            uint32_t p[2][HW];
#pragma unroll
            for (int i = 0; i < HW; ++i) {
                p[0][i] = w[i];
                p[1][i] = w[HW + i];
                spread_pieces(p[0][i], p[1][i]);
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                uint32_t d[8];
                const float s = value(sv, gsh, h, lg >> 1, f16), b = value(bv, gsh, h, lg >> 1, f16);
                dequant_half_run<BITS>(p[h], s, b, d);
                frag[2 * h] = u32x4_t{d[0], d[1], d[2], d[3]};
                frag[2 * h + 1] = u32x4_t{d[4], d[5], d[6], d[7]};
            }
        } else {
            // odd widths: dequantize the lane's own run (group lg >> gsh), then
            // spread its 16 bf16 pairs
            uint32_t d[16];
            const float s0 = value(sv, gsh, 0, lg & 1, f16), s1 = value(sv, gsh, 1, lg & 1, f16);
            const float b0 = value(bv, gsh, 0, lg & 1, f16), b1 = value(bv, gsh, 1, lg & 1, f16);
            dequant_run_bf16<BITS>(w, lg < 2 ? s0 : s1, lg < 2 ? b0 : b1, d);
#pragma unroll
            for (int i = 0; i < 8; ++i) spread_pieces(d[i], d[8 + i]);
#pragma unroll
            for (int j = 0; j < 4; ++j) frag[j] = u32x4_t{d[4 * j], d[4 * j + 1], d[4 * j + 2], d[4 * j + 3]};
        }
    }
    // Value of run 2 h + o of the span (h wave-uniform, o per lane).
    RQ_DEV static float value(const uint32_t* v, int gsh, int h, int o, bool f16) {
        if constexpr (SB32) {
            const uint32_t r = o ? v[2 * h + 1] : v[2 * h];
            return __uint_as_float(gsh == 0 ? r : (gsh == 1 ? v[h] : v[0]));
        } else {
            const int sh = gsh == 0 ? 16 * o : (gsh == 1 ? 16 * h : 0);
            const uint32_t r = ((gsh == 0 && h) ? v[1] : v[0]) >> sh;
            return f16 ? f16_bits_to_f32(r & 0xffffu) : bf16_bits_to_f32(r);
        }
    }
};

// Eight consecutive activations of one row, as they are loaded.  XF: fp32
// ones, rounded to bf16 (RNE) on their way to LDS; else 16-bit ones, f16
// converted when `f16`.
template <bool XF>
struct XPiece {
    u32x4_t v[XF ? 2 : 1];
    RQ_DEV void load(const uint8_t* base, uint32_t off) {
        const gbyte_t p = (gbyte_t)base + off;
        v[0] = *(gvec_a2_t)p;
        if constexpr (XF) v[1] = *((gvec_a2_t)p + 1);
    }
    // the first n of them (n < 8), zeros beyond
    RQ_DEV void load_part(const uint8_t* base, uint32_t off, int n) {
        const gbyte_t p = (gbyte_t)base + off;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if constexpr (XF) {
                v[0][e] = e < n ? ((gword_t)p)[e] : 0u;
                v[1][e] = 4 + e < n ? ((gword_t)p)[4 + e] : 0u;
            } else {
                v[0][e] = (2 * e < n ? (uint32_t)((ghalf_t)p)[2 * e] : 0u) |
                          (2 * e + 1 < n ? (uint32_t)((ghalf_t)p)[2 * e + 1] << 16 : 0u);
            }
        }
    }
    // what bf16() leaves of fp32 or f16 values, rounded to bf16
    RQ_DEV u32x4_t rest(u32x4_t hi) const {
        u32x4_t r;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float f0, f1;
            if constexpr (XF) {
                f0 = __uint_as_float(v[e >> 1][2 * (e & 1)]);
                f1 = __uint_as_float(v[e >> 1][2 * (e & 1) + 1]);
            } else {
                f0 = f16_bits_to_f32(v[0][e] & 0xffffu);
                f1 = f16_bits_to_f32(v[0][e] >> 16);
            }
            r[e] = pack_bf16x2(f0 - __uint_as_float(hi[e] << 16), f1 - __uint_as_float(hi[e] & 0xffff0000u));
        }
        return r;
    }
    RQ_DEV u32x4_t bf16(bool f16) const {
        if constexpr (XF) {
            return u32x4_t{pack_bf16x2(__uint_as_float(v[0][0]), __uint_as_float(v[0][1])),
                           pack_bf16x2(__uint_as_float(v[0][2]), __uint_as_float(v[0][3])),
                           pack_bf16x2(__uint_as_float(v[1][0]), __uint_as_float(v[1][1])),
                           pack_bf16x2(__uint_as_float(v[1][2]), __uint_as_float(v[1][3]))};
        } else {
            u32x4_t r = v[0];
            if (f16) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    r[e] = pack_bf16x2(f16_bits_to_f32(r[e] & 0xffffu), f16_bits_to_f32(r[e] >> 16));
            }
            return r;
        }
    }
};

// Four consecutive outputs of row m at columns n.. (rows >= M and columns >=
// ld are not written).
RQ_DEV void store_out4(const MidArgs& a, int64_t m, int64_t n, int64_t ld, f32x4_t v) {
    if (m >= a.M) return;
    const int64_t o = m * ld + n;
    if (a.y_vec && n + 4 <= ld) {
        if (a.y_dt == RQ_F32)
            *(f32x4_t*)((float*)a.y + o) = v;
        else
            *(u32x2_t*)((uint16_t*)a.y + o) =
                u32x2_t{pack2_dt(a.y_dt, v[0], v[1]), pack2_dt(a.y_dt, v[2], v[3])};
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (n + e < ld) store_dt(a.y, a.y_dt, o + e, v[e]);
}

// The QLoRA low-rank term of one 16x16 tile (outputs n0 + 4 lg .. +3 of row
// m0 + lr): v += scale * z . L^T, z [M, rank] and L [ncols, rank] bf16 (its
// transpose [rank, l_ld] when stored).
RQ_DEV f32x4_t add_lora(const rq::LoraArgs& lo, f32x4_t v, int64_t M, int64_t ncols, int64_t m0,
                        int64_t n0, int lane) {
    const int lg = lane >> 4, lr = lane & 15;
    const int64_t m = m0 + lr, n = n0 + lr;
    f32x4_t t = {0.f, 0.f, 0.f, 0.f};
    for (int j0 = 0; j0 < lo.rank; j0 += 32) {
        const int j = j0 + 8 * lg;
        u32x4_t zf = {0u, 0u, 0u, 0u}, lf = zf;
        if (j < lo.rank && m < M) zf = *(const u32x4_t*)((const uint16_t*)lo.z + m * lo.rank + j);
        if (j < lo.rank && n < ncols) {
            const uint16_t* l = (const uint16_t*)lo.l;
            if (lo.stored) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    lf[q] = (uint32_t)l[(j + 2 * q) * lo.l_ld + n] |
                            ((uint32_t)l[(j + 2 * q + 1) * lo.l_ld + n] << 16);
            } else {
                lf = *(const u32x4_t*)(l + n * lo.rank + j);
            }
        }
        t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, lf),
                                                    __builtin_bit_cast(bf16x8_t, zf), t, 0, 0, 0);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = fmaf(lo.scale, t[e], v[e]);
    return v;
}

// XD: halves of a span (64 k) of activations in flight ahead of the MFMAs.
template <int BITS, bool SB32, bool XF, int TM, int TN, int MAXW, int XD>
__global__ __launch_bounds__(64 * MAXW) void qmm_t_mid(const MidArgs a) {
    // per wave: its activation tile of 64 k (2 KB per 16 rows), later its
    // fp32 output tile [tile][lane]
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    constexpr int T = TM * TN;
    constexpr int ES = XF ? 4 : 2;
    constexpr int WB = mid_wave_bytes(TM, TN);
    const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lg = lane >> 4, lr = lane & 15;
    // consecutive blocks go to different XCDs: each XCD takes a contiguous
    // range of tiles, the row tiles of one weight panel next to each other
    const int nt = a.tiles_m * a.tiles_n, per = (nt + 7) >> 3;
    const int t0 = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (t0 >= nt) return;
    const int64_t n0 = (int64_t)(t0 / a.tiles_m) * (16 * TN), m0 = (int64_t)(t0 % a.tiles_m) * (16 * TM);

    const int runs = (int)(a.K >> 5);
    const int sp0 = wave * a.spw, nspan = (runs + 3) >> 2;
    const int sp1 = sp0 + a.spw < nspan ? sp0 + a.spw : nspan;
    const int64_t wpr = (int64_t)runs * BITS, G = a.K >> a.gs_shift;
    const int gsh = a.gs_shift - 5;
    constexpr int SBS = SB32 ? 4 : 2;

    const uint8_t* wbase = (const uint8_t*)(a.wq + n0 * wpr);
    uint32_t woff[TN];  // this lane's weight rows, the last row for those past it
    gbyte_t sbp[TN];    // and their scales (even lane groups) or biases
#pragma unroll
    for (int b = 0; b < TN; ++b) {
        const int left = a.R - n0 < 16 * TN ? (int)(a.R - n0) : 16 * TN;
        const int nr = 16 * b + lr < left ? 16 * b + lr : left - 1;
        woff[b] = (uint32_t)nr * (uint32_t)wpr * 4;
        sbp[b] = (gbyte_t)((lg & 1) ? a.biases : a.scales) + ((n0 + nr) * G + ((4 * sp0) >> gsh)) * SBS;
    }
    SpanRegs<BITS, SB32> cur[TN], nxt[TN];
    auto load_span = [&](SpanRegs<BITS, SB32>(&r)[TN], int sp) {
        // a run past the row's end reads the last one; its k-steps are not run
        const int run = 4 * sp + lg < runs ? 4 * sp + lg : runs - 1;
#pragma unroll
        for (int b = 0; b < TN; ++b) r[b].load_codes(wbase, woff[b] + run * BITS * 4);
        if (lg < 2) {
            const int left = (runs - 4 * sp + (1 << gsh) - 1) >> gsh, ng = 4 >> gsh;
#pragma unroll
            for (int b = 0; b < TN; ++b)
                r[b].load_sb(sbp[b] + (int64_t)((4 * (sp - sp0)) >> gsh) * SBS, gsh, left < ng ? left : ng);
        }
    };
    // Activations: load q covers rows 8q .. 8q+7 of the tile, 64 k (one whole
    // 128-byte line a row in 16 bits): eight consecutive lanes read one row.
    // Groups of rows past M repeat the last one.
    const int qlast = (a.M - m0 < 16 * TM ? (int)(a.M - m0) - 1 : 16 * TM - 1) >> 3;
    const int rem = a.M - m0 - 8 * qlast < 8 ? (int)(a.M - m0) - 8 * qlast : 8;
    const int xr = lane >> 3, xc = lane & 7;
    const uint32_t xfull = (uint32_t)xr * (uint32_t)a.K * ES;
    const uint32_t xpart = (uint32_t)(xr < rem ? xr : rem - 1) * (uint32_t)a.K * ES;
    const uint8_t* xbase = a.x + m0 * a.K * ES;
    XPiece<XF> xv[XD][2 * TM];
    auto load_x = [&](XPiece<XF>(&v)[2 * TM], int half) {  // half: index of the 64 k
        // a k past the row's end reads the half's first 32 (never used)
        const int c = 64 * half + 8 * xc < a.K ? xc : xc & 3;
        const uint32_t ko = (64 * half + 8 * c) * ES;
#pragma unroll
        for (int q = 0; q < 2 * TM; ++q) {
            const int qe = q < qlast ? q : qlast;
            v[q].load(xbase + (int64_t)(8 * qe) * a.K * ES, (qe == qlast ? xpart : xfull) + ko);
        }
    };
    // LDS tile: 16-byte chunk c of row r at (c ^ (r & 7)), 128 bytes a row
    uint8_t* xs = lds + wave * WB;
    uint8_t* xw = xs + xr * 128 + ((xc ^ xr) << 4);
    const uint32_t xrd = wave * WB + lr * 128 + (((2 * lg) ^ (lr & 7)) << 4);

    f32x4_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int b = 0; b < TN; ++b) acc[i][b] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    const int h1 = 2 * sp1 < (runs + 1) >> 1 ? 2 * sp1 : (runs + 1) >> 1;  // halves of the slice end here
    load_span(cur, sp0);
#pragma unroll
    for (int d = 0; d < XD; ++d)
        if (2 * sp0 + d < h1) load_x(xv[d], 2 * sp0 + d);
    for (int sp = sp0; sp < sp1; ++sp) {
        if (sp + 1 < sp1) load_span(nxt, sp + 1);
        u32x4_t wf[TN][4];
#pragma unroll
        for (int b = 0; b < TN; ++b) cur[b].fragments(gsh, lg, a.sb_f16, wf[b]);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int half = 2 * sp + h;
            if (half < h1) {
                // x past the row's end is 0
                if (64 * half + 64 > a.K && xc >= 4) {
#pragma unroll
                    for (int q = 0; q < 2 * TM; ++q) *(u32x4_t*)(xw + q * 1024) = u32x4_t{0u, 0u, 0u, 0u};
                } else {
#pragma unroll
                    for (int q = 0; q < 2 * TM; ++q) *(u32x4_t*)(xw + q * 1024) = xv[h % XD][q].bf16(a.x_f16);
                }
                if (half + XD < h1) load_x(xv[h % XD], half + XD);
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int i = 0; i < TM; ++i) {
                        const bf16x8_t xf = __builtin_bit_cast(
                            bf16x8_t, *(const u32x4_t*)(lds + (xrd ^ (16 * j)) + i * 2048));
#pragma unroll
                        for (int b = 0; b < TN; ++b)
                            acc[i][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                __builtin_bit_cast(bf16x8_t, wf[b][2 * h + j]), xf, acc[i][b], 0, 0, 0);
                    }
            }
        }
#pragma unroll
        for (int b = 0; b < TN; ++b) cur[b] = nxt[b];
    }

    if (nw > 1) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int b = 0; b < TN; ++b)
                *(f32x4_t*)(xs + ((i * TN + b) * 64 + lane) * 16) = acc[i][b];
        __syncthreads();
        for (int t = wave; t < T; t += nw) {
            const uint8_t* p = lds + (t * 64 + lane) * 16;
            f32x4_t v = *(const f32x4_t*)p;
            for (int w = 1; w < nw; ++w) {
                const f32x4_t u = *(const f32x4_t*)(p + w * WB);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] += u[e];
            }
            const int64_t m = m0 + 16 * (t / TN), n = n0 + 16 * (t % TN);
            if (a.lora.z) v = add_lora(a.lora, v, a.M, a.R, m, n, lane);
            store_out4(a, m + lr, n + 4 * lg, a.R, v);
        }
    } else {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int b = 0; b < TN; ++b) {
                const int64_t m = m0 + 16 * i, n = n0 + 16 * b;
                f32x4_t v = acc[i][b];
                if (a.lora.z) v = add_lora(a.lora, v, a.M, a.R, m, n, lane);
                store_out4(a, m + lr, n + 4 * lg, a.R, v);
            }
    }
}

// --------------------------------------------------------------- qmv_mid
//
// The decode GEMV of up to 16 activation rows for launches of few weight rows
// (one projection, or the independent ones of a layer): one block per 16
// weight rows, its waves over slices of the contraction as in qmm_t_mid.  The
// weights are not rounded: the codes enter the MFMA as integers (exact in
// bf16) and each group's scale and bias are applied to its sums in fp32, acc +=
// s D + b X, X the group's activation sums from a second MFMA against ones.
// The activations are the A operand, so an accumulator column is one weight
// row and a lane needs one (scale, bias) per group.  An MFMA contracts 32
// consecutive k, inside one group at every group size.  xsplit: rows m/2 .. m-1
// hold what bf16 leaves of the fp32 or f16 activations of rows 0 .. m/2-1 (m at
// most 4), and the two are added before the store.
struct QmvMidArgs {
    rq_problem p[RQ_MAX_GROUPED];
    int block_start[RQ_MAX_GROUPED + 1];
    int n, m, sb_f16, x_f16, y_dt, spw;
    int xsplit;
};

// 4 x 4 transpose of (lane group, register): afterwards register j of lane
// group g holds what register g of lane group j held.
RQ_DEV void transpose_lane_groups(uint32_t& a, uint32_t& b, uint32_t& c, uint32_t& d) {
    const auto r0 = __builtin_amdgcn_permlane32_swap(a, c, false, false);
    const auto r1 = __builtin_amdgcn_permlane32_swap(b, d, false, false);
    const auto r2 = __builtin_amdgcn_permlane16_swap(r0[0], r1[0], false, false);
    const auto r3 = __builtin_amdgcn_permlane16_swap(r0[1], r1[1], false, false);
    a = r2[0]; b = r2[1]; c = r3[0]; d = r3[1];
}

// A lane's run of codes -> the four fragments of the span as bf16 integers:
// frag[j] holds, in lane (lg, lr), k = 32 j + 8 lg .. +7 of row lr.
template <int BITS>
RQ_DEV void code_fragments(const uint32_t* words, u32x4_t* frag) {
    if constexpr (BITS == 4 || BITS == 8) {
        // eight codes are whole words: spread the packed words
        constexpr int HW = BITS / 4;
        uint32_t w[4 * HW];
#pragma unroll
        for (int i = 0; i < 4 * HW; ++i) w[i] = words[i];
#pragma unroll
        for (int i = 0; i < HW; ++i) transpose_lane_groups(w[i], w[HW + i], w[2 * HW + i], w[3 * HW + i]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if constexpr (BITS == 4) {
                typedef float f32x2_t __attribute__((ext_vector_type(2)));
                const uint32_t lo = w[j] & 0x0F0F0F0Fu, hi = (w[j] >> 4) & 0x0F0F0F0Fu;
                const f32x2_t l0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(lo, 512.f, false);
                const f32x2_t l1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(lo, 512.f, true);
                const f32x2_t h0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(hi, 512.f, false);
                const f32x2_t h1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(hi, 512.f, true);
                frag[j] = u32x4_t{pack_bf16x2(l0[0], h0[0]), pack_bf16x2(l0[1], h0[1]),
                                  pack_bf16x2(l1[0], h1[0]), pack_bf16x2(l1[1], h1[1])};
            } else {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    uint32_t v = w[2 * j + h];
                    asm("" : "+v"(v));
                    frag[j][2 * h] = pack_bf16x2((float)(uint8_t)v, (float)(uint8_t)(v >> 8));
                    frag[j][2 * h + 1] = pack_bf16x2((float)(uint8_t)(v >> 16), (float)(uint8_t)(v >> 24));
                }
            }
        }
    } else {
        uint32_t d[16];
#pragma unroll
        for (int i = 0; i < 16; ++i)
            d[i] = pack_bf16x2((float)run_code<BITS>(words, 2 * i), (float)run_code<BITS>(words, 2 * i + 1));
#pragma unroll
        for (int e = 0; e < 4; ++e) transpose_lane_groups(d[e], d[4 + e], d[8 + e], d[12 + e]);
#pragma unroll
        for (int j = 0; j < 4; ++j) frag[j] = u32x4_t{d[4 * j], d[4 * j + 1], d[4 * j + 2], d[4 * j + 3]};
    }
}

template <int BITS, bool SB32, bool XF, int GSH>
__global__ __launch_bounds__(1024) void qmv_mid(const QmvMidArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];  // 2 KB per wave
    constexpr int ES = XF ? 4 : 2, SBS = SB32 ? 4 : 2;
    constexpr int gsh = GSH - 5, KG = 1 << gsh;  // 32-wide k-steps per group
    const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lg = lane >> 4, lr = lane & 15;
    int lo = 0, hi = a.n - 1;  // last problem whose first block is not past this one
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (a.block_start[mid] <= (int)blockIdx.x) lo = mid; else hi = mid - 1;
    }
    const rq_problem& P = a.p[lo];
    const int64_t R = P.rows, K = P.cols;
    const int64_t n0 = (int64_t)((int)blockIdx.x - a.block_start[lo]) * 16;
    const int runs = (int)(K >> 5), nspan = (runs + 3) >> 2;
    const int sp0 = wave * a.spw, sp1 = sp0 + a.spw < nspan ? sp0 + a.spw : nspan;
    const int64_t wpr = (int64_t)runs * BITS, G = K >> GSH;

    const uint8_t* wbase = (const uint8_t*)(P.w_q + n0 * wpr);
    const int nr = R - n0 < 16 && lr >= (int)(R - n0) ? (int)(R - n0) - 1 : lr;
    const uint32_t woff = (uint32_t)nr * (uint32_t)wpr * 4;
    const gbyte_t sbp = (gbyte_t)((lg & 1) ? P.biases : P.scales) + ((n0 + nr) * G + ((4 * sp0) >> gsh)) * SBS;
    SpanRegs<BITS, SB32> cur, nxt;
    auto load_span = [&](SpanRegs<BITS, SB32>& r, int sp) {
        // a run past the row's end reads the last one; its k-step is not run
        const int run = 4 * sp + lg < runs ? 4 * sp + lg : runs - 1;
        r.load_codes(wbase, woff + run * BITS * 4);
        if (lg < 2) {
            const int left = (runs - 4 * sp + KG - 1) >> gsh, ng = 4 >> gsh;
            r.load_sb(sbp + (int64_t)((4 * (sp - sp0)) >> gsh) * SBS, gsh, left < ng ? left : ng);
        }
    };
    // activations as in qmm_t_mid, one 16-row tile: rows past m repeat the last
    const int xr = lane >> 3, xc = lane & 7;
    const int xm = a.xsplit ? a.m >> 1 : a.m;
    const bool xlo = a.xsplit && xr >= xm && xr < a.m;
    uint32_t xoff[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int r = 8 * q + xr - (xlo && q == 0 ? xm : 0);
        xoff[q] = (uint32_t)(r < xm ? r : xm - 1) * (uint32_t)K * ES;
    }
    XPiece<XF> xv[2][2];
    auto load_x = [&](XPiece<XF>(&v)[2], int half) {
        // a k past the row's end reads the half's first 32 (its k-step is not run)
        const int c = 64 * half + 8 * xc < K ? xc : xc & 3;
#pragma unroll
        for (int q = 0; q < 2; ++q) v[q].load((const uint8_t*)P.x, xoff[q] + (uint32_t)(64 * half + 8 * c) * ES);
    };
    uint8_t* xs = lds + wave * 2048;
    uint8_t* xw = xs + xr * 128 + ((xc ^ xr) << 4);
    const uint32_t xrd = wave * 2048 + lr * 128 + ((lg ^ (lr & 7)) << 4);

    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    const bf16x8_t ones = __builtin_bit_cast(bf16x8_t, u32x4_t{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u});
    f32x4_t acc = zero;
    const int h1 = 2 * sp1 < (runs + 1) >> 1 ? 2 * sp1 : (runs + 1) >> 1;
    load_span(cur, sp0);
    load_x(xv[0], 2 * sp0);
    if (2 * sp0 + 1 < h1) load_x(xv[1], 2 * sp0 + 1);
    for (int sp = sp0; sp < sp1; ++sp) {
        if (sp + 1 < sp1) load_span(nxt, sp + 1);
        uint32_t sv[SpanRegs<BITS, SB32>::NW], bv[SpanRegs<BITS, SB32>::NW];
        cur.spread_sb(sv, bv);
        u32x4_t wf[4];
        code_fragments<BITS>(cur.w, wf);
        f32x4_t D = zero, X = zero;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int half = 2 * sp + h;
            if (half < h1) {
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    u32x4_t v = xv[h][q].bf16(a.x_f16);
                    if (xlo && q == 0) v = xv[h][q].rest(v);
                    *(u32x4_t*)(xw + q * 1024) = v;
                }
                if (half + 2 < h1) load_x(xv[h], half + 2);
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int j = 2 * h + i;
                    if (2 * half + i < runs) {
                        const bf16x8_t xf =
                            __builtin_bit_cast(bf16x8_t, *(const u32x4_t*)(lds + (xrd ^ (64 * i))));
                        const bool first = j % KG == 0;
                        D = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf, __builtin_bit_cast(bf16x8_t, wf[j]),
                                                                    first ? zero : D, 0, 0, 0);
                        X = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf, ones, first ? zero : X, 0, 0, 0);
                        if (j % KG == KG - 1) {  // the group's last k-step (groups are whole)
                            const float s = SpanRegs<BITS, SB32>::group_value(sv, j >> gsh, a.sb_f16);
                            const float b = SpanRegs<BITS, SB32>::group_value(bv, j >> gsh, a.sb_f16);
#pragma unroll
                            for (int e = 0; e < 4; ++e) acc[e] = fmaf(s, D[e], fmaf(b, X[e], acc[e]));
                        }
                    }
                }
            }
        }
        cur = nxt;
    }
    if (nw > 1) {
        *(f32x4_t*)(xs + lane * 16) = acc;
        __syncthreads();
        if (wave) return;
        for (int w = 1; w < nw; ++w) {
            const f32x4_t u = *(const f32x4_t*)(lds + w * 2048 + lane * 16);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] += u[e];
        }
    }
    // lane (lg, lr): activation rows 4 lg + e, weight row lr
    if (a.xsplit) {
        acc[0] += xm == 1 ? acc[1] : acc[2];
        acc[1] += acc[3];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (4 * lg + e < xm && n0 + lr < R) store_dt(P.y, a.y_dt, (4 * lg + e) * R + n0 + lr, acc[e]);
}

// ------------------------------------------------------------- qmm_n_mid
//
// y[m, k] = sum_r x[m, r] * ŵ[r, k].  The contraction runs over the weight
// rows, the packed codes along k.  The MFMA's output index along k is free to
// be any permutation of the tile's columns, so no transpose is needed: lane
// (lg, lr) holds the NC (8 or 4) codes at columns NC lr .. of the rows 8 lg ..
// +7 of a 32-row step, and the c-th of NC MFMAs contracts those 32 rows for the
// columns {NC lr + c}, its operand the c-th code of the lane's eight rows.  A
// block is a tile of 16*TM activation rows x 16*NC columns; its waves take
// contiguous slices of the weight rows and add their tiles through LDS in wave
// order.  A load instruction reads 4 rows x 16*NC codes.  (The codes loaded as
// whole row segments and read back through LDS: the same times; what bounds it
// is the ~2.5 VALU instructions per code, and with few columns the number of
// blocks, since a block dequantizes all rows of its columns.)
// The step's scales and biases (32 rows x the tile's groups) come in one load
// and go through wave-private LDS as fp32 pairs; activations are staged as in
// qmm_t_mid, 64 weight rows at a time.

// NC (4 or 8) consecutive codes of one row in one load: the bytes they fill at
// 2, 4 and 8 bits, else two words of the run shifted so that they start at bit 0.
template <int BITS, int NC>
struct Codes {
    static constexpr int NB = BITS * NC;  // bits
    static constexpr bool SH = BITS == 3 || BITS >= 5 && BITS < 8;
    static constexpr int NW = SH || NB > 32 ? 2 : 1;
    uint32_t w[NW];
    // piece p of a run: byte offset of the load within the run, and the shift
    RQ_DEV static int offset(int p) {
        if constexpr (!SH) return p * (NB / 8);
        const int o = (p * NB) >> 5;
        return 4 * (o < BITS - 2 ? o : BITS - 2);
    }
    RQ_DEV static int shift(int p) {
        if constexpr (!SH) return 0;
        return p * NB - 8 * offset(p);
    }
    RQ_DEV void load(const uint8_t* base, uint32_t off) {
        const gbyte_t p = (gbyte_t)base + off;
        if constexpr (NW == 2) {
            const u32x2_t v = *(gvec2_a4_t)p;
            w[0] = v[0];
            w[1] = v[1];
        } else if constexpr (NB == 32) {
            w[0] = *(gword_t)p;
        } else if constexpr (NB == 16) {
            w[0] = *(ghalf_t)p;
        } else {
            static_assert(NB == 8, "");
            w[0] = *p;
        }
    }
    // scale * code + bias, fp32
    RQ_DEV void values(int sh, float s, float b, float* out) const {
        if constexpr (BITS == 4) {
            typedef float f32x2_t __attribute__((ext_vector_type(2)));
            const uint32_t lo = w[0] & 0x0F0F0F0Fu, hi = (w[0] >> 4) & 0x0F0F0F0Fu;
#pragma unroll
            for (int i = 0; i < NC / 4; ++i) {
                const f32x2_t l = i ? __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(lo, 512.f, true)
                                    : __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(lo, 512.f, false);
                const f32x2_t h = i ? __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(hi, 512.f, true)
                                    : __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(hi, 512.f, false);
                out[4 * i] = fmaf(s, l[0], b);
                out[4 * i + 1] = fmaf(s, h[0], b);
                out[4 * i + 2] = fmaf(s, l[1], b);
                out[4 * i + 3] = fmaf(s, h[1], b);
            }
        } else if constexpr (BITS == 8) {
#pragma unroll
            for (int h = 0; h < NC / 4; ++h) {
                uint32_t v = w[h];
                asm("" : "+v"(v));
#pragma unroll
                for (int i = 0; i < 4; ++i) out[4 * h + i] = fmaf(s, (float)(uint8_t)(v >> (8 * i)), b);
            }
        } else if constexpr (BITS == 2) {
#pragma unroll
            for (int i = 0; i < NC; ++i) out[i] = fmaf(s, (float)((w[0] >> (2 * i)) & 3u), b);
        } else {
            const uint64_t v = (((uint64_t)w[1] << 32) | w[0]) >> sh;
            const uint32_t d[2] = {(uint32_t)v, (uint32_t)(v >> 32)};
#pragma unroll
            for (int i = 0; i < NC; ++i) out[i] = fmaf(s, (float)run_code<BITS>(d, i), b);
        }
    }
};

// LDS of a wave: activations (2 KB per 16 rows) and the (scale, bias) pairs of
// a step (256 B per group); later 16x16 tiles of its fp32 output, `pass` row
// tiles at a time.
__host__ __device__ constexpr int mid_n_pass(int tm, int nc) { return tm * nc <= 16 ? tm : 16 / nc; }
__host__ __device__ constexpr int mid_n_wave_bytes(int tm, int nc) {
    const int in = 2048 * tm + 256 * (nc / 2), out = 1024 * nc * mid_n_pass(tm, nc);
    return in > out ? in : out;
}
// fp32 row stride of the block's output tile
__host__ __device__ constexpr int mid_n_out_row(int nc) { return 16 * nc + 4; }
__host__ __device__ constexpr int mid_n_out_bytes(int tm, int nc) {
    return 16 * mid_n_pass(tm, nc) * mid_n_out_row(nc) * 4;
}

template <int BITS, bool SB32, bool XF, int TM, int NC, int MAXW>
__global__ __launch_bounds__(64 * MAXW) void qmm_n_mid(const MidArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    constexpr int ES = XF ? 4 : 2, SBS = SB32 ? 4 : 2, CT = 16 * NC;
    constexpr int WB = mid_n_wave_bytes(TM, NC), TP = mid_n_pass(TM, NC);
    const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lg = lane >> 4, lr = lane & 15;
    const int nt = a.tiles_m * a.tiles_n, per = (nt + 7) >> 3;
    const int t0 = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (t0 >= nt) return;
    const int64_t c0 = (int64_t)(t0 / a.tiles_m) * CT, m0 = (int64_t)(t0 % a.tiles_m) * (16 * TM);

    const int64_t wpr = (a.K >> 5) * BITS, G = a.K >> a.gs_shift;
    const int gsh = a.gs_shift - 5;
    const int nhalf = (int)((a.R + 63) >> 6);  // 64 weight rows each
    const int h0 = wave * a.spw, h1 = h0 + a.spw < nhalf ? h0 + a.spw : nhalf;

    // codes: piece lr of the tile, the last piece of the row for those past it
    constexpr int PR = 32 / NC;  // pieces of a run
    const int pieces = a.K - c0 < CT ? (int)(a.K - c0) / NC : 16;
    const int pc = lr < pieces ? lr : pieces - 1;
    const uint8_t* wbase = (const uint8_t*)a.wq + (c0 >> 5) * (BITS * 4);
    const uint32_t wcol = (uint32_t)(pc / PR) * (BITS * 4) + Codes<BITS, NC>::offset(pc % PR);
    const uint32_t woff = (uint32_t)(8 * lg) * (uint32_t)wpr * 4 + wcol;
    const int csh = Codes<BITS, NC>::shift(pc % PR);
    // scales (lanes 0-31) and biases (lanes 32-63) of row lane % 32 of a step;
    // the tile's groups are those of a 128-wide span of twice the group size at NC = 4
    const int gst = NC == 8 ? gsh : (gsh < 2 ? gsh + 1 : 2);
    const int ngf = 4 >> gst, ngl = (int)(G - (c0 >> a.gs_shift)), ng = ngl < ngf ? ngl : ngf;
    const gbyte_t sbp = (gbyte_t)(lane < 32 ? a.scales : a.biases) + (c0 >> a.gs_shift) * SBS;

    const int rlive = (int)a.R - (lane & 31);  // row lane % 32 of a step is there below this
    Codes<BITS, NC> cw[2][8];
    SpanRegs<BITS, SB32> sbr[2];  // only its scale words are used
    auto load_step = [&](Codes<BITS, NC>(&c)[8], SpanRegs<BITS, SB32>& sb, int step) {
        const int64_t r0 = 32 * (int64_t)step;
        if (r0 + 32 <= a.R) {
#pragma unroll
            for (int i = 0; i < 8; ++i) c[i].load(wbase + (r0 + i) * wpr * 4, woff);
        } else {  // rows past the end repeat the last one's codes
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int64_t r = r0 + 8 * lg + i < a.R ? r0 + 8 * lg + i : a.R - 1;
                c[i].load(wbase + r * wpr * 4, wcol);
            }
        }
        const int64_t sr = r0 + (lane & 31) < a.R ? r0 + (lane & 31) : a.R - 1;
        sb.load_sb(sbp + sr * G * SBS, gst, ng);
    };
    // activations: as in qmm_t_mid, k -> weight row
    const int qlast = (a.M - m0 < 16 * TM ? (int)(a.M - m0) - 1 : 16 * TM - 1) >> 3;
    const int rem = a.M - m0 - 8 * qlast < 8 ? (int)(a.M - m0) - 8 * qlast : 8;
    const int xr = lane >> 3, xc = lane & 7;
    const uint32_t xfull = (uint32_t)xr * (uint32_t)a.R * ES;
    const uint32_t xpart = (uint32_t)(xr < rem ? xr : rem - 1) * (uint32_t)a.R * ES;
    const uint8_t* xbase = a.x + m0 * a.R * ES;
    XPiece<XF> xv[2 * TM];
    auto load_x = [&](int half) {
        const uint32_t ko = (uint32_t)(64 * half + 8 * xc) * ES;
        if (64 * (int64_t)half + 64 <= a.R) {
#pragma unroll
            for (int q = 0; q < 2 * TM; ++q) {
                const int qe = q < qlast ? q : qlast;
                xv[q].load(xbase + (int64_t)(8 * qe) * a.R * ES, (qe == qlast ? xpart : xfull) + ko);
            }
        } else {
            const int left = (int)(a.R - 64 * (int64_t)half) - 8 * xc;  // zeros past the last row
#pragma unroll
            for (int q = 0; q < 2 * TM; ++q) {
                const int qe = q < qlast ? q : qlast;
                xv[q].load_part(xbase + (int64_t)(8 * qe) * a.R * ES, (qe == qlast ? xpart : xfull) + ko,
                                left < 8 ? left : 8);
            }
        }
    };
    uint8_t* xs = lds + wave * WB;
    uint8_t* xw = xs + xr * 128 + ((xc ^ xr) << 4);
    const uint32_t xrd = wave * WB + lr * 128 + ((lg ^ (lr & 7)) << 4);
    // (scale, bias) pairs of a step: [group][row] behind the activations
    uint8_t* sbw = xs + TM * 2048 + (lane & 31) * 8 + (lane >> 5) * 4;
    const uint8_t* sbrd = xs + TM * 2048 + ((NC * lr) >> a.gs_shift) * 256 + lg * 64;

    f32x4_t acc[TM][NC];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[i][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    const int nstep = (int)((a.R + 31) >> 5), s1 = 2 * h1 < nstep ? 2 * h1 : nstep;
    load_step(cw[0], sbr[0], 2 * h0);
    load_x(h0);
    for (int half = h0; half < h1; ++half) {
#pragma unroll
        for (int q = 0; q < 2 * TM; ++q) *(u32x4_t*)(xw + q * 1024) = xv[q].bf16(a.x_f16);
        if (half + 1 < h1) load_x(half + 1);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int step = 2 * half + j;
            if (step < s1) {
                if (step + 1 < s1) load_step(cw[j ^ 1], sbr[j ^ 1], step + 1);
#pragma unroll
                for (int g = 0; g < NC / 2; ++g) {
                    if (g < ngf) {
                        float v;
                        if constexpr (SB32) {
                            v = __uint_as_float(sbr[j].sb[g]);
                        } else {
                            const uint32_t h = (g & 1) ? sbr[j].sb[g >> 1] >> 16 : sbr[j].sb[g >> 1] & 0xffffu;
                            v = a.sb_f16 ? f16_bits_to_f32(h) : bf16_bits_to_f32(h);
                        }
                        // rows past the end are 0, as x is there: an infinite weight times 0
                        // would be NaN (cleared here and not as they are loaded, where it
                        // waited for the load: [768, 768] at M = 200 6.7 us, 6.0 here)
                        *(float*)(sbw + g * 256) = 32 * step < rlive ? v : 0.f;
                    }
                }
                f32x4_t sb[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) sb[i] = *(const f32x4_t*)(sbrd + 16 * i);
                uint32_t wf[NC][4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float v0[NC], v1[NC];
                    cw[j][2 * i].values(csh, sb[i][0], sb[i][1], v0);
                    cw[j][2 * i + 1].values(csh, sb[i][2], sb[i][3], v1);
#pragma unroll
                    for (int c = 0; c < NC; ++c) wf[c][i] = pack_bf16x2(v0[c], v1[c]);
                }
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    const bf16x8_t xf =
                        __builtin_bit_cast(bf16x8_t, *(const u32x4_t*)(lds + (xrd ^ (64 * j)) + i * 2048));
#pragma unroll
                    for (int c = 0; c < NC; ++c)
                        acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(bf16x8_t, u32x4_t{wf[c][0], wf[c][1], wf[c][2], wf[c][3]}), xf,
                            acc[i][c], 0, 0, 0);
                }
            }
        }
    }

    // D element (row 4 lg + e, column lr) of MFMA c: column NC (4 lg + e) + c of
    // row lr.  TP row tiles a pass: the waves' tiles, their sums into the
    // block's tile [16 TP][CT], then its 16x16 pieces.
    constexpr int OR = mid_n_out_row(NC);
    float* out = (float*)(lds + nw * WB);
#pragma unroll
    for (int p = 0; p < TM; p += TP) {
        if (p) __syncthreads();
#pragma unroll
        for (int i = 0; i < TP; ++i)
#pragma unroll
            for (int c = 0; c < NC; ++c) *(f32x4_t*)(xs + ((i * NC + c) * 64 + lane) * 16) = acc[p + i][c];
        __syncthreads();
        for (int t = wave; t < NC * TP; t += nw) {
            const uint8_t* q = lds + (t * 64 + lane) * 16;
            f32x4_t v = *(const f32x4_t*)q;
            for (int w = 1; w < nw; ++w) {
                const f32x4_t u = *(const f32x4_t*)(q + w * WB);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] += u[e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
                out[(16 * (t / NC) + lr) * OR + NC * (4 * lg + e) + t % NC] = v[e];
        }
        __syncthreads();
        for (int t = wave; t < NC * TP; t += nw) {
            const int64_t m = m0 + 16 * (p + t / NC), n = c0 + 16 * (t % NC);
            if (m >= a.M || n >= a.K) continue;
            f32x4_t v = *(const f32x4_t*)(out + (16 * (t / NC) + lr) * OR + 16 * (t % NC) + 4 * lg);
            if (a.lora.z) v = add_lora(a.lora, v, a.M, a.K, m, n, lane);
            store_out4(a, m + lr, n + 4 * lg, a.K, v);
        }
    }
}

}  // namespace

namespace rq {

#define RQ_CAT2(a, b) a##b
#define RQ_CAT(a, b) RQ_CAT2(a, b)

template <bool SB32, bool XF, int TM, int TN, int MAXW>
static hipError_t launch_mid_t(MidArgs& a, const MidTile& plan, hipStream_t stream) {
    a.tiles_m = (int)((a.M + 16 * TM - 1) / (16 * TM));
    a.tiles_n = (int)((a.R + 16 * TN - 1) / (16 * TN));
    const int64_t tiles = (int64_t)a.tiles_m * a.tiles_n;
    const int nspan = (int)((a.K + 127) / 128);
    // about `waves` waves a CU, at least 4 a block ([16384, 4096] at M = 128, two
    // 4x4 blocks a CU: 38 us with 4 waves, 42 with 8; [8192, 2048] at M = 200
    // 21 against 25)
    const int64_t ptiles = ((a.M + 16 * plan.tm - 1) / (16 * plan.tm)) *
                           ((a.R + 16 * plan.tn - 1) / (16 * plan.tn));
    const int q = (int)((ptiles + 255) / 256);
    const int maxw = plan.waves / q > 4 ? plan.waves / q : 4;
    a.spw = (nspan + maxw - 1) / maxw;
    const int nw = (nspan + a.spw - 1) / a.spw;
    // activations in flight: two halves of a span where the registers allow
    constexpr int XD = !XF && TN == 1 ? 2 : 1;
    hipLaunchKernelGGL((qmm_t_mid<RQ_BITS, SB32, XF, TM, TN, MAXW, XD>),
                       dim3((unsigned)(((tiles + 7) / 8) * 8)), dim3(64 * nw),
                       nw * mid_wave_bytes(TM, TN), stream, a);
    return hipGetLastError();
}

template <bool SB32, bool XF>
static hipError_t launch_mid_t_tile(MidArgs& a, int tile, hipStream_t stream) {
    const MidTile& t = kMidTiles[tile];
    switch (tile) {
        case 0: return launch_mid_t<SB32, XF, 1, 1, 16>(a, t, stream);
        case 1: return launch_mid_t<SB32, XF, 2, 1, 16>(a, t, stream);
        case 2: return launch_mid_t<SB32, XF, 3, 1, 16>(a, t, stream);
        case 3: return launch_mid_t<SB32, XF, 2, 2, 16>(a, t, stream);
        case 4: return launch_mid_t<SB32, XF, 4, 2, 8>(a, t, stream);
        // 128 rows of fp32 activations in flight would spill: the same slices of
        // the contraction (so the same sums as bf16(x)) on two 64-row tiles
        case 5: return launch_mid_t<SB32, XF, XF ? 4 : 8, 2, 8>(a, t, stream);
        case 6: return launch_mid_t<SB32, XF, 3, 4, 8>(a, t, stream);
        default: return launch_mid_t<SB32, XF, 4, 4, 8>(a, t, stream);
    }
}

static MidArgs mid_args(const void* x, int x_dt, const uint32_t* wq, const void* scales,
                        const void* biases, int sb_dt, int64_t m, int64_t rows, int64_t cols, int gs,
                        void* y, int y_dt, int64_t n_out, const LoraArgs* lora) {
    MidArgs a{};
    a.x = (const uint8_t*)x;
    a.wq = wq;
    a.scales = scales;
    a.biases = biases;
    a.y = y;
    a.M = m;
    a.R = rows;
    a.K = cols;
    a.gs_shift = __builtin_ctz(gs);
    a.sb_f16 = sb_dt == RQ_F16;
    a.x_f16 = x_dt == RQ_F16;
    a.y_dt = y_dt;
    const int ysz = y_dt == RQ_F32 ? 16 : 8;  // four outputs
    a.y_vec = ((uintptr_t)y & (ysz - 1)) == 0 && n_out % 4 == 0;
    if (lora) a.lora = *lora;
    return a;
}

hipError_t RQ_CAT(launch_qmm_t_mid_b, RQ_BITS)(const void* x, int x_dt, const uint32_t* wq,
                                          const void* scales, const void* biases, int sb_dt,
                                          int64_t m, int64_t rows, int64_t cols, int gs, void* y,
                                          int y_dt, hipStream_t stream, const LoraArgs* lora) {
    MidArgs a = mid_args(x, x_dt, wq, scales, biases, sb_dt, m, rows, cols, gs, y, y_dt, rows, lora);
    const int tile = mid_pick(m, rows, cols, RQ_BITS);
    if (sb_dt == RQ_F32)
        return x_dt == RQ_F32 ? launch_mid_t_tile<true, true>(a, tile, stream)
                              : launch_mid_t_tile<true, false>(a, tile, stream);
    return x_dt == RQ_F32 ? launch_mid_t_tile<false, true>(a, tile, stream)
                          : launch_mid_t_tile<false, false>(a, tile, stream);
}

// qmm_n_mid tiles: 16*tm activation rows x 16*nc columns, the time per 64 weight
// rows as above (us; [2048, 2048] against [8192, 2048]).
static constexpr MidTile kMidNTiles[] = {{1, 4, 16, 0.22}, {2, 4, 8, 0.282}, {3, 4, 8, 0.29},
                                         {4, 4, 8, 0.322}, {2, 8, 8, 0.322}};

static int mid_n_pick(int64_t m, int64_t n_out, int64_t r) {
    int best = 0;
    double bt = 1e30;
    for (int i = 0; i < (int)(sizeof(kMidNTiles) / sizeof(kMidNTiles[0])); ++i) {
        const MidTile& t = kMidNTiles[i];
        const int64_t blocks = ((m + 16 * t.tm - 1) / (16 * t.tm)) * ((n_out + 16 * t.tn - 1) / (16 * t.tn));
        const double c = 3.0 + 0.12 * t.tm * t.tn +
                         (double)((blocks + 255) / 256) * (double)((r + 63) / 64) * t.span_us;
        if (c < bt) {
            bt = c;
            best = i;
        }
    }
    return best;
}

template <bool SB32, bool XF, int TM, int NC, int MAXW>
static hipError_t launch_mid_n(MidArgs& a, hipStream_t stream) {
    a.tiles_m = (int)((a.M + 16 * TM - 1) / (16 * TM));
    a.tiles_n = (int)((a.K + 16 * NC - 1) / (16 * NC));
    const int64_t tiles = (int64_t)a.tiles_m * a.tiles_n;
    const int nhalf = (int)((a.R + 63) / 64);
    const int q = (int)((tiles + 255) / 256);
    const int maxw = MAXW / q > 4 ? MAXW / q : 4;
    a.spw = (nhalf + maxw - 1) / maxw;
    const int nw = (nhalf + a.spw - 1) / a.spw;
    hipLaunchKernelGGL((qmm_n_mid<RQ_BITS, SB32, XF, TM, NC, MAXW>),
                       dim3((unsigned)(((tiles + 7) / 8) * 8)), dim3(64 * nw),
                       nw * mid_n_wave_bytes(TM, NC) + mid_n_out_bytes(TM, NC), stream, a);
    return hipGetLastError();
}

template <bool SB32, bool XF>
static hipError_t launch_mid_n_tile(MidArgs& a, int tile, hipStream_t stream) {
    switch (tile) {
        case 0: return launch_mid_n<SB32, XF, 1, 4, 16>(a, stream);
        case 1: return launch_mid_n<SB32, XF, 2, 4, 8>(a, stream);
        case 2: return launch_mid_n<SB32, XF, 3, 4, 8>(a, stream);
        case 3: return launch_mid_n<SB32, XF, 4, 4, 8>(a, stream);
        default: return launch_mid_n<SB32, XF, 2, 8, 8>(a, stream);
    }
}

hipError_t RQ_CAT(launch_qmm_n_mid_b, RQ_BITS)(const void* x, int x_dt, const uint32_t* wq,
                                          const void* scales, const void* biases, int sb_dt,
                                          int64_t m, int64_t rows, int64_t cols, int gs, void* y,
                                          int y_dt, hipStream_t stream, const LoraArgs* lora) {
    MidArgs a = mid_args(x, x_dt, wq, scales, biases, sb_dt, m, rows, cols, gs, y, y_dt, cols, lora);
    const int tile = mid_n_pick(m, cols, rows);
    if (sb_dt == RQ_F32)
        return x_dt == RQ_F32 ? launch_mid_n_tile<true, true>(a, tile, stream)
                              : launch_mid_n_tile<true, false>(a, tile, stream);
    return x_dt == RQ_F32 ? launch_mid_n_tile<false, true>(a, tile, stream)
                          : launch_mid_n_tile<false, false>(a, tile, stream);
}

// One launch of qmv_mid over n problems that share cols (n <= RQ_MAX_GROUPED); m
// counts MFMA activation rows (twice the problems' with xsplit).
hipError_t RQ_CAT(launch_qmv_mid_b, RQ_BITS)(const rq_problem* const* problems, int n, int x_dt,
                                        int sb_dt, int y_dt, int64_t m, int gs, bool xsplit,
                                        hipStream_t stream) {
    QmvMidArgs a{};
    int64_t blocks = 0;
    for (int i = 0; i < n; ++i) {
        a.p[i] = *problems[i];
        a.block_start[i] = (int)blocks;
        blocks += (problems[i]->rows + 15) / 16;
    }
    a.block_start[n] = (int)blocks;
    if (blocks == 0) return hipSuccess;
    a.n = n;
    a.m = (int)m;
    a.sb_f16 = sb_dt == RQ_F16;
    a.x_f16 = x_dt == RQ_F16;
    a.y_dt = y_dt;
    a.xsplit = xsplit;
    const int nspan = (int)((problems[0]->cols + 127) / 128);
    const int q = (int)((blocks + 255) / 256), maxw = 16 / q > 4 ? 16 / q : 4;
    a.spw = (nspan + maxw - 1) / maxw;
    const int nw = (nspan + a.spw - 1) / a.spw;
#define RQ_QMV_MID_G(SB, XFV, GSHV)                                                              \
    hipLaunchKernelGGL((qmv_mid<RQ_BITS, SB, XFV, GSHV>), dim3((unsigned)blocks), dim3(64 * nw),  \
                       nw * 2048, stream, a)
#define RQ_QMV_MID_X(SB, XFV)                          \
    switch (gs) {                                      \
        case 32: RQ_QMV_MID_G(SB, XFV, 5); break;      \
        case 64: RQ_QMV_MID_G(SB, XFV, 6); break;      \
        default: RQ_QMV_MID_G(SB, XFV, 7); break;      \
    }
#define RQ_QMV_MID(SB) \
    if (x_dt == RQ_F32) { RQ_QMV_MID_X(SB, true) } else { RQ_QMV_MID_X(SB, false) }
    if (sb_dt == RQ_F32) { RQ_QMV_MID(true) } else { RQ_QMV_MID(false) }
#undef RQ_QMV_MID
#undef RQ_QMV_MID_X
#undef RQ_QMV_MID_G
    return hipGetLastError();
}

}  // namespace rq
