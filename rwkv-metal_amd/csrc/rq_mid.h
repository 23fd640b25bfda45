// rq_mid.h -- which tile the short-batch GEMMs (rq_mid.hip) take and what it
// costs, and the choice between them, the large tiles and a split contraction.
#pragma once

#include <stdint.h>

#include "../../include/rwkvq.h"

namespace rq {

// qmm_t_k64's tiles: 128 rows below this many of 256, 64 below this many of 128
constexpr int kK64Bm128Below = 200, kK64Bm64Below = 128;

// 16*tm activation rows x 16*tn weight rows, `waves` at most, and the measured
// time per 128-wide span of a CU that runs one block of it (us; 4-bit codes,
// bf16 activations, [2048, 2048] against [2048, 8192]).  A wave dequantizes tn
// weight tiles and stages tm activation tiles per span, so wide tiles do less
// per output, and small ones fill the chip.
struct MidTile {
    int tm, tn, waves;
    double span_us;
};
constexpr MidTile kMidTiles[] = {{1, 1, 16, 0.123}, {2, 1, 16, 0.177}, {3, 1, 16, 0.204}, {2, 2, 16, 0.233},
                                 {4, 2, 8, 0.305},  {8, 2, 8, 0.475},  {3, 4, 8, 0.43},  {4, 4, 8, 0.479}};
constexpr int kMidTileCount = sizeof(kMidTiles) / sizeof(kMidTiles[0]);

// What dequantizing one 16-row weight tile's span costs beyond 4-bit codes
// (measured at 3, 5 and 8 bits).
inline double mid_bits_us(int bits) {
    return bits == 4 ? 0.0 : (bits == 8 ? 0.027 : (bits >= 5 ? 0.108 : 0.06));
}

// The tile with the least rounds x spans x time per span, plus the launch and
// the sum over the waves (3 + 0.2 us per 16x16 tile of the block).
inline int mid_pick(int64_t m, int64_t n_out, int64_t k, int bits, double* us = nullptr) {
    int best = 0;
    double bt = 1e30;
    for (int i = 0; i < kMidTileCount; ++i) {
        const MidTile& t = kMidTiles[i];
        const int64_t blocks = ((m + 16 * t.tm - 1) / (16 * t.tm)) * ((n_out + 16 * t.tn - 1) / (16 * t.tn));
        const double c = 3.0 + 0.2 * t.tm * t.tn +
                         (double)((blocks + 255) / 256) * (double)((k + 127) / 128) *
                             (t.span_us + mid_bits_us(bits) * t.tn);
        if (c < bt) {
            bt = c;
            best = i;
        }
    }
    if (us) *us = bt;
    return best;
}

// Fewer than 256 rows: the short-batch tiles with their output, and qmm_t_kernel's
// 128 x 128 tiles, two blocks a CU (us per 64 columns of a round of 512 tiles, and
// of 256 or fewer).  Over 7 weight shapes of 10240 to 65536 rows, 8 row counts, all
// six bit widths, bf16 and fp32 x, the form with the lower estimate is the faster
// one or within 6 % in 670 of 674, and within 11 % in the others.  One choice for
// both types of x: fp32 x gives the bits of bf16(x).
inline double mid_short_us(int64_t m, int64_t rows, int64_t cols, int bits) {
    double us;
    mid_pick(m, rows, cols, bits, &us);
    // fp32 x costs them more than the large tiles at 5 and 6 bits, where bf16 x is even
    return (bits == 5 || bits == 6 ? 1.05 : 1.0) * (us + 2.4e-6 * (double)(m * rows));
}
inline double t128_us(int64_t m, int64_t rows, int64_t cols, int bits) {
    const int64_t tiles = ((m + 127) / 128) * ((rows + 127) / 128), rest = tiles % 512;
    const bool odd = bits != 4 && bits != 8;
    const double two = bits == 4 ? 2.0 : (bits == 8 ? 2.4 : (bits < 4 ? 1.9 : 2.43));
    const double one = bits == 4 ? 1.63 : (bits == 8 ? 1.88 : (bits < 4 ? 1.39 : 1.73));
    const double round = (double)(tiles / 512) * two + (rest == 0 ? 0.0 : (rest <= 256 ? one : two));
    return (odd ? 10.0 : 1.5) + round * (double)((cols + 63) / 64) + 1.25e-6 * (double)(m * rows);
}

// Estimates of the forward GEMMs where the 64-wide stages apply (m >= 256; us, one
// MI355X), from both forms and the short-batch tiles timed over 17 weight
// shapes of 0.8 M to 38 M elements at 13 row counts of 256 to 3072 and 3, 4, 6
// and 8 bits: the plain ones are met within 2 % on average, the split ones
// within 3 %.
struct K64Tile {
    int bm, bn;
};

// qmm_t_k64's tile for a whole contraction.
inline K64Tile k64_tile(int64_t m, int64_t rows, int bits) {
    // 160-row tiles (whole rounds over 256 CUs for the 2560-wide RWKV-7 shapes) split
    // evenly into 8-code dequant jobs only at 4 bits
    const int bn = bits == 4 && rows % 160 == 0 ? 160 : 128;
    const int64_t tn = (rows + bn - 1) / bn;
    if (((m + 255) / 256) * tn >= kK64Bm128Below) return {256, bn};
    // 128-row tiles when 256-row ones leave most CUs idle (small M, narrow R), and at
    // 4 bits 64 x 96 tiles when 128-row ones still leave half of them idle
    // (M = 512 with 2560 outputs: 216 tiles instead of 64)
    if (bits == 4 && ((m + 127) / 128) * tn < kK64Bm64Below) return {64, 96};
    return {128, bn};
}

// us per 64-wide stage of a tile
inline double k64_stage_us(K64Tile t, int bits) {
    if (t.bm == 64) return 0.335;
    if (t.bn == 160) return t.bm == 128 ? 0.70 : 1.02;
    const bool small = t.bm == 128;
    if (bits == 4) return small ? 0.54 : 0.88;
    if (bits == 8) return small ? 0.59 : 0.92;
    return bits < 4 ? (small ? 0.77 : 0.95) : (small ? 0.87 : 1.01);
}

// Launch (4.6 us on 64-row tiles, 3.6 on others, 6.5 with the reduction; 11.5 more
// on 256-row tiles at the widths other than 4 and 8 bits), rounds over 256 CUs x
// stages, and the output: one store, or `splits` fp32 partial tiles written and
// read back by the reduction.
inline double k64_us(int64_t m, int64_t rows, int64_t cols, int gs, int bits, K64Tile t, int64_t splits) {
    const int64_t tiles = ((m + t.bm - 1) / t.bm) * ((rows + t.bn - 1) / t.bn) * splits;
    const int64_t nper = cols / (8 * (int64_t)gs);  // a split is of whole 8-group periods
    const int64_t stages = ((nper + splits - 1) / splits) * (gs / 8);
    const double mouts = 1e-6 * (double)(m * rows);
    double us = splits == 1 ? (t.bm == 64 ? 4.6 : 3.6) + 0.8 * mouts : 6.5 + 1.6 * (double)splits * mouts;
    if (t.bm == 256 && bits != 4 && bits != 8) us += 11.5;
    // measured 6 % longer on the smaller tiles of a split
    const double stage = k64_stage_us(t, bits) * (splits > 1 && t.bm == 128 ? 1.06 : 1.0);
    return us + (double)((tiles + 255) / 256) * (double)stages * stage;
}

// The short-batch tiles at 256 rows and more: beside mid_pick's estimate the
// output and what the tiles re-read from L2.
inline double mid_us(int64_t m, int64_t rows, int64_t cols, int bits) {
    double us;
    mid_pick(m, rows, cols, bits, &us);
    const double mouts = 1e-6 * (double)(m * rows);
    if (bits < 4) us *= 1.08;  // measured at 3 bits
    return us * (1.0 + 4e-6 * mouts * (double)cols) + 0.9 * mouts;
}

// The form with the least estimate.  Timed over those shapes at 2 to 5 bits it is
// 6.8 % faster on average than the plain and split forms alone ([1024, 4096] at
// M = 512, 4 bits, 17.3 -> 14.6 us, [768, 3072] 14.9 -> 11.9); the largest loss is
// [1536, 1536] at M = 512, 4 bits, 13.0 -> 13.9.  One estimator for all three:
// with another for the split, [3072, 3072] at M = 640 left its split (26 us) for
// short-batch tiles (30) and [12288, 3072] its large tiles (93) for them (106).
struct GemmPlan {
    bool mid = false;
    int bm = 0, splits = 1;  // > 1: qmm_t_k64 on bm-row tiles into partial tiles
};
inline GemmPlan gemm_plan(int64_t m, int64_t rows, int64_t cols, int gs, int bits, bool may_split) {
    GemmPlan p;
    const K64Tile t = k64_tile(m, rows, bits);
    double best = k64_us(m, rows, cols, gs, bits, t, 1);
    p.bm = t.bm;
    const int bn = bits == 4 && rows % 160 == 0 ? 160 : 128;
    const int64_t nper = cols / (8 * (int64_t)gs);
    for (int bm = 256; may_split && bm >= 128; bm /= 2) {
        const int64_t tiles = ((m + bm - 1) / bm) * ((rows + bn - 1) / bn);
        for (int64_t s = 2; s <= nper && s <= 32 && tiles * s <= 1024; ++s) {
            const double us = 1.02 * k64_us(m, rows, cols, gs, bits, {bm, bn}, s);  // not for a tie
            if (us < best) {
                best = us;
                p.bm = bm;
                p.splits = (int)s;
            }
        }
    }
    if (mid_us(m, rows, cols, bits) < best) {
        p.mid = true;
        p.splits = 1;
    }
    return p;
}

// 256 rows and more where the 64-wide stages do not apply (fp32 scales, groups that
// are no multiple of 8, f16 x): the 32-wide-stage GEMMs, 256-row tiles
// (qmm_t_ws, and with fp32 or f16 x qmm_t_big), against the short-batch tiles, whose
// fp32 rows are read again from L2 by every weight tile.  Both timed alone over 25
// weight shapes of 0.5 M to 67 M elements, M = 256 to 4096, 4, 5, 6 and 8 bits: of 924
// products 30 lose more than 5 % to the other form, most of them fp32 x at M = 4096.
inline double wide_us(int64_t m, int64_t rows, int64_t cols, int bits, bool x16) {
    const bool w160 = rows % 160 == 0;
    const int64_t bn = w160 ? 160 : 128;
    const int64_t tiles = ((m + 255) / 256) * ((rows + bn - 1) / bn);
    const double stages = (double)((tiles + 255) / 256) * (double)((cols + 31) / 32);
    const double mouts = 1e-6 * (double)(m * rows);
    if (!x16) return stages * (w160 ? 2.75 : 2.1) + 2.5 * mouts;
    const double stage = bits == 4 || bits == 8 ? (w160 ? 0.62 : 0.53) : (w160 ? 1.27 : 1.05);
    return 13.0 + stages * stage + 1.5 * mouts;
}
inline double mid_wide_us(int64_t m, int64_t rows, int64_t cols, int bits, bool x32) {
    double us;
    mid_pick(m, rows, cols, bits, &us);
    const double mouts = 1e-6 * (double)(m * rows);
    return us * (1.0 + (x32 ? 55e-6 : 7e-6) * mouts * (double)cols) + (x32 ? 4.8 : 2.2) * mouts;
}

// The short-batch GEMMs take weights of up to this many rows and columns (offsets
// inside a tile are 32-bit).
constexpr int64_t kMidMaxCols = 1 << 26;

// The decode GEMVs; m counts MFMA rows (two for each of fp32 or f16 x at one or two).

// Whether qmv_mid takes a small launch of more than 4 rows from the split GEMV,
// which makes two passes: few blocks of short rows, and at 7 and 8 rows (at 4 bits
// from 5, where long enough) more than two blocks a CU; slower between.  Split /
// qmv_mid in us: m = 8, 4 bits, [768, 768] 5.5 / 4.1, [2560, 2560] 7.5 / 6.6, [10240,
// 2560] 14.3 / 11.2, [8192, 2048] 8.1 / 8.3; m = 5 [16384, 768] 7.0 / 7.5, and at 6
// bits [2048, 2048] 7.4 / 8.3, at 2 [16384, 4096] 19.0 / 22.3.
inline bool qmv_mid_over_split(int x_dt, int64_t m, int64_t cols, int bits, int64_t rowblocks) {
    if (m <= 4) return false;
    if (m >= 7)
        return (rowblocks <= 192 && cols <= 4096) ||
               (rowblocks > 512 && !(bits == 5 && x_dt == RQ_F32));  // [10240, 2560] 17.4 / 20.0
    if (bits == 4) return (rowblocks <= 192 && cols <= 4096) || (rowblocks > 512 && cols >= 2048);
    return rowblocks <= 192 && cols < 2048;
}

// Whether qmv_mid takes a large launch (2048 blocks of 16 rows and more) that the
// streamed GEMVs do not cover from qmv_kernel.  Above 8 rows always ([65536, 768] at m
// = 12, 4 bits, 26 -> 17.6 us).  Below, qmv_kernel / qmv_mid in us:
//  * 16-bit scales: 3, 5 and 6 bits at 8 rows ([65536, 2048], 3 bits, 55.6 / 51.2) and
//    in rows of no whole 512 codes ([65536, 768], 6 bits, 35.9 / 30.0; 3 bits at m = 1
//    17.7 / 18.9); at 2 bits from 5 fp32 rows ([65536, 768], m = 8, 23.2 / 18.5, bf16
//    14.4 / 17.2).
//  * fp32 scales: 3, 5 and 6 bits but for up to 4 long rows in groups of 64 and more
//    ([65536, 2048], m = 1, 3 bits, group size 64, 42.1 / 50.0, 32 51 / 37); the other
//    widths in groups of 32 but for one or two short bf16 rows (4 bits, [65536, 2048],
//    m = 1 27.7 / 37.9, m = 8 57 / 40), in groups of 64 from 5 rows where x is fp32 or
//    long (m = 8, [49152, 3072] 47 / 43; m = 1 26.9 / 41.0, [65536, 768] 10.1 / 16.6).
inline bool qmv_large_takes_mid(int x_dt, int sb_dt, int64_t m, int64_t cols, int gs, int bits) {
    if (m > 8) return true;
    const bool odd = bits == 3 || bits == 5 || bits == 6;
    if (sb_dt != RQ_F32) {
        if (bits == 2) return x_dt == RQ_F32 && m >= 5 && (m == 8 || cols % 512 != 0);
        return odd && (m == 8 || (cols % 512 != 0 && !(bits == 3 && m == 1)));
    }
    if (odd) return gs == 32 || cols < 2048 || m > 4;
    if (gs == 32) return x_dt != RQ_BF16 || m > (bits == 8 ? 1 : 2) || cols > 2048;
    if (m <= 4) return bits == 8 && m >= 3 && cols < 2048;
    return x_dt == RQ_F32 || cols > 2048;
}

// Whether a small launch that the split GEMV does not take (fp32 scales, group counts
// that rule out whole-line loads) runs qmv_kernel with its waves splitting K, rather
// than qmv_mid: bf16 x of up to 3 rows, where qmv_mid's 16-row MFMA tile is mostly
// padding and its per-wave staging costs more than the weights.  fp32 scales, one
// row, qmv_kernel / qmv_mid in us: 4 bits, group size 64, [2048, 2048] 4.3 / 5.1, [8192,
// 2048] 6.3 / 8.7, [16384, 4096] 14.1 / 23.0 (3 rows 17.5 / 23.5, 4 rows 28.6 / 22.8); 8
// bits [16384, 4096] 19.9 / 27.5, [16384, 1024] 9.5 / 9.1; 3 bits [16384, 4096] 22.5 /
// 27.1, [10240, 2560] 14.9 / 13.5; group size 32, 4 bits, [8192, 2048] 7.2 / 8.2, [4096,
// 4096] 8.9 / 8.3.  5 and 6 bits never, nor fp32 x, which qmv_kernel converts again
// in every block, nor rows too long for its LDS ([2560, 10240], 3 rows, 17.8 / 12.8).
inline bool qmv_splits_k(int x_dt, int64_t m, int64_t cols, int gs, int bits, int64_t rowblocks) {
    // one long 8-bit form: [2560, 10240], bf16 scales, 2 rows, 13.7 / 15.8
    if (x_dt == RQ_BF16 && bits == 8 && m == 2 && gs >= 64 && cols >= 8192 && cols <= 10240)
        return rowblocks >= 128;
    if (x_dt != RQ_BF16 || m > 3 || bits == 5 || bits == 6 || m * cols > 12288) return false;
    if (gs == 32) return m <= 2 && rowblocks >= (bits == 2 || bits == 4 ? 512 : 1024);
    if (bits == 3) return m <= 2 && rowblocks >= 768 && cols >= 2048;
    if (bits == 8) return m <= 2 && rowblocks >= (m == 1 ? 128 : 256) && cols >= 1280;
    return rowblocks >= (m == 1 ? 128 : (m == 2 ? 256 : 512)) && (m < 3 || cols >= 2048);
}

// Whether a forward product runs the short-batch tiles.  k64: the 64-wide stages
// apply.  lora: with the low-rank term in its output stage, which of the others
// only the 64-wide stages can add; elsewhere it takes launches of its own, ~15 us and
// 24 bytes an output.
inline bool forward_takes_mid(int x_dt, bool k64, bool lora, int64_t m, int64_t rows, int64_t cols,
                              int gs, int bits) {
    if (cols > kMidMaxCols) return false;
    if (k64) return gemm_plan(m, rows, cols, gs, bits, /*may_split=*/false).mid;
    if (m < 256) return lora || mid_short_us(m, rows, cols, bits) <= t128_us(m, rows, cols, bits);
    const double term = lora ? 15.0 + 4.8e-6 * (double)(m * rows) : 0.0;
    return mid_wide_us(m, rows, cols, bits, x_dt == RQ_F32) <
           wide_us(m, rows, cols, bits, x_dt == RQ_BF16) + term;
}

}  // namespace rq
