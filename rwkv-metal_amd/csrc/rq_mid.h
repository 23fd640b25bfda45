// rq_mid.h -- which tile the short-batch GEMMs (rq_mid.hip) take and what it
// costs, for the launchers that choose between them and the large tiles.
#pragma once

#include <stdint.h>

namespace rq {

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

// Estimated us of the 64-wide-stage GEMM (qmm_t_k64) on its own tile choice
// (m >= 256): per 64-wide stage 0.43 us of a 64 x 96 tile, 0.7 (4 bits, 160
// columns) or 0.5 of a 128-row one, 1.0 of a 256-row one.
inline double k64_us(int64_t m, int64_t rows, int64_t cols, int bits) {
    const int64_t bn = bits == 4 && rows % 160 == 0 ? 160 : 128;
    const int64_t tn = (rows + bn - 1) / bn, t256 = ((m + 255) / 256) * tn, t128 = ((m + 127) / 128) * tn;
    int64_t tiles = t256;
    double stage = 1.0;
    if (t256 < 200) {
        tiles = t128;
        stage = bn == 160 ? 0.7 : 0.5;
        if (bits == 4 && t128 < 128) {
            tiles = ((m + 63) / 64) * ((rows + 95) / 96);
            stage = 0.43;
        }
    }
    return 2.8 + (double)((tiles + 255) / 256) * (double)(cols / 64) * stage;
}

// Estimated us of the 32-wide-stage GEMMs that take what qmm_t_k64 does not:
// 256-row tiles, 1.05 us per stage (qmm_t_ws), 2.0 with fp32 activations
// (qmm_t_big).
inline double wide_us(int64_t m, int64_t rows, int64_t cols, bool x32) {
    const int64_t bn = rows % 160 == 0 ? 160 : 128;
    const int64_t tiles = ((m + 255) / 256) * ((rows + bn - 1) / bn);
    return 3.0 + (double)((tiles + 255) / 256) * (double)((cols + 31) / 32) * (x32 ? 2.0 : 1.05);
}

}  // namespace rq
