// rq_store.h -- coalesced stores of dequantized 32-code runs.
#pragma once

#include "rq_common.h"

namespace {

template <int ODT>
constexpr int kRunChunks = ODT == RQ_F32 ? 8 : 4;  // 16-byte chunks of a run's 32 outputs

// Store a wave's 64 runs of 32 outputs (lane's run t lands at t * 32 of out, t
// consecutive over the lanes, runs at and past `total` dropped), rounded to
// ODT.  The wave's 2048 consecutive outputs are staged through `line` (64 *
// (kRunChunks + 1) chunks of LDS, its own) so that each store instruction
// writes 1 KB contiguous; stored straight from registers, the 16-byte stores
// of a lane sit 64 or 128 B apart, one request per lane and instruction.
// Lane L's chunk i sits at LDS chunk L * (kRunChunks + 1) + i (the pad spreads
// the banks).  Every lane of the wave calls it.
template <int ODT>
RQ_DEV void store_runs(const float* vals, uint4* line, int64_t t, int64_t total, void* out) {
    constexpr int NC = kRunChunks<ODT>;
    const int lane = threadIdx.x & 63;
    if constexpr (ODT == RQ_F32) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            line[lane * (NC + 1) + i] =
                make_uint4(__float_as_uint(vals[4 * i]), __float_as_uint(vals[4 * i + 1]),
                           __float_as_uint(vals[4 * i + 2]), __float_as_uint(vals[4 * i + 3]));
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t d[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float lo = vals[8 * i + 2 * j], hi = vals[8 * i + 2 * j + 1];
                d[j] = ODT == RQ_BF16 ? pack_bf16x2(lo, hi) : (f32_to_f16_bits(lo) | (f32_to_f16_bits(hi) << 16));
            }
            line[lane * (NC + 1) + i] = make_uint4(d[0], d[1], d[2], d[3]);
        }
    }
    __builtin_amdgcn_wave_barrier();  // LDS runs in order within the wave
    const int64_t t0 = t - lane;      // the wave's first run
    uint4* dst = (uint4*)((uint8_t*)out + t0 * (32 * (ODT == RQ_F32 ? 4 : 2)));
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        const int c = lane + 64 * i;  // chunk c of the wave's output: lane c / NC, its chunk c % NC
        const uint4 v = line[(c / NC) * (NC + 1) + c % NC];
        if (t0 + c / NC < total) dst[c] = v;
    }
}

}  // namespace
