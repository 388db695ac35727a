// trk_rules.h -- small rules that kernels and host code share (table indexes
// of a draw, launch shapes, budgets): functions of plain values without any
// HIP, so that a host compiler takes them too.
#pragma once

#include <stdint.h>
#include "trk_detmath.h"

namespace trk {

// The ion's energy-transfer draw RN in [b/kShiBuckets, (b+1)/kShiBuckets)
// finds its entry of a shell's inverse-path row between the entries that
// the bucket's two ends find (k_shi_buckets).
constexpr int kShiBuckets = 64;

// The bucket of a draw in (0, 1].  A draw is (u + 0.5) 2^-53, and for the
// largest u the sum rounds up: that draw is 1 and belongs to the last bucket.
TRK_FN int shi_bucket(double RN)
{
    const int b = (int)(RN * (double)kShiBuckets);
    return b < kShiBuckets ? b : kShiBuckets - 1;
}

// Waves per workgroup (one per SIMD) of a round with few particles.
constexpr int kSparseWaves = 4;

// The launch of one round's transport: workgroups, threads in each, and the
// lanes of a wave that take particles.
struct TransportShape {
    int64_t blocks;
    int threads, lane_cap;
};

// n particles on at most max_blocks resident workgroups of `full` threads.
// Few particles (the last rounds of a large run, all of a small one): as many
// waves as there are SIMDs, with as few particles each as that gives; a wave
// runs each category its particles want in turn, so a lone history goes faster
// the fewer share its wave.  From 64 particles per SIMD on, until they fill
// every resident workgroup: the waves they need spread over all of these, four
// to twelve each, rather than full workgroups on some CUs and none on others
// (37 to 100 oxide iterations pass through one or two such rounds: 2-4 % of
// the run in FP64, up to 2 % mixed).
inline TransportShape transport_shape(int64_t n, int64_t max_blocks, int full)
{
    TransportShape s;
    s.threads = full;
    s.lane_cap = 64;
    s.blocks = (n + full - 1) / full;
    if (n < 64 * kSparseWaves * max_blocks) {
        s.threads = 64 * kSparseWaves;
        s.lane_cap = (int)((n + kSparseWaves * max_blocks - 1) / (kSparseWaves * max_blocks));
        const int64_t per = (int64_t)kSparseWaves * s.lane_cap;
        s.blocks = (n + per - 1) / per;
    } else if (s.blocks < max_blocks) {
        const int64_t waves = (n + 63) / 64;
        s.threads = 64 * (int)((waves + max_blocks - 1) / max_blocks);
        s.blocks = (n + s.threads - 1) / s.threads;
    }
    if (s.blocks > max_blocks) s.blocks = max_blocks;
    return s;
}

}  // namespace trk
