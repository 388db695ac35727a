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

}  // namespace trk
