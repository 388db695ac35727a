// trk_mc_fp64.hip -- the event code of trk_events.inc compiled as the deterministic FP64 path (replays the oracle bit for bit): transport of single runs.
#include "trk_mc.h"

namespace trk {
namespace fp64 {
#define TRK_MX 0
#define TRK_PART TRK_PART_RUN
#include "trk_events.inc"
#undef TRK_MX
#undef TRK_PART

template __global__ void k_transport<true, false>(McDev din);
template __global__ void k_transport<false, false>(McDev din);
}  // namespace fp64
}  // namespace trk
