// trk_mc_fp64_general.hip -- the event code of trk_events.inc compiled as the deterministic FP64 path (replays the oracle bit for bit): the ions and the general transfers.
#include "trk_mc.h"

namespace trk {
namespace fp64 {
#define TRK_MX 0
#define TRK_PART TRK_PART_GENERAL
#include "trk_events.inc"
#undef TRK_MX
#undef TRK_PART

template __global__ void k_transport<true, true>(McDev din);
template __global__ void k_transport<false, true>(McDev din);
template __global__ void k_ions<true>(McDev din, int waves);
template __global__ void k_ions<false>(McDev din, int waves);
}  // namespace fp64
}  // namespace trk
