// trk_mc_mx_general.hip -- the event code of trk_events.inc compiled as the mixed-precision path (FP32 sampling, FP64 state, ledger and tallies): the ions and the general transfers.
#include "trk_mc.h"

namespace trk {
namespace mx {
#define TRK_MX 1
#define TRK_PART TRK_PART_GENERAL
#include "trk_events.inc"
#undef TRK_MX
#undef TRK_PART

template __global__ void k_transport<true, true>(McDev din);
template __global__ void k_transport<false, true>(McDev din);
template __global__ void k_ions<true>(McDev din, int waves);
template __global__ void k_ions<false>(McDev din, int waves);
}  // namespace mx
}  // namespace trk
