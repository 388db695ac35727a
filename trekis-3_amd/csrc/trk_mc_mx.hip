// trk_mc_mx.hip -- the event code of trk_events.inc compiled as the mixed-precision path (FP32 sampling, FP64 state, ledger and tallies): transport of single runs.
#include "trk_mc.h"

namespace trk {
namespace mx {
#define TRK_MX 1
#define TRK_PART TRK_PART_RUN
#include "trk_events.inc"
#undef TRK_MX
#undef TRK_PART

template __global__ void k_transport<true, false>(McDev din);
template __global__ void k_transport<false, false>(McDev din);
}  // namespace mx
}  // namespace trk
