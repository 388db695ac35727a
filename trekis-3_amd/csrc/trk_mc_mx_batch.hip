// trk_mc_mx_batch.hip -- the event code of trk_events.inc compiled as the mixed-precision path (FP32 sampling, FP64 state, ledger and tallies): batches.
#include "trk_mc.h"

namespace trk {
namespace mx {
#define TRK_MX 1
#define TRK_PART TRK_PART_BATCH
#include "trk_events.inc"
#undef TRK_MX
#undef TRK_PART

template __global__ void k_batch_ions<true>(BatchIons bi, int n_groups);
template __global__ void k_batch_ions<false>(BatchIons bi, int n_groups);
template __global__ void k_batch<true>(BatchCtl *ctl, int n_groups);
template __global__ void k_batch<false>(BatchCtl *ctl, int n_groups);
}  // namespace mx
}  // namespace trk
