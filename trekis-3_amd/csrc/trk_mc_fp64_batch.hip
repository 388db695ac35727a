// trk_mc_fp64_batch.hip -- the event code of trk_events.inc compiled as the deterministic FP64 path (replays the oracle bit for bit): batches.
#include "trk_mc.h"

namespace trk {
namespace fp64 {
#define TRK_MX 0
#define TRK_PART TRK_PART_BATCH
#include "trk_events.inc"
#undef TRK_MX
#undef TRK_PART

template __global__ void k_batch_ions<true>(BatchIons bi, int n_groups);
template __global__ void k_batch_ions<false>(BatchIons bi, int n_groups);
template __global__ void k_batch<true>(BatchCtl *ctl, int n_groups);
template __global__ void k_batch<false>(BatchCtl *ctl, int n_groups);
}  // namespace fp64
}  // namespace trk
