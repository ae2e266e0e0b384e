// Instantiations of the level-0 gradient pass dU_t = G_t H_{t-1}^T (CM_GRADU).
//
// Bound by HBM: U, V and G in, dU out.  R = 16, C = 48, L = 32768: 42 us (268 MB,
// 6.4 TB/s); before, the recomputed H was written by an OUTPUT pass (36 us) and
// read back by a kernel of one work-group per step (90 us): forward and backward
// of the scan 335 -> 257 us.
#include "dense_kernel.h"

namespace mogt {
template int dense_launch_gradu<float>(const ChunkParams&, int64_t, hipStream_t);
template int dense_launch_gradu<bf16_t>(const ChunkParams&, int64_t, hipStream_t);
}  // namespace mogt
