// The matrix-core attention kernels of head dim 224.
#include "attn_mfma_kernel.h"

namespace bc {
template bool mfma_launch<224>(int, int, const AttnArgs&, dim3, hipStream_t, int);
template int mfma_occupancy<224>(int, int);
}  // namespace bc
