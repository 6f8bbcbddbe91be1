// The matrix-core attention kernels of head dim 256.
#include "attn_mfma_kernel.h"

namespace bc {
template bool mfma_launch<256>(int, int, const AttnArgs&, dim3, hipStream_t, int);
template int mfma_occupancy<256>(int, int);
}  // namespace bc
