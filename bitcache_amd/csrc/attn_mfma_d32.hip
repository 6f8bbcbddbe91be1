// The matrix-core attention kernels of head dim 32.
#include "attn_mfma_kernel.h"

namespace bc {
template bool mfma_launch<32>(int, int, const AttnArgs&, dim3, hipStream_t, int);
template int mfma_occupancy<32>(int, int);
}  // namespace bc
