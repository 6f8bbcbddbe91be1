// Host dispatch of the matrix-core attention kernels (attn_mfma_kernel.h): one
// translation unit per head dim (attn_mfma_d*.hip) holds that head dim's
// instances, so that they compile in parallel.
#include "attn.h"

#include <map>
#include <mutex>
#include <tuple>

namespace bc {

#define BC_MFMA_DIMS(X) X(32) X(64) X(96) X(128) X(160) X(192) X(224) X(256)

#define BC_MFMA_EXTERN(D)                                                                              \
    extern template bool mfma_launch<D>(int, int, const AttnArgs&, dim3, hipStream_t, int);            \
    extern template int mfma_occupancy<D>(int, int);
BC_MFMA_DIMS(BC_MFMA_EXTERN)

int mfma_wgs_per_cu(int mode, int D, int G) {
    static std::mutex mu;
    static std::map<std::tuple<int, int, int, int>, int> cache;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    const auto key = std::make_tuple(dev, mode, D, G);
    std::lock_guard<std::mutex> lock(mu);
    const auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    int n = 0;
    switch (D) {
#define BC_MFMA_CASE(DD) case DD: n = mfma_occupancy<DD>(mode, G); break;
        BC_MFMA_DIMS(BC_MFMA_CASE)
#undef BC_MFMA_CASE
        default: n = 0;
    }
    cache[key] = n;
    return n;
}

bool mfma_split_ok(int D, int64_t chunk, int64_t head_groups) {
    if (!head_dim_ok(D) || head_groups > kMaxHeadGroups) return false;
    // buffer offsets are 32-bit and relative to a split's key range; the
    // prefetches reach up to 17 tiles (1088 keys) past its end.  The int8
    // value path adds at most 2^16 per tile to an int32 accumulator: a wave
    // takes at most 2^15 tiles (a split below 2^23 keys)
    return (chunk + 2048) * (D / 2) + 4096 < ((int64_t)1 << 31) && chunk < ((int64_t)1 << 23);
}

bool launch_mfma_split(int mode, int D, int G, const AttnArgs& a, dim3 grid, hipStream_t st, int nw) {
    if (!mfma_split_ok(D, a.chunk, (a.Hq / a.Hkv) / G)) return false;
    // adaptive mode reads the popcounts stored by the selection passes
    if (mode == MODE_ADAPTIVE && a.pcs == nullptr) return false;
    switch (D) {
#define BC_MFMA_CASE(DD) case DD: return mfma_launch<DD>(mode, G, a, grid, st, nw);
        BC_MFMA_DIMS(BC_MFMA_CASE)
#undef BC_MFMA_CASE
        default: return false;
    }
}

}  // namespace bc
