// lp_hash.h -- the per-frame hash table of the voxel and noise-cell stages.
#pragma once

#include "lp_internal.h"

namespace lp {

constexpr int kResetTiles = 16;  // workgroups per frame that a launch adds to clear the table

// Slots a stage occupied (slots[0 .. fs[count_slot])) back to their clean
// state, key -1 (free), count 0, aux kHashMinClean, by the threads t0, t0 +
// stride, ...; the whole table when the list is incomplete.
__device__ __forceinline__ void reset_slots(const DevBuf& d, const Layout& L, int f, const int32_t* slots,
                                            int count_slot, int t0, int stride) {
    const uint32_t cnt = d.fs[f * kFsCount + count_slot];
    const size_t ho = (size_t)f * L.hash_cap;
    if (cnt > static_cast<uint32_t>(L.N)) {
        for (int h = t0; h < L.hash_cap; h += stride) d.hslot[ho + h] = HashSlot{-1, 0u, 0, kHashMinClean};
        return;
    }
    for (int v = t0; v < static_cast<int>(cnt); v += stride) {
        const int32_t h = slots[(size_t)f * L.N + v];
        d.hslot[ho + h] = HashSlot{-1, 0u, 0, kHashMinClean};
    }
}

}  // namespace lp
