// lp_joins.h -- the neighbours of a voxel that its component search joins it with.
#pragma once

#include <stdint.h>

namespace lp {

// Half of the 26-neighbourhood (the other half is covered from the
// neighbour's side): offsets (dr, da, de) with (de, da, dr) > (0, 0, 0).
__constant__ static const int8_t kHalfNb[13][3] = {
    {1, 0, 0},  {-1, 1, 0}, {0, 1, 0},  {1, 1, 0},  {-1, -1, 1}, {0, -1, 1}, {1, -1, 1},
    {-1, 0, 1}, {0, 0, 1},  {1, 0, 1},  {-1, 1, 1}, {0, 1, 1},   {1, 1, 1}};

// Which of a voxel's forward neighbours it has to be joined with.  A voxel is
// joined with (1, 0, 0) always, so occupied cells that follow one another in
// range are one component already; of the three cells at the next azimuth one
// per such run is enough.  That joins all neighbours of one layer, so of the
// nine cells of the layer above one per group of cells that touch (in range or
// azimuth, diagonally too) is enough.  Each step leans only on the ones before
// it (never the other way round an azimuth ring), and two to three joins per
// voxel are left of up to thirteen.  Cell (da, dr) of the layer is bit
// 3 * (da + 1) + dr + 1, its centre bit 4.
struct LayerJoins {
    uint16_t of[512];
    constexpr LayerJoins() : of() {
        for (int m = 0; m < 512; ++m) {
            int left = m, joins = 0;
            while (left) {
                int first = 0;
                while (!((left >> first) & 1)) ++first;
                int group = 1 << first;
                for (bool grown = true; grown;) {
                    grown = false;
                    for (int a = 0; a < 9; ++a) {
                        if (!((left >> a) & 1) || ((group >> a) & 1)) continue;
                        for (int b = 0; b < 9; ++b) {
                            const int da = a / 3 - b / 3, dr = a % 3 - b % 3;
                            if (((group >> b) & 1) && da * da <= 1 && dr * dr <= 1) {
                                group |= 1 << a;
                                grown = true;
                                break;
                            }
                        }
                    }
                }
                joins |= (group & 16) ? 16 : 1 << first;
                left &= ~group;
            }
            of[m] = static_cast<uint16_t>(joins);
        }
    }
};
__constant__ static const LayerJoins kLayerJoins{};
constexpr int kMaxJoins = 7;  // one in range, two at the next azimuth, four in the layer above

// Bit q: join with neighbour q of kHalfNb; `found` has bit q when it is occupied.
__device__ __forceinline__ uint32_t joins_of(uint32_t found) {
    const uint32_t side = (found & 4u) ? 4u : found & 10u;
    return (found & 1u) | side | static_cast<uint32_t>(kLayerJoins.of[found >> 4]) << 4;
}

}  // namespace lp
