// lp_segment.hip -- polar grid, range-image winner, RECM and RANSAC on gfx950.
//
// Reference semantics (paths relative to the reference root):
//   constructPolarGrid   lidar_processing_lib/src/segmenter.cpp:103-204
//   RECM elevation map   lidar_processing_lib/src/segmenter.cpp:206-267
//   obstacle test        lidar_processing_lib/src/segmenter.cpp:269-283
//   RANSAC correction    lidar_processing_lib/src/segmenter.cpp:321-479
//   image transfer       lidar_processing_lib/src/segmenter.cpp:289-318
//
// Layout: points are CSR-packed per frame (FrameDesc::pt_off); per-frame
// arrays of cells / pixels / queue entries use fixed frame strides.  Grids
// are (tiles, frames) and sized for the batch capacity so one launch
// sequence (and one captured graph) serves every batch of a shape bucket.
#include "lp_hash.h"
#include "lp_kernels.h"
#include "lp_queue.h"

namespace lp {

using namespace lpd;

constexpr float kTwoPi = 6.28318548202514648438f;  // (float)(2*M_PI), segmenter.hpp:136
constexpr uint32_t kEmptyZ = 0x7fc00000u;           // NaN marks an empty cell

// ---------------------------------------------------------------------------
// Per-batch clear (fill kernels instead of memsets so the whole sequence can
// be captured in a graph).  The voxel hash is clean on entry (its previous
// users reset the slots they occupied).  Ahead of the noise filter it clears
// the filter's column bits and counters as well (a launch of their own took 4
// to 9 us of a 64x2048 frame); after it (the KD-tree search) the filter's
// counts stay.
__global__ void k_clear(DevBuf d, Layout L, bool noise) {
    const int f = blockIdx.y;
    const FrameDesc fd = d.frames[f];
    const int cells = fd.sc.cells;
    const int P = fd.sc.H * fd.sc.W;
    const int stride = gridDim.x * blockDim.x;
    const int t0 = blockIdx.x * blockDim.x + threadIdx.x;
    if (f == 0 && t0 < kWqCounters) d.wq[t0] = 0;
    for (int c = t0; c < cells; c += stride) d.cell_count[(size_t)f * L.cell_stride + c] = 0;
    for (int p = t0; p < P; p += stride) d.pix_key[fd.pix_off + p] = ~0ull;
    for (int k = t0; k < kRansacIters; k += stride) d.hyp_count[f * kRansacIters + k] = 0;
    if (noise)
        for (int q = t0; q < kNoiseOccWords; q += stride) d.nocc[(size_t)f * kNoiseOccWords + q] = 0;
    if (t0 < (noise ? static_cast<int>(kFsCount) : static_cast<int>(kFsKept))) d.fs[f * kFsCount + t0] = 0;
}

// ---------------------------------------------------------------------------
// One thread per point: polar cell, range-image pixel, cell histogram and the
// pixel winner.  The winner of a pixel is the first point, in (cell, input)
// order, with the smallest x*x+y*y (segmenter.cpp:291-318, strict `<`).
// Equal depth implies equal radial cell, so the order reduces to
// (depth, slice, index): packed into one 64-bit key and resolved with a
// single atomicMin.
__device__ __forceinline__ void project_tile(const DevBuf& d, const Layout& L, int f, int tile) {
    const FrameDesc& fd = d.frames[f];
    const int i = tile * blockDim.x + threadIdx.x;
    if (i >= fd.n) return;
    const SegConst& s = fd.sc;
    const int gi = fd.pt_off + i;
    const float x = d.x[gi], y = d.y[gi], z = d.z[gi];
    int cell = -1, pix = -1;
    const bool finite = isfinite(x) && isfinite(y) && isfinite(z);
    if (finite && !(z < s.zlo || z > s.zhi)) {
        const float dd = x * x + y * y;
        const float dist = sqrtf(dd);
        const int radial = static_cast<int>(dist / s.spacing);
        if (!(dist < s.min_d || dist > s.max_d || radial >= s.rings)) {
            float az = atan2_approx(y, x);
            az = (az < 0) ? (az + kTwoPi) : az;
            const int slice = min(static_cast<int>(az / s.slice_res), s.slices - 1);
            int row = -1;
            if (s.organized && fd.has_ring) {
                const int h = d.ring[gi];
                if (h < s.H) row = h;
            } else {
                const float elev = fdlibm_atanf(z / dist);
                const int hs = static_cast<int>((elev - s.down_rad) / s.per_pixel);
                if (hs >= 0 && hs < s.H) row = hs;
            }
            if (row >= 0) {
                const int col = static_cast<uint16_t>((s.w_minus_1 * az) / kTwoPi);
                cell = slice * s.rings + radial;
                pix = row * s.W + col;
                d.pt_loc[gi] = static_cast<int32_t>(wave_atomic_inc(&d.cell_count[(size_t)f * L.cell_stride + cell]));
                const unsigned long long key = (static_cast<unsigned long long>(f2u(dd)) << 32) |
                                               (static_cast<unsigned long long>(slice) << L.idx_bits) |
                                               static_cast<unsigned long long>(i);
                atomicMin(&d.pix_key[fd.pix_off + pix], key);
            }
        }
    }
    d.pt_cell[gi] = cell;
    d.pt_pix[gi] = pix;
    d.pt_xyzc[gi] = make_float4(x, y, z, __int_as_float(cell));
}

__global__ void k_project(DevBuf d, Layout L) { project_tile(d, L, blockIdx.y, blockIdx.x); }

__global__ __launch_bounds__(256) void k_project_q(DevBuf d, Layout L, int B) {
    wq_run(d.wq + kWqProject * 8, B, blockDim.x, [&](int f) { return d.frames[f].n; },
           [&](int f, int t) { project_tile(d, L, f, t); });
}

// Cell starts, the lists of non-empty cells for k_cell_sort, and the empty
// marker of every empty cell's minimum.  Where a cell's points lie does not
// matter, so each workgroup reserves room for its 2048 cells with one atomic
// per total instead of a scan over the frame by one workgroup (28 -> 6 us per
// frame).  Cells of up to kRowCell points are listed from the front of
// cell_list, larger ones from its back.
constexpr int kStartThreads = 256;
constexpr int kStartItems = 8;
constexpr uint32_t kRowCell = 16;  // points of a cell sorted by one 16-lane row

__global__ __launch_bounds__(kStartThreads) void k_cell_start(DevBuf d, Layout L) {
    __shared__ uint64_t lds[kStartThreads / kWave + 1];
    __shared__ uint32_t first[3];
    const int f = blockIdx.y;
    const int cells = d.frames[f].sc.cells;
    const int b = (blockIdx.x * kStartThreads + threadIdx.x) * kStartItems;
    if (static_cast<int>(blockIdx.x) * kStartThreads * kStartItems >= cells) return;
    const size_t co = (size_t)f * L.cell_stride;
    uint32_t v[kStartItems];
    uint64_t sum = 0;  // points in the low word, then small and large cells
#pragma unroll
    for (int k = 0; k < kStartItems; ++k) {
        v[k] = (b + k < cells) ? d.cell_count[co + b + k] : 0u;
        sum += v[k] + (v[k] ? (v[k] <= kRowCell ? 1ull << 32 : 1ull << 48) : 0ull);
    }
    uint64_t total;
    const uint64_t ex = block_exclusive_sum<kStartThreads>(sum, lds, &total);
    if (threadIdx.x < 3) {
        uint32_t* fs = d.fs + f * kFsCount;
        uint32_t* ctr = fs + (threadIdx.x == 0 ? kFsCellPoints : (threadIdx.x == 1 ? kFsCellsSmall : kFsCellsLarge));
        const uint32_t add = threadIdx.x == 0 ? static_cast<uint32_t>(total)
                                              : static_cast<uint32_t>(total >> (threadIdx.x == 1 ? 32 : 48)) & 0xffffu;
        first[threadIdx.x] = add ? atomicAdd(ctr, add) : 0u;
    }
    __syncthreads();
    uint32_t start = first[0] + static_cast<uint32_t>(ex);
    uint32_t small = first[1] + (static_cast<uint32_t>(ex >> 32) & 0xffffu);
    uint32_t large = first[2] + static_cast<uint32_t>(ex >> 48);
    uint4* list = d.cell_list + co;
#pragma unroll
    for (int k = 0; k < kStartItems; ++k) {
        if (b + k >= cells) break;
        d.cell_start[co + b + k] = start;
        const uint4 e = make_uint4(static_cast<uint32_t>(b + k), start, v[k], 0u);
        if (v[k] == 0)
            d.zmin[co + b + k] = u2f(kEmptyZ);
        else if (v[k] <= kRowCell)
            list[small++] = e;
        else
            list[L.cell_stride - 1 - static_cast<int>(large++)] = e;
        start += v[k];
    }
}

// Scatter point indices into their cells (unordered; sorted per cell next),
// each at the place the histogram's atomic add gave it, with its z key beside
// it for the robust minimum.
__global__ void k_cell_fill(DevBuf d, Layout L) {
    const int f = blockIdx.y;
    const FrameDesc& fd = d.frames[f];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= fd.n) return;
    const int gi = fd.pt_off + i;
    const int cell = d.pt_cell[gi];
    if (cell < 0) return;
    const uint32_t pos = d.cell_start[(size_t)f * L.cell_stride + cell] + static_cast<uint32_t>(d.pt_loc[gi]);
    d.cell_items[(size_t)f * L.N + pos] = i;
    d.cell_zkey[(size_t)f * L.N + pos] = ord_f32(d.z[gi]);
}

// Bitonic sort of m (power of two) u32 keys in LDS by NT cooperating
// threads (tid in [0, NT)); SYNC() orders the stages.
template <int NT, typename Sync>
__device__ __forceinline__ void bitonic_u32(uint32_t* a, int m, int tid, Sync sync) {
    for (int k = 2; k <= m; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int t = tid; t < (m >> 1); t += NT) {
                const int lo = ((t & ~(j - 1)) << 1) | (t & (j - 1));
                const int hi = lo + j;
                const uint32_t x = a[lo], y = a[hi];
                const bool up = (lo & k) == 0;
                if ((x > y) == up) {
                    a[lo] = y;
                    a[hi] = x;
                }
            }
            sync();
        }
    }
}

// Robust minimum of a sorted cell (segmenter.cpp:249-260): s[0], replaced by
// s[i] for the largest i in [1, n/2] with s[i] - s[i-1] > 0.5f.  `keys` hold
// ord_f32(z) sorted ascending.  Returns via max-reduction over candidate i.
__device__ __forceinline__ float unord_f32(uint32_t k) {
    return u2f((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

template <int NT, typename Sync, typename MaxReduce>
__device__ __forceinline__ float robust_min(const uint32_t* keys, int n, int tid, Sync sync, MaxReduce maxred) {
    int best = 0;
    for (int i = 1 + tid; i <= n / 2; i += NT) {
        const float a = unord_f32(keys[i]);
        const float b = unord_f32(keys[i - 1]);
        if (a - b > 0.5F) best = i;  // i grows with the loop, keep the last hit
    }
    best = maxred(best);
    return unord_f32(keys[best]);
}

// Sorted cell of up to 64*S points held in registers: the point indices
// ascending for the RANSAC cells, and z for the robust minimum.
template <int S>
__device__ __forceinline__ void sort_cell_regs(int32_t* items, const uint32_t* zkeys, int n, int radial,
                                               float* zmin_cell) {
    const int lane = lane_id();
    uint32_t key[S];
    if (radial < kRansacRadialBins) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int e = s * kWave + lane;
            key[s] = e < n ? static_cast<uint32_t>(items[e]) : 0xffffffffu;
        }
        reg_sort_u32<S>(key);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int e = s * kWave + lane;
            if (e < n) items[e] = static_cast<int32_t>(key[s]);
        }
    }
    if (radial >= 1) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int e = s * kWave + lane;
            key[s] = e < n ? zkeys[e] : 0xffffffffu;
        }
        reg_sort_u32<S>(key);
        // Robust minimum (segmenter.cpp:249-260): the largest i in [1, n/2]
        // with s[i] - s[i-1] > 0.5f, else 0.
        int best = 0;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int e = s * kWave + lane;
            const uint32_t up = __shfl_up(key[s], 1, kWave);
            const uint32_t wrap = __shfl(key[s > 0 ? s - 1 : 0], kWave - 1, kWave);
            const uint32_t prev = lane > 0 ? up : wrap;
            if (e >= 1 && e <= n / 2 && unord_f32(key[s]) - unord_f32(prev) > 0.5F) best = e;
        }
#pragma unroll
        for (int o = kWave / 2; o > 0; o >>= 1) best = max(best, __shfl_xor(best, o, kWave));
        uint32_t kb = 0;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const uint32_t v = __shfl(key[s], best % kWave, kWave);
            if (best / kWave == s) kb = v;
        }
        if (lane == 0) *zmin_cell = unord_f32(kb);
    }
}

// Ascending bitonic sort of 16 keys, one per lane of each 16-lane row (all
// exchanges are DPP moves inside the row).
__device__ __forceinline__ uint32_t row_sort16_u32(uint32_t key) {
    const int r = lane_id() & 15;
#pragma unroll
    for (int k = 2; k <= 16; k <<= 1) {
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1) {
            const uint32_t other = lane_xor(key, j);
            const bool asc = (r & k) == 0;
            const bool lower = (r & j) == 0;
            key = (lower == asc) ? min(key, other) : max(key, other);
        }
    }
    return key;
}

// sort_cell_regs for a cell of n <= 16 points held by one 16-lane row
// (element e = lane & 15); every lane of the row calls it.
__device__ __forceinline__ void sort_cell_row(int32_t* items, const uint32_t* zkeys, int n, int radial,
                                              float* zmin_cell) {
    const int e = lane_id() & 15;
    if (radial < kRansacRadialBins) {
        uint32_t key = e < n ? static_cast<uint32_t>(items[e]) : 0xffffffffu;
        key = row_sort16_u32(key);
        if (e < n) items[e] = static_cast<int32_t>(key);
    }
    if (radial >= 1) {
        uint32_t key = e < n ? zkeys[e] : 0xffffffffu;
        key = row_sort16_u32(key);
        // Robust minimum (segmenter.cpp:249-260): the largest i in [1, n/2]
        // with s[i] - s[i-1] > 0.5f, else 0.
        const uint32_t prev = __shfl_up(key, 1, 16);
        int best = (e >= 1 && e <= n / 2 && unord_f32(key) - unord_f32(prev) > 0.5F) ? e : 0;
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) best = max(best, static_cast<int>(lane_xor(static_cast<uint32_t>(best), o)));
        const uint32_t kb = __shfl(key, (lane_id() & ~15) + best, kWave);
        if (e == 0) *zmin_cell = unord_f32(kb);
    }
}

// Sorts the point indices of every RANSAC cell ascending (so the cell lists
// follow the reference's input order) and z for the robust minimum.  Cells of
// up to 16 points are sorted by one 16-lane row each (DPP bitonic), four to a
// wavefront; larger ones, up to kSmallCell (512) points, by a wavefront each in
// registers; beyond that they are queued for k_cell_sort_big.  The cells near
// the sensor are both the largest and neighbours in cell order, so taken in
// that order a wavefront got four of them in a row and was the launch's tail:
// 22 -> 14 us per frame with the large cells on a list of their own.
__global__ __launch_bounds__(256) void k_cell_sort(DevBuf d, Layout L) {
    static_assert(kSmallCell == 8 * kWave, "the register sorts cover cells up to kSmallCell points");
    int tile, f;
    xcd_tile_frame(tile, f);
    const FrameDesc& fd = d.frames[f];
    const SegConst& s = fd.sc;
    const int lane = lane_id();
    const size_t co = (size_t)f * L.cell_stride;
    const int small = static_cast<int>(d.fs[f * kFsCount + kFsCellsSmall]);
    const int large = static_cast<int>(d.fs[f * kFsCount + kFsCellsLarge]);
    const int waves = gridDim.x * 4;
    const int wave = tile * 4 + static_cast<int>(threadIdx.x) / kWave;
    float* zmin = d.zmin + co;
    const uint4* list = d.cell_list + co;
    for (int q = wave; q < large; q += waves) {
        const uint4 e = list[L.cell_stride - 1 - q];
        const int cell = __builtin_amdgcn_readfirstlane(static_cast<int>(e.x));
        const int n = __builtin_amdgcn_readfirstlane(static_cast<int>(e.z));
        const uint32_t start = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(e.y)));
        if (n > kSmallCell) {
            if (lane == 0) {
                const uint32_t k = atomicAdd(&d.fs[f * kFsCount + kFsNumBig], 1u);
                if (k < static_cast<uint32_t>(L.cell_stride)) d.big_cells[co + k] = cell;
            }
            continue;
        }
        int32_t* items = d.cell_items + (size_t)f * L.N + start;
        const uint32_t* zk = d.cell_zkey + (size_t)f * L.N + start;
        const int radial = cell % s.rings;
        if (n <= kWave)
            sort_cell_regs<1>(items, zk, n, radial, zmin + cell);
        else if (n <= 2 * kWave)
            sort_cell_regs<2>(items, zk, n, radial, zmin + cell);
        else if (n <= 4 * kWave)
            sort_cell_regs<4>(items, zk, n, radial, zmin + cell);
        else
            sort_cell_regs<8>(items, zk, n, radial, zmin + cell);
    }
    // Row g of the wavefront takes list entry q + g.  The wavefronts after
    // those with a large cell come first; an entry is loaded one iteration
    // ahead.
    const int g = lane >> 4;
    const int turn = (wave - large % waves + waves) % waves;
    const uint4 none = make_uint4(0u, 0u, 0u, 0u);
    uint4 next = turn * 4 + g < small ? list[turn * 4 + g] : none;
    for (int q = turn * 4; q < small; q += waves * 4) {
        const uint4 e = next;
        const int ahead = q + waves * 4 + g;
        next = ahead < small ? list[ahead] : none;
        const int cell = static_cast<int>(e.x);
        if (e.z)
            sort_cell_row(d.cell_items + (size_t)f * L.N + e.y, d.cell_zkey + (size_t)f * L.N + e.y,
                          static_cast<int>(e.z), cell % s.rings, zmin + cell);
    }
}

// Cells with more than kSmallCell points: one 1024-thread workgroup each.
__global__ __launch_bounds__(1024) void k_cell_sort_big(DevBuf d, Layout L) {
    __shared__ uint32_t a[kBigCell];
    __shared__ int red[1024 / kWave];
    const int f = blockIdx.y;
    const FrameDesc& fd = d.frames[f];
    const SegConst& s = fd.sc;
    const size_t co = (size_t)f * L.cell_stride;
    const uint32_t nbig = min(d.fs[f * kFsCount + kFsNumBig], static_cast<uint32_t>(L.cell_stride));
    const int tid = threadIdx.x;
    auto sync = [] { __syncthreads(); };
    for (uint32_t b = blockIdx.x; b < nbig; b += gridDim.x) {
        const int cell = d.big_cells[co + b];
        const uint32_t n = d.cell_count[co + cell];
        if (n > static_cast<uint32_t>(kBigCell)) {
            if (tid == 0) atomicOr(&d.fs[f * kFsCount + kFsErr], kErrCellCapacity);
            continue;
        }
        const uint32_t start = d.cell_start[(size_t)f * L.cell_stride + cell];
        int32_t* items = d.cell_items + (size_t)f * L.N + start;
        int m = 1;
        while (m < static_cast<int>(n)) m <<= 1;
        const int radial = cell % s.rings;
        if (radial < kRansacRadialBins) {
            for (int t = tid; t < m; t += 1024) a[t] = t < static_cast<int>(n) ? static_cast<uint32_t>(items[t]) : 0xffffffffu;
            __syncthreads();
            bitonic_u32<1024>(a, m, tid, sync);
            for (int t = tid; t < static_cast<int>(n); t += 1024) items[t] = static_cast<int32_t>(a[t]);
            __syncthreads();
        }
        if (radial >= 1) {
            for (int t = tid; t < m; t += 1024)
                a[t] = t < static_cast<int>(n) ? d.cell_zkey[(size_t)f * L.N + start + t] : 0xffffffffu;
            __syncthreads();
            bitonic_u32<1024>(a, m, tid, sync);
            const float r = robust_min<1024>(a, static_cast<int>(n), tid, sync, [&](int v) {
#pragma unroll
                for (int o = kWave / 2; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, kWave));
                if (lane_id() == 0) red[tid / kWave] = v;
                __syncthreads();
                int m2 = 0;
                for (int i = 0; i < 1024 / kWave; ++i) m2 = max(m2, red[i]);
                __syncthreads();
                return m2;
            });
            if (tid == 0) d.zmin[co + cell] = r;
        }
        __syncthreads();
    }
}

// RECM recurrence along each azimuth slice (segmenter.cpp:215-267).  The
// 49 float additions must happen in order (a log-step min-plus scan would
// re-associate them), so each slice is one sequential lane.
// One workgroup per 64 slices.  A slice's cells are contiguous (cell =
// slice * rings + r), so its 64 x rings minima are one contiguous block: four
// wavefronts load it into LDS with coalesced reads in flight together (one
// wavefront waited for them in 49 turns: 17 -> 8 us per frame), each lane
// of the first runs its slice's recurrence there, and the elevations go back
// the same way.  Grids with more than kRecmRings rings read and write global
// memory directly (eight rings' minima loaded ahead of their eight steps).
constexpr int kRecmRings = 64;
constexpr int kRecmThreads = 256;

__global__ __launch_bounds__(kRecmThreads) void k_recm(DevBuf d, Layout L) {
    __shared__ float blk[kWave * (kRecmRings + 1)];
    const int f = blockIdx.y;
    const SegConst& s = d.frames[f].sc;
    const int s0 = blockIdx.x * kWave;
    if (s0 >= s.slices) return;
    const int tid = threadIdx.x;
    const int R = s.rings;
    const size_t co = (size_t)f * L.cell_stride;
    float* E = d.elev + co;
    const float* zm = d.zmin + co;
    auto step = [&](float prev, float z) {
        const float b = prev + s.dz;
        if (f2u(z) == kEmptyZ) return b;
        return (b < z) ? b : z;  // std::min(curr_z_min, prev + dz)
    };
    if (R <= kRecmRings) {
        const int ns = min(kWave, s.slices - s0);
        const int total = ns * R;
        const float* src = zm + (size_t)s0 * R;
        // An odd row length keeps the lanes of the recurrence on different
        // banks.
        const int pitch = R | 1;
        constexpr int kTurns = kWave * kRecmRings / kRecmThreads;
        float v[kTurns];
#pragma unroll
        for (int k = 0; k < kTurns; ++k) {
            const int i = tid + k * kRecmThreads;
            v[k] = i < total ? src[i] : 0.0f;
        }
#pragma unroll
        for (int k = 0; k < kTurns; ++k) {
            const int i = tid + k * kRecmThreads;
            if (i < total) blk[(i / R) * pitch + i % R] = v[k];
        }
        __syncthreads();
        if (tid < ns) {
            float* row = blk + tid * pitch;
            float prev = s.e0;
            row[0] = prev;
            for (int r0 = 1; r0 < R; r0 += 8) {
                float z[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) z[k] = row[min(r0 + k, R - 1)];
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    if (r0 + k >= R) break;
                    prev = step(prev, z[k]);
                    row[r0 + k] = prev;
                }
            }
        }
        __syncthreads();
        float* dst = E + (size_t)s0 * R;
#pragma unroll
        for (int k = 0; k < kTurns; ++k) {
            const int i = tid + k * kRecmThreads;
            if (i < total) dst[i] = blk[(i / R) * pitch + i % R];
        }
        return;
    }
    const int sl = s0 + tid;
    if (tid >= kWave || sl >= s.slices) return;
    const int off = sl * R;
    E[off] = s.e0;
    float prev = s.e0;
    for (int r0 = 1; r0 < R; r0 += 8) {
        float zz[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) zz[k] = (r0 + k < R) ? zm[off + r0 + k] : 0.0f;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            if (r0 + k >= R) break;
            prev = step(prev, zz[k]);
            E[off + r0 + k] = prev;
        }
    }
}

// RANSAC candidate count per near cell, one wave per cell (a grid-stride
// loop over the frame's slices x 4 near cells), in the reference's iteration
// order: k = slice*4 + radial (segmenter.cpp:328-351).
__global__ __launch_bounds__(256) void k_cand_count(DevBuf d, Layout L) {
    const int f = blockIdx.y;
    const FrameDesc& fd = d.frames[f];
    const SegConst& s = fd.sc;
    const int w = threadIdx.x / kWave;
    const int lane = lane_id();
    for (int k = blockIdx.x * 4 + w; k < s.slices * kRansacRadialBins; k += gridDim.x * 4) {
    const int cell = (k / kRansacRadialBins) * s.rings + (k % kRansacRadialBins);
    const size_t co = (size_t)f * L.cell_stride;
    const uint32_t n = d.cell_count[co + cell];
    const uint32_t start = d.cell_start[(size_t)f * L.cell_stride + cell];
    const uint32_t* zk = d.cell_zkey + (size_t)f * L.N + start;  // the cell's z in any order
    const float e = d.elev[co + cell];
    uint32_t c = 0;
    for (uint32_t t = lane; t < n; t += kWave) {
        const float z = unord_f32(zk[t]);
        c += (fabsf(e - z) < s.two_thr) ? 1u : 0u;
    }
    c = wave_sum(c);
    if (lane == 0) d.cand_count[(size_t)f * L.cand_stride + k] = c;
    }
}

// Candidate compaction in the reference's order, a wavefront per near cell and
// four cells in a row per workgroup and turn.  A workgroup sums the counts of
// the cells before its own itself (a few reads per thread; a launch for their
// scan cost more than that); the one with the last cells writes the total.
__global__ __launch_bounds__(256) void k_cand_fill(DevBuf d, Layout L) {
    __shared__ uint32_t part[256 / kWave];
    const int f = blockIdx.y;
    const FrameDesc& fd = d.frames[f];
    const SegConst& s = fd.sc;
    const int w = threadIdx.x / kWave;
    const int lane = lane_id();
    const int cells = s.slices * kRansacRadialBins;
    const uint32_t* count = d.cand_count + (size_t)f * L.cand_stride;
    const size_t co = (size_t)f * L.cell_stride;
    const size_t ob = (size_t)f * L.N;
    uint32_t before = 0;  // candidates of the cells before k0
    int summed = 0;
    for (int k0 = blockIdx.x * 4; k0 < cells; k0 += gridDim.x * 4) {
        uint32_t sum = 0;
        for (int i = summed + threadIdx.x; i < k0; i += 256) sum += count[i];
        sum = wave_sum(sum);
        if (lane == 0) part[w] = sum;
        __syncthreads();
        before += part[0] + part[1] + part[2] + part[3];
        __syncthreads();
        summed = k0;
        uint32_t pos = before;
        for (int q = 0; q < w; ++q) pos += k0 + q < cells ? count[k0 + q] : 0u;
        const int k = k0 + w;
        if (k + 1 == cells && lane == 0) d.fs[f * kFsCount + kFsCands] = pos + count[k];
        if (k >= cells) continue;
        const int cell = (k / kRansacRadialBins) * s.rings + (k % kRansacRadialBins);
        const uint32_t n = d.cell_count[co + cell];
        const uint32_t start = d.cell_start[co + cell];
        const int32_t* items = d.cell_items + ob + start;
        const float e = d.elev[co + cell];
        for (uint32_t t0 = 0; t0 < n; t0 += kWave) {
            const uint32_t t = t0 + lane;
            bool pred = false;
            float x = 0, y = 0, z = 0;
            if (t < n) {
                const float4 pc = d.pt_xyzc[fd.pt_off + items[t]];  // one gather per point
                x = pc.x;
                y = pc.y;
                z = pc.z;
                pred = fabsf(e - z) < s.two_thr;
            }
            const uint64_t mask = __ballot(pred);
            if (pred) {
                const uint32_t o = pos + lanes_below(mask);
                d.cx[ob + o] = x;
                d.cy[ob + o] = y;
                d.cz[ob + o] = z;
            }
            pos += static_cast<uint32_t>(__popcll(mask));
        }
    }
}

// mt19937 with seed 42 (the reference's std::mt19937 gen{42},
// segmenter.cpp:369): the raw output stream does not depend on the frame, so
// it is generated once per context.  Standard MT19937 recurrence
// (Matsumoto & Nishimura 1998).
__global__ void k_mt19937(uint32_t* out, int count) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    uint32_t mt[624];
    mt[0] = 42u;
    for (int i = 1; i < 624; ++i) mt[i] = 1812433253u * (mt[i - 1] ^ (mt[i - 1] >> 30)) + static_cast<uint32_t>(i);
    int idx = 624;
    for (int k = 0; k < count; ++k) {
        if (idx >= 624) {
            for (int i = 0; i < 624; ++i) {
                const uint32_t yv = (mt[i] & 0x80000000u) | (mt[(i + 1) % 624] & 0x7fffffffu);
                mt[i] = mt[(i + 397) % 624] ^ (yv >> 1) ^ ((yv & 1u) ? 0x9908b0dfu : 0u);
            }
            idx = 0;
        }
        uint32_t yv = mt[idx++];
        yv ^= yv >> 11;
        yv ^= (yv << 7) & 0x9d2c5680u;
        yv ^= (yv << 15) & 0xefc60000u;
        yv ^= yv >> 18;
        out[k] = yv;
    }
}

// The index pairs of the 60 hypotheses by one lane: libstdc++'s
// uniform_int_distribution<uint32_t> for a 32-bit engine (Lemire's
// nearly-divisionless method, bits/uniform_int_dist.h) over the raw stream,
// redrawing p3 while it equals p2 (segmenter.cpp:379-386).  False when the
// stored stream ends.
__device__ bool draw_pairs(const uint32_t* raw, uint32_t n, uint2* pairs) {
    int pos = 0;
    bool good = true;
    auto draw = [&]() -> uint32_t {
        if (pos >= kMtRawCount) {
            good = false;
            return 0;
        }
        uint64_t prod = static_cast<uint64_t>(raw[pos]) * n;
        ++pos;
        uint32_t low = static_cast<uint32_t>(prod);
        if (low < n) {
            const uint32_t thresh = (0u - n) % n;
            while (low < thresh && good) {
                if (pos >= kMtRawCount) {
                    good = false;
                    break;
                }
                prod = static_cast<uint64_t>(raw[pos]) * n;
                ++pos;
                low = static_cast<uint32_t>(prod);
            }
        }
        return static_cast<uint32_t>(prod >> 32);
    };
    for (int it = 0; it < kRansacIters && good; ++it) {
        const uint32_t a = draw();
        uint32_t b = draw();
        while (b == a && good) b = draw();
        pairs[it] = make_uint2(a, b);
    }
    return good;
}

// Hypotheses and their inlier counts (segmenter.cpp:376-431).  Every workgroup
// draws the index pairs and builds the 60 planes itself, one per lane of its
// first wavefront, while the others' candidates are on their way: unless a
// draw is rejected or repeats (about one frame in a hundred; then one lane
// draws them all in order), pair `it` comes from values 2 it and 2 it + 1 of
// the stream.  Every candidate scores all planes with the reference's float
// expression; a wavefront counts a plane's hits with ballots over its rows,
// lane `it` keeps plane it's count, and the workgroup's counts meet in LDS
// before one atomic per plane.  With R = 1 candidate per thread more
// workgroups share a frame (few frames), with 4 each plane is read once for
// four rows.  Per frame with the serial draw in a launch of its own: 38 us,
// now 9.
template <int R>
__global__ __launch_bounds__(256) void k_ransac_count(DevBuf d, Layout L) {
    __shared__ uint32_t acc[kRansacIters];
    __shared__ float4 plane[kRansacIters];
    __shared__ uint2 pairs[kRansacIters];
    __shared__ uint32_t usable;
    static_assert(kRansacIters <= kWave, "one lane per hypothesis");
    const int f = blockIdx.y;
    const SegConst& s = d.frames[f].sc;
    const uint32_t n = d.fs[f * kFsCount + kFsCands];
    const uint32_t base = blockIdx.x * (256u * R);
    const int tid = threadIdx.x;
    const int lane = lane_id();
    if (n < 2) {  // without candidates the reference returns (segmenter.cpp:353-356); with one it never ends
        if (n == 1 && blockIdx.x == 0 && tid == 0) atomicOr(&d.fs[f * kFsCount + kFsErr], kErrRansacSingle);
        return;
    }
    if (base >= n) return;
    const size_t ob = (size_t)f * L.N;
    float x[R], y[R], z[R];
    bool act[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t t = base + r * 256u + tid;
        act[r] = t < n;
        x[r] = act[r] ? d.cx[ob + t] : 0.0f;
        y[r] = act[r] ? d.cy[ob + t] : 0.0f;
        z[r] = act[r] ? d.cz[ob + t] : 0.0f;
    }
    if (tid < kRansacIters) acc[tid] = 0;
    if (tid < kWave) {
        const int it = min(lane, kRansacIters - 1);
        const uint64_t pa = static_cast<uint64_t>(d.mt_raw[2 * it]) * n, pb = static_cast<uint64_t>(d.mt_raw[2 * it + 1]) * n;
        uint2 pr = make_uint2(static_cast<uint32_t>(pa >> 32), static_cast<uint32_t>(pb >> 32));
        bool ok = true;
        // A product whose low word is below n may be rejected.
        if (__ballot(static_cast<uint32_t>(pa) < n || static_cast<uint32_t>(pb) < n || pr.x == pr.y)) {
            if (lane == 0) usable = draw_pairs(d.mt_raw, n, pairs) ? 1u : 0u;
            wave_sync();
            ok = usable != 0;
            if (ok) pr = pairs[it];
            if (!ok && lane == 0 && blockIdx.x == 0) atomicOr(&d.fs[f * kFsCount + kFsErr], kErrRngExhausted);
        }
        wave_sync();
        if (lane == 0) usable = ok ? 1u : 0u;
        if (ok && lane < kRansacIters) {
            // Plane through the sensor's foot point and two candidates
            // (segmenter.cpp:389-418).
            const float p1x = 0.0f, p1y = 0.0f, p1z = s.neg_h;
            const float p2x = d.cx[ob + pr.x], p2y = d.cy[ob + pr.x], p2z = d.cz[ob + pr.x];
            const float p3x = d.cx[ob + pr.y], p3y = d.cy[ob + pr.y], p3z = d.cz[ob + pr.y];
            float nx = ((p2y - p1y) * (p3z - p1z)) - ((p2z - p1z) * (p3y - p1y));
            float ny = ((p2z - p1z) * (p3x - p1x)) - ((p2x - p1x) * (p3z - p1z));
            float nz = ((p2x - p1x) * (p3y - p1y)) - ((p2y - p1y) * (p3x - p1x));
            const float den2 = (nx * nx) + (ny * ny) + (nz * nz);
            uint32_t valid = 0;
            float pd = 0.0f;
            if (!(den2 < 1.0e-5F)) {
                const float norm = 1.0F / sqrtf(den2);
                nz *= norm;
                if (!(fabsf(nz) < s.cos_max)) {
                    nx *= norm;
                    ny *= norm;
                    pd = (nx * p1x) + (ny * p1y) + (nz * p1z);
                    valid = 1;
                }
            }
            // A plane that is not valid scores nothing: NaN compares false.
            plane[lane] = valid ? make_float4(nx, ny, nz, pd) : make_float4(0.0f, 0.0f, 0.0f, __builtin_nanf(""));
            if (blockIdx.x == 0) {
                reinterpret_cast<float4*>(d.hyp)[(size_t)f * kRansacIters + lane] = make_float4(nx, ny, nz, pd);
                d.hyp_valid[f * kRansacIters + lane] = valid;
            }
        }
    }
    __syncthreads();
    if (!usable) return;
    const float thr = s.thr;
    uint32_t mine = 0;
#pragma unroll 4
    for (int it = 0; it < kRansacIters; ++it) {
        const float4 p = plane[it];
        uint32_t c = 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float od = fabsf((p.x * x[r]) + (p.y * y[r]) + (p.z * z[r]) - p.w);
            c += static_cast<uint32_t>(__popcll(__ballot(act[r] && od < thr)));
        }
        mine += lane == it ? c : 0u;
    }
    if (lane < kRansacIters && mine) atomicAdd(&acc[lane], mine);
    __syncthreads();
    if (tid < kRansacIters && acc[tid]) atomicAdd(&d.hyp_count[f * kRansacIters + tid], acc[tid]);
}

// The best hypothesis, by every wavefront that needs it: the largest count,
// the first of equal ones (strict `>` in iteration order), then the sign flip
// (segmenter.cpp:433-453).  Returns its count, 0 when none applies.
__device__ __forceinline__ uint32_t best_plane(const DevBuf& d, int f, float4& plane) {
    const uint32_t* fs = d.fs + f * kFsCount;
    plane = make_float4(0.0f, 0.0f, 1.0f, 0.0f);
    if (fs[kFsCands] < 2 || (fs[kFsErr] & (kErrRansacSingle | kErrRngExhausted))) return 0;
    const int it = lane_id();
    uint64_t key = 0;
    if (it < kRansacIters && d.hyp_valid[f * kRansacIters + it])
        key = static_cast<uint64_t>(d.hyp_count[f * kRansacIters + it]) << 6 | static_cast<uint64_t>(kWave - 1 - it);
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        const uint64_t k = __shfl_xor(key, o, kWave);
        key = k > key ? k : key;
    }
    const uint32_t best = static_cast<uint32_t>(key >> 6);
    if (best == 0) return 0;
    const int at = kWave - 1 - static_cast<int>(key & (kWave - 1));
    plane = reinterpret_cast<const float4*>(d.hyp)[(size_t)f * kRansacIters + at];
    if (plane.z < 0) plane = make_float4(-plane.x, -plane.y, -plane.z, -plane.w);
    return best;
}

// Pixel states after RECM + RANSAC: the winner's label (segmenter.cpp:
// 278-281 and 466-475), its index (cloud_mapping_indices_) and xyz.
__global__ __launch_bounds__(256) void k_pixel_label(DevBuf d, Layout L) {
    const int f = blockIdx.y;
    const FrameDesc& fd = d.frames[f];
    const SegConst& s = fd.sc;
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (static_cast<int>(blockIdx.x * blockDim.x) >= s.H * s.W) return;
    const size_t po = fd.pix_off + p;
    const unsigned long long key = p < s.H * s.W ? d.pix_key[po] : ~0ull;
    float4 plane;
    const uint32_t best = best_plane(d, f, plane);
    if (p == 0 && d.fs[f * kFsCount + kFsCands] >= 2 &&
        !(d.fs[f * kFsCount + kFsErr] & (kErrRansacSingle | kErrRngExhausted))) {
        uint32_t* fs = d.fs + f * kFsCount;
        fs[kFsBest] = best;
        fs[kFsApplied] = best > 0 ? 1u : 0u;
        fs[kFsPlaneA] = f2u(plane.x);
        fs[kFsPlaneB] = f2u(plane.y);
        fs[kFsPlaneC] = f2u(plane.z);
        fs[kFsPlaneD] = f2u(plane.w);
    }
    if (p >= s.H * s.W) return;
    if (key == ~0ull) {
        d.state[po] = kEmpty;
        d.mapping[po] = -1;
        d.pxyz[po] = make_float4(0.0f, 0.0f, 0.0f, __int_as_float(-1));  // w: the winner, -1 for none
        return;
    }
    const int i = static_cast<int>(key & ((1ull << L.idx_bits) - 1));
    const float4 pc = d.pt_xyzc[fd.pt_off + i];  // one gather: x, y, z and the cell
    const float x = pc.x, y = pc.y, z = pc.z;
    const int cell = __float_as_int(pc.w);
    const float e = d.elev[(size_t)f * L.cell_stride + cell];
    uint8_t lab = (z >= e + s.thr) ? kObstacle : kGround;
    if (best > 0 && (cell % s.rings) < kRansacRadialBins) {
        const float sd = (plane.x * x) + (plane.y * y) + (plane.z * z) - plane.w;
        if (sd < s.thr) lab = kGround;
    }
    d.state[po] = lab;
    d.mapping[po] = i;
    d.pxyz[po] = make_float4(x, y, z, __int_as_float(i));
}

// ---------------------------------------------------------------------------
void launch_segment_front(lp_context* c, int B, bool cleared) {
    DevBuf& d = c->d;
    const Layout& L = c->L;
    hipStream_t st = c->stream;
    const int nb = (L.N + 255) / 256;
    if (!cleared) launch_clear(c, B, false);
    stage_mark(c, "project");
    const int wg = c->point_wg;
    if (c->persistent)
        hipLaunchKernelGGL(k_project_q, dim3(kPersistentWorkgroups), dim3(wg), 0, st, d, L, B);
    else
        hipLaunchKernelGGL(k_project, dim3((L.N + wg - 1) / wg, B), dim3(wg), 0, st, d, L);
    stage_mark(c, "cells");
    constexpr int kStartTile = kStartThreads * kStartItems;
    hipLaunchKernelGGL(k_cell_start, dim3((L.cell_stride + kStartTile - 1) / kStartTile, B), dim3(kStartThreads), 0, st, d, L);
    hipLaunchKernelGGL(k_cell_fill, dim3(nb, B), dim3(256), 0, st, d, L);
    // About 8192 wavefronts in all, at least 64 and at most 4096 per frame.
    hipLaunchKernelGGL(k_cell_sort, dim3(std::min(1024, std::max(16, 2048 / B)), B), dim3(256), 0, st, d, L);
    // Cells beyond kSmallCell points are rare: about 1024 workgroups in all.
    hipLaunchKernelGGL(k_cell_sort_big, dim3(std::min(64, std::max(4, 1024 / B)), B), dim3(1024), 0, st, d, L);
    stage_mark(c, "recm");
    hipLaunchKernelGGL(k_recm, dim3((L.cand_stride / kRansacRadialBins + kWave - 1) / kWave, B), dim3(kRecmThreads), 0,
                       st, d, L);
    stage_mark(c, "ransac");
    // A wavefront per near cell (slices x 4, 1440 by default) for few frames,
    // 512 wavefronts a frame on larger batches.
    const int cand_grid = std::min(384, std::max(128, 1536 / B));
    hipLaunchKernelGGL(k_cand_count, dim3(cand_grid, B), dim3(256), 0, st, d, L);
    hipLaunchKernelGGL(k_cand_fill, dim3(cand_grid, B), dim3(256), 0, st, d, L);
    // Few frames leave room for a candidate per thread: eight of 128x2048 22 us
    // (27 with four), of 64x2048 20 (24).  Twelve of 128x2048 are even, sixteen
    // 36 (30), 24 of 64x2048 are even, 32 34 (31).
    if (B <= 8)
        hipLaunchKernelGGL(k_ransac_count<1>, dim3((L.N + 255) / 256, B), dim3(256), 0, st, d, L);
    else
        hipLaunchKernelGGL(k_ransac_count<4>, dim3((L.N + 1023) / 1024, B), dim3(256), 0, st, d, L);
    stage_mark(c, "pixels");
    hipLaunchKernelGGL(k_pixel_label, dim3((L.P + 255) / 256, B), dim3(256), 0, st, d, L);
}

void launch_clear(lp_context* c, int B, bool noise) {
    stage_mark(c, "clear");
    hipLaunchKernelGGL(k_clear, dim3(256, B), dim3(256), 0, c->stream, c->d, c->L, noise);
}

// k_hash_reset clears the slots a stage occupied; k_hash_init clears every slot
// and the frames' scalars (context creation).
__global__ void k_hash_reset(DevBuf d, Layout L, const int32_t* slots, int count_slot) {
    reset_slots(d, L, blockIdx.y, slots, count_slot, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
}

__global__ void k_hash_init(DevBuf d, Layout L) {
    for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < L.B * kFsCount; q += gridDim.x * blockDim.x) d.fs[q] = 0;
    const size_t total = (size_t)L.B * L.hash_cap;
    for (size_t o = blockIdx.x * (size_t)blockDim.x + threadIdx.x; o < total; o += (size_t)gridDim.x * blockDim.x) {
        d.hslot[o] = HashSlot{-1, 0u, 0, kHashMinClean};
    }
}

void launch_hash_reset(lp_context* c, int B, const int32_t* slots, int count_slot) {
    hipLaunchKernelGGL(k_hash_reset, dim3(64, B), dim3(256), 0, c->stream, c->d, c->L, slots, count_slot);
}

void launch_hash_init(lp_context* c) {
    hipLaunchKernelGGL(k_hash_init, dim3(1024), dim3(256), 0, c->stream, c->d, c->L);
}

void launch_mt19937(uint32_t* out, int count, hipStream_t st) {
    hipLaunchKernelGGL(k_mt19937, dim3(1), dim3(1), 0, st, out, count);
}

}  // namespace lp
