// lp_cluster.hip -- curved-voxel clustering on gfx950.
//
// Reference: lidar_processing_lib/src/clusterer.cpp:55-239.  The reference
// hashes (range, azimuth, elevation) voxel keys into a linear-probing map
// (static_unordered_map.hpp) and labels voxels by BFS from each unlabelled
// point in input order over the 26-neighbourhood (range and elevation
// bounded, azimuth wrapping by one), numbering components in the order of
// their first point; removeSmallClusters then drops components with fewer
// than min_cluster_size points and renumbers the rest in order.  The result
// is therefore: label = rank, among surviving components, of the
// component's minimum point index.
//
// Here: voxel keys go into an open-addressing HBM hash set by atomicCAS
// (one dense id per occupied voxel, per-voxel point count and minimum point
// index by atomics on the voxel's own slot), components come from a
// lock-free union-find over dense ids (in LDS by one workgroup per frame, in
// global memory by the whole grid when a frame's voxels do not fit there), and
// a component's label is the rank of its first point among the surviving
// components'.
#include <algorithm>

#include "lp_kernels.h"
#include "lp_joins.h"
#include "lp_queue.h"

namespace lp {

using namespace lpd;

constexpr float kTwoPiF = 6.28318548202514648438f;   // Clusterer::TWO_M_PIf
constexpr float kHalfPiF = 1.57079637050628662109f;  // M_PI_2f
constexpr int kCcLds = 32768;                        // voxels per frame for the LDS union-find

__device__ __forceinline__ uint32_t max_bits(float v) {
    // Non-negative floats order like their bit patterns; -0 counts as +0
    // (only ceilf(max / res) is used, which is the same for both).
    const uint32_t u = f2u(v);
    return u == 0x80000000u ? 0u : u;
}

// Obstacle o: cartesianToSpherical (clusterer.cpp:55-100); m collects the
// maxima of range, azimuth and elevation.
__device__ __forceinline__ void spherical(const DevBuf& d, size_t o, float x, float y, float z, uint32_t (&m)[3]) {
    float az = fdlibm_atan2f(y, x);
    az = (az < 0) ? (az + kTwoPiF) : az;
    const float dsq = x * x + y * y;
    const float dist = sqrtf(dsq);
    const float range = sqrtf(dsq + z * z);
    const float el = fdlibm_atanf(z / dist) + kHalfPiF;
    d.sr[o] = range;
    d.sa[o] = az;
    d.se[o] = el;
    m[0] = max(m[0], max_bits(range));
    m[1] = max(m[1], max_bits(az));
    m[2] = max(m[2], max_bits(el));
}

// The frame maxima: wavefront maxima (DPP inside 16-lane rows, then two
// shuffles), the workgroup's in LDS, one atomic per workgroup and value
// (per wavefront, the per-frame counters were a contention point).  All
// threads of the workgroup call it.
__device__ __forceinline__ void frame_maxima(const DevBuf& d, int f, uint32_t (&m)[3]) {
    __shared__ uint32_t red[3][1024 / kWave];
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
#pragma unroll
        for (int q = 0; q < 3; ++q)
            m[q] = max(m[q], o < 16 ? lane_xor(m[q], o) : static_cast<uint32_t>(__shfl_xor(m[q], o, kWave)));
    }
    const int w = static_cast<int>(threadIdx.x) / kWave;
    if (lane_id() == 0)
        for (int q = 0; q < 3; ++q) red[q][w] = m[q];
    __syncthreads();
    if (threadIdx.x < 3) {
        uint32_t v = red[threadIdx.x][0];
        for (int q = 1; q < static_cast<int>(blockDim.x) / kWave; ++q) v = max(v, red[threadIdx.x][q]);
        atomicMax(&d.fs[f * kFsCount + kFsMaxR + threadIdx.x], v);
    }
}
static_assert(kFsMaxA == kFsMaxR + 1 && kFsMaxE == kFsMaxR + 2, "the maxima's slots follow one another");

// Obstacle split: input-order compaction of OBSTACLE points
// (processor.cpp:562-579) over tiles of 1024 points (two rows of 512,
// coalesced), after the points before it, of which the labels kernel left the
// obstacle count of every 64 in obs_rows.  cl_flag receives every point's
// exclusive obstacle count (the split into ground and unknown clouds reads
// it); the last tile writes the obstacle count.  A tile's obstacles meet in
// LDS, so their index and coordinates leave in full rows and every lane has
// one for the spherical coordinates, which took a launch and a pass of their
// own before.  Two rows per thread: what a frame's tiles wait for is the chain
// from labels to coordinates to atan2, so more, shorter ones are faster (one
// 64x2048 frame 26 -> 9 us with all three passes, 20 with tiles of 2048 points
// by 256 threads; four frames at a time 45 against 54 us).
constexpr int kObsTile = 1024;
constexpr int kObsThreads = 512;
constexpr int kObsRows = kObsTile / kObsThreads;

__global__ __launch_bounds__(kObsThreads) void k_obs_gather(DevBuf d, Layout L) {
    __shared__ uint32_t lds[kObsRows * kObsThreads / kWave + 1];
    __shared__ float4 obs[kObsTile];
    const int f = blockIdx.y;
    const FrameDesc& fd = d.frames[f];
    const int n = fd.n;
    const int tile = blockIdx.x;
    const int base = tile * kObsTile;
    if (base >= n) {
        if (tile == 0 && threadIdx.x == 0) d.fs[f * kFsCount + kFsObstacles] = 0;
        return;
    }
    const uint32_t* cnt = d.obs_rows + (size_t)f * L.obs_rows;
    uint32_t pre = 0;
    for (int i = threadIdx.x; i < tile * (kObsTile / kWave); i += kObsThreads) pre += cnt[i];
    uint32_t m = 0;
    float x[kObsRows], y[kObsRows], z[kObsRows];
#pragma unroll
    for (int k = 0; k < kObsRows; ++k) {
        const int i = base + k * kObsThreads + static_cast<int>(threadIdx.x);
        if (i < n && d.labels[fd.pt_off + i] == LP_LABEL_OBSTACLE) m |= 1u << k;
    }
#pragma unroll
    for (int k = 0; k < kObsRows; ++k) {
        const int gi = fd.pt_off + base + k * kObsThreads + static_cast<int>(threadIdx.x);
        if ((m >> k) & 1u) {
            x[k] = d.x[gi];
            y[k] = d.y[gi];
            z[k] = d.z[gi];
        }
    }
    uint32_t pre_total;
    block_exclusive_sum<kObsThreads>(pre, lds, &pre_total);
    uint32_t pos[kObsRows];
    const uint32_t total = tile_compact<kObsThreads, kObsRows>(m, pos, lds);
    const size_t ob = (size_t)f * L.N;
#pragma unroll
    for (int k = 0; k < kObsRows; ++k) {
        const int i = base + k * kObsThreads + static_cast<int>(threadIdx.x);
        if (i < n) d.cl_flag[ob + i] = pre_total + pos[k];
        if ((m >> k) & 1u) obs[pos[k]] = make_float4(x[k], y[k], z[k], __int_as_float(i));
    }
    __syncthreads();
    uint32_t mx[3] = {0, 0, 0};
    for (uint32_t q = threadIdx.x; q < total; q += kObsThreads) {
        const float4 p = obs[q];
        const size_t o = ob + pre_total + q;
        d.obs_src[o] = __float_as_int(p.w);
        d.ox[o] = p.x;
        d.oy[o] = p.y;
        d.oz[o] = p.z;
        spherical(d, o, p.x, p.y, p.z, mx);
    }
    frame_maxima(d, f, mx);
    if (threadIdx.x == 0 && base + kObsTile >= n) d.fs[f * kFsCount + kFsObstacles] = pre_total + total;
}

// Ground and unsegmented clouds of the same split (processor.cpp:565-577):
// with gnd_flag scanned into obs_flag and cl_flag still the obstacle scan,
// an UNKNOWN point's position among the unknowns is its index less the
// ground and obstacle points before it.  split_idx holds the ground indices
// followed by the unknown ones.
__global__ void k_label_split(DevBuf d, Layout L) {
    const int f = blockIdx.y;
    const FrameDesc& fd = d.frames[f];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= fd.n) return;
    const uint32_t lab = d.labels[fd.pt_off + i];
    if (lab == LP_LABEL_OBSTACLE) return;
    const size_t ob = (size_t)f * L.N;
    const uint32_t g = d.obs_flag[ob + i];
    if (lab == LP_LABEL_GROUND) {
        d.split_idx[ob + g] = i;
    } else {
        const uint32_t ng = d.fs[f * kFsCount + kFsGround];
        d.split_idx[ob + ng + (i - g - d.cl_flag[ob + i])] = i;
    }
}

// Standalone Clusterer::cluster input: the staged cloud is the obstacle cloud.
__global__ __launch_bounds__(256) void k_cluster_input(DevBuf d, Layout L) {
    const int f = blockIdx.y;
    const FrameDesc& fd = d.frames[f];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) d.fs[f * kFsCount + kFsObstacles] = static_cast<uint32_t>(fd.n);
    if (static_cast<int>(blockIdx.x * blockDim.x) >= fd.n) return;
    uint32_t mx[3] = {0, 0, 0};
    if (i < fd.n) {
        const size_t ob = (size_t)f * L.N;
        const int gi = fd.pt_off + i;
        const float x = d.x[gi], y = d.y[gi], z = d.z[gi];
        d.obs_src[ob + i] = i;
        d.ox[ob + i] = x;
        d.oy[ob + i] = y;
        d.oz[ob + i] = z;
        spherical(d, ob + i, x, y, z, mx);
    }
    frame_maxima(d, f, mx);
}

struct Dims {
    int32_t nr, na, ne;
};

// num_range / num_azimuth / num_elevation (clusterer.cpp:94-99).
__device__ __forceinline__ Dims dims_of(const DevBuf& d, int f, const CluConst& cc) {
    const uint32_t* fs = d.fs + f * kFsCount;
    Dims dm;
    dm.nr = static_cast<int32_t>(ceilf(u2f(fs[kFsMaxR]) / cc.res_r) + 1);
    dm.na = static_cast<int32_t>(ceilf(u2f(fs[kFsMaxA]) / cc.res_az) + 1);
    dm.ne = static_cast<int32_t>(ceilf(u2f(fs[kFsMaxE]) / cc.res_el) + 1);
    return dm;
}

__device__ __forceinline__ uint32_t hash_slot(int32_t key, uint32_t mask) {
    uint32_t h = static_cast<uint32_t>(key) * 0x9E3779B1u;
    h ^= h >> 15;
    return h & mask;
}

// Voxel keys (clusterer.cpp:102-120, flatVoxelIndex clusterer.hpp:135-141)
// inserted into the per-frame hash set.
constexpr int kVoxRows = 2;  // obstacles per thread: rows of blockDim.x, their atomics in flight together

// Obstacles tile * kVoxRows * blockDim.x + s * blockDim.x + threadIdx.x for
// the rows s: lanes of a wavefront hold consecutive obstacles.
__device__ __forceinline__ void voxel_insert_tile(const DevBuf& d, const Layout& L, int f, int tile) {
    const int nobs = static_cast<int>(d.fs[f * kFsCount + kFsObstacles]);
    const int base = tile * kVoxRows * static_cast<int>(blockDim.x);
    if (base >= nobs) return;
    const CluConst cc = *d.cc;
    const Dims dm = dims_of(d, f, cc);
    const size_t ob = (size_t)f * L.N;
    const uint32_t mask = static_cast<uint32_t>(L.hash_cap) - 1;
    const size_t ho = (size_t)f * L.hash_cap;
    const int lane = lane_id();
    int k[kVoxRows];
    int32_t key[kVoxRows];
#pragma unroll
    for (int s = 0; s < kVoxRows; ++s) {
        k[s] = base + s * static_cast<int>(blockDim.x) + static_cast<int>(threadIdx.x);
        key[s] = -2;  // past the obstacles: never a voxel key (keys are non-negative), inserts nothing
        if (k[s] < nobs) {
            const int32_t ri = static_cast<int32_t>(d.sr[ob + k[s]] / cc.res_r);
            const int32_t ai = static_cast<int32_t>(d.sa[ob + k[s]] / cc.res_az);
            const int32_t ei = static_cast<int32_t>(d.se[ob + k[s]] / cc.res_el);
            key[s] = dm.nr * (dm.na * ei + ai) + ri;
        }
    }
    // A run of lanes with the same voxel inserts once: its lowest lane (which
    // holds the run's smallest point index, lanes follow point order) probes
    // and records the run's count and minimum index; all runs of both rows
    // at once.
    WaveRun run[kVoxRows];
    bool lead[kVoxRows];
    uint32_t h[kVoxRows];
    int32_t prev[kVoxRows];
#pragma unroll
    for (int s = 0; s < kVoxRows; ++s) {
        run[s] = wave_runs(key[s]);
        lead[s] = lane == run[s].leader && key[s] >= 0;
        h[s] = hash_slot(key[s], mask);
        prev[s] = lead[s] ? atomicCAS(&d.hslot[ho + h[s]].key, -1, key[s]) : key[s];
    }
#pragma unroll
    for (int s = 0; s < kVoxRows; ++s) {
        for (uint32_t probe = 1; probe <= mask && prev[s] != -1 && prev[s] != key[s]; ++probe) {
            h[s] = (h[s] + 1) & mask;
            prev[s] = atomicCAS(&d.hslot[ho + h[s]].key, -1, key[s]);
        }
    }
    bool fresh[kVoxRows];
#pragma unroll
    for (int s = 0; s < kVoxRows; ++s) {
        fresh[s] = lead[s] && prev[s] == -1;
        if (lead[s]) {
            atomicMin(&d.hslot[ho + h[s]].aux, k[s]);
            atomicAdd(&d.hslot[ho + h[s]].count, run[s].count);
        }
    }
    // Dense ids of the new voxels, in any order.
    uint32_t pos[kVoxRows];
    __shared__ uint32_t rsv[1024 / kWave + 1];
    block_reserve<kVoxRows>(&d.fs[f * kFsCount + kFsVoxels], fresh, pos, rsv);
#pragma unroll
    for (int s = 0; s < kVoxRows; ++s) {
        if (fresh[s]) {
            if (pos[s] < static_cast<uint32_t>(L.N)) {
                d.vlist[ob + pos[s]] = static_cast<int32_t>(h[s]);
                d.vpar[ob + pos[s]] = static_cast<int32_t>(pos[s]);
                d.vmin[ob + pos[s]] = 0x7fffffff;
                d.vcnt[ob + pos[s]] = 0;
            }
            d.hslot[ho + h[s]].dense = static_cast<int32_t>(pos[s]);
        }
        const int32_t slot = static_cast<int32_t>(__shfl(h[s], run[s].leader, kWave));
        if (k[s] < nobs) d.vslot[ob + k[s]] = slot;
    }
}

__global__ void k_voxel_insert(DevBuf d, Layout L) {
    int tile, f;
    xcd_tile_frame(tile, f);
    voxel_insert_tile(d, L, f, tile);
}

__global__ __launch_bounds__(256) void k_voxel_insert_q(DevBuf d, Layout L, int B) {
    wq_run(d.wq + kWqVoxelInsert * 8, B, kVoxRows * blockDim.x,
           [&](int f) { return d.fs[f * kFsCount + kFsObstacles]; },
           [&](int f, int t) { voxel_insert_tile(d, L, f, t); });
}

// ---- union-find in LDS ----------------------------------------------------
__device__ __forceinline__ int32_t lds_find(volatile int32_t* par, int32_t x) {
    for (;;) {
        const int32_t p = par[x];
        if (p == x) return x;
        const int32_t gp = par[p];
        if (gp == p) return p;
        par[x] = gp;  // path halving; x is not a root, so no CAS targets it
        x = gp;
    }
}

// Joins the trees of a and b, climbing both at once; returns a node of the
// joined tree near its root, where the voxel's next join starts.
__device__ __forceinline__ int32_t lds_union(int32_t* parents, int32_t a, int32_t b) {
    volatile int32_t* par = parents;
    while (a != b) {
        const int32_t pa = par[a], pb = par[b];
        if (pa == a && pb == b) {
            const int32_t lo = min(a, b), hi = max(a, b);
            const int32_t old = atomicCAS(parents + hi, hi, lo);  // hook the larger root under the smaller
            if (old == hi) return lo;
            a = lo;
            b = old;
        } else {
            const int32_t ga = par[pa], gb = par[pb];
            if (ga != pa) par[a] = ga;  // path halving; a is no root any more, so no CAS targets it
            if (gb != pb) par[b] = gb;
            a = ga;
            b = gb;
        }
    }
    return a;
}

// ---- union-find in global memory -------------------------------------------
__device__ __forceinline__ int32_t load_parent(const int32_t* p, int32_t x) {
    return __hip_atomic_load(p + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int32_t g_find(int32_t* parent, int32_t x) {
    int32_t p = load_parent(parent, x);
    while (p != x) {
        const int32_t gp = load_parent(parent, p);
        if (gp != p) atomicCAS(parent + x, p, gp);
        x = p;
        p = gp;
    }
    return x;
}

// Joins the trees of a and b; returns a node of the joined tree at or above a
// (its root when last looked at, unless a was none to begin with).
__device__ __forceinline__ int32_t g_union(int32_t* parent, int32_t a, int32_t b) {
    for (;;) {
        b = g_find(parent, b);
        if (a == b) return a;
        const int32_t hi = a > b ? a : b, lo = a > b ? b : a;
        const int32_t old = atomicCAS(parent + hi, hi, lo);  // hook the larger root under the smaller
        if (old == hi) return lo;
        // The larger is no root any more: go on from its parent.
        a = lo;
        b = old;
        a = g_find(parent, a);
    }
}

// Forward neighbours of every voxel, looked up in the hash by the whole grid
// (the lookups are independent).  The dense ids of those to join it with go to
// vnb, the list ended by -1, for the union-find in LDS; a frame with more
// voxels than that holds joins them here, in global memory.  (That way for
// every frame keeps more of the chip busy than one workgroup per frame, but
// its chains of dependent loads cost more than the LDS ones at any size:
// neighbours and components 68 us against 37 for one 64x2048 frame, 76 against
// 70 for the 30 thousand voxels of a 128x2048 one, 74 against 42 for eight
// frames at a time.)
__global__ __launch_bounds__(256) void k_voxel_neighbours(DevBuf d, Layout L) {
    int tile, f;
    xcd_tile_frame(tile, f);
    // Voxel capacity (the reference's StaticUnorderedMap throws past it).
    if (tile == 0 && threadIdx.x == 0 && static_cast<int32_t>(d.fs[f * kFsCount + kFsVoxels]) > d.cc->max_voxels)
        atomicOr(&d.fs[f * kFsCount + kFsErr], kErrVoxelOverflow);
    const uint32_t U = min(d.fs[f * kFsCount + kFsVoxels], static_cast<uint32_t>(L.N));
    const uint32_t v = tile * blockDim.x + threadIdx.x;
    if (v >= U) return;
    const CluConst cc = *d.cc;
    const Dims dm = dims_of(d, f, cc);
    const size_t ob = (size_t)f * L.N;
    const size_t ho = (size_t)f * L.hash_cap;
    const uint32_t mask = static_cast<uint32_t>(L.hash_cap) - 1;
    const int32_t key = d.hslot[ho + d.vlist[ob + v]].key;
    // Neighbour q of the voxel (clusterer.cpp:150-176 bounds: range and
    // elevation in [0, num), azimuth wraps by one step) is its dense id, or -1
    // if that voxel is empty.  All 13 first probes are issued before any is
    // waited on (collisions, rare at the table's load, probe on afterwards).
    const int32_t ri = key % dm.nr;
    const int32_t rest = key / dm.nr;
    const int32_t ai = rest % dm.na;
    const int32_t ei = rest / dm.na;
    int32_t nk[13];
    uint32_t h[13];
    HashSlot rec[13];
#pragma unroll
    for (int q = 0; q < 13; ++q) {
        const int32_t rr = ri + kHalfNb[q][0];
        const int32_t ee = ei + kHalfNb[q][2];
        int32_t aa = ai + kHalfNb[q][1];
        if (aa < 0)
            aa += dm.na;
        else if (aa >= dm.na)
            aa -= dm.na;
        nk[q] = (rr < 0 || rr >= dm.nr || ee < 0 || ee >= dm.ne) ? -1 : dm.nr * (dm.na * ee + aa) + rr;
        h[q] = hash_slot(nk[q], mask);
        rec[q] = HashSlot{-1, 0u, -1, 0};
        if (nk[q] >= 0) rec[q] = d.hslot[ho + h[q]];
    }
    uint32_t found = 0;
#pragma unroll
    for (int q = 0; q < 13; ++q) {
        for (uint32_t probe = 1; probe <= mask && nk[q] >= 0 && rec[q].key != nk[q] && rec[q].key != -1; ++probe) {
            h[q] = (h[q] + 1) & mask;
            rec[q] = d.hslot[ho + h[q]];
        }
        if (nk[q] >= 0 && rec[q].key == nk[q]) found |= 1u << q;
    }
    const uint32_t joins = joins_of(found);
    if (U <= static_cast<uint32_t>(kCcLds)) {
        int32_t* nb = d.vnb + ob * 8;
        size_t at = v;
#pragma unroll
        for (int q = 0; q < 13; ++q) {
            if (!((joins >> q) & 1u)) continue;
            nb[at] = rec[q].dense;
            at += L.N;
        }
        nb[at] = -1;
    } else {
        int32_t a = static_cast<int32_t>(v);
#pragma unroll
        for (int q = 0; q < 13; ++q)
            if ((joins >> q) & 1u) a = g_union(d.vpar + ob, a, rec[q].dense);
    }
}

// Components of the frames whose voxels fit in LDS.  The loads of a voxel's
// joins and the chains of its finds are what this waits for: with all of up to
// thirteen neighbours joined, each loaded when its turn came, it took 43 us
// for one 64x2048 frame and 101 us for the 30 thousand voxels of a 128x2048
// one; 22 and 54 us with the joins chosen and loaded ahead, 21 and 46 with both
// ends of a join climbing together.
__global__ __launch_bounds__(1024) void k_voxel_cc(DevBuf d, Layout L) {
    __shared__ int32_t par[kCcLds];
    const int f = blockIdx.x;
    const int tid = threadIdx.x;
    const uint32_t U = min(d.fs[f * kFsCount + kFsVoxels], static_cast<uint32_t>(L.N));
    if (U > static_cast<uint32_t>(kCcLds)) return;
    const size_t ob = (size_t)f * L.N;
    const int32_t* nb = d.vnb + ob * 8;
    for (uint32_t v = tid; v < U; v += 1024) par[v] = static_cast<int32_t>(v);
    __syncthreads();
    // The first joins of the next voxel are loaded while this one's are made.
    constexpr int kFirst = 4;
    int32_t next[kFirst];
    auto load = [&](uint32_t v) {
#pragma unroll
        for (int q = 0; q < kFirst; ++q) next[q] = v < U ? nb[(size_t)q * L.N + v] : -1;
    };
    load(tid);
    for (uint32_t v = tid; v < U; v += 1024) {
        int32_t u[kFirst];
#pragma unroll
        for (int q = 0; q < kFirst; ++q) u[q] = next[q];
        load(v + 1024);
        bool more = true;
        int32_t a = static_cast<int32_t>(v);
#pragma unroll
        for (int q = 0; q < kFirst; ++q) {
            more = more && u[q] >= 0;
            if (more) a = lds_union(par, a, u[q]);
        }
        for (int q = kFirst; more && q < kMaxJoins; ++q) {
            const int32_t w = nb[(size_t)q * L.N + v];
            more = w >= 0;
            if (more) a = lds_union(par, a, w);
        }
    }
    __syncthreads();
    for (uint32_t v = tid; v < U; v += 1024) d.vpar[ob + v] = lds_find(par, static_cast<int32_t>(v));
}

// Component minimum point index and point count (removeSmallClusters counts
// points, clusterer.cpp:214-220): one atomic per voxel; the list of the roots;
// and every voxel's root in its hash slot, where its points find it.  After
// the global-memory union-find the roots are found first (all unions are done,
// so concurrent finds only shorten paths within one tree); the LDS union-find
// leaves the parents compressed already.
__global__ __launch_bounds__(256) void k_voxel_stats(DevBuf d, Layout L) {
    __shared__ uint32_t rsv[256 / kWave + 1];
    const int f = blockIdx.y;
    const uint32_t U = min(d.fs[f * kFsCount + kFsVoxels], static_cast<uint32_t>(L.N));
    if (blockIdx.x * blockDim.x >= U) return;
    const uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
    const size_t ob = (size_t)f * L.N;
    const size_t ho = (size_t)f * L.hash_cap;
    int32_t r = -1;
    int32_t mn = 0x7fffffff;
    uint32_t cnt = 0;
    if (v < U) {
        const size_t slot = ho + d.vlist[ob + v];
        const HashSlot hv = d.hslot[slot];
        mn = hv.aux;
        cnt = hv.count;
        r = U > static_cast<uint32_t>(kCcLds) ? g_find(d.vpar + ob, static_cast<int32_t>(v)) : d.vpar[ob + v];
        d.hslot[slot].dense = r;
    }
    // Voxels numbered one after the other mostly share a component: each run
    // of equal roots in the wavefront reduces its minimum and count first
    // (a segmented reduction down the run) and its leader adds them, so a
    // large component's root takes one atomic pair per run, not per voxel.
    const WaveRun run = wave_runs(r);
    const int lane = lane_id();
    const int end = run.leader + static_cast<int>(run.count);  // one past the run's last lane
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const int32_t omn = __shfl_down(mn, o, kWave);
        const uint32_t ocnt = __shfl_down(cnt, o, kWave);
        if (lane + o < end) {
            mn = min(mn, omn);
            cnt += ocnt;
        }
    }
    if (r >= 0 && lane == run.leader) {
        atomicMin(&d.vmin[ob + r], mn);
        atomicAdd(&d.vcnt[ob + r], cnt);
    }
    const bool root[1] = {v < U && r == static_cast<int32_t>(v)};
    uint32_t pos[1];
    block_reserve<1>(&d.fs[f * kFsCount + kFsRoots], root, pos, rsv);
    if (root[0]) d.vroots[ob + pos[0]] = r;
}

__device__ __forceinline__ int32_t root_of_point(const DevBuf& d, size_t ob, size_t ho, int k) {
    return d.hslot[ho + d.vslot[ob + k]].dense;
}

// Clusters in the order of their first point (the reference numbers them in
// input order): a component is a cluster when it has at least min_size points,
// and its first point is its minimum obstacle index.  Two forms, by the number
// of obstacles a frame can have (launch_cluster):
//
// Up to kRankPoints: one workgroup per frame marks the first points of the
// frame's components in an LDS bitmap, ranks them by the bits before them, and
// writes each cluster's size, member offset and empty cursors and each root's
// label (standalone, the labels only).  A frame has a few hundred components,
// for which the two passes below and the offsets' scan took 22 us of a 64x2048
// frame and this takes 5.  Where nearly every point is a component, it waits
// for the roots' gathers, eight a thread in flight: a standalone call with
// 200 000 isolated points takes 264 us, 387 with one gather at a time.
constexpr int kRankThreads = 1024;
constexpr int kRankItems = 8;
constexpr int kRankWords = kRankThreads * kRankItems;
constexpr int kRankPoints = kRankWords * 32;
constexpr int kRankRoots = 8;  // roots per thread and turn

// visit(root, first point, size) for every component, R roots per thread and
// turn.  (Most frames have one turn of one root: the unrolled code, cold in
// every launch, would cost them 0.7 us.)
template <int R, typename Visit>
__device__ __forceinline__ void for_components(const DevBuf& d, size_t ob, int roots, Visit visit) {
    for (int i0 = threadIdx.x; i0 < roots; i0 += kRankThreads * R) {
        int32_t r[R], first[R];
        uint32_t size[R];
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const int i = i0 + u * kRankThreads;
            r[u] = i < roots ? d.vroots[ob + i] : -1;
        }
#pragma unroll
        for (int u = 0; u < R; ++u) {
            if (r[u] < 0) continue;
            first[u] = d.vmin[ob + r[u]];
            size[u] = d.vcnt[ob + r[u]];
        }
#pragma unroll
        for (int u = 0; u < R; ++u)
            if (r[u] >= 0) visit(r[u], first[u], size[u]);
    }
}

// Member offsets: the exclusive sums of the K sizes, R per thread and turn.
template <int R>
__device__ __forceinline__ void member_offsets(const DevBuf& d, size_t ob, int K, uint32_t* lds) {
    uint32_t off = 0;
    for (int base = 0; base < K; base += kRankThreads * R) {
        const int b = base + static_cast<int>(threadIdx.x) * R;
        uint32_t v[R];
        uint32_t mine = 0;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            v[k] = b + k < K ? d.cl_size[ob + b + k] : 0u;
            mine += v[k];
        }
        uint32_t total;
        uint32_t at = block_exclusive_sum<kRankThreads>(mine, lds, &total) + off;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            if (b + k < K) d.cl_off[ob + b + k] = at;
            at += v[k];
        }
        off += total;
    }
}

template <bool kOffsets>
__global__ __launch_bounds__(kRankThreads) void k_component_rank(DevBuf d, Layout L) {
    __shared__ uint32_t bits[kRankWords];
    __shared__ uint32_t before[kRankWords];
    __shared__ uint32_t lds[kRankThreads / kWave + 1];
    const int f = blockIdx.x;
    const int tid = threadIdx.x;
    const int roots = static_cast<int>(d.fs[f * kFsCount + kFsRoots]);
    const uint32_t min_size = d.cc->min_size;
    const size_t ob = (size_t)f * L.N;
    // visit(root, first point, size) for every component.
    auto components = [&](auto visit) {
        if (roots <= 2 * kRankThreads)
            for_components<1>(d, ob, roots, visit);
        else
            for_components<kRankRoots>(d, ob, roots, visit);
    };
    for (int q = tid; q < kRankWords; q += kRankThreads) bits[q] = 0;
    __syncthreads();
    components([&](int32_t, int32_t at, uint32_t size) {
        if (size >= min_size) atomicOr(&bits[at >> 5], 1u << (at & 31));
    });
    __syncthreads();
    uint32_t sum = 0;
#pragma unroll
    for (int k = 0; k < kRankItems; ++k) sum += static_cast<uint32_t>(__popc(bits[tid * kRankItems + k]));
    uint32_t clusters;
    uint32_t ex = block_exclusive_sum<kRankThreads>(sum, lds, &clusters);
#pragma unroll
    for (int k = 0; k < kRankItems; ++k) {
        before[tid * kRankItems + k] = ex;
        ex += static_cast<uint32_t>(__popc(bits[tid * kRankItems + k]));
    }
    __syncthreads();
    components([&](int32_t r, int32_t at, uint32_t size) {
        if (size < min_size) {
            d.vlab[ob + r] = -1;
            return;
        }
        const uint32_t lab = before[at >> 5] + static_cast<uint32_t>(__popc(bits[at >> 5] & ((1u << (at & 31)) - 1u)));
        if (kOffsets) {
            d.cl_size[ob + lab] = size;
            d.cl_cursor[ob + lab] = 0;
            d.hc_count[ob + lab] = 0;  // the round-0 hull input count (first buffer)
        }
        d.vlab[ob + r] = static_cast<int32_t>(lab);
    });
    if (tid == 0) d.fs[f * kFsCount + kFsClusters] = clusters;
    if (!kOffsets) return;
    __syncthreads();
    const int K = static_cast<int>(clusters);
    if (K <= kRankThreads)
        member_offsets<1>(d, ob, K, lds);
    else
        member_offsets<kRankItems>(d, ob, K, lds);
}

// Beyond kRankPoints: two passes of the whole grid over tiles of 2048
// obstacles (eight rows of 256), the first points of every tile and then their
// numbers after the tiles before; the offsets are scanned afterwards.  (The
// form above in turns of kRankPoints, each over all components, took 6.1 ms of
// a standalone call with a million isolated points and 74 ms with four million;
// with these the calls take 0.84 and 3.3 ms.)
constexpr int kCompThreads = 256;
constexpr int kCompRows = 8;
constexpr int kCompTile = kCompThreads * kCompRows;

// The thread's points that are a component's first, of them the clusters'.
__device__ __forceinline__ uint32_t first_points(const DevBuf& d, size_t ob, size_t ho, int base, int nobs,
                                                 uint32_t min_size, int32_t (&root)[kCompRows],
                                                 uint32_t (&size)[kCompRows], uint32_t& clusters) {
    uint32_t m = 0;
    clusters = 0;
#pragma unroll
    for (int k = 0; k < kCompRows; ++k) {
        const int q = base + k * kCompThreads + static_cast<int>(threadIdx.x);
        if (q >= nobs) continue;
        root[k] = root_of_point(d, ob, ho, q);
        size[k] = d.vcnt[ob + root[k]];
        if (d.vmin[ob + root[k]] != q) continue;
        m |= 1u << k;
        if (size[k] >= min_size) clusters |= 1u << k;
    }
    return m;
}

__global__ __launch_bounds__(kCompThreads) void k_component_count(DevBuf d, Layout L) {
    __shared__ uint32_t lds[kCompThreads / kWave + 1];
    const int f = blockIdx.y;
    const int nobs = static_cast<int>(d.fs[f * kFsCount + kFsObstacles]);
    const int base = blockIdx.x * kCompTile;
    if (base >= nobs) return;
    int32_t root[kCompRows];
    uint32_t size[kCompRows], clusters;
    first_points(d, (size_t)f * L.N, (size_t)f * L.hash_cap, base, nobs, d.cc->min_size, root, size, clusters);
    uint32_t total;
    block_exclusive_sum<kCompThreads>(static_cast<uint32_t>(__popc(clusters)), lds, &total);
    if (threadIdx.x == 0) d.blk[(size_t)f * L.blk_stride + blockIdx.x] = total;
}

__global__ __launch_bounds__(kCompThreads) void k_component_number(DevBuf d, Layout L) {
    __shared__ uint32_t lds[kCompRows * kCompThreads / kWave + 1];
    const int f = blockIdx.y;
    const int nobs = static_cast<int>(d.fs[f * kFsCount + kFsObstacles]);
    const int tile = blockIdx.x;
    const int base = tile * kCompTile;
    if (base >= nobs) {
        if (tile == 0 && threadIdx.x == 0) d.fs[f * kFsCount + kFsClusters] = 0;
        return;
    }
    const uint32_t* blk = d.blk + (size_t)f * L.blk_stride;
    uint32_t pre = 0;
    for (int i = threadIdx.x; i < tile; i += kCompThreads) pre += blk[i];
    uint32_t pre_total;
    block_exclusive_sum<kCompThreads>(pre, lds, &pre_total);
    const size_t ob = (size_t)f * L.N;
    int32_t root[kCompRows];
    uint32_t size[kCompRows], clusters;
    const uint32_t first = first_points(d, ob, (size_t)f * L.hash_cap, base, nobs, d.cc->min_size, root, size, clusters);
    uint32_t pos[kCompRows];
    const uint32_t total = tile_compact<kCompThreads, kCompRows>(clusters, pos, lds);
#pragma unroll
    for (int k = 0; k < kCompRows; ++k) {
        if (!((first >> k) & 1u)) continue;
        const uint32_t lab = pre_total + pos[k];
        const bool cluster = (clusters >> k) & 1u;
        d.vlab[ob + root[k]] = cluster ? static_cast<int32_t>(lab) : -1;
        if (!cluster) continue;
        d.cl_size[ob + lab] = size[k];
        d.cl_cursor[ob + lab] = 0;
        d.hc_count[ob + lab] = 0;
    }
    if (threadIdx.x == 0 && base + kCompTile >= nobs) d.fs[f * kFsCount + kFsClusters] = pre_total + total;
}

// True when the obstacle at input index i (pixel pix of a frame W pixels
// wide) has, in the two range-image rows above it in its column, obstacles
// of its own cluster with exactly its x and y.  Vertical surfaces repeat one
// (x, y) down a column; such a point is never a hull vertex while a copy of
// it stays in the hull input, and down every column run of copies the top
// two never pass this test, so each run keeps two copies (a cluster of one
// repeated point keeps the two copies the reference returns for it).
__device__ __forceinline__ bool column_repeat(const DevBuf& d, const Layout& L, const FrameDesc& fd, size_t ob,
                                              size_t ho, int k, int i, float x, float y, int32_t root) {
    const int pix = d.pt_pix[fd.pt_off + i];
    const int W = fd.sc.W;
    const bool inside = pix >= 2 * W;
    const unsigned long long imask = (1ull << L.idx_bits) - 1;
    // Both rows' loads go out together; a row that is out of the question
    // loads this point's own values.
    bool same[2];
    int at[2];
    int32_t r[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const unsigned long long key = inside ? d.pix_key[fd.pix_off + pix - (q + 1) * W] : ~0ull;
        same[q] = key != ~0ull;
        at[q] = same[q] ? static_cast<int>(key & imask) : i;
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int g = fd.pt_off + at[q];
        const uint32_t lab = d.labels[g], o = d.cl_flag[ob + at[q]];
        const float px = d.x[g], py = d.y[g];
        same[q] = same[q] && lab == LP_LABEL_OBSTACLE && px == x && py == y;
        at[q] = same[q] ? static_cast<int>(o) : k;
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) r[q] = root_of_point(d, ob, ho, at[q]);
    return same[0] && same[1] && r[0] == root && r[1] == root;
}

// Every obstacle's cluster label; with kScatter also the members of each
// cluster (unordered within the cluster) and the round-0 hull input: the
// cluster's points as PointXY doubles (processor.cpp:647), less the column
// repeats (their own count, in the first hull buffer).  A thread waits for
// its chain of dependent loads, so the point's label, the rows above it and
// then both counters are each read side by side (labels and scatter of one
// 64x2048 frame 22 -> 12.5 us).
template <bool kScatter>
__global__ void k_cluster_label(DevBuf d, Layout L) {
    const int f = blockIdx.y;
    const int nobs = static_cast<int>(d.fs[f * kFsCount + kFsObstacles]);
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nobs) return;
    const size_t ob = (size_t)f * L.N;
    const size_t ho = (size_t)f * L.hash_cap;
    const int32_t r = root_of_point(d, ob, ho, k);
    if (!kScatter) {
        d.clabel[ob + k] = d.vlab[ob + r];
        return;
    }
    const float x = d.ox[ob + k], y = d.oy[ob + k];
    const bool repeat = column_repeat(d, L, d.frames[f], ob, ho, k, d.obs_src[ob + k], x, y, r);
    const int32_t lab = d.vlab[ob + r];
    d.clabel[ob + k] = lab;
    // The lanes of one cluster take their places together: one atomic pair for
    // each cluster in the wavefront.
    const uint64_t all = __ballot(1), inputs = __ballot(!repeat);
    uint64_t mine = 0;
    for (uint64_t left = all & __ballot(lab >= 0); left;) {
        const int32_t one = __builtin_amdgcn_readlane(lab, __ffsll(static_cast<unsigned long long>(left)) - 1);
        const uint64_t group = __ballot(lab == one);
        if (lab == one) mine = group;
        left &= ~group;
    }
    if (lab < 0) return;
    const int lane = lane_id();
    const uint64_t below = (1ull << lane) - 1ull;
    const int leader = __ffsll(static_cast<unsigned long long>(mine)) - 1;
    const uint32_t off = d.cl_off[ob + lab];
    uint32_t mpos = 0, hpos = 0;
    if (lane == leader) {
        mpos = atomicAdd(&d.cl_cursor[ob + lab], static_cast<uint32_t>(__popcll(mine)));
        hpos = atomicAdd(&d.hc_count[ob + lab], static_cast<uint32_t>(__popcll(mine & inputs)));
    }
    mpos = off + __shfl(mpos, leader, kWave) + static_cast<uint32_t>(__popcll(mine & below));
    hpos = off + __shfl(hpos, leader, kWave) + static_cast<uint32_t>(__popcll(mine & inputs & below));
    d.cl_members[ob + mpos] = k;
    if (repeat) return;
    d.hcx[ob + hpos] = static_cast<double>(x);
    d.hcy[ob + hpos] = static_cast<double>(y);
    d.hci[ob + hpos] = k;
}

void launch_cluster(lp_context* c, int B, bool from_split) {
    DevBuf& d = c->d;
    const Layout& L = c->L;
    hipStream_t st = c->stream;
    const int nb = (L.N + 255) / 256;
    stage_mark(c, "split");
    if (from_split) {
        hipLaunchKernelGGL(k_obs_gather, dim3((L.N + kObsTile - 1) / kObsTile, B), dim3(kObsThreads), 0, st, d, L);
        if (c->clouds_on) {
            launch_scan(c, B, d.gnd_flag, d.obs_flag, L.N, kCountPoints, 0, kFsGround);
            hipLaunchKernelGGL(k_label_split, dim3(nb, B), dim3(256), 0, st, d, L);
        }
    } else {
        hipLaunchKernelGGL(k_cluster_input, dim3(nb, B), dim3(256), 0, st, d, L);
    }
    stage_mark(c, "voxels");
    const int wg = c->point_wg;
    if (c->persistent)
        hipLaunchKernelGGL(k_voxel_insert_q, dim3(kPersistentWorkgroups), dim3(wg), 0, st, d, L, B);
    else
        hipLaunchKernelGGL(k_voxel_insert, dim3((L.N + kVoxRows * wg - 1) / (kVoxRows * wg), B), dim3(wg), 0, st, d,
                           L);
    stage_mark(c, "components");
    hipLaunchKernelGGL(k_voxel_neighbours, dim3(nb, B), dim3(256), 0, st, d, L);
    hipLaunchKernelGGL(k_voxel_cc, dim3(B), dim3(1024), 0, st, d, L);
    hipLaunchKernelGGL(k_voxel_stats, dim3(nb, B), dim3(256), 0, st, d, L);
    // Obstacles a frame can have: of the split, each has a pixel of its own (by
    // the capacity, so that a graph holds for every batch); standalone, the
    // cloud's points.
    const int most = from_split ? std::min(L.N, L.P) : c->frames.front().n;
    if (most > kRankPoints) {
        const int ct = (L.N + kCompTile - 1) / kCompTile;
        hipLaunchKernelGGL(k_component_count, dim3(ct, B), dim3(kCompThreads), 0, st, d, L);
        hipLaunchKernelGGL(k_component_number, dim3(ct, B), dim3(kCompThreads), 0, st, d, L);
        if (from_split) launch_scan(c, B, d.cl_size, d.cl_off, L.N, kCountSlot, kFsClusters, -1);
    } else if (from_split) {
        hipLaunchKernelGGL(k_component_rank<true>, dim3(B), dim3(kRankThreads), 0, st, d, L);
    } else {
        hipLaunchKernelGGL(k_component_rank<false>, dim3(B), dim3(kRankThreads), 0, st, d, L);
    }
    if (from_split) {
        hipLaunchKernelGGL(k_cluster_label<true>, dim3(nb, B), dim3(256), 0, st, d, L);
    } else {
        hipLaunchKernelGGL(k_cluster_label<false>, dim3(nb, B), dim3(256), 0, st, d, L);
    }
    // The hull stage clears the voxel table; here nothing follows.
    if (!from_split) launch_hash_reset(c, B, d.vlist, kFsVoxels);
}

}  // namespace lp
