// lp_api.hip -- context, staging, launch sequence and the C ABI.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "lp_kernels.h"

namespace {

thread_local std::string g_last_error;

int fail(int code, const std::string& msg) {
    g_last_error = msg;
    return code;
}

#define LP_HIP(call)                                                                         \
    do {                                                                                     \
        hipError_t e_ = (call);                                                              \
        if (e_ != hipSuccess) return fail(LP_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

constexpr float kDegToRad = static_cast<float>(M_PI / 180.0);  // segmenter.hpp:135
constexpr float kTwoPi = static_cast<float>(2.0 * M_PI);        // segmenter.hpp:136

int ceil_log2(int64_t v) {
    int b = 0;
    while ((int64_t{1} << b) < v) ++b;
    return b;
}

}  // namespace

namespace lp {

int set_last_error(int code, const char* msg) { return fail(code, msg); }

void stage_mark(lp_context* c, const char* name) {
    if (!c->profiling) return;
    hipEvent_t e;
    if (hipEventCreate(&e) != hipSuccess) return;
    (void)hipEventRecord(e, c->stream);
    c->events.push_back(e);
    c->stage_names.push_back(name);
}

// Derived segmenter constants, computed with host libm in float exactly as
// Segmenter::config / constructPolarGrid / RECM / RANSAC / JCP do.
static bool derive_seg(const lp_segmenter_config& g, const Layout& L, SegConst& s, std::string& why) {
    if (g.image_width <= 0 || g.image_height <= 0 || g.image_width > L.W || g.image_height > L.H) {
        why = "image size outside the context capacity";
        return false;
    }
    s.H = g.image_height;
    s.W = g.image_width;
    s.slice_res = g.grid_slice_resolution_deg * kDegToRad;
    s.rings = static_cast<int32_t>(g.max_distance_m / g.grid_radial_spacing_m);
    s.slices = static_cast<int32_t>(kTwoPi / s.slice_res);
    s.cells = s.rings * s.slices;
    if (s.rings < kRansacRadialBins || s.slices < 1) {
        why = "polar grid needs at least 4 radial rings and one slice";
        return false;
    }
    if (s.cells > L.cell_stride || s.slices * kRansacRadialBins > L.cand_stride ||
        s.slices >= (1 << (32 - L.idx_bits))) {
        why = "polar grid larger than the context capacity";
        return false;
    }
    s.organized = g.assume_unorganized_cloud ? 0 : 1;
    s.zlo = -g.sensor_height_m + g.z_min_m;
    s.zhi = -g.sensor_height_m + g.z_max_m;
    s.spacing = g.grid_radial_spacing_m;
    s.min_d = g.min_distance_m;
    s.max_d = g.max_distance_m;
    const float up = g.elevation_up_deg * kDegToRad;
    s.down_rad = g.elevation_down_deg * kDegToRad;
    s.per_pixel = (up - s.down_rad) / g.image_height;
    s.w_minus_1 = static_cast<float>(g.image_width - 1);
    s.thr = g.ground_height_threshold_m;
    s.two_thr = 2.0F * g.ground_height_threshold_m;
    s.dz = std::min(g.grid_radial_spacing_m * std::tan(g.road_maximum_slope_m_per_m),
                    g.ground_height_threshold_m - FLT_EPSILON);
    s.e0 = -g.sensor_height_m + g.ground_height_threshold_m;
    s.neg_h = -g.sensor_height_m;
    s.cos_max = std::cos(std::tan(g.road_maximum_slope_m_per_m));
    s.kthr2 = g.kernel_threshold_distance_m * g.kernel_threshold_distance_m;
    s.neg_amp = -g.amplification_factor;
    return true;
}

static void derive_clu(const lp_clusterer_config& g, int32_t max_voxels, CluConst& c) {
    c.res_r = g.voxel_grid_range_resolution_m;
    c.res_az = g.voxel_grid_azimuth_resolution_deg * kDegToRad;
    c.res_el = g.voxel_grid_elevation_resolution_deg * kDegToRad;
    c.min_size = g.min_cluster_size;
    c.max_voxels = max_voxels;
}

// De-interleave a raw AoS record buffer into the SoA inputs.
__global__ void k_deinterleave(const uint8_t* raw, int n, int stride, int ox, int oy, int oz, int oring,
                               float* x, float* y, float* z, uint16_t* ring) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint8_t* r = raw + static_cast<size_t>(i) * stride;
    float v;
    memcpy(&v, r + ox, 4);
    x[i] = v;
    memcpy(&v, r + oy, 4);
    y[i] = v;
    memcpy(&v, r + oz, 4);
    z[i] = v;
    if (oring >= 0) {
        uint16_t q;
        memcpy(&q, r + oring, 2);
        ring[i] = q;
    }
}

// Frames one staging launch describes: their descriptors travel as kernel
// arguments (2.7 KB of the 4 KB a launch may carry).
constexpr int kStageFrames = 16;

// A frame's points where the gather reads them: n points, `stride` bytes
// apart; n = 0 when they are copied by other means.
struct StageCloud {
    const uint8_t* x;
    const uint8_t* y;
    const uint8_t* z;
    const uint8_t* ring;
    int32_t stride, ring_stride;
    int32_t n;
};

struct StageArgs {
    FrameDesc fd[kStageFrames];
    StageCloud cl[kStageFrames];
    CluConst cc;
    NoiseConst nc;
    int32_t first;  // index of fd[0] in the batch
};

constexpr int kStageRows = 4;  // points per thread, 256 apart

__device__ __forceinline__ float load_f32(const uint8_t* p) {
    float v;
    memcpy(&v, p, 4);
    return v;
}

__device__ __forceinline__ uint16_t load_u16(const uint8_t* p) {
    uint16_t v;
    memcpy(&v, p, 2);
    return v;
}

// Stages a batch: descriptors and constants from the arguments, and the
// points of the clouds that are in this device's memory, whatever their
// strides.  One launch for up to 16 frames instead of four copies per frame
// and three for the descriptors (a copy costs 3 to 5 us of host time and a
// gap on the stream; the points themselves move at memory speed): staging 128
// frames of 128 k points on four streams takes 65 us of host time and 55 us
// of waiting, one frame 7 + 13 us; with the copies it was several
// milliseconds and about 60 us.
__global__ __launch_bounds__(256) void k_stage(StageArgs a, float* x, float* y, float* z, uint16_t* ring,
                                               FrameDesc* frames, CluConst* cc, NoiseConst* nc) {
    const int f = blockIdx.y;
    if (blockIdx.x == 0) {
        constexpr int kWords = sizeof(FrameDesc) / 4;
        static_assert(sizeof(FrameDesc) % 4 == 0 && kWords <= 256, "one thread per descriptor word");
        if (threadIdx.x < kWords)
            reinterpret_cast<uint32_t*>(frames + a.first + f)[threadIdx.x] =
                reinterpret_cast<const uint32_t*>(&a.fd[f])[threadIdx.x];
        if (f == 0 && threadIdx.x == 0) {
            *cc = a.cc;
            *nc = a.nc;
        }
    }
    const StageCloud& c = a.cl[f];
    const int off = a.fd[f].pt_off;
    const int base = blockIdx.x * (256 * kStageRows) + threadIdx.x;
    float vx[kStageRows], vy[kStageRows], vz[kStageRows];
    uint16_t vr[kStageRows];
#pragma unroll
    for (int k = 0; k < kStageRows; ++k) {
        const int i = base + k * 256;
        if (i >= c.n) continue;
        const size_t o = static_cast<size_t>(i) * c.stride;
        vx[k] = load_f32(c.x + o);
        vy[k] = load_f32(c.y + o);
        vz[k] = load_f32(c.z + o);
        if (c.ring) vr[k] = load_u16(c.ring + static_cast<size_t>(i) * c.ring_stride);
    }
#pragma unroll
    for (int k = 0; k < kStageRows; ++k) {
        const int i = base + k * 256;
        if (i >= c.n) continue;
        x[off + i] = vx[k];
        y[off + i] = vy[k];
        z[off + i] = vz[k];
        if (c.ring) ring[off + i] = vr[k];
    }
}

// One array on its way to the host: `elem` bytes times a count, which is
// fs[frame][slot] (at most `count`) or `count` itself (slot < 0).  The unknown
// cloud (kUnknownCloud) follows the ground cloud in memory and holds what the
// ground and obstacle points leave of that count.
struct OutItem {
    const uint8_t* src;
    uint8_t* dst;   // where the kernel writes: the caller's page-locked memory or the bounce buffer
    uint32_t elem;
    int32_t count;
    int32_t frame;
    int16_t slot;
    int16_t rules;  // OutRule bits
    int32_t hull_capacity;
};
enum OutRule : int16_t {
    kSkipFailed = 1,    // nothing when the frame failed
    kSkipHullOver = 2,  // nothing when the frame has more than hull_capacity hull vertices
    kUnknownCloud = 4
};
constexpr int kOutItems = 64;  // items of one launch (2.6 KB of arguments)
struct OutArgs {
    OutItem item[kOutItems];
};

// Bytes of an item, by the frame's scalars (the same on host and device).
__host__ __device__ inline uint32_t out_bytes(const OutItem& it, const uint32_t* fs) {
    const uint32_t* s = fs + static_cast<size_t>(it.frame) * kFsCount;
    if ((it.rules & kSkipFailed) && (s[kFsErr] | s[kFsNoiseErr]) != 0) return 0;
    const int32_t hull = static_cast<int32_t>(s[kFsHullTotal]);
    if ((it.rules & kSkipHullOver) && hull > 0 && hull > it.hull_capacity) return 0;
    const uint32_t cap = static_cast<uint32_t>(it.count);
    uint32_t n = it.slot < 0 ? cap : (s[it.slot] < cap ? s[it.slot] : cap);
    if (it.rules & kUnknownCloud) {
        const uint32_t known = s[kFsGround] + s[kFsObstacles];
        n = known < n ? n - known : 0u;
    }
    return n * it.elem;
}

__host__ __device__ inline const uint8_t* out_src(const OutItem& it, const uint32_t* fs) {
    const uint32_t skipped = it.rules & kUnknownCloud ? fs[static_cast<size_t>(it.frame) * kFsCount + kFsGround] : 0u;
    return it.src + static_cast<size_t>(skipped) * it.elem;
}

// Writes the outputs of a run straight into host memory: one launch for up to
// 64 arrays, whose sizes it reads on the device, so the host waits once
// instead of once for the counts and once more for a copy per array.  Bound
// by the host link on large batches: 2.5 ms for the 140 MB of 128 full frames
// (56 GB/s; a plain copy reaches 57), where 770 copies took 6; one frame
// 34 us.
__global__ __launch_bounds__(256) void k_copy_out(OutArgs a, const uint32_t* fs) {
    const OutItem& it = a.item[blockIdx.y];
    const uint32_t bytes = out_bytes(it, fs);
    const uint8_t* src = out_src(it, fs);
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t step = gridDim.x * blockDim.x;
    const uintptr_t mix = reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(it.dst);
    uint32_t done = 0;
    if ((mix & 15) == 0) {
        const uint32_t n = bytes / 16;
        for (uint32_t i = t; i < n; i += step)
            reinterpret_cast<uint4*>(it.dst)[i] = reinterpret_cast<const uint4*>(src)[i];
        done = n * 16;
    } else if ((mix & 3) == 0) {
        const uint32_t n = bytes / 4;
        for (uint32_t i = t; i < n; i += step)
            reinterpret_cast<uint32_t*>(it.dst)[i] = reinterpret_cast<const uint32_t*>(src)[i];
        done = n * 4;
    }
    for (uint32_t i = done + t; i < bytes; i += step) it.dst[i] = src[i];
}

}  // namespace lp

using namespace lp;

namespace {

// Kind of the memory around a pointer of the caller, and whether a kernel of
// this device may touch all of [p, p + bytes).  Allocations seen are kept for
// one call only (a batch's arrays mostly share a few allocations).
class CallerMemory {
   public:
    enum Kind { kDevice, kPinned, kPageable, kOther };

    explicit CallerMemory(int device) : device_(device) {}

    // *dev receives the address to use on the device (kDevice, kPinned).
    Kind find(const void* p, size_t bytes, uint8_t** dev) {
        const uintptr_t a = reinterpret_cast<uintptr_t>(p);
        for (const Range& r : ranges_)
            if (a >= r.lo && a + bytes <= r.hi) {
                *dev = reinterpret_cast<uint8_t*>(a + r.delta);
                return r.kind;
            }
        hipPointerAttribute_t at{};
        if (hipPointerGetAttributes(&at, p) != hipSuccess) {
            (void)hipGetLastError();
            return kPageable;  // not known to the runtime
        }
        if (at.type == hipMemoryTypeUnregistered) return kPageable;
        if ((at.type != hipMemoryTypeDevice && at.type != hipMemoryTypeHost) || at.device != device_ ||
            !at.devicePointer)
            return kOther;
        hipDeviceptr_t base = nullptr;
        size_t size = 0;
        if (hipMemGetAddressRange(&base, &size, reinterpret_cast<hipDeviceptr_t>(at.devicePointer)) != hipSuccess) {
            (void)hipGetLastError();
            return kOther;
        }
        const uintptr_t d = reinterpret_cast<uintptr_t>(at.devicePointer);
        const uintptr_t b = reinterpret_cast<uintptr_t>(base);
        if (d < b || d + bytes > b + size) return kOther;
        const Kind kind = at.type == hipMemoryTypeDevice ? kDevice : kPinned;
        ranges_.insert(ranges_.begin(), Range{a - (d - b), a - (d - b) + size, d - a, kind});
        if (ranges_.size() > 16) ranges_.pop_back();
        *dev = reinterpret_cast<uint8_t*>(d);
        return kind;
    }

   private:
    struct Range {
        uintptr_t lo, hi, delta;
        Kind kind;
    };
    int device_;
    std::vector<Range> ranges_;
};

template <typename T>
T* carve(char*& p, size_t count) {
    T* r = reinterpret_cast<T*>(p);
    size_t bytes = (count * sizeof(T) + 255) & ~size_t{255};
    p += bytes;
    return r;
}

size_t layout_bytes(const Layout& L, DevBuf* d, char* base) {
    char* p = base;
    const size_t B = L.B, N = L.N, P = L.P, C = L.cell_stride, HC = L.hash_cap;
    auto go = [&](auto*& dst, size_t count) {
        using T = std::remove_reference_t<decltype(*dst)>;
        T* r = carve<T>(p, count);
        if (d) dst = r;
    };
    DevBuf tmp{};
    DevBuf& x = d ? *d : tmp;
    go(x.x, B * N);
    go(x.y, B * N);
    go(x.z, B * N);
    go(x.ring, B * N);
    go(x.rx, B * N);
    go(x.ry, B * N);
    go(x.rz, B * N);
    go(x.rring, B * N);
    go(x.noise, B * N);
    go(x.dsort, B * N);
    go(x.spos, B * N);
    go(x.nocc, B * kNoiseOccWords);
    go(x.ncell_slot, B * N);
    go(x.pt_cell, B * N);
    go(x.pt_xyzc, B * N);
    go(x.pt_pix, B * N);
    go(x.labels, B * N);
    go(x.obs_flag, B * N);
    go(x.obs_src, B * N);
    go(x.obs_rows, B * static_cast<size_t>(L.obs_rows));
    go(x.ox, B * N);
    go(x.oy, B * N);
    go(x.oz, B * N);
    go(x.sr, B * N);
    go(x.sa, B * N);
    go(x.se, B * N);
    go(x.vslot, B * N);
    go(x.cl_flag, B * N);
    go(x.clabel, B * N);
    x.nloc = x.clabel;
    go(x.cell_count, B * C);
    go(x.cell_start, B * C);
    go(x.pt_loc, B * N);
    go(x.cell_items, B * N);
    go(x.cell_zkey, B * N);
    x.hc_chunk_c = x.cell_items;
    go(x.hc_chunk_b, B * N);
    x.hc_chunk_i = x.cell_zkey;
    go(x.zmin, B * C);
    go(x.elev, B * C);
    go(x.big_cells, B * C);
    go(x.cell_list, B * C);
    go(x.cand_count, B * L.cand_stride);
    go(x.cx, B * N);
    go(x.cy, B * N);
    go(x.cz, B * N);
    go(x.hyp, B * kRansacIters * 4);
    go(x.hyp_valid, B * kRansacIters);
    go(x.hyp_count, B * kRansacIters);
    go(x.mt_raw, kMtRawCount);
    go(x.pix_key, B * P);
    go(x.state, B * P);
    go(x.mapping, B * P);
    go(x.pxyz, B * P);
    go(x.qmask, B * static_cast<size_t>(L.qruns));
    go(x.qmap, B * P);
    go(x.qlist, B * P);
    go(x.qrow, B * (L.H + 1));
    go(x.slot_rec, B * P * (kSlotRecordBytes / sizeof(uint4)));
    go(x.fin, B * P);
    go(x.hslot, B * HC);
    go(x.vlist, B * N);
    go(x.vpar, B * N);
    go(x.vnb, B * N * 8);
    go(x.vmin, B * N);
    go(x.vcnt, B * N);
    go(x.vlab, B * N);
    go(x.cl_size, B * N);
    go(x.cl_off, B * N);
    go(x.cl_cursor, B * N);
    x.hull_flag = x.cl_cursor;
    go(x.cl_members, B * N);
    x.nopen = x.cl_members;
    go(x.hcx, 2 * B * N);
    go(x.hcy, 2 * B * N);
    go(x.hci, 2 * B * N);
    go(x.hc_count, 2 * B * N);
    go(x.hc_open, B * N + 1);  // standalone lists: their offsets, one more than there are lists
    go(x.hull_idx, B * N);
    go(x.hull_count, B * N);
    go(x.hull_off, B * N);
    go(x.hull_local, B * N);
    x.vroots = x.hull_local;
    go(x.blk, B * L.blk_stride);
    go(x.fs, B * kFsCount);
    go(x.wq, kWqCounters);
    go(x.frames, B);
    go(x.cc, 1);
    go(x.nc, 1);
    go(x.boxes, B * static_cast<size_t>(L.box_stride));
    go(x.vclass, B * static_cast<size_t>(L.box_stride));
    return static_cast<size_t>(p - base);
}

// Field offsets of an AoS cloud relative to its lowest field.
struct AosLayout {
    const uint8_t* lo = nullptr;
    int fx = 0, fy = 0, fz = 0, fr = -1;
    int stride = 0;
    int span = 0;   // bytes from `lo` to the end of the last field of a record
};

bool aos_layout(const lp_cloud& cl, AosLayout& a, std::string& why) {
    const uint8_t* lo = static_cast<const uint8_t*>(cl.x);
    for (const void* q : {cl.y, cl.z, cl.ring})
        if (q && static_cast<const uint8_t*>(q) < lo) lo = static_cast<const uint8_t*>(q);
    auto field = [&](const void* q) { return static_cast<int64_t>(static_cast<const uint8_t*>(q) - lo); };
    const int64_t fx = field(cl.x), fy = field(cl.y), fz = field(cl.z), fr = cl.ring ? field(cl.ring) : -1;
    const int64_t stride = cl.xyz_stride;
    if (stride < 12 || fx + 4 > stride || fy + 4 > stride || fz + 4 > stride || (fr >= 0 && fr + 2 > stride) ||
        (cl.ring && cl.ring_stride != stride)) {
        why = "unsupported point layout: fields must share one record stride";
        return false;
    }
    a.lo = lo;
    a.fx = static_cast<int>(fx);
    a.fy = static_cast<int>(fy);
    a.fz = static_cast<int>(fz);
    a.fr = static_cast<int>(fr);
    a.stride = static_cast<int>(stride);
    a.span = static_cast<int>(std::max({fx + 4, fy + 4, fz + 4, fr >= 0 ? fr + 2 : int64_t{0}}));
    return true;
}

// Device bytes at slot_rec used for staging (the records are written after it).
size_t raw_staging_bytes(const lp_context* c) {
    constexpr size_t kPerPixel = 96;
    static_assert(kPerPixel <= kSlotRecordBytes, "the staging area is part of the slot records");
    return static_cast<size_t>(c->L.B) * static_cast<size_t>(c->L.P) * kPerPixel;
}

}  // namespace

namespace lp {

// The per-frame checks lp_batch_stage makes, without staging anything.
int validate_frame(const lp_context* c, const lp_segmenter_config& cfg, const lp_cloud& cl) {
    if (cl.num_points < 0 || cl.num_points > c->L.N)
        return fail(LP_ERR_CAPACITY, "frame has more points than max_points_per_frame");
    if (cl.num_points > 0 && (!cl.x || !cl.y || !cl.z)) return fail(LP_ERR_INVALID_ARGUMENT, "null coordinates");
    SegConst sc{};
    std::string why;
    if (!derive_seg(cfg, c->L, sc, why)) return fail(LP_ERR_INVALID_ARGUMENT, why);
    const bool soa = cl.xyz_stride == 4 && (cl.ring == nullptr || cl.ring_stride == 2);
    if (cl.num_points > 0 && !soa) {
        AosLayout a;
        if (!aos_layout(cl, a, why)) return fail(LP_ERR_INVALID_ARGUMENT, why);
        if (raw_staging_bytes(c) < static_cast<size_t>(a.stride))
            return fail(LP_ERR_CAPACITY, "point record larger than the staging area");
    }
    return LP_OK;
}

}  // namespace lp

namespace {

// Whether k_stage may read the cloud where it is: device memory of this
// device, every field inside its allocation.
bool gathers(CallerMemory& mem, const lp_cloud& cl, StageCloud& g) {
    if (!cl.on_device || cl.num_points == 0 || cl.xyz_stride < 4 || (cl.ring && cl.ring_stride < 2)) return false;
    const size_t last = static_cast<size_t>(cl.num_points) - 1;
    uint8_t *x, *y, *z, *r = nullptr;
    const size_t span = last * static_cast<size_t>(cl.xyz_stride) + 4;
    if (mem.find(cl.x, span, &x) != CallerMemory::kDevice || mem.find(cl.y, span, &y) != CallerMemory::kDevice ||
        mem.find(cl.z, span, &z) != CallerMemory::kDevice ||
        (cl.ring && mem.find(cl.ring, last * static_cast<size_t>(cl.ring_stride) + 2, &r) != CallerMemory::kDevice))
        return false;
    g = StageCloud{x, y, z, r, cl.xyz_stride, cl.ring_stride, cl.num_points};
    return true;
}

// Copies a cloud into the packed inputs (x, y, z, ring at offset `off`) of d.
int stage_cloud(lp_context* c, const DevBuf& d, const lp_cloud& cl, int32_t off, uint8_t* raw_dev) {
    const int n = cl.num_points;
    if (n == 0) return LP_OK;
    const hipMemcpyKind kind = cl.on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice;
    const bool soa = cl.xyz_stride == 4 && (cl.ring == nullptr || cl.ring_stride == 2);
    if (soa) {
        LP_HIP(hipMemcpyAsync(d.x + off, cl.x, n * 4, kind, c->stream));
        LP_HIP(hipMemcpyAsync(d.y + off, cl.y, n * 4, kind, c->stream));
        LP_HIP(hipMemcpyAsync(d.z + off, cl.z, n * 4, kind, c->stream));
        if (cl.ring) LP_HIP(hipMemcpyAsync(d.ring + off, cl.ring, n * 2, kind, c->stream));
        return LP_OK;
    }
    // AoS: all fields inside one record of xyz_stride bytes, staged through
    // the device area at raw_dev in chunks of whole records.
    AosLayout a;
    std::string why;
    if (!aos_layout(cl, a, why)) return fail(LP_ERR_INVALID_ARGUMENT, why);
    const size_t stride = static_cast<size_t>(a.stride);
    const size_t chunk = raw_staging_bytes(c) / stride;
    if (chunk == 0) return fail(LP_ERR_CAPACITY, "point record larger than the staging area");
    for (size_t first = 0; first < static_cast<size_t>(n); first += chunk) {
        const int cnt = static_cast<int>(std::min(chunk, static_cast<size_t>(n) - first));
        // The last record is read up to its last field only: the caller's
        // array may end there.
        const size_t bytes = (static_cast<size_t>(cnt) - 1) * stride + static_cast<size_t>(a.span);
        LP_HIP(hipMemcpyAsync(raw_dev, a.lo + first * stride, bytes, kind, c->stream));
        const int o = off + static_cast<int>(first);
        hipLaunchKernelGGL(k_deinterleave, dim3((cnt + 255) / 256), dim3(256), 0, c->stream, raw_dev, cnt, a.stride,
                           a.fx, a.fy, a.fz, a.fr, d.x + o, d.y + o, d.z + o, d.ring + o);
        LP_HIP(hipGetLastError());
    }
    return LP_OK;
}

// Stages the clouds of c->frames (descriptors ready, constants given) into
// the packed inputs, or into the noise filter's raw inputs when `raw_inputs`.
// Clouds in host memory, or in memory a kernel may not read, are copied (AoS
// records through a device area, free at this point of the pipeline).
int stage_frames(lp_context* c, const lp_cloud* clouds, const CluConst& cc, const NoiseConst& nc, bool raw_inputs) {
    DevBuf d = c->d;
    if (raw_inputs) {
        d.x = d.rx;
        d.y = d.ry;
        d.z = d.rz;
        d.ring = d.rring;
    }
    uint8_t* raw = reinterpret_cast<uint8_t*>(c->d.slot_rec);
    CallerMemory mem(c->device);
    const int B = static_cast<int>(c->frames.size());
    for (int f0 = 0; f0 < B; f0 += kStageFrames) {
        StageArgs a{};
        a.cc = cc;
        a.nc = nc;
        a.first = f0;
        const int cnt = std::min(kStageFrames, B - f0);
        int most = 0;
        for (int k = 0; k < cnt; ++k) {
            const lp_cloud& cl = clouds[f0 + k];
            a.fd[k] = c->frames[f0 + k];
            std::string why;
            AosLayout layout;
            const bool soa = cl.xyz_stride == 4 && (cl.ring == nullptr || cl.ring_stride == 2);
            if (cl.num_points > 0 && !soa) {
                if (!aos_layout(cl, layout, why)) return fail(LP_ERR_INVALID_ARGUMENT, why);
                if (raw_staging_bytes(c) < static_cast<size_t>(layout.stride))
                    return fail(LP_ERR_CAPACITY, "point record larger than the staging area");
            }
            if (gathers(mem, cl, a.cl[k])) {
                most = std::max(most, cl.num_points);
                continue;
            }
            const int st = stage_cloud(c, d, cl, c->frames[f0 + k].pt_off, raw);
            if (st != LP_OK) return st;
        }
        const int tiles = std::max(1, (most + 256 * kStageRows - 1) / (256 * kStageRows));
        hipLaunchKernelGGL(k_stage, dim3(tiles, cnt), dim3(256), 0, c->stream, a, d.x, d.y, d.z, d.ring, d.frames, d.cc,
                           d.nc);
    }
    LP_HIP(hipGetLastError());
    return LP_OK;
}

int run_pipeline(lp_context* c, int B, bool segment_only) {
    c->L.B_active = B;
    const bool radius_rule = c->staged_filtered && !segment_only && !c->noise_kdtree;
    if (c->staged_filtered && !segment_only) {
        if (c->noise_kdtree)
            launch_noise_kdtree(c, B, true);
        else
            launch_noise(c, B, true);
    }
    launch_segment_front(c, B, radius_rule);
    launch_jcp(c, B);
    if (!segment_only) {
        launch_cluster(c, B, true);
        launch_hull(c, B);
        if (c->boxes_on || c->vehicles_on) launch_boxes(c, B);
        if (c->vehicles_on) launch_vehicles(c, B);
    }
    LP_HIP(hipGetLastError());
    return LP_OK;
}

// NoiseRemover::filter constants (noise_remover.cpp:44-48).
NoiseConst noise_const(const lp_noise_config& cfg) {
    NoiseConst nc{};
    nc.scaling = std::pow(static_cast<double>(cfg.radius_multiplier_m_per_m), 2.0);
    nc.min_sqr = cfg.min_search_radius_m * cfg.min_search_radius_m;
    nc.k = cfg.min_neighbours;
    return nc;
}

int status_of(uint32_t err) {
    if (err & kErrVoxelOverflow) return fail(LP_ERR_VOXEL_OVERFLOW, "more occupied voxels than max_voxels");
    if (err & kErrRansacSingle)
        return fail(LP_ERR_RANSAC_SINGLE_CANDIDATE, "exactly one RANSAC candidate (reference never terminates)");
    if (err & kErrNoiseInput)
        return fail(LP_ERR_INVALID_ARGUMENT,
                    "non-finite coordinates: the KD-tree search (std::nth_element) has no order for them");
    if (err & kErrNoiseCapacity)
        return fail(LP_ERR_CAPACITY, "KD-tree noise search: more pending search entries than the device holds");
    if (err & kErrHullFuzzyOrder)
        return fail(LP_ERR_INVALID_ARGUMENT,
                    "hull points with distinct x closer than DBL_EPSILON: the reference's sort comparator "
                    "(polygonizer.cpp:52-59) is not an ordering there");
    if (err & (kErrCellCapacity | kErrQueueCapacity | kErrHullCapacity | kErrRngExhausted | kErrBoxCapacity))
        return fail(LP_ERR_CAPACITY, "a device capacity was exceeded (cell, JCP queue, hull, box or RNG stream)");
    return LP_OK;
}

}  // namespace

namespace {

// Whether kernels of two streams run side by side: one waits for the other's
// mark, for kProbeTicks of the 100 MHz counter at most.
constexpr unsigned long long kProbeTicks = 20000;

__global__ void k_probe_wait(uint32_t* mark, uint32_t* seen) {
    const unsigned long long t0 = wall_clock64();
    uint32_t m = 0;
    for (int i = 0; i < 100000 && !m && wall_clock64() - t0 < kProbeTicks; ++i) {
        m = __hip_atomic_load(mark, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __builtin_amdgcn_s_sleep(8);
    }
    *seen = m;
}

__global__ void k_probe_mark(uint32_t* mark) {
    __hip_atomic_store(mark, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

bool side_by_side(hipStream_t a, hipStream_t b, uint32_t* words) {
    volatile uint32_t* w = words;
    // The first round brings up the kernels and the queues.
    for (int round = 0; round < 2; ++round) {
        w[0] = w[1] = 0;
        hipLaunchKernelGGL(k_probe_wait, dim3(1), dim3(1), 0, a, words, words + 1);
        hipLaunchKernelGGL(k_probe_mark, dim3(1), dim3(1), 0, b, words);
        if (hipStreamSynchronize(b) != hipSuccess || hipStreamSynchronize(a) != hipSuccess) return true;
        if (w[1]) return true;
    }
    return false;
}

}  // namespace

// The runtime has a few hardware queues (four by default) and gives a new
// stream the one with the fewest streams, so after other streams came and went
// two lanes can land on one queue and run one after the other, while another
// queue idles: 32 mixed frames in four lanes 650 us with a queue each, 1090 us
// with two lanes on one.  A stream that shares its queue with an earlier one
// is replaced, by the first of a few new ones that does not; the ones passed
// over go when all are placed, so that each new one lands elsewhere.
int lp::spread_streams(const std::vector<lp_context*>& contexts) {
    constexpr int kTries = 8;
    constexpr size_t kQueues = 4;
    if (contexts.size() < 2) return LP_OK;
    uint32_t* words = nullptr;
    LP_HIP(hipHostMalloc(reinterpret_cast<void**>(&words), 64, hipHostMallocDefault));
    std::vector<hipStream_t> placed, passed;
    int tries = 0;
    hipError_t err = hipSuccess;
    auto alone = [&](hipStream_t s) {
        for (hipStream_t o : placed)
            if (!side_by_side(o, s, words)) return false;
        return true;
    };
    for (lp_context* c : contexts) {
        if (placed.size() == kQueues || tries == kTries || err != hipSuccess) break;
        bool found = alone(c->stream);
        while (!found && tries < kTries) {
            ++tries;
            hipStream_t s = nullptr;
            err = hipStreamCreateWithFlags(&s, hipStreamNonBlocking);
            if (err != hipSuccess) break;
            found = alone(s);
            if (found) std::swap(c->stream, s);
            passed.push_back(s);
        }
        if (found) placed.push_back(c->stream);
    }
    for (hipStream_t s : passed) (void)hipStreamDestroy(s);
    (void)hipHostFree(words);
    LP_HIP(err);
    return LP_OK;
}

extern "C" {

void lp_segmenter_config_default(lp_segmenter_config* c) {
    c->elevation_up_deg = 2.0F;
    c->elevation_down_deg = -24.8F;
    c->image_width = 2048;
    c->image_height = 64;
    c->assume_unorganized_cloud = 0;
    c->grid_radial_spacing_m = 2.0F;
    c->grid_slice_resolution_deg = 1.0F;
    c->ground_height_threshold_m = 0.2F;
    c->road_maximum_slope_m_per_m = 0.2F;
    c->min_distance_m = 2.0F;
    c->max_distance_m = 100.0F;
    c->sensor_height_m = 1.73F;
    c->kernel_threshold_distance_m = 1.0F;
    c->amplification_factor = 5.0F;
    c->z_min_m = -3.0F;
    c->z_max_m = 4.0F;
}

void lp_clusterer_config_default(lp_clusterer_config* c) {
    c->voxel_grid_range_resolution_m = 0.4F;
    c->voxel_grid_azimuth_resolution_deg = 1.0F;
    c->voxel_grid_elevation_resolution_deg = 1.5F;
    c->min_cluster_size = 3;
}

void lp_clusterer_config_shipped(lp_clusterer_config* c) {
    lp_clusterer_config_default(c);
    c->voxel_grid_elevation_resolution_deg = 3.0F;
}

void lp_capacity_default(lp_capacity* cap) {
    cap->max_frames = 1;
    cap->max_points_per_frame = 200000;  // Segmenter::MAX_CLOUD_SIZE, segmenter.hpp:151
    cap->max_image_height = 64;
    cap->max_image_width = 2048;
    cap->max_voxels = 200000;            // clusterer.cpp:36
    cap->device = 0;
    cap->streams = 1;
    cap->hash_load_factor = 0.5F;
}

const char* lp_last_error(void) { return g_last_error.c_str(); }

namespace {

int create_lane(const lp_capacity* cap, lp_context** out);

}  // namespace

int lp_context_create(const lp_capacity* cap, lp_context** out) {
    if (!cap || !out) return fail(LP_ERR_INVALID_ARGUMENT, "null argument");
    *out = nullptr;
    if (cap->streams < 1 || cap->streams > 8) return fail(LP_ERR_INVALID_ARGUMENT, "streams must be 1..8");
    const int S = std::min(cap->streams, std::max(cap->max_frames, 1));
    lp_capacity lc = *cap;
    lc.streams = 1;
    lc.max_frames = (cap->max_frames + S - 1) / S;
    lp_context* c = nullptr;
    int st = create_lane(&lc, &c);
    if (st != LP_OK) return st;
    for (int k = 1; k < S; ++k) {
        lp_context* lane = nullptr;
        st = create_lane(&lc, &lane);
        hipEvent_t ev = nullptr;
        if (st == LP_OK) {
            const hipError_t e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
            if (e != hipSuccess) {
                lp_context_destroy(lane);
                st = fail(LP_ERR_HIP, std::string("lane event: ") + hipGetErrorString(e));
            }
        }
        if (st != LP_OK) {
            lp_context_destroy(c);
            return st;
        }
        c->lanes.push_back(lane);
        c->lane_done.push_back(ev);
    }
    std::vector<lp_context*> lanes{c};
    lanes.insert(lanes.end(), c->lanes.begin(), c->lanes.end());
    st = lp::spread_streams(lanes);
    if (st != LP_OK) {
        lp_context_destroy(c);
        return st;
    }
    *out = c;
    return LP_OK;
}

namespace {

// One lane: buffers, stream and graph cache for cap->max_frames frames.
int create_lane(const lp_capacity* cap, lp_context** out) {
    *out = nullptr;
    if (cap->max_frames < 1 || cap->max_points_per_frame < 1 || cap->max_image_height < 1 ||
        cap->max_image_width < 1 || cap->max_image_height > 1024 || cap->max_voxels < 1)
        return fail(LP_ERR_INVALID_ARGUMENT, "invalid capacity");
    if (!(cap->hash_load_factor >= 0.5F && cap->hash_load_factor <= 0.9F))
        return fail(LP_ERR_INVALID_ARGUMENT, "hash_load_factor must be in [0.5, 0.9]");
    int ndev = 0;
    LP_HIP(hipGetDeviceCount(&ndev));
    if (cap->device < 0 || cap->device >= ndev) return fail(LP_ERR_INVALID_ARGUMENT, "no such HIP device");
    LP_HIP(hipSetDevice(cap->device));
    auto* c = new lp_context();
    c->device = cap->device;
    c->cap = *cap;
    Layout& L = c->L;
    L.B = cap->max_frames;
    L.N = cap->max_points_per_frame;
    L.H = cap->max_image_height;
    L.W = cap->max_image_width;
    L.P = L.H * L.W;
    L.B_active = 0;
    L.idx_bits = std::max(1, ceil_log2(L.N));
    if (L.idx_bits > 24) {
        delete c;
        return fail(LP_ERR_INVALID_ARGUMENT, "max_points_per_frame above 2^24");
    }
    L.cell_stride = 32768;
    L.cand_stride = 4 * 4096;
    // Every point could occupy its own cell or voxel: the table holds N keys
    // at the chosen worst-case load.
    L.hash_cap = 1 << ceil_log2(static_cast<int64_t>(std::ceil(L.N / static_cast<double>(cap->hash_load_factor))));
    L.blk_stride = (L.N + 1023) / 1024 + 1;
    L.box_stride = L.N / 3 + 1024;
    L.obs_rows = (L.N + 63) / 64;
    L.qruns = L.H * ((L.W + 63) / 64);
    const size_t bytes = layout_bytes(L, nullptr, nullptr);
    hipError_t e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipMalloc(&c->arena, bytes);
    if (e != hipSuccess) {
        if (c->stream) (void)hipStreamDestroy(c->stream);
        delete c;
        return fail(LP_ERR_HIP, std::string("context allocation: ") + hipGetErrorString(e));
    }
    c->arena_bytes = bytes;
    layout_bytes(L, &c->d, static_cast<char*>(c->arena));
    launch_mt19937(c->d.mt_raw, kMtRawCount, c->stream);
    launch_hash_init(c);
    e = hipStreamSynchronize(c->stream);
    if (e != hipSuccess) {
        lp_context_destroy(c);
        return fail(LP_ERR_HIP, std::string("context init: ") + hipGetErrorString(e));
    }
    *out = c;
    return LP_OK;
}

}  // namespace

int lp_context_destroy(lp_context* c) {
    if (!c) return LP_OK;
    for (auto* lane : c->lanes) lp_context_destroy(lane);
    for (auto e : c->lane_done) (void)hipEventDestroy(e);
    (void)hipSetDevice(c->device);
    for (auto& g : c->graphs) {
        (void)hipGraphExecDestroy(g.exec);
        (void)hipGraphDestroy(g.graph);
    }
    for (auto e : c->events) (void)hipEventDestroy(e);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    if (c->arena) (void)hipFree(c->arena);
    if (c->clouds_mem) (void)hipFree(c->clouds_mem);
    if (c->kd_mem) (void)hipFree(c->kd_mem);
    if (c->image_dev) (void)hipFree(c->image_dev);
    if (c->pinned) (void)hipHostFree(c->pinned);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
    return LP_OK;
}

void* lp_context_stream(lp_context* c) { return c ? c->stream : nullptr; }

namespace {

int stage_batch(lp_context* c, const lp_segmenter_config* seg_cfgs, int32_t num_seg_cfgs,
                const lp_clusterer_config* ccfg, int32_t num_frames, const lp_cloud* clouds, bool filter) {
    if (!c || !seg_cfgs || !ccfg || !clouds) return fail(LP_ERR_INVALID_ARGUMENT, "null argument");
    if (num_frames < 1 || num_frames > c->L.B) return fail(LP_ERR_CAPACITY, "batch larger than max_frames");
    if (num_seg_cfgs != 1 && num_seg_cfgs != num_frames)
        return fail(LP_ERR_INVALID_ARGUMENT, "num_seg_cfgs must be 1 or num_frames");
    LP_HIP(hipSetDevice(c->device));
    c->frames.assign(num_frames, FrameDesc{});
    int32_t off = 0;
    for (int f = 0; f < num_frames; ++f) {
        const lp_cloud& cl = clouds[f];
        if (cl.num_points < 0 || cl.num_points > c->L.N)
            return fail(LP_ERR_CAPACITY, "frame has more points than max_points_per_frame");
        if (cl.num_points > 0 && (!cl.x || !cl.y || !cl.z)) return fail(LP_ERR_INVALID_ARGUMENT, "null coordinates");
        FrameDesc& fd = c->frames[f];
        std::string why;
        if (!derive_seg(seg_cfgs[num_seg_cfgs == 1 ? 0 : f], c->L, fd.sc, why))
            return fail(LP_ERR_INVALID_ARGUMENT, why);
        fd.pt_off = off;
        fd.n = cl.num_points;
        fd.n_raw = cl.num_points;
        fd.pix_off = f * c->L.P;
        fd.has_ring = cl.ring != nullptr ? 1 : 0;
        off += cl.num_points;
    }
    // With the noise filter on the points land in its raw inputs and the
    // filter writes the kept ones where the segmenter reads them.
    derive_clu(*ccfg, c->cap.max_voxels, c->cc);
    const int st = stage_frames(c, clouds, c->cc, c->nc, filter);
    if (st != LP_OK) return st;
    c->staged_filtered = filter;
    c->num_frames = num_frames;
    c->staged_points = off;
    return LP_OK;
}

}  // namespace

int lp_batch_stage(lp_context* c, const lp_segmenter_config* seg_cfgs, int32_t num_seg_cfgs,
                   const lp_clusterer_config* ccfg, int32_t num_frames, const lp_cloud* clouds) {
    if (!c) return fail(LP_ERR_INVALID_ARGUMENT, "null context");
    if (c->lanes.empty()) return stage_batch(c, seg_cfgs, num_seg_cfgs, ccfg, num_frames, clouds, c->noise_on);
    const int S = 1 + static_cast<int>(c->lanes.size());
    if (!seg_cfgs || !clouds) return fail(LP_ERR_INVALID_ARGUMENT, "null argument");
    if (num_frames < 1 || num_frames > c->L.B * S) return fail(LP_ERR_CAPACITY, "batch larger than max_frames");
    if (num_seg_cfgs != 1 && num_seg_cfgs != num_frames)
        return fail(LP_ERR_INVALID_ARGUMENT, "num_seg_cfgs must be 1 or num_frames");
    // Contiguous shares, as even as possible, lane 0 first.
    const int g = (num_frames + S - 1) / S;
    c->lane_frames.assign(S, 0);
    for (int k = 0; k < S; ++k) {
        lp_context* lane = k == 0 ? c : c->lanes[k - 1];
        const int lo = k * g;
        const int cnt = std::max(0, std::min(g, num_frames - lo));
        if (cnt == 0) {
            lane->num_frames = 0;
            continue;
        }
        const int st = stage_batch(lane, num_seg_cfgs == 1 ? seg_cfgs : seg_cfgs + lo, num_seg_cfgs == 1 ? 1 : cnt,
                                   ccfg, cnt, clouds + lo, lane->noise_on);
        if (st != LP_OK) return st;
        c->lane_frames[k] = cnt;
    }
    return LP_OK;
}

namespace {

int run_lane(lp_context* c, int32_t use_graph) {
    LP_HIP(hipSetDevice(c->device));
    const int B = c->num_frames;
    if (!use_graph) return run_pipeline(c, B, false);
    const int options = (c->staged_filtered ? 1 : 0) | (c->boxes_on ? 2 : 0) | (c->clouds_on ? 4 : 0) |
                        (c->vehicles_on ? 8 : 0) | (c->staged_filtered && c->noise_kdtree ? 16 : 0) |
                        (c->persistent ? 32 : 0) | (c->point_wg << 8) | (c->mark_tile << 20);
    lp_context::GraphEntry* ge = nullptr;
    for (auto& g : c->graphs)
        if (g.frames == B && g.options == options) ge = &g;
    if (!ge) {
        LP_HIP(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
        const int st = run_pipeline(c, B, false);
        hipGraph_t g = nullptr;
        const hipError_t e = hipStreamEndCapture(c->stream, &g);
        if (st != LP_OK) {
            if (g) (void)hipGraphDestroy(g);
            return st;
        }
        if (e != hipSuccess) return fail(LP_ERR_HIP, std::string("graph capture: ") + hipGetErrorString(e));
        hipGraphExec_t ex = nullptr;
        const hipError_t ei = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
        if (ei != hipSuccess) {
            (void)hipGraphDestroy(g);
            return fail(LP_ERR_HIP, std::string("graph instantiate: ") + hipGetErrorString(ei));
        }
        c->graphs.push_back({B, options, g, ex});
        ge = &c->graphs.back();
    }
    c->L.B_active = B;
    LP_HIP(hipGraphLaunch(ge->exec, c->stream));
    return LP_OK;
}

}  // namespace

int lp_batch_run(lp_context* c, int32_t use_graph) {
    if (!c || c->num_frames < 1) return fail(LP_ERR_INVALID_ARGUMENT, "nothing staged");
    int st = run_lane(c, use_graph);
    for (size_t k = 0; st == LP_OK && k < c->lanes.size(); ++k) {
        lp_context* lane = c->lanes[k];
        if (lane->num_frames < 1) continue;
        st = run_lane(lane, use_graph);
        if (st != LP_OK) break;
        LP_HIP(hipEventRecord(c->lane_done[k], lane->stream));
        LP_HIP(hipStreamWaitEvent(c->stream, c->lane_done[k], 0));
    }
    return st;
}

int lp_synchronize(lp_context* c) {
    if (!c) return fail(LP_ERR_INVALID_ARGUMENT, "null context");
    LP_HIP(hipStreamSynchronize(c->stream));
    return LP_OK;
}

int lp_query(lp_context* c) {
    if (!c) return fail(LP_ERR_INVALID_ARGUMENT, "null context");
    const hipError_t e = hipStreamQuery(c->stream);
    if (e == hipSuccess) return 1;
    if (e == hipErrorNotReady) return 0;
    LP_HIP(e);
    return LP_OK;
}

namespace {

// Host memory a context keeps for outputs that go to pageable memory: at
// most this much, beyond it such arrays are copied one by one.
constexpr size_t kBounceMax = size_t{64} << 20;

// The arrays one call returns, and where each goes.  add() them, launch()
// the copies behind the run, finish() waits and hands the pageable ones over.
class Outputs {
   public:
    explicit Outputs(lp_context* c) : c_(c), mem_(c->device) {}

    // `count` elements of `elem` bytes at src (fewer if fs[frame][slot] says so).
    void add(void* user, const void* src, size_t elem, int count, int frame = 0, int slot = -1, int rules = 0,
             int hull_capacity = 0) {
        if (!user || count <= 0) return;
        Entry e{};
        e.it = OutItem{static_cast<const uint8_t*>(src), nullptr, static_cast<uint32_t>(elem), count, frame,
                       static_cast<int16_t>(slot), static_cast<int16_t>(rules), hull_capacity};
        e.user = user;
        const size_t bytes = elem * static_cast<size_t>(count);
        e.kind = mem_.find(user, bytes, &e.it.dst);
        if (e.kind == CallerMemory::kDevice) e.kind = CallerMemory::kOther;
        if (e.kind == CallerMemory::kPageable) {
            e.bounce = (need_ + 255) & ~size_t{255};
            if (e.bounce + bytes > kBounceMax)
                e.kind = CallerMemory::kOther;
            else
                need_ = e.bounce + bytes;
        }
        entries_.push_back(e);
    }

    // Queues the copies and the scalars of `frames` frames.
    int launch(int frames) {
        const size_t scalars = (static_cast<size_t>(c_->L.B) * kFsCount * 4 + 255) & ~size_t{255};
        const size_t want = scalars + need_;
        if (want > c_->pinned_bytes) {
            if (c_->pinned) (void)hipHostFree(c_->pinned);
            c_->pinned = nullptr;
            c_->pinned_bytes = 0;
            LP_HIP(hipHostMalloc(&c_->pinned, want, hipHostMallocDefault));
            c_->pinned_bytes = want;
        }
        bounce_ = static_cast<uint8_t*>(c_->pinned) + scalars;
        OutArgs a{};
        a.item[0] = OutItem{reinterpret_cast<const uint8_t*>(c_->d.fs), static_cast<uint8_t*>(c_->pinned), 4,
                            frames * kFsCount, 0, -1, 0, 0};
        int k = 1;
        size_t most = 0;
        auto flush = [&] {
            // 16 bytes a thread, at most 64 workgroups an item: a few
            // hundred KB in flight fill the host link.
            const int tiles = static_cast<int>(std::min<size_t>(64, std::max<size_t>(1, (most + 4095) / 4096)));
            hipLaunchKernelGGL(k_copy_out, dim3(tiles, k), dim3(256), 0, c_->stream, a, c_->d.fs);
            k = 0;
            most = 0;
        };
        for (Entry& e : entries_) {
            if (e.kind == CallerMemory::kOther) continue;
            if (e.kind == CallerMemory::kPageable) e.it.dst = bounce_ + e.bounce;
            if (k == kOutItems) flush();
            a.item[k++] = e.it;
            most = std::max(most, static_cast<size_t>(e.it.elem) * e.it.count);
        }
        if (k) flush();
        LP_HIP(hipGetLastError());
        return LP_OK;
    }

    // The scalars, valid after finish().
    const uint32_t* scalars() const { return static_cast<const uint32_t*>(c_->pinned); }

    int finish() {
        LP_HIP(hipStreamSynchronize(c_->stream));
        bool more = false;
        for (const Entry& e : entries_) {
            const uint32_t bytes = e.kind == CallerMemory::kPinned ? 0 : out_bytes(e.it, scalars());
            if (!bytes) continue;
            if (e.kind == CallerMemory::kPageable) {
                std::memcpy(e.user, bounce_ + e.bounce, bytes);
            } else {
                LP_HIP(hipMemcpyAsync(e.user, out_src(e.it, scalars()), bytes, hipMemcpyDeviceToHost, c_->stream));
                more = true;
            }
        }
        if (more) LP_HIP(hipStreamSynchronize(c_->stream));
        return LP_OK;
    }

   private:
    struct Entry {
        OutItem it;
        void* user;
        size_t bounce;
        CallerMemory::Kind kind;
    };
    lp_context* c_;
    CallerMemory mem_;
    std::vector<Entry> entries_;
    size_t need_ = 0;
    uint8_t* bounce_ = nullptr;
};

// Queues the outputs of a lane's frames behind its run.
int queue_fetch(lp_context* c, const lp_frame_outputs* outputs, Outputs& out) {
    LP_HIP(hipSetDevice(c->device));
    const int B = c->num_frames;
    const Layout& L = c->L;
    const bool boxes = c->boxes_on || c->vehicles_on;
    for (int f = 0; f < B && outputs; ++f) {
        const FrameDesc& fd = c->frames[f];
        const lp_frame_outputs& o = outputs[f];
        const size_t ob = static_cast<size_t>(f) * L.N;
        const size_t kb = static_cast<size_t>(f) * L.box_stride;
        const int n = fd.n;
        // Points the segmenter saw: the noise filter's kept count when it ran.
        const int points = c->staged_filtered ? kFsKept : -1;
        // A cluster has at least min_size of them.
        const int k = n / std::max(1, static_cast<int>(std::min(c->cc.min_size, 1u << 30)));
        if (c->staged_filtered) out.add(o.noise_labels, c->d.noise + ob, 1, fd.n_raw, f);
        out.add(o.seg_labels, c->d.labels + fd.pt_off, 4, n, f, points);
        out.add(o.obstacle_index, c->d.obs_src + ob, 4, n, f, kFsObstacles, kSkipFailed);
        out.add(o.cluster_labels, c->d.clabel + ob, 4, n, f, kFsObstacles, kSkipFailed);
        out.add(o.hull_offsets, c->d.hull_off + ob, 4, k, f, kFsClusters, kSkipFailed);
        const int hc = o.hull_capacity;
        const int rules = kSkipFailed | (o.hull_indices ? kSkipHullOver : 0);
        out.add(o.hull_indices, c->d.hull_local + ob, 4, std::min(n, hc), f, kFsHullTotal, rules, hc);
        if (boxes) out.add(o.boxes, c->d.boxes + kb, sizeof(lp_bounding_box), std::min(k, L.box_stride), f, kFsClusters,
                           rules, hc);
        if (c->vehicles_on) out.add(o.vehicle_class, c->d.vclass + kb, 4, std::min(k, L.box_stride), f, kFsClusters,
                                    rules, hc);
        if (c->clouds_on) {
            out.add(o.ground_index, c->d.split_idx + ob, 4, n, f, kFsGround, rules, hc);
            out.add(o.unknown_index, c->d.split_idx + ob, 4, n, f, points, rules | kUnknownCloud, hc);
        }
    }
    return out.launch(B);
}

// Waits for a lane's outputs and reports its frames.
int finish_fetch(lp_context* c, const lp_frame_outputs* outputs, lp_frame_result* results, Outputs& out) {
    LP_HIP(hipSetDevice(c->device));
    const int st = out.finish();
    if (st != LP_OK) return st;
    int overall = LP_OK;
    for (int f = 0; f < c->num_frames; ++f) {
        const uint32_t* s = out.scalars() + static_cast<size_t>(f) * kFsCount;
        const FrameDesc& fd = c->frames[f];
        lp_frame_result r{};
        r.status = status_of(s[kFsErr] | s[kFsNoiseErr]);
        const int n = c->staged_filtered ? static_cast<int>(s[kFsKept]) : fd.n;
        r.num_points = n;
        r.num_noise = c->staged_filtered ? static_cast<int32_t>(s[kFsNoise]) : 0;
        r.num_noise_searched = c->staged_filtered ? static_cast<int32_t>(s[kFsNoiseHard]) : 0;
        const bool boxes = c->boxes_on || c->vehicles_on;
        r.num_boxes = boxes ? static_cast<int32_t>(s[kFsBoxes]) : 0;
        r.num_obstacles = static_cast<int32_t>(s[kFsObstacles]);
        r.num_voxels = static_cast<int32_t>(s[kFsVoxels]);
        r.num_clusters = static_cast<int32_t>(s[kFsClusters]);
        r.num_hull_vertices = static_cast<int32_t>(s[kFsHullTotal]);
        r.jcp_queue = static_cast<int32_t>(s[kFsQueue]);
        if (c->clouds_on) {
            r.num_ground = static_cast<int32_t>(s[kFsGround]);
            r.num_unknown = n - r.num_ground - r.num_obstacles;
        }
        r.num_vehicles = c->vehicles_on ? static_cast<int32_t>(s[kFsVehicles]) : 0;
        r.num_hull_inexact = static_cast<int32_t>(s[kFsHullInexact]);
        r.num_hull_rounded = static_cast<int32_t>(s[kFsHullRounded]);
        r.ransac.candidates = s[kFsCands];
        r.ransac.best_inliers = s[kFsBest];
        r.ransac.applied = static_cast<int32_t>(s[kFsApplied]);
        uint32_t pl[4] = {s[kFsPlaneA], s[kFsPlaneB], s[kFsPlaneC], s[kFsPlaneD]};
        if (!r.ransac.applied) {
            const float dflt[4] = {0.0F, 0.0F, 1.0F, 0.0F};
            std::memcpy(pl, dflt, sizeof(pl));
        }
        std::memcpy(r.ransac.plane, pl, sizeof(pl));
        if (results) results[f] = r;
        if (r.status != LP_OK && overall == LP_OK) overall = r.status;
        if (!outputs || r.status != LP_OK) continue;
        const lp_frame_outputs& o = outputs[f];
        if (o.hull_offsets) o.hull_offsets[r.num_clusters] = r.num_hull_vertices;
        if (o.hull_indices && r.num_hull_vertices > 0 && r.num_hull_vertices > o.hull_capacity) {
            if (results) results[f].status = fail(LP_ERR_CAPACITY, "hull_capacity too small");
            overall = LP_ERR_CAPACITY;
        }
    }
    return overall;
}

}  // namespace

int lp_batch_fetch(lp_context* c, const lp_frame_outputs* outputs, lp_frame_result* results) {
    if (!c || c->num_frames < 1) return fail(LP_ERR_INVALID_ARGUMENT, "nothing staged");
    if (c->lanes.empty()) {
        Outputs out(c);
        const int st = queue_fetch(c, outputs, out);
        return st != LP_OK ? st : finish_fetch(c, outputs, results, out);
    }
    // Every lane's copies are queued before the first is waited for, so a
    // lane that is done sends its outputs while the others still run.
    std::vector<Outputs> outs;
    outs.reserve(c->lane_frames.size());
    int overall = LP_OK, off = 0;
    auto each = [&](auto step) {
        off = 0;
        for (size_t k = 0; k < c->lane_frames.size(); ++k) {
            if (c->lane_frames[k] == 0) continue;
            lp_context* lane = k == 0 ? c : c->lanes[k - 1];
            const int st = step(lane, outputs ? outputs + off : nullptr, results ? results + off : nullptr);
            if (st != LP_OK && overall == LP_OK) overall = st;
            off += c->lane_frames[k];
        }
    };
    each([&](lp_context* lane, const lp_frame_outputs* o, lp_frame_result*) {
        outs.emplace_back(lane);
        return queue_fetch(lane, o, outs.back());
    });
    if (overall != LP_OK) {
        // A lane failed to queue: nothing is left writing to the caller's memory.
        each([&](lp_context* lane, const lp_frame_outputs*, lp_frame_result*) -> int {
            LP_HIP(hipStreamSynchronize(lane->stream));
            return LP_OK;
        });
        return overall;
    }
    size_t next = 0;
    each([&](lp_context* lane, const lp_frame_outputs* o, lp_frame_result* r) {
        return finish_fetch(lane, o, r, outs[next++]);
    });
    return overall;
}

int lp_process_frames(lp_context* c, const lp_segmenter_config* seg_cfgs, int32_t num_seg_cfgs,
                      const lp_clusterer_config* ccfg, int32_t num_frames, const lp_cloud* clouds,
                      const lp_frame_outputs* outputs, lp_frame_result* results) {
    int st = lp_batch_stage(c, seg_cfgs, num_seg_cfgs, ccfg, num_frames, clouds);
    if (st != LP_OK) return st;
    st = lp_batch_run(c, 0);
    if (st != LP_OK) return st;
    return lp_batch_fetch(c, outputs, results);
}

int lp_segment(lp_context* c, const lp_segmenter_config* cfg, const lp_cloud* cloud, uint32_t* labels,
               lp_ransac_result* ransac) {
    if (!c || !cfg || !cloud || (!labels && cloud->num_points > 0))
        return fail(LP_ERR_INVALID_ARGUMENT, "null argument");
    lp_clusterer_config cc;
    lp_clusterer_config_shipped(&cc);
    int st = stage_batch(c, cfg, 1, &cc, 1, cloud, false);
    if (st != LP_OK) return st;
    st = run_pipeline(c, 1, true);
    if (st != LP_OK) return st;
    Outputs out(c);
    out.add(labels, c->d.labels, 4, cloud->num_points);
    st = out.launch(1);
    if (st == LP_OK) st = out.finish();
    if (st != LP_OK) return st;
    const uint32_t* fs = out.scalars();
    st = status_of(fs[kFsErr] & ~(kErrVoxelOverflow | kErrHullCapacity));
    if (ransac) {
        ransac->candidates = fs[kFsCands];
        ransac->best_inliers = fs[kFsBest];
        ransac->applied = static_cast<int32_t>(fs[kFsApplied]);
        if (ransac->applied) {
            std::memcpy(ransac->plane, &fs[kFsPlaneA], 16);
        } else {
            const float dflt[4] = {0.0F, 0.0F, 1.0F, 0.0F};
            std::memcpy(ransac->plane, dflt, 16);
        }
    }
    return st;
}

int lp_cluster(lp_context* c, const lp_clusterer_config* cfg, const lp_cloud* cloud, int32_t* labels) {
    if (!c || !cfg || !cloud || (!labels && cloud->num_points > 0))
        return fail(LP_ERR_INVALID_ARGUMENT, "null argument");
    if (cloud->num_points < 0 || cloud->num_points > c->L.N)
        return fail(LP_ERR_CAPACITY, "cloud has more points than max_points_per_frame");
    LP_HIP(hipSetDevice(c->device));
    FrameDesc fd{};
    fd.pt_off = 0;
    fd.n = cloud->num_points;
    fd.n_raw = cloud->num_points;
    fd.pix_off = 0;
    fd.has_ring = 0;  // no polar grid, no image: the clear stage only resets the voxel state
    c->frames.assign(1, fd);
    lp_cloud xyz = *cloud;
    xyz.ring = nullptr;
    derive_clu(*cfg, c->cap.max_voxels, c->cc);
    int st = stage_frames(c, &xyz, c->cc, c->nc, false);
    if (st != LP_OK) return st;
    c->num_frames = 1;
    c->L.B_active = 1;
    launch_clear(c, 1, false);
    launch_cluster(c, 1, false);
    LP_HIP(hipGetLastError());
    Outputs out(c);
    out.add(labels, c->d.clabel, 4, cloud->num_points);
    st = out.launch(1);
    if (st == LP_OK) st = out.finish();
    if (st != LP_OK) return st;
    c->num_frames = 0;  // the staged frame is not a full-pipeline batch
    return status_of(out.scalars()[kFsErr]);
}

void lp_noise_config_default(lp_noise_config* cfg) {
    cfg->radius_multiplier_m_per_m = 0.02F;
    cfg->min_search_radius_m = 0.1F;
    cfg->min_neighbours = 4U;
}

int lp_set_noise_filter(lp_context* c, const lp_noise_config* cfg) {
    if (!c) return fail(LP_ERR_INVALID_ARGUMENT, "null context");
    if (!cfg) {
        c->noise_on = false;
        for (auto* lane : c->lanes) lane->noise_on = false;
        return LP_OK;
    }
    if (c->noise_kdtree && cfg->min_neighbours > kKdMaxNeighbours)
        return fail(LP_ERR_INVALID_ARGUMENT, "the KD-tree noise search supports min_neighbours up to 7");
    c->nc = noise_const(*cfg);
    c->noise_on = true;
    for (auto* lane : c->lanes) lp_set_noise_filter(lane, cfg);
    return LP_OK;
}

int lp_set_persistent(lp_context* c, int32_t enable) {
    if (!c) return fail(LP_ERR_INVALID_ARGUMENT, "null context");
    c->persistent = enable != 0;
    for (auto* lane : c->lanes) lane->persistent = c->persistent;
    return LP_OK;
}

int lp_set_launch_shape(lp_context* c, int32_t point_workgroup, int32_t mark_tile_width) {
    if (!c) return fail(LP_ERR_INVALID_ARGUMENT, "null context");
    auto ok = [](int32_t v) { return v == 64 || v == 128 || v == 256; };
    if (!ok(point_workgroup) || !ok(mark_tile_width))
        return fail(LP_ERR_INVALID_ARGUMENT, "workgroup size and tile width must be 64, 128 or 256");
    c->point_wg = point_workgroup;
    c->mark_tile = mark_tile_width;
    for (auto* lane : c->lanes) {
        lane->point_wg = point_workgroup;
        lane->mark_tile = mark_tile_width;
    }
    return LP_OK;
}

int lp_set_noise_search(lp_context* c, int32_t mode) {
    if (!c) return fail(LP_ERR_INVALID_ARGUMENT, "null context");
    if (mode != LP_NOISE_RULE && mode != LP_NOISE_KDTREE) return fail(LP_ERR_INVALID_ARGUMENT, "unknown noise search");
    // The KD-tree kernels (lp_noise_ref.hip) stay compiled but unreachable:
    // their first device run left the GPU faulted, and no cause has been
    // shown yet.
    if (mode == LP_NOISE_KDTREE && kKdSearchDisabled)
        return fail(LP_ERR_INVALID_ARGUMENT, "the KD-tree noise search is switched off in this build");
    if (mode == LP_NOISE_KDTREE) {
        if (c->noise_on && c->nc.k > static_cast<uint32_t>(kKdMaxNeighbours))
            return fail(LP_ERR_INVALID_ARGUMENT, "the KD-tree noise search supports min_neighbours up to 7");
        if (!c->kd_mem) {
            LP_HIP(hipSetDevice(c->device));
            const size_t cnt = static_cast<size_t>(c->L.B) * c->L.N;
            const size_t ent = cnt * kKdEntriesPerPoint;
            const size_t bytes = cnt * (sizeof(float4) + 2 * sizeof(int32_t) + sizeof(uint2) + 4 * sizeof(uint32_t) +
                                        kKdRecInts * sizeof(int32_t)) + 2 * ent * sizeof(uint64_t);
            LP_HIP(hipMalloc(&c->kd_mem, bytes));
            char* p = static_cast<char*>(c->kd_mem);
            auto take = [&](size_t b) { char* r = p; p += b; return r; };
            c->d.kd_csr = reinterpret_cast<uint64_t*>(take(ent * sizeof(uint64_t)));
            c->d.kd_live = reinterpret_cast<uint64_t*>(take(ent * sizeof(uint64_t)));
            c->d.kd = reinterpret_cast<float4*>(take(cnt * sizeof(float4)));
            c->d.kd_q = reinterpret_cast<uint2*>(take(cnt * sizeof(uint2)));
            c->d.kd_tl = reinterpret_cast<int32_t*>(take(cnt * sizeof(int32_t)));
            c->d.kd_tr = reinterpret_cast<int32_t*>(take(cnt * sizeof(int32_t)));
            c->d.kd_lcnt = reinterpret_cast<uint32_t*>(take(cnt * sizeof(uint32_t)));
            c->d.kd_loff = reinterpret_cast<uint32_t*>(take(cnt * sizeof(uint32_t)));
            c->d.kd_dflag = reinterpret_cast<uint32_t*>(take(cnt * sizeof(uint32_t)));
            c->d.kd_dpos = reinterpret_cast<uint32_t*>(take(cnt * sizeof(uint32_t)));
            c->d.kd_drec = reinterpret_cast<int32_t*>(take(cnt * kKdRecInts * sizeof(int32_t)));
        }
    }
    c->noise_kdtree = mode == LP_NOISE_KDTREE;
    for (auto* lane : c->lanes) {
        const int st = lp_set_noise_search(lane, mode);
        if (st != LP_OK) return st;
    }
    return LP_OK;
}

int lp_set_oriented_boxes(lp_context* c, int32_t enable) {
    if (!c) return fail(LP_ERR_INVALID_ARGUMENT, "null context");
    c->boxes_on = enable != 0;
    for (auto* lane : c->lanes) lane->boxes_on = c->boxes_on;
    return LP_OK;
}

int lp_set_label_clouds(lp_context* c, int32_t enable) {
    if (!c) return fail(LP_ERR_INVALID_ARGUMENT, "null context");
    if (enable && !c->clouds_mem) {
        LP_HIP(hipSetDevice(c->device));
        const size_t count = static_cast<size_t>(c->L.B) * c->L.N;
        LP_HIP(hipMalloc(&c->clouds_mem, 2 * count * sizeof(uint32_t)));
        c->d.gnd_flag = static_cast<uint32_t*>(c->clouds_mem);
        c->d.split_idx = reinterpret_cast<int32_t*>(c->d.gnd_flag + count);
    }
    c->clouds_on = enable != 0;
    for (auto* lane : c->lanes) {
        const int st = lp_set_label_clouds(lane, enable);
        if (st != LP_OK) return st;
    }
    return LP_OK;
}

int lp_set_vehicle_boxes(lp_context* c, int32_t enable) {
    if (!c) return fail(LP_ERR_INVALID_ARGUMENT, "null context");
    c->vehicles_on = enable != 0;
    for (auto* lane : c->lanes) lane->vehicles_on = c->vehicles_on;
    return LP_OK;
}

int lp_remove_noise(lp_context* c, const lp_noise_config* cfg, const lp_cloud* cloud, uint8_t* labels) {
    if (!c || !cfg || !cloud || (!labels && cloud->num_points > 0))
        return fail(LP_ERR_INVALID_ARGUMENT, "null argument");
    if (cloud->num_points < 0 || cloud->num_points > c->L.N)
        return fail(LP_ERR_CAPACITY, "cloud has more points than max_points_per_frame");
    if (cloud->num_points > 0 && (!cloud->x || !cloud->y || !cloud->z))
        return fail(LP_ERR_INVALID_ARGUMENT, "null coordinates");
    if (c->noise_kdtree && cfg->min_neighbours > kKdMaxNeighbours)
        return fail(LP_ERR_INVALID_ARGUMENT, "the KD-tree noise search supports min_neighbours up to 7");
    if (cloud->num_points == 0) return LP_OK;
    LP_HIP(hipSetDevice(c->device));
    FrameDesc fd{};
    fd.n = cloud->num_points;
    fd.n_raw = cloud->num_points;
    c->frames.assign(1, fd);
    lp_cloud xyz = *cloud;
    xyz.ring = nullptr;
    int st = stage_frames(c, &xyz, c->cc, noise_const(*cfg), true);
    if (st != LP_OK) return st;
    c->num_frames = 0;
    c->L.B_active = 1;
    if (c->noise_kdtree) {
        launch_noise_kdtree(c, 1, false);
    } else {
        launch_noise(c, 1, false);
    }
    LP_HIP(hipGetLastError());
    Outputs out(c);
    out.add(labels, c->d.noise, 1, cloud->num_points);
    st = out.launch(1);
    if (st == LP_OK) st = out.finish();
    if (st != LP_OK) return st;
    return c->noise_kdtree ? status_of(out.scalars()[kFsNoiseErr]) : LP_OK;
}

namespace {

// Stages num_polygons point lists (x, y packed by offsets) as frame 0's hull
// coordinates and runs `launch` over them; boxes[k] receives list k's box.
int polygon_boxes(lp_context* c, const double* x, const double* y, const int32_t* offsets, int32_t num_polygons,
                  lp_bounding_box* boxes, void (*launch)(lp_context*, int)) {
    if (!c || !offsets || num_polygons < 0 || (num_polygons > 0 && !boxes))
        return fail(LP_ERR_INVALID_ARGUMENT, "null argument");
    if (num_polygons == 0) return LP_OK;
    const int32_t total = offsets[num_polygons];
    if (offsets[0] != 0 || total < 0 || total > c->L.N || num_polygons > c->L.box_stride || num_polygons > c->L.N)
        return fail(LP_ERR_CAPACITY, "polygons exceed the context capacity");
    for (int k = 0; k < num_polygons; ++k)
        if (offsets[k + 1] < offsets[k]) return fail(LP_ERR_INVALID_ARGUMENT, "offsets must be non-decreasing");
    if (total > 0 && (!x || !y)) return fail(LP_ERR_INVALID_ARGUMENT, "null coordinates");
    LP_HIP(hipSetDevice(c->device));
    const size_t BN = static_cast<size_t>(c->L.B) * c->L.N;
    std::vector<uint32_t> fs(kFsCount, 0u);
    fs[kFsClusters] = static_cast<uint32_t>(num_polygons);
    fs[kFsHullTotal] = static_cast<uint32_t>(total);
    LP_HIP(hipMemcpyAsync(c->d.fs, fs.data(), kFsCount * 4, hipMemcpyHostToDevice, c->stream));
    LP_HIP(hipMemcpyAsync(c->d.hull_off, offsets, num_polygons * sizeof(int32_t), hipMemcpyHostToDevice, c->stream));
    if (total) {
        LP_HIP(hipMemcpyAsync(c->d.hcx + BN, x, total * sizeof(double), hipMemcpyHostToDevice, c->stream));
        LP_HIP(hipMemcpyAsync(c->d.hcy + BN, y, total * sizeof(double), hipMemcpyHostToDevice, c->stream));
    }
    c->num_frames = 0;
    c->L.B_active = 1;
    launch(c, num_polygons);
    LP_HIP(hipGetLastError());
    Outputs out(c);
    out.add(boxes, c->d.boxes, sizeof(lp_bounding_box), num_polygons);
    int st = out.launch(1);
    if (st == LP_OK) st = out.finish();
    if (st != LP_OK) return st;
    if (out.scalars()[kFsErr] & kErrBoxCapacity) return fail(LP_ERR_CAPACITY, "a polygon exceeds the box kernel's capacity");
    return LP_OK;
}

}  // namespace

int lp_oriented_boxes(lp_context* c, const double* x, const double* y, const int32_t* offsets, int32_t num_polygons,
                      lp_bounding_box* boxes) {
    return polygon_boxes(c, x, y, offsets, num_polygons, boxes,
                         [](lp_context* ctx, int) { launch_boxes(ctx, 1); });
}

int lp_pca_boxes(lp_context* c, const double* x, const double* y, const int32_t* offsets, int32_t num_polygons,
                 lp_bounding_box* boxes) {
    return polygon_boxes(c, x, y, offsets, num_polygons, boxes,
                         [](lp_context* ctx, int k) { launch_pca_boxes(ctx, k); });
}

int lp_add_ring_info(lp_context* c, const float* x, const float* y, int32_t n, uint16_t* ring) {
    if (!c || n < 0 || (n > 0 && (!x || !y || !ring))) return fail(LP_ERR_INVALID_ARGUMENT, "null argument");
    if (n > c->L.N) return fail(LP_ERR_CAPACITY, "cloud has more points than max_points_per_frame");
    if (n == 0) return LP_OK;
    LP_HIP(hipSetDevice(c->device));
    FrameDesc fd{};
    fd.n = n;
    c->frames.assign(1, fd);
    c->num_frames = 0;
    LP_HIP(hipMemcpyAsync(c->d.frames, &fd, sizeof(FrameDesc), hipMemcpyHostToDevice, c->stream));
    LP_HIP(hipMemcpyAsync(c->d.x, x, n * 4, hipMemcpyHostToDevice, c->stream));
    LP_HIP(hipMemcpyAsync(c->d.y, y, n * 4, hipMemcpyHostToDevice, c->stream));
    launch_ring_info(c, n);
    LP_HIP(hipGetLastError());
    LP_HIP(hipMemcpyAsync(ring, c->d.ring, n * 2, hipMemcpyDeviceToHost, c->stream));
    LP_HIP(hipStreamSynchronize(c->stream));
    return LP_OK;
}

int lp_convex_hulls(lp_context* c, const double* x, const double* y, const int32_t* offsets, int32_t num_lists,
                    int32_t* hull_offsets, int32_t* hull_indices, int32_t hull_capacity) {
    if (!c || !offsets || !hull_offsets || num_lists < 0) return fail(LP_ERR_INVALID_ARGUMENT, "null argument");
    if (num_lists == 0) {
        hull_offsets[0] = 0;
        return LP_OK;
    }
    const int32_t total = offsets[num_lists];
    if (offsets[0] != 0 || total < 0 || total > c->L.N || num_lists > c->L.N)
        return fail(LP_ERR_CAPACITY, "point lists exceed max_points_per_frame");
    for (int k = 0; k < num_lists; ++k)
        if (offsets[k + 1] < offsets[k]) return fail(LP_ERR_INVALID_ARGUMENT, "offsets must be non-decreasing");
    if (total > 0 && (!x || !y)) return fail(LP_ERR_INVALID_ARGUMENT, "null coordinates");
    LP_HIP(hipSetDevice(c->device));
    c->L.B_active = 1;
    LP_HIP(hipMemcpyAsync(c->d.hc_open, offsets, (num_lists + 1) * sizeof(int32_t), hipMemcpyHostToDevice,
                          c->stream));
    if (total) {
        LP_HIP(hipMemcpyAsync(c->d.hcx, x, total * sizeof(double), hipMemcpyHostToDevice, c->stream));
        LP_HIP(hipMemcpyAsync(c->d.hcy, y, total * sizeof(double), hipMemcpyHostToDevice, c->stream));
    }
    launch_hull_lists(c, num_lists, total);
    LP_HIP(hipGetLastError());
    Outputs out(c);
    out.add(hull_offsets, c->d.hull_off, sizeof(int32_t), num_lists);
    out.add(hull_indices, c->d.hull_local, sizeof(int32_t), std::min(c->L.N, hull_capacity), 0, kFsHullTotal,
            kSkipHullOver, hull_capacity);
    int st = out.launch(1);
    if (st == LP_OK) st = out.finish();
    if (st != LP_OK) return st;
    const uint32_t* fs = out.scalars();
    const int32_t V = static_cast<int32_t>(fs[kFsHullTotal]);
    if (fs[kFsErr] & kErrHullCapacity) return fail(LP_ERR_CAPACITY, "hull candidates exceed the device capacity");
    if (V > hull_capacity || (V > 0 && !hull_indices)) return fail(LP_ERR_CAPACITY, "hull_capacity too small");
    hull_offsets[num_lists] = V;
    c->num_frames = 0;
    return LP_OK;
}

int lp_debug_fetch(lp_context* c, int32_t frame, int32_t which, void* dst, int32_t capacity) {
    if (!c || frame < 0 || frame >= static_cast<int32_t>(c->frames.size()) || !dst)
        return fail(LP_ERR_INVALID_ARGUMENT, "bad debug request");
    LP_HIP(hipSetDevice(c->device));
    LP_HIP(hipStreamSynchronize(c->stream));
    const FrameDesc& fd = c->frames[frame];
    const Layout& L = c->L;
    const int32_t P = fd.sc.H * fd.sc.W;
    const size_t po = static_cast<size_t>(frame) * L.P;
    uint32_t fs[kFsCount];
    LP_HIP(hipMemcpy(fs, c->d.fs + static_cast<size_t>(frame) * kFsCount, sizeof(fs), hipMemcpyDeviceToHost));
    const int32_t nq = static_cast<int32_t>(fs[kFsQueue]);
    switch (which) {
        case LP_DEBUG_ELEVATION_MAP: {
            const int32_t n = fd.sc.cells;
            if (n <= capacity)
                LP_HIP(hipMemcpy(dst, c->d.elev + static_cast<size_t>(frame) * L.cell_stride, n * 4,
                                 hipMemcpyDeviceToHost));
            return n;
        }
        case LP_DEBUG_MAPPING:
            if (P <= capacity) LP_HIP(hipMemcpy(dst, c->d.mapping + po, P * 4, hipMemcpyDeviceToHost));
            return P;
        case LP_DEBUG_STATE_RECM:
            if (P <= capacity) LP_HIP(hipMemcpy(dst, c->d.state + po, P, hipMemcpyDeviceToHost));
            return P;
        case LP_DEBUG_JCP_QUEUE:
            if (nq <= capacity && nq > 0) LP_HIP(hipMemcpy(dst, c->d.qlist + po, nq * 4, hipMemcpyDeviceToHost));
            return nq;
        case LP_DEBUG_STATE_FINAL: {
            if (P > capacity) return P;
            std::vector<uint8_t> st(P), fin(std::max(nq, 1));
            std::vector<int32_t> qm(P);
            LP_HIP(hipMemcpy(st.data(), c->d.state + po, P, hipMemcpyDeviceToHost));
            LP_HIP(hipMemcpy(qm.data(), c->d.qmap + po, P * 4, hipMemcpyDeviceToHost));
            if (nq > 0) LP_HIP(hipMemcpy(fin.data(), c->d.fin + po, nq, hipMemcpyDeviceToHost));
            uint8_t* o = static_cast<uint8_t*>(dst);
            for (int32_t p = 0; p < P; ++p) o[p] = qm[p] >= 0 ? fin[qm[p]] : st[p];
            return P;
        }
        default:
            return fail(LP_ERR_INVALID_ARGUMENT, "unknown debug buffer");
    }
}

int lp_frame_image(lp_context* c, int32_t frame, uint8_t* bgr, int32_t capacity) {
    if (!c || frame < 0 || !bgr) return fail(LP_ERR_INVALID_ARGUMENT, "bad image request");
    // The lane that ran the frame: lane k holds the k-th contiguous share.
    lp_context* lane = c;
    int32_t f = frame;
    if (!c->lanes.empty()) {
        size_t k = 0;
        while (k < c->lane_frames.size() && f >= c->lane_frames[k]) f -= c->lane_frames[k++];
        if (k == c->lane_frames.size()) return fail(LP_ERR_INVALID_ARGUMENT, "frame not in the last batch");
        lane = k == 0 ? c : c->lanes[k - 1];
    }
    if (f >= lane->num_frames || f >= static_cast<int32_t>(lane->frames.size()))
        return fail(LP_ERR_INVALID_ARGUMENT, "frame not in the last batch");
    const SegConst& sc = lane->frames[f].sc;
    const int32_t pixels = sc.H * sc.W;
    const int32_t bytes = 3 * pixels;
    if (bytes > capacity) return bytes;
    LP_HIP(hipSetDevice(lane->device));
    if (!lane->image_dev) LP_HIP(hipMalloc(&lane->image_dev, 3 * static_cast<size_t>(lane->L.P)));
    launch_label_image(lane, f, pixels, lane->image_dev);
    LP_HIP(hipGetLastError());
    LP_HIP(hipMemcpyAsync(bgr, lane->image_dev, bytes, hipMemcpyDeviceToHost, lane->stream));
    LP_HIP(hipStreamSynchronize(lane->stream));
    return bytes;
}

int lp_stage_names(lp_context* c, char* buf, int32_t buf_len) {
    if (!c || !buf || buf_len <= 0) return fail(LP_ERR_INVALID_ARGUMENT, "null argument");
    std::string s;
    for (size_t i = 0; i < c->stage_names.size(); ++i) {
        if (i) s += ",";
        s += c->stage_names[i];
    }
    std::snprintf(buf, static_cast<size_t>(buf_len), "%s", s.c_str());
    return static_cast<int>(c->stage_names.size());
}

int lp_profile_run(lp_context* c, int32_t runs, float* stage_ms, int32_t max_stages, int32_t* num_stages) {
    if (!c || c->num_frames < 1 || runs < 1) return fail(LP_ERR_INVALID_ARGUMENT, "nothing staged");
    LP_HIP(hipSetDevice(c->device));
    std::vector<float> acc;
    for (int r = 0; r < runs; ++r) {
        for (auto e : c->events) (void)hipEventDestroy(e);
        c->events.clear();
        c->stage_names.clear();
        c->profiling = true;
        const int st = run_pipeline(c, c->num_frames, false);
        stage_mark(c, "end");
        c->profiling = false;
        if (st != LP_OK) return st;
        LP_HIP(hipStreamSynchronize(c->stream));
        acc.resize(c->events.size() - 1, 0.0f);
        for (size_t i = 0; i + 1 < c->events.size(); ++i) {
            float ms = 0.0f;
            LP_HIP(hipEventElapsedTime(&ms, c->events[i], c->events[i + 1]));
            acc[i] += ms;
        }
    }
    const int ns = static_cast<int>(acc.size());
    for (int i = 0; i < ns && i < max_stages; ++i) stage_ms[i] = acc[i] / runs;
    if (num_stages) *num_stages = ns;
    c->stage_names.pop_back();
    return LP_OK;
}

// PointCloud2 field dispatch of Processor::run (src/processor/src/
// processor.cpp:494-549) and the per-layout conversions convert<PointT>
// (processor.cpp:42-179): the reference copies every point into a
// pcl::PointCloud; here the message buffer itself becomes the lp_cloud
// (byte-strided views), so the points go to the GPU straight from it.
static bool field_names_are(const lp_point_field* f, int32_t n, std::initializer_list<const char*> want) {
    if (n != static_cast<int32_t>(want.size())) return false;
    int32_t k = 0;
    for (const char* w : want) {
        if (!f[k].name || std::strcmp(f[k].name, w) != 0) return false;
        ++k;
    }
    return true;
}

int lp_cloud_from_pointcloud2(const uint8_t* data, uint32_t width, uint32_t height, uint32_t point_step,
                              uint32_t row_step, const lp_point_field* fields, int32_t num_fields, lp_cloud* cloud) {
    if (!fields || !cloud || num_fields < 0) return fail(LP_ERR_INVALID_ARGUMENT, "null argument");
    int ring_field = -1;
    if (field_names_are(fields, num_fields, {"x", "y", "z"}) ||
        field_names_are(fields, num_fields, {"x", "y", "z", "intensity"})) {
        ring_field = -1;
    } else if (field_names_are(fields, num_fields, {"x", "y", "z", "ring"})) {
        ring_field = 3;
    } else if (field_names_are(fields, num_fields, {"x", "y", "z", "intensity", "ring"})) {
        ring_field = 4;
    } else {
        return fail(LP_ERR_INVALID_ARGUMENT,
                    "Unsupported point format. Acceptable formats: pcl::PointXYZ, pcl::PointXYZI, "
                    "pcl::PointXYZR, pcl::PointXYZIR");
    }
    const uint64_t n = static_cast<uint64_t>(width) * height;
    if (n > 0x7fffffffull) return fail(LP_ERR_CAPACITY, "more than 2^31 - 1 points");
    if (height > 1 && static_cast<uint64_t>(row_step) != static_cast<uint64_t>(width) * point_step)
        return fail(LP_ERR_INVALID_ARGUMENT, "rows are not packed (row_step != width * point_step)");
    if (point_step > 0x7fffffffu) return fail(LP_ERR_INVALID_ARGUMENT, "point_step too large");
    for (int k = 0; k < 3; ++k)
        if (static_cast<uint64_t>(fields[k].offset) + 4 > point_step)
            return fail(LP_ERR_INVALID_ARGUMENT, "a coordinate field lies outside the point");
    if (ring_field >= 0 && static_cast<uint64_t>(fields[ring_field].offset) + 2 > point_step)
        return fail(LP_ERR_INVALID_ARGUMENT, "the ring field lies outside the point");
    if (n > 0 && !data) return fail(LP_ERR_INVALID_ARGUMENT, "null data");
    lp_cloud c{};
    c.num_points = static_cast<int32_t>(n);
    c.xyz_stride = static_cast<int32_t>(point_step);
    c.ring_stride = static_cast<int32_t>(point_step);
    c.on_device = 0;
    c.x = data ? data + fields[0].offset : nullptr;
    c.y = data ? data + fields[1].offset : nullptr;
    c.z = data ? data + fields[2].offset : nullptr;
    c.ring = (ring_field >= 0 && data) ? data + fields[ring_field].offset : nullptr;
    *cloud = c;
    return LP_OK;
}

}  // extern "C"
