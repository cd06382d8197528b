// lp_jcp.hip -- Jump-Convolution-Process on the range image, exact.
//
// Reference: lidar_processing_lib/src/segmenter.cpp:481-638 (JCP) and
// :640-669 (populateLabels).  The reference dilates the obstacle mask with a
// 5x5 rectangle (out-of-image pixels never contribute), queues every ground
// pixel next to an obstacle in raster order, and then visits the queue
// sequentially.  Each visit reads the CURRENT label of its 24 neighbours and
// writes 24 weight / label slots that are member arrays reset only once per
// frame: a slot whose neighbour falls outside the image is skipped without
// being rewritten, so it keeps the value of the last earlier queue pixel for
// which that slot was inside the image ("stale" slots).
//
// Parallel form used here (exactly equivalent):
//   * every dependency of a queue pixel p is on raster-earlier queue pixels;
//   * all of them lie in earlier image rows, except the two same-row
//     neighbours (0,-1) and (0,-2) -- a stale slot's writer and the writer's
//     neighbour are always in earlier rows or static;
//   * so rows are solved in order, and inside a row a pixel's label is a
//     function of the labels of the two queue pixels before it: an
//     associative scan of these maps solves the row at once.
// The weights w_i = u_i / sum do not depend on labels and are precomputed
// for all queue pixels in parallel (k_jcp_slots).  A label is the sign of
// (obstacle weights - ground weights); the row solve forms that difference
// once and only where it is within rounding of zero evaluates the reference's
// ordered float sums.
#include "lp_kernels.h"
#include "lp_queue.h"

namespace lp {

using namespace lpd;

__constant__ static const int8_t kOffR[24] = {-2, -2, -2, -2, -2, -1, -1, -1, -1, -1, 0, 0,
                                              0,  0,  1,  1,  1,  1,  1,  2,  2,  2,  2, 2};
__constant__ static const int8_t kOffC[24] = {-2, -1, 0, 1, 2, -2, -1, 0, 1, 2, -2, -1,
                                              1,  2,  -2, -1, 0, 1, 2, -2, -1, 0, 1, 2};

// Slot label sources: >= 0 a queue index (dynamic), else a static label.
constexpr int32_t kSrcUnknown = -1;
constexpr int32_t kSrcGround = -2;
constexpr int32_t kSrcObstacle = -3;

// Queue membership: a ground pixel with an obstacle pixel in its clipped 5x5
// window (cv::dilate of the red channel, then the raster scan of
// segmenter.cpp:491-514).
// Queue flags: a ground pixel with an obstacle pixel in its 5x5 window
// clipped to the image (the dilated red channel of segmenter.cpp:484-513).
// Each workgroup takes T columns of one row (T = 64, 128 or 256, the
// tile width the launch chooses) and stages rows r-2..r+2 of columns
// c0-2..c0+T+1 in LDS (out-of-image pixels read as empty).  The flags of a
// wavefront's 64 columns leave as one word, bit b for column 64 * k + b of the
// row's run k.
__device__ __forceinline__ int queue_runs(int W) { return (W + kWave - 1) / kWave; }  // runs per row

template <int T>
__global__ __launch_bounds__(T) void k_jcp_mark(DevBuf d, Layout L) {
    constexpr int kSpan = T + 4;
    __shared__ uint8_t win[5][kSpan];
    const int f = blockIdx.y;
    const FrameDesc& fd = d.frames[f];
    const int H = fd.sc.H, W = fd.sc.W;
    const int tpr = (W + T - 1) / T;
    const int r = static_cast<int>(blockIdx.x) / tpr, c0 = (static_cast<int>(blockIdx.x) % tpr) * T;
    if (r >= H) return;
    const uint8_t* st = d.state + fd.pix_off;
    for (int q = threadIdx.x; q < 5 * kSpan; q += blockDim.x) {
        const int rr = r + q / kSpan - 2, cc = c0 - 2 + q % kSpan;
        win[q / kSpan][q % kSpan] = (rr >= 0 && rr < H && cc >= 0 && cc < W) ? st[rr * W + cc] : kEmpty;
    }
    __syncthreads();
    const int c = c0 + static_cast<int>(threadIdx.x);
    uint32_t q = 0;
    if (c < W && win[2][threadIdx.x + 2] == kGround) {
#pragma unroll
        for (int dr = 0; dr < 5; ++dr)
#pragma unroll
            for (int dc = 0; dc < 5; ++dc) q |= win[dr][threadIdx.x + dc] == kObstacle ? 1u : 0u;
    }
    const uint64_t mask = __ballot(q != 0);
    if (lane_id() == 0 && c < W) d.qmask[(size_t)f * L.qruns + r * queue_runs(W) + c / kWave] = mask;
}

// The queue in raster order: a workgroup compacts 32 runs of 64 pixels, after
// the queue pixels of the runs before, which it counts itself (a launch that
// left the count of every tile cost more: one 64x2048 frame 13.3 -> 7.5 us).
// qlist[j] is the pixel of queue entry j, qmap[p] the queue index of pixel p
// or, for a pixel that is not queued, its static label source (negative),
// qrow[r] the first queue index at or after row r's first pixel (kept for the
// row solve); the last tile writes the queue length.
constexpr int kFillThreads = 256;
constexpr int kFillRuns = 8;  // per wavefront, their loads in flight together
constexpr int kFillTile = kFillRuns * kFillThreads / kWave;

__global__ __launch_bounds__(kFillThreads) void k_jcp_fill(DevBuf d, Layout L) {
    __shared__ uint32_t lds[kFillThreads / kWave + 1];
    const int f = blockIdx.y;
    const FrameDesc& fd = d.frames[f];
    const int W = fd.sc.W;
    const int per_row = queue_runs(W);
    const int runs = fd.sc.H * per_row;
    const int first = static_cast<int>(blockIdx.x) * kFillTile;
    if (first >= runs) return;
    const uint64_t* mask = d.qmask + (size_t)f * L.qruns;
    const int lane = lane_id();
    const int w = static_cast<int>(threadIdx.x) / kWave;
    const size_t po = (size_t)f * L.P;
    int p[kFillRuns];
    uint8_t st[kFillRuns];
#pragma unroll
    for (int k = 0; k < kFillRuns; ++k) {
        const int run = first + w * kFillRuns + k;
        const int c = run % per_row * kWave + lane;
        p[k] = run < runs && c < W ? run / per_row * W + c : -1;
        st[k] = d.state[fd.pix_off + max(p[k], 0)];
    }
    // Every wavefront has the tile's masks and their sums, a run per lane.
    const uint64_t mine = lane < kFillTile && first + lane < runs ? mask[first + lane] : 0ull;
    uint32_t before = 0, base;
    for (int i = threadIdx.x; i < first; i += kFillThreads) before += static_cast<uint32_t>(__popcll(mask[i]));
    block_exclusive_sum<kFillThreads>(before, lds, &base);
    const uint32_t incl = base + wave_inclusive_sum(static_cast<uint32_t>(__popcll(mine)));
#pragma unroll
    for (int k = 0; k < kFillRuns; ++k) {
        const uint64_t m = __shfl(mine, w * kFillRuns + k, kWave);
        const uint32_t end = __shfl(incl, w * kFillRuns + k, kWave);
        if (p[k] < 0) continue;
        const int j = static_cast<int>(end - static_cast<uint32_t>(__popcll(m >> lane)));
        if (p[k] % W == 0) d.qrow[(size_t)f * (L.H + 1) + p[k] / W] = j;
        if ((m >> lane) & 1ull) {
            d.qlist[po + j] = p[k];
            d.qmap[po + p[k]] = j;
        } else {
            d.qmap[po + p[k]] = st[k] == kGround ? kSrcGround : (st[k] == kObstacle ? kSrcObstacle : kSrcUnknown);
        }
    }
    if (threadIdx.x == kWave - 1 && first + kFillTile >= runs) d.fs[f * kFsCount + kFsQueue] = incl;
}

// A queue pixel's slots, as the row solve reads them: the head slots 0..11
// (rows -2, -1 and the two left neighbours) with their weights and label
// entries, and the tail slots 12..23 (right neighbours, rows +1, +2).  A tail
// slot names a neighbour raster-after its writer (the pixel itself or, stale,
// an earlier queue pixel), so its label is static or pending and its weight is
// stored with a sign: + obstacle, - ground, 0 neither.
// A record is eight 16-byte parts, part k of queue pixel j at [k * P + j] of
// the frame's records, so neighbouring lanes read neighbouring addresses:
//   0..2  head weights 0..11 (float)
//   3     head entries 0..7, 16 bits each (low half; see kLabelBase)
//   4     head entries 8..11, the sum of the tail (float), flags
//   5..7  tail weights 12..23 (float)
// flags: bits 0..11 bit 16 of the entries; bits kRecScale.. log2 of the
// weights' sum, rounded up; kRecTail, kRecOk.  The solve's fast path reads
// parts 0 to 4.
constexpr int kRecordParts = 8;
static_assert(kRecordParts * 16 == kSlotRecordBytes, "slot records fill their array");
constexpr int kRecScale = 12;
constexpr uint32_t kRecTail = 1u << 30;  // some tail weight is not zero
constexpr uint32_t kRecOk = 1u << 31;    // the weight sum passes the reference's test

// Label entries: 0, 1, 2 are the static sources kSrcObstacle, kSrcGround and
// kSrcUnknown, queue pixel j is entry j + kLabelBase.  A label is +1 for an
// obstacle, -1 for ground and 0 for neither.
constexpr int kLabelBase = 3;
static_assert(kSrcObstacle + kLabelBase == 0 && kSrcGround + kLabelBase == 1 && kSrcUnknown + kLabelBase == 2,
              "static sources are the first three label entries");

struct SlotVal {
    float u;
    int32_t src;
    bool near;
};

// Slot value computed by evaluator pixel `pe` (core point `core`) for its
// neighbour pixel np with record nb and source qm (segmenter.cpp:558-606).
__device__ __forceinline__ SlotVal eval_slot(const SegConst& s, int pe, float4 core, int np, float4 nb, int qm) {
    SlotVal v{0.0f, kSrcUnknown, false};
    if (__float_as_int(nb.w) == -1) return v;  // w holds the pixel's winner, -1 when empty
    const float dx = core.x - nb.x;
    const float dy = core.y - nb.y;
    const float dz = core.z - nb.z;
    const float d2 = dx * dx + dy * dy + dz * dz;
    if (d2 > s.kthr2) return v;
    v.u = glibc_expf(s.neg_amp * sqrtf(d2));
    v.near = true;
    v.src = (qm >= 0 && np >= pe) ? kSrcUnknown : qm;  // later queue pixels are still pending
    return v;
}

// Per queue pixel: the 24 slot weights w_i = u_i / sum and label sources,
// including stale slots resolved through their writer.  A workgroup takes 64
// queue pixels and a wavefront four slots of each, lane by lane consecutive
// pixels, so its reads are mostly neighbours; the slots meet in LDS for the
// ordered sums.  With a lane doing all 24 slots of a pixel the code was long,
// straight and cold in every launch, and few wavefronts had work (35 us for
// one 64x2048 frame with the records read one after the other, 22 with all of
// them requested first, now 8.5; 32x1024 20 -> 7.3; eight 128x2048 frames 28 ->
// 19; 32 frames of 64x2048 keep the chip busy either way, 51 us).
constexpr int kSlotWaves = 6;
constexpr int kWaveSlots = 24 / kSlotWaves;
static_assert(kWaveSlots == 4, "a wavefront's weights are one part of the record");

__global__ __launch_bounds__(kSlotWaves* kWave) void k_jcp_slots(DevBuf d, Layout L) {
    __shared__ float lw[24][kWave];     // u, then the weights
    __shared__ float ltail[12][kWave];  // signed tail weights
    __shared__ uint32_t lent[12][kWave];
    int tile, f;
    xcd_tile_frame(tile, f);
    const FrameDesc& fd = d.frames[f];
    const SegConst& s = fd.sc;
    const int nq = static_cast<int>(d.fs[f * kFsCount + kFsQueue]);
    const int lane = lane_id();
    const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
    const int H = s.H, W = s.W;
    const float4* px = d.pxyz + fd.pix_off;
    const size_t qo = (size_t)f * L.P;
    const int32_t* qm = d.qmap + qo;
    const int32_t* ql = d.qlist + qo;
    const int32_t* qrow = d.qrow + (size_t)f * (L.H + 1);
    const size_t P = static_cast<size_t>(L.P);
    for (int j0 = tile * kWave; j0 < nq; j0 += static_cast<int>(gridDim.x) * kWave) {
        const int j = min(j0 + lane, nq - 1);  // past the end: the last one again, not written
        const bool mine = j0 + lane < nq;
        const int p = ql[j];
        const int r = p / W, c = p % W;
        const float4 core = px[p];
        float4 nb[kWaveSlots];
        int32_t nq_src[kWaveSlots];
    #pragma unroll
        for (int k = 0; k < kWaveSlots; ++k) {
            const int i = w * kWaveSlots + k;
            const int np = min(max(r + kOffR[i], 0), H - 1) * W + min(max(c + kOffC[i], 0), W - 1);
            nb[k] = px[np];
            nq_src[k] = qm[np];
        }
        float u[kWaveSlots];
        int32_t src[kWaveSlots];
    #pragma unroll
        for (int k = 0; k < kWaveSlots; ++k) {
            const int dr = kOffR[w * kWaveSlots + k], dc = kOffC[w * kWaveSlots + k];
            const int nr = r + dr, nc = c + dc;
            SlotVal v{0.0f, kSrcUnknown, false};  // slots start at zero / UNKNOWN (segmenter.cpp:523-525)
            if (nr >= 0 && nr < H && nc >= 0 && nc < W) {
                v = eval_slot(s, p, core, nr * W + nc, nb[k], nq_src[k]);
            } else {
                // Stale slot: find the last earlier queue pixel for which this
                // slot was inside the image.
                const int rlo = max(0, -dr), rhi = min(H, H - dr);
                const int clo = max(0, -dc), chi = min(W, W - dc);
                // None in an image too small for the slot: rows rlo .. rhi - 1
                // exist below.
                int khi = rlo < rhi ? j - 1 : -1, klo = 0;
                // First queue index at or after a row's first pixel: qrow.
                if (rlo < rhi && rhi < H) khi = min(khi, qrow[rhi] - 1);
                if (rlo < rhi && rlo > 0) klo = qrow[rlo];
                int q = -1;
                for (int e = khi; e >= klo && q < 0; --e) {
                    const int pk = ql[e], qc = pk % W;
                    if (qc >= clo && qc < chi) q = pk;
                }
                if (q >= 0) {
                    const int np = (q / W + dr) * W + q % W + dc;
                    v = eval_slot(s, q, px[q], np, px[np], qm[np]);
                    v.near = false;  // no part of this pixel's sum
                }
            }
            u[k] = v.u;
            src[k] = v.src;
            // What the sum takes: slots without a near neighbour add nothing
            // (their u is +0 as the sum's start is, so adding it changes nothing).
            lw[w * kWaveSlots + k][lane] = v.near ? v.u : 0.0f;
        }
        __syncthreads();
        float sum = 0.0f;
    #pragma unroll
        for (int i = 0; i < 24; ++i) sum += lw[i][lane];
        __syncthreads();
        const bool ok = fabsf(sum) > 1.1920928955078125e-07f;  // FLT_EPSILON
        // An infinite sum makes every weight 0 or NaN: the reference's comparison
        // is false then, as it is without any weight.
        const bool weigh = ok && sum < __builtin_inff();
        uint4* rec = d.slot_rec + qo * kRecordParts + j;
        float part[kWaveSlots];
    #pragma unroll
        for (int k = 0; k < kWaveSlots; ++k) {
            const int i = w * kWaveSlots + k;
            const float t = weigh ? u[k] / sum : 0.0f;
            lw[i][lane] = t;
            if (i < 12) {
                part[k] = t;
                lent[i][lane] = static_cast<uint32_t>((t > 0.0f ? src[k] : kSrcUnknown) + kLabelBase);
            } else {
                part[k] = src[k] == kSrcObstacle ? t : (src[k] == kSrcGround ? -t : 0.0f);
                ltail[i - 12][lane] = part[k];
            }
        }
        if (mine)
            rec[(w < 3 ? w : w + 2) * P] = make_uint4(__float_as_uint(part[0]), __float_as_uint(part[1]),
                                                      __float_as_uint(part[2]), __float_as_uint(part[3]));
        __syncthreads();
        if (w == 0 && mine) {
            uint32_t flags = ok ? kRecOk : 0u;
            float tail_sum = 0.0f, total = 0.0f;
            uint32_t entry[12];
        #pragma unroll
            for (int i = 0; i < 12; ++i) {
                const uint32_t e = lent[i][lane];
                entry[i] = e & 0xffffu;
                flags |= (e >> 16) << i;
                const float t = ltail[i][lane];
                tail_sum += t;
                if (t != 0.0f) flags |= kRecTail;
                total += lw[i][lane] + lw[12 + i][lane];
            }
            // The pixel's own weights sum to 1; stale ones come on top, divided by a
            // sum they are not part of.
            if (total > 1.5f) flags |= min(((__float_as_uint(total) >> 23) & 0xffu) - 126u, 140u) << kRecScale;
            rec[3 * P] = make_uint4(entry[0] | entry[1] << 16, entry[2] | entry[3] << 16, entry[4] | entry[5] << 16,
                                    entry[6] | entry[7] << 16);
            rec[4 * P] =
                make_uint4(entry[8] | entry[9] << 16, entry[10] | entry[11] << 16, __float_as_uint(tail_sum), flags);
        }
        __syncthreads();
    }
}

constexpr int kSolveThreads = 512;
constexpr int kSolveWaves = kSolveThreads / kWave;
constexpr int kQueueMax = 65536;  // labels of one frame's queue in LDS
constexpr int kSolveRows = 1024;  // image rows
constexpr int kSolveAhead = 4;    // chunks whose records are in registers
constexpr int kSolveChunks = kSolveRows + kQueueMax / kSolveThreads;  // at most: one per row, and per full chunk

// A difference of weight sums further than this from zero, times the power of
// two at or above the weights' sum (1 without stale weights), has the sign of
// the reference's: its two ordered float sums and the difference formed here
// are each within some 24 * 2^-24 of that sum (4.3e-6 in all).
constexpr float kSumMargin = 1.0e-5f;

// Parts 0..4 of a record, and the flags of one of the two records before the
// wavefront's (lane 0 the last, lane 1 the one before).
struct SlotData {
    uint4 part[5];
    uint32_t before;
};

// Records of the chunk [first, end), first <= nq.  Lanes past its end read its
// last record: a wavefront without a pixel reads one line a load.
__device__ __forceinline__ void load_slots(const uint4* rec, size_t P, int first, int end, SlotData& sd) {
    const int last = max(end - 1, 0);
    // 32-bit byte offsets from each part's (uniform) base.
    const uint32_t o = static_cast<uint32_t>(min(first + static_cast<int>(threadIdx.x), last)) * 16u;
#pragma unroll
    for (int k = 0; k < 5; ++k)
        sd.part[k] = *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(rec + k * P) + o);
    const int wave_first = first + (static_cast<int>(threadIdx.x) & ~(kWave - 1));
    const uint32_t b = static_cast<uint32_t>(min(max(wave_first - 1 - (lane_id() & 1), 0), last)) * 16u;
    sd.before = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(rec + 4 * P) + 12 + b);
}

// Transfer map of a queue pixel: the pair state 2 * (label of j - 2 is
// obstacle) + (label of j - 1 is obstacle) to the next one, byte k the image
// of state k.  Composing f after g is one byte permute.  A pixel left pending
// counts as ground here; the pixels after it do not weigh it.
constexpr uint32_t kMapIdentity = 0x03020100u;
constexpr uint32_t kMapShift = 0x02000200u;  // state k with its older label dropped and a ground appended

__device__ __forceinline__ uint32_t map_compose(uint32_t f, uint32_t g) { return __builtin_amdgcn_perm(f, f, g); }

template <int kCtrl, int kRowMask>
__device__ __forceinline__ uint32_t map_dpp(uint32_t m) {
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(static_cast<int>(kMapIdentity), static_cast<int>(m), kCtrl,
                                                             kRowMask, 0xf, false));
}

// Inclusive scan of the wavefront's maps, m := m_lane o ... o m_0: row
// shifts by 1, 2, 4 and 8 inside each 16-lane row, then lane 15 of rows 0 / 2
// into rows 1 / 3 and lane 31 into rows 2 and 3.
__device__ __forceinline__ uint32_t map_wave_scan(uint32_t m) {
    m = map_compose(m, map_dpp<0x111, 0xf>(m));
    m = map_compose(m, map_dpp<0x112, 0xf>(m));
    m = map_compose(m, map_dpp<0x114, 0xf>(m));
    m = map_compose(m, map_dpp<0x118, 0xf>(m));
    m = map_compose(m, map_dpp<0x142, 0xa>(m));
    m = map_compose(m, map_dpp<0x143, 0xc>(m));
    return m;
}

// Value of the lane below (lane 0 reads `first`).
__device__ __forceinline__ uint32_t lane_below(uint32_t v, uint32_t first) {
    return static_cast<uint32_t>(
        __builtin_amdgcn_update_dpp(static_cast<int>(first), static_cast<int>(v), 0x138, 0xf, 0xf, false));
}

// Row-ordered exact solve, one workgroup per frame.  A chunk is up to 512
// queue pixels of one row; all labels of earlier chunks are final in LDS.
// Each pixel sums its known slots (at most twelve label reads); open are at
// most the two queue pixels before it, with weights a1 and a2, so its label as
// a function of theirs is four signs, and the row is a scan of four-byte maps.
// Signs within rounding of zero are taken from the reference's ordered sums.
// The kernel is a chain of rows, bound by latency: each chunk is an LDS read,
// some 120 instructions and two barriers, and the records are read
// kSolveAhead - 1 chunks ahead, more than the time of a memory access.  140 ->
// 63 us for a 64x2048 frame of 16 000 queue pixels (154 -> 68 us for 32): a
// chunk took nine-entry maps built from nine pairs of ordered sums before.
// Label entries beyond 16 bits occur in queues of more than 65533 pixels only
// (kWide): their upper bit costs every slot two instructions.
struct SolveLds {
    int8_t lab[kLabelBase + kQueueMax];
    int chunk_base[kSolveChunks + 2 + kSolveAhead];
    uint32_t wtot[kSolveWaves];
    int scan[kSolveWaves + 1];
};

template <bool kWide>
__device__ __forceinline__ void solve_rows(const uint4* rec, size_t P, int nq, int chunks, SolveLds& lds) {
    const int tid = threadIdx.x;
    const int w = tid / kWave;
    const int lane = lane_id();
    int8_t* lab = lds.lab;
    const int* chunk_base = lds.chunk_base;
    uint32_t* wtot = lds.wtot;
    auto chunk = [&](SlotData& sd, int base, int end, int ahead, int ahead_end) {
        const int j = base + tid;
        const bool any = base + w * kWave < end;
        uint32_t m = kMapIdentity;
        const uint32_t flags = sd.part[4].w;
        if (any) {
            float hw[12];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                hw[4 * k] = __uint_as_float(sd.part[k].x);
                hw[4 * k + 1] = __uint_as_float(sd.part[k].y);
                hw[4 * k + 2] = __uint_as_float(sd.part[k].z);
                hw[4 * k + 3] = __uint_as_float(sd.part[k].w);
            }
            const uint32_t ew[6] = {sd.part[3].x, sd.part[3].y, sd.part[3].z, sd.part[3].w, sd.part[4].x, sd.part[4].y};
            int e[12], l[12];
#pragma unroll
            for (int i = 0; i < 12; ++i) e[i] = static_cast<int>((i & 1) ? ew[i / 2] >> 16 : ew[i / 2] & 0xffffu);
            if (kWide) {
#pragma unroll
                for (int i = 0; i < 12; ++i) e[i] |= static_cast<int>(((flags >> i) & 1u) << 16);
            }
            // Slots 10 and 11 may name the two queue pixels before this one
            // in the chunk; a pending one has no label.
            const int first = base + kLabelBase;
            const bool in10 = e[10] >= first, in11 = e[11] >= first;
            const uint32_t ok = flags >> 31;
            const uint32_t ok1 = lane_below(ok, static_cast<uint32_t>(__builtin_amdgcn_readlane(
                                                    static_cast<int>(sd.before), 0)) >> 31);
            const uint32_t ok2 = lane_below(ok1, static_cast<uint32_t>(__builtin_amdgcn_readlane(
                                                     static_cast<int>(sd.before), 1)) >> 31);
            const bool one = e[10] == j - 1 + kLabelBase;
            float a1 = in11 ? hw[11] : 0.0f, a2 = in10 && !one ? hw[10] : 0.0f;
            if (in10 && one) a1 += hw[10];
            if (!ok1) a1 = 0.0f;
            if (!ok2) a2 = 0.0f;
            if (in10) e[10] = 2;
            if (in11) e[11] = 2;
#pragma unroll
            for (int i = 0; i < 12; ++i) l[i] = lab[e[i]];
            float d0 = __uint_as_float(sd.part[4].z);
            int seen = 0;
#pragma unroll
            for (int i = 0; i < 12; ++i) {
                d0 = __builtin_fmaf(hw[i], static_cast<float>(l[i]), d0);
                seen |= l[i];
            }
            // Without any other label the sign of a1, a2 is exact (and 0 is
            // ground, as in the reference).
            const bool alone = seen == 0 && !(flags & kRecTail);
            const float margin =
                alone ? -1.0f : __uint_as_float(__float_as_uint(kSumMargin) + (((flags >> kRecScale) & 0xffu) << 23));
            const float p = d0 + a1, q = d0 - a1;
            const float v0 = q - a2, v1 = p - a2, v2 = q + a2, v3 = p + a2;
            m = kMapShift | (v0 > 0.0f ? 1u : 0u) | (v1 > 0.0f ? 1u << 8 : 0u) | (v2 > 0.0f ? 1u << 16 : 0u) |
                (v3 > 0.0f ? 1u << 24 : 0u);
            const float least = fminf(fminf(fabsf(v0), fabsf(v1)), fminf(fabsf(v2), fabsf(v3)));
            if (j < end && ok && !(least > margin)) {
                // The ordered sums of segmenter.cpp:613-626 (wg += w for a
                // GROUND slot, wo += w for an OBSTACLE slot, as adds of w or
                // +0: weights are +0 or positive and the sums start at +0, so
                // adding +0 changes nothing), for each pair of open labels.
                float tail[12];
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const uint4 t = rec[(5 + k) * P + j];
                    tail[4 * k] = __uint_as_float(t.x);
                    tail[4 * k + 1] = __uint_as_float(t.y);
                    tail[4 * k + 2] = __uint_as_float(t.z);
                    tail[4 * k + 3] = __uint_as_float(t.w);
                }
                m = kMapShift;
                const bool open = a1 > 0.0f || a2 > 0.0f;  // else one pair stands for all
#pragma nounroll
                for (int k = 0; k < (open ? 4 : 1); ++k) {
                    const int s1 = ok1 ? 2 * (k & 1) - 1 : 0, s2 = ok2 ? (k & 2) - 1 : 0;
                    float g = 0.0f, o = 0.0f;
#pragma unroll
                    for (int i = 0; i < 12; ++i) {
                        int v = l[i];
                        if (i == 10 && in10) v = one ? s1 : s2;
                        if (i == 11 && in11) v = s1;
                        g += v < 0 ? hw[i] : 0.0f;
                        o += v > 0 ? hw[i] : 0.0f;
                    }
#pragma unroll
                    for (int i = 0; i < 12; ++i) {
                        g += tail[i] < 0.0f ? -tail[i] : 0.0f;
                        o += tail[i] > 0.0f ? tail[i] : 0.0f;
                    }
                    if (o > g) m |= open ? 1u << (8 * k) : 0x01010101u;
                }
            }
            if (!ok) m = kMapShift;
            if (j >= end) m = kMapIdentity;
            m = map_wave_scan(m);
        }
        if (lane == kWave - 1) wtot[w] = m;
        __syncthreads();
        // State before the wavefront: the totals of the wavefronts before it,
        // from state 0 (nothing in a chunk hangs on pixels before it).
        uint32_t t = lane < kSolveWaves ? wtot[lane] : kMapIdentity;
        load_slots(rec, P, ahead, ahead_end, sd);
        t = map_compose(t, map_dpp<0x111, 0xf>(t));
        t = map_compose(t, map_dpp<0x112, 0xf>(t));
        t = map_compose(t, map_dpp<0x114, 0xf>(t));
        static_assert(kSolveWaves <= 8, "three row-shift steps scan at most 8 wavefront totals");
        const uint32_t state = w > 0 ? static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(t), w - 1)) & 3u : 0u;
        if (j < end) {
            const uint32_t s = (m >> (8 * state)) & 1u;
            lab[j + kLabelBase] = static_cast<int8_t>((flags & kRecOk) ? (s ? 1 : -1) : 0);
        }
        __syncthreads();
    };
    int base[kSolveAhead + 2];
    SlotData sd[kSolveAhead];
#pragma unroll
    for (int k = 0; k <= kSolveAhead + 1; ++k) base[k] = __builtin_amdgcn_readfirstlane(chunk_base[min(k, chunks)]);
    // Records of the chunk kSolveAhead further replace those just used; the
    // index is clamped and the order of the loads is kept, so every path has
    // the same loads in flight and the compiler waits for the oldest only.
#pragma unroll
    for (int k = 0; k < kSolveAhead; ++k) {
        load_slots(rec, P, base[k], base[k + 1], sd[k]);
        __builtin_amdgcn_sched_barrier(0);
    }
    // (The steps are not left early for the same reason: past the last chunk
    // they have no pixel.)
    for (int c = 0; c < chunks; c += kSolveAhead) {
#pragma unroll
        for (int k = 0; k < kSolveAhead; ++k) {
            const int after = chunk_base[min(c + k + kSolveAhead + 2, chunks)];
            chunk(sd[k], base[0], base[1], base[kSolveAhead], base[kSolveAhead + 1]);
#pragma unroll
            for (int q = 0; q <= kSolveAhead; ++q) base[q] = base[q + 1];
            base[kSolveAhead + 1] = __builtin_amdgcn_readfirstlane(after);
        }
    }
}

__global__ __launch_bounds__(kSolveThreads) void k_jcp_solve(DevBuf d, Layout L) {
    __shared__ SolveLds lds;
    const int f = blockIdx.x;
    const FrameDesc& fd = d.frames[f];
    const int H = fd.sc.H;
    const int nq = static_cast<int>(d.fs[f * kFsCount + kFsQueue]);
    const int tid = threadIdx.x;
    if (nq > kQueueMax || H > kSolveRows) {
        if (tid == 0) atomicOr(&d.fs[f * kFsCount + kFsErr], kErrQueueCapacity);
        return;
    }
    if (nq == 0) return;
    const size_t qo = (size_t)f * L.P;
    const uint4* rec = d.slot_rec + qo * kRecordParts;
    const size_t P = static_cast<size_t>(L.P);
    // Chunks in queue order, two rows per thread: a row's chunks start at its
    // first queue pixel and every kSolveThreads further.  A chunk ends where
    // the next begins; past the last one every base is nq.
    const int32_t* qrow = d.qrow + (size_t)f * (L.H + 1);
    auto row_at = [&](int r) { return r < H ? qrow[r] : nq; };
    const int r0 = 2 * tid, b0 = row_at(r0), b1 = row_at(r0 + 1), b2 = row_at(r0 + 2);
    const int n0 = (b1 - b0 + kSolveThreads - 1) / kSolveThreads, n1 = (b2 - b1 + kSolveThreads - 1) / kSolveThreads;
    int chunks;
    const int c0 = block_exclusive_sum<kSolveThreads>(n0 + n1, lds.scan, &chunks);
    for (int k = 0; k < n0; ++k) lds.chunk_base[c0 + k] = b0 + k * kSolveThreads;
    for (int k = 0; k < n1; ++k) lds.chunk_base[c0 + n0 + k] = b1 + k * kSolveThreads;
    if (tid < 2 + kSolveAhead) lds.chunk_base[chunks + tid] = nq;
    if (tid < kLabelBase) lds.lab[tid] = static_cast<int8_t>(tid == 0 ? 1 : (tid == 1 ? -1 : 0));
    __syncthreads();
    chunks = __builtin_amdgcn_readfirstlane(chunks);
    if (nq > (1 << 16) - kLabelBase)
        solve_rows<true>(rec, P, nq, chunks, lds);
    else
        solve_rows<false>(rec, P, nq, chunks, lds);
    for (int j = tid; j < nq; j += kSolveThreads) {
        const int v = lds.lab[j + kLabelBase];
        d.fin[qo + j] = v < 0 ? kGround : (v > 0 ? kObstacle : kPending);
    }
}

// Labels per input point (populateLabels, segmenter.cpp:640-669): only the
// winner of a pixel gets its pixel's final label; PENDING stays UNKNOWN.
__device__ __forceinline__ void seg_labels_tile(const DevBuf& d, const Layout& L, int f, int tile) {
    const FrameDesc& fd = d.frames[f];
    const int i = tile * blockDim.x + threadIdx.x;
    if (i >= fd.n) return;
    const int gi = fd.pt_off + i;
    uint32_t lab = LP_LABEL_UNKNOWN;
    const int pix = d.pt_pix[gi];
    if (pix >= 0) {
        const unsigned long long key = d.pix_key[fd.pix_off + pix];
        if (static_cast<int>(key & ((1ull << L.idx_bits) - 1)) == i) {
            const int qm = d.qmap[(size_t)f * L.P + pix];
            const uint8_t st = qm >= 0 ? d.fin[(size_t)f * L.P + qm] : d.state[fd.pix_off + pix];
            lab = st == kGround ? LP_LABEL_GROUND : (st == kObstacle ? LP_LABEL_OBSTACLE : LP_LABEL_UNKNOWN);
        }
    }
    d.labels[gi] = lab;
    // Obstacles of every 64 points, for the split that follows.
    const uint64_t obs = __ballot(lab == LP_LABEL_OBSTACLE);
    if (lane_id() == 0) d.obs_rows[(size_t)f * L.obs_rows + i / kWave] = static_cast<uint32_t>(__popcll(obs));
    if (d.gnd_flag) d.gnd_flag[(size_t)f * L.N + i] = lab == LP_LABEL_GROUND ? 1u : 0u;
}

__global__ void k_seg_labels(DevBuf d, Layout L) { seg_labels_tile(d, L, blockIdx.y, blockIdx.x); }

__global__ __launch_bounds__(256) void k_seg_labels_q(DevBuf d, Layout L, int B) {
    wq_run(d.wq + kWqSegLabels * 8, B, blockDim.x, [&](int f) { return d.frames[f].n; },
           [&](int f, int t) { seg_labels_tile(d, L, f, t); });
}

// Segmenter::image after segment() (segmenter.hpp:163-166), as BGR bytes.
// The winners paint ground green and obstacles red (segmenter.cpp:288-318);
// the red channel is dilated with a 5x5 rectangle whose out-of-image part
// never contributes (:484-489), which turns empty pixels near an obstacle
// red and ground pixels near one yellow; yellow pixels with a point become
// the blue JCP queue (:491-513) and take the JCP colour where the weights
// resolve (:626-635).  A yellow pixel without a point (white, :510) cannot
// occur: only a winner paints green.
__global__ void k_label_image(DevBuf d, Layout L, int f, uint8_t* img) {
    const FrameDesc& fd = d.frames[f];
    const int H = fd.sc.H, W = fd.sc.W;
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= H * W) return;
    const uint8_t* st = d.state + fd.pix_off;
    const int qm = d.qmap[(size_t)f * L.P + p];
    uint8_t b = 0, g = 0, r = 0;
    const uint8_t s = qm >= 0 ? d.fin[(size_t)f * L.P + qm] : st[p];
    if (s == kGround) {
        g = 255;
    } else if (s == kObstacle) {
        r = 255;
    } else if (s == kPending) {
        b = 255;
    } else {
        const int row = p / W, col = p % W;
        for (int dr = -2; dr <= 2 && !r; ++dr) {
            const int rr = row + dr;
            if (rr < 0 || rr >= H) continue;
            for (int dc = -2; dc <= 2; ++dc) {
                const int cc = col + dc;
                if (cc >= 0 && cc < W && st[rr * W + cc] == kObstacle) {
                    r = 255;
                    break;
                }
            }
        }
    }
    img[3 * p + 0] = b;
    img[3 * p + 1] = g;
    img[3 * p + 2] = r;
}

void launch_jcp(lp_context* c, int B) {
    DevBuf& d = c->d;
    const Layout& L = c->L;
    hipStream_t st = c->stream;
    stage_mark(c, "jcp_queue");
    const int mt = c->mark_tile;
    if (mt == 64)
        hipLaunchKernelGGL(k_jcp_mark<64>, dim3(L.H * ((L.W + 63) / 64), B), dim3(64), 0, st, d, L);
    else if (mt == 128)
        hipLaunchKernelGGL(k_jcp_mark<128>, dim3(L.H * ((L.W + 127) / 128), B), dim3(128), 0, st, d, L);
    else
        hipLaunchKernelGGL(k_jcp_mark<256>, dim3(L.H * ((L.W + 255) / 256), B), dim3(256), 0, st, d, L);
    hipLaunchKernelGGL(k_jcp_fill, dim3((L.qruns + kFillTile - 1) / kFillTile, B), dim3(kFillThreads), 0, st, d, L);
    stage_mark(c, "jcp_slots");
    // A workgroup for each 64 pixels of a frame's queue when they are few; on
    // larger batches about 4096 in all, several turns each (most of a frame's
    // pixels are not queued, so one for each 64 of them would mostly be empty).
    hipLaunchKernelGGL(k_jcp_slots, dim3(std::min((L.P + kWave - 1) / kWave, std::max(64, 4096 / B)), B),
                       dim3(kSlotWaves * kWave), 0, st, d, L);
    stage_mark(c, "jcp_solve");
    hipLaunchKernelGGL(k_jcp_solve, dim3(B), dim3(kSolveThreads), 0, st, d, L);
    stage_mark(c, "labels");
    const int wg = c->point_wg;
    if (c->persistent)
        hipLaunchKernelGGL(k_seg_labels_q, dim3(kPersistentWorkgroups), dim3(wg), 0, st, d, L, B);
    else
        hipLaunchKernelGGL(k_seg_labels, dim3((L.N + wg - 1) / wg, B), dim3(wg), 0, st, d, L);
}

void launch_label_image(lp_context* c, int f, int pixels, uint8_t* img) {
    hipLaunchKernelGGL(k_label_image, dim3((pixels + 255) / 256), dim3(256), 0, c->stream, c->d, c->L, f, img);
}

}  // namespace lp
