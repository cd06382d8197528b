// lp_scan.hip -- reduce-then-scan exclusive prefix sums over per-frame
// arrays whose lengths are only known on the device (point counts, queue
// lengths, obstacle counts), so the launch shape stays fixed for graphs.
#include "lp_kernels.h"

namespace lp {

using namespace lpd;

constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;

__device__ __forceinline__ int scan_count(const DevBuf& d, int f, ScanCount kind, int slot) {
    const FrameDesc& fd = d.frames[f];
    if (kind == kCountPoints) return fd.n;
    if (kind == kCountRawPoints) return fd.n_raw;
    return static_cast<int>(d.fs[f * kFsCount + slot]);
}

__global__ __launch_bounds__(kScanThreads) void k_scan_reduce(DevBuf d, Layout L, const uint32_t* in, size_t stride,
                                                              ScanCount kind, int slot) {
    __shared__ uint32_t lds[kScanThreads / kWave + 1];
    const int f = blockIdx.y;
    const int n = scan_count(d, f, kind, slot);
    const int base = blockIdx.x * kScanTile;
    if (base >= n) return;
    uint32_t s = 0;
    const int b = base + threadIdx.x * kScanItems;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k)
        if (b + k < n) s += in[(size_t)f * stride + b + k];
    uint32_t total;
    block_exclusive_sum<kScanThreads>(s, lds, &total);
    if (threadIdx.x == 0) d.blk[(size_t)f * L.blk_stride + blockIdx.x] = total;
}

// Down pass: each tile adds the totals of the tiles before it (read straight
// from the reduce pass, at most blk_stride of them) to its own exclusive
// scan; the last tile writes the frame total.  Two launches per scan.
__global__ __launch_bounds__(kScanThreads) void k_scan_down(DevBuf d, Layout L, const uint32_t* in, uint32_t* out,
                                                            size_t stride, ScanCount kind, int slot,
                                                            int total_slot) {
    __shared__ uint32_t lds[kScanThreads / kWave + 1];
    const int f = blockIdx.y;
    const int n = scan_count(d, f, kind, slot);
    const int tile = blockIdx.x;
    const int base = tile * kScanTile;
    if (base >= n) {
        if (tile == 0 && threadIdx.x == 0 && total_slot >= 0) d.fs[f * kFsCount + total_slot] = 0;
        return;
    }
    const uint32_t* blk = d.blk + (size_t)f * L.blk_stride;
    uint32_t pre = 0;
    for (int i = threadIdx.x; i < tile; i += kScanThreads) pre += blk[i];
    uint32_t pre_total;
    block_exclusive_sum<kScanThreads>(pre, lds, &pre_total);
    uint32_t* o = out + (size_t)f * stride;
    uint32_t v[kScanItems];
    uint32_t s = 0;
    const int b = base + threadIdx.x * kScanItems;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        v[k] = (b + k < n) ? in[(size_t)f * stride + b + k] : 0u;
        s += v[k];
    }
    uint32_t total;
    uint32_t ex = block_exclusive_sum<kScanThreads>(s, lds, &total) + pre_total;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        if (b + k < n) o[b + k] = ex;
        ex += v[k];
    }
    if (threadIdx.x == 0 && total_slot >= 0 && base + kScanTile >= n)
        d.fs[f * kFsCount + total_slot] = pre_total + total;
}

void launch_scan(lp_context* c, int B, const uint32_t* in, uint32_t* out, size_t stride, ScanCount kind,
                 int count_slot, int total_slot) {
    const Layout& L = c->L;
    const int nb = (static_cast<int>(stride) + kScanTile - 1) / kScanTile;
    hipLaunchKernelGGL(k_scan_reduce, dim3(nb, B), dim3(kScanThreads), 0, c->stream, c->d, L, in, stride, kind,
                       count_slot);
    hipLaunchKernelGGL(k_scan_down, dim3(nb, B), dim3(kScanThreads), 0, c->stream, c->d, L, in, out, stride, kind,
                       count_slot, total_slot);
}

}  // namespace lp
