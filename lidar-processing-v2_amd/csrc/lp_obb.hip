// lp_obb.hip -- rotating-calipers oriented bounding boxes of hull polygons.
//
// Reference: lidar_processing_lib/src/polygonizer.cpp:93-161
// (findAntipodalPairsOfConvexHull, Shamos' walk with areaOfTriangle,
// polygonizer.hpp:228-231) and :163-278 (boundingBoxRotatingCalipers).  For
// every antipodal pair (i, j), for index in {i, j}, for offset in {-1, +1},
// the edge (index, index+offset) of length >= 1e-6 defines a frame in which
// the polygon's extents give a box; the first candidate, in that order, whose
// double area is below the running minimum replaces the box.  The running
// minimum is the box's float `area` member, so near-ties are decided against
// the float-rounded value exactly as the reference does.
//
// Polygons of up to 64 vertices (nearly all hulls) take one wavefront each,
// larger ones a workgroup, in one launch.  The antipodal walk is a serial
// chain (about 2.5 steps per vertex, 300 cycles each: two thirds of the
// stage's time when one lane walked it), but its state at every vertex i is
// where the area of (i, i+1, j) stops growing, so all rows are found at once
// by binary search and the whole walk is then checked step by step in
// parallel with the reference's own comparisons; a walk that differs anywhere
// (rounded ties, polygons that are not convex) is redone by one lane.  The
// candidates (i, -1) and (i - 1, +1) share one edge with opposite directions,
// which negates every rotated coordinate exactly and leaves the area
// bit-identical, so one area is evaluated per edge, O(n) each, a lane per
// edge; the sequential selection rule over the candidates is applied by two
// reductions.  64x2048 frame of 40 cars: 96 -> 19 us (two launches before),
// 331 polygons of 13 vertices on average: 81 -> 19 us.
#include <algorithm>

#include "lp_device.h"
#include "lp_internal.h"
#include "lp_kernels.h"

namespace lp {

using namespace lpd;

namespace {

constexpr int kBoxThreads = 256;
// Polygons of up to kBoxVerts vertices are held in LDS (larger: capacity
// error).
constexpr int kBoxVerts = 1024;

// areaOfTriangle (polygonizer.hpp:228-231), same operand order.
__device__ __forceinline__ double tri_area(const double2& a, const double2& b, const double2& c) {
    return fabs((a.x * (b.y - c.y) + b.x * (c.y - a.y) + c.x * (a.y - b.y)) * 0.5);
}

__device__ __forceinline__ int wrap(int k, int n) { return k >= n ? k - n : k; }

// Antipodal pairs of polygon V (n >= 3 vertices) in the reference's order
// (polygonizer.cpp:93-161), walked as one sequential chain with the areas of
// the running pair carried from step to step.  emit(i, j) receives the pairs.
// Returns false when the walk exceeds 4n + 8 steps or `cap` pairs (the
// reference's loop need not end on degenerate input).
template <typename Emit>
__device__ __forceinline__ bool antipodal_walk(const double2* V, int n, int cap, Emit emit) {
    const int i0 = n - 1;
    const int limit = 4 * n + 8;
    int guard = 0, count = 0;
    int i = 0, j = 1;
    double2 vi = V[0], vi1 = V[1], vj = V[1];
    int jn = wrap(2, n);
    double2 vn = V[jn];
    double a_cur = tri_area(vi, vi1, vj);
    // while (area(i, i+1, j+1) > area(i, i+1, j)) ++j
    for (;;) {
        const double a_nx = tri_area(vi, vi1, vn);
        if (!(a_nx > a_cur)) break;
        j = jn;
        vj = vn;
        a_cur = a_nx;
        jn = wrap(j + 1, n);
        vn = V[jn];
        if (++guard > limit) return false;
    }
    const int j0 = j;
    while (i != j0) {
        i = wrap(i + 1, n);
        vi = vi1;
        const int i1 = wrap(i + 1, n);
        vi1 = V[i1];
        if (count++ >= cap) return false;
        emit(i, j);
        a_cur = tri_area(vi, vi1, vj);
        for (;;) {
            const double a_nx = tri_area(vi, vi1, vn);
            if (!(a_nx > a_cur)) break;
            j = jn;
            vj = vn;
            a_cur = a_nx;
            jn = wrap(j + 1, n);
            vn = V[jn];
            if (i == j0 && j == i0) return true;
            if (count++ >= cap) return false;
            emit(i, j);
            if (++guard > limit) return false;
        }
        // areaOfTriangle(j, i+1, j+1) == areaOfTriangle(i, i+1, j)
        if (tri_area(vj, vi1, vn) == a_cur) {
            if (count++ >= cap) return false;
            if (i == j0 && j == i0)
                emit(i1, j);
            else
                emit(i, jn);
        }
        if (++guard > limit) return false;
    }
    return true;
}

// Extents of the polygon rotated into the frame of unit direction (ux, uy)
// about (cx, cy), as the reference computes them (std::min / std::max order).
struct Extent {
    double mnx, mxx, mny, mxy;
};

__device__ __forceinline__ void extent_add(Extent& e, double rx, double ry) {
    e.mnx = (rx < e.mnx) ? rx : e.mnx;  // std::min(min_x, x)
    e.mxx = (e.mxx < rx) ? rx : e.mxx;  // std::max(max_x, x)
    e.mny = (ry < e.mny) ? ry : e.mny;
    e.mxy = (e.mxy < ry) ? ry : e.mxy;
}

__device__ __forceinline__ Extent extent_init() {
    return Extent{1.7976931348623157e308, -1.7976931348623157e308, 1.7976931348623157e308,
                  -1.7976931348623157e308};
}

// Candidate edge (idx, idx + off) of the reference: unit direction, or
// false when shorter than 1e-6.
__device__ __forceinline__ bool cand_dir(const double2* V, int n, int idx, int off, double& ux, double& uy) {
    int nb = idx + off;
    if (nb < 0)
        nb += n;
    else if (nb >= n)
        nb -= n;
    const double ex = V[nb].x - V[idx].x;
    const double ey = V[nb].y - V[idx].y;
    const double len = sqrt(ex * ex + ey * ey);
    if (len < 1.0e-6) return false;
    ux = ex / len;
    uy = ey / len;
    return true;
}

// Area of the box in the frame of edge e (e -> e+1), or NaN when the edge is
// shorter than 1e-6.  The candidates (e, +1) and (e + 1, -1) share it.
// fmin / fmax keep the same extents as extent_add up to the sign of a zero,
// which can only show in an area of zero: such an edge is evaluated again in
// the reference's own order.
__device__ __forceinline__ double edge_box_area(const double2* V, int n, int e, double cx, double cy) {
    double ux, uy;
    if (!cand_dir(V, n, e, 1, ux, uy)) return __builtin_nan("");
    Extent ex = extent_init();
#pragma unroll 4
    for (int q = 0; q < n; ++q) {
        const double tx = V[q].x - cx;
        const double ty = V[q].y - cy;
        const double rx = tx * ux + ty * uy;
        const double ry = -tx * uy + ty * ux;
        ex.mnx = fmin(ex.mnx, rx);
        ex.mxx = fmax(ex.mxx, rx);
        ex.mny = fmin(ex.mny, ry);
        ex.mxy = fmax(ex.mxy, ry);
    }
    const double area = (ex.mxx - ex.mnx) * (ex.mxy - ex.mny);
    if (area != 0.0) return area;
    ex = extent_init();
    for (int q = 0; q < n; ++q) {
        const double tx = V[q].x - cx;
        const double ty = V[q].y - cy;
        extent_add(ex, tx * ux + ty * uy, -tx * uy + ty * ux);
    }
    return (ex.mxx - ex.mnx) * (ex.mxy - ex.mny);
}

// A group of NT threads (a wavefront, or the whole workgroup).
template <int NT>
__device__ __forceinline__ void group_sync() {
    if (NT == kWave)
        wave_sync();
    else
        __syncthreads();
}

// Whether `v` holds on any thread of the group; the group is in step
// afterwards.
template <int NT>
__device__ __forceinline__ bool group_any(bool v) {
    if (NT == kWave) {
        const bool r = __ballot(v) != 0;
        wave_sync();
        return r;
    }
    return __syncthreads_or(v ? 1 : 0) != 0;
}

// The smallest (area, position) pair and the last position are kept with the
// candidate they belong to: vertex * 2 + (offset + 1) / 2.
struct CandMin {
    double area;
    int pos;
    int cand;
};

__device__ __forceinline__ void cand_min(CandMin& m, double area, int pos, int cand) {
    if (area < m.area || (area == m.area && pos < m.pos)) m = CandMin{area, pos, cand};
}

// The candidate that the reference's sequential rule ends with, for a walk
// done by all NT threads: cand (as in CandMin) and the smallest area, or -1
// when no candidate has an area, or kWalkSerial when the sequential walk has
// to decide.  V, area in LDS; J (n entries), par (n / 32 + 1 words) and red
// (NT / 64 entries) are LDS scratch.
//
// Walk: row i starts at j = J[i - 1] (row 0 at 1) and advances to J[i], the
// first j whose next vertex does not enlarge the triangle (j runs on past n;
// vertex j - n is meant); rows run to j0 = J[0].  Element t of the walk is
// (i, t - i + 1) with i the first row with J[i] - 1 + i >= t.  Every element
// but a row's last must advance and the last must not; with that the rows are
// the sequential walk's, whatever guessed them.  Row j0 ends the walk when it
// advances to vertex n - 1.
//
// Rule: a candidate replaces the box when its area is below the float of the
// smallest area before it (float rounding is monotone, so that is the float
// running minimum of polygonizer.cpp:257).  After the first candidate of the
// overall smallest area m only areas below float(m) replace, so the last of
// those is the answer; without one it is that first candidate, if m is below
// the float of the smallest area before it.  If it is not (the sides of a
// straight wall give areas that agree in float), the last candidate below the
// float of the smallest area before it is found from prefix minima over the
// walk, NT elements at a time; that case took the walk by one lane before
// (eight 128x2048 frames with facades 112 -> 27 us, 32 of 64x2048 68 -> 43).
constexpr int kWalkSerial = -2;

template <int NT>
__device__ int choose_candidate(const double2* V, const double* area, int n, int cap, int tid, uint16_t* J,
                                uint32_t* par, CandMin* red, double& smallest) {
    auto advances = [&](int i, int j) {
        const double2 a = V[i], b = V[wrap(i + 1, n)];
        return tri_area(a, b, V[wrap(j + 1, n)]) > tri_area(a, b, V[wrap(j, n)]);
    };
    for (int i = tid; i < n; i += NT) {
        int lo = i + 1, hi = i + n - 1;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (advances(i, mid))
                lo = mid + 1;
            else
                hi = mid;
        }
        J[i] = static_cast<uint16_t>(lo);
    }
    for (int q = tid; q <= n >> 5; q += NT) par[q] = 0;
    group_sync<NT>();
    const int j0 = J[0];  // 1 .. n - 1
    const bool early = J[j0 - 1] < n - 1 && J[j0] >= n - 1;
    const int jl = early ? n - 1 : J[j0];
    bool bad = false;
    for (int i = 1 + tid; i <= j0; i += NT) bad |= J[i] < J[i - 1];
    if (group_any<NT>(bad)) return kWalkSerial;
    if (tid == 0) J[j0] = static_cast<uint16_t>(jl);
    group_sync<NT>();
    const int elements = jl + j0;
    auto row_of = [&](int t) {
        int lo = 0, hi = j0;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (J[mid] - 1 + mid >= t)
                hi = mid;
            else
                lo = mid + 1;
        }
        return lo;
    };
    for (int t = tid; t < elements; t += NT) {
        const int i = row_of(t), j = t - i + 1;
        const bool end = j == J[i];
        const bool last = end && early && i == j0;
        bad |= !last && advances(i, j) == end;
        if (end && !last && i > 0) {
            const double2 vi1 = V[wrap(i + 1, n)];
            const double2 vj = V[wrap(j, n)];
            if (tri_area(vj, vi1, V[wrap(j + 1, n)]) == tri_area(V[i], vi1, vj))
                atomicOr(&par[i >> 5], 1u << (i & 31));
        }
    }
    if (group_any<NT>(bad)) return kWalkSerial;
    int pairs = elements - j0 - (early ? 1 : 0);  // row 0 has j0 elements and no pairs
    for (int q = 0; q <= j0 >> 5; ++q) pairs += __popc(par[q]);
    if (pairs > cap) return kWalkSerial;
    // Candidates of the walk's pairs: visit(position, vertex, offset bit).
    auto candidates_at = [&](int t, auto visit) {
        const int i = row_of(t), j = t - i + 1;
        if (early && i == j0 && j == n - 1) return;
        int before = t - j0;
        for (int q = 0; q < i >> 5; ++q) before += __popc(par[q]);
        before += __popc(par[i >> 5] & ((1u << (i & 31)) - 1u));
        const bool twin = j == J[i] && ((par[i >> 5] >> (i & 31)) & 1u);
        const bool wrapped = i == j0 && j == n - 1;
        for (int p = 0; p <= (twin ? 1 : 0); ++p) {
            const int a = p && wrapped ? wrap(i + 1, n) : i;
            const int b = wrap(p && !wrapped ? j + 1 : j, n);
            visit(4 * (before + p) + 0, a, 0);
            visit(4 * (before + p) + 1, a, 1);
            visit(4 * (before + p) + 2, b, 0);
            visit(4 * (before + p) + 3, b, 1);
        }
    };
    auto candidates = [&](auto visit) {
        for (int t = j0 + tid; t < elements; t += NT) candidates_at(t, visit);
    };
    auto area_of = [&](int v, int up) { return area[up ? v : (v == 0 ? n - 1 : v - 1)]; };
    // Candidate of the smallest area, the first of equal ones.
    CandMin m{__builtin_inf(), 0x7fffffff, -1};
    candidates([&](int pos, int v, int up) { cand_min(m, area_of(v, up), pos, 2 * v + up); });
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1)
        cand_min(m, __shfl_xor(m.area, o, kWave), __shfl_xor(m.pos, o, kWave), __shfl_xor(m.cand, o, kWave));
    if (NT > kWave) {
        if (lane_id() == 0) red[tid / kWave] = m;
        __syncthreads();
        for (int q = 0; q < NT / kWave; ++q) cand_min(m, red[q].area, red[q].pos, red[q].cand);
        __syncthreads();
    }
    smallest = m.area;
    if (!(m.area < __builtin_inf())) return -1;
    // The last later candidate below float(m), and the smallest area before.
    const double fm = static_cast<double>(static_cast<float>(m.area));
    CandMin later{__builtin_inf(), -1, -1};
    double before = __builtin_inf();
    candidates([&](int pos, int v, int up) {
        const double a = area_of(v, up);
        if (pos > m.pos && a < fm && pos > later.pos) {
            later.pos = pos;
            later.cand = 2 * v + up;
        }
        if (pos < m.pos) before = fmin(before, a);
    });
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        const int p = __shfl_xor(later.pos, o, kWave), c = __shfl_xor(later.cand, o, kWave);
        if (p > later.pos) {
            later.pos = p;
            later.cand = c;
        }
        before = fmin(before, __shfl_xor(before, o, kWave));
    }
    later.area = before;
    if (NT > kWave) {
        if (lane_id() == 0) red[tid / kWave] = later;
        __syncthreads();
        for (int q = 0; q < NT / kWave; ++q) {
            if (red[q].pos > later.pos) later = CandMin{later.area, red[q].pos, red[q].cand};
            later.area = fmin(later.area, red[q].area);
        }
        __syncthreads();
    }
    if (later.pos >= 0) return later.cand;
    if (m.area < static_cast<double>(static_cast<float>(later.area))) return m.cand;
    double carry = __builtin_inf();  // smallest area of the elements before these NT
    CandMin last{0.0, -1, -1};
    for (int t0 = j0; t0 < elements; t0 += NT) {
        const int t = t0 + tid;
        double mine = __builtin_inf();
        if (t < elements) candidates_at(t, [&](int, int v, int up) { mine = fmin(mine, area_of(v, up)); });
        double incl = mine;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const double x = __shfl_up(incl, o, kWave);
            if (lane_id() >= o) incl = fmin(incl, x);
        }
        double run = __shfl_up(incl, 1, kWave);
        run = fmin(lane_id() > 0 ? run : __builtin_inf(), carry);
        double total = __shfl(incl, kWave - 1, kWave);
        if (NT > kWave) {
            if (lane_id() == 0) red[tid / kWave].area = total;
            __syncthreads();
            for (int q = 0; q < NT / kWave; ++q) {
                if (q < tid / kWave) run = fmin(run, red[q].area);
                total = fmin(total, red[q].area);
            }
            __syncthreads();
        }
        carry = fmin(carry, total);
        if (t < elements)
            candidates_at(t, [&](int pos, int v, int up) {
                const double a = area_of(v, up);
                if (a < static_cast<double>(static_cast<float>(run))) {
                    last.pos = pos;
                    last.cand = 2 * v + up;
                }
                run = fmin(run, a);
            });
    }
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        const int p = __shfl_xor(last.pos, o, kWave), c = __shfl_xor(last.cand, o, kWave);
        if (p > last.pos) {
            last.pos = p;
            last.cand = c;
        }
    }
    if (NT > kWave) {
        if (lane_id() == 0) red[tid / kWave] = last;
        __syncthreads();
        for (int q = 0; q < NT / kWave; ++q)
            if (red[q].pos > last.pos) last = red[q];
        __syncthreads();
    }
    return last.cand;
}

// The same by one lane: the reference's walk and its sequential rule.  False
// when the walk does not end.
__device__ bool choose_serial(const double2* V, const double* area, int n, int cap, int& cand, float& best) {
    best = __builtin_inff();  // float(DBL_MAX)
    cand = -1;
    return antipodal_walk(V, n, cap, [&](int i, int j) {
        for (int q = 0; q < 4; ++q) {
            const int v = q < 2 ? i : j;
            const double a = area[(q & 1) ? v : (v == 0 ? n - 1 : v - 1)];
            if (a < static_cast<double>(best)) {
                best = static_cast<float>(a);
                cand = 2 * v + (q & 1);
            }
        }
    });
}

// Box of the chosen candidate in its own direction, by one whole wavefront
// (every lane returns the same box).
__device__ void candidate_box(const double2* V, int n, int cand, double cx, double cy, lp_bounding_box& box) {
    const int lane = lane_id();
    double ux = 0.0, uy = 0.0;
    cand_dir(V, n, cand >> 1, (cand & 1) ? 1 : -1, ux, uy);
    // Lanes take every 64th vertex; the reduction keeps, among equal values,
    // the one of the lowest vertex index, which is what the sequential
    // std::min / std::max keep (equal values differ at most in the sign of a
    // zero).
    Extent ex = extent_init();
    int qa = n, qb = n, qc = n, qd = n;
    for (int q = lane; q < n; q += kWave) {
        const double tx = V[q].x - cx;
        const double ty = V[q].y - cy;
        const double rx = tx * ux + ty * uy, ry = -tx * uy + ty * ux;
        if (rx < ex.mnx) { ex.mnx = rx; qa = q; }
        if (ex.mxx < rx) { ex.mxx = rx; qb = q; }
        if (ry < ex.mny) { ex.mny = ry; qc = q; }
        if (ex.mxy < ry) { ex.mxy = ry; qd = q; }
    }
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        const double a0 = __shfl_xor(ex.mnx, o, kWave), a1 = __shfl_xor(ex.mxx, o, kWave);
        const double a2 = __shfl_xor(ex.mny, o, kWave), a3 = __shfl_xor(ex.mxy, o, kWave);
        const int b0 = __shfl_xor(qa, o, kWave), b1 = __shfl_xor(qb, o, kWave);
        const int b2 = __shfl_xor(qc, o, kWave), b3 = __shfl_xor(qd, o, kWave);
        if (a0 < ex.mnx || (a0 == ex.mnx && b0 < qa)) { ex.mnx = a0; qa = b0; }
        if (ex.mxx < a1 || (a1 == ex.mxx && b1 < qb)) { ex.mxx = a1; qb = b1; }
        if (a2 < ex.mny || (a2 == ex.mny && b2 < qc)) { ex.mny = a2; qc = b2; }
        if (ex.mxy < a3 || (a3 == ex.mxy && b3 < qd)) { ex.mxy = a3; qd = b3; }
    }
    box.corners[0] = ex.mnx * ux - ex.mny * uy + cx;
    box.corners[1] = ex.mnx * uy + ex.mny * ux + cy;
    box.corners[2] = ex.mxx * ux - ex.mny * uy + cx;
    box.corners[3] = ex.mxx * uy + ex.mny * ux + cy;
    box.corners[4] = ex.mxx * ux - ex.mxy * uy + cx;
    box.corners[5] = ex.mxx * uy + ex.mxy * ux + cy;
    box.corners[6] = ex.mnx * ux - ex.mxy * uy + cx;
    box.corners[7] = ex.mnx * uy + ex.mxy * ux + cy;
    box.angle_rad = atan2_approx(static_cast<float>(uy), static_cast<float>(ux));
    box.is_valid = 1;
}

__device__ __forceinline__ lp_bounding_box empty_box() {
    lp_bounding_box box;
    for (int q = 0; q < 8; ++q) box.corners[q] = 0.0;
    box.area = 0.0f;
    box.angle_rad = 0.0f;
    box.is_valid = 0;
    box.reserved = 0;
    return box;
}

// LDS of one polygon of up to N vertices worked on by W wavefronts.
template <int N, int W>
struct BoxLds {
    double2 V[N];
    double area[N];  // per edge e (e -> e+1); NaN when too short
    uint16_t J[N];
    uint32_t par[N / 32 + 1];
    CandMin red[W];
    int cand;
    float best;
    int ok;
};

// Box of polygon k of frame f, vertices VX/VY[v0 .. v0 + n), 3 <= n <= N, by
// the group's NT threads.
template <int NT, int N>
__device__ __forceinline__ void polygon_box(const DevBuf& d, const Layout& L, int f, int k, const double* VX,
                                            const double* VY, int n, int tid, BoxLds<N, NT / kWave>& s) {
    for (int q = tid; q < n; q += NT) s.V[q] = make_double2(VX[q], VY[q]);
    group_sync<NT>();
    // Centroid: the vertices summed in order, as the reference does.
    double cx = 0.0, cy = 0.0;
#pragma unroll 4
    for (int q = 0; q < n; ++q) {
        cx += s.V[q].x;
        cy += s.V[q].y;
    }
    cx /= n;
    cy /= n;
    for (int e = tid; e < n; e += NT) s.area[e] = edge_box_area(s.V, n, e, cx, cy);
    group_sync<NT>();
    double smallest = 0.0;
    int cand = choose_candidate<NT>(s.V, s.area, n, 2 * N, tid, s.J, s.par, s.red, smallest);
    float best = static_cast<float>(smallest);
    bool ok = true;
    if (cand == kWalkSerial) {
        if (tid == 0) s.ok = choose_serial(s.V, s.area, n, 2 * N, s.cand, s.best) ? 1 : 0;
        group_sync<NT>();
        cand = s.cand;
        best = s.best;
        ok = s.ok != 0;
    }
    if (!ok && tid == 0) atomicOr(&d.fs[f * kFsCount + kFsErr], kErrBoxCapacity);
    if (tid < kWave) {
        lp_bounding_box box = empty_box();
        if (ok && cand >= 0) {
            box.area = best;
            candidate_box(s.V, n, cand, cx, cy, box);
        }
        if (tid == 0) {
            d.boxes[(size_t)f * L.box_stride + k] = box;
            if (box.is_valid) atomicAdd(&d.fs[f * kFsCount + kFsBoxes], 1u);
        }
    }
    group_sync<NT>();
}

// One launch for all polygons.  Polygon k of frame f: vertices
// VX/VY[ob + off[k] .. off[k+1]) with the offsets' end given by `total`.  The
// first `large_tiles` workgroups of a frame take its polygons of more than 64
// vertices (up to kBoxVerts; larger: capacity error): each lists them all
// from the offsets, in order, and takes every large_tiles-th, so the few long
// polygons start at once and run beside the small ones.  The other workgroups
// take the small polygons, a wavefront each, in a grid-stride loop.
constexpr int kBoxWaves = kBoxThreads / kWave;

__global__ __launch_bounds__(kBoxThreads) void k_boxes(DevBuf d, Layout L, const double* VX, const double* VY,
                                                       const uint32_t* off, int large_tiles) {
    union Lds {
        BoxLds<kBoxVerts, kBoxWaves> large;
        BoxLds<kWave, 1> small[kBoxWaves];
        __device__ Lds() {}
    };
    __shared__ Lds lds;
    __shared__ int row_cnt[kBoxWaves];
    int tile, f;
    xcd_tile_frame(tile, f);
    const int tid = threadIdx.x;
    const int w = tid / kWave;
    const int lane = lane_id();
    const uint32_t* fs = d.fs + f * kFsCount;
    const int K = static_cast<int>(fs[kFsClusters]);
    const uint32_t total = fs[kFsHullTotal];
    const size_t ob = (size_t)f * L.N;
    if (K > L.box_stride) {
        if (tile == 0 && tid == 0) atomicOr(&d.fs[f * kFsCount + kFsErr], kErrBoxCapacity);
        return;
    }
    auto range = [&](int k, uint32_t& v0) {
        v0 = off[ob + k];
        return static_cast<int>((k + 1 < K ? off[ob + k + 1] : total) - v0);
    };
    if (tile >= large_tiles) {
        const int tiles = static_cast<int>(gridDim.x) - large_tiles;
        for (int k = (tile - large_tiles) * kBoxWaves + w; k < K; k += tiles * kBoxWaves) {
            uint32_t v0;
            const int n = range(k, v0);
            if (n > kWave) continue;
            if (n < 3) {
                if (lane == 0) d.boxes[(size_t)f * L.box_stride + k] = empty_box();
                continue;
            }
            polygon_box<kWave, kWave>(d, L, f, k, VX + ob + v0, VY + ob + v0, n, lane, lds.small[w]);
        }
        return;
    }
    int seen = 0;  // large polygons before this row of 256
    for (int k0 = 0; k0 < K; k0 += kBoxThreads) {
        uint32_t v0 = 0;
        const int k = k0 + tid;
        const int n = k < K ? range(k, v0) : 0;
        const uint64_t big = __ballot(n > kWave);
        if (lane == 0) row_cnt[w] = __popcll(big);
        __syncthreads();
        int before = seen;
        for (int q = 0; q < w; ++q) before += row_cnt[q];
        int all = 0;
        for (int q = 0; q < kBoxWaves; ++q) all += row_cnt[q];
        before += static_cast<int>(lanes_below(big));
        // This workgroup's polygons of the row, one after the other: `before`
        // is the polygon's number among the large ones.
        const uint64_t mine = __ballot(n > kWave && before % large_tiles == tile);
        __syncthreads();
        seen += all;
        if (all == 0) continue;
        // Every wavefront goes through every wavefront's polygons.
        for (int q = 0; q < kBoxWaves; ++q) {
            if (w == q && lane == 0) {
                lds.large.par[0] = static_cast<uint32_t>(mine);
                lds.large.par[1] = static_cast<uint32_t>(mine >> 32);
            }
            __syncthreads();
            uint64_t todo = lds.large.par[0] | (static_cast<uint64_t>(lds.large.par[1]) << 32);
            __syncthreads();
            while (todo) {
                const int kk = k0 + q * kWave + __ffsll(static_cast<unsigned long long>(todo)) - 1;
                todo &= todo - 1;
                uint32_t vv;
                const int nn = range(kk, vv);
                if (nn > kBoxVerts) {
                    if (tid == 0) {
                        atomicOr(&d.fs[f * kFsCount + kFsErr], kErrBoxCapacity);
                        d.boxes[(size_t)f * L.box_stride + kk] = empty_box();
                    }
                    continue;
                }
                polygon_box<kBoxThreads, kBoxVerts>(d, L, f, kk, VX + ob + vv, VY + ob + vv, nn, tid, lds.large);
            }
        }
    }
}

// Vehicle size classes of the processor's polygon simplification
// (src/processor/src/processor.hpp:78-192): the five base dimension ranges
// widened by the length / width / height tolerances, their volume and area
// bounds, and the loosest height and volume bounds over all five.
struct VehicleConst {
    double dims[5][6];    // min/max length, width, height
    double bounds[5][4];  // min/max volume, min/max area
    double min_h, max_h, min_vol, max_vol;
};

VehicleConst vehicle_const() {
    static const double base[5][6] = {{4.3, 4.6, 1.6, 1.9, 1.4, 1.5},
                                      {4.6, 5.0, 1.6, 1.9, 1.4, 1.5},
                                      {4.6, 5.2, 1.7, 2.1, 1.7, 1.8},
                                      {5.2, 5.8, 1.9, 2.2, 1.8, 2.0},
                                      {4.9, 5.2, 1.7, 2.1, 1.7, 1.8}};
    const double tol[3] = {0.8, 0.5, 0.5};
    VehicleConst v{};
    v.min_h = 1.7976931348623157e308;
    v.max_h = -1.7976931348623157e308;
    v.min_vol = 1.7976931348623157e308;
    v.max_vol = -1.7976931348623157e308;
    for (int i = 0; i < 5; ++i) {
        for (int k = 0; k < 3; ++k) {
            v.dims[i][2 * k] = base[i][2 * k] - tol[k];
            v.dims[i][2 * k + 1] = base[i][2 * k + 1] + tol[k];
        }
        const double* a = v.dims[i];
        v.bounds[i][0] = a[0] * a[2] * a[4];
        v.bounds[i][1] = a[1] * a[3] * a[5];
        v.bounds[i][2] = a[0] * a[2];
        v.bounds[i][3] = a[1] * a[3];
        if (a[4] < v.min_h) v.min_h = a[4];
        if (a[5] > v.max_h) v.max_h = a[5];
        if (v.bounds[i][0] < v.min_vol) v.min_vol = v.bounds[i][0];
        if (v.bounds[i][1] > v.max_vol) v.max_vol = v.bounds[i][1];
    }
    return v;
}

__device__ __forceinline__ double dist_xy(double ax, double ay, double bx, double by) {
    const double dx = ax - bx;
    const double dy = ay - by;
    return sqrt(dx * dx + dy * dy);
}

// Processor::run's polygon simplification test (processor.cpp:680-757), one
// wavefront per cluster: the cluster's z range over its points, then on the
// first lane the shoelace area of the hull in hull order (polygonArea,
// polygonizer.hpp:185-198), the volume and box tests and the first vehicle
// class whose strict bounds all hold.  The box is the cluster hull's
// rotating-calipers box of the preceding stage.
__global__ __launch_bounds__(256) void k_vehicles(DevBuf d, Layout L, VehicleConst vc) {
    const int f = blockIdx.y;
    const uint32_t* fs = d.fs + f * kFsCount;
    const int K = min(static_cast<int>(fs[kFsClusters]), L.box_stride);
    const size_t ob = (size_t)f * L.N;
    const size_t BN = (size_t)L.B * L.N;
    const int lane = lane_id();
    const int waves = gridDim.x * (blockDim.x / kWave);
    for (int c = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; c < K; c += waves) {
        const uint32_t size = d.cl_size[ob + c];
        const uint32_t base = d.cl_off[ob + c];
        float zlo = 3.402823466e38f, zhi = -3.402823466e38f;
        for (uint32_t j = lane; j < size; j += kWave) {
            const float z = d.oz[ob + d.cl_members[ob + base + j]];
            zlo = z < zlo ? z : zlo;
            zhi = zhi < z ? z : zhi;
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
            const float a = __shfl_xor(zlo, o, kWave), b = __shfl_xor(zhi, o, kWave);
            zlo = a < zlo ? a : zlo;
            zhi = zhi < b ? b : zhi;
        }
        if (lane == 0) {
            int32_t cls = -1;
            const int nv = static_cast<int>(d.hull_count[ob + c]);
            const double height = static_cast<double>(zhi) - static_cast<double>(zlo);
            if (nv >= 3 && size > 150u && height > vc.min_h && height < vc.max_h) {
                const double* X = d.hcx + BN + ob + d.hull_off[ob + c];
                const double* Y = d.hcy + BN + ob + d.hull_off[ob + c];
                double area = 0.0;
                for (int i = 0; i < nv - 1; ++i) area += X[i] * Y[i + 1] - X[i + 1] * Y[i];
                area += X[nv - 1] * Y[0] - X[0] * Y[nv - 1];
                area = fabs(area) * 0.5;
                const double volume = area * height;
                const lp_bounding_box& box = d.boxes[(size_t)f * L.box_stride + c];
                if (volume > vc.min_vol && volume < vc.max_vol && box.is_valid &&
                    area / static_cast<double>(box.area) > 0.4) {
                    const double* q = box.corners;
                    const double e1 = dist_xy(q[0], q[1], q[2], q[3]);
                    const double e2 = dist_xy(q[2], q[3], q[4], q[5]);
                    const double len = e1 < e2 ? e2 : e1;  // std::max
                    const double wid = e2 < e1 ? e2 : e1;  // std::min
                    for (int i = 0; i < 5; ++i) {
                        const double* v = vc.dims[i];
                        const double* b = vc.bounds[i];
                        if (len > v[0] && len < v[1] && wid > v[2] && wid < v[3] && height > v[4] && height < v[5] &&
                            volume > b[0] && volume < b[1] && area > b[2] && area < b[3]) {
                            cls = i;
                            break;
                        }
                    }
                }
            }
            d.vclass[(size_t)f * L.box_stride + c] = cls;
            if (cls >= 0) atomicAdd(&d.fs[f * kFsCount + kFsVehicles], 1u);
        }
    }
}

// One Jacobi rotation (c, s) of the 2x2 SVD sweep: the rotation that
// diagonalises the symmetric 2x2 [[x, y], [y, z]] (Golub & Van Loan's
// symmetric Schur step, with the sign choice t = 1 / (tau +- sqrt(tau^2 + 1))).
__device__ __forceinline__ void jacobi_rot(double x, double y, double z, double& c, double& s) {
    const double deno = 2.0 * fabs(y);
    if (deno < 2.2250738585072014e-308) {
        c = 1.0;
        s = 0.0;
        return;
    }
    const double tau = (x - z) / deno;
    const double w = sqrt(tau * tau + 1.0);
    const double t = tau > 0.0 ? 1.0 / (tau + w) : 1.0 / (tau - w);
    const double sign_t = t > 0.0 ? 1.0 : -1.0;
    const double n = 1.0 / sqrt(t * t + 1.0);
    s = -sign_t * (y / fabs(y)) * fabs(t) * n;
    c = n;
}

// Right singular vectors of the 2x2 covariance by two-sided Jacobi sweeps
// (the real 2x2 step: a rotation making the block symmetric, then the
// symmetric Schur rotation), largest singular value first.  v = [v00 v01;
// v10 v11], columns are the vectors.  False for a non-finite matrix.
__device__ bool svd2_v(const double (&a)[2][2], double (&v)[2][2]) {
    double scale = fmax(fmax(fabs(a[0][0]), fabs(a[0][1])), fmax(fabs(a[1][0]), fabs(a[1][1])));
    if (!isfinite(scale)) return false;
    if (scale == 0.0) scale = 1.0;
    double w[2][2] = {{a[0][0] / scale, a[0][1] / scale}, {a[1][0] / scale, a[1][1] / scale}};
    v[0][0] = 1.0;
    v[0][1] = 0.0;
    v[1][0] = 0.0;
    v[1][1] = 1.0;
    const double precision = 2.0 * 2.220446049250313e-16;
    double max_diag = fmax(fabs(w[0][0]), fabs(w[1][1]));
    // p = 1, q = 0 throughout (the only off-diagonal pair of a 2x2).
    for (int sweep = 0; sweep < 64; ++sweep) {
        const double thr = fmax(2.2250738585072014e-308, precision * max_diag);
        if (!(fabs(w[1][0]) > thr || fabs(w[0][1]) > thr)) break;
        // Block m = [[w11, w10], [w01, w00]] in (p, q) order.
        const double m00 = w[1][1], m01 = w[1][0], m10 = w[0][1], m11 = w[0][0];
        double c1 = 1.0, s1 = 0.0;
        const double tt = m00 + m11, dd = m10 - m01;
        if (!(fabs(dd) < 2.2250738585072014e-308)) {
            const double u = tt / dd;
            const double tmp = sqrt(1.0 + u * u);
            s1 = 1.0 / tmp;
            c1 = u / tmp;
        }
        // m <- rot1 applied on the left (rows 0, 1 of m); the symmetric
        // rotation reads m00, m01 and m11 of the result.
        double n00 = m00, n01 = m01, n11 = m11;
        if (!(c1 == 1.0 && s1 == 0.0)) {
            n00 = c1 * m00 + s1 * m10;
            n01 = c1 * m01 + s1 * m11;
            n11 = -s1 * m01 + c1 * m11;
        }
        double cr, sr;
        jacobi_rot(n00, n01, n11, cr, sr);
        // left = rot1 * right^T, right^T = (cr, -sr).
        const double cl = c1 * cr - s1 * (-sr);
        const double sl = c1 * (-sr) + s1 * cr;
        // w.applyOnTheLeft(p=1, q=0, left): x = row 1, y = row 0.
        if (!(cl == 1.0 && sl == 0.0)) {
            for (int k = 0; k < 2; ++k) {
                const double xi = w[1][k], yi = w[0][k];
                w[1][k] = cl * xi + sl * yi;
                w[0][k] = -sl * xi + cl * yi;
            }
        }
        // w and v .applyOnTheRight(p=1, q=0, right): x = column 1, y = column 0,
        // rotated by right^T = (cr, -sr).
        if (!(cr == 1.0 && -sr == 0.0)) {
            for (int k = 0; k < 2; ++k) {
                const double xi = w[k][1], yi = w[k][0];
                w[k][1] = cr * xi + (-sr) * yi;
                w[k][0] = -(-sr) * xi + cr * yi;
                const double vx = v[k][1], vy = v[k][0];
                v[k][1] = cr * vx + (-sr) * vy;
                v[k][0] = -(-sr) * vx + cr * vy;
            }
        }
        max_diag = fmax(max_diag, fmax(fabs(w[1][1]), fabs(w[0][0])));
    }
    const double sv0 = fabs(w[0][0]) * scale, sv1 = fabs(w[1][1]) * scale;
    if (sv0 != 0.0 || sv1 != 0.0) {
        if (sv1 > sv0) {
            const double t0 = v[0][0], t1 = v[1][0];
            v[0][0] = v[0][1];
            v[1][0] = v[1][1];
            v[0][1] = t0;
            v[1][1] = t1;
        }
    }
    return true;
}

// Polygonizer::boundingBoxPrincipalComponentAnalysis (polygonizer.cpp:280-360),
// one wavefront per list.  Every lane evaluates the mean and the covariance
// in the same sequential order (so all lanes hold identical values with no
// exchange), the lanes share the rotation of the centred points and the
// extents, and lane 0 writes the box.
__global__ __launch_bounds__(256) void k_pca_boxes(DevBuf d, Layout L, const double* VX, const double* VY,
                                                  const uint32_t* off) {
    const uint32_t* fs = d.fs;
    const int K = static_cast<int>(fs[kFsClusters]);
    const uint32_t total = fs[kFsHullTotal];
    const int lane = lane_id();
    const int waves = gridDim.x * (blockDim.x / kWave);
    for (int k = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; k < K; k += waves) {
        const uint32_t beg = off[k];
        const uint32_t end = k + 1 < K ? off[k + 1] : total;
        const int n = static_cast<int>(end - beg);
        const double* X = VX + beg;
        const double* Y = VY + beg;
        lp_bounding_box box{};
        double v[2][2] = {{1.0, 0.0}, {0.0, 1.0}};
        bool ok = n >= 3;
        double mx = 0.0, my = 0.0;
        if (ok) {
            double sx = X[0], sy = Y[0];
            for (int i = 1; i < n; ++i) {
                sx += X[i];
                sy += Y[i];
            }
            mx = sx / static_cast<double>(n);
            my = sy / static_cast<double>(n);
            double c00 = 0.0, c01 = 0.0, c11 = 0.0;
            for (int i = 0; i < n; ++i) {
                const double cx = X[i] - mx, cy = Y[i] - my;
                c00 += cx * cx;
                c01 += cx * cy;
                c11 += cy * cy;
            }
            const double dn = static_cast<double>(static_cast<uint32_t>(n - 1));
            const double a[2][2] = {{c00 / dn, c01 / dn}, {c01 / dn, c11 / dn}};
            ok = svd2_v(a, v);
        }
        if (ok) {
            Extent e = extent_init();
            for (int i = lane; i < n; i += kWave) {
                const double cx = X[i] - mx, cy = Y[i] - my;
                extent_add(e, cx * v[0][0] + cy * v[1][0], cx * v[0][1] + cy * v[1][1]);
            }
#pragma unroll
            for (int o = 32; o >= 1; o >>= 1) {
                const double a0 = __shfl_xor(e.mnx, o, kWave), a1 = __shfl_xor(e.mxx, o, kWave);
                const double a2 = __shfl_xor(e.mny, o, kWave), a3 = __shfl_xor(e.mxy, o, kWave);
                e.mnx = a0 < e.mnx ? a0 : e.mnx;
                e.mxx = e.mxx < a1 ? a1 : e.mxx;
                e.mny = a2 < e.mny ? a2 : e.mny;
                e.mxy = e.mxy < a3 ? a3 : e.mxy;
            }
            const double cxs[4] = {e.mnx, e.mxx, e.mxx, e.mnx};
            const double cys[4] = {e.mny, e.mny, e.mxy, e.mxy};
            for (int j = 0; j < 4; ++j) {
                box.corners[2 * j] = (cxs[j] * v[0][0] + cys[j] * v[0][1]) + mx;
                box.corners[2 * j + 1] = (cxs[j] * v[1][0] + cys[j] * v[1][1]) + my;
            }
            box.area = static_cast<float>((e.mxx - e.mnx) * (e.mxy - e.mny));
            box.angle_rad = static_cast<float>(atan2(v[1][0], v[0][0]));
            box.is_valid = 1;
        }
        if (lane == 0) d.boxes[k] = box;
    }
}

}  // namespace

void launch_vehicles(lp_context* c, int B) {
    stage_mark(c, "vehicles");
    hipLaunchKernelGGL(k_vehicles, dim3(64, B), dim3(256), 0, c->stream, c->d, c->L, vehicle_const());
}

void launch_pca_boxes(lp_context* c, int num_polygons) {
    const size_t BN = (size_t)c->L.B * c->L.N;
    const int blocks = std::max(1, std::min(1024, (num_polygons + 3) / 4));
    hipLaunchKernelGGL(k_pca_boxes, dim3(blocks), dim3(256), 0, c->stream, c->d, c->L, c->d.hcx + BN,
                       c->d.hcy + BN, c->d.hull_off);
}

void launch_boxes(lp_context* c, int B) {
    DevBuf& d = c->d;
    const Layout& L = c->L;
    hipStream_t st = c->stream;
    const size_t BN = (size_t)L.B * L.N;
    stage_mark(c, "boxes");
    // Four small polygons per workgroup, about 128 wavefronts per frame on
    // large batches, more for few frames (standalone polygon lists); ahead of
    // them enough workgroups that each takes at most one of a frame's few
    // large polygons.
    const int small_tiles = std::min(1024, std::max(32, 4096 / B));
    const int large_tiles = std::min(256, std::max(8, 1024 / B));
    hipLaunchKernelGGL(k_boxes, dim3(large_tiles + small_tiles, B), dim3(kBoxThreads), 0, st, d, L, d.hcx + BN,
                       d.hcy + BN, d.hull_off, large_tiles);
}

}  // namespace lp
