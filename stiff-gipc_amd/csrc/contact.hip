// Contact-pair generation and the barrier of every pair type, for gfx950.
//
// Reference: the LBVH self queries of StiffGIPC/mlbvh.cu (leaf boxes and
// Morton keys :1146-1225, radix tree :133-227,1247-1267, refit :1269-1296,
// point-face query :1306-1407, edge-edge query :1509-1632) with the
// distance-type narrow phase and pair encoding of _checkPTintersection /
// _checkEEintersection (:229-533, :535-1060, smooth = false), and the RANK 2 /
// NEWF branches of _calBarrierGradientAndHessian (StiffGIPC/GIPC.cu:3176-4984).
//
// Differences by design:
//   * in place of a radix tree walked by one thread per query, the sorted
//     primitives form clusters of 64 (and tops of 64 clusters) that a whole
//     wave tests at once (scan_wave); the float boxes of the tree only
//     preselect, the FP64 leaf boxes decide which pairs are examined;
//   * the reference appends pairs with atomic counters, so their order (and
//     every MatIndex) changes from run to run; here the pairs found are sorted
//     by (query primitive, found primitive): point-face pairs by (surface
//     slot, face), then edge-edge pairs by (edge, edge).  MatIndex counts each
//     class in that order, so a detection is reproducible bit for bit.
#include <algorithm>
#include <cmath>
#include <limits>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "contact.hpp"
#include "pcg.hpp"
#include "vertex_sums.hpp"
#include "wave_ops.hpp"

namespace sgipc {

namespace {

inline int g256(long n) { return (int)((n + 255) / 256); }

// ------------------------------------------------------------ small vectors
struct V3 {
    double x, y, z;
};
__device__ __forceinline__ V3 ld3(const double* p, long i) { return V3{p[3 * i], p[3 * i + 1], p[3 * i + 2]}; }
__device__ __forceinline__ V3 operator-(V3 a, V3 b) { return V3{a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ double dot(V3 a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ V3 cross(V3 a, V3 b)
{
    return V3{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ double det_cols(V3 c0, V3 c1, V3 c2) { return dot(c0, cross(c1, c2)); }

// squared distances (mlbvh.cu:229-271)
__device__ __forceinline__ double sq_pp(V3 a, V3 b)
{
    const V3 d = a - b;
    return dot(d, d);
}
__device__ __forceinline__ double sq_pe(V3 p, V3 a, V3 b)
{
    const V3 c = cross(a - p, b - p), e = b - a;
    return dot(c, c) / dot(e, e);
}
__device__ __forceinline__ double sq_pt(V3 p, V3 a, V3 b, V3 c)
{
    const V3 nv = cross(b - a, c - a);
    const double s = dot(p - a, nv);
    return s * s / dot(nv, nv);
}
__device__ __forceinline__ double sq_ee(V3 a0, V3 a1, V3 b0, V3 b1)
{
    const V3 nv = cross(a1 - a0, b1 - b0);
    const double s = dot(b0 - a0, nv);
    return s * s / dot(nv, nv);
}

// p in the frame (edge ab, in-plane normal of the edge, triangle normal)
__device__ __forceinline__ void edge_frame(V3 p, V3 a, V3 b, V3 nv, double& s, double& t)
{
    const V3 e = b - a, m = cross(e, nv), w = p - a;
    const double D = det_cols(e, m, nv);
    s = det_cols(w, m, nv) / D;
    t = det_cols(e, w, nv) / D;
}

// closest feature of triangle (t0, t1, t2) to p (mlbvh.cu:288-447)
__device__ int feature_pt(V3 p, V3 t0, V3 t1, V3 t2)
{
    const V3 nv = cross(t1 - t0, t2 - t0);
    double s0, u0, s1, u1, s2, u2;
    edge_frame(p, t0, t1, nv, s0, u0);
    if (s0 > 0.0 && s0 < 1.0 && u0 >= 0.0) return 3;
    edge_frame(p, t1, t2, nv, s1, u1);
    if (s1 > 0.0 && s1 < 1.0 && u1 >= 0.0) return 4;
    edge_frame(p, t2, t0, nv, s2, u2);
    if (s2 > 0.0 && s2 < 1.0 && u2 >= 0.0) return 5;
    if (s0 <= 0.0 && s2 >= 1.0) return 0;
    if (s1 <= 0.0 && s0 >= 1.0) return 1;
    if (s2 <= 0.0 && s1 >= 1.0) return 2;
    return 6;
}

// closest features of segments a0a1, b0b1 (mlbvh.cu:449-533)
__device__ int feature_ee(V3 a0, V3 a1, V3 b0, V3 b1)
{
    const V3 u = a1 - a0, v = b1 - b0, w = a0 - b0;
    const double a = dot(u, u), b = dot(u, v), c = dot(v, v), d = dot(u, w), e = dot(v, w);
    const double D = a * c - b * b;
    double tD = D, tN;
    int res = 8;
    const double sN = b * e - c * d;
    if (sN <= 0.0) {
        tN = e;
        tD = c;
        res = 2;
    } else if (sN >= D) {
        tN = e + b;
        tD = c;
        res = 5;
    } else {
        tN = a * e - b * d;
        const V3 uv = cross(u, v);
        if (tN > 0.0 && tN < tD && (dot(w, uv) == 0.0 || dot(uv, uv) < 1.0e-20 * a * c)) {
            tN = sN < D / 2 ? e : e + b;
            tD = c;
            res = sN < D / 2 ? 2 : 5;
        }
    }
    if (tN <= 0.0) return (-d <= 0.0) ? 0 : ((-d >= a) ? 3 : 6);
    if (tN >= tD) return ((-d + b) <= 0.0) ? 1 : (((-d + b) >= a) ? 4 : 7);
    return res;
}

struct Found {
    int4 pr;
    int cls;  // 2 PP, 3 PE, 4 PT/EE; 0: no contact
};

// _checkPTintersection (mlbvh.cu:535-651)
__device__ Found narrow_pt(const double* __restrict__ x, int p, int t0, int t1, int t2, double dsq)
{
    const V3 P = ld3(x, p), A = ld3(x, t0), B = ld3(x, t1), C = ld3(x, t2);
    Found f{make_int4(0, 0, 0, 0), 0};
    const int m = -p - 1;
    switch (feature_pt(P, A, B, C)) {
    case 0: if (sq_pp(P, A) < dsq) f = Found{make_int4(m, t0, -1, -1), 2}; break;
    case 1: if (sq_pp(P, B) < dsq) f = Found{make_int4(m, t1, -1, -1), 2}; break;
    case 2: if (sq_pp(P, C) < dsq) f = Found{make_int4(m, t2, -1, -1), 2}; break;
    case 3: if (sq_pe(P, A, B) < dsq) f = Found{make_int4(m, t0, t1, -1), 3}; break;
    case 4: if (sq_pe(P, B, C) < dsq) f = Found{make_int4(m, t1, t2, -1), 3}; break;
    case 5: if (sq_pe(P, C, A) < dsq) f = Found{make_int4(m, t2, t0, -1), 3}; break;
    default: if (sq_pt(P, A, B, C) < dsq) f = Found{make_int4(m, t0, t1, t2), 4}; break;
    }
    return f;
}

// _checkEEintersection, smooth = false (mlbvh.cu:685-1060): w of a
// point-point / point-edge pair is -obj - 2 for edges nearly parallel at rest
__device__ Found narrow_ee(const double* __restrict__ x, const double* __restrict__ rest, int a0, int a1, int b0, int b1,
                           int obj, double dsq)
{
    const V3 A0 = ld3(x, a0), A1 = ld3(x, a1), B0 = ld3(x, b0), B1 = ld3(x, b1);
    const int t = feature_ee(A0, A1, B0, B1);
    const V3 c = cross(A0 - A1, B0 - B1);
    const double ex = 1e-3 * sq_pp(ld3(rest, a0), ld3(rest, a1)) * sq_pp(ld3(rest, b0), ld3(rest, b1));
    const int we = dot(c, c) < ex ? -obj - 2 : -1;
    Found f{make_int4(0, 0, 0, 0), 0};
    switch (t) {
    case 0: if (sq_pp(A0, B0) < dsq) f = Found{make_int4(-a0 - 1, b0, -1, we), 2}; break;
    case 1: if (sq_pp(A0, B1) < dsq) f = Found{make_int4(-a0 - 1, b1, -1, we), 2}; break;
    case 2: if (sq_pe(A0, B0, B1) < dsq) f = Found{make_int4(-a0 - 1, b0, b1, we), 3}; break;
    case 3: if (sq_pp(A1, B0) < dsq) f = Found{make_int4(-a1 - 1, b0, -1, we), 2}; break;
    case 4: if (sq_pp(A1, B1) < dsq) f = Found{make_int4(-a1 - 1, b1, -1, we), 2}; break;
    case 5: if (sq_pe(A1, B0, B1) < dsq) f = Found{make_int4(-a1 - 1, b0, b1, we), 3}; break;
    case 6: if (sq_pe(B0, A0, A1) < dsq) f = Found{make_int4(-b0 - 1, a0, a1, we), 3}; break;
    case 7: if (sq_pe(B1, A0, A1) < dsq) f = Found{make_int4(-b1 - 1, a0, a1, we), 3}; break;
    default: if (sq_ee(A0, A1, B0, B1) < dsq) f = Found{make_int4(a0, a1, b0, b1), 4}; break;
    }
    return f;
}

// ------------------------------------------------------------ broad phase
// Boxes of every primitive: faces, then edges, then points (surface
// vertices), FP64; with dir they also cover x - alpha dir (swept boxes of the
// CCD queries, mlbvh.cu:1171-1204).  Each block also leaves the union of its
// boxes (part, 6 per block) for the Morton grid.
__global__ __launch_bounds__(256) void k_boxes(BroadSets bs, const double* __restrict__ x,
                                               const uint32_t* __restrict__ faces, const uint32_t* __restrict__ edges,
                                               const uint32_t* __restrict__ points, const double* __restrict__ dir,
                                               double alpha, double* __restrict__ box, double* __restrict__ part)
{
    __shared__ double sm[6][4];
    double u[6] = {1e32, 1e32, 1e32, -1e32, -1e32, -1e32};
    const int n = bs.total();
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int set = bs.set_of(i);
        const int e = i - bs.start(set), k = 3 - set;  // 3, 2, 1 vertices
        const uint32_t* v = set == 0 ? faces + 3L * e : (set == 1 ? edges + 2L * e : points + e);
        double lo[3] = {1e32, 1e32, 1e32}, hi[3] = {-1e32, -1e32, -1e32};
        for (int a = 0; a < k; ++a) {
            const long w = v[a];
            for (int d = 0; d < 3; ++d) {
                const double c = x[3 * w + d];
                lo[d] = fmin(lo[d], c);
                hi[d] = fmax(hi[d], c);
                if (dir != nullptr) {
                    const double m = c - dir[3 * w + d] * alpha;
                    lo[d] = fmin(lo[d], m);
                    hi[d] = fmax(hi[d], m);
                }
            }
        }
        for (int d = 0; d < 3; ++d) {
            box[6L * i + d] = lo[d];
            box[6L * i + 3 + d] = hi[d];
            u[d] = fmin(u[d], lo[d]);
            u[3 + d] = fmax(u[3 + d], hi[d]);
        }
    }
    for (int d = 0; d < 6; ++d) {
        double v = u[d];
        for (int off = 32; off >= 1; off >>= 1) {
            const double o = __shfl_xor(v, off, 64);
            v = d < 3 ? fmin(v, o) : fmax(v, o);
        }
        if ((threadIdx.x & 63) == 0) sm[d][threadIdx.x >> 6] = v;
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int d = threadIdx.x;
        double v = sm[d][0];
        for (int q = 1; q < 4; ++q) v = d < 3 ? fmin(v, sm[d][q]) : fmax(v, sm[d][q]);
        part[6L * blockIdx.x + d] = v;
    }
}

// 10 bits per axis, interleaved (x highest)
__device__ __forceinline__ uint32_t spread10(uint32_t v)
{
    v &= 0x3FFu;
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

// key = set (2 bits) above the 30-bit Morton code of the box centre, so one
// sort orders the three sets.  The grid's cells are cubes: with cells scaled
// to each axis' extent, thin sheets were split by the height of their
// vertices first, and clusters reached far across them (pair queries of two
// 256^2 sheets: 2.6 and 2.2 ms against 0.28 and 0.33 ms).  They hold 10 bits
// of the largest extent, so a far vertex coarsens the clusters of the rest
// (two 192^2 sheets in random order: 0.92 ms, 24 with a vertex 1 km away; a
// radix tree of per-axis cells 12.9 and 62.9).
__global__ __launch_bounds__(256) void k_morton(BroadSets bs, const double* __restrict__ box,
                                                const double* __restrict__ part, int n_part,
                                                uint32_t* __restrict__ keys, int* __restrict__ idx)
{
    __shared__ double sm[6][4], scene[6];
    for (int d = 0; d < 6; ++d) {
        double v = d < 3 ? 1e32 : -1e32;
        for (int q = threadIdx.x; q < n_part; q += blockDim.x)
            v = d < 3 ? fmin(v, part[6L * q + d]) : fmax(v, part[6L * q + d]);
        for (int off = 32; off >= 1; off >>= 1) {
            const double o = __shfl_xor(v, off, 64);
            v = d < 3 ? fmin(v, o) : fmax(v, o);
        }
        if ((threadIdx.x & 63) == 0) sm[d][threadIdx.x >> 6] = v;
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int d = threadIdx.x;
        double v = sm[d][0];
        for (int q = 1; q < 4; ++q) v = d < 3 ? fmin(v, sm[d][q]) : fmax(v, sm[d][q]);
        scene[d] = v;
    }
    __syncthreads();
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= bs.total()) return;
    uint32_t q[3];
    const double ext = fmax(scene[3] - scene[0], fmax(scene[4] - scene[1], scene[5] - scene[2]));
    for (int d = 0; d < 3; ++d) {
        const double c = 0.5 * (box[6L * i + d] + box[6L * i + 3 + d]) - scene[d];
        double u = ext > 0.0 ? c / ext * 1024.0 : 0.0;
        u = fmin(fmax(u, 0.0), 1023.0);
        q[d] = (uint32_t)u;
    }
    const int set = bs.set_of(i);
    keys[i] = ((uint32_t)set << 30) | (spread10(q[0]) << 2) | (spread10(q[1]) << 1) | spread10(q[2]);
    idx[i] = i - bs.start(set);
}

// FP64 bound widened to a float at least one float step outside it: the tree
// tests then never drop a pair the FP64 box test keeps
__device__ __forceinline__ float below(double v)
{
    return nextafterf(__double2float_rd(v), -INFINITY);
}
__device__ __forceinline__ float above(double v)
{
    return nextafterf(__double2float_ru(v), INFINITY);
}

// Float leaf boxes in sorted order (6 arrays of bs.slots entries, every set
// padded to whole clusters of 64 with boxes that overlap nothing) and the
// union of each cluster; one wave per cluster.
__global__ __launch_bounds__(256) void k_clusters(BroadSets bs, const double* __restrict__ box,
                                                  const int* __restrict__ sidx, float* __restrict__ leaf,
                                                  float* __restrict__ l1)
{
    const int c = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (c >= bs.slots / 64) return;
    const int set = bs.set_of_slot(64 * c);
    const int p = 64 * c + lane - bs.slot0[set];  // sorted position inside the set
    float b[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    if (p < bs.n[set]) {
        const long i = bs.start(set) + sidx[bs.start(set) + p];
        for (int d = 0; d < 3; ++d) {
            b[d] = below(box[6 * i + d]);
            b[3 + d] = above(box[6 * i + 3 + d]);
        }
    }
    for (int d = 0; d < 6; ++d) {
        leaf[(long)d * bs.slots + 64 * c + lane] = b[d];
        float v = b[d];
        for (int off = 32; off >= 1; off >>= 1) {
            const float o = __shfl_xor(v, off, 64);
            v = d < 3 ? fminf(v, o) : fmaxf(v, o);
        }
        if (lane == 0) l1[(long)d * (bs.slots / 64) + c] = v;
    }
}

// Union of 64 clusters (of one set) each: the top level, scanned linearly.
__global__ __launch_bounds__(256) void k_tops(BroadSets bs, const float* __restrict__ l1, float* __restrict__ l2)
{
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (t >= bs.tops) return;
    const int set = t >= bs.top0[2] ? 2 : (t >= bs.top0[1] ? 1 : 0);
    const int c = bs.slot0[set] / 64 + 64 * (t - bs.top0[set]) + lane;
    const bool in = c < bs.slot_end(set) / 64;
    for (int d = 0; d < 6; ++d) {
        float v = in ? l1[(long)d * (bs.slots / 64) + c] : (d < 3 ? INFINITY : -INFINITY);
        for (int off = 32; off >= 1; off >>= 1) {
            const float o = __shfl_xor(v, off, 64);
            v = d < 3 ? fminf(v, o) : fmaxf(v, o);
        }
        if (lane == 0) l2[(long)d * bs.tops + t] = v;
    }
}

// the FP64 box test that decides which pairs reach the narrow phase
__device__ __forceinline__ bool boxes_overlap(const double* q, const double* __restrict__ b, double gap)
{
#pragma unroll
    for (int d = 0; d < 3; ++d)
        if ((b[d] - q[3 + d]) >= gap || (q[d] - b[3 + d]) >= gap) return false;
    return true;
}

// Box queries of 16 consecutive sorted queries per wave against the clusters
// of a target set.  What bounds a tree walk per thread here is divergence and
// its stack; a wave instead tests 64 boxes at a time: tops, the 64 clusters
// of a hit top, the 64 leaves of a hit cluster against the union of its
// queries, and then the leaves that remain, 4 per step, against the 16 single
// queries.  Pairs that overlap go to a queue in LDS; whenever it holds 64,
// visit(query position, target position) runs on all lanes at once (inactive
// lanes get -1).  kSelf: queries and targets are one set and each pair comes
// once, with the target at the higher sorted position.
// Two 256^2 sheets (390k edges, 131k points, 260k faces, 1.77 M pairs): 0.33
// ms for the edges and 0.28 ms for the faces, and 0.2 ms for the sorted
// clusters.  The depth-first FP64 walk it replaced took 4.3 and 1.3 ms, each
// twice (a counting and a writing pass), its radix tree's refit with a device
// fence per node 4.8 ms.
constexpr int kQ = 16;
struct WaveScan {
    float tb[6][64];  // leaves of the cluster under test that overlap the queries' union
    int tp[64];       // their sorted positions
    int2 queue[128];
};
template <bool kSelf, typename F>
__device__ __forceinline__ void scan_wave(WaveScan& w, const BroadSets& bs, int qset, int tset, int q0,
                                          const float* __restrict__ leaf, const float* __restrict__ l1,
                                          const float* __restrict__ l2, float gap, F&& visit)
{
    const int lane = threadIdx.x & 63;
    const int nl1 = bs.slots / 64;
    const int qp = q0 + (lane & (kQ - 1));
    float lo[3], hi[3], ulo[3], uhi[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        // the query set is padded to whole clusters: in range for every lane
        lo[d] = nextafterf(leaf[(long)d * bs.slots + bs.slot0[qset] + qp] - gap, -INFINITY);
        hi[d] = nextafterf(leaf[(long)(3 + d) * bs.slots + bs.slot0[qset] + qp] + gap, INFINITY);
        ulo[d] = lo[d];
        uhi[d] = hi[d];
        for (int off = kQ / 2; off >= 1; off >>= 1) {
            ulo[d] = fminf(ulo[d], __shfl_xor(ulo[d], off, 64));
            uhi[d] = fmaxf(uhi[d], __shfl_xor(uhi[d], off, 64));
        }
    }
    // all six bounds loaded before any is compared (one memory round trip)
    auto load = [](const float* __restrict__ src, long stride, long i, float* b) {
#pragma unroll
        for (int d = 0; d < 6; ++d) b[d] = src[d * stride + i];
    };
    auto hits = [&](const float* b) {
        return (b[0] <= uhi[0]) & (b[3] >= ulo[0]) & (b[1] <= uhi[1]) & (b[4] >= ulo[1]) & (b[2] <= uhi[2]) &
               (b[5] >= ulo[2]);
    };
    float tb[6];
    int qn = 0;  // queue length (wave-uniform)
    const int c0 = bs.slot0[tset] / 64, c1 = bs.slot_end(tset) / 64;
    const int nt = bs.n_tops(tset);
    for (int t0 = 0; t0 < nt; t0 += 64) {
        const int t = t0 + lane;
        load(l2, bs.tops, bs.top0[tset] + min(t, nt - 1), tb);
        // kSelf: tops, clusters and leaves that end at or before the first query hold no partner
        bool h = (t < nt) & !(kSelf && 4096L * (t + 1) <= q0 + 1) & hits(tb);
        for (uint64_t mt = __ballot(h); mt; mt &= mt - 1) {
            const int cf = 64 * (t0 + __ffsll((unsigned long long)mt) - 1);  // first cluster of the top
            const int c = c0 + cf + lane;
            load(l1, nl1, min(c, c1 - 1), tb);
            h = (c < c1) & !(kSelf && 64L * (cf + lane + 1) <= q0 + 1) & hits(tb);
            for (uint64_t mc = __ballot(h); mc; mc &= mc - 1) {
                const int base = 64 * (cf + __ffsll((unsigned long long)mc) - 1);  // first leaf position
                load(leaf, bs.slots, (long)bs.slot0[tset] + base + lane, tb);
                h = (base + lane < bs.n[tset]) & !(kSelf && base + lane <= q0) & hits(tb);
                const uint64_t ml = __ballot(h);
                if (!ml) continue;
                const int at = __popcll(ml & ((1ull << lane) - 1ull));
                if (h) {
#pragma unroll
                    for (int d = 0; d < 6; ++d) w.tb[d][at] = tb[d];
                    w.tp[at] = base + lane;
                }
                const int m = __popcll(ml);
                wave_lds_sync();
                for (int k0 = 0; k0 < m; k0 += 64 / kQ) {
                    const int k = min(k0 + lane / kQ, 63);
                    const int tp = w.tp[k];
                    const bool ok = (k < m) & (w.tb[0][k] <= hi[0]) & (w.tb[3][k] >= lo[0]) & (w.tb[1][k] <= hi[1]) &
                                    (w.tb[4][k] >= lo[1]) & (w.tb[2][k] <= hi[2]) & (w.tb[5][k] >= lo[2]) &
                                    !(kSelf && tp <= qp) & (k0 + lane / kQ < m);
                    const uint64_t mo = __ballot(ok);
                    if (!mo) continue;
                    if (ok) w.queue[qn + __popcll(mo & ((1ull << lane) - 1ull))] = make_int2(qp, tp);
                    qn += __popcll(mo);
                    wave_lds_sync();
                    if (qn >= 64) {
                        const int2 e = w.queue[lane];
                        const int2 rest = w.queue[64 + lane];
                        wave_lds_sync();
                        w.queue[lane] = rest;
                        qn -= 64;
                        wave_lds_sync();
                        visit(e.x, e.y);
                    }
                }
                wave_lds_sync();
            }
        }
    }
    if (qn > 0) {
        const int2 e = w.queue[lane];
        const bool in = lane < qn;
        visit(in ? e.x : -1, in ? e.y : -1);
    }
}

__device__ __forceinline__ bool all_fixed(const int* __restrict__ bt, int a, int b, int c, int d)
{
    return bt != nullptr && bt[a] >= 2 && bt[b] >= 2 && bt[c] >= 2 && bt[d] >= 2;
}

// Pairs found by a workgroup, gathered in LDS so that one atomic per
// workgroup reserves their place in the output; pairs past the LDS buffer are
// written at a place their wave reserves.
constexpr int kOut = 512;
struct PairOut {
    uint64_t key[kOut];
    int4 pair[kOut];
    int n, base;
};
__device__ __forceinline__ void put_pair(uint64_t* __restrict__ rkey, int4* __restrict__ rpair, int cap, int at,
                                         uint64_t key, int4 pr)
{
    if (at < cap) {
        rkey[at] = key;
        rpair[at] = pr;
    }
}
// every lane of the wave calls it
__device__ __forceinline__ void push_pairs(PairOut& o, bool found, uint64_t key, int4 pr, uint64_t* __restrict__ rkey,
                                           int4* __restrict__ rpair, int cap, int* __restrict__ total)
{
    const uint64_t m = __ballot(found);
    if (!m) return;
    const int lane = threadIdx.x & 63;
    const uint64_t before = (1ull << lane) - 1ull;
    int at = 0;
    if (lane == 0) at = atomicAdd(&o.n, __popcll(m));
    at = __shfl(at, 0, 64) + __popcll(m & before);
    const bool in = found && at < kOut;
    if (in) {
        o.key[at] = key;
        o.pair[at] = pr;
    }
    const bool over = found && !in;
    const uint64_t mo = __ballot(over);
    if (!mo) return;
    int g = 0;
    if (lane == 0) g = atomicAdd(total, __popcll(mo));
    g = __shfl(g, 0, 64) + __popcll(mo & before);
    if (over) put_pair(rkey, rpair, cap, g, key, pr);
}
__device__ __forceinline__ void flush_pairs(PairOut& o, uint64_t* __restrict__ rkey, int4* __restrict__ rpair, int cap,
                                            int* __restrict__ total)
{
    __syncthreads();
    const int n = min(o.n, kOut);
    if (threadIdx.x == 0 && n > 0) o.base = atomicAdd(total, n);
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += blockDim.x) put_pair(rkey, rpair, cap, o.base + i, o.key[i], o.pair[i]);
}

// point-face pairs (mlbvh.cu:1306-1407) and edge-edge pairs (:1509-1632, each
// pair once), with their sort keys (query, found; edge-edge pairs above all
// point-face pairs); total counts every pair, also past cap
__global__ __launch_bounds__(256) void k_pairs_vf(BroadSets bs, const float* __restrict__ leaf,
                                                  const float* __restrict__ l1, const float* __restrict__ l2,
                                                  const int* __restrict__ sidx, const double* __restrict__ box,
                                                  const double* __restrict__ x, const uint32_t* __restrict__ faces,
                                                  const uint32_t* __restrict__ surf, const int* __restrict__ body,
                                                  const int* __restrict__ bt, double dsq, float gapf, int fbits,
                                                  uint64_t* __restrict__ rkey, int4* __restrict__ rpair, int cap,
                                                  int* __restrict__ total)
{
    __shared__ WaveScan ws[4];
    __shared__ PairOut out;
    if (threadIdx.x == 0) out.n = 0;
    __syncthreads();
    const int q0 = kQ * (blockIdx.x * 4 + (threadIdx.x >> 6));
    const double gap = sqrt(dsq);
    if (q0 < bs.n[2])
        scan_wave<false>(ws[threadIdx.x >> 6], bs, 2, 0, q0, leaf, l1, l2, gapf, [&](int qp, int tp) {
            Found fd{make_int4(0, 0, 0, 0), 0};
            int q = 0, f = 0;
            if (qp >= 0 && qp < bs.n[2]) {
                q = sidx[bs.start(2) + qp];
                f = sidx[tp];
                const int p = (int)surf[q];
                const int t0 = (int)faces[3L * f], t1 = (int)faces[3L * f + 1], t2 = (int)faces[3L * f + 2];
                const V3 P = ld3(x, p);
                const double qb[6] = {P.x, P.y, P.z, P.x, P.y, P.z};
                if (p != t0 && p != t1 && p != t2 && boxes_overlap(qb, box + 6L * f, gap) &&
                    !(body != nullptr && body[p] == body[t0] && body[p] != -1) && !all_fixed(bt, p, t0, t1, t2))
                    fd = narrow_pt(x, p, t0, t1, t2, dsq);
            }
            push_pairs(out, fd.cls != 0, ((uint64_t)(uint32_t)q << fbits) | (uint32_t)f, fd.pr, rkey, rpair, cap,
                       total);
        });
    flush_pairs(out, rkey, rpair, cap, total);
}

__global__ __launch_bounds__(256) void k_pairs_ee(BroadSets bs, const float* __restrict__ leaf,
                                                  const float* __restrict__ l1, const float* __restrict__ l2,
                                                  const int* __restrict__ sidx, const double* __restrict__ box,
                                                  const double* __restrict__ x, const double* __restrict__ rest,
                                                  const uint32_t* __restrict__ edges, const int* __restrict__ body,
                                                  const int* __restrict__ bt, double dsq, float gapf, int ebits,
                                                  int topbit, uint64_t* __restrict__ rkey, int4* __restrict__ rpair,
                                                  int cap, int* __restrict__ total)
{
    __shared__ WaveScan ws[4];
    __shared__ PairOut out;
    if (threadIdx.x == 0) out.n = 0;
    __syncthreads();
    const int q0 = kQ * (blockIdx.x * 4 + (threadIdx.x >> 6));
    const double gap = sqrt(dsq);
    if (q0 < bs.n[1])
        scan_wave<true>(ws[threadIdx.x >> 6], bs, 1, 1, q0, leaf, l1, l2, gapf, [&](int qp, int tp) {
            Found fd{make_int4(0, 0, 0, 0), 0};
            int e = 0, o = 0;
            if (qp >= 0 && qp < bs.n[1]) {
                const int i = sidx[bs.start(1) + qp], j = sidx[bs.start(1) + tp];
                e = min(i, j);
                o = max(i, j);
                const int a0 = (int)edges[2L * e], a1 = (int)edges[2L * e + 1];
                const int b0 = (int)edges[2L * o], b1 = (int)edges[2L * o + 1];
                if (a0 != b0 && a0 != b1 && a1 != b0 && a1 != b1 &&
                    boxes_overlap(box + 6L * (bs.start(1) + e), box + 6L * (bs.start(1) + o), gap) &&
                    !(body != nullptr && body[a0] == body[b0] && body[a0] != -1) && !all_fixed(bt, a0, a1, b0, b1))
                    fd = narrow_ee(x, rest, a0, a1, b0, b1, o, dsq);
            }
            push_pairs(out, fd.cls != 0, (1ull << topbit) | ((uint64_t)(uint32_t)e << ebits) | (uint32_t)o, fd.pr,
                       rkey, rpair, cap, total);
        });
    flush_pairs(out, rkey, rpair, cap, total);
}

__global__ void k_iota(int n, int* __restrict__ a)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = i;
}

// class of an encoded pair: 2 point-point, 3 point-edge, 4 otherwise
__device__ __forceinline__ int pair_class(int4 pr)
{
    return pr.x >= 0 ? 4 : (pr.z < 0 ? 2 : (pr.w < 0 ? 3 : 4));
}

// pairs in sorted order, and what the MatIndex scan counts: point-point pairs
// in the low, point-edge pairs in the high 32 bits (the rest is class 4)
__global__ void k_emit(int n, const int* __restrict__ order, const int4* __restrict__ rpair, int4* __restrict__ pairs,
                       uint64_t* __restrict__ cls)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int4 pr = rpair[order[i]];
    pairs[i] = pr;
    const int c = pair_class(pr);
    cls[i] = c == 2 ? 1ull : (c == 3 ? 1ull << 32 : 0ull);
}

__global__ void k_mat_index(int n, const int4* __restrict__ pairs, const uint64_t* __restrict__ scan,
                            int* __restrict__ mat_index)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int c = pair_class(pairs[i]);
    const int n2 = (int)(uint32_t)scan[i], n3 = (int)(scan[i] >> 32);  // inclusive
    mat_index[i] = c == 2 ? n2 - 1 : (c == 3 ? n3 - 1 : i - n2 - n3);
}

// ------------------------------------------------------------ barrier
__device__ __forceinline__ double barrier_lam0(double I5, double dh, double kappa)
{
    const double L = log(I5);
    return -(4.0 * kappa * dh * dh *
             (4.0 * I5 + L - 3.0 * I5 * I5 * L * L + 6.0 * I5 * L - 2.0 * I5 * I5 + I5 * L * L - 7.0 * I5 * I5 * L - 2.0)) /
           I5;
}

// One thread per pair: the gradient of dist / sqrt(dHat) in closest-point
// form (point-point, point-line foot, point-plane foot with barycentric
// weights, line-line closest points), the reference's squared distance,
// then the rank-1 Hessian lambda0 g g^T and the gradient g s pk.
// The kernel is bound by its stores (80 B per block, 4 to 16 blocks a pair):
// each thread leaves g, lambda0 and the vertices of its pair in LDS and the
// wave then writes pair after pair, lanes over the pair's consecutive values.
// 1.77 M pairs, 1.48 GB: 0.45 ms with the gradient summed per workgroup first (0.88
// ms with an atomic to memory per component; 1.03 ms when every thread wrote its own
// blocks, at a stride of its pair's size between lanes).
struct PairRec {
    double g[13];  // g, lambda0
};
template <int NV>
__device__ __forceinline__ void write_pair_blocks(const double* __restrict__ g, const int* __restrict__ v, long base,
                                                  int hess_offset, double* __restrict__ tvals, int* __restrict__ trows,
                                                  int* __restrict__ tcols)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int e0 = 0; e0 < 9 * NV * NV; e0 += 64) {
        const int e = e0 + lane;
        if (e < 9 * NV * NV) {
            const int blk = e / 9, k = e % 9, ii = blk / NV, jj = blk % NV;
            const double h = g[12] * g[3 * ii + k % 3] * g[3 * jj + k / 3];
            tvals[9 * base + e] = v[ii] <= v[jj] ? h : 0.0;
        }
    }
    if (lane < NV * NV) {
        const int a = v[lane / NV] + hess_offset, b = v[lane % NV] + hess_offset;
        trows[base + lane] = min(a, b);
        tcols[base + lane] = max(a, b);
    }
}

__global__ __launch_bounds__(128) void k_barrier_pairs(int np, const double* __restrict__ x,
                                                       const int4* __restrict__ pairs,
                                                       const int* __restrict__ mat_index, int n4, int n3, double dh,
                                                       double kappa, int hess_offset, double* __restrict__ grad,
                                                       double* __restrict__ tvals, int* __restrict__ trows,
                                                       int* __restrict__ tcols, int* __restrict__ bad)
{
    __shared__ PairRec rec[128];
    __shared__ int vids[128][4];
    __shared__ long bases[128];
    __shared__ int nvs[128];
    __shared__ VertexSums<256> sums;
    if (grad != nullptr) sums.init();
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    const int4 pr = p < np ? pairs[p] : make_int4(0, 0, 0, -1);
    int vid[4] = {0, 0, 0, 0};
    int k = 0;  // 2 .. 5; 0: nothing to write
    if (p >= np) {
    } else if (pr.x >= 0) {
        // a negative w is a smooth-encoded edge-edge pair: not produced by the detection
        if (pr.w < 0) atomicOr(bad, 1);
        else k = 5;
        vid[0] = pr.x; vid[1] = pr.y; vid[2] = pr.z; vid[3] = pr.w;
    } else {
        vid[0] = -pr.x - 1;
        vid[1] = pr.y;
        if (pr.y < 0) {
            atomicOr(bad, 1);
        } else if (pr.z < 0) {
            k = 2;
        } else if (pr.w < 0) {
            vid[2] = pr.z;
            k = 3;
        } else {
            vid[2] = pr.z;
            vid[3] = pr.w;
            k = 4;
        }
    }
    const int nv = k == 5 ? 4 : k;
    nvs[threadIdx.x] = nv;
    if (k > 0) {
        V3 P[4];
#pragma unroll
        for (int a = 0; a < 4; ++a) P[a] = ld3(x, a < nv ? vid[a] : vid[0]);
        V3 r;
        double coef[4] = {0.0, 0.0, 0.0, 0.0};
        double d2;
        if (k == 2) {
            r = P[0] - P[1];
            coef[0] = 1.0;
            coef[1] = -1.0;
            d2 = sq_pp(P[0], P[1]);
        } else if (k == 3) {
            const V3 e = P[2] - P[1], u = P[0] - P[1];
            const double t = dot(u, e) / dot(e, e);
            r = V3{u.x - t * e.x, u.y - t * e.y, u.z - t * e.z};
            coef[0] = 1.0;
            coef[1] = -(1.0 - t);
            coef[2] = -t;
            d2 = sq_pe(P[0], P[1], P[2]);
        } else if (k == 4) {
            const V3 e1 = P[2] - P[1], e2 = P[3] - P[1], w = P[0] - P[1], nrm = cross(e1, e2);
            const double nn = dot(nrm, nrm);
            const double b1 = dot(cross(w, e2), nrm) / nn, b2 = dot(cross(e1, w), nrm) / nn;
            const double s = dot(w, nrm) / nn;
            r = V3{s * nrm.x, s * nrm.y, s * nrm.z};
            coef[0] = 1.0;
            coef[1] = -(1.0 - b1 - b2);
            coef[2] = -b1;
            coef[3] = -b2;
            d2 = sq_pt(P[0], P[1], P[2], P[3]);
        } else {
            const V3 ea = P[1] - P[0], eb = P[3] - P[2], w0 = P[0] - P[2];
            const double a = dot(ea, ea), b = dot(ea, eb), c = dot(eb, eb), dd = dot(ea, w0), e = dot(eb, w0);
            const double D = a * c - b * b;
            const double s = (b * e - c * dd) / D, t = (a * e - b * dd) / D;
            r = V3{w0.x + s * ea.x - t * eb.x, w0.y + s * ea.y - t * eb.y, w0.z + s * ea.z - t * eb.z};
            coef[0] = 1.0 - s;
            coef[1] = s;
            coef[2] = -(1.0 - t);
            coef[3] = -t;
            d2 = sq_ee(P[0], P[1], P[2], P[3]);
        }
        const double sq = sqrt(dh);
        const double rl = sqrt(dot(r, r));
        const double ux = r.x / rl / sq, uy = r.y / rl / sq, uz = r.z / rl / sq;
        double g[12];
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            g[3 * a] = coef[a] * ux;
            g[3 * a + 1] = coef[a] * uy;
            g[3 * a + 2] = coef[a] * uz;
        }
        const double I5 = d2 / dh;
        const double lam0 = barrier_lam0(d2 < 1e-6 * dh ? 1e-6 : I5, dh, kappa);
        if (grad != nullptr) {
            const double L = log(I5);
            const double pk = 2.0 * (2.0 * kappa * dh * dh * L * (I5 - 1.0) * (I5 + I5 * L - 1.0)) / I5;
            const double sc = sqrt(d2) / sq * pk;
#pragma unroll
            for (int a = 0; a < 4; ++a)
                if (a < nv) sums.add(vid[a], g[3 * a] * sc, g[3 * a + 1] * sc, g[3 * a + 2] * sc, grad);
        }
        const int mi = mat_index[p];
        bases[threadIdx.x] = nv == 4 ? 16L * mi : (nv == 3 ? 16L * n4 + 9L * mi : 16L * n4 + 9L * n3 + 4L * mi);
        PairRec& w = rec[threadIdx.x];
#pragma unroll
        for (int a = 0; a < 12; ++a) w.g[a] = g[a];
        w.g[12] = lam0;
#pragma unroll
        for (int a = 0; a < 4; ++a) vids[threadIdx.x][a] = vid[a];
    }
    __syncthreads();
    if (grad != nullptr) sums.flush(grad);
    // each wave writes its own 64 pairs
    const int w0 = threadIdx.x & ~63;
    for (int q = w0; q < w0 + 64; ++q) {
        const int m = nvs[q];
        if (m == 4)
            write_pair_blocks<4>(rec[q].g, vids[q], bases[q], hess_offset, tvals, trows, tcols);
        else if (m == 3)
            write_pair_blocks<3>(rec[q].g, vids[q], bases[q], hess_offset, tvals, trows, tcols);
        else if (m == 2)
            write_pair_blocks<2>(rec[q].g, vids[q], bases[q], hess_offset, tvals, trows, tcols);
    }
}

// ------------------------------------------------------------ feasible step
// distance of the closest features (ACCD.cu:317-371)
__device__ double pt_dist_any(V3 p, V3 a, V3 b, V3 c)
{
    switch (feature_pt(p, a, b, c)) {
    case 0: return sq_pp(p, a);
    case 1: return sq_pp(p, b);
    case 2: return sq_pp(p, c);
    case 3: return sq_pe(p, a, b);
    case 4: return sq_pe(p, b, c);
    case 5: return sq_pe(p, c, a);
    default: return sq_pt(p, a, b, c);
    }
}
__device__ double ee_dist_any(V3 a0, V3 a1, V3 b0, V3 b1)
{
    switch (feature_ee(a0, a1, b0, b1)) {
    case 0: return sq_pp(a0, b0);
    case 1: return sq_pp(a0, b1);
    case 2: return sq_pe(a0, b0, b1);
    case 3: return sq_pp(a1, b0);
    case 4: return sq_pp(a1, b1);
    case 5: return sq_pe(a1, b0, b1);
    case 6: return sq_pe(b0, a0, a1);
    case 7: return sq_pe(b1, a0, a1);
    default: return sq_ee(a0, a1, b0, b1);
    }
}

// Additive CCD (ACCD.cu:373-534): conservative advancement of the four points
// moving by D (centred), with eta = 1 - slackness and zero thickness; the time
// of contact in [0, 1], at most 50000 steps.
__device__ double accd_toc(V3 P[4], V3 D[4], bool ee, double eta)
{
    const V3 mov{-0.25 * (D[0].x + D[1].x + D[2].x + D[3].x), -0.25 * (D[0].y + D[1].y + D[2].y + D[3].y),
                 -0.25 * (D[0].z + D[1].z + D[2].z + D[3].z)};
    for (int a = 0; a < 4; ++a) D[a] = V3{D[a].x + mov.x, D[a].y + mov.y, D[a].z + mov.z};
    const double maxd = ee ? sqrt(fmax(dot(D[0], D[0]), dot(D[1], D[1]))) + sqrt(fmax(dot(D[2], D[2]), dot(D[3], D[3])))
                           : sqrt(dot(D[0], D[0])) +
                                 sqrt(fmax(dot(D[1], D[1]), fmax(dot(D[2], D[2]), dot(D[3], D[3]))));
    if (maxd == 0.0) return 1.0;
    auto dist2 = [&]() {
        if (!ee) return pt_dist_any(P[0], P[1], P[2], P[3]);
        double d2 = ee_dist_any(P[0], P[1], P[2], P[3]);
        if (d2 <= 0.0)
            d2 = fmin(fmin(sq_pp(P[0], P[2]), sq_pp(P[0], P[3])), fmin(sq_pp(P[1], P[2]), sq_pp(P[1], P[3])));
        return d2;
    };
    double d2 = dist2(), dc = sqrt(d2);
    const double gap = eta * d2 / dc;
    double toc = 0.0;
    for (int count = 1;; ++count) {
        if (count > 50000) return toc;
        const double tlb = (1.0 - eta) * d2 / (dc * maxd);
        for (int a = 0; a < 4; ++a) P[a] = V3{P[a].x + D[a].x * tlb, P[a].y + D[a].y * tlb, P[a].z + D[a].z * tlb};
        d2 = dist2();
        dc = sqrt(d2);
        if (toc != 0.0 && d2 / dc < gap) break;
        toc += tlb;
        if (toc > 1.0) return 1.0;
    }
    return toc;
}

// largest 1 / toc and candidate count of the workgroup
__device__ __forceinline__ void ccd_result(double best, int m, double* __restrict__ inv_toc, int* __restrict__ cnt)
{
    __shared__ double sb[4];
    __shared__ int sc[4];
    for (int off = 32; off >= 1; off >>= 1) {
        best = fmax(best, __shfl_xor(best, off, 64));
        m += __shfl_xor(m, off, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        sb[threadIdx.x >> 6] = best;
        sc[threadIdx.x >> 6] = m;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        inv_toc[blockIdx.x] = fmax(fmax(sb[0], sb[1]), fmax(sb[2], sb[3]));
        cnt[blockIdx.x] = sc[0] + sc[1] + sc[2] + sc[3];
    }
}

// point-face candidates of the swept boxes (mlbvh.cu:1408-1508 with
// _checkPTintersection_fullCCD, :653-683)
__global__ __launch_bounds__(256) void k_ccd_vf(BroadSets bs, const float* __restrict__ leaf,
                                                const float* __restrict__ l1, const float* __restrict__ l2,
                                                const int* __restrict__ sidx, const double* __restrict__ box,
                                                const double* __restrict__ x, const double* __restrict__ dir,
                                                double alpha, const uint32_t* __restrict__ faces,
                                                const uint32_t* __restrict__ surf, const int* __restrict__ body,
                                                const int* __restrict__ bt, double dsq, float gapf, double eta,
                                                double* __restrict__ inv_toc, int* __restrict__ cnt)
{
    __shared__ WaveScan ws[4];
    const int q0 = kQ * (blockIdx.x * 4 + (threadIdx.x >> 6));
    const double gap = sqrt(dsq);
    double best = 1.0;
    int m = 0;
    if (q0 < bs.n[2])
        scan_wave<false>(ws[threadIdx.x >> 6], bs, 2, 0, q0, leaf, l1, l2, gapf, [&](int qp, int tp) {
            if (qp < 0 || qp >= bs.n[2]) return;
            const int p = (int)surf[sidx[bs.start(2) + qp]], f = sidx[tp];
            const int t0 = (int)faces[3L * f], t1 = (int)faces[3L * f + 1], t2 = (int)faces[3L * f + 2];
            const V3 P = ld3(x, p), Pd = ld3(dir, p);
            const double qb[6] = {fmin(P.x, P.x - Pd.x * alpha), fmin(P.y, P.y - Pd.y * alpha),
                                  fmin(P.z, P.z - Pd.z * alpha), fmax(P.x, P.x - Pd.x * alpha),
                                  fmax(P.y, P.y - Pd.y * alpha), fmax(P.z, P.z - Pd.z * alpha)};
            if (!boxes_overlap(qb, box + 6L * f, gap)) return;
            if (body != nullptr && body[p] == body[t0] && body[p] != -1) return;
            if (p == t0 || p == t1 || p == t2) return;
            if (all_fixed(bt, p, t0, t1, t2)) return;
            const V3 A = ld3(x, t0), B = ld3(x, t1), C = ld3(x, t2);
            if (feature_pt(P, A, B, C) == 6 && dot(cross(B - A, C - A), P - A) < 0.0) return;
            ++m;
            V3 Q[4] = {P, A, B, C};
            const V3 da = ld3(dir, t0), db = ld3(dir, t1), dc = ld3(dir, t2);
            V3 D[4] = {V3{-Pd.x, -Pd.y, -Pd.z}, V3{-da.x, -da.y, -da.z}, V3{-db.x, -db.y, -db.z},
                       V3{-dc.x, -dc.y, -dc.z}};
            best = fmax(best, 1.0 / accd_toc(Q, D, false, eta));
        });
    ccd_result(best, m, inv_toc, cnt);
}

// edge-edge candidates of the swept boxes (mlbvh.cu:1634-1774)
__global__ __launch_bounds__(256) void k_ccd_ee(BroadSets bs, const float* __restrict__ leaf,
                                                const float* __restrict__ l1, const float* __restrict__ l2,
                                                const int* __restrict__ sidx, const double* __restrict__ box,
                                                const double* __restrict__ x, const double* __restrict__ dir,
                                                const uint32_t* __restrict__ edges, const int* __restrict__ body,
                                                const int* __restrict__ bt, double dsq, float gapf, double eta,
                                                double* __restrict__ inv_toc, int* __restrict__ cnt)
{
    __shared__ WaveScan ws[4];
    const int q0 = kQ * (blockIdx.x * 4 + (threadIdx.x >> 6));
    const double gap = sqrt(dsq);
    double best = 1.0;
    int m = 0;
    if (q0 < bs.n[1])
        scan_wave<true>(ws[threadIdx.x >> 6], bs, 1, 1, q0, leaf, l1, l2, gapf, [&](int qp, int tp) {
            if (qp < 0 || qp >= bs.n[1]) return;
            const int i = sidx[bs.start(1) + qp], j = sidx[bs.start(1) + tp];
            const int e = min(i, j), o = max(i, j);
            const int a0 = (int)edges[2L * e], a1 = (int)edges[2L * e + 1];
            const int b0 = (int)edges[2L * o], b1 = (int)edges[2L * o + 1];
            if (a0 == b0 || a0 == b1 || a1 == b0 || a1 == b1) return;
            if (!boxes_overlap(box + 6L * (bs.start(1) + e), box + 6L * (bs.start(1) + o), gap)) return;
            if (body != nullptr && body[a0] == body[b0] && body[a0] != -1) return;
            if (all_fixed(bt, a0, a1, b0, b1)) return;
            ++m;
            V3 Q[4] = {ld3(x, a0), ld3(x, a1), ld3(x, b0), ld3(x, b1)};
            const int id[4] = {a0, a1, b0, b1};
            V3 D[4];
            for (int a = 0; a < 4; ++a) {
                const V3 dv = ld3(dir, id[a]);
                D[a] = V3{-dv.x, -dv.y, -dv.z};
            }
            best = fmax(best, 1.0 / accd_toc(Q, D, true, eta));
        });
    ccd_result(best, m, inv_toc, cnt);
}

// ground (GIPC.cu:6945-7020): coef / (dist slackness) for vertices moving
// toward the plane
__global__ void k_ground_step(int n, const uint32_t* __restrict__ surf, const double* __restrict__ x,
                              const double* __restrict__ nrm, double offset, const double* __restrict__ dir,
                              double slackness, double* __restrict__ inv_t)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    const V3 nv{nrm[0], nrm[1], nrm[2]};
    const int v = (int)surf[q];
    const double coef = dot(nv, ld3(dir, v));
    double t = 1.0;
    if (coef > 0.0) t = coef / ((dot(nv, ld3(x, v)) - offset) * slackness);
    inv_t[q] = t;
}

// tet injectivity (GIPC.cu:1130-1300,7022-7094): the smallest t > 0 at which
// the tet's volume shrinks to slackness times its current one; the
// reference's quadratic and linear branches below error_rate, the smallest
// positive root of the cubic otherwise (a case the reference leaves undefined)
__global__ void k_injective_step(int n, const uint32_t* __restrict__ tets, const double* __restrict__ x,
                                 const double* __restrict__ dir, double slackness, double error_rate,
                                 double* __restrict__ inv_t)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    int t[4];
    for (int a = 0; a < 4; ++a) t[a] = (int)tets[4L * e + a];
    const V3 x0 = ld3(x, t[0]), d0 = ld3(dir, t[0]);
    V3 A[3], Bm[3];
    for (int c = 0; c < 3; ++c) {
        A[c] = ld3(x, t[c + 1]) - x0;
        const V3 dc = ld3(dir, t[c + 1]);
        Bm[c] = V3{-dc.x + d0.x, -dc.y + d0.y, -dc.z + d0.z};
    }
    const double c0 = det_cols(A[0], A[1], A[2]), c3 = det_cols(Bm[0], Bm[1], Bm[2]);
    const double c1 = det_cols(Bm[0], A[1], A[2]) + det_cols(A[0], Bm[1], A[2]) + det_cols(A[0], A[1], Bm[2]);
    const double c2 = det_cols(A[0], Bm[1], Bm[2]) + det_cols(Bm[0], A[1], Bm[2]) + det_cols(Bm[0], Bm[1], A[2]);
    const double k0 = (1.0 - slackness) * c0;
    double ts = 1.0;
    if (fabs(c3) <= error_rate) {
        if (fabs(c2) <= error_rate) {
            ts = -k0 / c1;
        } else {
            const double disc = c1 * c1 - 4.0 * c2 * k0;
            if (disc > 0) {
                ts = (-c1 - sqrt(disc)) / (2.0 * c2);
                if (ts < 0) ts = (-c1 + sqrt(disc)) / (2.0 * c2);
            }
        }
    } else {
        double best = -1.0, tlo = 0.0, glo = k0;
        for (int s = 1; s <= 256 && best < 0.0; ++s) {
            const double th = 4.0 * s / 256;
            const double gh = ((c3 * th + c2) * th + c1) * th + k0;
            if ((glo > 0) != (gh > 0) || gh == 0.0) {
                double lo = tlo, hi = th;
                for (int it = 0; it < 100; ++it) {
                    const double mm = 0.5 * (lo + hi), gm = ((c3 * mm + c2) * mm + c1) * mm + k0;
                    if ((gm > 0) == (glo > 0)) lo = mm;
                    else hi = mm;
                }
                best = 0.5 * (lo + hi);
            }
            tlo = th;
            glo = gh;
        }
        ts = best > 0.0 ? best : 1.0;
    }
    if (ts <= 0.0) ts = 1.0;
    inv_t[e] = 1.0 / ts;
}

// max of n values and sum of n ints -> out[blockIdx.x], icnt[blockIdx.x]
__global__ __launch_bounds__(256) void k_max_reduce(long n, const double* __restrict__ v, const int* __restrict__ c,
                                                    double* __restrict__ out, int* __restrict__ icnt)
{
    __shared__ double sm[4];
    __shared__ int si[4];
    double m = 1.0;
    int k = 0;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        m = fmax(m, v[i]);
        if (c != nullptr) k += c[i];
    }
    for (int off = 32; off >= 1; off >>= 1) {
        m = fmax(m, __shfl_xor(m, off, 64));
        k += __shfl_xor(k, off, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        sm[threadIdx.x >> 6] = m;
        si[threadIdx.x >> 6] = k;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = sm[0];
        int rk = si[0];
        for (int w = 1; w < (int)(blockDim.x >> 6); ++w) {
            r = fmax(r, sm[w]);
            rk += si[w];
        }
        out[blockIdx.x] = r;
        icnt[blockIdx.x] = rk;
    }
}

}  // namespace

void BroadPhase::build(hipStream_t s, const double* x, const uint32_t* faces, int n_faces, const uint32_t* edges,
                       int n_edges, const uint32_t* points, int n_points, const double* dir, double alpha)
{
    sets = BroadSets{};
    const int cnt[3] = {n_faces, n_edges, n_points};
    long total = 0, slots = 0, tops = 0;
    for (int k = 0; k < 3; ++k) {
        total += cnt[k];
        slots += (cnt[k] + 63L) / 64 * 64;
        tops += (cnt[k] + 4095L) / 4096;
    }
    SGIPC_CHECK(slots < (1L << 31), SGIPC_CAPACITY, "too many surface primitives");
    for (int k = 0, sl = 0, tp = 0; k < 3; ++k) {
        sets.n[k] = cnt[k];
        sets.slot0[k] = sl;
        sets.top0[k] = tp;
        sl += (cnt[k] + 63) / 64 * 64;
        tp += (cnt[k] + 4095) / 4096;
    }
    sets.slots = (int)slots;
    sets.tops = (int)tops;
    const int n = (int)total;
    if (n == 0) return;
    box.reserve(6 * total);
    const int gb = std::min(g256(n), 256);
    part_.reserve(6L * gb);
    keys_.reserve(n);
    skeys_.reserve(n);
    idx_.reserve(n);
    sidx.reserve(n);
    leaf.reserve(6 * slots);
    l1.reserve(6 * (slots / 64));
    l2.reserve(6 * tops);
    k_boxes<<<gb, 256, 0, s>>>(sets, x, faces, edges, points, dir, alpha, box.get(), part_.get());
    SGIPC_LAUNCH_CHECK();
    k_morton<<<g256(n), 256, 0, s>>>(sets, box.get(), part_.get(), gb, keys_.get(), idx_.get());
    SGIPC_LAUNCH_CHECK();
    size_t need = 0;
    SGIPC_HIP(rocprim::radix_sort_pairs(nullptr, need, keys_.get(), skeys_.get(), idx_.get(), sidx.get(), (size_t)n, 0,
                                        32, s));
    temp_.reserve(need);
    SGIPC_HIP(rocprim::radix_sort_pairs(temp_.get(), need, keys_.get(), skeys_.get(), idx_.get(), sidx.get(),
                                        (size_t)n, 0, 32, s));
    k_clusters<<<(sets.slots / 64 + 3) / 4, 256, 0, s>>>(sets, box.get(), sidx.get(), leaf.get(), l1.get());
    SGIPC_LAUNCH_CHECK();
    k_tops<<<(sets.tops + 3) / 4, 256, 0, s>>>(sets, l1.get(), l2.get());
    SGIPC_LAUNCH_CHECK();
}

namespace {
int bits_of(int n)
{
    int b = 1;
    while (b < 31 && (1L << b) < (long)n) ++b;
    return b;
}
// the query boxes' margin: sqrt(dhat_sq), rounded up past what adding it to a
// float bound can round away (the bounds already lie a float step outside)
float gap_above(double dsq)
{
    return std::nextafter((float)std::sqrt(dsq), std::numeric_limits<float>::infinity());
}
int scan_grid(int queries) { return (queries + 4 * kQ - 1) / (4 * kQ); }
}  // namespace

ContactCounts ContactDetector::detect(hipStream_t s, const double* x, const double* rest, int n_verts,
                                      const uint32_t* faces, int n_faces, const uint32_t* edges, int n_edges,
                                      const uint32_t* surf, int n_surf, const int* body_id, const int* btype,
                                      double dhat_sq, int* pairs, int* mat_index, int capacity)
{
    (void)n_verts;
    ContactCounts out;
    last_total = 0;
    const int nq_vf = (n_faces > 0) ? n_surf : 0;
    const int nq_ee = n_edges > 1 ? n_edges : 0;
    if (nq_vf + (long)nq_ee == 0) return out;
    broad_.build(s, x, faces, nq_vf > 0 ? n_faces : 0, edges, nq_ee, surf, nq_vf, nullptr, 0.0);
    const BroadSets& bs = broad_.sets;
    // sort key: found primitive, query above it, the edge-edge flag on top
    const int fbits = bits_of(n_faces), ebits = bits_of(n_edges);
    const int topbit = std::max(bits_of(n_surf) + fbits, 2 * ebits);
    const float gapf = gap_above(dhat_sq);
    total_.reserve(1);
    // the pairs are found in no fixed order into a buffer that is enlarged
    // (and the queries run again) when it was too small
    if (raw_cap_ == 0) raw_cap_ = std::max(1024L, 4L * (nq_vf + (long)nq_ee));
    int total = 0;
    while (true) {
        const int cap = (int)std::min<long>(raw_cap_, std::max(capacity, 1));
        rkey_.reserve(cap);
        rpair_.reserve(cap);
        launch_fill<int>(s, total_.get(), 0, 1);
        if (nq_vf > 0) {
            k_pairs_vf<<<scan_grid(nq_vf), 256, 0, s>>>(bs, broad_.leaf.get(), broad_.l1.get(), broad_.l2.get(),
                                                        broad_.sidx.get(), broad_.box.get(), x, faces, surf, body_id,
                                                        btype, dhat_sq, gapf, fbits, rkey_.get(), rpair_.get(), cap,
                                                        total_.get());
            SGIPC_LAUNCH_CHECK();
        }
        if (nq_ee > 0) {
            k_pairs_ee<<<scan_grid(nq_ee), 256, 0, s>>>(bs, broad_.leaf.get(), broad_.l1.get(), broad_.l2.get(),
                                                        broad_.sidx.get(), broad_.box.get(), x, rest, edges, body_id,
                                                        btype, dhat_sq, gapf, ebits, topbit, rkey_.get(),
                                                        rpair_.get(), cap, total_.get());
            SGIPC_LAUNCH_CHECK();
        }
        SGIPC_HIP(hipMemcpyAsync(&total, total_.get(), sizeof(int), hipMemcpyDeviceToHost, s));
        SGIPC_HIP(hipStreamSynchronize(s));
        if (total <= cap || total > capacity) break;
        raw_cap_ = total + total / 4L;
    }
    out.c[0] = total;
    last_total = total;
    SGIPC_CHECK(total <= capacity, SGIPC_CAPACITY, "contact pairs exceed the output capacity");
    if (total == 0) return out;
    rkey_sorted_.reserve(total);
    rid_.reserve(total);
    rid_sorted_.reserve(total);
    cls_.reserve(total);
    cls_scan_.reserve(total);
    // canonical order: by key
    k_iota<<<g256(total), 256, 0, s>>>(total, rid_.get());
    SGIPC_LAUNCH_CHECK();
    const int end_bit = topbit + (nq_ee > 0 ? 1 : 0);
    size_t need = 0, need2 = 0;
    SGIPC_HIP(rocprim::radix_sort_pairs(nullptr, need, rkey_.get(), rkey_sorted_.get(), rid_.get(), rid_sorted_.get(),
                                        (size_t)total, 0, end_bit, s));
    SGIPC_HIP(rocprim::inclusive_scan(nullptr, need2, cls_.get(), cls_scan_.get(), (size_t)total,
                                      rocprim::plus<uint64_t>(), s));
    temp_.reserve(std::max(need, need2));
    SGIPC_HIP(rocprim::radix_sort_pairs(temp_.get(), need, rkey_.get(), rkey_sorted_.get(), rid_.get(),
                                        rid_sorted_.get(), (size_t)total, 0, end_bit, s));
    k_emit<<<g256(total), 256, 0, s>>>(total, rid_sorted_.get(), rpair_.get(), reinterpret_cast<int4*>(pairs),
                                       cls_.get());
    SGIPC_LAUNCH_CHECK();
    SGIPC_HIP(rocprim::inclusive_scan(temp_.get(), need2, cls_.get(), cls_scan_.get(), (size_t)total,
                                      rocprim::plus<uint64_t>(), s));
    k_mat_index<<<g256(total), 256, 0, s>>>(total, reinterpret_cast<const int4*>(pairs), cls_scan_.get(), mat_index);
    SGIPC_LAUNCH_CHECK();
    uint64_t last = 0;
    SGIPC_HIP(hipMemcpyAsync(&last, cls_scan_.get() + total - 1, sizeof(last), hipMemcpyDeviceToHost, s));
    SGIPC_HIP(hipStreamSynchronize(s));
    out.c[2] = (int)(uint32_t)last;
    out.c[3] = (int)(last >> 32);
    out.c[4] = total - out.c[2] - out.c[3];
    return out;
}

double StepReducer::max_inv(hipStream_t s, const double* v, const int* c, long n, long* total)
{
    const int gb = (int)std::min<long>(256, (n + 255) / 256);
    part_.reserve(gb + 1);
    ipart_.reserve(gb + 1);
    k_max_reduce<<<gb, 256, 0, s>>>(n, v, c, part_.get(), ipart_.get());
    SGIPC_LAUNCH_CHECK();
    k_max_reduce<<<1, 256, 0, s>>>(gb, part_.get(), ipart_.get(), part_.get() + gb, ipart_.get() + gb);
    SGIPC_LAUNCH_CHECK();
    double h = 1.0;
    int hk = 0;
    SGIPC_HIP(hipMemcpyAsync(&h, part_.get() + gb, sizeof(double), hipMemcpyDeviceToHost, s));
    SGIPC_HIP(hipMemcpyAsync(&hk, ipart_.get() + gb, sizeof(int), hipMemcpyDeviceToHost, s));
    SGIPC_HIP(hipStreamSynchronize(s));
    if (total) *total = hk;
    return h;
}

double ContactDetector::ccd_step(hipStream_t s, const double* x, const double* dir, double alpha,
                                 const uint32_t* faces, int n_faces, const uint32_t* edges, int n_edges,
                                 const uint32_t* surf, int n_surf, const int* body_id, const int* btype,
                                 double dhat_sq, double slackness, long* n_candidates)
{
    const double eta = 1.0 - slackness;
    const int nq_vf = n_faces > 0 ? n_surf : 0;
    const int nq_ee = n_edges > 1 ? n_edges : 0;
    double inv = 1.0;
    long cand = 0;
    const int g_vf = scan_grid(nq_vf), g_ee = scan_grid(nq_ee);
    if (g_vf + g_ee > 0) {
        broad_.build(s, x, faces, nq_vf > 0 ? n_faces : 0, edges, nq_ee, surf, nq_vf, dir, alpha);
        const BroadSets& bs = broad_.sets;
        const float gapf = gap_above(dhat_sq);
        vals_.reserve(g_vf + g_ee);
        cnt_.reserve(g_vf + g_ee);
        if (nq_vf > 0) {
            k_ccd_vf<<<g_vf, 256, 0, s>>>(bs, broad_.leaf.get(), broad_.l1.get(), broad_.l2.get(), broad_.sidx.get(),
                                          broad_.box.get(), x, dir, alpha, faces, surf, body_id, btype, dhat_sq, gapf,
                                          eta, vals_.get(), cnt_.get());
            SGIPC_LAUNCH_CHECK();
        }
        if (nq_ee > 0) {
            k_ccd_ee<<<g_ee, 256, 0, s>>>(bs, broad_.leaf.get(), broad_.l1.get(), broad_.l2.get(), broad_.sidx.get(),
                                          broad_.box.get(), x, dir, edges, body_id, btype, dhat_sq, gapf, eta,
                                          vals_.get() + g_vf, cnt_.get() + g_vf);
            SGIPC_LAUNCH_CHECK();
        }
        inv = std::max(inv, red_.max_inv(s, vals_.get(), cnt_.get(), g_vf + g_ee, &cand));
    }
    if (n_candidates) *n_candidates = cand;
    return 1.0 / inv;
}

double ground_step(hipStream_t s, StepReducer& red, DevBuf<double>& vals, const double* x, const uint32_t* surf,
                   int n_surf, const double* normal, double offset, const double* dir, double slackness)
{
    if (n_surf <= 0) return 1.0;
    vals.reserve(n_surf);
    k_ground_step<<<g256(n_surf), 256, 0, s>>>(n_surf, surf, x, normal, offset, dir, slackness, vals.get());
    SGIPC_LAUNCH_CHECK();
    return 1.0 / red.max_inv(s, vals.get(), nullptr, n_surf, nullptr);
}

double injective_step(hipStream_t s, StepReducer& red, DevBuf<double>& vals, const double* x, const uint32_t* tets,
                      int n_tets, const double* dir, double slackness, double error_rate)
{
    if (n_tets <= 0) return 1.0;
    vals.reserve(n_tets);
    k_injective_step<<<g256(n_tets), 256, 0, s>>>(n_tets, tets, x, dir, slackness, error_rate, vals.get());
    SGIPC_LAUNCH_CHECK();
    return 1.0 / red.max_inv(s, vals.get(), nullptr, n_tets, nullptr);
}

void launch_barrier_pairs(hipStream_t s, int n_pairs, const double* x, const int* pairs, const int* mat_index, int n4,
                          int n3, double dhat_sq, double kappa, int hess_offset, double* grad, double* tvals,
                          int* trows, int* tcols, int* bad)
{
    if (n_pairs <= 0) return;
    k_barrier_pairs<<<(n_pairs + 127) / 128, 128, 0, s>>>(n_pairs, x, reinterpret_cast<const int4*>(pairs), mat_index,
                                                          n4, n3, dhat_sq, kappa, hess_offset, grad, tvals, trows,
                                                          tcols, bad);
    SGIPC_LAUNCH_CHECK();
}

}  // namespace sgipc
