// dA/dt of a block of placements at the mesh nodes (solver/coil/dadt.cu:27-104 of the reference
// evaluates the same sum directly): dA/dt(r) = scale sum_j m_j x (r - s_j) / |r - s_j|^3.
//
// Away from the dipoles each component is a harmonic function, smooth on the scale of its distance
// from them, so most of the n x n_dip terms are redundant: n nodes fill a box far from the coil
// much more densely than the field varies there. The nodes' Morton order gives boxes (octants of
// the bounding box) that are contiguous runs of nodes. A cluster of dipoles far from a box (its
// bounding sphere at least eta half-widths from the box's centre) is summed at the box's p^3
// Chebyshev points only; box values go down to the children by polynomial interpolation, and from
// the leaf boxes' points to the nodes. Clusters near a leaf are summed at its nodes directly. Each
// cluster is taken at the coarsest level where it is far.
//
// Orders and distances: 8 points per axis at 3.5 half-widths above the leaves, 6 points at 5.5 in
// the leaves. Against the closed form in FP64 that truncates the field of a 2,400-dipole figure-8
// coil 4 mm off a 92 mm head by 1e-7 of its 2-norm, against 2.5e-6 that the FP32 pair terms of the
// nearest dipoles cost (8e-6 for a coil bent around the head): those are formed as
// |r|^2 + |s|^2 - 2 r.s, as the reference does. The box points' terms use r - s itself.
//
// A coil whose moments differ in direction may be bent around the head until its dipoles all but
// touch nodes. There W x r - P (below) cancels to the last digits, so the runs of 64 nodes within
// kCloseMm of such a coil's clusters, and every node of a mesh without boxes, take all its dipoles in
// the caller's order, one sum per node. Half a millimetre from a dipole that sum itself is off by up to
// 1e-3 of the 2-norm over the nearest 600 nodes (4e-6 to 1e-4 on finer meshes); any other order or form
// gives other last digits, 2.5 % of E in places.
//
// The sum of a placement does not depend on the block it is in: the dipoles are always summed in
// the same 8 slices, each in order, and the slices added in order, whichever waves take them.
#include "dipole.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

namespace cn {

namespace {

constexpr int kSlices = 8;
constexpr int kLeafValues = 3 * kLeafOrder * kLeafOrder * kLeafOrder;
constexpr int kSliceClusters = kClusters / kSlices;
constexpr int kDipoleThreads = kSlices * kWave;

constexpr double kUpperDistance = 3.5;  // admissible distance over the largest half-width
constexpr double kLeafDistance = 5.5;
constexpr double kCloseMm = 10.0;

// The box method is taken from these sizes up; below them the launches of the levels, and boxes that are
// near most clusters, cost more than the pairs they save. Whether it pays depends on the block's width
// too, but a placement's sum must not, so the lines lie where the widths from 1 to 32 balance, later where
// the leaves are one level deeper. Flat coil, us without and with boxes at widths 1, 4, 16 and 32: 400
// dipoles at 125,000 nodes 34 87 284 530 and 57 114 302 547, at 213,000 46 136 454 879 and 66 138 402 732;
// 600 at 125,000 43 117 400 772 and 67 137 377 677; 400 at 412,000 69 236 854 1684 and 117 283 845 1922,
// 600 there 96 343 1255 2471 and 129 319 964 2129; 260 at 966,000 107 380 1251 2489 and 125 385 1026 2194.
// Moments that differ (near chunks take every dipole either way): 600 dipoles at 213,000 nodes 76 205 701
// 1367 and 122 249 739 1278; 1,800 at 125,000 165 370 1239 2413 and 265 470 1338 2239; 964 at 412,000 182
// 636 2218 4275 and 283 598 1807 3652; 400 at 667,000 114 382 1412 2787 and 184 460 1407 2790; 260 at
// 966,000 105 366 1337 2644 and 161 469 1432 2866.
constexpr std::int64_t kBoxMinNodes = 100000;
constexpr std::int64_t kBoxMinDipoles = 256;
constexpr std::int64_t kBoxMinPairs = 80000000, kBoxMinPairsDeep = 200000000;
constexpr std::int64_t kBoxMinGeneralPairs = 240000000, kBoxMinGeneralPairsDeep = 320000000;
// Leaves one level deeper from here. Sweeps 16 wide at 412,000 nodes, 4,000 dipoles: 28.1 ms with the
// shallower leaves and 27.6 deeper (flat coil), 34.2 and 32.0 (moments that differ), 400 dipoles 23.5 and
// 24.1; at 214,000 nodes, 8,700 chunks deeper against 4,500, most leaves would hold fewer nodes than the
// 216 points they take. At the deepest level a placement's box values take up to 100 MB.
constexpr std::int64_t kBoxDeepNodes = 400000;
constexpr std::int64_t kBoxDeeperNodes = 3200000;

// Chunks from which a wide block's node pass takes a block per chunk (4,500 chunks at 213,000 nodes: 16
// and 32 placements of 1,800 dipoles 1102 and 2116 us so, 994 and 1836 with waves sharing a chunk; 8,000
// at 412,000: 1623 and 3323 so, 1659 and 3432 shared), and
// (chunk, placement) tasks below which eight and four waves share one (one placement at 7,400 nodes has
// 116 tasks: 15 us for 964 dipoles).
constexpr int kWideMinChunks = 8192;
constexpr int kNarrow = 4;  // placements up to which a block of the box passes takes two points a lane
constexpr std::int64_t kSplitTasks8 = 2048;
constexpr std::int64_t kSplitTasks4 = 8192;

// (chunk, placement) tasks from which near chunks go on a list: 4 placements of 4,000 dipoles at 213,000
// nodes (18,000 tasks) 1175 us without and 1204 with it, 16 (72,000) 3604 and 3102; 16 at 125,000 (39,000)
// 2712 and 2594; 4 at 667,000 (41,000) 1938 and 1728.
constexpr std::int64_t kListTasks = 32768;
static_assert(kListTasks <= 9 * kWideMinChunks, "node_wide_kernel leaves near chunks to the list");

// LDS added to a workgroup that runs beside a solve, so that it leaves the solve's kernels their wave
// slots: of 160 KB a CU holds one workgroup of the box passes or of node_split_kernel with shared waves,
// two of the other node passes (16-wide sweeps: at 213,000 nodes 25.6 ms with the CUs filled, 24.8 so; at
// 966,000 nodes 97.3 and 96.4; a general coil's at 95,000 nodes 28.3 and 25.2). The box and node passes
// of many dipoles whose moments differ take longer than the solves beside them, and then take more of
// the machine (32-wide sweeps at 138,000 nodes: 4,000 dipoles 32.3 ms with the wide pad, 28.4 so, 2,600
// 26.3 and 24.9, 1,800 22.6 and 22.8; of 4,000, 8 wide 13.5 and 12.8, 4 wide 9.6 and 10.0).
constexpr std::size_t kBesideLds = 60 * 1024;
constexpr std::size_t kBesideHeavyLds = 24 * 1024;
constexpr int kHeavyDipoles = 2304, kHeavyWidth = 8;

// tables layout (floats): points of order 8, points of order 6, then for child order 8 and 6 the
// matrices T[half][child point][parent point] (parent order 8).
constexpr int kTabX8 = 0;
constexpr int kTabX6 = 8;
constexpr int kTabT8 = 16;
constexpr int kTabT6 = kTabT8 + 2 * 8 * 8;
constexpr int kTabLen = kTabT6 + 2 * 6 * 8;

// Read-only arrays at wave-uniform addresses, in the constant address space: scalar loads also where
// the kernel writes something else in the same loop.
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef const floatx4 __attribute__((address_space(4)))* UniformQuads;
typedef const float __attribute__((address_space(4)))* UniformFloats;

__device__ __forceinline__ UniformQuads uniform(const float4* p) {
    return reinterpret_cast<UniformQuads>(reinterpret_cast<std::uintptr_t>(p));
}
__device__ __forceinline__ UniformFloats uniform(const float* p) {
    return reinterpret_cast<UniformFloats>(reinterpret_cast<std::uintptr_t>(p));
}

// v_rsq_f32 without rsqrtf's denormal rescale (a squared coil-to-node distance is never denormal).
__device__ __forceinline__ float rsq_normal(float x) { return __builtin_amdgcn_rsqf(x); }

__global__ void leaf_first_kernel(const std::uint64_t* __restrict__ keys, std::int64_t n, int shift,
                                  std::int32_t* __restrict__ first) {
    const std::int64_t i = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const std::uint64_t b = keys[i] >> shift;
    if (i == 0 || (keys[i - 1] >> shift) != b) first[b] = static_cast<std::int32_t>(i);
}

__global__ void fill_i32_kernel(std::int32_t* __restrict__ p, std::int64_t n, std::int32_t v) {
    const std::int64_t i = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// World-axis dipoles relative to each placement's coil origin, transformed in FP64
// (fem/placement.py:294-313) and rounded once. When every moment lies along `dir` (m = mu dir):
// wide (s, mu); close (-2 s, |s|^2), (mu, mu s). Else wide (s, 0), (m, 0); close (s, |s|^2),
// (m, (m x s).x), ((m x s).y, (m x s).z, 0, 0), and the same in the caller's order in `given`.
__global__ void pack_kernel(const double* __restrict__ coil, int n_dip, const double* __restrict__ tf, int k,
                            double d0, double d1, double d2, bool parallel,
                            const std::int32_t* __restrict__ order, float4* __restrict__ wide,
                            float4* __restrict__ close, float4* __restrict__ given, double* __restrict__ origin,
                            float* __restrict__ dirs) {
    const std::int64_t t = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= static_cast<std::int64_t>(k) * n_dip) return;
    const int c = static_cast<int>(t / n_dip), j = static_cast<int>(t % n_dip);
    const double* f = tf + 16 * c;
    const double* p = coil + 6 * static_cast<std::int64_t>(j);
    double sd[3], md[3];
    for (int r = 0; r < 3; ++r) {
        const double o = f[4 * r + 3] * 1e-3;
        double acc = 0.0, am = 0.0;
        for (int q = 0; q < 3; ++q) {
            acc += p[q] * 1e3 * f[4 * r + q];
            am += p[3 + q] * f[4 * r + q];
        }
        sd[r] = (acc + f[4 * r + 3]) * 1e-3 - o;
        md[r] = am;
        if (j == 0) {
            origin[3 * c + r] = o;
            dirs[3 * c + r] = static_cast<float>(d0 * f[4 * r] + d1 * f[4 * r + 1] + d2 * f[4 * r + 2]);
        }
    }
    const float s[3] = {static_cast<float>(sd[0]), static_cast<float>(sd[1]), static_cast<float>(sd[2])};
    const float sn = s[0] * s[0] + s[1] * s[1] + s[2] * s[2];
    if (parallel) {
        const double mu = p[3] * d0 + p[4] * d1 + p[5] * d2;
        const float m = static_cast<float>(mu);
        wide[t] = make_float4(s[0], s[1], s[2], m);
        close[2 * t] = make_float4(-2.0f * s[0], -2.0f * s[1], -2.0f * s[2], sn);
        close[2 * t + 1] = make_float4(m, static_cast<float>(mu * sd[0]), static_cast<float>(mu * sd[1]),
                                       static_cast<float>(mu * sd[2]));
    } else {
        const float m[3] = {static_cast<float>(md[0]), static_cast<float>(md[1]), static_cast<float>(md[2])};
        const float x[3] = {static_cast<float>(md[1] * sd[2] - md[2] * sd[1]),
                            static_cast<float>(md[2] * sd[0] - md[0] * sd[2]),
                            static_cast<float>(md[0] * sd[1] - md[1] * sd[0])};
        wide[2 * t] = make_float4(s[0], s[1], s[2], 0.f);
        wide[2 * t + 1] = make_float4(m[0], m[1], m[2], 0.f);
        close[3 * t] = make_float4(s[0], s[1], s[2], sn);
        close[3 * t + 1] = make_float4(m[0], m[1], m[2], x[0]);
        close[3 * t + 2] = make_float4(x[1], x[2], 0.f, 0.f);
        const std::int64_t g = static_cast<std::int64_t>(c) * n_dip + order[j];
        for (int q = 0; q < 3; ++q) given[3 * g + q] = close[3 * t + q];
    }
}

// far[box, c], bit q: cluster q of placement c is far from the box or from one of its ancestors.
// One wavefront per (box, placement), lane q testing cluster q.
__global__ void __launch_bounds__(kBlock) far_kernel(const double* __restrict__ center,
                                                     const std::int32_t* __restrict__ parent,
                                                     const double* __restrict__ rule, int4 first, int total,
                                                     const double* __restrict__ spheres, const double* __restrict__ tf,
                                                     int k, unsigned long long* __restrict__ far) {
    const std::int64_t w = static_cast<std::int64_t>(blockIdx.x) * (kBlock / kWave) + threadIdx.x / kWave;
    if (w >= static_cast<std::int64_t>(total) * k) return;  // whole wavefronts
    const int lane = threadIdx.x & (kWave - 1);
    const int box = static_cast<int>(w / k), c = static_cast<int>(w % k);
    const double* f = tf + 16 * c;
    const double* sp = spheres + 4 * lane;
    double p[3];
    for (int r = 0; r < 3; ++r)
        p[r] = (sp[0] * f[4 * r] + sp[1] * f[4 * r + 1] + sp[2] * f[4 * r + 2]) + f[4 * r + 3] * 1e-3;
    bool is_far = false;
    for (int b = box; b >= 0; b = parent[b]) {
        const int level = (b >= first.y) + (b >= first.z) + (b >= first.w);
        const double dx = center[3 * b] * 1e-3 - p[0], dy = center[3 * b + 1] * 1e-3 - p[1],
                     dz = center[3 * b + 2] * 1e-3 - p[2];
        is_far |= sqrt(dx * dx + dy * dy + dz * dz) - sp[3] >= rule[level];
    }
    const unsigned long long m = __ballot(is_far);
    if (lane == 0) far[w] = m;
}

// Bounding ball (mm) of each chunk's nodes: the middle and half diagonal of their extents. One
// wavefront per chunk.
__global__ void __launch_bounds__(kBlock) chunk_ball_kernel(const double* __restrict__ nodes_mm, int n_chunks,
                                                            const std::int32_t* __restrict__ chunk_node,
                                                            const std::int32_t* __restrict__ chunk_end,
                                                            double* __restrict__ ball) {
    const int w = static_cast<int>(blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave);
    if (w >= n_chunks) return;  // whole wavefronts
    const int lane = threadIdx.x & (kWave - 1);
    const std::int64_t node = min(chunk_node[w] + lane, chunk_end[w] - 1);
    double r2 = 0.0;
    for (int d = 0; d < 3; ++d) {
        double lo = nodes_mm[3 * node + d], hi = lo;
#pragma unroll
        for (int off = kWave / 2; off > 0; off >>= 1) {
            lo = fmin(lo, __shfl_xor(lo, off, kWave));
            hi = fmax(hi, __shfl_xor(hi, off, kWave));
        }
        r2 += 0.25 * (hi - lo) * (hi - lo);
        if (lane == 0) ball[4 * static_cast<std::int64_t>(w) + d] = 0.5 * (lo + hi);
    }
    if (lane == 0) ball[4 * static_cast<std::int64_t>(w) + 3] = sqrt(r2);
}

// a += sum over the dipoles [j, e) of mu (r - s) / |r - s|^3 (parallel moments) or
// m x (r - s) / |r - s|^3, for U points. The dipoles' addresses are wave-uniform, so they come
// through the scalar cache into scalar registers and cost the vector units nothing.
template <bool PAR, int U>
__device__ __forceinline__ void add_dipoles(UniformQuads dip, int j, int e, const float (&rx)[U],
                                            const float (&ry)[U], const float (&rz)[U], float (&ax)[U],
                                            float (&ay)[U], float (&az)[U]) {
#pragma unroll 4
    for (; j < e; ++j) {
        const floatx4 s = dip[PAR ? j : 2 * j];
        floatx4 m = {0.f, 0.f, 0.f, 0.f};
        if constexpr (!PAR) m = dip[2 * j + 1];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const float dx = rx[u] - s.x, dy = ry[u] - s.y, dz = rz[u] - s.z;
            const float inv = rsq_normal(fmaf(dz, dz, fmaf(dy, dy, dx * dx)));
            if constexpr (PAR) {
                const float w = (inv * s.w) * (inv * inv);
                ax[u] = fmaf(w, dx, ax[u]);
                ay[u] = fmaf(w, dy, ay[u]);
                az[u] = fmaf(w, dz, az[u]);
            } else {
                const float w = inv * (inv * inv);
                const float ex = w * dx, ey = w * dy, ez = w * dz;
                ax[u] = fmaf(m.y, ez, fmaf(-m.z, ey, ax[u]));
                ay[u] = fmaf(m.z, ex, fmaf(-m.x, ez, ay[u]));
                az[u] = fmaf(m.x, ey, fmaf(-m.y, ex, az[u]));
            }
        }
    }
}

__device__ __forceinline__ int cluster_begin(int q, int n_dip) {
    return static_cast<int>(static_cast<std::int64_t>(q) * n_dip / kClusters);
}

// Values at the Chebyshev points of one level's boxes: the sum over the clusters first far at this
// level, plus the parent's values interpolated. blockIdx.x = box * PARTS + part, blockIdx.y the
// placement; a block takes U x 64 (of order 8) or U x 54 (order 6) of the box's points, U per lane, and
// wave w the clusters of slice w. Bound by the vector ALUs where a level has pairs to sum (3.2e12
// pairs/s) and by its LDS passes where it only interpolates. U = 4 passes the parent's values down
// fewer times; U = 2 halves the longest block, which is what a narrow block of placements waits for.
// Values are stored (z, y, component, x), the order the node pass reads.
template <int P, bool PAR, int U>
__global__ void __launch_bounds__(kDipoleThreads) box_points_kernel(
    const double* __restrict__ center, double hx, double hy, double hz, const std::int32_t* __restrict__ parent,
    const std::int32_t* __restrict__ octant, int first, int parent_first, const unsigned long long* __restrict__ far,
    const float4* __restrict__ packed, int n_dip, const double* __restrict__ origin, int k,
    const float* __restrict__ tables, const float* __restrict__ up, float* __restrict__ values) {
    constexpr int P3 = P * P * P;
    constexpr int LANES = P == 8 ? 64 : 54;
    constexpr int PARTS = P3 / (U * LANES);
    static_assert(PARTS * U * LANES == P3, "whole blocks of points");
    constexpr int Q = kUpperOrder, Q3 = Q * Q * Q;
    __shared__ float part_s[kSlices][U][3][kWave];
    __shared__ float pv[3 * Q3], xs[3 * P * Q * Q];
    __shared__ float T[3][P * Q];
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int local = blockIdx.x / PARTS, part = blockIdx.x % PARTS, c = blockIdx.y;
    const int box = first + local;
    const int par = parent[box];
    const unsigned long long cum = far[static_cast<std::int64_t>(box) * k + c];
    if (cum == 0) return;  // nothing reaches this box through points
    const unsigned long long above = par >= 0 ? far[static_cast<std::int64_t>(par) * k + c] : 0ull;
    const unsigned long long mine = cum & ~above;
    if (above != 0) {
        const float* src = up + (static_cast<std::int64_t>(par - parent_first) * k + c) * 3 * Q3;
        for (int e = threadIdx.x; e < 3 * Q3; e += kDipoleThreads) pv[e] = src[e];
        const int oct = octant[box];
        for (int e = threadIdx.x; e < 3 * P * Q; e += kDipoleThreads) {
            const int d = e / (P * Q);
            T[d][e % (P * Q)] = tables[(P == 8 ? kTabT8 : kTabT6) + ((oct >> d) & 1) * P * Q + e % (P * Q)];
        }
    }
    if (mine != 0) {
        const float* xc = tables + (P == 8 ? kTabX8 : kTabX6);
        const double hw[3] = {hx, hy, hz};
        float r[3][U], a[3][U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int q = (part * U + u) * LANES + min(lane, LANES - 1);
            const int i[3] = {q % P, (q / P) % P, q / (P * P)};
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const double x = center[3 * box + d] + static_cast<double>(xc[i[d]]) * hw[d];
                r[d][u] = static_cast<float>(x * 1e-3 - origin[3 * c + d]);
                a[d][u] = 0.f;
            }
        }
        const UniformQuads dip = uniform(packed + static_cast<std::int64_t>(c) * n_dip * (PAR ? 1 : 2));
        unsigned m = static_cast<unsigned>(mine >> (kSliceClusters * wave)) & ((1u << kSliceClusters) - 1u);
        m = __builtin_amdgcn_readfirstlane(m);
        while (m != 0) {  // runs of neighbouring clusters are one run of dipoles
            const int q0 = __builtin_ctz(m);
            const int len = __builtin_ctz(~(m >> q0));
            const int q = kSliceClusters * wave + q0;
            add_dipoles<PAR, U>(dip, cluster_begin(q, n_dip), cluster_begin(q + len, n_dip), r[0], r[1], r[2], a[0], a[1],
                                a[2]);
            m &= ~(((1u << len) - 1u) << q0);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int d = 0; d < 3; ++d) part_s[wave][u][d][lane] = a[d][u];
    }
    __syncthreads();
    if (above != 0) {  // the parent's values along x, then y, then (below) z
        for (int e = threadIdx.x; e < 3 * P * Q * Q; e += kDipoleThreads) {  // e = ((z Q + y) 3 + d) P + i
            const int i = e % P, zyd = e / P;
            float v = 0.f;
#pragma unroll
            for (int x = 0; x < Q; ++x) v = fmaf(T[0][i * Q + x], pv[zyd * Q + x], v);
            xs[e] = v;
        }
        __syncthreads();
        for (int e = threadIdx.x; e < 3 * P * P * Q; e += kDipoleThreads) {  // e = ((z P + j) 3 + d) P + i
            const int id = e % (3 * P), j = (e / (3 * P)) % P, z = e / (3 * P * P);
            float v = 0.f;
#pragma unroll
            for (int y = 0; y < Q; ++y) v = fmaf(T[1][j * Q + y], xs[(z * Q + y) * 3 * P + id], v);
            pv[e] = v;
        }
        __syncthreads();
    }
    float* dst = values + (static_cast<std::int64_t>(local) * k + c) * 3 * P3;
    for (int e = threadIdx.x; e < 3 * U * LANES; e += kDipoleThreads) {  // this block's run of ((z P + y) 3 + d) P + x
        const int f = part * 3 * U * LANES + e;
        const int i = f % P, d = (f / P) % 3, zy = f / (3 * P);
        const int l = zy * P + i - part * U * LANES;
        float v = 0.f;
        if (mine != 0)
#pragma unroll
            for (int w = 0; w < kSlices; ++w) v += part_s[w][l / LANES][d][l % LANES];
        if (above != 0) {
            const int kz = zy / P, jdi = f % (3 * P * P);
            float t = 0.f;
#pragma unroll
            for (int z = 0; z < Q; ++z) t = fmaf(T[2][kz * Q + z], pv[z * 3 * P * P + jdi], t);
            v += t;
        }
        dst[f] = v;
    }
}

// Lagrange weights of the order-6 Chebyshev points at u (in [-1, 1] over the box).
__device__ __forceinline__ void leaf_weights(const float* __restrict__ x, float u, float (&w)[kLeafOrder]) {
#pragma unroll
    for (int i = 0; i < kLeafOrder; ++i) {
        float num = 1.f, den = 1.f;
#pragma unroll
        for (int j = 0; j < kLeafOrder; ++j) {
            if (j == i) continue;
            num *= u - x[j];
            den *= x[i] - x[j];
        }
        w[i] = num / den;
    }
}

// What the node passes read.
struct NodeArgs {
    const double* nodes_mm;
    std::int64_t n;
    int n_chunks;  // 64 nodes of one leaf each (any 64 nodes, every dipole near, without boxes)
    const std::int32_t *chunk_node, *chunk_end, *chunk_leaf;
    int leaf_first;
    const double* center;
    double half[3];
    const float* tables;
    const unsigned long long* far;
    const float* values;
    const float4 *close, *given;
    const double *ball, *spheres, *frames;
    int n_dip;
    const double* origin;
    const float* dirs;
    int k, K;
    float scale;
    float* out;
    const unsigned char* near_flag;  // (n_chunks, k): the chunks on the list
};

struct Chunk {
    std::int64_t n0;
    int cnt, leaf, id;
};

__device__ __forceinline__ Chunk chunk_at(const NodeArgs& a, int chunk) {
    if (a.chunk_leaf != nullptr)
        return {a.chunk_node[chunk], a.chunk_end[chunk] - a.chunk_node[chunk], a.chunk_leaf[chunk], chunk};
    const std::int64_t n0 = static_cast<std::int64_t>(chunk) * kWave;
    return {n0, static_cast<int>(min(static_cast<std::int64_t>(kWave), a.n - n0)), -1, chunk};
}

// The middle of cluster q of placement c (m).
__device__ __forceinline__ void cluster_at(const NodeArgs& a, int c, int q, double* p) {
    const double* f = a.frames + 16 * c;
    const double* sp = a.spheres + 4 * q;
    for (int r = 0; r < 3; ++r)
        p[r] = (sp[0] * f[4 * r] + sp[1] * f[4 * r + 1] + sp[2] * f[4 * r + 2]) + f[4 * r + 3] * 1e-3;
}

// Whether a cluster around p (m) lies within kCloseMm of a chunk's ball (mm).
__device__ __forceinline__ bool within_close(const double* ball, const double* p, double radius) {
    double d2 = 0.0;
    for (int r = 0; r < 3; ++r) {
        const double d = ball[r] * 1e-3 - p[r];
        d2 += d * d;
    }
    return sqrt(d2) - radius < (kCloseMm + ball[3]) * 1e-3;
}

// Whether some cluster (lane q testing cluster q) of placement c lies within kCloseMm of this chunk.
__device__ __forceinline__ bool close_by(const NodeArgs& a, const Chunk& ch, int c) {
    const int q = threadIdx.x & (kWave - 1);
    double p[3];
    cluster_at(a, c, q, p);
    return __ballot(within_close(a.ball + 4 * static_cast<std::int64_t>(ch.id), p, a.spheres[4 * q + 3])) != 0;
}

// How a node pass treats the chunks near a coil: a planar coil's like any other; else it sums every dipole
// there in the caller's order itself, or leaves that to near_given_kernel (as near_chunks_kernel has found;
// the pass keeps its registers for the rest).
enum class Near { kPlain, kSum, kListed };

template <Near NEAR>
__device__ __forceinline__ bool takes_given(const NodeArgs& a, const Chunk& ch, int c) {
    if constexpr (NEAR == Near::kListed) return a.near_flag[static_cast<std::int64_t>(ch.id) * a.k + c] != 0;
    if constexpr (NEAR == Near::kSum) return close_by(a, ch, c);
    return false;
}

struct Weights {
    float x[kLeafOrder], y[kLeafOrder], z[kLeafOrder];
};

__device__ __forceinline__ void node_weights(const NodeArgs& a, const Chunk& ch, const double (&x)[3], Weights& w) {
    if (ch.leaf < 0) return;
    const double* ctr = a.center + 3 * static_cast<std::int64_t>(ch.leaf);
    leaf_weights(a.tables + kTabX6, static_cast<float>((x[0] - ctr[0]) / a.half[0]), w.x);
    leaf_weights(a.tables + kTabX6, static_cast<float>((x[1] - ctr[1]) / a.half[1]), w.y);
    leaf_weights(a.tables + kTabX6, static_cast<float>((x[2] - ctr[2]) / a.half[2]), w.z);
}

// The leaf's values at this lane's node, planes z in 3 H .. 3 H + 2. The values are wave-uniform.
template <int H>
__device__ __forceinline__ void interpolate(UniformFloats v, const Weights& w, float& ax, float& ay,
                                            float& az) {
    constexpr int P = kLeafOrder;
    ax = ay = az = 0.f;
#pragma unroll
    for (int iz = 3 * H; iz < 3 * H + 3; ++iz)
#pragma unroll
        for (int iy = 0; iy < P; ++iy) {
            const UniformFloats row = v + (iz * P + iy) * 3 * P;
            float tx = 0.f, ty = 0.f, tz = 0.f;
#pragma unroll
            for (int ix = 0; ix < P; ++ix) {
                tx = fmaf(w.x[ix], row[ix], tx);
                ty = fmaf(w.x[ix], row[P + ix], ty);
                tz = fmaf(w.x[ix], row[2 * P + ix], tz);
            }
            const float f = w.y[iy] * w.z[iz];
            ax = fmaf(f, tx, ax);
            ay = fmaf(f, ty, ay);
            az = fmaf(f, tz, az);
            // Three rows' values (54 scalar registers) in flight: hoisting more of them spills.
            if (iy % 3 == 2) __builtin_amdgcn_sched_barrier(0);
        }
}

__device__ __forceinline__ void add_general(floatx4 s, floatx4 mo, floatx4 x, const float (&r)[3], float rn, float& w0,
                                            float& w1, float& w2, float& p0, float& p1, float& p2) {
    const float rs = fmaf(r[2], s.z, fmaf(r[1], s.y, r[0] * s.x));
    const float inv = rsq_normal(fmaf(-2.f, rs, rn + s.w));
    const float w = inv * inv * inv;
    w0 = fmaf(w, mo.x, w0);
    w1 = fmaf(w, mo.y, w1);
    w2 = fmaf(w, mo.z, w2);
    p0 = fmaf(w, mo.w, p0);
    p1 = fmaf(w, x.x, p1);
    p2 = fmaf(w, x.y, p2);
}

// Slice sl of the dipoles near a leaf at this lane's node r: with w_j = |r - s_j|^-3,
// sum_j w_j mu_j (r - s_j) = S0 r - S for parallel moments, else sum_j w_j m_j x (r - s_j) = W x r - P.
template <bool PAR>
__device__ __forceinline__ void near_slice(const NodeArgs& a, unsigned long long cum, int sl, int c, const float (&r)[3],
                                           float (&v)[3]) {
    const UniformQuads dip = uniform(a.close + static_cast<std::int64_t>(c) * a.n_dip * (PAR ? 2 : 3));
    unsigned m = static_cast<unsigned>(~cum >> (kSliceClusters * sl)) & ((1u << kSliceClusters) - 1u);
    m = __builtin_amdgcn_readfirstlane(m);
    const float rn = fmaf(r[2], r[2], fmaf(r[1], r[1], r[0] * r[0]));
    float w0 = 0.f, w1 = 0.f, w2 = 0.f, p0 = 0.f, p1 = 0.f, p2 = 0.f;
    while (m != 0) {
        const int q0 = __builtin_ctz(m);
        const int len = __builtin_ctz(~(m >> q0));
        const int q = kSliceClusters * sl + q0;
        const int e = cluster_begin(q + len, a.n_dip);
#pragma unroll 4
        for (int j = cluster_begin(q, a.n_dip); j < e; ++j) {
            if constexpr (PAR) {
                const floatx4 s = dip[2 * j], mu = dip[2 * j + 1];
                const float d2 = fmaf(r[2], s.z, fmaf(r[1], s.y, fmaf(r[0], s.x, s.w))) + rn;
                const float inv = rsq_normal(d2);
                const float w = inv * inv * inv;
                w0 = fmaf(w, mu.x, w0);
                p0 = fmaf(w, mu.y, p0);
                p1 = fmaf(w, mu.z, p1);
                p2 = fmaf(w, mu.w, p2);
            } else {
                const floatx4 s = dip[3 * j], mo = dip[3 * j + 1], x = dip[3 * j + 2];
                add_general(s, mo, x, r, rn, w0, w1, w2, p0, p1, p2);
            }
        }
        m &= ~(((1u << len) - 1u) << q0);
    }
    if constexpr (PAR) {
        v[0] = w0 * r[0] - p0;
        v[1] = w0 * r[1] - p1;
        v[2] = w0 * r[2] - p2;
    } else {
        v[0] = (w1 * r[2] - w2 * r[1]) - p0;
        v[1] = (w2 * r[0] - w0 * r[2]) - p1;
        v[2] = (w0 * r[1] - w1 * r[0]) - p2;
    }
}

// Every dipole of placement c in the caller's order: W x r - P as one sum.
__device__ __forceinline__ void given_sum(const NodeArgs& a, int c, const float (&r)[3], float (&v)[3]) {
    const UniformQuads dip = uniform(a.given + static_cast<std::int64_t>(c) * a.n_dip * 3);
    const float rn = fmaf(r[2], r[2], fmaf(r[1], r[1], r[0] * r[0]));
    float w0 = 0.f, w1 = 0.f, w2 = 0.f, p0 = 0.f, p1 = 0.f, p2 = 0.f;
#pragma unroll 4
    for (int j = 0; j < a.n_dip; ++j) {
        const floatx4 s = dip[3 * j], mo = dip[3 * j + 1], x = dip[3 * j + 2];
        add_general(s, mo, x, r, rn, w0, w1, w2, p0, p1, p2);
    }
    v[0] = (w1 * r[2] - w2 * r[1]) - p0;
    v[1] = (w2 * r[0] - w0 * r[2]) - p1;
    v[2] = (w0 * r[1] - w1 * r[0]) - p2;
}

template <bool PAR>
__device__ __forceinline__ void turn(const NodeArgs& a, int c, float ax, float ay, float az, float (&o)[3]) {
    if constexpr (PAR) {
        const float d0 = a.dirs[3 * c], d1 = a.dirs[3 * c + 1], d2 = a.dirs[3 * c + 2];
        o[0] = a.scale * (d1 * az - d2 * ay);
        o[1] = a.scale * (d2 * ax - d0 * az);
        o[2] = a.scale * (d0 * ay - d1 * ax);
    } else {
        o[0] = a.scale * ax;
        o[1] = a.scale * ay;
        o[2] = a.scale * az;
    }
}

// The nodes of wide blocks on large meshes: one chunk per block and pass, a wave taking every eighth
// placement. The chunk's (64, 3, K) outputs are gathered in LDS and written as one contiguous run (a
// wave's own three stores touch 64 lines of 12 K bytes each; eight placements a block measured 15 %
// slower). Bound by the latency of the values' scalar loads. Chunks taken in the caller's order are left
// to near_given_kernel.
template <bool PAR>
__global__ void __launch_bounds__(kDipoleThreads) __attribute__((amdgpu_waves_per_eu(6))) node_wide_kernel(NodeArgs a) {
    constexpr Near NEAR = PAR ? Near::kPlain : Near::kListed;
    extern __shared__ float lds[];  // (64, 3 K + 1)
    const int K = a.K, k = a.k, ld = 3 * K + 1;
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int chunk = blockIdx.x; chunk < a.n_chunks; chunk += gridDim.x) {
        const Chunk ch = chunk_at(a, chunk);
        const std::int64_t node = ch.n0 + min(lane, ch.cnt - 1);
        const double x[3] = {a.nodes_mm[3 * node], a.nodes_mm[3 * node + 1], a.nodes_mm[3 * node + 2]};
        Weights w;
        node_weights(a, ch, x, w);
        for (int c = wave; c < K; c += kSlices) {
            float o[3] = {0.f, 0.f, 0.f};
            if (c < k) {
                const bool given = takes_given<NEAR>(a, ch, c);
                const unsigned long long cum = ch.leaf >= 0 ? a.far[static_cast<std::int64_t>(ch.leaf) * k + c] : 0ull;
                const float r[3] = {static_cast<float>(x[0] * 1e-3 - a.origin[3 * c]),
                                    static_cast<float>(x[1] * 1e-3 - a.origin[3 * c + 1]),
                                    static_cast<float>(x[2] * 1e-3 - a.origin[3 * c + 2])};
                float ax = 0.f, ay = 0.f, az = 0.f;
                if (!given && cum != 0) {
                    const UniformFloats v =
                        uniform(a.values + (static_cast<std::int64_t>(ch.leaf - a.leaf_first) * k + c) * kLeafValues);
                    float bx, by, bz;
                    interpolate<0>(v, w, ax, ay, az);
                    interpolate<1>(v, w, bx, by, bz);
                    ax += bx;
                    ay += by;
                    az += bz;
                }
                if (!given && ~cum != 0) {
#pragma unroll 1
                    for (int sl = 0; sl < kSlices; ++sl) {
                        float v[3];
                        near_slice<PAR>(a, cum, sl, c, r, v);
                        ax += v[0];
                        ay += v[1];
                        az += v[2];
                    }
                }
                turn<PAR>(a, c, ax, ay, az, o);
            }
            float* p = lds + lane * ld + c;
            p[0] = o[0];
            p[K] = o[1];
            p[2 * K] = o[2];
        }
        __syncthreads();
        float* dst = a.out + ch.n0 * 3 * K;
        for (int e = threadIdx.x; e < ch.cnt * 3 * K; e += kDipoleThreads) dst[e] = lds[(e / (3 * K)) * ld + e % (3 * K)];
        __syncthreads();
    }
}

// The nodes of narrow blocks, and of meshes with few chunks: WP waves share one chunk of one placement
// (a slice each of the near dipoles, the first two half of the interpolation), so that a single
// placement still fills the machine.
template <Near NEAR, int WP>
__global__ void __launch_bounds__(kDipoleThreads) node_split_kernel(NodeArgs a) {
    constexpr bool PAR = NEAR == Near::kPlain;
    static_assert(WP >= 2, "the interpolation is shared by two waves");
    constexpr int GROUPS = kSlices / WP, PER = kSlices / WP;
    __shared__ float part[GROUPS][kSlices + 2][3][kWave];
    const int K = a.K, k = a.k;
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = wave / WP, q = wave % WP;
    const std::int64_t tasks = static_cast<std::int64_t>(a.n_chunks) * K;
    for (std::int64_t t0 = static_cast<std::int64_t>(blockIdx.x) * GROUPS; t0 < tasks;
         t0 += static_cast<std::int64_t>(gridDim.x) * GROUPS) {
        const std::int64_t t = min(t0 + g, tasks - 1);
        const int chunk = static_cast<int>(t / K), c = static_cast<int>(t % K);
        const Chunk ch = chunk_at(a, chunk);
        const std::int64_t node = ch.n0 + min(lane, ch.cnt - 1);
        unsigned long long cum = 0;
        bool given = false;
        if (c < k) {
            given = takes_given<NEAR>(a, ch, c);
            cum = ch.leaf >= 0 ? a.far[static_cast<std::int64_t>(ch.leaf) * k + c] : 0ull;
            const double x[3] = {a.nodes_mm[3 * node], a.nodes_mm[3 * node + 1], a.nodes_mm[3 * node + 2]};
            const float r[3] = {static_cast<float>(x[0] * 1e-3 - a.origin[3 * c]),
                                static_cast<float>(x[1] * 1e-3 - a.origin[3 * c + 1]),
                                static_cast<float>(x[2] * 1e-3 - a.origin[3 * c + 2])};
            if (given) {
                if constexpr (NEAR == Near::kSum) {
                    if (q == 0) {
                        float v[3];
                        given_sum(a, c, r, v);
#pragma unroll
                        for (int d = 0; d < 3; ++d) part[g][0][d][lane] = v[d];
                    }
                }
            } else if (q < 2) {
                float ax = 0.f, ay = 0.f, az = 0.f;
                if (cum != 0) {
                    Weights w;
                    node_weights(a, ch, x, w);
                    const UniformFloats v =
                        uniform(a.values + (static_cast<std::int64_t>(ch.leaf - a.leaf_first) * k + c) * kLeafValues);
                    if (q == 0)
                        interpolate<0>(v, w, ax, ay, az);
                    else
                        interpolate<1>(v, w, ax, ay, az);
                }
                part[g][q][0][lane] = ax;
                part[g][q][1][lane] = ay;
                part[g][q][2][lane] = az;
            }
            if (!given && ~cum != 0) {
#pragma unroll 1
                for (int i = 0; i < PER; ++i) {
                    const int sl = q * PER + i;
                    float v[3];
                    near_slice<PAR>(a, cum, sl, c, r, v);
#pragma unroll
                    for (int d = 0; d < 3; ++d) part[g][2 + sl][d][lane] = v[d];
                }
            }
        }
        __syncthreads();
        if (q == 0 && t0 + g < tasks && lane < ch.cnt && !(NEAR == Near::kListed && given)) {
            float o[3] = {0.f, 0.f, 0.f};
            if (c < k) {
                float v[3];
#pragma unroll
                for (int d = 0; d < 3; ++d) v[d] = given ? part[g][0][d][lane] : part[g][0][d][lane] + part[g][1][d][lane];
                if (!given && ~cum != 0)
                    for (int i = 0; i < kSlices; ++i)
#pragma unroll
                        for (int d = 0; d < 3; ++d) v[d] += part[g][2 + i][d][lane];
                turn<PAR>(a, c, v[0], v[1], v[2], o);
            }
            float* p = a.out + node * 3 * K + c;
            p[0] = o[0];
            p[K] = o[1];
            p[2 * K] = o[2];
        }
        __syncthreads();
    }
}

// Placement c's sum in the caller's order at this lane's node, written there.
__device__ __forceinline__ void write_given(const NodeArgs& a, int c, std::int64_t node, bool mine) {
    const float r[3] = {static_cast<float>(a.nodes_mm[3 * node] * 1e-3 - a.origin[3 * c]),
                        static_cast<float>(a.nodes_mm[3 * node + 1] * 1e-3 - a.origin[3 * c + 1]),
                        static_cast<float>(a.nodes_mm[3 * node + 2] * 1e-3 - a.origin[3 * c + 2])};
    float v[3], o[3];
    given_sum(a, c, r, v);
    turn<false>(a, c, v[0], v[1], v[2], o);
    if (!mine) return;
    float* p = a.out + node * 3 * a.K + c;
    p[0] = o[0];
    p[a.K] = o[1];
    p[2 * a.K] = o[2];
}

// Every node of a mesh without boxes, for a coil whose moments differ in direction: one node a lane, so
// that small meshes fill the machine (eight nodes a thread, the shape of the raw entry point's kernel,
// took 383 us for 89,000 nodes and 1,500 dipoles). A capped grid walks the nodes.
__global__ void __launch_bounds__(kBlock) node_given_kernel(NodeArgs a) {
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const std::int64_t tasks = static_cast<std::int64_t>(a.n_chunks) * a.K;
    for (std::int64_t t = static_cast<std::int64_t>(blockIdx.x) * (kBlock / kWave) + wave; t < tasks;
         t += static_cast<std::int64_t>(gridDim.x) * (kBlock / kWave)) {
        const int c = static_cast<int>(t % a.K);
        const std::int64_t i = t / a.K * kWave + lane, node = min(i, a.n - 1);
        if (c < a.k) {
            write_given(a, c, node, i < a.n);
        } else if (i < a.n) {
            float* p = a.out + node * 3 * a.K + c;
            p[0] = p[a.K] = p[2 * a.K] = 0.f;
        }
    }
}

// flag[chunk, c]: whether placement c = blockIdx.y takes the chunk in the caller's order (close_by, one
// chunk a lane); near[c] = those chunks, in no order. `count` starts at zero; one addition a wavefront
// (one a near chunk took 200 us of 16 placements at 966,000 nodes).
__global__ void __launch_bounds__(kBlock) near_chunks_kernel(NodeArgs a, unsigned char* __restrict__ flag,
                                                             std::int32_t* __restrict__ near,
                                                             std::int32_t* __restrict__ count) {
    __shared__ double sphere[kClusters][4];
    const int c = blockIdx.y, t = threadIdx.x;
    if (t < kClusters) {
        cluster_at(a, c, t, sphere[t]);
        sphere[t][3] = a.spheres[4 * t + 3];
    }
    __syncthreads();
    const int chunk = static_cast<int>(blockIdx.x) * kBlock + t;
    bool given = false;
    if (chunk < a.n_chunks) {
        const double* ball = a.ball + 4 * static_cast<std::int64_t>(chunk);
        const double b[4] = {ball[0], ball[1], ball[2], ball[3]};
        for (int q = 0; q < kClusters && !given; ++q) given = within_close(b, sphere[q], sphere[q][3]);
        flag[static_cast<std::int64_t>(chunk) * a.k + c] = given;
    }
    const unsigned long long m = __ballot(given);
    if (m == 0) return;  // whole wavefronts
    const int lane = t & (kWave - 1);
    int at = lane == 0 ? atomicAdd(count + c, __popcll(m)) : 0;
    at = __shfl(at, 0, kWave) + __popcll(m & ((1ull << lane) - 1ull));
    if (given) near[static_cast<std::int64_t>(c) * a.n_chunks + at] = chunk;
}

// Placement blockIdx.y at its near chunks, one a wavefront: in the node passes of a wide block the waves
// that share a chunk, or a block, would wait for the one that sums every dipole (32 placements of 4,000
// dipoles at 125,000 nodes: 5.0 to 4.5 ms; with two chunks a wavefront 4.9, with four 5.5).
__global__ void __launch_bounds__(kBlock) near_given_kernel(NodeArgs a, const std::int32_t* __restrict__ near,
                                                            const std::int32_t* __restrict__ count) {
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = blockIdx.y, chunks = count[c];
    for (int q = static_cast<int>(blockIdx.x) * (kBlock / kWave) + wave; q < chunks;
         q += static_cast<int>(gridDim.x) * (kBlock / kWave)) {
        const Chunk ch = chunk_at(a, near[static_cast<std::int64_t>(c) * a.n_chunks + q]);
        write_given(a, c, ch.n0 + min(lane, ch.cnt - 1), lane < ch.cnt);
    }
}

double cheb_point(int i, int p) { return std::cos((i + 0.5) * M_PI / p); }

// Lagrange weight of point i of order p at u.
double lagrange(int i, int p, double u) {
    double w = 1.0;
    for (int j = 0; j < p; ++j)
        if (j != i) w *= (u - cheb_point(j, p)) / (cheb_point(i, p) - cheb_point(j, p));
    return w;
}

// The direction every dipole moment lies along, if there is one (coil models of planar windings
// put all their moments on the coil normal): |m_j x d| <= 1e-12 |m_j| for all j. Writes the unit
// direction of the largest moment.
bool common_moment_direction(const double* mom, std::int64_t n_dip, double* d) {
    std::int64_t big = 0;
    double best = 0.0;
    for (std::int64_t j = 0; j < n_dip; ++j) {
        const double q = mom[3 * j] * mom[3 * j] + mom[3 * j + 1] * mom[3 * j + 1] + mom[3 * j + 2] * mom[3 * j + 2];
        if (q > best) {
            best = q;
            big = j;
        }
    }
    if (!(best > 0.0)) return false;
    const double nb = std::sqrt(best);
    for (int r = 0; r < 3; ++r) d[r] = mom[3 * big + r] / nb;
    for (std::int64_t j = 0; j < n_dip; ++j) {
        const double* m = mom + 3 * j;
        const double cx = m[1] * d[2] - m[2] * d[1], cy = m[2] * d[0] - m[0] * d[2], cz = m[0] * d[1] - m[1] * d[0];
        const double mm = m[0] * m[0] + m[1] * m[1] + m[2] * m[2];
        if (cx * cx + cy * cy + cz * cz > 1e-24 * mm) return false;
    }
    return true;
}

struct Site {
    float x[3];
    std::int32_t i;
};

// Splits p[at(q0), at(q1)) (the clusters q0 .. q1 - 1) into four along its longest axis, and each of
// those again: by 256 bins and a stable counting sort, 40 us for 2,400 dipoles where bisection by
// selection took 350.
void split_clusters(Site* p, Site* tmp, int n_dip, int q0, int q1) {
    if (q1 - q0 < 4) return;
    const auto at = [n_dip](int q) { return static_cast<int>(static_cast<std::int64_t>(q) * n_dip / kClusters); };
    const int b = at(q0), e = at(q1);
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int j = b; j < e; ++j)
        for (int d = 0; d < 3; ++d) {
            lo[d] = std::min(lo[d], p[j].x[d]);
            hi[d] = std::max(hi[d], p[j].x[d]);
        }
    int axis = 0;
    for (int d = 1; d < 3; ++d)
        if (hi[d] - lo[d] > hi[axis] - lo[axis]) axis = d;
    const float width = hi[axis] - lo[axis], scale = width > 0.f ? 255.f / width : 0.f;
    const auto bin = [&](const Site& s) {
        const float v = (s.x[axis] - lo[axis]) * scale;
        return v > 0.f ? std::min(static_cast<int>(std::min(v, 255.f)), 255) : 0;  // NaN falls in bin 0
    };
    int start[257] = {};
    for (int j = b; j < e; ++j) ++start[1 + bin(p[j])];
    for (int k = 0; k < 256; ++k) start[k + 1] += start[k];
    for (int j = b; j < e; ++j) tmp[b + start[bin(p[j])]++] = p[j];
    std::copy(tmp + b, tmp + e, p + b);
    const int q = (q1 - q0) / 4;
    for (int k = 0; k < 4; ++k) split_clusters(p, tmp, n_dip, q0 + k * q, q0 + (k + 1) * q);
}

}  // namespace

void build_box_tree(BoxTree& t, const double* nodes_mm, std::int64_t n, hipStream_t s) {
    t.levels = 0;
    t.n = n;
    if (n < kBoxMinNodes) return;
    const int leaf_level = n >= kBoxDeeperNodes ? 5 : n >= kBoxDeepNodes ? 4 : 3;
    const int levels = leaf_level - kTopLevel + 1;
    double lo[3], span[3];
    bounding_box(nodes_mm, n, lo, span, s);
    DeviceBuffer<std::uint64_t> keys(n, "box keys");
    morton_keys(nodes_mm, n, keys.get(), s);
    const std::int64_t cells = 1ll << (3 * leaf_level);
    DeviceBuffer<std::int32_t> d_first(cells, "leaf starts");
    fill_i32_kernel<<<grid_for(cells), kBlock, 0, s>>>(d_first.get(), cells, -1);
    leaf_first_kernel<<<grid_for(n), kBlock, 0, s>>>(keys.get(), n, 63 - 3 * leaf_level, d_first.get());
    std::vector<std::int32_t> start(cells);
    d2h(start.data(), d_first.get(), cells, s);
    sync(s, "leaf starts");
    // Boxes of every level, in key order; the leaves in node order with them.
    std::vector<double> center;
    std::vector<std::int32_t> parent, octant, leaf_start;
    std::vector<std::int32_t> index, above;  // box of a cell at the current and the coarser level
    int total = 0;
    for (int li = 0; li < levels; ++li) {
        const int level = kTopLevel + li;
        const std::int64_t nc = 1ll << (3 * level), per = 1ll << (3 * (leaf_level - level));
        above.swap(index);
        index.assign(nc, -1);
        t.first[li] = total;
        for (int d = 0; d < 3; ++d) t.half[li][d] = std::ldexp(span[d], -level - 1);
        for (std::int64_t cell = 0; cell < nc; ++cell) {
            bool any = false;
            for (std::int64_t q = cell * per; q < (cell + 1) * per && !any; ++q) any = start[q] >= 0;
            if (!any) continue;
            index[cell] = total++;
            for (int d = 0; d < 3; ++d) {
                std::int64_t i = 0;
                for (int b = 0; b < level; ++b) i |= ((cell >> (3 * b + d)) & 1) << b;
                center.push_back(lo[d] + (2 * i + 1) * t.half[li][d]);
            }
            parent.push_back(li == 0 ? -1 : above[cell >> 3]);
            octant.push_back(static_cast<std::int32_t>(cell & 7));
            if (li == levels - 1) leaf_start.push_back(start[cell]);
        }
        t.n_box[li] = total - t.first[li];
    }
    for (int li = levels; li < kMaxBoxLevels; ++li) t.first[li] = total;
    leaf_start.push_back(static_cast<std::int32_t>(n));
    std::vector<std::int32_t> cn, ce, cl;
    for (int b = 0; b < t.n_box[levels - 1]; ++b)
        for (std::int32_t i = leaf_start[b]; i < leaf_start[b + 1]; i += kWave) {
            cn.push_back(i);
            ce.push_back(std::min(i + kWave, leaf_start[b + 1]));
            cl.push_back(t.first[levels - 1] + b);
        }
    std::vector<double> rule(kMaxBoxLevels, INFINITY);
    for (int li = 0; li < levels; ++li)
        rule[li] = (li == levels - 1 ? kLeafDistance : kUpperDistance) * 1e-3 *
                   std::max(t.half[li][0], std::max(t.half[li][1], t.half[li][2]));
    std::vector<float> tab(kTabLen);
    for (int i = 0; i < 8; ++i) tab[kTabX8 + i] = static_cast<float>(cheb_point(i, 8));
    for (int i = 0; i < 6; ++i) tab[kTabX6 + i] = static_cast<float>(cheb_point(i, 6));
    for (int half = 0; half < 2; ++half)
        for (int j = 0; j < 8; ++j) {
            const double off = half ? 0.5 : -0.5;
            for (int i = 0; i < 8; ++i)
                tab[kTabT8 + (half * 8 + i) * 8 + j] = static_cast<float>(lagrange(j, 8, off + 0.5 * cheb_point(i, 8)));
            for (int i = 0; i < 6; ++i)
                tab[kTabT6 + (half * 6 + i) * 8 + j] = static_cast<float>(lagrange(j, 8, off + 0.5 * cheb_point(i, 6)));
        }
    t.total = total;
    t.n_chunks = static_cast<int>(cn.size());
    t.center = upload(center.data(), center.size(), s, "box centres");
    t.parent = upload(parent.data(), parent.size(), s, "box parents");
    t.octant = upload(octant.data(), octant.size(), s, "box octants");
    t.rule = upload(rule.data(), rule.size(), s, "box rule");
    t.tables = upload(tab.data(), tab.size(), s, "box tables");
    t.chunk_node = upload(cn.data(), cn.size(), s, "chunks");
    t.chunk_end = upload(ce.data(), ce.size(), s, "chunks");
    t.chunk_leaf = upload(cl.data(), cl.size(), s, "chunks");
    t.chunk_ball.reset(4 * cn.size(), "chunk balls");
    chunk_ball_kernel<<<grid_for(t.n_chunks, kBlock / kWave), kBlock, 0, s>>>(
        nodes_mm, t.n_chunks, t.chunk_node.get(), t.chunk_end.get(), t.chunk_ball.get());
    sync(s, "box tree");  // the sources above are function-local
    t.levels = levels;
}

void set_coil(DipoleSet& d, const BoxTree& t, const double* pos_m, const double* mom,
              std::int64_t n_dip, hipStream_t s) {
    require(n_dip >= 1 && n_dip <= INT32_MAX / 6, "dipole count out of range");
    d.n = static_cast<int>(n_dip);
    d.parallel = common_moment_direction(mom, n_dip, d.dir);
    const bool deep = t.n >= kBoxDeepNodes;
    const std::int64_t pairs = d.parallel ? (deep ? kBoxMinPairsDeep : kBoxMinPairs)
                                          : (deep ? kBoxMinGeneralPairsDeep : kBoxMinGeneralPairs);
    d.boxes = t.levels > 0 && n_dip >= kBoxMinDipoles && t.n * n_dip >= pairs;
    std::vector<std::int32_t> order(static_cast<std::size_t>(n_dip));
    for (int i = 0; i < d.n; ++i) order[i] = i;
    if (d.boxes) {
        std::vector<Site> site(2 * static_cast<std::size_t>(n_dip));
        for (int i = 0; i < d.n; ++i) {
            for (int q = 0; q < 3; ++q) site[i].x[q] = static_cast<float>(pos_m[3 * static_cast<std::int64_t>(i) + q]);
            site[i].i = i;
        }
        split_clusters(site.data(), site.data() + n_dip, d.n, 0, kClusters);
        for (int i = 0; i < d.n; ++i) order[i] = site[i].i;
    }
    const std::size_t sphere_at = 6 * static_cast<std::size_t>(n_dip), order_at = sphere_at + 4 * kClusters;
    const std::size_t order_bytes = sizeof(std::int32_t) * static_cast<std::size_t>(n_dip);
    double* h = static_cast<double*>(d.stage_coil.fill(sizeof(double) * order_at + order_bytes));
    std::memcpy(h + order_at, order.data(), order_bytes);
    for (int i = 0; i < d.n; ++i)
        for (int q = 0; q < 3; ++q) {
            h[6 * i + q] = pos_m[3 * static_cast<std::int64_t>(order[i]) + q];
            h[6 * i + 3 + q] = mom[3 * static_cast<std::int64_t>(order[i]) + q];
        }
    if (d.boxes) {
        for (int q = 0; q < kClusters; ++q) {
            const std::int64_t a = static_cast<std::int64_t>(q) * d.n / kClusters,
                               b = static_cast<std::int64_t>(q + 1) * d.n / kClusters;
            double lo[3], hi[3], r2 = 0.0;
            double* o = h + sphere_at + 4 * q;
            for (int x = 0; x < 3; ++x) {
                lo[x] = hi[x] = h[6 * a + x];
                for (std::int64_t i = a; i < b; ++i) {
                    lo[x] = std::min(lo[x], h[6 * i + x]);
                    hi[x] = std::max(hi[x], h[6 * i + x]);
                }
                o[x] = 0.5 * (lo[x] + hi[x]);
            }
            for (std::int64_t i = a; i < b; ++i) {
                double e = 0.0;
                for (int x = 0; x < 3; ++x) e += (h[6 * i + x] - o[x]) * (h[6 * i + x] - o[x]);
                r2 = std::max(r2, e);
            }
            o[3] = std::sqrt(r2);
        }
    }
    d.coil.ensure(sphere_at, "coil dipoles");
    d.spheres.ensure(4 * kClusters, "coil clusters");
    d.stage_coil.send(d.coil.get(), 0, sizeof(double) * sphere_at, s);
    d.order.ensure(static_cast<std::size_t>(n_dip), "coil order");
    d.stage_coil.send(d.order.get(), sizeof(double) * order_at, order_bytes, s);
    if (d.boxes) d.stage_coil.send(d.spheres.get(), sizeof(double) * sphere_at, sizeof(double) * 4 * kClusters, s);
    d.stage_coil.done(s);
}

void dadt_block(DipoleSet& d, const BoxTree& t, const double* nodes_mm, std::int64_t n, const double* tf, int k, int K,
                float scale, float* out, int max_blocks, bool beside, hipStream_t s) {
    if (n <= 0 || k <= 0) return;
    const bool heavy = d.boxes && !d.parallel && d.n >= kHeavyDipoles && k >= kHeavyWidth;
    const std::size_t pad = !beside ? 0 : heavy ? kBesideHeavyLds : kBesideLds;
    require(d.n >= 1, "no coil has been set");
    d.frames.ensure(16 * static_cast<std::size_t>(k), "coil frames");
    d.origin.ensure(3 * static_cast<std::size_t>(k), "coil origins");
    d.dirs.ensure(3 * static_cast<std::size_t>(k), "moment directions");
    d.wide.ensure(static_cast<std::size_t>(k) * d.n * (d.parallel ? 1 : 2), "packed dipoles");
    d.close.ensure(static_cast<std::size_t>(k) * d.n * (d.parallel ? 2 : 3), "packed dipoles");
    if (!d.parallel) d.given.ensure(static_cast<std::size_t>(k) * d.n * 3, "packed dipoles");
    d.stage_frames.put(d.frames.get(), tf, 16 * static_cast<std::size_t>(k), s);
    pack_kernel<<<grid_for(static_cast<std::int64_t>(k) * d.n), kBlock, 0, s>>>(
        d.coil.get(), d.n, d.frames.get(), k, d.dir[0], d.dir[1], d.dir[2], d.parallel,
        d.order.get(), d.wide.get(), d.close.get(), d.given.get(), d.origin.get(), d.dirs.get());
    const int leaf = t.levels - 1;
    if (d.boxes) {
        d.far.ensure(static_cast<std::size_t>(t.total) * k, "far clusters");
        far_kernel<<<grid_for(static_cast<std::int64_t>(t.total) * k, kBlock / kWave), kBlock, 0, s>>>(
            t.center.get(), t.parent.get(), t.rule.get(), make_int4(t.first[0], t.first[1], t.first[2], t.first[3]),
            t.total, d.spheres.get(), d.frames.get(), k, d.far.get());
        for (int li = 0; li < t.levels; ++li) {
            const int p = li == leaf ? kLeafOrder : kUpperOrder;
            d.values[li].ensure(static_cast<std::size_t>(t.n_box[li]) * k * 3 * p * p * p, "box values");
            const int u = k <= kNarrow ? 2 : 4;
            const int parts = li == leaf ? 4 / u : 8 / u;
            const dim3 grid(static_cast<unsigned>(t.n_box[li] * parts), static_cast<unsigned>(k));
            auto go = [&](auto kernel) {
                kernel<<<grid, kDipoleThreads, pad, s>>>(
                    t.center.get(), t.half[li][0], t.half[li][1], t.half[li][2], t.parent.get(), t.octant.get(),
                    t.first[li], li > 0 ? t.first[li - 1] : 0, d.far.get(), d.wide.get(), d.n, d.origin.get(), k,
                    t.tables.get(), li > 0 ? d.values[li - 1].get() : nullptr, d.values[li].get());
            };
            auto order = [&](auto par) {
                constexpr bool PAR = decltype(par)::value;
                if (li == leaf)
                    u == 2 ? go(box_points_kernel<kLeafOrder, PAR, 2>) : go(box_points_kernel<kLeafOrder, PAR, 4>);
                else
                    u == 2 ? go(box_points_kernel<kUpperOrder, PAR, 2>) : go(box_points_kernel<kUpperOrder, PAR, 4>);
            };
            d.parallel ? order(std::true_type{}) : order(std::false_type{});
        }
    }
    NodeArgs a{};
    a.nodes_mm = nodes_mm;
    a.n = n;
    a.n_chunks = static_cast<int>((n + kWave - 1) / kWave);
    a.close = d.close.get();
    a.given = d.given.get();
    a.n_dip = d.n;
    a.origin = d.origin.get();
    a.dirs = d.dirs.get();
    a.k = k;
    a.K = K;
    a.scale = scale;
    a.out = out;
    if (d.boxes) {
        a.n_chunks = t.n_chunks;
        a.chunk_node = t.chunk_node.get();
        a.chunk_end = t.chunk_end.get();
        a.chunk_leaf = t.chunk_leaf.get();
        a.leaf_first = t.first[leaf];
        a.center = t.center.get();
        for (int i = 0; i < 3; ++i) a.half[i] = t.half[leaf][i];
        a.tables = t.tables.get();
        a.far = d.far.get();
        a.ball = t.chunk_ball.get();
        a.spheres = d.spheres.get();
        a.frames = d.frames.get();
        a.values = d.values[leaf].get();
    }
    const auto capped = [max_blocks](std::int64_t grid) {
        return static_cast<unsigned>(max_blocks > 0 ? std::min<std::int64_t>(grid, max_blocks) : grid);
    };
    const std::int64_t tasks = static_cast<std::int64_t>(a.n_chunks) * K;
    // Wide blocks of a coil whose moments differ: the near chunks on a list.
    const bool listed = !d.parallel && d.boxes && static_cast<std::int64_t>(a.n_chunks) * k >= kListTasks;
    if (listed) {
        const std::int64_t pairs = static_cast<std::int64_t>(a.n_chunks) * k;
        d.near.ensure(static_cast<std::size_t>(pairs), "near chunks");
        d.near_flag.ensure(static_cast<std::size_t>(pairs), "near chunks");
        d.near_count.ensure(static_cast<std::size_t>(k), "near chunks");
        fill_i32_kernel<<<1, kBlock, 0, s>>>(d.near_count.get(), k, 0);
        near_chunks_kernel<<<dim3(grid_for(a.n_chunks), static_cast<unsigned>(k)), kBlock, 0, s>>>(
            a, d.near_flag.get(), d.near.get(), d.near_count.get());
        a.near_flag = d.near_flag.get();
    }
    if (!d.parallel && !d.boxes) {
        node_given_kernel<<<capped((tasks + kBlock / kWave - 1) / (kBlock / kWave)), kBlock, pad, s>>>(a);
    } else if (k > 8 && a.n_chunks >= kWideMinChunks) {
        const std::size_t lds = std::max(sizeof(float) * static_cast<std::size_t>(kWave) * (3 * K + 1), pad);
        const unsigned grid = capped(a.n_chunks);
        if (d.parallel)
            node_wide_kernel<true><<<grid, kDipoleThreads, lds, s>>>(a);
        else
            node_wide_kernel<false><<<grid, kDipoleThreads, lds, s>>>(a);
    } else {
        const auto go = [&](auto kernel, int groups) {
            kernel<<<capped((tasks + groups - 1) / groups), kDipoleThreads, pad, s>>>(a);
        };
        const auto split = [&](auto near) {
            constexpr Near NEAR = decltype(near)::value;
            if (tasks < kSplitTasks8)
                go(node_split_kernel<NEAR, 8>, 1);
            else if (tasks < kSplitTasks4)
                go(node_split_kernel<NEAR, 4>, 2);
            else
                go(node_split_kernel<NEAR, 2>, 4);
        };
        if (d.parallel)
            split(std::integral_constant<Near, Near::kPlain>{});
        else if (listed)
            split(std::integral_constant<Near, Near::kListed>{});
        else
            split(std::integral_constant<Near, Near::kSum>{});
    }
    if (listed) {
        const std::int64_t blocks = (a.n_chunks + kBlock / kWave - 1) / (kBlock / kWave);
        near_given_kernel<<<dim3(std::max(1u, max_blocks > 0 ? capped(blocks) / k : capped(blocks)), k), kBlock, pad, s>>>(
            a, d.near.get(), d.near_count.get());
    }
    check(hipGetLastError(), "dA/dt launch");
}

}  // namespace cn
