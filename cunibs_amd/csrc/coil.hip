// Coil side of a block of placements: scalp projection and coil frames, the dipole dA/dt N-body,
// the node-to-element average and the right-hand side.
//
// Layouts. Per-placement arrays are placement-major: dA/dt at nodes (k, n, 3), at elements
// (k, m, 3). The right-hand side goes straight into the solver's (n_red, K) row-major block with
// the grounded node dropped.
#include <cfloat>

#include "coil.hpp"

namespace cn {

namespace {

struct Candidate {
    double d2;
    int tri;
};

__device__ __forceinline__ bool closer(const Candidate& x, const Candidate& y) {
    return x.d2 < y.d2 || (x.d2 == y.d2 && x.tri < y.tri);
}

__device__ __forceinline__ double dot3(const double* a, const double* b) {
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
}

// Closest point on triangle (a, b, c) to p (Ericson), solver/coil/place.cu:66-119.
__device__ double closest_on_tri(const double* p, const double* a, const double* b, const double* c, double* q) {
    double ab[3], ac[3], ap[3], bp[3], cp[3];
    for (int i = 0; i < 3; ++i) {
        ab[i] = b[i] - a[i];
        ac[i] = c[i] - a[i];
        ap[i] = p[i] - a[i];
        bp[i] = p[i] - b[i];
        cp[i] = p[i] - c[i];
    }
    const double d1 = dot3(ab, ap), d2 = dot3(ac, ap);
    const double d3 = dot3(ab, bp), d4 = dot3(ac, bp);
    const double d5 = dot3(ab, cp), d6 = dot3(ac, cp);
    const double vc = d1 * d4 - d3 * d2;
    const double vb = d5 * d2 - d1 * d6;
    const double va = d3 * d6 - d5 * d4;
    if (d1 <= 0.0 && d2 <= 0.0) {
        for (int i = 0; i < 3; ++i) q[i] = a[i];
    } else if (d3 >= 0.0 && d4 <= d3) {
        for (int i = 0; i < 3; ++i) q[i] = b[i];
    } else if (vc <= 0.0 && d1 >= 0.0 && d3 <= 0.0) {
        const double t = d1 / (d1 - d3);
        for (int i = 0; i < 3; ++i) q[i] = a[i] + t * ab[i];
    } else if (d6 >= 0.0 && d5 <= d6) {
        for (int i = 0; i < 3; ++i) q[i] = c[i];
    } else if (vb <= 0.0 && d2 >= 0.0 && d6 <= 0.0) {
        const double t = d2 / (d2 - d6);
        for (int i = 0; i < 3; ++i) q[i] = a[i] + t * ac[i];
    } else if (va <= 0.0 && (d4 - d3) >= 0.0 && (d5 - d6) >= 0.0) {
        const double t = (d4 - d3) / ((d4 - d3) + (d5 - d6));
        for (int i = 0; i < 3; ++i) q[i] = b[i] + t * (c[i] - b[i]);
    } else {
        const double denom = 1.0 / (va + vb + vc);
        const double v = vb * denom, w = vc * denom;
        for (int i = 0; i < 3; ++i) q[i] = a[i] + v * ab[i] + w * ac[i];
    }
    const double dx = q[0] - p[0], dy = q[1] - p[1], dz = q[2] - p[2];
    return dx * dx + dy * dy + dz * dz;
}

// place.cu:122-150: one block per (placement, triangle chunk); the minimum over the total order
// (d^2, triangle index) within the chunk.
__global__ void __launch_bounds__(kBlock) place_scan_kernel(const double* __restrict__ centers,
                                                            const double* __restrict__ ta,
                                                            const double* __restrict__ tb,
                                                            const double* __restrict__ tc, int n_tri,
                                                            int n_chunks, Candidate* __restrict__ cand) {
    __shared__ double sd[kBlock];
    __shared__ int st[kBlock];
    const int p = blockIdx.x, chunk = blockIdx.y;
    const int per = (n_tri + n_chunks - 1) / n_chunks;
    const int lo = chunk * per, hi = min(lo + per, n_tri);
    const double ctr[3] = {centers[3 * p], centers[3 * p + 1], centers[3 * p + 2]};
    Candidate best{DBL_MAX, INT_MAX};
    double q[3];
    for (int j = lo + static_cast<int>(threadIdx.x); j < hi; j += kBlock) {
        const double d2 = closest_on_tri(ctr, ta + 3 * static_cast<std::int64_t>(j), tb + 3 * static_cast<std::int64_t>(j),
                                         tc + 3 * static_cast<std::int64_t>(j), q);
        if (d2 < best.d2) best = {d2, j};
    }
    sd[threadIdx.x] = best.d2;
    st[threadIdx.x] = best.tri;
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) {
            const Candidate o{sd[threadIdx.x + w], st[threadIdx.x + w]};
            const Candidate m{sd[threadIdx.x], st[threadIdx.x]};
            if (closer(o, m)) {
                sd[threadIdx.x] = o.d2;
                st[threadIdx.x] = o.tri;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) cand[static_cast<std::int64_t>(p) * n_chunks + chunk] = {sd[0], st[0]};
}

// place.cu:153-230: frame [x | y | z | c] per placement, z the inward normal, y the in-plane
// handle direction, c the projection lifted `distance` along the outward normal.
__global__ void place_frame_kernel(const double* __restrict__ centers, const double* __restrict__ handles,
                                   const double* __restrict__ dists, const double* __restrict__ ta,
                                   const double* __restrict__ tb, const double* __restrict__ tc,
                                   const double* __restrict__ tn, const Candidate* __restrict__ cand,
                                   int n_pl, int n_chunks, int n_tri, double* __restrict__ out,
                                   int* __restrict__ degenerate) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_pl) return;
    const Candidate* mine = cand + static_cast<std::int64_t>(p) * n_chunks;
    Candidate best = mine[0];
    for (int i = 1; i < n_chunks; ++i)
        if (closer(mine[i], best)) best = mine[i];
    // Every distance was NaN only if the inputs were; the host rejects non-finite centres, and a
    // frame built on triangle 0 then stays in bounds rather than reading past the surface.
    const std::int64_t tri = (best.tri >= 0 && best.tri < n_tri) ? best.tri : 0;
    const double ctr[3] = {centers[3 * p], centers[3 * p + 1], centers[3 * p + 2]};
    double proj[3];
    closest_on_tri(ctr, ta + 3 * tri, tb + 3 * tri, tc + 3 * tri, proj);
    const double nrm[3] = {tn[3 * tri], tn[3 * tri + 1], tn[3 * tri + 2]};
    const double z[3] = {-nrm[0], -nrm[1], -nrm[2]};
    double y[3];
    bool from_handle = false;
    if (handles != nullptr) {
        for (int i = 0; i < 3; ++i) y[i] = handles[3 * p + i] - proj[i];
        if (dot3(y, y) > 0.0) {
            const double inv = 1.0 / sqrt(dot3(y, y));
            for (int i = 0; i < 3; ++i) y[i] *= inv;
            const double cz = dot3(y, z);
            if ((1.0 - cz * cz) > 1e-12) {
                for (int i = 0; i < 3; ++i) y[i] -= z[i] * cz;
                const double inv2 = 1.0 / sqrt(dot3(y, y));
                for (int i = 0; i < 3; ++i) y[i] *= inv2;
                from_handle = true;
            }
        }
    }
    if (!from_handle) {
        int m = 0;
        if (fabs(z[1]) < fabs(z[m])) m = 1;
        if (fabs(z[2]) < fabs(z[m])) m = 2;
        double ref[3] = {0.0, 0.0, 0.0};
        ref[m] = 1.0;
        y[0] = z[1] * ref[2] - z[2] * ref[1];
        y[1] = z[2] * ref[0] - z[0] * ref[2];
        y[2] = z[0] * ref[1] - z[1] * ref[0];
        const double inv = 1.0 / sqrt(dot3(y, y));
        for (int i = 0; i < 3; ++i) y[i] *= inv;
    }
    if (degenerate != nullptr) degenerate[p] = from_handle ? 0 : 1;
    const double x[3] = {y[1] * z[2] - y[2] * z[1], y[2] * z[0] - y[0] * z[2], y[0] * z[1] - y[1] * z[0]};
    double* o = out + 16 * static_cast<std::int64_t>(p);
    for (int i = 0; i < 16; ++i) o[i] = 0.0;
    for (int r = 0; r < 3; ++r) {
        o[4 * r + 0] = x[r];
        o[4 * r + 1] = y[r];
        o[4 * r + 2] = z[r];
        o[4 * r + 3] = proj[r] + dists[p] * nrm[r];
    }
    o[15] = 1.0;
}

constexpr int kDadtBlock = 256;
constexpr int kDipTile = 256;
constexpr int kNodesPerThread = 8;

// The direct sum over dipoles given with their m x s and |s|^2 (dadt.cu:27-104), for the kernel-level
// entry point; a block's dA/dt is formed in dipole.hip. Dipole tiles staged in LDS, 8 nodes per
// thread in registers. The reciprocal square root is the bare v_rsq_f32: rsqrtf wraps the same
// instruction in a denormal rescale, and a squared coil-to-node distance is never denormal.
__device__ __forceinline__ float rsq_normal(float x) { return __builtin_amdgcn_rsqf(x); }

__global__ void __launch_bounds__(kDadtBlock) dadt_kernel(const float* __restrict__ dip, int n_dip,
                                                          const double* __restrict__ nodes_mm, std::int64_t n,
                                                          const double* __restrict__ origin, float scale, int K,
                                                          float* __restrict__ out) {
    __shared__ float s_s[kDipTile * 3];
    __shared__ float s_mp[kDipTile * 6];
    __shared__ float s_sn[kDipTile];
    const int c = blockIdx.y;
    const float* dp = dip + static_cast<std::int64_t>(c) * n_dip * 10;  // per placement: s(3) mp(6) sn(1)
    const double ox = origin[3 * c], oy = origin[3 * c + 1], oz = origin[3 * c + 2];
    const std::int64_t T = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
    const std::int64_t t = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    float rx[kNodesPerThread], ry[kNodesPerThread], rz[kNodesPerThread], rn[kNodesPerThread];
    float wx[kNodesPerThread], wy[kNodesPerThread], wz[kNodesPerThread];
    float px[kNodesPerThread], py[kNodesPerThread], pz[kNodesPerThread];
#pragma unroll
    for (int k = 0; k < kNodesPerThread; ++k) {
        const std::int64_t node = t + k * T;
        rx[k] = ry[k] = rz[k] = rn[k] = 0.f;
        if (node < n) {
            rx[k] = static_cast<float>(nodes_mm[3 * node] * 1e-3 - ox);
            ry[k] = static_cast<float>(nodes_mm[3 * node + 1] * 1e-3 - oy);
            rz[k] = static_cast<float>(nodes_mm[3 * node + 2] * 1e-3 - oz);
            rn[k] = fmaf(rz[k], rz[k], fmaf(ry[k], ry[k], rx[k] * rx[k]));
        }
        wx[k] = wy[k] = wz[k] = px[k] = py[k] = pz[k] = 0.f;
    }
    for (int base = 0; base < n_dip; base += kDipTile) {
        const int tile = min(kDipTile, n_dip - base);
        __syncthreads();
        for (int i = threadIdx.x; i < tile; i += kDadtBlock) {
            const float* d = dp + static_cast<std::int64_t>(base + i) * 10;
            s_s[3 * i] = d[0];
            s_s[3 * i + 1] = d[1];
            s_s[3 * i + 2] = d[2];
            for (int q = 0; q < 6; ++q) s_mp[6 * i + q] = d[3 + q];
            s_sn[i] = d[9];
        }
        __syncthreads();
#pragma unroll 4
        for (int j = 0; j < tile; ++j) {
            const float sx = s_s[3 * j], sy = s_s[3 * j + 1], sz = s_s[3 * j + 2], snj = s_sn[j];
            const float m0 = s_mp[6 * j], m1 = s_mp[6 * j + 1], m2 = s_mp[6 * j + 2];
            const float m3 = s_mp[6 * j + 3], m4 = s_mp[6 * j + 4], m5 = s_mp[6 * j + 5];
#pragma unroll
            for (int k = 0; k < kNodesPerThread; ++k) {
                const float rs = fmaf(rz[k], sz, fmaf(ry[k], sy, rx[k] * sx));
                const float d2 = fmaf(-2.f, rs, rn[k] + snj);
                const float inv = rsq_normal(d2);
                const float w = inv * inv * inv;
                wx[k] = fmaf(w, m0, wx[k]);
                wy[k] = fmaf(w, m1, wy[k]);
                wz[k] = fmaf(w, m2, wz[k]);
                px[k] = fmaf(w, m3, px[k]);
                py[k] = fmaf(w, m4, py[k]);
                pz[k] = fmaf(w, m5, pz[k]);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < kNodesPerThread; ++k) {
        const std::int64_t node = t + k * T;
        if (node < n) {
            float* o = out + node * 3 * K + c;
            o[0] = scale * ((wy[k] * rz[k] - wz[k] * ry[k]) - px[k]);
            o[K] = scale * ((wz[k] * rx[k] - wx[k] * rz[k]) - py[k]);
            o[2 * K] = scale * ((wx[k] * ry[k] - wy[k] * rx[k]) - pz[k]);
        }
    }
}

// Element pass over (element, placement), placements fastest so the K lanes of an element read
// and write contiguous memory:
//   dadt_elm = mean of the four nodal vectors       (dadt_element.cu:6-21)
//   q[corner] = dadt_elm . (g[corner] * neg_vc)     (rhs.cu:65-80, the staged corner terms, FP32)
// Placements beyond k (block padding) get zeros, so their right-hand-side columns are zero.
// With `sigma_tag` (K x n_sigma, FP32), placement c weighs element e by -(vol_e * sigma_c[tag_e])
// instead of neg_vc[e] (the same FP32 product the context's neg_vc holds for its own table).
__global__ void element_pass_kernel(const float* __restrict__ nodal, const std::int32_t* __restrict__ tets,
                                    const float* __restrict__ g, const float* __restrict__ neg_vc, std::int64_t m,
                                    int k, int K, float* __restrict__ elm, float* __restrict__ q,
                                    const std::int32_t* __restrict__ corner_pos, const float* __restrict__ vols,
                                    const std::int32_t* __restrict__ tags, const float* __restrict__ sigma_tag,
                                    int n_sigma) {
    const std::int64_t t = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= m * K) return;
    const std::int64_t e = t / K;
    const int c = static_cast<int>(t % K);
    float d[3] = {0.f, 0.f, 0.f};
    if (c < k) {
        const int4 tt = reinterpret_cast<const int4*>(tets)[e];
        const std::int64_t stride = 3 * static_cast<std::int64_t>(K);
        for (int a = 0; a < 3; ++a) {
            const float v0 = nodal[tt.x * stride + a * K + c], v1 = nodal[tt.y * stride + a * K + c];
            const float v2 = nodal[tt.z * stride + a * K + c], v3 = nodal[tt.w * stride + a * K + c];
            d[a] = 0.25f * (((v0 + v1) + v2) + v3);
        }
    }
    if (elm != nullptr)
        for (int a = 0; a < 3; ++a) elm[(e * 3 + a) * K + c] = d[a];
    const float w = sigma_tag != nullptr ? -(vols[e] * sigma_tag[c * n_sigma + tags[e]]) : neg_vc[e];
    for (int i = 0; i < 4; ++i) {
        const float* gc = g + (4 * e + i) * 3;
        const float w0 = gc[0] * w, w1 = gc[1] * w, w2 = gc[2] * w;
        q[static_cast<std::int64_t>(corner_pos[4 * e + i]) * K + c] = fmaf(d[2], w2, fmaf(d[1], w1, d[0] * w0));
    }
}

// Node gather (rhs.cu:84-104): b[node] = sum of its corners' q in node2corner order, written to
// the solver block with the ground row dropped, and optionally to (k, n) full-node storage. The
// element pass stored the corner terms in that order, so a node's terms are one contiguous run. A
// block takes kRhsRows nodes and writes their columns' FP64 sums (fixed tree) to sums (blocks, K).
constexpr int kRhsRows = kWave;

// sums[block, c] = the FP64 sum of a block's kRhsRows rows of column c, a butterfly per column.
__device__ __forceinline__ void block_sums(const float (*tile)[kRhsRows + 1], int K, double* __restrict__ sums) {
    const int lane = threadIdx.x & (kWave - 1), waves = blockDim.x / kWave;
    for (int c = threadIdx.x / kWave; c < K; c += waves) {
        double v = static_cast<double>(tile[c][lane]);
#pragma unroll
        for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
        if (lane == 0) sums[static_cast<std::int64_t>(blockIdx.x) * K + c] = v;
    }
}

__global__ void node_rhs_kernel(const float* __restrict__ q, const std::int32_t* __restrict__ ptr, std::int64_t n,
                                int k, int K, int ground, float* __restrict__ B, float* __restrict__ b_full,
                                float* __restrict__ b_ground, double* __restrict__ sums) {
    __shared__ float tile[32][kRhsRows + 1];  // K <= 32
    const std::int64_t n0 = static_cast<std::int64_t>(blockIdx.x) * kRhsRows;
    for (int t = threadIdx.x; t < kRhsRows * K; t += blockDim.x) {
        const std::int64_t node = n0 + t / K;
        const int c = t % K;
        float acc = 0.f;
        if (node < n) {
            for (int p = ptr[node]; p < ptr[node + 1]; ++p) acc += q[static_cast<std::int64_t>(p) * K + c];
            if (b_full != nullptr && c < k) b_full[c * n + node] = acc;
            if (node != ground)
                B[(node - (node > ground)) * K + c] = acc;
            else if (b_ground != nullptr)
                b_ground[c] = acc;
        }
        tile[c][t / K] = acc;
    }
    __syncthreads();
    if (sums != nullptr) block_sums(tile, K, sums);
}

// The same sums of right-hand sides that were combined from the tissues' (nr, K), with the ground node's
// entry of each (the sum of its tissues' by the column's conductivities) as a last row.
__global__ void combined_sums_kernel(const float* __restrict__ B, std::int64_t nr, int k, int K,
                                     const float* __restrict__ b_ground, int T, const double* __restrict__ sigma,
                                     double* __restrict__ sums) {
    __shared__ float tile[32][kRhsRows + 1];  // K <= 32
    const std::int64_t r0 = static_cast<std::int64_t>(blockIdx.x) * kRhsRows;
    for (int t = threadIdx.x; t < kRhsRows * K; t += blockDim.x) {
        const std::int64_t row = r0 + t / K;
        const int c = t % K;
        float v = 0.f;
        if (row < nr) {
            v = B[row * K + c];
        } else if (row == nr && c < k) {
            double acc = 0.0;
            for (int q = 0; q < T; ++q) acc = fma(sigma[c * T + q], static_cast<double>(b_ground[q]), acc);
            v = static_cast<float>(acc);
        }
        tile[c][t / K] = v;
    }
    __syncthreads();
    block_sums(tile, K, sums);
}

// The right-hand side of a field without sources sums to zero over all nodes; its FP32 rounding
// does not, and whatever is left (5e-8 of the norm) flows to the ground node, which shifts the whole
// potential by 1e-6 to 4e-5 of its norm. The sum of each column is taken back from kBalanceRows rows
// spread over the mesh, each rounded value's error carried to the next, which leaves less than one
// rounding of one entry (the potential's error: 3e-7, that of the solve). One block per column; the
// sum does not depend on the block's width. The carried chain takes 4 us whatever the mesh; the rows
// rounded side by side, with the remainder in one of them, took none of that, but any other rounding
// moves single potentials by the solve's error (2e-6 at five placements of 127,000 nodes).
constexpr int kBalanceRows = kBlock;

__global__ void __launch_bounds__(kBlock) balance_rhs_kernel(const double* __restrict__ sums, std::int64_t blocks,
                                                             std::int64_t n, int K, int ground, float* __restrict__ B,
                                                             float* __restrict__ b_full) {
    __shared__ double s[kBlock];
    __shared__ float v[kBalanceRows];
    const int c = blockIdx.x, t = threadIdx.x;
    double acc = 0.0;
#pragma unroll 8
    for (std::int64_t b = t; b < blocks; b += kBlock) acc += sums[b * K + c];  // eight loads in flight
    s[t] = acc;
    const std::int64_t nr = n - 1;
    const int rows = static_cast<int>(min(static_cast<std::int64_t>(kBalanceRows), nr));
    const std::int64_t row = static_cast<std::int64_t>(t) * nr / rows;
    if (t < rows) v[t] = B[row * K + c];
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if (t < w) s[t] += s[t + w];
        __syncthreads();
    }
    if (t == 0 && s[0] != 0.0) {
        const double share = -s[0] / rows;
        double carry = 0.0;
        for (int i = 0; i < rows; ++i) {
            const double x = static_cast<double>(v[i]) + (share + carry);
            v[i] = static_cast<float>(x);
            carry = x - static_cast<double>(v[i]);
        }
    }
    __syncthreads();
    if (t < rows) {
        B[row * K + c] = v[t];
        if (b_full != nullptr) b_full[c * n + row + (row >= ground)] = v[t];
    }
}

__global__ void corner_pos_kernel(const std::int32_t* __restrict__ idx, std::int64_t count,
                                  std::int32_t* __restrict__ corner_pos) {
    const std::int64_t p = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (p < count) corner_pos[idx[p]] = static_cast<std::int32_t>(p);
}

}  // namespace

void place_transforms(const double* centers, const double* handles, const double* dists, int n_pl, const double* ta,
                      const double* tb, const double* tc, const double* tn, int n_tri, double* out, int* degenerate,
                      int n_cu, hipStream_t s) {
    if (n_pl <= 0 || n_tri <= 0) return;
    const int for_occ = (n_cu + n_pl - 1) / n_pl;
    const int for_size = (n_tri + 1023) / 1024;
    const int n_chunks = std::max(1, std::min(for_occ, for_size));
    DeviceBuffer<Candidate> cand(static_cast<std::size_t>(n_pl) * n_chunks, "placement candidates");
    place_scan_kernel<<<dim3(n_pl, n_chunks), kBlock, 0, s>>>(centers, ta, tb, tc, n_tri, n_chunks, cand.get());
    place_frame_kernel<<<grid_for(n_pl), kBlock, 0, s>>>(centers, handles, dists, ta, tb, tc, tn, cand.get(), n_pl,
                                                         n_chunks, n_tri, out, degenerate);
    sync(s, "placement");
}

void dadt_nbody(const float* dip, int n_dip, const double* nodes_mm, std::int64_t n, const double* origins, int k,
                int K, float scale, float* out, hipStream_t s) {
    if (n <= 0 || k <= 0) return;
    const std::int64_t threads = (n + kNodesPerThread - 1) / kNodesPerThread;
    const unsigned gx = grid_for(threads, kDadtBlock);
    dadt_kernel<<<dim3(gx, k), kDadtBlock, 0, s>>>(dip, n_dip, nodes_mm, n, origins, scale, K, out);
}

void element_pass(const float* nodal, const std::int32_t* tets, const float* g, const float* neg_vc, std::int64_t m,
                  int k, int K, float* elm, float* q, const std::int32_t* corner_pos, hipStream_t s, const float* vols,
                  const std::int32_t* tags, const float* sigma_tag, int n_sigma) {
    if (const unsigned gr = grid_for(m * K))
        element_pass_kernel<<<gr, kBlock, 0, s>>>(nodal, tets, g, neg_vc, m, k, K, elm, q, corner_pos, vols, tags,
                                                  sigma_tag, n_sigma);
}

void corner_positions(const std::int32_t* idx, std::int64_t count, std::int32_t* corner_pos, hipStream_t s) {
    if (const unsigned gr = grid_for(count)) corner_pos_kernel<<<gr, kBlock, 0, s>>>(idx, count, corner_pos);
}

void node_rhs(const float* q, const std::int32_t* ptr, std::int64_t n, int k, int K, int ground, float* B,
              float* b_full, DeviceBuffer<double>& sums, hipStream_t s) {
    const std::int64_t blocks = (n + kRhsRows - 1) / kRhsRows;
    if (blocks <= 0) return;
    sums.ensure(static_cast<std::size_t>(blocks) * K, "right-hand-side sums");
    node_rhs_kernel<<<static_cast<unsigned>(blocks), std::min(kRhsRows * K, 1024), 0, s>>>(
        q, ptr, n, k, K, ground, B, b_full, nullptr, sums.get());
    if (n > 1 && k > 0)
        balance_rhs_kernel<<<static_cast<unsigned>(k), kBlock, 0, s>>>(sums.get(), blocks, n, K, ground, B, b_full);
}

void tissue_rhs(const float* q, const std::int32_t* ptr, std::int64_t n, int ground, float* b, float* b_ground,
                hipStream_t s) {
    if (const unsigned blocks = grid_for(n, kRhsRows))
        node_rhs_kernel<<<blocks, kRhsRows, 0, s>>>(q, ptr, n, 1, 1, ground, b, nullptr, b_ground, nullptr);
}

void balance_combined(float* B, std::int64_t nr, int k, int K, const float* b_ground, int T, const double* sigma,
                      DeviceBuffer<double>& sums, hipStream_t s) {
    if (nr <= 0 || k <= 0) return;
    const std::int64_t blocks = (nr + 1 + kRhsRows - 1) / kRhsRows;
    sums.ensure(static_cast<std::size_t>(blocks) * K, "right-hand-side sums");
    combined_sums_kernel<<<static_cast<unsigned>(blocks), std::min(kRhsRows * K, 1024), 0, s>>>(B, nr, k, K, b_ground, T,
                                                                                               sigma, sums.get());
    balance_rhs_kernel<<<static_cast<unsigned>(k), kBlock, 0, s>>>(sums.get(), blocks, nr + 1, K, 0, B, nullptr);
}

}  // namespace cn
