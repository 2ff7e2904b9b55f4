// The learned part of the warm start: a small MLP (inputs -> hidden -> hidden -> outputs, GELU)
// trained on the GPU with the library's own kernels, mapping a placement's pose (and tissue
// conductivities) to coefficients in the reduced basis of solver-generated solutions.
//
// Training runs in FP32: GEMMs on the FP32 matrix cores for the forward pass, the backward pass and
// the weight gradients, with the bias, an exact GELU (erf form), its derivative and the bias gradient
// in the same kernels, and Adam on FP32 master weights. Inference uses
// BF16 copies of the weights: each layer is a v_mfma_f32_16x16x16bf16_1k GEMM with FP32
// accumulation, the activations rounded to BF16 between layers.
//
// No reference counterpart (cuNIBS has no learned component).
#include <algorithm>
#include <cmath>
#include <random>
#include <vector>

#include "mlp.hpp"

namespace cn {

namespace {

typedef __attribute__((__vector_size__(4 * sizeof(short)))) short bf16x4_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4_t;

__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }

__device__ __forceinline__ float gelu_grad(float x) {
    return 0.5f * (1.0f + erff(x * 0.70710678118654752f)) + x * 0.39894228040143268f * expf(-0.5f * x * x);
}

constexpr int kTile = 64;    // output tile of the FP32 GEMM: 64 x 64 per block, 32 x 32 per wavefront
constexpr int kTileK = 32;   // K chunk staged in LDS
constexpr int kPitch = kTileK + 4;
constexpr int kGemmThreads = 256;

enum Epilogue : int {
    kPlain = 0,     // C = acc
    kBias = 1,      // C = acc + bias
    kGelu = 2,      // C = z = acc + bias, H = gelu(z)
    kGeluGrad = 3,  // C = acc gelu'(Z)
};

struct GemmArgs {
    int M, N, K;
    const float* A;  // A(i, k): A[i * lda + k], or A[k * lda + i] transposed
    int lda;
    const float* B;  // B(k, j): B[k * ldb + j], or B[j * ldb + k] transposed
    int ldb;
    float* C;  // (M, N), the split's part of the partials when K is split
    const float* bias;
    const float* Z;
    float* H;
    float* colsum;  // kPlain: column sums of B over its K rows (the bias gradient)
    int k_per;      // K rows per split, a multiple of kTileK (blockIdx.z = split)
};

// One operand's 64 x kTileK chunk into registers: two float4 a thread along the contiguous dimension
// (leading dimensions and contiguous extents are multiples of 4), zeros past the edges.
// KC: k is contiguous. `r` counts rows of the tile, `R` the extent of that dimension.
template <bool KC>
__device__ __forceinline__ void load_chunk(const float* __restrict__ p, int ld, int r0, int R, int k0, int k1,
                                           float4 (&v)[2]) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int t = threadIdx.x + u * kGemmThreads;
        const int r = r0 + (KC ? t / (kTileK / 4) : 4 * (t % (kTile / 4)));
        const int k = k0 + (KC ? 4 * (t % (kTileK / 4)) : t / (kTile / 4));
        v[u] = (r < R && k < k1) ? *reinterpret_cast<const float4*>(p + (KC ? static_cast<long>(r) * ld + k
                                                                             : static_cast<long>(k) * ld + r))
                                 : make_float4(0.f, 0.f, 0.f, 0.f);
    }
}

// The chunk into LDS as rows of kTileK consecutive k.
template <bool KC>
__device__ __forceinline__ void store_chunk(const float4 (&v)[2], float (&s)[kTile][kPitch]) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int t = threadIdx.x + u * kGemmThreads;
        if constexpr (KC) {
            *reinterpret_cast<float4*>(&s[t / (kTileK / 4)][4 * (t % (kTileK / 4))]) = v[u];
        } else {
            const int r = 4 * (t % (kTile / 4)), k = t / (kTile / 4);
            s[r][k] = v[u].x;
            s[r + 1][k] = v[u].y;
            s[r + 2][k] = v[u].z;
            s[r + 3][k] = v[u].w;
        }
    }
}

// C = A B on the FP32 matrix cores (v_mfma_f32_16x16x4f32, FP32 products and sums). Each wavefront
// keeps 2 x 2 tiles of 16 x 16; a lane reads four consecutive k of its row of either operand in one
// 16-byte LDS read and feeds them to four products, so product u of a 16-k group takes the k's
// 4 (l / 16) + u of both. The next chunk's global loads are in flight during the products.
// The weight gradients have few tiles (64 for 512 x 512) and a long K, so they split K over
// blockIdx.z until 512 blocks are in flight, partials added in order. The gradients of a 2048-row
// batch at 512 hidden and 256 outputs: 3.4 ms with vector-ALU tiles, unsplit, and a bias gradient
// serial in the rows; 0.7 ms now with the copies, 0.16 ms of it in these kernels (24 us for the
// 2048 x 512 x 512 product, 45 TFLOP/s: its 256 blocks are one wavefront a SIMD).
template <bool AKC, bool BKC, int EPI>
__global__ void __launch_bounds__(kGemmThreads) gemm_f32_kernel(GemmArgs g) {
    __shared__ __align__(16) float As[kTile][kPitch];
    __shared__ __align__(16) float Bs[kTile][kPitch];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row = lane & 15, quad = lane >> 4;
    const int wi = 32 * (wave >> 1), wj = 32 * (wave & 1);
    const int i0 = blockIdx.y * kTile, j0 = blockIdx.x * kTile;
    const int k0 = blockIdx.z * g.k_per, k1 = min(k0 + g.k_per, g.K);
    floatx4_t acc[2][2] = {};
    float sum = 0.0f;
    float4 av[2], bv[2];
    load_chunk<AKC>(g.A, g.lda, i0, g.M, k0, k1, av);
    load_chunk<BKC>(g.B, g.ldb, j0, g.N, k0, k1, bv);
    for (int k = k0; k < k1; k += kTileK) {
        store_chunk<AKC>(av, As);
        store_chunk<BKC>(bv, Bs);
        __syncthreads();
        load_chunk<AKC>(g.A, g.lda, i0, g.M, k + kTileK, k1, av);
        load_chunk<BKC>(g.B, g.ldb, j0, g.N, k + kTileK, k1, bv);
#pragma unroll
        for (int c = 0; c < kTileK; c += 16) {
            floatx4_t a[2], b[2];
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                a[x] = *reinterpret_cast<const floatx4_t*>(&As[wi + 16 * x + row][c + 4 * quad]);
                b[x] = *reinterpret_cast<const floatx4_t*>(&Bs[wj + 16 * x + row][c + 4 * quad]);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int x = 0; x < 2; ++x)
#pragma unroll
                    for (int y = 0; y < 2; ++y)
                        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[x][u], b[y][u], acc[x][y], 0, 0, 0);
        }
        if constexpr (EPI == kPlain) {
            if (g.colsum != nullptr && blockIdx.y == 0 && threadIdx.x < kTile)
                for (int kk = 0; kk < kTileK; ++kk) sum += Bs[threadIdx.x][kk];
        }
        __syncthreads();
    }
    const long part = static_cast<long>(blockIdx.z) * g.M * g.N;
    if constexpr (EPI == kPlain) {
        if (g.colsum != nullptr && blockIdx.y == 0 && threadIdx.x < kTile && j0 + static_cast<int>(threadIdx.x) < g.N)
            g.colsum[static_cast<long>(blockIdx.z) * g.N + j0 + threadIdx.x] = sum;
    }
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = i0 + wi + 16 * x + 4 * quad + v, j = j0 + wj + 16 * y + row;
                if (i >= g.M || j >= g.N) continue;
                const long at = static_cast<long>(i) * g.N + j;
                float r = acc[x][y][v];
                if constexpr (EPI == kBias || EPI == kGelu) r += g.bias[j];
                if constexpr (EPI == kGeluGrad) r *= gelu_grad(g.Z[at]);
                g.C[part + at] = r;
                if constexpr (EPI == kGelu) g.H[at] = gelu(r);
            }
}

// out = the splits' partials added in order: the product's `count` values, then the bias gradient's N.
__global__ void sum_splits_kernel(long count, int N, int splits, const float* __restrict__ parts,
                                  const float* __restrict__ cols, float* __restrict__ out, float* __restrict__ db) {
    const long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= count + N) return;
    const float* p = i < count ? parts + i : cols + (i - count);
    const long step = i < count ? count : N;
    float acc = p[0];
    for (int z = 1; z < splits; ++z) acc += p[z * step];
    (i < count ? out[i] : db[i - count]) = acc;
}

// Mean squared error over the batch: dy = 2 (y - t) / (B * N); per-row partial losses in FP64.
__global__ void mse_kernel(int B, int N, const float* __restrict__ y, const float* __restrict__ t,
                           float* __restrict__ dy, double* __restrict__ row_loss) {
    const int r = blockIdx.x;
    double acc = 0.0;
    for (int j = threadIdx.x; j < N; j += blockDim.x) {
        const float d = y[static_cast<long>(r) * N + j] - t[static_cast<long>(r) * N + j];
        dy[static_cast<long>(r) * N + j] = 2.0f * d / static_cast<float>(B * N);
        acc += static_cast<double>(d) * d;
    }
    __shared__ double s[256];
    s[threadIdx.x] = acc;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) row_loss[r] = s[0];
}

__device__ __forceinline__ unsigned short to_bf16(float x) {
    const unsigned u = __float_as_uint(x);
    return static_cast<unsigned short>((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

// Adam on the FP32 master weights, then the BF16 copy used by inference.
__global__ void adam_kernel(long count, float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m,
                            float* __restrict__ v, float lr, float b1, float b2, float eps, float c1, float c2,
                            unsigned short* __restrict__ w16) {
    const long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    w[i] = wi;
    w16[i] = to_bf16(wi);
}

__global__ void to_bf16_kernel(long count, const float* __restrict__ x, unsigned short* __restrict__ y) {
    const long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < count) y[i] = to_bf16(x[i]);
}

// Y (M, N) FP32 = act(X (M, K) BF16 . W (K, N) BF16 + bias), one wavefront per 16 x 16 tile,
// K stepped by 16 (M, N, K multiples of 16). Lane l supplies A[l % 16][4 (l / 16) + j],
// B[4 (l / 16) + j][l % 16] and receives D[4 (l / 16) + j][l % 16]. With gelu set, the output is
// GELU-activated and also written as BF16 for the next layer.
__global__ void __launch_bounds__(256) mfma_layer_kernel(int M, int N, int K, const unsigned short* __restrict__ X,
                                                         const unsigned short* __restrict__ W,
                                                         const float* __restrict__ bias, int gelu_act,
                                                         float* __restrict__ Y, unsigned short* __restrict__ Y16) {
    const int lane = threadIdx.x & 63;
    const int tile = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int tiles_n = N / 16;
    if (tile >= (M / 16) * tiles_n) return;
    const int i0 = (tile / tiles_n) * 16, j0 = (tile % tiles_n) * 16;
    const int i = lane & 15, q = lane >> 4;
    floatx4_t acc = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < K; k0 += 16) {
        bf16x4_t a, b;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            a[j] = static_cast<short>(X[static_cast<long>(i0 + i) * K + k0 + 4 * q + j]);
            b[j] = static_cast<short>(W[static_cast<long>(k0 + 4 * q + j) * N + j0 + i]);
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const long r = i0 + 4 * q + j;
        const int c = j0 + i;
        float v = acc[j] + bias[c];
        if (gelu_act) v = gelu(v);
        Y[r * N + c] = v;
        if (Y16) Y16[r * N + c] = to_bf16(v);
    }
}

template <bool AKC, bool BKC, int EPI>
void gemm(GemmArgs g, int splits, hipStream_t s) {
    const int chunks = (g.K + kTileK - 1) / kTileK;
    g.k_per = (chunks + splits - 1) / splits * kTileK;
    const dim3 grid((g.N + kTile - 1) / kTile, (g.M + kTile - 1) / kTile, splits);
    gemm_f32_kernel<AKC, BKC, EPI><<<grid, kGemmThreads, 0, s>>>(g);
}

// Splits of the batch in a weight gradient: until 512 blocks are in flight, each of at least 256 rows.
int grad_splits(int M, int N, int B) {
    const int tiles = ((M + kTile - 1) / kTile) * ((N + kTile - 1) / kTile);
    return std::max(1, std::min({512 / tiles, B / 256, 64}));
}

}  // namespace

Mlp::Mlp(int n_in, int n_hidden, int n_out, unsigned seed, hipStream_t s)
    : n_in_(n_in), n_hidden_(n_hidden), n_out_(n_out), s_(s) {
    require(n_in >= 1 && n_in <= 16, "the MLP takes 1 to 16 inputs");
    require(n_hidden >= 16 && n_hidden % 16 == 0 && n_hidden <= 4096, "hidden width must be a multiple of 16");
    require(n_out >= 16 && n_out % 16 == 0 && n_out <= 4096, "output width must be a multiple of 16");
    const int shapes[3][2] = {{kInPad, n_hidden}, {n_hidden, n_hidden}, {n_hidden, n_out}};
    std::mt19937 rng(seed);
    std::vector<float> host;
    for (int l = 0; l < 3; ++l) {
        const int fan_in = l == 0 ? n_in : shapes[l][0];
        offset_[l] = static_cast<long>(host.size());
        std::normal_distribution<float> nd(0.0f, std::sqrt(2.0f / static_cast<float>(fan_in)));
        for (int r = 0; r < shapes[l][0]; ++r)
            for (int c = 0; c < shapes[l][1]; ++c) host.push_back((l == 0 && r >= n_in) ? 0.0f : nd(rng));
        boffset_[l] = static_cast<long>(host.size());
        for (int c = 0; c < shapes[l][1]; ++c) host.push_back(0.0f);
    }
    n_params_ = static_cast<long>(host.size());
    w_.reset(n_params_, "mlp weights");
    g_.reset(n_params_, "mlp grads");
    m_.reset(n_params_, "adam m");
    v_.reset(n_params_, "adam v");
    w16_.reset(n_params_, "mlp bf16 weights");
    set_params(host.data());
    std::vector<float> zeros(n_params_, 0.0f);
    h2d(m_.get(), zeros.data(), n_params_, s_);
    h2d(v_.get(), zeros.data(), n_params_, s_);
    sync(s_, "mlp init");
}

void Mlp::set_params(const float* host) {
    h2d(w_.get(), host, n_params_, s_);
    to_bf16_kernel<<<grid_for(n_params_), kBlock, 0, s_>>>(n_params_, w_.get(), w16_.get());
    sync(s_, "mlp params");
}

void Mlp::get_params(float* host) const {
    d2h(host, w_.get(), n_params_, s_);
    sync(s_, "mlp params");
}

void Mlp::ensure_batch(int B) {
    if (B <= cap_batch_) return;
    const long hb = static_cast<long>(B) * n_hidden_;
    x_.reset(static_cast<long>(B) * kInPad, "mlp x");
    z1_.reset(hb, "z1");
    h1_.reset(hb, "h1");
    z2_.reset(hb, "z2");
    h2_.reset(hb, "h2");
    y_.reset(static_cast<long>(B) * n_out_, "y");
    t_.reset(static_cast<long>(B) * n_out_, "t");
    dy_.reset(static_cast<long>(B) * n_out_, "dy");
    dz_.reset(hb, "dz");
    dz1_.reset(hb, "dz1");
    const int shapes[3][2] = {{kInPad, n_hidden_}, {n_hidden_, n_hidden_}, {n_hidden_, n_out_}};
    std::size_t parts = 1;  // at most 512 tiles of partials; a smaller batch splits no further
    for (const auto& m : shapes)
        if (const int z = grad_splits(m[0], m[1], B); z > 1)
            parts = std::max(parts, static_cast<std::size_t>(z) * (m[0] + 1) * m[1]);
    parts_.reset(parts, "gradient partials");
    loss_.reset(B, "row loss");
    x16_.reset(static_cast<long>(B) * kInPad, "x16");
    h16a_.reset(hb, "h16a");
    h16b_.reset(hb, "h16b");
    cap_batch_ = B;
}

// X (B, n_in) host-padded to (B, kInPad) on upload.
void Mlp::upload_inputs(const float* X, int B) {
    const std::size_t count = static_cast<std::size_t>(B) * kInPad;
    float* pad = static_cast<float*>(stage_.fill(count * sizeof(float)));
    std::fill(pad, pad + count, 0.0f);
    for (int r = 0; r < B; ++r)
        for (int c = 0; c < n_in_; ++c) pad[static_cast<std::size_t>(r) * kInPad + c] = X[static_cast<std::size_t>(r) * n_in_ + c];
    stage_.send(x_.get(), 0, count * sizeof(float), s_);
    stage_.done(s_);
}

double Mlp::forward_backward(int B) {
    const int H = n_hidden_, O = n_out_;
    const float* W1 = w_.get() + offset_[0];
    const float* b1 = w_.get() + boffset_[0];
    const float* W2 = w_.get() + offset_[1];
    const float* b2 = w_.get() + boffset_[1];
    const float* W3 = w_.get() + offset_[2];
    const float* b3 = w_.get() + boffset_[2];
    // forward
    gemm<true, false, kGelu>({B, H, kInPad, x_.get(), kInPad, W1, H, z1_.get(), b1, nullptr, h1_.get()}, 1, s_);
    gemm<true, false, kGelu>({B, H, H, h1_.get(), H, W2, H, z2_.get(), b2, nullptr, h2_.get()}, 1, s_);
    gemm<true, false, kBias>({B, O, H, h2_.get(), H, W3, O, y_.get(), b3}, 1, s_);
    mse_kernel<<<B, 256, 0, s_>>>(B, O, y_.get(), t_.get(), dy_.get(), loss_.get());
    // backward: dW3 = h2^T dy and db3, dz2 = (dy W3^T) gelu'(z2), dW2 = h1^T dz2, ...
    float* G = g_.get();
    auto weight_grad = [&](int M, int N, const float* in, const float* d, int l) {
        const int splits = grad_splits(M, N, B);
        GemmArgs a{M, N, B, in, M, d, N, G + offset_[l]};
        a.colsum = G + boffset_[l];
        if (splits == 1) {
            gemm<false, false, kPlain>(a, 1, s_);
            return;
        }
        const long count = static_cast<long>(M) * N;
        a.C = parts_.get();
        a.colsum = parts_.get() + splits * count;
        gemm<false, false, kPlain>(a, splits, s_);
        sum_splits_kernel<<<grid_for(count + N), kBlock, 0, s_>>>(count, N, splits, parts_.get(), a.colsum,
                                                                  G + offset_[l], G + boffset_[l]);
    };
    weight_grad(H, O, h2_.get(), dy_.get(), 2);
    gemm<true, true, kGeluGrad>({B, H, O, dy_.get(), O, W3, O, dz_.get(), nullptr, z2_.get()}, 1, s_);
    weight_grad(H, H, h1_.get(), dz_.get(), 1);
    gemm<true, true, kGeluGrad>({B, H, H, dz_.get(), H, W2, H, dz1_.get(), nullptr, z1_.get()}, 1, s_);
    weight_grad(kInPad, H, x_.get(), dz1_.get(), 0);
    check(hipGetLastError(), "mlp launches");
    std::vector<double> rl(B);
    d2h(rl.data(), loss_.get(), B, s_);
    sync(s_, "mlp step");
    double loss = 0.0;
    for (double v : rl) loss += v;
    return loss / (static_cast<double>(B) * O);
}

double Mlp::gradients(const float* X, const float* T, int B, float* grads_host) {
    ensure_batch(B);
    upload_inputs(X, B);
    h2d(t_.get(), T, static_cast<std::size_t>(B) * n_out_, s_);
    const double loss = forward_backward(B);
    d2h(grads_host, g_.get(), n_params_, s_);
    sync(s_, "mlp grads");
    return loss;
}

double Mlp::train(const float* X, const float* T, long N, int epochs, int batch, float lr, unsigned seed) {
    require(N >= 1 && batch >= 1 && epochs >= 1, "bad training arguments");
    const int B = static_cast<int>(std::min<long>(batch, N));
    ensure_batch(B);
    std::mt19937 rng(seed);
    std::vector<long> order(N);
    for (long i = 0; i < N; ++i) order[i] = i;
    std::vector<float> xb(static_cast<std::size_t>(B) * n_in_), tb(static_cast<std::size_t>(B) * n_out_);
    double last = 0.0;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    for (int ep = 0; ep < epochs; ++ep) {
        std::shuffle(order.begin(), order.end(), rng);
        double sum = 0.0;
        int steps = 0;
        for (long at = 0; at + B <= N; at += B) {
            for (int r = 0; r < B; ++r) {
                const long src = order[at + r];
                std::copy(X + src * n_in_, X + (src + 1) * n_in_, xb.begin() + static_cast<long>(r) * n_in_);
                std::copy(T + src * n_out_, T + (src + 1) * n_out_, tb.begin() + static_cast<long>(r) * n_out_);
            }
            upload_inputs(xb.data(), B);
            h2d(t_.get(), tb.data(), tb.size(), s_);
            sum += forward_backward(B);
            ++steps_;
            ++steps;
            const float c1 = 1.0f - std::pow(b1, static_cast<float>(steps_));
            const float c2 = 1.0f - std::pow(b2, static_cast<float>(steps_));
            adam_kernel<<<grid_for(n_params_), kBlock, 0, s_>>>(n_params_, w_.get(), g_.get(), m_.get(), v_.get(), lr,
                                                                 b1, b2, eps, c1, c2, w16_.get());
        }
        last = steps ? sum / steps : 0.0;
    }
    sync(s_, "mlp train");
    return last;
}

void Mlp::predict(const float* X, int B, float* Y_host) {
    const int Bp = (B + 15) / 16 * 16;
    ensure_batch(Bp);
    std::vector<float> pad(static_cast<std::size_t>(Bp) * n_in_, 0.0f);
    std::copy(X, X + static_cast<std::size_t>(B) * n_in_, pad.begin());
    upload_inputs(pad.data(), Bp);
    const long xin = static_cast<long>(Bp) * kInPad;
    to_bf16_kernel<<<grid_for(xin), kBlock, 0, s_>>>(xin, x_.get(), x16_.get());
    const int H = n_hidden_, O = n_out_;
    auto layer = [&](const unsigned short* in, int K, int N, int l, bool act, float* out, unsigned short* out16) {
        const int tiles = (Bp / 16) * (N / 16);
        mfma_layer_kernel<<<(tiles + 3) / 4, 256, 0, s_>>>(Bp, N, K, in, w16_.get() + offset_[l],
                                                           w_.get() + boffset_[l], act ? 1 : 0, out, out16);
    };
    layer(x16_.get(), kInPad, H, 0, true, h1_.get(), h16a_.get());
    layer(h16a_.get(), H, H, 1, true, h2_.get(), h16b_.get());
    layer(h16b_.get(), H, O, 2, false, y_.get(), nullptr);
    d2h(Y_host, y_.get(), static_cast<std::size_t>(B) * O, s_);
    sync(s_, "mlp predict");
}

}  // namespace cn
