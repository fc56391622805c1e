// rf_mlp.hip -- the learned initial guess on gfx950: per-fiber features from
// the 16 nearest fibers, a 113-128-128-128-15 tanh MLP (FP32) that predicts
// the fiber's force coefficients in its own frame, and its training
// (forward, backward, mean-squared-error loss, Adam), all hand-written.
//
// Local frame of fiber i: e1 = t_i, e2 = normalize(z x t_i) (x x t_i when t_i
// is parallel to z), e3 = e1 x e2.  Features (113): for each of the 16
// nearest fibers j (segment-segment distance, ascending) the relative centre
// (x_j - x_i)/2, the orientation t_j with the sign that makes t_j.e1 >= 0
// (a fiber is the same segment for +t and -t), both in the local frame, and
// the proximity 0.1/(d_ij + 0.1); then t_i.z.  Targets (15): the coefficients
// a_i^k (k = 1..M, M = 5) in the local frame.
//
// Weight blob (floats): in_mean[113] in_std[113] W1[128x113] b1[128]
// W2[128x128] b2[128] W3[128x128] b3[128] W4[15x128] b4[15] out_mean[15]
// out_std[15].  W is row-major [out][in].
#include "rf_internal.h"
#include "rf_mlp.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

namespace rf {
namespace {

// ---- features / frames ---------------------------------------------------

__device__ __forceinline__ void local_frame(const double* t, double* e1, double* e2, double* e3)
{
    e1[0] = t[0];
    e1[1] = t[1];
    e1[2] = t[2];
    // e2 = z x t  (or x x t)
    double a0 = -t[1], a1 = t[0], a2 = 0.0;
    double nrm = sqrt(a0 * a0 + a1 * a1);
    if (nrm < 1e-6) {
        a0 = 0.0;
        a1 = -t[2];
        a2 = t[1];
        nrm = sqrt(a1 * a1 + a2 * a2);
    }
    e2[0] = a0 / nrm;
    e2[1] = a1 / nrm;
    e2[2] = a2 / nrm;
    e3[0] = e1[1] * e2[2] - e1[2] * e2[1];
    e3[1] = e1[2] * e2[0] - e1[0] * e2[2];
    e3[2] = e1[0] * e2[1] - e1[1] * e2[0];
}

__global__ void features_kernel(int N, int ldn, const double* __restrict__ pos, const double* __restrict__ orient,
                                const int* __restrict__ nbr, const double* __restrict__ nbr_dist,
                                float* __restrict__ X)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    double e1[3], e2[3], e3[3];
    local_frame(orient + 3 * i, e1, e2, e3);
    float* xi = X + (size_t)i * kMlpIn;
    const double* ci = pos + 3 * i;
    for (int r = 0; r < kMlpNeighbours; ++r) {
        const int j = nbr[(size_t)i * ldn + r];
        const double d = nbr_dist[(size_t)i * ldn + r];
        const double dx = pos[3 * j] - ci[0], dy = pos[3 * j + 1] - ci[1], dz = pos[3 * j + 2] - ci[2];
        const double* tj = orient + 3 * j;
        double u1 = tj[0] * e1[0] + tj[1] * e1[1] + tj[2] * e1[2];
        double u2 = tj[0] * e2[0] + tj[1] * e2[1] + tj[2] * e2[2];
        double u3 = tj[0] * e3[0] + tj[1] * e3[1] + tj[2] * e3[2];
        const double sg = (u1 > 0.0 || (u1 == 0.0 && (u2 > 0.0 || (u2 == 0.0 && u3 >= 0.0)))) ? 1.0 : -1.0;
        float* f = xi + 7 * r;
        f[0] = (float)(0.5 * (dx * e1[0] + dy * e1[1] + dz * e1[2]));
        f[1] = (float)(0.5 * (dx * e2[0] + dy * e2[1] + dz * e2[2]));
        f[2] = (float)(0.5 * (dx * e3[0] + dy * e3[1] + dz * e3[2]));
        f[3] = (float)(sg * u1);
        f[4] = (float)(sg * u2);
        f[5] = (float)(sg * u3);
        f[6] = (float)(0.1 / (d + 0.1));
    }
    xi[7 * kMlpNeighbours] = (float)e1[2];
}

// coefficients (global, fiber-major 3M) <-> local frame (M=5 -> 15 values)
__global__ void to_local_kernel(int N, int M, const double* __restrict__ orient, const double* __restrict__ x,
                                float* __restrict__ Y)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    double e1[3], e2[3], e3[3];
    local_frame(orient + 3 * i, e1, e2, e3);
    for (int k = 0; k < M; ++k) {
        const double* a = x + (size_t)i * 3 * M + 3 * k;
        Y[(size_t)i * 3 * M + 3 * k + 0] = (float)(a[0] * e1[0] + a[1] * e1[1] + a[2] * e1[2]);
        Y[(size_t)i * 3 * M + 3 * k + 1] = (float)(a[0] * e2[0] + a[1] * e2[1] + a[2] * e2[2]);
        Y[(size_t)i * 3 * M + 3 * k + 2] = (float)(a[0] * e3[0] + a[1] * e3[1] + a[2] * e3[2]);
    }
}

__global__ void to_global_kernel(int N, int M, const double* __restrict__ orient, const float* __restrict__ Y,
                                 const float* __restrict__ out_mean, const float* __restrict__ out_std,
                                 double* __restrict__ x)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    double e1[3], e2[3], e3[3];
    local_frame(orient + 3 * i, e1, e2, e3);
    for (int k = 0; k < M; ++k) {
        const int q = 3 * k;
        const float* y = Y + (size_t)i * kMlpOut + q;
        const double l1 = (double)y[0] * out_std[q] + out_mean[q];
        const double l2 = (double)y[1] * out_std[q + 1] + out_mean[q + 1];
        const double l3 = (double)y[2] * out_std[q + 2] + out_mean[q + 2];
        double* a = x + (size_t)i * 3 * M + q;
        a[0] = l1 * e1[0] + l2 * e2[0] + l3 * e3[0];
        a[1] = l1 * e1[1] + l2 * e2[1] + l3 * e3[1];
        a[2] = l1 * e1[2] + l2 * e2[2] + l3 * e3[2];
    }
}

// ---- the network -----------------------------------------------------------
// One workgroup carries 16 rows of the batch through every layer: forward,
// and for a gradient the loss and all deltas back to the first hidden layer,
// the activations in LDS.  Every product is v_mfma_f32_16x16x4f32 (FP32
// operands and accumulation): lane l supplies A[l%16][l/16] and B[l/16][l%16]
// and holds D[4(l/16) + r][l%16].  The K index of a product is permuted, the
// same way in both operands: step r of a group of 16 takes k = 4(l/16) + r, so
// one 16-byte read of LDS feeds four steps.  The weights (200 KB) stream from
// L2; a layer's loads are issued before its products.
// What bounds it: seven dependent layers of L2 and LDS latency.  16 rows per
// workgroup (the rows of one matrix instruction) give 256 workgroups at 4096
// rows: 35 us for forward, loss and deltas, where one tiled product per layer
// and pass took 640 us.
typedef float f4v __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));  // weight rows are only 4-byte aligned
typedef float f2v __attribute__((ext_vector_type(2)));

constexpr int kRowTile = 16;   // rows per workgroup
constexpr int kActStride = 132;  // LDS row stride: 16-byte aligned, rows four banks apart
constexpr int kZStride = 128;  // standardised input, zero-padded
constexpr int kDStride = 16;   // output deltas, zero-padded

struct RowsArgs {
    const float* w;
    int W[4], b[4], in_mean, in_std, out_mean, out_std;
    int B;
    const float* X;
    const float* Y;
    const int64_t* idx;  // row of X and Y taken as batch row q (nullptr: q itself)
    float* Yhat;
    float* Z;            // gradient only, as everything below
    float* H[3];
    float* D[4];
    float* partial;
};

__device__ __forceinline__ f4v mfma_f32(float a, float b, f4v c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// acc = act[16 rows][0, K) W^T for the output columns n0..n0+15 (n < O), W row-major [O][K].
template <int K, int O>
__device__ __forceinline__ f4v layer_tile(const float (&act)[kRowTile][kActStride], const float* __restrict__ W, int n0,
                                          int lr, int lk)
{
    constexpr int G = (K + 15) / 16;
    const int n = n0 + lr;
    f4v wv[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const int k = 16 * g + 4 * lk;
        if (n < O && k + 3 < K) {
            wv[g] = *reinterpret_cast<const f4u*>(W + n * K + k);
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) wv[g][r] = (n < O && k + r < K) ? W[n * K + k + r] : 0.f;
        }
    }
    f4v acc = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const f4v a = *reinterpret_cast<const f4v*>(&act[lr][16 * g + 4 * lk]);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc = mfma_f32(a[r], wv[g][r], acc);
    }
    return acc;
}

// acc = delta[16 rows][0, O) W for the input columns n0..n0+15, W row-major [O][128].
template <int O>
__device__ __forceinline__ f4v back_tile(const float (&delta)[kRowTile][kActStride], const float* __restrict__ W, int n0,
                                         int lr, int lk)
{
    constexpr int G = (O + 15) / 16;
    f4v wv[G];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int o = 16 * g + 4 * lk + r;
            wv[g][r] = (o < O) ? W[o * kMlpHidden + n0 + lr] : 0.f;
        }
    f4v acc = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const f4v a = *reinterpret_cast<const f4v*>(&delta[lr][16 * g + 4 * lk]);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc = mfma_f32(a[r], wv[g][r], acc);
    }
    return acc;
}

template <bool GRAD>
__global__ void __launch_bounds__(256) mlp_rows_kernel(const RowsArgs a)
{
    __shared__ __attribute__((aligned(16))) float act[2][kRowTile][kActStride];
    const int t = threadIdx.x, lane = t & 63;
    const int wave = t >> 6;
    const int lr = lane & 15, lk = lane >> 4;
    const int row0 = blockIdx.x * kRowTile;
    for (int e = t; e < kRowTile * kZStride; e += 256) {  // standardised input
        const int r = e / kZStride, c = e % kZStride;
        const int row = row0 + r;
        float z = 0.f;
        if (row < a.B && c < kMlpIn) {
            const int64_t src = a.idx ? a.idx[row] : row;
            z = (a.X[src * kMlpIn + c] - a.w[a.in_mean + c]) / a.w[a.in_std + c];
        }
        act[0][r][c] = z;
        if (GRAD && row < a.B) a.Z[(int64_t)row * kZStride + c] = z;
    }
    __syncthreads();
    float h[3][2][4];  // this lane's activations (rows 4 lk + r, columns 32 wave + 16 u + lr)
#pragma unroll
    for (int l = 0; l < 3; ++l) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int n0 = 32 * wave + 16 * u;
            const f4v acc = (l == 0) ? layer_tile<kMlpIn, kMlpHidden>(act[0], a.w + a.W[0], n0, lr, lk)
                                     : layer_tile<kMlpHidden, kMlpHidden>(act[l & 1], a.w + a.W[l], n0, lr, lk);
            const float bias = a.w[a.b[l] + n0 + lr];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float v = tanhf(acc[r] + bias);
                h[l][u][r] = v;
                act[(l + 1) & 1][4 * lk + r][n0 + lr] = v;
                const int row = row0 + 4 * lk + r;
                if (GRAD && row < a.B) a.H[l][(int64_t)row * kMlpHidden + n0 + lr] = v;
            }
        }
        __syncthreads();
    }
    // output layer (one tile): the third activation is in act[1]
    if (wave == 0) {
        const f4v acc = layer_tile<kMlpHidden, kMlpOut>(act[1], a.w + a.W[3], 0, lr, lk);
        const float bias = (lr < kMlpOut) ? a.w[a.b[3] + lr] : 0.f;
        float loss = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = row0 + 4 * lk + r;
            const float y = acc[r] + bias;
            const bool live = row < a.B && lr < kMlpOut;
            if (live && a.Yhat) a.Yhat[(int64_t)row * kMlpOut + lr] = y;
            if constexpr (GRAD) {
                // mean squared error on standardised targets
                float d = 0.f, sq = 0.f;
                if (live) {
                    const int64_t src = a.idx ? a.idx[row] : row;
                    const float diff = y - (a.Y[src * kMlpOut + lr] - a.w[a.out_mean + lr]) / a.w[a.out_std + lr];
                    d = 2.f * diff / (float)((int64_t)a.B * kMlpOut);
                    sq = diff * diff;
                }
                act[0][4 * lk + r][lr] = d;
                loss += sq;
                if (row < a.B) a.D[3][(int64_t)row * kDStride + lr] = d;
            }
        }
        if constexpr (GRAD) {
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off, 64);
            if (lane == 0) a.partial[blockIdx.x] = loss;
        }
    }
    if constexpr (!GRAD) return;
    __syncthreads();
    // deltas of the hidden layers: (delta W) (1 - h^2)
#pragma unroll
    for (int l = 2; l >= 0; --l) {
        const int in = l & 1;  // delta 3 in act[0], 2 in act[1], 1 in act[0]
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int n0 = 32 * wave + 16 * u;
            const f4v acc = (l == 2) ? back_tile<kMlpOut>(act[in], a.w + a.W[3], n0, lr, lk)
                                     : back_tile<kMlpHidden>(act[in], a.w + a.W[l + 1], n0, lr, lk);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float hv = h[l][u][r];
                const float d = acc[r] * (1.f - hv * hv);
                act[in ^ 1][4 * lk + r][n0 + lr] = d;
                const int row = row0 + 4 * lk + r;
                if (row < a.B) a.D[l][(int64_t)row * kMlpHidden + n0 + lr] = d;
            }
        }
        __syncthreads();
    }
}

// dW_l[o][i] = sum_b delta_l[b][o] in_l[b][i] and db_l[o] = sum_b delta_l[b][o]
// for all four layers in one launch: workgroup = (layer, 64 rows o, 32 columns
// i) x one split of the batch, each wavefront a quarter of the split, the four
// sums met in LDS.  A lane's 16-byte read of a delta row covers o = o0 + 4 lr
// .. + 3 and feeds four 16 x 16 blocks, its 8-byte read of an input row two.
// The split partials (blob order, from first_param) are added in a fixed order
// by grad_reduce_kernel.  Bound by L2 reads of the deltas and activations; at
// 4096 rows 13 us + 5 us for the sum, against 2.9 ms for four products over
// the whole batch by four workgroups each and 2.9 ms for serial bias sums.
constexpr int kGradTasks = 28;  // 8 + 8 + 8 (128 x 128 in 64 x 32) + 4 (15 x 128)
constexpr int kMaxGradSplits = 32;

struct GradArgs {
    int B, splits;
    const float* Z;
    const float* H[3];
    const float* D[4];
    int W[4], b[4];  // offsets from first_param
    float* out;      // [splits][stride]
    int64_t stride;
};

__global__ void __launch_bounds__(256) mlp_grad_kernel(const GradArgs a)
{
    __shared__ float red[4][64 * 32];
    __shared__ float redb[4][64];
    const int task = blockIdx.x;
    const int l = (task < 24) ? task / 8 : 3, tl = (l < 3) ? task % 8 : task - 24;
    const int o0 = (l < 3) ? 64 * (tl / 4) : 0, i0 = 32 * (tl % 4);
    const int O = (l < 3) ? kMlpHidden : kMlpOut, I = (l == 0) ? kMlpIn : kMlpHidden;
    const int ldd = (l < 3) ? kMlpHidden : kDStride;
    const float* delta = a.D[l];
    const float* in = (l == 0) ? a.Z : a.H[l - 1];  // row stride 128 either way
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int lr = lane & 15, lk = lane >> 4;
    const int per = ((a.B + a.splits - 1) / a.splits + 15) / 16 * 16;  // rows per split
    const int b0 = blockIdx.y * per + wave * (per / 4);
    const int b1 = min(a.B, b0 + per / 4);
    const bool dl = l < 3 || lr < 4;  // 4 lr < kDStride
    f4v acc[4][2];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int u = 0; u < 2; ++u) acc[m][u] = f4v{0.f, 0.f, 0.f, 0.f};
    f4v bs = f4v{0.f, 0.f, 0.f, 0.f};
    for (int b = b0; b < b1; b += 16) {  // per / 4 is a multiple of 4: guard each row
        f4v dv[4];
        f2v iv[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int row = b + 4 * q + lk;
            const bool live = row < b1;
            dv[q] = (live && dl) ? *reinterpret_cast<const f4v*>(delta + (int64_t)row * ldd + o0 + 4 * lr)
                                 : f4v{0.f, 0.f, 0.f, 0.f};
            iv[q] = live ? *reinterpret_cast<const f2v*>(in + (int64_t)row * 128 + i0 + 2 * lr) : f2v{0.f, 0.f};
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            bs += dv[q];
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int u = 0; u < 2; ++u) acc[m][u] = mfma_f32(dv[q][m], iv[q][u], acc[m][u]);
        }
    }
    // block (m, u), value r of this lane: o = o0 + 4 (4 lk + r) + m, i = i0 + 2 lr + u
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[wave][(4 * (4 * lk + r) + m) * 32 + 2 * lr + u] = acc[m][u][r];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        float v = bs[m];
        v += __shfl_xor(v, 16, 64);
        v += __shfl_xor(v, 32, 64);
        if (lk == 0) redb[wave][4 * lr + m] = v;
    }
    __syncthreads();
    float* out = a.out + blockIdx.y * a.stride;
    for (int e = t; e < 64 * 32; e += 256) {
        const int o = o0 + e / 32, i = i0 + e % 32;
        if (o < O && i < I) out[a.W[l] + (int64_t)o * I + i] = (red[0][e] + red[1][e]) + (red[2][e] + red[3][e]);
    }
    if (i0 == 0 && t < 64 && o0 + t < O)
        out[a.b[l] + o0 + t] = (redb[0][t] + redb[1][t]) + (redb[2][t] + redb[3][t]);
}

// g[p] = sum of the split partials (no splits: g is complete), and in the last
// workgroup acc[0] += the batch's partial losses.
__global__ void __launch_bounds__(256) grad_reduce_kernel(int n, int splits, int64_t stride,
                                                          const float* __restrict__ part, float* __restrict__ g,
                                                          int losses, const float* __restrict__ partial,
                                                          double* __restrict__ acc)
{
    if (blockIdx.x == gridDim.x - 1) {
        __shared__ double sh[256];
        double s = 0.0;
        for (int i = threadIdx.x; i < losses; i += 256) s += partial[i];
        sh[threadIdx.x] = s;
        __syncthreads();
        for (int st = 128; st > 0; st >>= 1) {
            if (threadIdx.x < st) sh[threadIdx.x] += sh[threadIdx.x + st];
            __syncthreads();
        }
        if (threadIdx.x == 0) acc[0] += sh[0];
        return;
    }
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= n) return;
    float s = 0.f;
    for (int k = 0; k < splits; ++k) s += part[k * stride + p];
    g[p] = s;
}

__global__ void adam_kernel(int n, float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m,
                            float* __restrict__ v, float lr, float b1, float b2, float eps, float c1, float c2)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const float gt = g[t];
    const float mt = b1 * m[t] + (1.f - b1) * gt;
    const float vt = b2 * v[t] + (1.f - b2) * gt * gt;
    m[t] = mt;
    v[t] = vt;
    w[t] -= lr * (mt / c1) / (sqrtf(vt / c2) + eps);
}

inline dim3 grid1(int64_t n, int bs = 256) { return dim3((unsigned)((n + bs - 1) / bs)); }

}  // namespace

MlpLayout mlp_layout()
{
    MlpLayout L;
    int64_t o = 0;
    L.in_mean = o;
    o += kMlpIn;
    L.in_std = o;
    o += kMlpIn;
    const int dims[5] = {kMlpIn, kMlpHidden, kMlpHidden, kMlpHidden, kMlpOut};
    L.first_param = o;
    for (int l = 0; l < 4; ++l) {
        L.W[l] = o;
        o += (int64_t)dims[l + 1] * dims[l];
        L.b[l] = o;
        o += dims[l + 1];
    }
    L.num_params = o - L.first_param;
    L.out_mean = o;
    o += kMlpOut;
    L.out_std = o;
    o += kMlpOut;
    L.total = o;
    return L;
}

hipError_t mlp_features(int N, int ldn, const double* pos, const double* orient, const int* nbr,
                        const double* nbr_dist, float* X, hipStream_t s)
{
    hipLaunchKernelGGL(features_kernel, grid1(N, 128), dim3(128), 0, s, N, ldn, pos, orient, nbr, nbr_dist, X);
    return hipGetLastError();
}

hipError_t mlp_targets(int N, int M, const double* orient, const double* x, float* Y, hipStream_t s)
{
    hipLaunchKernelGGL(to_local_kernel, grid1(N, 128), dim3(128), 0, s, N, M, orient, x, Y);
    return hipGetLastError();
}

namespace {

inline int64_t pad64(int64_t x) { return (x + 63) / 64 * 64; }
inline int loss_blocks(int rows) { return (rows + kRowTile - 1) / kRowTile; }

// Splits of the batch in mlp_grad_kernel: about 256 rows each, so that 28
// tasks x splits fill the chip from a batch of 2048 on; a training batch of
// 256 takes one split and writes the gradient directly.
inline int grad_splits(int rows) { return std::max(1, std::min(kMaxGradSplits, (rows + 255) / 256)); }

RowsArgs rows_args(const float* w, int B, const float* X, float* Yhat)
{
    const MlpLayout L = mlp_layout();
    RowsArgs a{};
    a.w = w;
    for (int l = 0; l < 4; ++l) {
        a.W[l] = (int)L.W[l];
        a.b[l] = (int)L.b[l];
    }
    a.in_mean = (int)L.in_mean;
    a.in_std = (int)L.in_std;
    a.out_mean = (int)L.out_mean;
    a.out_std = (int)L.out_std;
    a.B = B;
    a.X = X;
    a.Yhat = Yhat;
    return a;
}

}  // namespace

// Normalised output Yhat [B][15] of B rows of X.
hipError_t mlp_forward(const float* w, int B, const float* X, float* Yhat, hipStream_t s)
{
    const RowsArgs a = rows_args(w, B, X, Yhat);
    hipLaunchKernelGGL(mlp_rows_kernel<false>, dim3(loss_blocks(B)), dim3(256), 0, s, a);
    return hipGetLastError();
}

// Gradient of the mean squared error of B rows of (X, Y) (rows idx[0..B) of
// them when idx is given) into g (same offsets as the weight blob;
// normalisation entries untouched); acc[0] += the sum of squared errors.
hipError_t mlp_gradient(const float* w, int B, const float* X, const float* Y, const int64_t* idx, MlpBuffers& buf,
                        float* g, double* acc, hipStream_t s)
{
    const MlpLayout L = mlp_layout();
    RowsArgs a = rows_args(w, B, X, nullptr);
    a.Y = Y;
    a.idx = idx;
    a.Z = buf.Z;
    a.partial = buf.partial;
    GradArgs ga{};
    ga.B = B;
    ga.splits = grad_splits(B);
    ga.Z = buf.Z;
    for (int l = 0; l < 3; ++l) ga.H[l] = a.H[l] = buf.H[l];
    for (int l = 0; l < 4; ++l) {
        ga.D[l] = a.D[l] = buf.D[l];
        ga.W[l] = (int)(L.W[l] - L.first_param);
        ga.b[l] = (int)(L.b[l] - L.first_param);
    }
    ga.out = (ga.splits > 1) ? buf.gpart : g + L.first_param;
    ga.stride = pad64(L.num_params);
    hipLaunchKernelGGL(mlp_rows_kernel<true>, dim3(loss_blocks(B)), dim3(256), 0, s, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(mlp_grad_kernel, dim3(kGradTasks, ga.splits), dim3(256), 0, s, ga);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    const int n = (ga.splits > 1) ? (int)L.num_params : 0;
    hipLaunchKernelGGL(grad_reduce_kernel, dim3((n + 255) / 256 + 1), dim3(256), 0, s, n, ga.splits, ga.stride,
                       buf.gpart, g + L.first_param, loss_blocks(B), buf.partial, acc);
    return hipGetLastError();
}

hipError_t mlp_to_global(int N, int M, const double* orient, const float* w, const float* Yhat, double* x,
                         hipStream_t s)
{
    const MlpLayout L = mlp_layout();
    hipLaunchKernelGGL(to_global_kernel, grid1(N, 128), dim3(128), 0, s, N, M, orient, Yhat, w + L.out_mean,
                       w + L.out_std, x);
    return hipGetLastError();
}

hipError_t mlp_adam(int n, float* w, const float* g, float* m, float* v, float lr, int step, hipStream_t s)
{
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - std::pow(b1, (float)step), c2 = 1.f - std::pow(b2, (float)step);
    hipLaunchKernelGGL(adam_kernel, grid1(n), dim3(256), 0, s, n, w, g, m, v, lr, b1, b2, 1e-8f, c1, c2);
    return hipGetLastError();
}

int64_t mlp_buffer_floats(int rows)
{
    const int64_t r = rows;
    const int splits = grad_splits(rows);
    return pad64(r * kZStride) + 6 * pad64(r * kMlpHidden) + pad64(r * kDStride) + pad64(loss_blocks(rows)) +
           (splits > 1 ? splits * pad64(mlp_layout().num_params) : 0);
}

void mlp_buffer_bind(float* base, int rows, MlpBuffers* b)
{
    const int64_t r = rows;
    float* q = base;
    b->rows = rows;
    b->Z = q;
    q += pad64(r * kZStride);
    for (int l = 0; l < 3; ++l) {
        b->H[l] = q;
        q += pad64(r * kMlpHidden);
    }
    for (int l = 0; l < 3; ++l) {
        b->D[l] = q;
        q += pad64(r * kMlpHidden);
    }
    b->D[3] = q;
    q += pad64(r * kDStride);
    b->partial = q;
    q += pad64(loss_blocks(rows));
    b->gpart = q;
}

// Glorot-uniform weights from SplitMix64 ((u >> 11) * 2^-53), zero biases.
void mlp_init_weights(uint64_t seed, float* w)
{
    const MlpLayout L = mlp_layout();
    uint64_t state = seed;
    auto next = [&state]() {
        uint64_t z = (state += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
    };
    const int dims[5] = {kMlpIn, kMlpHidden, kMlpHidden, kMlpHidden, kMlpOut};
    for (int l = 0; l < 4; ++l) {
        const double lim = std::sqrt(6.0 / (dims[l] + dims[l + 1]));
        for (int64_t t = 0; t < (int64_t)dims[l + 1] * dims[l]; ++t) {
            const double u = (double)(next() >> 11) * 0x1.0p-53;
            w[L.W[l] + t] = (float)((2.0 * u - 1.0) * lim);
        }
        for (int t = 0; t < dims[l + 1]; ++t) w[L.b[l] + t] = 0.f;
    }
}

// Column means and deviations (floored) of the samples into the blob.
void mlp_set_standardisation(const float* X, const float* Y, int64_t count, float* w)
{
    const MlpLayout L = mlp_layout();
    auto stats = [count](const float* D, int cols, float* mean, float* sd, double floor_sd) {
        for (int c = 0; c < cols; ++c) {
            double s1 = 0.0, s2 = 0.0;
            for (int64_t r = 0; r < count; ++r) s1 += D[r * cols + c];
            const double mu = s1 / (double)count;
            for (int64_t r = 0; r < count; ++r) {
                const double d = D[r * cols + c] - mu;
                s2 += d * d;
            }
            mean[c] = (float)mu;
            sd[c] = (float)std::max(std::sqrt(s2 / (double)count), floor_sd);
        }
    };
    stats(X, kMlpIn, w + L.in_mean, w + L.in_std, 1e-6);
    stats(Y, kMlpOut, w + L.out_mean, w + L.out_std, 1e-12);
}

// Minibatch Adam with a cosine learning-rate schedule over `epochs` passes
// of `count` device samples (dX, dY); one shuffle per epoch (SplitMix64).
hipError_t mlp_train(float* w, const float* dX, const float* dY, int64_t count, int epochs, int batch, float lr,
                     uint64_t seed, float* loss_per_epoch, hipStream_t s)
{
    const MlpLayout L = mlp_layout();
    if (batch > count) batch = (int)count;
    const int64_t nb = count / batch;
    float* work = nullptr;
    const int64_t nbuf = mlp_buffer_floats(batch);
    const int64_t lt = pad64(L.total);
    const int64_t need = 3 * lt + nbuf;
    hipError_t e = hipMalloc(&work, sizeof(float) * need);
    if (e != hipSuccess) return e;
    int64_t* didx = nullptr;
    double* dacc = nullptr;
    e = hipMalloc(&didx, sizeof(int64_t) * count);
    if (e == hipSuccess) e = hipMalloc(&dacc, sizeof(double));
    std::vector<int64_t> idx(count);
    for (int64_t i = 0; i < count; ++i) idx[i] = i;
    uint64_t state = seed ^ 0xA0761D6478BD642Full;
    auto next = [&state]() {
        uint64_t z = (state += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
    };
    float* g = work;
    float* m = g + lt;
    float* v = m + lt;
    MlpBuffers buf;
    mlp_buffer_bind(v + lt, batch, &buf);
    if (e == hipSuccess) e = hipMemsetAsync(work, 0, sizeof(float) * 3 * lt, s);
    int step = 0;
    for (int ep = 0; ep < epochs && e == hipSuccess; ++ep) {
        for (int64_t i = count - 1; i > 0; --i) std::swap(idx[i], idx[(int64_t)(next() % (uint64_t)(i + 1))]);
        if ((e = hipMemcpyAsync(didx, idx.data(), sizeof(int64_t) * count, hipMemcpyHostToDevice, s)) != hipSuccess) break;
        if ((e = hipMemsetAsync(dacc, 0, sizeof(double), s)) != hipSuccess) break;
        const float lr_e = lr * 0.5f * (1.f + std::cos(3.14159265358979f * (float)ep / (float)epochs));
        for (int64_t b = 0; b < nb && e == hipSuccess; ++b) {
            const int64_t* ib = didx + b * batch;
            if ((e = mlp_gradient(w, batch, dX, dY, ib, buf, g, dacc, s)) != hipSuccess) break;
            e = mlp_adam((int)L.num_params, w + L.first_param, g + L.first_param, m + L.first_param,
                         v + L.first_param, lr_e, ++step, s);
        }
        if (e != hipSuccess) break;
        double acc = 0.0;
        if ((e = hipMemcpyAsync(&acc, dacc, sizeof(double), hipMemcpyDeviceToHost, s)) != hipSuccess) break;
        if ((e = hipStreamSynchronize(s)) != hipSuccess) break;
        if (loss_per_epoch) loss_per_epoch[ep] = (float)(acc / ((double)nb * batch * kMlpOut));
    }
    hipError_t e2 = hipStreamSynchronize(s);
    if (e == hipSuccess) e = e2;
    (void)hipFree(work);
    if (didx) (void)hipFree(didx);
    if (dacc) (void)hipFree(dacc);
    return e;
}

}  // namespace rf
