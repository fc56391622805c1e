// rf_precond.hip -- fiber neighbourhoods on gfx950: k nearest fibers by
// segment-segment distance, and the neighbour-coupled block-Jacobi
// (restricted additive Schwarz) preconditioner built on them.
//
// The diagonal blocks of the system matrix are exactly the identity
// (fortran/matrix_assembly.f90:308-311), so a per-fiber block-Jacobi
// preconditioner is the identity.  The ill-conditioning comes from fibers in
// near contact, whose mutual blocks are large.  For every fiber i the cluster
// C_i = {i} + its K nearest fibers is solved exactly:
//     z_i = [ (A_{C_i C_i})^{-1} r_{C_i} ]_i
// The 3M rows of the cluster inverse that belong to fiber i are precomputed
// once per assembly (Gauss-Jordan in registers, one workgroup per fiber), so
// one application is a gather + small dense product per fiber.
#include "rf_internal.h"
#include "rf_precond.h"

#include <algorithm>
#include <type_traits>

namespace rf {
namespace {

// Distance between the segments c1 + s t1 and c2 + u t2, |s|,|u| <= 1
// (closest points, clamped to both segments).
__device__ __forceinline__ double segment_distance(const double* c1, const double* t1, const double* c2,
                                                   const double* t2)
{
    const double w0[3] = {c1[0] - c2[0], c1[1] - c2[1], c1[2] - c2[2]};
    const double a = t1[0] * t1[0] + t1[1] * t1[1] + t1[2] * t1[2];
    const double b = t1[0] * t2[0] + t1[1] * t2[1] + t1[2] * t2[2];
    const double c = t2[0] * t2[0] + t2[1] * t2[1] + t2[2] * t2[2];
    const double d = t1[0] * w0[0] + t1[1] * w0[1] + t1[2] * w0[2];
    const double e = t2[0] * w0[0] + t2[1] * w0[1] + t2[2] * w0[2];
    const double den = a * c - b * b;
    double s = (den > 1e-12) ? (b * e - c * d) / den : 0.0;
    s = fmin(1.0, fmax(-1.0, s));
    double u = (b * s + e) / c;
    u = fmin(1.0, fmax(-1.0, u));
    s = fmin(1.0, fmax(-1.0, (b * u - d) / a));
    const double dx = w0[0] + s * t1[0] - u * t2[0];
    const double dy = w0[1] + s * t1[1] - u * t2[1];
    const double dz = w0[2] + s * t1[2] - u * t2[2];
    return sqrt(dx * dx + dy * dy + dz * dz);
}

// One wavefront per fiber i: every lane keeps a sorted top-K list of its
// share of the sources, then K rounds of a wavefront min-reduction merge the
// lists (ties broken by the smaller index, so the result is deterministic).
template <int KMAX>
__global__ void __launch_bounds__(256) knn_kernel(int N, int K, const double* __restrict__ pos,
                                                  const double* __restrict__ orient, int* __restrict__ nbr,
                                                  double* __restrict__ nbr_dist)
{
    const int lane = threadIdx.x & 63;
    const int i = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (i >= N) return;
    const double ci[3] = {pos[3 * i], pos[3 * i + 1], pos[3 * i + 2]};
    const double ti[3] = {orient[3 * i], orient[3 * i + 1], orient[3 * i + 2]};
    double dl[KMAX];
    int il[KMAX];
#pragma unroll
    for (int q = 0; q < KMAX; ++q) {
        dl[q] = 1e300;
        il[q] = N;
    }
    for (int j = lane; j < N; j += 64) {
        if (j == i) continue;
        const double cj[3] = {pos[3 * j], pos[3 * j + 1], pos[3 * j + 2]};
        const double tj[3] = {orient[3 * j], orient[3 * j + 1], orient[3 * j + 2]};
        double dv = segment_distance(ci, ti, cj, tj);
        int iv = j;
        if (dv < dl[KMAX - 1]) {
            // insertion into the sorted local list
#pragma unroll
            for (int q = 0; q < KMAX; ++q) {
                if (dv < dl[q]) {
                    const double td = dl[q];
                    const int ti2 = il[q];
                    dl[q] = dv;
                    il[q] = iv;
                    dv = td;
                    iv = ti2;
                }
            }
        }
    }
    int head = 0;
    for (int r = 0; r < K; ++r) {
        double hv = 1e300;
        int hi = N;
#pragma unroll
        for (int q = 0; q < KMAX; ++q)
            if (q == head) {
                hv = dl[q];
                hi = il[q];
            }
        double bv = hv;
        int bi = hi;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const double ov = __shfl_xor(bv, off, 64);
            const int oi = __shfl_xor(bi, off, 64);
            if (ov < bv || (ov == bv && oi < bi)) {
                bv = ov;
                bi = oi;
            }
        }
        if (hi == bi && hv == bv && head < KMAX) ++head;  // the winning lane pops its head
        if (lane == 0) {
            nbr[(size_t)i * K + r] = (bi < N) ? bi : i;
            nbr_dist[(size_t)i * K + r] = bv;
        }
    }
}

// The largest key of the wavefront, in every lane.
__device__ __forceinline__ unsigned long long wave_max(unsigned long long v)
{
    auto join = [](unsigned hi, unsigned lo) { return ((unsigned long long)hi << 32) | lo; };
    auto dpp = [&](auto ctrl) {
        constexpr int C = decltype(ctrl)::value;
        const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)v, C, 0xf, 0xf, true);
        const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(v >> 32), C, 0xf, 0xf, true);
        v = max(v, join(hi, lo));
    };
    dpp(std::integral_constant<int, 0xB1>{});   // lane ^ 1
    dpp(std::integral_constant<int, 0x4E>{});   // lane ^ 2
    dpp(std::integral_constant<int, 0x141>{});  // mirrored in its eight
    dpp(std::integral_constant<int, 0x128>{});  // lane ^ 8
    auto lo = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
    auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(v >> 32), (unsigned)(v >> 32), false, false);
    v = max(join(hi[0], lo[0]), join(hi[1], lo[1]));
    lo = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
    hi = __builtin_amdgcn_permlane32_swap((unsigned)(v >> 32), (unsigned)(v >> 32), false, false);
    return max(join(hi[0], lo[0]), join(hi[1], lo[1]));
}

// body(integral constants 0 .. N-1): register arrays are only indexed by constants
template <int N, typename F, int I = 0>
__device__ __forceinline__ void static_for(F&& body)
{
    if constexpr (I < N) {
        body(std::integral_constant<int, I>{});
        static_for<N, F, I + 1>(static_cast<F&&>(body));
    }
}

// One workgroup per fiber: Gauss-Jordan with partial pivoting on the
// transposed cluster matrix augmented with the first bs unit vectors, which
// leaves in the augmented columns the rows of A_CC^{-1} that belong to fiber
// i.  B[i] is stored as [dim][bs] (bs = 3M, dim = bs (K+1)).
// The matrix stays in registers, element (ty + TY a, tx + TX b) in thread
// (ty, tx) of TY x TX: a step passes only the pivot's column and row through
// LDS and needs two barriers, the rows are not swapped (a row is its unknown's
// once it has been the pivot row) and eliminated columns are skipped.
// The work around a step's update (pivot search, quotient, addresses) is per
// wavefront, so few threads with many elements each are better than 256 with
// few, as far as registers go: 1000 clusters of 75 rows take 111 us with
// 16 x 8 threads, 122 with 16 x 16, 154 with 8 x 8; 421 of 105 rows 161 us with
// 16 x 16, 167 with 16 x 8.  With the matrix in LDS, every column updated in
// every step and five barriers a step they took 932 and 1952 us.
template <typename T, int TY, int TX, int RA, int AB>
__global__ void __launch_bounds__(TY* TX) ras_setup_kernel(int K, int ldn, int bs, const int* __restrict__ nbr,
                                                           const T* __restrict__ A, int64_t lda,
                                                           double* __restrict__ B, int* __restrict__ info)
{
    constexpr int DM = TY * RA, CA = DM / TX;
    static_assert(CA * TX == DM && DM <= 128, "whole column blocks");
    __shared__ double col[2][DM], row[DM + TX * AB], rscale[DM];
    __shared__ int rowcol[DM];  // the unknown of a row: the step it was pivot row in
    __shared__ int fib[kMaxRasNeighbours + 1];
    const int dim = bs * (K + 1), i = blockIdx.x, tid = threadIdx.x;
    const int tx = tid % TX, ty = tid / TX, lane = tid & 63;
    if (tid <= K) fib[tid] = tid == 0 ? i : nbr[(size_t)i * ldn + tid - 1];
    __syncthreads();
    // x[a][b] = A_CC[c][r], r = ty + TY a, c = tx + TX b; cluster index q is
    // global (fib[q / bs] bs + q % bs); rows past dim stay 0 and are no pivots
    double x[RA][CA], g[RA][AB];
    int grow[CA];
#pragma unroll
    for (int b = 0; b < CA; ++b) {
        const int c = min(tx + TX * b, dim - 1);
        grow[b] = fib[c / bs] * bs + c % bs;
    }
#pragma unroll
    for (int a = 0; a < RA; ++a) {
        const int r = min(ty + TY * a, dim - 1);
        const T* at = A + ((int64_t)fib[r / bs] * bs + r % bs) * lda;
#pragma unroll
        for (int b = 0; b < CA; ++b) {
            const double v = (double)at[grow[b]];
            x[a][b] = (ty + TY * a < dim && tx + TX * b < dim) ? v : 0.0;
        }
#pragma unroll
        for (int b = 0; b < AB; ++b) g[a][b] = (ty + TY * a == tx + TX * b && tx + TX * b < bs) ? 1.0 : 0.0;
    }
    auto publish_col = [&](auto kb, int k) {
        if (tx != k % TX) return;
#pragma unroll
        for (int a = 0; a < RA; ++a) col[k & 1][ty + TY * a] = x[a][decltype(kb)::value];
    };
    publish_col(std::integral_constant<int, 0>{}, 0);
    bool singular = false;
    int used = 0;  // bit q: row lane + 64 q has been pivot row
    static_for<CA>([&](auto block) {
        constexpr int KB = decltype(block)::value;  // columns TX KB .. of the steps
        for (int k = TX * KB; k < min(dim, TX * KB + TX); ++k) {
            __syncthreads();
            // the pivot row: largest magnitude among the rows not used yet, the
            // first of equal ones (the last 8 bits of the magnitude give way to it)
            const double* ck = col[k & 1];
            unsigned long long key = 0;
#pragma unroll
            for (int q = 0; q < (DM + 63) / 64; ++q) {
                const int r = lane + 64 * q;
                if (r < dim && !((used >> q) & 1)) {
                    const unsigned long long bits = (unsigned long long)__double_as_longlong(ck[r]) & 0x7FFFFFFFFFFFFFFFull;
                    key = max(key, (bits & ~255ull) | (unsigned)(255 - r));
                }
            }
            const int p = __builtin_amdgcn_readfirstlane(255 - (int)(wave_max(key) & 255ull));
            if (lane == (p & 63)) used |= 1 << (p >> 6);
            const double pv = ck[p];
            singular |= pv == 0.0;  // the same for every thread; goes on (one way out of the loop) with inf and NaN
            const double rp = 1.0 / pv;
            static_for<RA>([&](auto aa) {
                constexpr int a = decltype(aa)::value;
                if (ty + TY * a == p) {
#pragma unroll
                    for (int b = KB; b < CA; ++b) row[tx + TX * b] = x[a][b];
#pragma unroll
                    for (int b = 0; b < AB; ++b) row[DM + tx + TX * b] = g[a][b];
                }
            });
            __syncthreads();
            if (tid == 0) {
                rowcol[p] = k;
                rscale[p] = rp;
            }
            // every other row loses column k; the pivot row is scaled at the end
            double f[RA];
#pragma unroll
            for (int a = 0; a < RA; ++a) f[a] = (ty + TY * a == p) ? 0.0 : ck[ty + TY * a] * rp;
#pragma unroll
            for (int b = KB; b < CA; ++b) {
                const double v = row[tx + TX * b];
#pragma unroll
                for (int a = 0; a < RA; ++a) x[a][b] -= f[a] * v;
            }
#pragma unroll
            for (int b = 0; b < AB; ++b) {
                const double v = row[DM + tx + TX * b];
#pragma unroll
                for (int a = 0; a < RA; ++a) g[a][b] -= f[a] * v;
            }
            if (k + 1 < dim) {
                if ((k + 1) % TX != 0)
                    publish_col(block, k + 1);
                else
                    publish_col(std::integral_constant<int, (KB + 1 < CA ? KB + 1 : KB)>{}, k + 1);
            }
        }
    });
    if (singular) {
        if (tid == 0) atomicExch(info, i + 1);
        return;
    }
    __syncthreads();
    // augmented column q of unknown c = row q of A_CC^{-1}: B[i][c][q]
    double* Bi = B + (size_t)i * dim * bs;
#pragma unroll
    for (int a = 0; a < RA; ++a) {
        const int r = ty + TY * a;
        if (r >= dim) continue;
        const int c = rowcol[r];
        const double sc = rscale[r];
#pragma unroll
        for (int b = 0; b < AB; ++b)
            if (tx + TX * b < bs) Bi[(size_t)c * bs + tx + TX * b] = g[a][b] * sc;
    }
}

// z_i = B_i r_{C_i}: a workgroup per fiber, its lanes in groups of bs that take
// every G-th cluster row, so consecutive lanes read consecutive words of B and
// all loads of a group are in flight together.  A thread per (fiber, row of
// B_i) is 59 workgroups at N = 1000, M = 5 and reads one row after the other.
// N = 1000, M = 5, K = 4: 22 -> 5.4 us; N = 4000 26 -> 11 us (36 MB of B).
constexpr int kRasApplyThreads = 256;
__global__ void __launch_bounds__(kRasApplyThreads) ras_apply_kernel(int K, int ldn, int bs, const int* __restrict__ nbr,
                                                                     const double* __restrict__ B,
                                                                     const double* __restrict__ r,
                                                                     double* __restrict__ z)
{
    __shared__ double part[kRasApplyThreads];
    const int i = blockIdx.x, dim = bs * (K + 1);
    const int G = kRasApplyThreads / bs, grp = threadIdx.x / bs, q = threadIdx.x % bs;
    double s = 0.0;
    if (grp < G) {
        const double* Bi = B + (size_t)i * dim * bs + q;
#pragma unroll 4
        for (int c = grp; c < dim; c += G) {
            const int m = c / bs;
            const int f = m == 0 ? i : nbr[(size_t)i * ldn + m - 1];
            s += Bi[(size_t)c * bs] * r[(size_t)f * bs + c % bs];
        }
    }
    part[threadIdx.x] = s;
    __syncthreads();
    if (grp == 0) {
        for (int h = 1; h < G; ++h) s += part[h * bs + q];
        z[(size_t)i * bs + q] = s;
    }
}

}  // namespace

hipError_t launch_knn(int N, int K, const double* pos, const double* orient, int* nbr, double* nbr_dist,
                      hipStream_t s)
{
    if (K < 1 || K > kMaxNeighbours || K > N - 1) return hipErrorInvalidValue;
    const int fibers_per_block = 4;
    hipLaunchKernelGGL(knn_kernel<kMaxNeighbours>, dim3((N + fibers_per_block - 1) / fibers_per_block),
                       dim3(64 * fibers_per_block), 0, s, N, K, pos, orient, nbr, nbr_dist);
    return hipGetLastError();
}

hipError_t launch_ras_setup(int N, int K, int ldn, int bs, const int* nbr, const void* A, int elem_bytes,
                            int64_t lda, double* B, int* info, hipStream_t s)
{
    const int dim = bs * (K + 1);
    if (K < 1 || K > kMaxRasNeighbours || K > ldn || bs < 1 || bs > 24 || dim > kMaxRasRows) return hipErrorInvalidValue;
    // TY x TX threads with RA rows each; AB covers bs <= 16 or bs <= 24
    auto launch = [&](auto ty, auto tx, auto ra) {
        constexpr int TY = decltype(ty)::value, TX = decltype(tx)::value, RA = decltype(ra)::value;
        auto go = [&](auto* At, auto ab) {
            using T = std::remove_const_t<std::remove_pointer_t<decltype(At)>>;
            hipLaunchKernelGGL((ras_setup_kernel<T, TY, TX, RA, decltype(ab)::value>), dim3(N), dim3(TY * TX), 0, s, K,
                               ldn, bs, nbr, At, lda, B, info);
        };
        auto go_t = [&](auto* At) {
            if (bs <= 16)
                go(At, std::integral_constant<int, (16 + TX - 1) / TX>{});
            else
                go(At, std::integral_constant<int, (24 + TX - 1) / TX>{});
        };
        if (elem_bytes == 8)
            go_t(static_cast<const double*>(A));
        else
            go_t(static_cast<const float*>(A));
    };
    using I8 = std::integral_constant<int, 8>;
    using I16 = std::integral_constant<int, 16>;
    using R4 = std::integral_constant<int, 4>;
    if (dim <= 32)
        launch(I8{}, I8{}, R4{});
    else if (dim <= 64)
        launch(I16{}, I8{}, R4{});
    else if (dim <= 80)
        launch(I16{}, I8{}, std::integral_constant<int, 5>{});
    else if (dim <= 112)
        launch(I16{}, I16{}, std::integral_constant<int, 7>{});
    else
        launch(I16{}, I16{}, std::integral_constant<int, 8>{});
    return hipGetLastError();
}

hipError_t launch_ras_apply(int N, int K, int ldn, int bs, const int* nbr, const double* B, const double* r,
                            double* z, hipStream_t s)
{
    hipLaunchKernelGGL(ras_apply_kernel, dim3(N), dim3(kRasApplyThreads), 0, s, K, ldn, bs, nbr, B, r, z);
    return hipGetLastError();
}

}  // namespace rf
