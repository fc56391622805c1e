// rf_linalg.hip -- HBM-bound vector kernels of the solver on gfx950:
// column-major GEMV (the GMRES matvec of fortran/coeffs_and_vels.f90:299,483
// and the velocity-operator product), deterministic multi-dot reductions and
// Gram-Schmidt updates of the Arnoldi basis.
//
// All arithmetic is FP64.  The matrix may be stored as double or float; the
// float case (mixed precision) halves the bytes streamed from HBM while the
// products and sums stay FP64.
#include "rf_internal.h"

#include <algorithm>

namespace rf {
namespace {

constexpr int kGemvThreads = 256;  // 4 wavefronts per workgroup
constexpr int kGemvUnroll = 8;     // columns in flight per wavefront

// 16-byte vectors of the matrix, read with non-temporal (streaming) loads:
// the matrix is read once per GEMV and should not evict the vectors.
typedef double d2v __attribute__((ext_vector_type(2)));
typedef float f4v __attribute__((ext_vector_type(4)));

template <typename T>
struct Vec16;
template <>
struct Vec16<double> {
    using type = d2v;
    static constexpr int n = 2;
};
template <>
struct Vec16<float> {
    using type = f4v;
    static constexpr int n = 4;
};

template <typename V, int N>
__device__ __forceinline__ void unpack(const V& v, double (&o)[N])
{
#pragma unroll
    for (int r = 0; r < N; ++r) o[r] = (double)v[r];
}

// parts[split][row] = sum_{c in split} A[row + c*ld] * x[c]
// Workgroup: 64*RPL consecutive rows x one column split.  Wavefront w of the
// workgroup takes columns c0+w, c0+w+4, ...; each lane loads 16 bytes (RPL
// rows) per column, so one wavefront load is a 1 KiB contiguous segment.
template <typename T>
__global__ void __launch_bounds__(kGemvThreads) gemv_parts_kernel(int cols, int64_t ld, const T* __restrict__ A,
                                                                  const double* __restrict__ x,
                                                                  double* __restrict__ parts, int64_t pstride,
                                                                  int cols_per_split)
{
    using V = typename Vec16<T>::type;
    constexpr int RPL = Vec16<T>::n;
    constexpr int ROWS = 64 * RPL;
    __shared__ double red[4][ROWS];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t row0 = (int64_t)blockIdx.x * ROWS + lane * RPL;
    const int c0 = blockIdx.y * cols_per_split;
    const int c1 = min(cols, c0 + cols_per_split);
    double acc[RPL];
#pragma unroll
    for (int r = 0; r < RPL; ++r) acc[r] = 0.0;
    const T* Ab = A + row0;
    int c = c0 + wave;
    for (; c + 4 * (kGemvUnroll - 1) < c1; c += 4 * kGemvUnroll) {
        V v[kGemvUnroll];
        double xv[kGemvUnroll];
#pragma unroll
        for (int u = 0; u < kGemvUnroll; ++u) {
            v[u] = __builtin_nontemporal_load(reinterpret_cast<const V*>(Ab + (int64_t)(c + 4 * u) * ld));
            xv[u] = x[c + 4 * u];
        }
#pragma unroll
        for (int u = 0; u < kGemvUnroll; ++u) {
            double e[RPL];
            unpack(v[u], e);
#pragma unroll
            for (int r = 0; r < RPL; ++r) acc[r] += e[r] * xv[u];
        }
    }
    for (; c < c1; c += 4) {
        const V v = __builtin_nontemporal_load(reinterpret_cast<const V*>(Ab + (int64_t)c * ld));
        const double xv = x[c];
        double e[RPL];
        unpack(v, e);
#pragma unroll
        for (int r = 0; r < RPL; ++r) acc[r] += e[r] * xv;
    }
#pragma unroll
    for (int r = 0; r < RPL; ++r) red[wave][lane * RPL + r] = acc[r];
    __syncthreads();
    for (int rr = threadIdx.x; rr < ROWS; rr += kGemvThreads) {
        const double s = (red[0][rr] + red[1][rr]) + (red[2][rr] + red[3][rr]);
        parts[(int64_t)blockIdx.y * pstride + (int64_t)blockIdx.x * ROWS + rr] = s;
    }
}

// y[i] = sum_s parts[s][i]  (mode 0)  or  b[i] - sum_s parts[s][i]  (mode 1).
// Eight lanes per row: lane q sums the splits q, q+8, ... (all its loads in
// flight together), and the eight partial sums meet in a fixed xor tree, so
// the result is deterministic.
constexpr int kSplitLanes = 8;

__global__ void reduce_splits_kernel(const double* __restrict__ parts, int splits, int64_t stride, int n,
                                     const double* __restrict__ b, int mode, double* __restrict__ y)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int i = (int)(t / kSplitLanes), q = (int)(t % kSplitLanes);
    double s = 0.0;
    if (i < n) {
        int k = q;
        for (; k + 3 * kSplitLanes < splits; k += 4 * kSplitLanes) {
            double v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = parts[(int64_t)(k + u * kSplitLanes) * stride + i];
#pragma unroll
            for (int u = 0; u < 4; ++u) s += v[u];
        }
        for (; k < splits; k += kSplitLanes) s += parts[(int64_t)k * stride + i];
    }
#pragma unroll
    for (int off = 1; off < kSplitLanes; off <<= 1) s += __shfl_xor(s, off, 64);
    if (q == 0 && i < n) y[i] = (mode == 1) ? b[i] - s : s;
}

constexpr int kDotThreads = 256;

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

__device__ __forceinline__ double block_sum(double v, double* sh)
{
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) sh[w] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0) {
        for (int k = 0; k < (int)(blockDim.x >> 6); ++k) s += sh[k];
    }
    __syncthreads();
    return s;  // valid in thread 0
}

// Block (bx, j): partial of dot(V[:,j], w) (j < k) or dot(w,w) (j == k) over a
// row chunk.  The last workgroup to finish sums the partials in a fixed order
// (deterministic) into out[0..k] and resets the counter.
__global__ void __launch_bounds__(kDotThreads) multidot_kernel(const double* __restrict__ V, int64_t ldv, int k,
                                                               const double* __restrict__ w, int n,
                                                               double* __restrict__ parts,
                                                               unsigned int* counter, double* __restrict__ out)
{
    __shared__ double sh[kDotThreads / 64];
    __shared__ bool last;
    const int j = blockIdx.y;
    const int nbx = gridDim.x;
    const double* a = (j < k) ? V + (int64_t)j * ldv : w;
    double s = 0.0;
    for (int i = blockIdx.x * kDotThreads + threadIdx.x; i < n; i += nbx * kDotThreads) s += a[i] * w[i];
    s = block_sum(s, sh);
    if (threadIdx.x == 0) {
        parts[(int64_t)j * nbx + blockIdx.x] = s;
        __threadfence();
        const unsigned int total = gridDim.x * gridDim.y;
        const unsigned int prev = atomicAdd(counter, 1u);
        last = (prev == total - 1);
    }
    __syncthreads();
    if (last) {
        __threadfence();
        for (int jj = threadIdx.x; jj <= k; jj += kDotThreads) {
            double t = 0.0;
            for (int b = 0; b < nbx; ++b)
                t += __hip_atomic_load(&parts[(int64_t)jj * nbx + b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            out[jj] = t;
        }
        if (threadIdx.x == 0) atomicExch(counter, 0u);
    }
}

// ---------------------------------------------------------------------------
// One Arnoldi step after the product (or the norm of a residual) in one launch:
//     w = sum of the product's column splits (or b minus it, or w as it is),
//     h1 = V^T w, w -= V h1, h2 = V^T w, w -= V h2, |w|^2, v_next = w / |w|,
// h1, h2 and |w|^2 to the host.  As separate kernels (split sums, dots, update
// with dots, update with norm, scaling) the step is up to five launches whose
// time is latency: 26 us of an iteration at n = 1500, 31 at n = 4995, 36 at
// n = 15000 and 72 at n = 60000; in one launch it is 8.7, 11.6, 13.3 and 28 us,
// bound by the three exchanges and, from a few rows a thread on, by the loads
// of V (n = 15000 with 16 workgroups and two rows a thread: 23 us).
//
// Up to 32 workgroups split the rows, each thread its own; the sums cross the
// workgroups three times.  A workgroup publishes its partial sums as they are,
// with agent-scope stores into slots that hold kEmpty until then, and reads
// those of all others in the same fixed order (so every workgroup computes the
// same bits): no counter, and no release fence, which would write a whole L2
// back.  A launch uses one of two sets of slots and empties its own slots of
// the other set for the next launch on the stream.
// The workgroups wait for each other, so all of them must be resident at once.
// Two fit a CU (128 registers), 512 the chip: the launches of 32 streams to
// n = 8192 (16 workgroups) and of 16 above, where a process has four hardware
// queues by default; any other kernel that holds a place ends
// by itself.  The wait is bounded all the same: after kSpinLimit polls a
// workgroup goes on with NaN and the host's words stay empty, which the host
// reports.  Those words are published like the slots, each by itself (the
// host empties them before the launch): a sequence word after them needs a
// system-scope fence that the whole step would wait for.
constexpr int kArnThreads = 512;
constexpr int kArnWaves = kArnThreads / 64;
constexpr int kArnMaxK = 64;             // basis vectors at most
constexpr int kArnBlocks = 32;           // workgroups at most (a power of two)
constexpr int kSpinLimit = 1 << 22;      // a few seconds
constexpr unsigned long long kEmpty = kArnoldiEmpty, kNaN = 0x7FF8000000000000ull;

struct ArnArgs {
    const double* parts;  // [splits][pstride]: w is their sum; null: w as it is
    int splits;
    int64_t pstride;
    const double* b;      // not null: w = b - the sum
    double* w;
    double* V;
    int64_t ldv;
    int k, n;
    double* v_next;       // w / |w|, or null
    unsigned long long* slots;  // [2][3][slot_rows][gridDim.x]
    int set, slot_rows;
    double* nrm_out;      // |w|^2 on the device
    unsigned long long* host;  // h1 at 0, h2 at ld_host, |w|^2 at 2 ld_host
    int ld_host;
};

// v of the lane across offset OFF (for 4: the lane mirrored within its eight,
// which differs in bit 2 too), by DPP.
template <int OFF>
__device__ __forceinline__ double dpp_across(double v)
{
    constexpr int ctrl = OFF == 1 ? 0xB1 : OFF == 2 ? 0x4E : OFF == 4 ? 0x141 : 0x128;
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), ctrl, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), ctrl, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
// OFF = 32, 16: a in the lanes below and b in those above, each summed over
// the pair of lanes, by the half (row) swap that exchanges both at once.
template <int OFF>
__device__ __forceinline__ double swap_sum(double a, double b)
{
    auto swap = [](unsigned x, unsigned y) {
        if constexpr (OFF == 32)
            return __builtin_amdgcn_permlane32_swap(x, y, false, false);
        else
            return __builtin_amdgcn_permlane16_swap(x, y, false, false);
    };
    const auto lo = swap((unsigned)__double2loint(a), (unsigned)__double2loint(b));
    const auto hi = swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b));
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
// a[0..CH) (CH = 16 or 32) summed over the wavefront; lane l ends with the sum
// of index arn_index<CH>(l) in a[0].  Each step halves the values a lane
// keeps; it stays in the vector unit (through LDS the 32 exchanges of two
// words by eight wavefronts took about 1 us a reduction).
template <int CH>
__device__ __forceinline__ int arn_index(int lane)
{
    int j = 0;
#pragma unroll
    for (int bit = 5, half = CH / 2; half >= 1; --bit, half /= 2) j += ((lane >> bit) & 1) * half;
    return j;
}
template <int CH, int HALF = CH / 2, int OFF = 32>
__device__ __forceinline__ void wave_sums(double (&a)[CH], int lane)
{
    if constexpr (OFF >= 16) {
#pragma unroll
        for (int u = 0; u < HALF; ++u) a[u] = swap_sum<OFF>(a[u], a[u + HALF]);
        wave_sums<CH, HALF / 2, OFF / 2>(a, lane);
    } else if constexpr (HALF >= 1) {
        const bool hi = (lane & OFF) != 0;
#pragma unroll
        for (int u = 0; u < HALF; ++u) {
            const double send = hi ? a[u] : a[u + HALF];
            const double keep = hi ? a[u + HALF] : a[u];
            a[u] = keep + dpp_across<OFF>(send);
        }
        wave_sums<CH, HALF / 2, OFF / 2>(a, lane);
    } else if constexpr (OFF >= 1) {
        a[0] += dpp_across<OFF>(a[0]);
        wave_sums<CH, 0, OFF / 2>(a, lane);
    }
}

struct ArnShared {
    double sh[kArnWaves][32];
    double h[2][kArnMaxK];
    double nrm;
    int late;  // a wait ran out
};

// The workgroup's sums of a[0..count) into slots [row0 + j][block].
template <int CH>
__device__ __forceinline__ void arn_publish(double (&a)[CH], int count, unsigned long long* slots, ArnShared& S)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    wave_sums<CH>(a, lane);
    if ((lane & (64 / CH - 1)) == 0) S.sh[wave][arn_index<CH>(lane)] = a[0];
    __syncthreads();
    if ((int)threadIdx.x < count) {
        double t = 0.0;
#pragma unroll
        for (int q = 0; q < kArnWaves; ++q) t += S.sh[q][threadIdx.x];
        unsigned long long bits = __double_as_longlong(t);
        if (bits == kEmpty) bits = kNaN;
        __hip_atomic_store(&slots[(size_t)threadIdx.x * gridDim.x + blockIdx.x], bits, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
}

// out[j] = the sum over all workgroups of slot row j, j < count.
__device__ __forceinline__ void arn_gather(int count, unsigned long long* slots, double* out, ArnShared& S)
{
    const int nb = gridDim.x;  // a power of two up to 32: a row's slots share a wavefront
    for (int e = threadIdx.x; e < count * nb; e += kArnThreads) {
        unsigned long long bits = kEmpty;
        for (int spin = 0; spin < kSpinLimit && bits == kEmpty; ++spin)
            bits = __hip_atomic_load(&slots[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (bits == kEmpty) S.late = 1;
        double v = __longlong_as_double(bits);
        if (nb > 1) v += dpp_across<1>(v);
        if (nb > 2) v += dpp_across<2>(v);
        if (nb > 4) v += dpp_across<4>(v);
        if (nb > 8) v += dpp_across<8>(v);
        if (nb > 16) v = swap_sum<16>(v, v);
        if (e % nb == 0) out[e / nb] = v;
    }
    __syncthreads();
}

// ONE: one row a thread and k <= 32: w and the thread's row of V stay in
// registers, V is read once.
template <bool ONE>
__global__ void __launch_bounds__(kArnThreads, 4) arnoldi_kernel(const ArnArgs a)
{
    constexpr int CH = ONE ? 32 : 16;  // basis vectors held at a time
    __shared__ ArnShared S;
    const int tid = threadIdx.x, nb = gridDim.x, k = a.k, n = a.n;
    const int step = nb * kArnThreads;
    const int first = blockIdx.x * kArnThreads + tid;
    const size_t set = (size_t)3 * a.slot_rows * nb;
    unsigned long long* slots = a.slots + (size_t)a.set * set;
    unsigned long long* other = a.slots + (size_t)(1 - a.set) * set;
    for (int e = tid; e < 3 * a.slot_rows; e += kArnThreads)
        __hip_atomic_store(&other[(size_t)e * nb + blockIdx.x], kEmpty, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (tid == 0) S.late = 0;
    auto phase = [&](int ph, int row) { return slots + ((size_t)ph * a.slot_rows + row) * nb; };
    // w of rows i and i2 (the same row: once)
    auto product2 = [&](int i, int i2, double& w1, double& w2) {
        w1 = w2 = 0.0;
        if (!a.parts) return;
        for (int q = 0; q < a.splits; q += 16) {
            double p1[16], p2[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                const double* row = a.parts + (int64_t)min(q + u, a.splits - 1) * a.pstride;
                p1[u] = row[i];
                if constexpr (!ONE) p2[u] = row[i2];
            }
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                w1 += (q + u < a.splits) ? p1[u] : 0.0;
                if constexpr (!ONE) w2 += (q + u < a.splits) ? p2[u] : 0.0;
            }
        }
        if (a.b) {
            w1 = a.b[i] - w1;
            w2 = a.b[i2] - w2;
        }
    };
    // columns c0.. of V at row i; past the last vector, the last one again
    auto load = [&](int i, int c0, double (&v)[CH]) {
#pragma unroll
        for (int g = 0; g < CH; g += 8) {
#pragma unroll
            for (int u = 0; u < 8; ++u) v[g + u] = 0.0;
            if (c0 + g < k) {
#pragma unroll
                for (int u = 0; u < 8; ++u) v[g + u] = a.V[(int64_t)min(c0 + g + u, k - 1) * a.ldv + i];
            }
        }
    };
    auto subtract = [&](double w, const double (&v)[CH], const double* h) {
#pragma unroll
        for (int g = 0; g < CH; ++g) w -= v[g] * h[g];
        return w;
    };
    if (tid < kArnMaxK) S.h[0][tid] = S.h[1][tid] = 0.0;  // zero past k
    double w = 0.0, v[CH], acc[CH];
    auto clear = [&] {
#pragma unroll
        for (int j = 0; j < CH; ++j) acc[j] = 0.0;
    };
    if constexpr (ONE) {
        const int i = min(first, n - 1);
        if (k > 0) load(i, 0, v);
        double same;
        if (a.parts)
            product2(i, i, w, same);
        else
            w = a.w[i];
        if (first >= n) w = 0.0;
        if (k == 0 && a.parts && first < n) a.w[i] = w;
        for (int ph = 0; ph < 2 && k > 0; ++ph) {
#pragma unroll
            for (int j = 0; j < CH; ++j) acc[j] = v[j] * w;
            arn_publish(acc, k, phase(ph, 0), S);
            arn_gather(k, phase(ph, 0), S.h[ph], S);
            w = (first < n) ? subtract(w, v, S.h[ph]) : 0.0;
        }
        clear();
        acc[0] = w * w;
    } else {
        // two rows at a time: i and i + step (past the end, row i again with w = 0)
        double v2[CH], w2 = 0.0;
        auto rows = [&](auto body) {
            for (int i = first; i < n; i += 2 * step) body(i, i + step < n ? i + step : i, i + step < n);
        };
        auto load2 = [&](int i, int i2, bool two) {
            w = a.w[i];
            w2 = two ? a.w[i2] : 0.0;
        };
        auto store2 = [&](int i, int i2, bool two) {
            a.w[i] = w;
            if (two) a.w[i2] = w2;
        };
        rows([&](int i, int i2, bool two) {
            product2(i, i2, w, w2);
            if (a.parts) store2(i, i2, two);
        });
        for (int ph = 0; ph < 2 && k > 0; ++ph) {
            for (int c0 = 0; c0 < k; c0 += CH) {
                clear();
                rows([&](int i, int i2, bool two) {
                    load(i, c0, v);
                    load(i2, c0, v2);
                    load2(i, i2, two);
                    if (ph == 1 && k <= CH) {  // the update with its dots
                        w = subtract(w, v, S.h[0]);
                        w2 = two ? subtract(w2, v2, S.h[0]) : 0.0;
                        store2(i, i2, two);
                    }
#pragma unroll
                    for (int j = 0; j < CH; ++j) acc[j] += v[j] * w + v2[j] * w2;
                });
                arn_publish(acc, min(CH, k - c0), phase(ph, c0), S);
            }
            arn_gather(k, phase(ph, 0), S.h[ph], S);
            if (ph == 0 && k <= CH) continue;
            clear();
            rows([&](int i, int i2, bool two) {
                load2(i, i2, two);
                for (int c0 = 0; c0 < k; c0 += CH) {
                    load(i, c0, v);
                    load(i2, c0, v2);
                    w = subtract(w, v, S.h[ph] + c0);
                    w2 = subtract(w2, v2, S.h[ph] + c0);
                }
                if (!two) w2 = 0.0;
                store2(i, i2, two);
                acc[0] += w * w + w2 * w2;
            });
        }
        if (k == 0) {
            clear();
            rows([&](int i, int i2, bool two) {
                load2(i, i2, two);
                acc[0] += w * w + w2 * w2;
            });
        }
    }
    arn_publish(acc, 1, phase(2, 0), S);
    arn_gather(1, phase(2, 0), &S.nrm, S);
    const double nrm = S.nrm;
    if (blockIdx.x == 0) {
        if (tid == 0) *a.nrm_out = nrm;
        auto send = [&](int at, double v) {
            unsigned long long bits = __double_as_longlong(v);
            if (bits == kEmpty) bits = kNaN;
            __hip_atomic_store(&a.host[at], bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        };
        if (!S.late) {
            if (tid < k) {
                send(tid, S.h[0][tid]);
                send(a.ld_host + tid, S.h[1][tid]);
            }
            if (tid == 0) send(2 * a.ld_host, nrm);
        }
    }
    if (a.v_next) {
        const double inv = 1.0 / sqrt(nrm);
        if constexpr (ONE) {
            if (first < n) a.v_next[first] = w * inv;
        } else {
            for (int i = first; i < n; i += step) a.v_next[i] = a.w[i] * inv;
        }
    }
}

__global__ void fill_slots_kernel(unsigned long long* slots, int count)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) slots[i] = kEmpty;
}

// v = w / sqrt(nrm2[idx])
__global__ void scale_copy_kernel(const double* __restrict__ w, const double* __restrict__ nrm2, int idx, int n,
                                  double* __restrict__ v)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double inv = 1.0 / sqrt(nrm2[idx]);
    v[i] = w[i] * inv;
}

// xc = x + V[:, :k] y with y passed by value (the host's least-squares
// solution: a host-to-device copy before the launch would stall the queue)
constexpr int kYArg = 64;
struct YArg {
    double v[kYArg];
};

__global__ void vy_plus_x_kernel(const double* __restrict__ V, int64_t ldv, int k, YArg y, const double* x, int n,
                                 double* xc)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double s = 0.0;
    for (int j = 0; j < k; ++j) s += V[(int64_t)j * ldv + i] * y.v[j];
    xc[i] = x ? x[i] + s : s;
}

__global__ void copy_vec_kernel(const double* __restrict__ src, double* __restrict__ dst, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

__global__ void copy_kernel(const double4* __restrict__ src, double4* __restrict__ dst, size_t n4)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += (size_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

__global__ void f64_to_f32_kernel(const double* __restrict__ src, float* __restrict__ dst, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        dst[i] = (float)src[i];
}

// A few words into coherent pinned host memory, by one workgroup: the
// runtime's device-to-host copy ends with a system-scope release that stalls
// the queue ~15 us, once per GMRES iteration.
// With seq_word, the copy ends with `seq` stored there at system scope after
// every thread's data stores have been fenced at system scope, so a host that
// reads the expected sequence number reads the data of this copy.
__global__ void to_host_kernel(const unsigned* __restrict__ src, unsigned* dst, int words, unsigned* seq_word,
                               unsigned seq)
{
    for (int i = threadIdx.x; i < words; i += blockDim.x) dst[i] = src[i];
    if (seq_word) {
        __threadfence_system();
        __syncthreads();
        if (threadIdx.x == 0) __hip_atomic_store(seq_word, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

}  // namespace

hipError_t launch_to_host(const void* src, void* host_dst, size_t bytes, hipStream_t s, unsigned* host_seq_word,
                          unsigned seq)
{
    if (bytes % sizeof(unsigned) != 0 || bytes > 64 * 1024) return hipErrorInvalidValue;
    hipLaunchKernelGGL(to_host_kernel, dim3(1), dim3(256), 0, s, static_cast<const unsigned*>(src),
                       static_cast<unsigned*>(host_dst), (int)(bytes / sizeof(unsigned)), host_seq_word, seq);
    return hipGetLastError();
}

hipError_t launch_f64_to_f32(const double* src, float* dst, size_t n, hipStream_t s)
{
    const size_t blocks = std::min<size_t>((n + 255) / 256, 65536);
    hipLaunchKernelGGL(f64_to_f32_kernel, dim3((unsigned)blocks), dim3(256), 0, s, src, dst, n);
    return hipGetLastError();
}

hipError_t launch_copy(const void* src, void* dst, size_t bytes, hipStream_t s)
{
    const size_t n4 = bytes / sizeof(double4);
    hipLaunchKernelGGL(copy_kernel, dim3(4096), dim3(256), 0, s, static_cast<const double4*>(src),
                       static_cast<double4*>(dst), n4);
    return hipGetLastError();
}

GemvPlan plan_gemv(int rows, int cols, int64_t ld, int elem_bytes, int num_cus)
{
    GemvPlan p;
    p.rows = rows;
    p.cols = cols;
    p.ld = ld;
    p.elem_bytes = elem_bytes;
    const int rows_per_block = 64 * (16 / elem_bytes);
    p.row_blocks = (int)((ld + rows_per_block - 1) / rows_per_block);
    // about 24 workgroups per CU (measured best for n = 15000..60000 with
    // streaming loads), but keep >= 32 columns per wavefront
    const int target = std::max(1, num_cus) * 24;
    int splits = (target + p.row_blocks - 1) / p.row_blocks;
    splits = std::min(splits, std::max(1, cols / 128));
    p.splits = std::max(1, std::min(splits, 256));
    return p;
}

int64_t gemv_parts_stride(const GemvPlan& p)
{
    return (int64_t)p.row_blocks * 64 * (16 / p.elem_bytes);
}

size_t gemv_parts_elems(const GemvPlan& p)
{
    return (size_t)p.splits * (size_t)gemv_parts_stride(p);
}

hipError_t launch_gemv(const GemvPlan& p, const void* A, const double* x, double* parts, double* y, const double* b,
                       int mode, hipStream_t s, hipEvent_t ev0, hipEvent_t ev1)
{
    const int rows_per_block = 64 * (16 / p.elem_bytes);
    if (p.ld % rows_per_block != 0) return hipErrorInvalidValue;  // loads assume whole row blocks
    const int64_t pstride = gemv_parts_stride(p);
    const int cps = (p.cols + p.splits - 1) / p.splits;
    dim3 grid(p.row_blocks, p.splits);
    if (ev0) {
        hipError_t e0 = hipEventRecord(ev0, s);
        if (e0 != hipSuccess) return e0;
    }
    if (p.elem_bytes == 8)
        hipLaunchKernelGGL(gemv_parts_kernel<double>, grid, dim3(kGemvThreads), 0, s, p.cols, p.ld,
                           static_cast<const double*>(A), x, parts, pstride, cps);
    else
        hipLaunchKernelGGL(gemv_parts_kernel<float>, grid, dim3(kGemvThreads), 0, s, p.cols, p.ld,
                           static_cast<const float*>(A), x, parts, pstride, cps);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (ev1) {
        e = hipEventRecord(ev1, s);
        if (e != hipSuccess) return e;
    }
    if (!y) return hipSuccess;  // the partial sums are what the caller wants
    hipLaunchKernelGGL(reduce_splits_kernel, dim3((p.rows * kSplitLanes + 255) / 256), dim3(256), 0, s, parts,
                       p.splits, pstride, p.rows, b, mode, y);
    return hipGetLastError();
}

hipError_t launch_reduce_splits(const double* parts, int splits, int64_t stride, int n, double* out, hipStream_t s)
{
    hipLaunchKernelGGL(reduce_splits_kernel, dim3((n * kSplitLanes + 255) / 256), dim3(256), 0, s, parts, splits,
                       stride, n, nullptr, 0, out);
    return hipGetLastError();
}

int multidot_blocks(int n)
{
    return std::max(1, std::min(kMaxDotBlocks, (n + 4 * kDotThreads - 1) / (4 * kDotThreads)));
}

hipError_t launch_multidot(const double* V, int64_t ldv, int k, const double* w, int n, double* parts,
                           unsigned int* counter, double* out, hipStream_t s)
{
    dim3 grid(multidot_blocks(n), k + 1);
    hipLaunchKernelGGL(multidot_kernel, grid, dim3(kDotThreads), 0, s, V, ldv, k, w, n, parts, counter, out);
    return hipGetLastError();
}

// workgroups of an n-row step: one row a thread as far as 32 go
static int arnoldi_blocks(int n)
{
    int nb = 1;
    while (nb < kArnBlocks && nb * kArnThreads < n) nb *= 2;
    return nb;
}

size_t arnoldi_slots(int max_k)
{
    return (size_t)2 * 3 * std::max(1, max_k) * kArnBlocks;
}

hipError_t launch_arnoldi_init(unsigned long long* slots, int max_k, hipStream_t s)
{
    const int count = (int)arnoldi_slots(max_k);
    hipLaunchKernelGGL(fill_slots_kernel, dim3((count + 255) / 256), dim3(256), 0, s, slots, count);
    return hipGetLastError();
}

hipError_t launch_arnoldi(const ArnoldiStep& st, hipStream_t s)
{
    if (st.n < 1 || st.k < 0 || st.k > st.max_k || st.max_k > kArnMaxK || !st.w || !st.slots || !st.host ||
        !st.nrm_out)
        return hipErrorInvalidValue;
    ArnArgs a;
    a.parts = st.product ? st.parts : nullptr;
    a.splits = st.product ? st.product->splits : 0;
    a.pstride = st.product ? gemv_parts_stride(*st.product) : 0;
    a.b = st.b;
    a.w = st.w;
    a.V = st.V;
    a.ldv = st.ldv;
    a.k = st.k;
    a.n = st.n;
    a.v_next = st.v_next;
    a.slots = st.slots;
    a.set = st.set & 1;
    a.slot_rows = std::max(1, st.max_k);
    a.nrm_out = st.nrm_out;
    a.host = st.host;
    a.ld_host = st.ld_host;
    const int nb = arnoldi_blocks(st.n);
    if (st.n <= nb * kArnThreads && st.k <= 32)
        hipLaunchKernelGGL(arnoldi_kernel<true>, dim3(nb), dim3(kArnThreads), 0, s, a);
    else
        hipLaunchKernelGGL(arnoldi_kernel<false>, dim3(nb), dim3(kArnThreads), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_scale_copy(const double* w, const double* nrm2, int idx, int n, double* v, hipStream_t s)
{
    hipLaunchKernelGGL(scale_copy_kernel, dim3((n + 255) / 256), dim3(256), 0, s, w, nrm2, idx, n, v);
    return hipGetLastError();
}

hipError_t launch_vy_plus_x(const double* V, int64_t ldv, int k, const double* y_host, const double* x, int n,
                            double* xc, hipStream_t s)
{
    for (int c = 0; c < k || c == 0; c += kYArg) {  // chunks of 64 basis vectors
        YArg y{};
        const int kc = std::min(kYArg, k - c);
        for (int j = 0; j < kc; ++j) y.v[j] = y_host[c + j];
        hipLaunchKernelGGL(vy_plus_x_kernel, dim3((n + 255) / 256), dim3(256), 0, s, V + (int64_t)c * ldv, ldv,
                           std::max(0, kc), y, c == 0 ? x : xc, n, xc);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        if (kc <= 0) break;
    }
    return hipSuccess;
}

hipError_t launch_copy_vec(const double* src, double* dst, int n, hipStream_t s)
{
    hipLaunchKernelGGL(copy_vec_kernel, dim3((n + 255) / 256), dim3(256), 0, s, src, dst, n);
    return hipGetLastError();
}

}  // namespace rf
