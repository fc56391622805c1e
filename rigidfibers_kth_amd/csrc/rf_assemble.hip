// rf_assemble.hip -- pairwise assembly of the rigid-fiber linear system on
// gfx950.
//
// For every ordered pair (target fiber i, source fiber j != i) the kernel
// computes the outer integrals
//     Theta^{ij}_{kl} = sum_p w_p P_k(s_p) G_l(x_i + s_p t_i),  k,l = 0..M,
// where G_l is the inner integral over fiber j of the Stokeslet+doublet
// kernel times P_l (3x3 symmetric, 6 components):
//   analytic: fortran/Int_analytical.f90:5-293,663-767 (moments I,J,S with
//             forward recurrence for c<10, backward from n=27 otherwise);
//   numeric : fortran/quadrature.f90:100-164 (LQ-point Gauss quadrature).
// From Theta it writes
//   * A (column-major): rows (i,k,a), k=1..M, cols (j,l,b), l=1..M,
//       k=1: D1 t_a (Theta_kl t)_b ;  k>=2: gamma_k (Theta_kl,ab - E_k t_a (Theta_kl t)_b)
//     (fortran/matrix_assembly.f90:341-395), identity on the diagonal blocks;
//   * partial right-hand sides from Theta_{k0} f0_j
//     (fortran/matrix_assembly.f90:632-905), one slice per source split;
//   * the velocity operator W: rows (i, r in {V,Omega}, c), cols (j,l,c'),
//     W = Theta_{r l} (P_0 and P_1 outer weights of
//     fortran/coeffs_and_vels.f90:612-620,715-724), so the velocities of the
//     step are one GEMV with [F/2, a^1..a^M] per source fiber.
#include "rf_inner.h"
#include "rf_internal.h"

#include <algorithm>

namespace rf {
namespace {

// body(integral constant M)
template <typename F>
hipError_t with_terms(int M, F&& body)
{
    switch (M) {
    case 1: return body(std::integral_constant<int, 1>{});
    case 2: return body(std::integral_constant<int, 2>{});
    case 3: return body(std::integral_constant<int, 3>{});
    case 4: return body(std::integral_constant<int, 4>{});
    case 5: return body(std::integral_constant<int, 5>{});
    case 6: return body(std::integral_constant<int, 6>{});
    case 7: return body(std::integral_constant<int, 7>{});
    case 8: return body(std::integral_constant<int, 8>{});
    }
    return hipErrorInvalidValue;
}

// ---------------------------------------------------------------------------
// A wavefront (its own workgroup) owns up to kTW
// consecutive targets and a range of sources.  For a source it sorts the
// targets into near and far pairs (the operator's first far class: centres 4.2
// apart, 5.2 for M > 5, and not within 0.1 of the source's axis line) and takes
// as many pairs of a kind at a time as fill its lanes: a lane evaluates the
// outer points h and n-1-h of a pair.
//   * near: the closed-form moments at the n = LQ points;
//   * far: 11 Gauss nodes on the source, n = 14 outer nodes with the weights
//     that stand for the composite rule;
//   * numeric inner integrals: every pair is near, with the LQ-point rule on
//     the source.
// Each way the lane has G_l = al_l I + be_l V V^T + ga_l (t V^T + V t^T)
// + de_l t t^T, V = R0 or (numeric) its part across t.  Two l at a time the 6 components go to LDS as G(h) +- G(n-1-h)
// (P_k is even or odd, so each k needs one of the two: half the products), a
// lane per (pair, l, c) contracts them over h with weights in scalar registers,
// and a lane per (pair, l, k) writes the 9 entries of A, and of W for k = 0, 1.
// LDS is the wavefront's own, so nothing waits for another wavefront.
// What bounds it is instruction issue (59 % of cycles in the vector unit at two
// wavefronts a SIMD; without its stores it takes 1.29 of 1.41 ms), about 420
// vector instructions a pair where a thread per (target, point) with all pairs
// through the moments, LDS weights and three barriers took over twice that:
// N = 1000, M = 5 FP64 2.11 -> 1.41 ms, mixed 1.94 -> 1.19 ms; N = 4000 mixed
// 28.5 -> 15.3 ms; N = 421, M = 7 1.02 -> 0.50 ms.  Streaming (non-temporal)
// stores of the 24-byte pieces take 3.1 ms in FP64.
constexpr int kTW = 20;          // targets of a wavefront at most (20 fills 5 near or 9 far pairs at a time well)
constexpr int kFarPairs = 9;     // pairs at a time at most
constexpr int kGBuf = 12 * (2 * 64 + 4 * kFarPairs);  // doubles: 12 rows a pair of 2 H + 2..4

typedef const __attribute__((address_space(4))) double* const_ptr;  // uniform reads through the scalar cache

struct AKArgs {
    int N, n, LQ, targets, src_per_split, rhs_z_only;
    int64_t lda, ldw;
    double eps, D1, far_dist2;
    int far_n, far_q;
    double Ek[kMaxTerms + 1], gam[kMaxTerms + 1];
    const double* pos;
    const double* orient;
    const double* force;
    const double* near_node;  // [LQ]
    const double* far_node;   // [far_n]
    const double* near_w;     // [H][M+1]: w_p P_k(s_p) of the first half of the points
    const double* far_w;      // [H][M+1]
    const double* inner;      // [far_q][M+4]: s_q, w_q P_l(s_q) for l = 0..M+2
    const double* numeric;    // [LQ][M+2]: s_q, w_q P_l(s_q)
    void* A;
    void* W;
    double* bpart;
};

// al_l, be_l, ga_l, de_l at X from the moments (RB: see analytic_moments).
template <int M, typename RB>
__device__ __forceinline__ void near_coefficients(const double (&X)[3], const double* xj, const double* tj, double e2,
                                                  double e6, double (&co)[4][M + 1])
{
    Moments<M> mo;
    analytic_moments<M, RB, kByDistance, true>(X[0], X[1], X[2], xj, tj, mo);
#pragma unroll
    for (int l = 0; l <= M; ++l) {
        double L11 = 0, L12 = 0, L13 = 0, L14 = 0, L22 = 0, L23 = 0, L24 = 0;
#pragma unroll
        for (int m = 0; m <= M; ++m) {
            if (m <= l && kLeg[l][m] != 0.0) {
                const double cf = kLeg[l][m];
                L11 += cf * mo.I[m];
                L12 += cf * mo.J[m];
                L13 += cf * mo.J[m + 1];
                L14 += cf * mo.J[m + 2];
                L22 += cf * mo.S[m];
                L23 += cf * mo.S[m + 1];
                L24 += cf * mo.S[m + 2];
            }
        }
        co[0][l] = L11 + e2 * L12;
        co[1][l] = L12 - e6 * L22;
        co[2][l] = e6 * L23 - L13;
        co[3][l] = L14 - e6 * L24;
    }
}

// The same by quadrature over the source: sums of the kernel with P_l, the
// factors -s and s^2 of ga and de by the recurrence of s P_l.
template <int M>
__device__ __forceinline__ void far_coefficients(const double (&R0)[3], const double* tj, double e2, double e6, int Q,
                                                 const_ptr inner, double (&co)[4][M + 1])
{
    const double b = -2.0 * (tj[0] * R0[0] + tj[1] * R0[1] + tj[2] * R0[2]);
    const double c = R0[0] * R0[0] + R0[1] * R0[1] + R0[2] * R0[2];
    double be[M + 3], s1[M + 2];
#pragma unroll
    for (int l = 0; l <= M; ++l) co[0][l] = 0.0;
#pragma unroll
    for (int l = 0; l < M + 3; ++l) be[l] = 0.0;
    for (int q = 0; q < Q; ++q) {
        const_ptr row = inner + q * (M + 4);
        const double s = row[0];
        const double x = fma(s, b + s, c);  // |R|^2
        const double y = __builtin_amdgcn_rsq(x);
        const double e = fma(-x * y, y, 1.0);
        const double inv = fma(y * e, fma(e, 0.375, 0.5), y);  // 1/|R|: the estimate and a third-order step
        const double inv2 = inv * inv, inv3 = inv2 * inv;
        const double dg = inv + e2 * inv3, of = inv3 - e6 * inv3 * inv2;
#pragma unroll
        for (int l = 0; l < M + 3; ++l) {
            if (l <= M) co[0][l] += row[1 + l] * dg;
            be[l] += row[1 + l] * of;
        }
    }
#pragma unroll
    for (int l = 0; l < M + 2; ++l) s1[l] = ((l + 1) * be[l + 1] + (l > 0 ? l * be[l > 0 ? l - 1 : 0] : 0.0)) * (1.0 / (2 * l + 1));
#pragma unroll
    for (int l = 0; l <= M; ++l) {
        co[1][l] = be[l];
        co[2][l] = -s1[l];
        co[3][l] = ((l + 1) * s1[l + 1] + (l > 0 ? l * s1[l > 0 ? l - 1 : 0] : 0.0)) * (1.0 / (2 * l + 1));
    }
}

// Numeric inner integrals (fortran/quadrature.f90:121-155) at two points:
// with R(s) = V + (h - s) t, |R|^2 = |V|^2 + (h - s)^2 keeps its relative
// accuracy where the fibers come close.  43 operations a point and node in
// place of 64 with the six components accumulated, and one read of the node's
// weights (scalar registers) for both points: N = 333, M = 5, LQ = 24 510 -> 203 us
// with the wavefront's other steps.
template <int M>
__device__ __forceinline__ void numeric_coefficients(double (&R1)[3], double (&R2)[3], const double* tj, double e2,
                                                     double e6, int LQ, const_ptr table, double (&c1)[4][M + 1],
                                                     double (&c2)[4][M + 1])
{
    double h[2], d[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        double(&R)[3] = p ? R2 : R1;
        h[p] = tj[0] * R[0] + tj[1] * R[1] + tj[2] * R[2];
#pragma unroll
        for (int x = 0; x < 3; ++x) R[x] -= h[p] * tj[x];
        d[p] = R[0] * R[0] + R[1] * R[1] + R[2] * R[2];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int l = 0; l <= M; ++l) c1[e][l] = c2[e][l] = 0.0;
    for (int q = 0; q < LQ; ++q) {
        const_ptr row = table + q * (M + 2);
        const double s = row[0];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            double(&co)[4][M + 1] = p ? c2 : c1;
            const double u = h[p] - s, x = fma(u, u, d[p]);
            const double y = __builtin_amdgcn_rsq(x);
            const double e = fma(-x * y, y, 1.0);
            const double inv = fma(y * e, fma(e, 0.375, 0.5), y);
            const double inv2 = inv * inv, inv3 = inv2 * inv;
            const double dg = inv + e2 * inv3, of = inv3 - e6 * inv3 * inv2;
            const double of1 = of * u, of2 = of1 * u;
#pragma unroll
            for (int l = 0; l <= M; ++l) {
                co[0][l] += row[1 + l] * dg;
                co[1][l] += row[1 + l] * of;
                co[2][l] += row[1 + l] * of1;
                co[3][l] += row[1 + l] * of2;
            }
        }
    }
}

// LDS written by some lanes of the wavefront is read by others
__device__ __forceinline__ void wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// three consecutive rows of a column
__device__ __forceinline__ void store3(double* p, double x, double y, double z)
{
    p[0] = x;
    p[1] = y;
    p[2] = z;
}
__device__ __forceinline__ void store3(float* p, double x, double y, double z)
{
    p[0] = (float)x;
    p[1] = (float)y;
    p[2] = (float)z;
}

template <int M, typename AT, bool NUMERIC>
__global__ void __launch_bounds__(64, 2) assemble_kernel(const AKArgs a)
{
    constexpr int NL = M + 1, NCH = (NL + 1) / 2;
    typedef double d2 __attribute__((ext_vector_type(2)));
    __shared__ __align__(16) double buf[kGBuf];  // G of a stage, then Theta of it
    __shared__ double rhs[kTW][3 * M];
    __shared__ double tgt[kTW][6];
    __shared__ double kc[NL][2];  // entry = kc[k][0] Theta_ab + kc[k][1] t_a (Theta t)_b
    __shared__ unsigned char list[2][32];
    const int lane = threadIdx.x, N = a.N;
    const int i0 = blockIdx.x * a.targets, T = min(a.targets, N - i0);
    const int jb = blockIdx.y * a.src_per_split, je = min(N, jb + a.src_per_split);
    const double e2 = 2.0 * a.eps * a.eps, e6 = 6.0 * a.eps * a.eps;
    AT* A = reinterpret_cast<AT*>(a.A);
    AT* W = reinterpret_cast<AT*>(a.W);
    const_ptr pos = (const_ptr)a.pos, orient = (const_ptr)a.orient, force = (const_ptr)a.force;
    const double* pos_v = a.pos;
    const double* orient_v = a.orient;
    for (int e = lane; e < kTW * 3 * M; e += 64) rhs[0][e] = 0.0;
    for (int e = lane; e < T * 3; e += 64) {
        tgt[e / 3][e % 3] = pos_v[3 * i0 + e];
        tgt[e / 3][3 + e % 3] = orient_v[3 * i0 + e];
    }
    if (lane < NL) {
        kc[lane][0] = (lane <= 1) ? 0.0 : a.gam[lane];
        kc[lane][1] = (lane == 1) ? a.D1 : -a.gam[lane] * a.Ek[lane];
    }
    // what the two kinds of pairs differ in: points, lanes and pairs at a time
    const int LQ = a.LQ, nn[2] = {LQ, a.far_n};
    const int H[2] = {(LQ + 1) / 2, (a.far_n + 1) / 2};
    const int pairs_max[2] = {min(kFarPairs, 64 / H[0]), min(kFarPairs, 64 / H[1])};
    int slot_of[2], h_of[2];
    double node1[2], node2[2];
    bool mid[2];
#pragma unroll
    for (int f = 0; f < 2; ++f) {
        slot_of[f] = lane / H[f];
        h_of[f] = lane - slot_of[f] * H[f];
        const double* node = f ? a.far_node : a.near_node;
        node1[f] = node[h_of[f]];
        node2[f] = node[nn[f] - 1 - h_of[f]];
        mid[f] = h_of[f] == nn[f] - 1 - h_of[f];
    }
    wave_fence();
    for (int j = jb; j < je; ++j) {
        const double xj[3] = {pos[3 * j], pos[3 * j + 1], pos[3 * j + 2]};
        const double tj[3] = {orient[3 * j], orient[3 * j + 1], orient[3 * j + 2]};
        int cls = -1;
        if (lane < T && i0 + lane != j) {
            const double* g = tgt[lane];
            const double dx = g[0] - xj[0], dy = g[1] - xj[1], dz = g[2] - xj[2];
            const double D2 = dx * dx + dy * dy + dz * dz;
            // least distance squared of the target segment from the source's axis line
            const double dl = dx * tj[0] + dy * tj[1] + dz * tj[2], tl = g[3] * tj[0] + g[4] * tj[1] + g[5] * tj[2];
            const double dt = dx * g[3] + dy * g[4] + dz * g[5];
            const double aq = 1.0 - tl * tl, bq = dt - dl * tl, cq = D2 - dl * dl;
            const double s = (aq > 1e-12) ? fmin(1.0, fmax(-1.0, -bq / aq)) : 0.0;
            cls = (!NUMERIC && D2 >= a.far_dist2 && cq + s * (2.0 * bq + s * aq) >= 1e-2) ? 1 : 0;
        }
        int count[2];
#pragma unroll
        for (int f = 0; f < 2; ++f) {
            const unsigned long long in = __ballot(cls == f);
            if (cls == f) list[f][__popcll(in & ((1ull << lane) - 1ull))] = (unsigned char)lane;
            count[f] = __popcll(in);
        }
        wave_fence();
        if (j >= i0 && j < i0 + T) {  // the diagonal block: the identity, and nothing of W
            for (int e = lane; e < 9 * M * M; e += 64) {
                const int col = e / (3 * M), row = e - col * (3 * M);
                A[((int64_t)j * 3 * M + col) * a.lda + (int64_t)j * 3 * M + row] = (AT)(row == col ? 1.0 : 0.0);
            }
            if (W)
                for (int e = lane; e < 18 * NL; e += 64)
                    W[((int64_t)j * 3 * NL + e / 6) * a.ldw + (int64_t)j * 6 + e % 6] = (AT)0.0;
        }
        for (int f = 0; f < (NUMERIC ? 1 : 2); ++f) {
            const int Hf = f ? H[1] : H[0];
            const int slot = f ? slot_of[1] : slot_of[0], h = f ? h_of[1] : h_of[0];
            const int stride = 2 * Hf + ((Hf & 1) ? 4 : 2);  // an odd number of 16-byte words
            const const_ptr wk = (const_ptr)(f ? a.far_w : a.near_w);
            const int most = f ? pairs_max[1] : pairs_max[0], total = f ? count[1] : count[0];
            for (int base = 0; base < total; base += most) {
                const int pairs = min(most, total - base);
                const bool on = slot < pairs;
                const double* g = tgt[list[f][base + (on ? slot : 0)]];
                const double s1 = f ? node1[1] : node1[0], s2 = f ? node2[1] : node2[0];
                const double X1[3] = {g[0] + s1 * g[3], g[1] + s1 * g[4], g[2] + s1 * g[5]};
                const double X2[3] = {g[0] + s2 * g[3], g[1] + s2 * g[4], g[2] + s2 * g[5]};
                double R1[3] = {X1[0] - xj[0], X1[1] - xj[1], X1[2] - xj[2]};
                double R2[3] = {X2[0] - xj[0], X2[1] - xj[1], X2[2] - xj[2]};
                double c1[4][NL], c2[4][NL];
                if constexpr (NUMERIC) {
                    numeric_coefficients<M>(R1, R2, tj, e2, e6, LQ, (const_ptr)a.numeric, c1, c2);
                } else if (f == 0) {
                    near_coefficients<M, AT>(X1, xj, tj, e2, e6, c1);
                    near_coefficients<M, AT>(X2, xj, tj, e2, e6, c2);
                } else {
                    far_coefficients<M>(R1, tj, e2, e6, a.far_q, (const_ptr)a.inner, c1);
                    far_coefficients<M>(R2, tj, e2, e6, a.far_q, (const_ptr)a.inner, c2);
                }
                if (f ? mid[1] : mid[0]) {  // the middle point is its own mirror image
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int l = 0; l < NL; ++l) c2[e][l] = 0.0;
                }
#pragma unroll
                for (int ch = 0; ch < NCH; ++ch) {
                    // G(h) +- G(n-1-h) of two l, G = al I + (be R + ga t) R^T + (ga R + de t) t^T
                    if (on) {
#pragma unroll
                        for (int li = 0; li < 2; ++li) {
                            const int l = 2 * ch + li;
                            if (l > M) continue;
                            double u1[3], v1[3], u2[3], v2[3];
#pragma unroll
                            for (int x = 0; x < 3; ++x) {
                                u1[x] = c1[1][l] * R1[x] + c1[2][l] * tj[x];
                                v1[x] = c1[2][l] * R1[x] + c1[3][l] * tj[x];
                                u2[x] = c2[1][l] * R2[x] + c2[2][l] * tj[x];
                                v2[x] = c2[2][l] * R2[x] + c2[3][l] * tj[x];
                            }
#pragma unroll
                            for (int c = 0; c < 6; ++c) {
                                const int x = c < 3 ? c : c == 5 ? 1 : 0, y = c < 3 ? c : c == 3 ? 1 : 2;
                                const double g1 = u1[x] * R1[y] + (v1[x] * tj[y] + (c < 3 ? c1[0][l] : 0.0));
                                const double g2 = u2[x] * R2[y] + (v2[x] * tj[y] + (c < 3 ? c2[0][l] : 0.0));
                                d2 v;
                                v[0] = g1 + g2;
                                v[1] = g1 - g2;
                                *reinterpret_cast<d2*>(&buf[((slot * 2 + li) * 6 + c) * stride + 2 * h]) = v;
                            }
                        }
                    }
                    wave_fence();
                    // Theta_k of (pair, l, c): even k from the sums, odd k from the differences
                    double acc[2][NL];
                    const int rows = pairs * 12;
#pragma unroll
                    for (int r = 0; r < 2; ++r) {
                        if (64 * r >= rows) break;
                        const double* gr = &buf[min(lane + 64 * r, rows - 1) * stride];
#pragma unroll
                        for (int k = 0; k < NL; ++k) acc[r][k] = 0.0;
#pragma unroll 4
                        for (int p = 0; p < Hf; ++p) {
                            const d2 v = *reinterpret_cast<const d2*>(&gr[2 * p]);
#pragma unroll
                            for (int k = 0; k < NL; ++k) acc[r][k] += wk[p * NL + k] * v[k & 1];
                        }
                    }
                    wave_fence();
#pragma unroll
                    for (int r = 0; r < 2; ++r) {
                        const int task = lane + 64 * r;
                        if (task < rows) {
#pragma unroll
                            for (int k = 0; k < NL; ++k) buf[((task / 6) * NL + k) * 6 + task % 6] = acc[r][k];
                        }
                    }
                    wave_fence();
                    // entries of (l, pair, k)
                    for (int task = lane; task < 2 * pairs * NL; task += 64) {
                        const int half = task >= pairs * NL;
                        const int rem = task - half * pairs * NL, sl = rem / NL, k = rem - sl * NL;
                        const int l = 2 * ch + half;
                        if (l > M) continue;
                        const double* th = &buf[((sl * 2 + half) * NL + k) * 6];
                        double t6[6];
#pragma unroll
                        for (int c = 0; c < 6; ++c) t6[c] = th[c];
                        const int t = list[f][base + sl];
                        const int64_t i = i0 + t;
                        const double tx = tgt[t][3], ty = tgt[t][4], tz = tgt[t][5];
                        if (k >= 1) {
                            const double p0 = kc[k][0], p1 = kc[k][1];
                            if (l >= 1) {
                                AT* Ac = A + ((int64_t)j * 3 * M + (l - 1) * 3) * a.lda + i * 3 * M + 3 * (k - 1);
#pragma unroll
                                for (int b = 0; b < 3; ++b) {
                                    const double q = p1 * (t6[sym6(b, 0)] * tx + t6[sym6(b, 1)] * ty + t6[sym6(b, 2)] * tz);
                                    store3(Ac + b * a.lda, p0 * t6[sym6(0, b)] + q * tx, p0 * t6[sym6(1, b)] + q * ty,
                                           p0 * t6[sym6(2, b)] + q * tz);
                                }
                            } else {  // the force term: Theta_k0 f0_j
                                const double F0 = a.rhs_z_only ? 0.0 : 0.5 * force[3 * j];
                                const double F1 = a.rhs_z_only ? 0.0 : 0.5 * force[3 * j + 1];
                                const double F2 = 0.5 * force[3 * j + 2];
                                const double r0 = t6[0] * F0 + t6[3] * F1 + t6[4] * F2;
                                const double r1 = t6[3] * F0 + t6[1] * F1 + t6[5] * F2;
                                const double r2 = t6[4] * F0 + t6[5] * F1 + t6[2] * F2;
                                const double q = p1 * (tx * r0 + ty * r1 + tz * r2);
                                double* b = &rhs[t][3 * (k - 1)];
                                b[0] -= p0 * r0 + q * tx;
                                b[1] -= p0 * r1 + q * ty;
                                b[2] -= p0 * r2 + q * tz;
                            }
                        }
                        if (k < 2 && W) {
                            AT* Wc = W + ((int64_t)j * 3 * NL + l * 3) * a.ldw + i * 6 + 3 * k;
#pragma unroll
                            for (int b = 0; b < 3; ++b)
                                store3(Wc + b * a.ldw, t6[sym6(0, b)], t6[sym6(1, b)], t6[sym6(2, b)]);
                        }
                    }
                    wave_fence();
                }
            }
        }
    }
    wave_fence();
    for (int e = lane; e < T * 3 * M; e += 64)
        a.bpart[(size_t)blockIdx.y * a.n + (size_t)i0 * 3 * M + e] = rhs[0][e];
}

}  // namespace

int assemble_targets(int N)
{
    // fewer where the pairs are too few for two fillings of all wavefronts (N = 100: 54 -> 29 us)
    return 5 * (int)std::min<int64_t>(kTW / 5, std::max<int64_t>(1, (int64_t)N * N / (5 * 2 * 2048)));
}

hipError_t launch_assemble(const Tables& t, const AssembleArgs& a, hipStream_t s)
{
    AKArgs k;
    k.N = a.N;
    k.n = a.n;
    k.LQ = t.LQ;
    k.targets = assemble_targets(a.N);
    k.src_per_split = (a.N + a.splits - 1) / a.splits;
    k.rhs_z_only = a.analytic ? a.rhs_z_only : 0;
    k.lda = a.lda;
    k.ldw = a.ldw;
    k.eps = t.eps;
    k.D1 = t.D1;
    k.far_dist2 = t.fc[0].dist2;
    k.far_n = t.fc[0].n;
    k.far_q = t.fc[0].q;
    for (int i = 0; i <= kMaxTerms; ++i) {
        k.Ek[i] = t.Ek[i];
        k.gam[i] = t.gammak[i];
    }
    k.pos = a.pos;
    k.orient = a.orient;
    k.force = a.force;
    k.near_node = a.pv;
    k.far_node = a.far + t.fc[0].node;
    k.near_w = a.far + t.asm_near;
    k.far_w = a.far + t.asm_far;
    k.inner = a.far + t.asm_inner;
    k.numeric = a.far + t.asm_numeric;
    k.A = a.A;
    k.W = a.W;
    k.bpart = a.bpart;
    const dim3 grid((a.N + k.targets - 1) / k.targets, a.splits);
    auto launch = [&](auto mm) {
        constexpr int MM = decltype(mm)::value;
        if (a.analytic && a.mixed)
            hipLaunchKernelGGL((assemble_kernel<MM, float, false>), grid, dim3(64), 0, s, k);
        else if (a.analytic)
            hipLaunchKernelGGL((assemble_kernel<MM, double, false>), grid, dim3(64), 0, s, k);
        else if (a.mixed)
            hipLaunchKernelGGL((assemble_kernel<MM, float, true>), grid, dim3(64), 0, s, k);
        else
            hipLaunchKernelGGL((assemble_kernel<MM, double, true>), grid, dim3(64), 0, s, k);
        return hipGetLastError();
    };
    return with_terms(t.M, launch);
}

}  // namespace rf
