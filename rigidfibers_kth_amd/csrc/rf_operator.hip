// rf_operator.hip -- the matrix-free FP64 operator of the fiber system on
// gfx950: y = A x, the right-hand side b, the residual b - A x and the
// velocity sums, without storing A or W.
//
// mat_prod of fortran/matrix_assembly.f90:159-265 (numeric inner integrals
// G_f_GQ, fortran/quadrature.f90:166-223), extended to the analytic inner
// integrals (fortran/Int_analytical.f90:5-293,663-767) and to the force term
// of the right-hand side (fortran/matrix_assembly.f90:632-905) and of the
// velocities (fortran/coeffs_and_vels.f90:543-746).
//
// For target fiber i and Legendre index k = 0..M the kernel forms
//     IF_k(i) = sum_{j != i} sum_p w_p P_k(s_p) g_j(x_i + s_p t_i),
//     g_j(X)  = sum_{l=0..M} G_l(X; j) a_{j,l},
// the inner integral over fiber j of the kernel times j's force density
// f_j(s) = sum_l a_{j,l} P_l(s) (a_{j,0} = F_j/2 or 0, a_{j,l} = the
// coefficients x).  Both sums are linear, so thread (target i, point p) adds
// g_j(x_i + s_p t_i) over all sources j in three registers, and the
// contraction over p with w_p P_k happens once per target at the end.
// Sources are read with wavefront-uniform addresses (scalar loads).
//
// Analytic: G_l = al_l I + be_l R R^T + ga_l (t R^T + R t^T) + de_l t t^T with
// al_l, ..., de_l Legendre combinations of the moments I_m, J_m, S_m.  Moving
// the Legendre coefficients onto the source vector (c_m = sum_l C[l][m] a_l,
// the monomial coefficients of f_j) gives
//     g = sum_m (I_m + 2e^2 J_m) c_m + q sum_m [be_m (q.c_m) + gq_m (t.c_m)]
//                                    + t sum_m [gq_m (q.c_m) + dq_m (t.c_m)],
// q = R - h t, h = t.R, be_m = J_m - 6e^2 S_m, ga_m = 6e^2 S_{m+1} - J_{m+1},
// gq_m = h be_m + ga_m, dq_m = h (gq_m + ga_m) + J_{m+2} - 6e^2 S_{m+2}:
// about 35 flops per m on top of the moments.
// Numeric: g = sum_q [ (1/|R| + 2e^2/|R|^3) f_q + (1/|R|^3 - 6e^2/|R|^5) R (R.f_q) ],
// R = X - x_j - s_q t_j, f_q = w_q f_j(s_q).
//
// Analytic far pairs.  A pair whose centres are more than about four apart is
// smooth on both fibers: 8 to 10 Gauss nodes give its inner integrals and 10
// to 14 outer nodes carry the LQ-point outer rule (Tables::FarClass), about
// 110 kernel evaluations of 30 operations in place of 24 moment evaluations
// of 700 (two logarithms, square roots, divisions, 26-step recurrences).
// Near pairs keep the moments, and so does a far pair whose target comes
// within 0.1 of the source's axis line: there the closed forms cancel
// (1/d, d the distance squared from the axis) and their rounding, which this
// path does not share, would show.
#include "rf_inner.h"
#include "rf_internal.h"
#include "rigidfibers.h"

#include <algorithm>
#include <mutex>
#include <string>

namespace rf {
namespace {

struct OpKArgs {
    int N, LQ, T, src_per_split, src_stride;
    double eps;
    const double* pos;
    const double* orient;
    const double* src;  // per source fiber [LQ][4]
    const double* wp;   // [M+1][LQ] w_p P_k(s_p)
    const double* pv;   // [LQ]
    double* part;       // [splits][N][M+1][3]
};

// Inner nodes and weights of the far classes (Tables::far at tab; no nodes: none)
struct OpFarSources {
    int q[Tables::kFarClasses] = {0, 0, 0}, wP[Tables::kFarClasses] = {0, 0, 0};
    const double* tab = nullptr;
};

// Source vectors of the operator.  a_{j,0} (force term): mode 0 none; modes
// 1, 2 the right-hand side's F/2 (only F_z with analytic integrals,
// fortran/matrix_assembly.f90:857-859); mode 3 F/2.  a_{j,l}, l >= 1: the
// coefficients x (none in mode 2).  The host turns the mode into the masks
// fmask (force components on) and x_on.
__global__ void op_source_kernel(int N, int M, int LQ, int analytic, int fmask, int x_on,
                                 const double* __restrict__ force, const double* __restrict__ x,
                                 const double* __restrict__ orient, const double* __restrict__ wp,
                                 double* __restrict__ src, int stride, OpFarSources far)
{
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    const int per = analytic ? (M + 1) + far.q[0] + far.q[1] + far.q[2] : LQ;
    if (idx >= N * per) return;
    const int j = idx / per, r = idx - j * per;
    double a[kMaxTerms + 1][3];
#pragma unroll
    for (int c = 0; c < 3; ++c) a[0][c] = ((fmask >> c) & 1) ? 0.5 * force[3 * j + c] : 0.0;
    for (int l = 1; l <= M; ++l)
#pragma unroll
        for (int c = 0; c < 3; ++c) a[l][c] = x_on ? x[(size_t)j * 3 * M + (l - 1) * 3 + c] : 0.0;
    double v[3] = {0.0, 0.0, 0.0};
    if (analytic && r > M) {
        // w_q f_j(s_q) at node q of a far class
        int c = 0, q = r - (M + 1);
        while (q >= far.q[c]) q -= far.q[c++];
        for (int l = 0; l <= M; ++l) {
            const double w = far.tab[far.wP[c] + l * far.q[c] + q];
#pragma unroll
            for (int d = 0; d < 3; ++d) v[d] += w * a[l][d];
        }
        double* o = src + (size_t)j * stride + 4 * (M + 1) + 3 * (r - (M + 1));
        o[0] = v[0];
        o[1] = v[1];
        o[2] = v[2];
        return;
    }
    if (analytic) {
        // monomial coefficient m = r of f_j(s) = sum_l a_l P_l(s)
        for (int l = r; l <= M; ++l) {
            const double cf = kLeg[l][r];
#pragma unroll
            for (int c = 0; c < 3; ++c) v[c] += cf * a[l][c];
        }
    } else {
        // w_q f_j(s_q), q = r
        for (int l = 0; l <= M; ++l) {
            const double w = wp[l * LQ + r];
#pragma unroll
            for (int c = 0; c < 3; ++c) v[c] += w * a[l][c];
        }
    }
    double* o = src + (size_t)j * stride + 4 * r;
    o[0] = v[0];
    o[1] = v[1];
    o[2] = v[2];
    o[3] = analytic ? (orient[3 * j] * v[0] + orient[3 * j + 1] * v[1] + orient[3 * j + 2] * v[2]) : 0.0;
}

// Numeric inner integrals: thread (target, point), sources in turn.
template <int M>
__global__ void __launch_bounds__(512) operator_numeric_kernel(const OpKArgs a)
{
    constexpr int NL = M + 1;
    extern __shared__ double sg[];  // [T][LQ][3]
    const int T = a.T, LQ = a.LQ, N = a.N;
    const int tid = threadIdx.x;
    const int i0 = blockIdx.x * T;
    const int jb = blockIdx.y * a.src_per_split;
    const int je = min(N, jb + a.src_per_split);
    const double e2 = 2.0 * a.eps * a.eps, e6 = 6.0 * a.eps * a.eps;
    const int t1 = tid / LQ, p1 = tid - t1 * LQ;
    const int i1 = i0 + t1;
    const bool on = (t1 < T) && (i1 < N);
    double X0 = 0, X1 = 0, X2 = 0;
    if (on) {
        const double s = a.pv[p1];
        X0 = a.pos[3 * i1 + 0] + s * a.orient[3 * i1 + 0];
        X1 = a.pos[3 * i1 + 1] + s * a.orient[3 * i1 + 1];
        X2 = a.pos[3 * i1 + 2] + s * a.orient[3 * i1 + 2];
    }
    double g0 = 0.0, g1 = 0.0, g2 = 0.0;
    for (int j = jb; j < je; ++j) {
        if (!on || j == i1) continue;
        const double xj[3] = {a.pos[3 * j], a.pos[3 * j + 1], a.pos[3 * j + 2]};
        const double tj[3] = {a.orient[3 * j], a.orient[3 * j + 1], a.orient[3 * j + 2]};
        const double* cs = a.src + (size_t)j * a.src_stride;
        const double bx = X0 - xj[0], by = X1 - xj[1], bz = X2 - xj[2];
        double h0 = 0.0, h1 = 0.0, h2 = 0.0;
        for (int q = 0; q < LQ; ++q) {
            const double s = a.pv[q];
            const double fx = cs[4 * q], fy = cs[4 * q + 1], fz = cs[4 * q + 2];
            const double rx = bx - tj[0] * s, ry = by - tj[1] * s, rz = bz - tj[2] * s;
            const double r2 = rx * rx + ry * ry + rz * rz;
            const double inv = 1.0 / sqrt(r2);
            const double inv2 = inv * inv, inv3 = inv * inv2, inv5 = inv3 * inv2;
            const double dg = inv + e2 * inv3, of = inv3 - e6 * inv5;
            const double rf = of * (rx * fx + ry * fy + rz * fz);
            h0 += dg * fx + rf * rx;
            h1 += dg * fy + rf * ry;
            h2 += dg * fz + rf * rz;
        }
        g0 += h0;
        g1 += h1;
        g2 += h2;
    }
    if (t1 < T) {
        sg[(t1 * LQ + p1) * 3 + 0] = g0;
        sg[(t1 * LQ + p1) * 3 + 1] = g1;
        sg[(t1 * LQ + p1) * 3 + 2] = g2;
    }
    __syncthreads();
    // IF_k(i) partial of this source split: sum_p w_p P_k(s_p) g(p)
    for (int it = tid; it < T * NL * 3; it += blockDim.x) {
        const int t = it / (NL * 3), rem = it - t * (NL * 3);
        const int k = rem / 3, c = rem - k * 3;
        const int i = i0 + t;
        if (i >= N) continue;
        double acc = 0.0;
        for (int p = 0; p < LQ; ++p) acc += a.wp[k * LQ + p] * sg[(t * LQ + p) * 3 + c];
        a.part[((size_t)blockIdx.y * N + i) * (NL * 3) + rem] = acc;
    }
}

// g_j at the point (X0, X1, X2) from the moments; cs: the source's monomial
// vectors.  With R(s) = q + (h - s) t, q the part of R0 across t, the large
// near-contact terms (S ~ 1/d^2, |q|^2 = d) cancel in the coefficients, which
// are the same for every x, and not in the sums over c_m: on a state with
// fibers in near contact the FP64 residual of a solve, which rounding held at
// 1e-10 to 3e-10 of |b|, now falls to 4e-13.
template <int M, MomentBranch BRANCH>
__device__ __forceinline__ void analytic_g(double X0, double X1, double X2, const double* xj, const double* tj,
                                           const double* __restrict__ cs, double e2, double e6, double (&g)[3])
{
    Moments<M> mo;
    analytic_moments<M, double, BRANCH>(X0, X1, X2, xj, tj, mo);
    const double h = mo.r0x * tj[0] + mo.r0y * tj[1] + mo.r0z * tj[2];
    const double qx = mo.r0x - h * tj[0], qy = mo.r0y - h * tj[1], qz = mo.r0z - h * tj[2];
    double ax = 0.0, ay = 0.0, az = 0.0, sQ = 0.0, sT = 0.0;
#pragma unroll
    for (int m = 0; m <= M; ++m) {
        const double cx = cs[4 * m], cy = cs[4 * m + 1], cz = cs[4 * m + 2], tc = cs[4 * m + 3];
        const double al = mo.I[m] + e2 * mo.J[m];
        ax += al * cx;
        ay += al * cy;
        az += al * cz;
        const double qc = qx * cx + qy * cy + qz * cz;
        const double be = mo.J[m] - e6 * mo.S[m];
        const double ga = e6 * mo.S[m + 1] - mo.J[m + 1];
        const double de = mo.J[m + 2] - e6 * mo.S[m + 2];
        const double gq = h * be + ga, dq = h * (gq + ga) + de;
        sQ += be * qc + gq * tc;
        sT += gq * qc + dq * tc;
    }
    g[0] = ax + sQ * qx + sT * tj[0];
    g[1] = ay + sQ * qy + sT * tj[1];
    g[2] = az + sQ * qz + sT * tj[2];
}

// 1/sqrt(x) for ordinary positive x: the hardware estimate and one
// third-order (Halley) step.
__device__ __forceinline__ double inv_sqrt(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(e, 0.375, 0.5), y);
}

// g_j at K points X (R0 = X - x_j) by Q-point quadrature over the source: fq
// holds w_q f_j(s_q), read once for the K points.  |R|^2 is the closed forms'
// c + b s + s^2 (|t| = 1).
template <int Q, int K>
__device__ __forceinline__ void quadrature_g(const double (&r0)[K][3], const double* tj, const double* sq,
                                             const double* __restrict__ fq, double e2, double e6, double (&g)[K][3])
{
    double b[K], c[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        b[k] = -2.0 * (tj[0] * r0[k][0] + tj[1] * r0[k][1] + tj[2] * r0[k][2]);
        c[k] = r0[k][0] * r0[k][0] + r0[k][1] * r0[k][1] + r0[k][2] * r0[k][2];
        g[k][0] = g[k][1] = g[k][2] = 0.0;
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const double s = sq[q];
        const double fx = fq[3 * q], fy = fq[3 * q + 1], fz = fq[3 * q + 2];
        const double sx = s * tj[0], sy = s * tj[1], sz = s * tj[2];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const double rx = r0[k][0] - sx, ry = r0[k][1] - sy, rz = r0[k][2] - sz;
            const double inv = inv_sqrt(fma(s, b[k] + s, c[k]));
            const double inv2 = inv * inv, inv3 = inv2 * inv;
            const double dg = inv + e2 * inv3, of = inv3 - e6 * inv3 * inv2;
            const double rf = of * (rx * fx + ry * fy + rz * fz);
            g[k][0] += dg * fx + rf * rx;
            g[k][1] += dg * fy + rf * ry;
            g[k][2] += dg * fz + rf * rz;
        }
    }
}

// Analytic inner integrals.  A workgroup takes one target fiber and one split
// of the sources, a wavefront a quarter of the split.  Each wavefront first
// sorts its sources into the near list and the far classes (in LDS, in order:
// every sum is deterministic), then its lanes take the elements (source, outer
// node) of one list after the other, so all 64 lanes run the same path: with
// a thread per (target, point) and sources in turn, near and far neighbours
// shared a wavefront and both paths ran for all of it.  IF_k is accumulated
// per lane with the node's weights and summed over the workgroup at the end.
// FP64 vector work and the source vectors' loads bound it, at two wavefronts a
// SIMD (224 registers at M = 5; a bound of three spills and is slower, and near
// and far pairs in kernels of their own, 168 and 108 registers, take longer
// together: 68 / 553 / 8015 us).  In a far class a lane takes two outer nodes,
// so a source vector is loaded once for both: 7037 us, one node a lane 8167.
// M = 5, LQ = 24, N = 250 / 1000 / 6000: 52 / 440 / 7100 us; a thread per
// (target, point) with every pair through the moments: 59 / 796 / 27062 us.
constexpr int kFarSplit = 2048;           // sources per workgroup at a time
constexpr int kFarWave = kFarSplit / 4;   // and per wavefront

struct FarKArgs {
    int N, LQ, src_per_split, src_stride, far_total, use_far;
    double eps, point_c;
    Tables::FarClass fc[Tables::kFarClasses];
    const double* pos;
    const double* orient;
    const double* src;  // [N][src_stride]: [M+1][4], then the classes' [q][3]
    const double* wp;   // [M+1][LQ]
    const double* pv;   // [LQ]
    const double* far;  // Tables::far
    double* part;       // [splits][N][M+1][3]
};

template <int M>
__global__ void __launch_bounds__(256, 2) operator_kernel(const FarKArgs a)
{
    constexpr int NL = M + 1, NC = Tables::kFarClasses;
    extern __shared__ double tab[];  // pv[LQ], wp[NL][LQ], far[far_total]
    __shared__ unsigned short list[4][NC + 1][kFarWave];
    __shared__ unsigned short queue[4][3][128];
    __shared__ double red[4][NL * 3];
    const int LQ = a.LQ, N = a.N;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = blockIdx.x;
    const double e2 = 2.0 * a.eps * a.eps, e6 = 6.0 * a.eps * a.eps;
    double* tpv = tab;
    double* twp = tab + LQ;
    double* tfar = twp + NL * LQ;
    for (int e = tid; e < LQ; e += 256) tpv[e] = a.pv[e];
    for (int e = tid; e < NL * LQ; e += 256) twp[e] = a.wp[e];
    for (int e = tid; e < a.far_total; e += 256) tfar[e] = a.far[e];
    const double x0 = a.pos[3 * i], x1 = a.pos[3 * i + 1], x2 = a.pos[3 * i + 2];
    const double t0 = a.orient[3 * i], t1 = a.orient[3 * i + 1], t2 = a.orient[3 * i + 2];
    constexpr double kUnit2 = 1.0 + 1e-6;
    const double tt = t0 * t0 + t1 * t1 + t2 * t2;
    const int split_end = min(N, (int)(blockIdx.y + 1) * a.src_per_split);
    double acc[NL * 3];
#pragma unroll
    for (int e = 0; e < NL * 3; ++e) acc[e] = 0.0;
    __syncthreads();  // the tables; the lists are each wavefront's own
    for (int sb = blockIdx.y * a.src_per_split; sb < split_end; sb += kFarSplit) {
        const int se = min(split_end, sb + kFarSplit);
        const int per = (se - sb + 3) / 4;
        const int jb = sb + wave * per, je = min(se, jb + per);
        // ---- lists: 0 near, 1 + c far class c ----
        int count[NC + 1] = {};
        for (int j0 = jb; j0 < je; j0 += 64) {
            const int j = j0 + lane;
            int cls = -1;
            if (j < je && j != i) {
                const double dx = x0 - a.pos[3 * j], dy = x1 - a.pos[3 * j + 1], dz = x2 - a.pos[3 * j + 2];
                const double ux = a.orient[3 * j], uy = a.orient[3 * j + 1], uz = a.orient[3 * j + 2];
                const double D2 = dx * dx + dy * dy + dz * dz;
                cls = 0;
                // (the classes hold for |t| = 1; a caller's longer vectors stay near)
                const bool unit = tt <= kUnit2 && ux * ux + uy * uy + uz * uz <= kUnit2;
                if (a.use_far && unit && D2 >= a.fc[0].dist2) {
                    // least distance squared of the target segment from the source's axis line
                    const double dl = dx * ux + dy * uy + dz * uz, tl = t0 * ux + t1 * uy + t2 * uz;
                    const double dt = dx * t0 + dy * t1 + dz * t2;
                    const double aq = 1.0 - tl * tl, bq = dt - dl * tl, cq = D2 - dl * dl;
                    const double s = (aq > 1e-12) ? fmin(1.0, fmax(-1.0, -bq / aq)) : 0.0;
                    if (cq + s * (2.0 * bq + s * aq) >= 1e-2)
                        cls = (D2 >= a.fc[2].dist2) ? 3 : (D2 >= a.fc[1].dist2) ? 2 : 1;
                }
            }
#pragma unroll
            for (int c = 0; c <= NC; ++c) {
                const unsigned long long in = __ballot(cls == c);
                if (cls == c) list[wave][c][count[c] + __popcll(in & ((1ull << lane) - 1ull))] = (unsigned short)(j - jb);
                count[c] += __popcll(in);
            }
        }
        // Near sources: element e is entry e / LQ of the list at point e % LQ.
        // Each goes to the queue of its path -- forward recurrences
        // (|R|^2 < 10), quadrature, or backward recurrences (closer than 0.1
        // to the axis line) -- and 64 queued elements are evaluated together.
        auto element = [&](int id, int& j, int& p, double (&X)[3]) {  // id: list position << 7 | point
            j = jb + (id >> 7);
            p = id & 127;
            const double s = tpv[p];
            X[0] = x0 + s * t0;
            X[1] = x1 + s * t1;
            X[2] = x2 + s * t2;
        };
        auto evaluate = [&](auto path, int k) {  // the first k entries of a queue
            constexpr int Pt = decltype(path)::value;
            if (lane >= k) return;
            int j, p;
            double X[3], gv[1][3];
            double(&g)[3] = gv[0];
            element(queue[wave][Pt][lane], j, p, X);
            const double xj[3] = {a.pos[3 * j], a.pos[3 * j + 1], a.pos[3 * j + 2]};
            const double tj[3] = {a.orient[3 * j], a.orient[3 * j + 1], a.orient[3 * j + 2]};
            const double* cs = a.src + (size_t)j * a.src_stride;
            if constexpr (Pt == 1) {
                const double r0[1][3] = {{X[0] - xj[0], X[1] - xj[1], X[2] - xj[2]}};
                quadrature_g<far_inner_nodes(M, 0), 1>(r0, tj, tfar + a.fc[0].sq, cs + 4 * NL, e2, e6, gv);
            } else {
                analytic_g<M, Pt == 0 ? kForward : kBackward>(X[0], X[1], X[2], xj, tj, cs, e2, e6, g);
            }
#pragma unroll
            for (int kk = 0; kk < NL; ++kk) {
                const double w = twp[kk * LQ + p];
#pragma unroll
                for (int c = 0; c < 3; ++c) acc[3 * kk + c] += w * g[c];
            }
        };
        int queued[3] = {0, 0, 0};
        auto drain = [&](auto path, int least) {  // evaluates full queues, or whatever is left (least = 1)
            constexpr int Pt = decltype(path)::value;
            if (queued[Pt] < least) return;
            const int k = min(64, queued[Pt]);
            evaluate(path, k);
            queued[Pt] -= k;
            if (lane < queued[Pt]) queue[wave][Pt][lane] = queue[wave][Pt][64 + lane];
        };
        {
            int at = lane / LQ, p = lane % LQ;
            const int da = 64 / LQ, dp = 64 % LQ;
            const int total = count[0] * LQ;
            for (int e = lane; e - lane < total; e += 64) {
                int path = -1, id = 0;
                if (e < total) {
                    const int li = list[wave][0][at];
                    int j;
                    double X[3];
                    id = li << 7 | p;
                    element(id, j, p, X);
                    const double rx = X[0] - a.pos[3 * j], ry = X[1] - a.pos[3 * j + 1], rz = X[2] - a.pos[3 * j + 2];
                    const double ux = a.orient[3 * j], uy = a.orient[3 * j + 1], uz = a.orient[3 * j + 2];
                    const double h = rx * ux + ry * uy + rz * uz;
                    const double c = rx * rx + ry * ry + rz * rz;
                    const bool smooth = c >= a.point_c && c - h * h >= 1e-2 && ux * ux + uy * uy + uz * uz <= kUnit2;
                    path = (c < 10.0) ? 0 : (a.use_far && smooth) ? 1 : 2;
                }
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    const unsigned long long in = __ballot(path == q);
                    if (path == q) queue[wave][q][queued[q] + __popcll(in & ((1ull << lane) - 1ull))] = (unsigned short)id;
                    queued[q] += __popcll(in);
                }
                drain(std::integral_constant<int, 0>{}, 64);
                drain(std::integral_constant<int, 1>{}, 64);
                drain(std::integral_constant<int, 2>{}, 64);
                at += da;
                p += dp;
                if (p >= LQ) {
                    p -= LQ;
                    ++at;
                }
            }
            drain(std::integral_constant<int, 0>{}, 1);
            drain(std::integral_constant<int, 1>{}, 1);
            drain(std::integral_constant<int, 2>{}, 1);
        }
        auto far = [&](auto cc) {
            constexpr int c = decltype(cc)::value, Q = far_inner_nodes(M, c);
            const int n = a.fc[c].n;
            int off = 4 * NL;  // the class's source vectors
#pragma unroll
            for (int b = 0; b < c; ++b) off += 3 * far_inner_nodes(M, b);
            // a lane takes the outer nodes p and p + h of a source
            const int h = (n + 1) / 2;
            int at = lane / h, p = lane % h;
            const int da = 64 / h, dp = 64 % h;
            for (; at < count[c + 1]; at += da) {
                const int j = jb + list[wave][c + 1][at];
                const double tj[3] = {a.orient[3 * j], a.orient[3 * j + 1], a.orient[3 * j + 2]};
                const double dx = x0 - a.pos[3 * j], dy = x1 - a.pos[3 * j + 1], dz = x2 - a.pos[3 * j + 2];
                const bool two = p + h < n;
                const int p2 = two ? p + h : p;
                const double s = tfar[a.fc[c].node + p], s2 = tfar[a.fc[c].node + p2];
                const double r0[2][3] = {{dx + s * t0, dy + s * t1, dz + s * t2}, {dx + s2 * t0, dy + s2 * t1, dz + s2 * t2}};
                double g[2][3];
                quadrature_g<Q, 2>(r0, tj, tfar + a.fc[c].sq, a.src + (size_t)j * a.src_stride + off, e2, e6, g);
#pragma unroll
                for (int k = 0; k < NL; ++k) {
                    const double* W = tfar + a.fc[c].W + k * n;
                    const double w = W[p], w2 = two ? W[p2] : 0.0;
#pragma unroll
                    for (int d = 0; d < 3; ++d) acc[3 * k + d] += w * g[0][d] + w2 * g[1][d];
                }
                p += dp;
                if (p >= h) {
                    p -= h;
                    ++at;
                }
            }
        };
        if (a.use_far) {
            far(std::integral_constant<int, 0>{});
            far(std::integral_constant<int, 1>{});
            far(std::integral_constant<int, 2>{});
        }
    }
#pragma unroll
    for (int e = 0; e < NL * 3; ++e) {
        double v = acc[e];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        if (lane == 0) red[wave][e] = v;
    }
    __syncthreads();
    if (tid < NL * 3)
        a.part[((size_t)blockIdx.y * N + i) * (NL * 3) + tid] =
            (red[0][tid] + red[1][tid]) + (red[2][tid] + red[3][tid]);
}

// Sums the split partials in a fixed order and applies the output map of the
// mode (one thread per (fiber, k)):
//   mode 0: y = x + P(IF)       (A x)
//   mode 1: y = -(x + P(IF))    (b - A x; the force term is in IF)
//   mode 2: y = -P(IF)          (b)
//   mode 3: y6[6i + 3k + c] = IF_k(i)_c for k = 0, 1  (the velocity sums)
// with P_k(IF) = D1 t (t.IF_1) for k = 1 and gamma_k (IF_k - E_k t (t.IF_k))
// for k >= 2 (fortran/matrix_assembly.f90:341-395).
struct OpEpiArgs {
    int N, M, splits, mode;
    int use_x;    // modes 0, 1: the identity term x
    double sign;  // +1 mode 0, -1 modes 1, 2
    double D1;
    double Ek[kMaxTerms + 1], gam[kMaxTerms + 1];
    const double* orient;
    const double* part;
    const double* x;
    double* y;
};

__global__ void operator_epilogue_kernel(const OpEpiArgs a)
{
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    const int NL = a.M + 1;
    if (idx >= a.N * NL) return;
    const int i = idx / NL, k = idx - i * NL;
    const size_t stride = (size_t)a.N * NL * 3;
    double s[3] = {0.0, 0.0, 0.0};
    const double* pp = a.part + (size_t)i * NL * 3 + 3 * k;
    for (int sp = 0; sp < a.splits; ++sp) {
#pragma unroll
        for (int c = 0; c < 3; ++c) s[c] += pp[sp * stride + c];
    }
    if (a.mode == 3) {
        if (k <= 1) {
#pragma unroll
            for (int c = 0; c < 3; ++c) a.y[6 * (size_t)i + 3 * k + c] = s[c];
        }
        return;
    }
    if (k == 0) return;
    const double t0 = a.orient[3 * i], t1 = a.orient[3 * i + 1], t2 = a.orient[3 * i + 2];
    const double td = t0 * s[0] + t1 * s[1] + t2 * s[2];
    const double tt[3] = {t0, t1, t2};
    const size_t row = (size_t)i * 3 * a.M + 3 * (k - 1);
    // One arithmetic form for modes 0..2 (y = sign (x + P) with x = 0 in
    // mode 2): a three-way branch on the mode here was compiled to a store
    // of an undefined register for mode 2.
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const double pc = (k == 1) ? a.D1 * td * tt[c] : a.gam[k] * (s[c] - a.Ek[k] * td * tt[c]);
        const double xv = a.use_x ? a.x[row + c] : 0.0;
        a.y[row + c] = a.sign * (xv + pc);
    }
}

}  // namespace

OperatorPlan plan_operator(int N, int M, int LQ, int analytic, int num_cus, int far)
{
    OperatorPlan p;
    p.N = N;
    p.M = M;
    p.LQ = LQ;
    p.analytic = analytic;
    if (analytic) {
        // A workgroup per target and split; two fit a CU.  As many splits as
        // one filling of the places takes with at least 16 sources each (fewer
        // leave lanes without elements), and two beyond that where the
        // wavefronts still have some 800 points each: N = 150 44 us (51 with
        // five), N = 600 198 us (one 224, three 207), N = 390 with 12 points 78
        // us (two 84).
        p.far = far;
        p.T = 1;
        p.threads = 256;
        p.splits = std::max(1, std::min(2 * num_cus / N, N / 16));
        if (p.splits == 1 && (int64_t)N * LQ >= 6400) p.splits = 2;
        p.src_stride = 4 * (M + 1);
        for (int c = 0; c < Tables::kFarClasses && far; ++c) p.src_stride += 3 * far_inner_nodes(M, c);
    } else {
        // T targets per workgroup, one thread per (target, point): prefer whole
        // 64-wide wavefronts and at most 512 threads.
        int T = 0;
        for (int t = 16; t >= 1; --t)
            if (t * LQ <= 512 && (t * LQ) % 64 == 0) {
                T = t;
                break;
            }
        if (T == 0) T = std::max(1, std::min(16, 256 / LQ));
        p.T = T;
        p.threads = T * LQ;
        const int tiles = (N + T - 1) / T;
        // enough workgroups for every CU several times over, with at least 8
        // sources per split
        const int want = (4 * num_cus + tiles - 1) / tiles;
        p.splits = std::max(1, std::min(want, std::max(1, N / 8)));
        p.src_stride = 4 * LQ;
    }
    p.src_per_split = (N + p.splits - 1) / p.splits;
    p.splits = (N + p.src_per_split - 1) / p.src_per_split;
    return p;
}

size_t operator_scratch_doubles(const OperatorPlan& p)
{
    return (size_t)p.N * p.src_stride + (size_t)p.splits * p.N * (p.M + 1) * 3;
}

hipError_t launch_operator(const OperatorPlan& p, const Tables& t, int mode, const double* pos, const double* orient,
                           const double* force, const double* x, const double* wp, const double* pv, const double* far,
                           double* scratch, double* y, hipStream_t s)
{
    if (mode < 0 || mode > 3 || p.M != t.M || p.LQ != t.LQ || p.threads > 512) return hipErrorInvalidValue;
    double* src = scratch;
    double* part = scratch + (size_t)p.N * p.src_stride;
    {
        OpFarSources fs;
        int per = p.analytic ? (p.M + 1) : p.LQ;
        if (p.analytic && p.far) {
            fs.tab = far;
            for (int c = 0; c < Tables::kFarClasses; ++c) {
                fs.q[c] = t.fc[c].q;
                fs.wP[c] = t.fc[c].wP;
                per += fs.q[c];
            }
        }
        const int64_t tot = (int64_t)p.N * per;
        // force term: none for A x; F_z only for the analytic right-hand side
        const int fmask = (mode == 0) ? 0 : ((mode == 1 || mode == 2) && p.analytic) ? 4 : 7;
        const int x_on = (mode == 2) ? 0 : 1;
        hipLaunchKernelGGL(op_source_kernel, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s, p.N, p.M, p.LQ,
                           p.analytic, fmask, x_on, force, x, orient, wp, src, p.src_stride, fs);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    hipError_t e = hipErrorInvalidValue;
    auto launch = [&](auto mm) {
        constexpr int M = decltype(mm)::value;
        if (p.analytic) {
            FarKArgs k;
            k.N = p.N;
            k.LQ = p.LQ;
            k.src_per_split = p.src_per_split;
            k.src_stride = p.src_stride;
            k.use_far = p.far;
            k.far_total = p.far ? t.far_total : 0;
            k.eps = t.eps;
            k.point_c = t.point_c;
            for (int c = 0; c < Tables::kFarClasses; ++c) k.fc[c] = t.fc[c];
            k.pos = pos;
            k.orient = orient;
            k.src = src;
            k.wp = wp;
            k.pv = pv;
            k.far = far;
            k.part = part;
            const size_t lds = sizeof(double) * (size_t)((M + 2) * p.LQ + k.far_total);
            hipLaunchKernelGGL(operator_kernel<M>, dim3(p.N, p.splits), dim3(256), lds, s, k);
        } else {
            OpKArgs k;
            k.N = p.N;
            k.LQ = p.LQ;
            k.T = p.T;
            k.src_per_split = p.src_per_split;
            k.src_stride = p.src_stride;
            k.eps = t.eps;
            k.pos = pos;
            k.orient = orient;
            k.src = src;
            k.wp = wp;
            k.pv = pv;
            k.part = part;
            const size_t lds = sizeof(double) * (size_t)p.T * p.LQ * 3;
            hipLaunchKernelGGL(operator_numeric_kernel<M>, dim3((p.N + p.T - 1) / p.T, p.splits), dim3(p.threads), lds,
                               s, k);
        }
        return hipGetLastError();
    };
    switch (p.M) {
    case 1: e = launch(std::integral_constant<int, 1>{}); break;
    case 2: e = launch(std::integral_constant<int, 2>{}); break;
    case 3: e = launch(std::integral_constant<int, 3>{}); break;
    case 4: e = launch(std::integral_constant<int, 4>{}); break;
    case 5: e = launch(std::integral_constant<int, 5>{}); break;
    case 6: e = launch(std::integral_constant<int, 6>{}); break;
    case 7: e = launch(std::integral_constant<int, 7>{}); break;
    case 8: e = launch(std::integral_constant<int, 8>{}); break;
    }
    if (e != hipSuccess) return e;
    return launch_operator_epilogue(p, t, mode, orient, x, scratch, y, s);
}

hipError_t launch_operator_epilogue(const OperatorPlan& p, const Tables& t, int mode, const double* orient,
                                    const double* x, const double* scratch, double* y, hipStream_t s)
{
    if (mode < 0 || mode > 3 || p.M != t.M) return hipErrorInvalidValue;
    const double* part = scratch + (size_t)p.N * p.src_stride;
    OpEpiArgs ea;
    ea.N = p.N;
    ea.M = p.M;
    ea.splits = p.splits;
    ea.mode = mode;
    ea.use_x = (mode == 0 || mode == 1) ? 1 : 0;
    ea.sign = (mode == 0) ? 1.0 : -1.0;
    ea.D1 = t.D1;
    for (int i = 0; i <= kMaxTerms; ++i) {
        ea.Ek[i] = t.Ek[i];
        ea.gam[i] = t.gammak[i];
    }
    ea.orient = orient;
    ea.part = part;
    ea.x = x;
    ea.y = y;
    const int tot = p.N * (p.M + 1);
    hipLaunchKernelGGL(operator_epilogue_kernel, dim3((tot + 255) / 256), dim3(256), 0, s, ea);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// The operator on caller-provided device buffers without any allocation
// (rf_operator_noalloc).  Its scratch -- the quadrature tables, the
// velocity sums and the operator's source vectors and split partials -- is
// one file-scope device array per GPU, resolved once per device with
// hipGetSymbolAddress; host code uses only that address.
// ---------------------------------------------------------------------------
namespace {

constexpr size_t kNoAllocScratchDoubles = size_t(1) << 22;  // 32 MiB per GPU
constexpr size_t kTableDoubles = 1024;                      // wp[(M+1) LQ] (<= 864), then pv[LQ]
constexpr size_t kFarTableDoubles = 704;                    // then Tables::far
constexpr int kMaxDevices = 64;

static __device__ __align__(256) double scratch[kNoAllocScratchDoubles];

std::mutex g_scratch_mutex;
double* g_scratch_ptr[kMaxDevices] = {nullptr};

// up to 448 table values per launch, passed by value
constexpr int kChunk = 448;
struct TableChunk {
    int offset, count;
    double v[kChunk];
};

__global__ void store_table_kernel(double* __restrict__ dst, const TableChunk c)
{
    const int i = threadIdx.x;
    if (i < c.count) dst[c.offset + i] = c.v[i];
}

// wp, pv and (far) the far tables, one after the other at dst
hipError_t store_tables(double* dst, const Tables& t, bool far, hipStream_t s)
{
    TableChunk c;
    c.offset = c.count = 0;
    auto flush = [&]() -> hipError_t {
        if (c.count == 0) return hipSuccess;
        hipLaunchKernelGGL(store_table_kernel, dim3(1), dim3(kChunk), 0, s, dst, c);
        c.offset += c.count;
        c.count = 0;
        return hipGetLastError();
    };
    hipError_t e = hipSuccess;
    auto put = [&](const double* src, int count) {
        for (int i = 0; i < count && e == hipSuccess; ++i) {
            c.v[c.count++] = src[i];
            if (c.count == kChunk) e = flush();
        }
    };
    put(t.wp, (t.M + 1) * t.LQ);
    put(t.pv, t.LQ);
    if (far) put(t.far, t.far_total);
    return e == hipSuccess ? flush() : e;
}

}  // namespace

// The device address of this GPU's scratch array (set-up once per device).
static int noalloc_scratch(double** out)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        set_error("rf_operator_noalloc: no current HIP device");
        return RF_EHIP;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            set_error(std::string("rf_operator_noalloc: hipGetSymbolAddress: ") + hipGetErrorString(e));
            return RF_EHIP;
        }
        g_scratch_ptr[dev] = static_cast<double*>(ptr);
    }
    *out = g_scratch_ptr[dev];
    return RF_OK;
}

}  // namespace rf

extern "C" int rf_operator_noalloc(const rf_params* params, int32_t num_fibers, int32_t mode, const double* pos,
                                   const double* orient, const double* force, const double* x, double* y,
                                   void* stream)
{
    using namespace rf;
    if (!params || !pos || !orient || !force || !y || (mode != RF_OP_RHS && !x) || mode < RF_OP_AX ||
        mode > RF_OP_VELOCITY) {
        set_error("rf_operator_noalloc: null buffer or unknown mode");
        return RF_EINVAL;
    }
    const rf_params& P = *params;
    if (num_fibers < 2 || P.num_terms < 1 || P.num_terms > kMaxTerms || P.num_quad_intervals < 1 ||
        3 * P.num_quad_intervals > kMaxQuad || !(P.slenderness > 0.0)) {
        set_error("rf_operator_noalloc: invalid parameters (need N>=2, 1<=M<=8, 1<=NoQI<=32, eps>0)");
        return RF_EINVAL;
    }
    Tables tab;
    build_tables(P.num_terms, P.num_quad_intervals, P.slenderness, &tab);
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
        set_error("rf_operator_noalloc: cannot query the device");
        return RF_EHIP;
    }
    const int N = num_fibers;
    // What is rejected does not depend on the far pairs' tables and source
    // vectors: a system too large for them takes every pair through the moments.
    const int analytic = P.use_analytical_integration ? 1 : 0;
    OperatorPlan plan = plan_operator(N, tab.M, tab.LQ, analytic, cus);
    const size_t per_split = (size_t)N * (tab.M + 1) * 3;
    auto fixed = [&] {
        return kTableDoubles + (plan.far ? kFarTableDoubles : 0) + 6 * (size_t)N + (size_t)N * plan.src_stride;
    };
    if (analytic && fixed() + per_split > kNoAllocScratchDoubles)
        plan = plan_operator(N, tab.M, tab.LQ, analytic, cus, 0);
    if (fixed() + per_split > kNoAllocScratchDoubles) {
        set_error("rf_operator_noalloc: " + std::to_string(N) + " fibers need " +
                  std::to_string((fixed() + per_split) * sizeof(double)) + " bytes of scratch; the maximum is " +
                  std::to_string(kNoAllocScratchDoubles * sizeof(double)) + " (rf_operator has no limit)");
        return RF_EINVAL;
    }
    const size_t max_splits = (kNoAllocScratchDoubles - fixed()) / per_split;
    if ((size_t)plan.splits > max_splits) {
        plan.splits = (int)max_splits;
        plan.src_per_split = (N + plan.splits - 1) / plan.splits;
        plan.splits = (N + plan.src_per_split - 1) / plan.src_per_split;
    }
    double* base = nullptr;
    int rc = noalloc_scratch(&base);
    if (rc) return rc;
    double* wp = base;
    double* pv = wp + (size_t)(tab.M + 1) * tab.LQ;
    double* far = pv + tab.LQ;
    double* y6 = base + kTableDoubles + (plan.far ? kFarTableDoubles : 0);
    double* work = y6 + 6 * (size_t)N;
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipError_t e = store_tables(base, tab, plan.far != 0, s);
    const int kmode = (mode == RF_OP_AX) ? kOpAx : (mode == RF_OP_RESIDUAL) ? kOpResidual
                                                : (mode == RF_OP_RHS) ? kOpRhs : kOpVelocity;
    if (e == hipSuccess)
        e = launch_operator(plan, tab, kmode, pos, orient, force, x, wp, pv, far, work,
                            (mode == RF_OP_VELOCITY) ? y6 : y, s);
    if (e == hipSuccess && mode == RF_OP_VELOCITY)
        e = launch_velocity_epilogue(N, tab.d, tab.e, P.shear_rate, pos, orient, force, y6, y, y + 3 * (size_t)N, s);
    if (e != hipSuccess) {
        set_error(std::string("rf_operator_noalloc: ") + hipGetErrorString(e));
        return RF_EHIP;
    }
    return RF_OK;
}
