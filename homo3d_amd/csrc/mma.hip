// GPU MMA step (homo::MMAOptimizer, optimization/mmaOptimizer.cu:18-77, and mmasub_g / subsolv_g,
// optimization/mmaOpt.cu:429-1062), everything in FP64: the per-variable work and its reductions run
// over the whole GPU, the m-sized dual variables, the (m+1) x (m+1) Newton system (solveLinearHost,
// mmaOpt.cpp:48-73; here Gaussian elimination with partial pivoting), the step lengths and the line
// search's decisions in one-workgroup control kernels on the device.  The host only queues rounds and
// looks, a round behind, whether the interior-point method has ended.
//
// What bounds a step: an interior-point step needs each variable's data three times (Newton sums, step
// length, line search), and there are a few hundred of them, so the bytes per variable and pass count.
// A variable's 13 + 3 FP64 coefficients of the convex approximation (p0, q0, P_i, Q_i, alfa, beta) are
// functions of the FP32 design and gradients, the bounds and the asymptotes; they are formed again in
// each pass from those (72 bytes a variable for m = 2 instead of 104, and no coefficient is ever
// written), and so is the Newton direction (from the last point and multipliers) instead of being
// stored.  The line search tries kMmaCand halvings per pass over the variables: it needs 5.2 on average
// at 128^3, m = 2 (a step took 39.1 ms with four a pass where it took 36.1 with eight, both with as many
// search workgroups as the other passes have).  There a step of 269 Newton steps takes 35 ms (188 with the
// direction and every trial point stored, a trial per pass and three host waits a Newton step); the passes
// 31.3 us (Newton sums, with the iterate's update), 24.2 us (step length, 6.2 TB/s of the 151 MB it reads,
// which stay in the last-level cache) and 48.7 us (eight trials, bound by FP64 arithmetic), the control
// kernels 5-8 us each.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "../../include/homo3d.h"

namespace {

constexpr int kMmaMaxM = 4;
constexpr int kMmaBlocks = 1024;   // workgroups of the per-variable passes
constexpr int kMmaSearchBlocks = 768;  // of the search pass, whose registers allow three a CU (1024: 52 us, 768: 49)
constexpr int kMmaThreads = 256;
constexpr int kMmaCand = 8;        // line-search steps tried per pass: steg, steg / 2, ..., steg / 128
constexpr int kMmaCtlThreads = 1024;
constexpr int kMmaSums = kMmaCand * (2 + kMmaMaxM);  // most quantities a pass reduces
constexpr int kMmaNewton = 200;    // most Newton steps of one epsi

enum { kPhaseNewton = 0, kPhaseSearch = 1, kPhaseResid = 2, kPhaseDone = 3 };

// The small state of subsolv_g (mmaOpt.cu:429-834), on the device.
struct MmaState {
    int phase, status;      // status 1: singular Newton system
    int itera, ittt, itto;  // Newton steps in all, of this epsi, and trials of the running line search
    int pending;            // x, xsi, eta still lack steg times the direction of (lamo, dlam, epsd)
    double a0, a[kMmaMaxM], c[kMmaMaxM], d[kMmaMaxM], b[kMmaMaxM], gval[kMmaMaxM];
    double epsi, residunorm, steg, epsd;
    double y[kMmaMaxM], lam[kMmaMaxM], mu[kMmaMaxM], s[kMmaMaxM], z, zet;
    double yo[kMmaMaxM], lamo[kMmaMaxM], muo[kMmaMaxM], so[kMmaMaxM], zo, zeto;  // before the running step
    double dy[kMmaMaxM], dlam[kMmaMaxM], dmu[kMmaMaxM], ds[kMmaMaxM], dz, dzet;  // its direction
    double gvec[kMmaMaxM];
};

// Per-variable arrays of one step.
struct MmaVars {
    long n;
    const float *x0, *df, *dg;  // design, objective gradient, m constraint gradients [m][n]
    const double *lo, *up, *xmin, *xmax;
    double *x, *xsi, *eta;      // the subproblem's iterate
};

// One variable: iterate and convex approximation (mmasub_ker, mmaOpt.cu:864-989; move = 1).
template <int M>
struct MmaVar {
    double x, xsi, eta, lo, up, alfa, beta, p0, q0, P[M], Q[M];
    __device__ __forceinline__ void load(const MmaVars& v, long j) {
        const double x0 = (double)v.x0[j], xl = v.xmin[j], xu = v.xmax[j], dx = xu - xl;
        const double g0 = (double)v.df[j];
        double g[M];
#pragma unroll
        for (int i = 0; i < M; i++) g[i] = (double)v.dg[(size_t)i * v.n + j];
        lo = v.lo[j];
        up = v.up[j];
        x = v.x[j];
        xsi = v.xsi[j];
        eta = v.eta[j];
        const double raa0 = 1e-5, albefa = 0.1;
        alfa = fmax(fmax(lo + albefa * (x0 - lo), x0 - dx), xl);
        beta = fmin(fmin(up - albefa * (up - x0), x0 + dx), xu);
        const double ux1 = up - x0, xl1 = x0 - lo, ux2 = ux1 * ux1, xl2 = xl1 * xl1;
        const double r = raa0 * (1.0 / fmax(dx, 1e-5));
        const double dp = fmax(g0, 0.0), dm = fmax(-g0, 0.0), pq0 = 1e-3 * (dp + dm) + r;
        p0 = (dp + pq0) * ux2;
        q0 = (dm + pq0) * xl2;
#pragma unroll
        for (int i = 0; i < M; i++) {
            const double pp = fmax(g[i], 0.0), qq = fmax(-g[i], 0.0), pq = 1e-3 * (pp + qq) + r;
            P[i] = (pp + pq) * ux2;
            Q[i] = (qq + pq) * xl2;
        }
    }
    // Newton terms at the iterate for multipliers lam: delx, diagx and gg (subsolv_g, mmaOpt.cu:560-640)
    __device__ __forceinline__ void newton(const double* lam, double epsi, double& dl, double& dg, double (&gg)[M],
                                           double& ia, double& ib) const {
        ia = 1.0 / (x - alfa);
        ib = 1.0 / (beta - x);
        const double ux1 = up - x, xl1 = x - lo, r = 1.0 / (ux1 * xl1), iu = r * xl1, il = r * ux1;
        const double iu2 = iu * iu, il2 = il * il;
        double pl = p0, ql = q0;
#pragma unroll
        for (int i = 0; i < M; i++) {
            pl += P[i] * lam[i];
            ql += Q[i] * lam[i];
            gg[i] = P[i] * iu2 - Q[i] * il2;
        }
        dl = (pl * iu2 - ql * il2) - epsi * ia + epsi * ib;
        dg = 2 * (pl * iu2 * iu + ql * il2 * il) + xsi * ia + eta * ib;
    }
    // Newton direction (mmaOpt.cu:680-700), and 1 / (x - alfa), 1 / (beta - x)
    __device__ __forceinline__ void direction(const double* lam, const double* dlam, double epsi, double& dx,
                                              double& dxsi, double& deta, double& ia, double& ib) const {
        double dl, dg, gg[M];
        newton(lam, epsi, dl, dg, gg, ia, ib);
        double t = dl;
#pragma unroll
        for (int i = 0; i < M; i++) t += gg[i] * dlam[i];
        dx = -t / dg;
        dxsi = -xsi + epsi * ia - (xsi * dx) * ia;
        deta = -eta + epsi * ib + (eta * dx) * ib;
    }
};

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}
__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_down(v, off, 64));
    return v;
}

// part[q * nb + block] of NS block sums (and, with MAX, one more quantity in the NS-th place: a maximum)
template <int NS, bool MAX>
__device__ __forceinline__ void block_parts(const double (&sum)[NS > 0 ? NS : 1], double mx, double* part) {
    __shared__ double sh[kMmaThreads / 64][NS + 1];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < NS; q++) {
        const double t = wave_sum(sum[q]);
        if (lane == 0) sh[w][q] = t;
    }
    if constexpr (MAX) {
        const double t = wave_max(mx);
        if (lane == 0) sh[w][NS] = t;
    }
    __syncthreads();
    if ((int)threadIdx.x < NS + (MAX ? 1 : 0)) {
        const int q = threadIdx.x;
        double t = sh[0][q];
        for (int k = 1; k < kMmaThreads / 64; k++) t = MAX && q == NS ? fmax(t, sh[k][q]) : t + sh[k][q];
        part[(size_t)q * gridDim.x + blockIdx.x] = t;
    }
}

// Asymptotes and the iterate's start (mmaOpt.cu:864-989; subsolv_g's initial point), block sums of
// P_i / (upp - x) + Q_i / (x - low).
template <int M>
__global__ __launch_bounds__(kMmaThreads) void k_mma_setup(MmaVars v, int iter, const double* __restrict__ xold1,
                                                           const double* __restrict__ xold2, double* lo_,
                                                           double* up_, double* __restrict__ part) {
    const double asyinit = 0.5, asyincr = 1.2, asydecr = 0.7;
    double bs[M] = {};
    for (long j = (long)blockIdx.x * blockDim.x + threadIdx.x; j < v.n; j += (long)gridDim.x * blockDim.x) {
        const double xj = (double)v.x0[j], dx = v.xmax[j] - v.xmin[j];
        double lo, up;
        if (iter <= 2) {
            lo = xj - asyinit * dx;
            up = xj + asyinit * dx;
        } else {
            const double zzz = (xj - xold1[j]) * (xold1[j] - xold2[j]);
            const double fac = zzz > 0 ? asyincr : (zzz < 0 ? asydecr : 1.0);
            lo = xj - fac * (xold1[j] - lo_[j]);
            up = xj + fac * (up_[j] - xold1[j]);
            lo = fmax(lo, xj - 10 * dx);
            lo = fmin(lo, xj - 0.01 * dx);
            up = fmin(up, xj + 10 * dx);
            up = fmax(up, xj + 0.01 * dx);
        }
        lo_[j] = lo;
        up_[j] = up;
        MmaVar<M> a;
        a.load(v, j);  // with this thread's own lo, up (v.lo, v.up are lo_, up_); the iterate is not used
        const double xs = 0.5 * (a.alfa + a.beta);
        v.x[j] = xs;
        v.xsi[j] = fmax(1.0 / (xs - a.alfa), 1.0);
        v.eta[j] = fmax(1.0 / (a.beta - xs), 1.0);
#pragma unroll
        for (int i = 0; i < M; i++) bs[i] += a.P[i] / (up - xj) + a.Q[i] / (xj - lo);
    }
    block_parts<M, false>(bs, 0.0, part);
}

// First pass of a Newton step: the accepted step of the line search before it is applied to the
// iterate, then the sums of the Newton system: gg_i delx / diagx and gg_i gg_k / diagx (k >= i).
template <int M>
__global__ __launch_bounds__(kMmaThreads, M <= 2 ? 4 : 2) void k_mma_newton(MmaVars v, const MmaState* __restrict__ st,
                                                               double* __restrict__ part) {
    if (st->phase != kPhaseNewton) return;
    constexpr int NS = M + M * (M + 1) / 2;
    double acc[NS] = {};
    const double epsi = st->epsi, epsd = st->epsd, steg = st->steg;
    const int pending = st->pending;
    double lam[M], lamo[M], dlam[M];
#pragma unroll
    for (int i = 0; i < M; i++) {
        lam[i] = st->lam[i];
        lamo[i] = st->lamo[i];
        dlam[i] = st->dlam[i];
    }
    for (long j = (long)blockIdx.x * blockDim.x + threadIdx.x; j < v.n; j += (long)gridDim.x * blockDim.x) {
        MmaVar<M> a;
        a.load(v, j);
        if (pending) {
            double dx, dxsi, deta, ia, ib;
            a.direction(lamo, dlam, epsd, dx, dxsi, deta, ia, ib);
            v.x[j] = a.x = a.x + steg * dx;
            v.xsi[j] = a.xsi = a.xsi + steg * dxsi;
            v.eta[j] = a.eta = a.eta + steg * deta;
        }
        double dl, dg, gg[M], ia, ib;
        a.newton(lam, epsi, dl, dg, gg, ia, ib);
        const double ig = 1.0 / dg;
        int k = M;
#pragma unroll
        for (int i = 0; i < M; i++) {
            acc[i] += gg[i] * dl * ig;
#pragma unroll
            for (int q = i; q < M; q++) acc[k++] += gg[i] * gg[q] * ig;
        }
    }
    block_parts<NS, false>(acc, 0.0, part);
}

// Second pass: the largest step-length ratio of the variables (stepxx / stepalfa / stepbeta).
template <int M>
__global__ __launch_bounds__(kMmaThreads, M <= 2 ? 4 : 2) void k_mma_length(MmaVars v, const MmaState* __restrict__ st,
                                                               double* __restrict__ part) {
    if (st->phase != kPhaseNewton) return;
    const double epsi = st->epsi;
    double lam[M], dlam[M];
#pragma unroll
    for (int i = 0; i < M; i++) {
        lam[i] = st->lam[i];
        dlam[i] = st->dlam[i];
    }
    double stm = -1e300;
    for (long j = (long)blockIdx.x * blockDim.x + threadIdx.x; j < v.n; j += (long)gridDim.x * blockDim.x) {
        MmaVar<M> a;
        a.load(v, j);
        double dx, dxsi, deta, ia, ib;
        a.direction(lam, dlam, epsi, dx, dxsi, deta, ia, ib);
        stm = fmax(stm, fmax(fmax(-1.01 * dxsi / a.xsi, -1.01 * deta / a.eta), fmax(-1.01 * dx * ia, 1.01 * dx * ib)));
    }
    const double none[1] = {};
    block_parts<0, true>(none, stm, part);
}

// Third pass: the residual's sums at the points x + steg 2^-k dx, k < CAND (the line search), or with
// CAND = 1 at the accepted point alone.  Per candidate: squared norm, the m constraint sums, and the
// largest entry.
template <int M, int CAND>
__device__ __forceinline__ void mma_search(const MmaVars& v, const MmaState* __restrict__ st,
                                           double* __restrict__ part) {
    const double epsi = st->epsi, epsd = st->epsd, steg = st->steg;
    const int dir = st->phase == kPhaseSearch || st->pending;
    double lamo[M], dlam[M], sum[CAND * (1 + M)] = {}, mx[CAND];
#pragma unroll
    for (int i = 0; i < M; i++) {
        lamo[i] = dir ? st->lamo[i] : st->lam[i];
        dlam[i] = dir ? st->dlam[i] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < CAND; k++) mx[k] = 0.0;
    for (long j = (long)blockIdx.x * blockDim.x + threadIdx.x; j < v.n; j += (long)gridDim.x * blockDim.x) {
        MmaVar<M> a;
        a.load(v, j);
        double dx = 0.0, dxsi = 0.0, deta = 0.0, ia, ib;
        if (dir) a.direction(lamo, dlam, epsd, dx, dxsi, deta, ia, ib);
        // everything a candidate needs is linear in its step, and its two reciprocals share one division
        const double ux0 = a.up - a.x, xl0 = a.x - a.lo, xa0 = a.x - a.alfa, bx0 = a.beta - a.x;
        double pl0 = a.p0, ql0 = a.q0, dpl = 0.0, dql = 0.0;
#pragma unroll
        for (int i = 0; i < M; i++) {
            pl0 += a.P[i] * lamo[i];
            ql0 += a.Q[i] * lamo[i];
            dpl += a.P[i] * dlam[i];
            dql += a.Q[i] * dlam[i];
        }
        double sk = steg;
#pragma unroll
        for (int k = 0; k < CAND; k++) {
            const double ux1 = ux0 - sk * dx, xl1 = xl0 + sk * dx, xsi = a.xsi + sk * dxsi, eta = a.eta + sk * deta;
            const double r = 1.0 / (ux1 * xl1), iu = r * xl1, il = r * ux1;
#pragma unroll
            for (int i = 0; i < M; i++) sum[k * (1 + M) + 1 + i] += a.P[i] * iu + a.Q[i] * il;
            const double rex = ((pl0 + sk * dpl) * (iu * iu) - (ql0 + sk * dql) * (il * il)) - xsi + eta;
            const double rexsi = xsi * (xa0 + sk * dx) - epsi, reeta = eta * (bx0 - sk * dx) - epsi;
            sum[k * (1 + M)] += rex * rex + rexsi * rexsi + reeta * reeta;
            mx[k] = fmax(mx[k], fmax(fabs(rex), fmax(fabs(rexsi), fabs(reeta))));
            sk *= 0.5;
        }
    }
    __shared__ double sh[kMmaThreads / 64][CAND * (2 + M)];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < CAND; k++) {
#pragma unroll
        for (int q = 0; q <= M; q++) {
            const double t = wave_sum(sum[k * (1 + M) + q]);
            if (lane == 0) sh[w][k * (2 + M) + q] = t;
        }
        const double t = wave_max(mx[k]);
        if (lane == 0) sh[w][k * (2 + M) + 1 + M] = t;
    }
    __syncthreads();
    if (threadIdx.x < CAND * (2 + M)) {
        const int q = threadIdx.x;
        const bool is_max = q % (2 + M) == 1 + M;
        double t = sh[0][q];
        for (int k = 1; k < kMmaThreads / 64; k++) t = is_max ? fmax(t, sh[k][q]) : t + sh[k][q];
        part[(size_t)q * gridDim.x + blockIdx.x] = t;
    }
}

template <int M>
__global__ __launch_bounds__(kMmaThreads, 2) void k_mma_search(MmaVars v, const MmaState* __restrict__ st,
                                                               double* __restrict__ part) {
    if (st->phase == kPhaseSearch)
        mma_search<M, kMmaCand>(v, st, part);
    else if (st->phase == kPhaseResid)
        mma_search<M, 1>(v, st, part);
}

// ---------------------------------------------------------------------------------------------
// Control kernels: one workgroup; the waves reduce the block sums, thread 0 does the m-sized algebra.
// ---------------------------------------------------------------------------------------------
// total[q] of NQ quantities of nb block values; every (period)-th one (is_max) by its maximum
__device__ __forceinline__ void reduce_parts(const double* __restrict__ part, int nb, int nq, int period,
                                             double* total) {
    const int lane = threadIdx.x & 63;
    for (int q = threadIdx.x >> 6; q < nq; q += kMmaCtlThreads / 64) {
        const bool is_max = period && q % period == period - 1;
        const double* p = part + (size_t)q * nb;
        const double none = is_max ? -1e300 : 0.0;
        double v[kMmaBlocks / 64];
#pragma unroll
        for (int i = 0; i < kMmaBlocks / 64; i++) v[i] = lane + 64 * i < nb ? p[lane + 64 * i] : none;
        double t = none;
#pragma unroll
        for (int i = 0; i < kMmaBlocks / 64; i++) t = is_max ? fmax(t, v[i]) : t + v[i];
        t = is_max ? wave_max(t) : wave_sum(t);
        if (lane == 0) total[q] = t;
    }
    __syncthreads();
}

// The small variables at one point.
template <int M>
struct MmaSmall {
    double y[M], lam[M], mu[M], s[M], z, zet;
};

// The small part of the residual at v added to the variables' squared norm and maximum (subsolv_g's
// resi, mmaOpt.cu:700-790).
template <int M>
__device__ __forceinline__ void small_residual(const MmaState* __restrict__ st, const MmaSmall<M>& v,
                                               const double* gvec, double& s2, double& m2) {
    const double epsi = st->epsi;
    auto acc = [&](double r) {
        s2 += r * r;
        const double ar = fabs(r);
        if (m2 < ar) m2 = ar;
    };
    double alam = 0;
#pragma unroll
    for (int i = 0; i < M; i++) {
        acc(st->c[i] + st->d[i] * v.y[i] - v.mu[i] - v.lam[i]);
        alam += st->a[i] * v.lam[i];
    }
    acc(st->a0 - v.zet - alam);
#pragma unroll
    for (int i = 0; i < M; i++) acc(gvec[i] - st->a[i] * v.z - v.y[i] + v.s[i] - st->b[i]);
#pragma unroll
    for (int i = 0; i < M; i++) acc(v.mu[i] * v.y[i] - epsi);
    acc(v.zet * v.z - epsi);
#pragma unroll
    for (int i = 0; i < M; i++) acc(v.lam[i] * v.s[i] - epsi);
}

// After a residual that ends a Newton step or opens an epsi: what comes next.
__device__ __forceinline__ void next_phase(MmaState* st, double residumax) {
    const double epsi = st->epsi;
    if (residumax > 0.9 * epsi && st->ittt < kMmaNewton) {
        st->phase = kPhaseNewton;
        return;
    }
    st->epsi = epsi * 0.1;
    st->ittt = 0;
    st->phase = epsi * 0.1 > 1e-7 ? kPhaseResid : kPhaseDone;
}

template <int M>
__global__ __launch_bounds__(kMmaCtlThreads) void k_mma_begin(MmaState* st, const double* __restrict__ part, int nb) {
    __shared__ double total[kMmaSums];
    reduce_parts(part, nb, M, 0, total);
    if (threadIdx.x) return;
    MmaState& t = *st;
    for (int i = 0; i < M; i++) {
        t.b[i] = total[i] - t.gval[i];
        t.y[i] = t.lam[i] = t.s[i] = 1.0;
        t.mu[i] = fmax(1.0, 0.5 * t.c[i]);
    }
    t.z = t.zet = t.epsi = 1.0;
    t.phase = kPhaseResid;
}

// The (m+1) x (m+1) Newton system and the direction of the small variables.
template <int M>
__global__ __launch_bounds__(kMmaCtlThreads) void k_mma_solve(MmaState* st, const double* __restrict__ part, int nb) {
    if (st->phase != kPhaseNewton) return;
    __shared__ double total[kMmaSums];
    reduce_parts(part, nb, M + M * (M + 1) / 2, 0, total);
    if (threadIdx.x) return;
    MmaState t = *st;
    t.ittt++;
    t.itera++;
    t.pending = 0;
    t.epsd = t.epsi;
    double A[M + 1][M + 1], rhs[M + 1], dely[M], diagy[M], sol[M + 1];
    double alam = 0;
#pragma unroll
    for (int i = 0; i < M; i++) alam += t.a[i] * t.lam[i];
    int k = M;
#pragma unroll
    for (int i = 0; i < M; i++) {
        dely[i] = t.c[i] + t.d[i] * t.y[i] - t.lam[i] - t.epsi / t.y[i];
        const double dellam = t.gvec[i] - t.a[i] * t.z - t.y[i] - t.b[i] + t.epsi / t.lam[i];
        diagy[i] = t.d[i] + t.mu[i] / t.y[i];
        rhs[i] = dellam + dely[i] / diagy[i] - total[i];
#pragma unroll
        for (int q = i; q < M; q++) A[i][q] = A[q][i] = total[k++];
    }
#pragma unroll
    for (int i = 0; i < M; i++) {
        A[i][i] += t.s[i] / t.lam[i] + 1.0 / diagy[i];
        A[i][M] = A[M][i] = t.a[i];
    }
    A[M][M] = -t.zet / t.z;
    rhs[M] = t.a0 - alam - t.epsi / t.z;
    // elimination with partial pivoting; every index is a constant, so the system stays in registers
#pragma unroll
    for (int c = 0; c <= M; c++) {
        int pr = c;
        double best = fabs(A[c][c]);
#pragma unroll
        for (int i = c + 1; i <= M; i++)
            if (fabs(A[i][c]) > best) {
                pr = i;
                best = fabs(A[i][c]);
            }
#pragma unroll
        for (int i = c + 1; i <= M; i++)
            if (i == pr) {
#pragma unroll
                for (int q = 0; q <= M; q++) {
                    const double x = A[c][q];
                    A[c][q] = A[i][q];
                    A[i][q] = x;
                }
                const double x = rhs[c];
                rhs[c] = rhs[i];
                rhs[i] = x;
            }
        if (A[c][c] == 0) {
            st->status = 1;
            st->phase = kPhaseDone;
            return;
        }
#pragma unroll
        for (int i = c + 1; i <= M; i++) {
            const double f = A[i][c] / A[c][c];
#pragma unroll
            for (int q = c; q <= M; q++) A[i][q] -= f * A[c][q];
            rhs[i] -= f * rhs[c];
        }
    }
#pragma unroll
    for (int c = M; c >= 0; c--) {
        double x = rhs[c];
#pragma unroll
        for (int q = c + 1; q <= M; q++) x -= A[c][q] * sol[q];
        sol[c] = x / A[c][c];
    }
    t.dz = sol[M];
#pragma unroll
    for (int i = 0; i < M; i++) {
        t.dlam[i] = sol[i];
        t.dy[i] = -dely[i] / diagy[i] + sol[i] / diagy[i];
        t.dmu[i] = -t.mu[i] + t.epsi / t.y[i] - (t.mu[i] * t.dy[i]) / t.y[i];
        t.ds[i] = -t.s[i] + t.epsi / t.lam[i] - (t.s[i] * sol[i]) / t.lam[i];
        t.yo[i] = t.y[i];
        t.lamo[i] = t.lam[i];
        t.muo[i] = t.mu[i];
        t.so[i] = t.s[i];
    }
    t.dzet = -t.zet + t.epsi / t.z - t.zet * t.dz / t.z;
    t.zo = t.z;
    t.zeto = t.zet;
    *st = t;
}

// The step length and the start of the line search (subsolv_g's resinew = 2 residunorm).
template <int M>
__global__ __launch_bounds__(kMmaCtlThreads) void k_mma_steplen(MmaState* st, const double* __restrict__ part, int nb) {
    if (st->phase != kPhaseNewton) return;
    __shared__ double total[kMmaSums];
    reduce_parts(part, nb, 1, 1, total);
    if (threadIdx.x) return;
    MmaState& t = *st;
    double stm = 1.0;
    auto up = [&](double v) {
        if (stm < v) stm = v;
    };
    up(total[0]);
    for (int i = 0; i < M; i++) {
        up(-1.01 * t.dy[i] / t.y[i]);
        up(-1.01 * t.dlam[i] / t.lam[i]);
        up(-1.01 * t.dmu[i] / t.mu[i]);
        up(-1.01 * t.ds[i] / t.s[i]);
    }
    up(-1.01 * t.dz / t.z);
    up(-1.01 * t.dzet / t.zet);
    // The line search goes on while the residual is not below the one before, starting from twice that: it is
    // not entered from a residual that is not a number (a variable with equal bounds, an infinite gradient).
    // The point stays, and with it all that the further steps of this epsi would compute.
    if (!(2 * t.residunorm > t.residunorm)) {
        t.itera += kMmaNewton - t.ittt;
        t.ittt = kMmaNewton;
        next_phase(st, 0.0);
        return;
    }
    t.steg = 1.0 / stm;
    t.itto = 0;
    t.phase = kPhaseSearch;
}

// The line search's decision over the candidates of one pass, or the residual of a new epsi.
template <int M>
__global__ __launch_bounds__(kMmaCtlThreads) void k_mma_accept(MmaState* st, const double* __restrict__ part, int nb) {
    const int phase = st->phase;
    if (phase != kPhaseSearch && phase != kPhaseResid) return;
    __shared__ double total[kMmaSums];
    constexpr int per = 2 + M;
    reduce_parts(part, nb, (phase == kPhaseSearch ? kMmaCand : 1) * per, per, total);
    if (threadIdx.x >= 64) return;
    // a lane forms each candidate's residual, the first that is taken goes on
    const int k = (int)threadIdx.x, tries = phase == kPhaseSearch ? kMmaCand : 1, itto = st->itto;
    const double* q = total + (k < tries ? k : 0) * per;
    double steg = st->steg;
    for (int i = 0; i < k && i < tries; i++) steg *= 0.5;
    MmaSmall<M> v;
    if (phase == kPhaseSearch) {
#pragma unroll
        for (int i = 0; i < M; i++) {
            v.y[i] = st->yo[i] + steg * st->dy[i];
            v.lam[i] = st->lamo[i] + steg * st->dlam[i];
            v.mu[i] = st->muo[i] + steg * st->dmu[i];
            v.s[i] = st->so[i] + steg * st->ds[i];
        }
        v.z = st->zo + steg * st->dz;
        v.zet = st->zeto + steg * st->dzet;
    } else {
#pragma unroll
        for (int i = 0; i < M; i++) {
            v.y[i] = st->y[i];
            v.lam[i] = st->lam[i];
            v.mu[i] = st->mu[i];
            v.s[i] = st->s[i];
        }
        v.z = st->z;
        v.zet = st->zet;
    }
    double s2 = q[0], m2 = q[1 + M];
    small_residual<M>(st, v, q + 1, s2, m2);
    const double resinew = sqrt(s2);
    const bool taken = k < tries && !(phase == kPhaseSearch && resinew > st->residunorm && itto + k + 1 < 50);
    const unsigned long long any = __ballot(taken);
    if (!any) {  // every candidate refused: the next pass goes on from here
        if (k == tries) {
            st->itto = itto + tries;
            st->steg = steg;
        }
        return;
    }
    if (k != __ffsll(any) - 1) return;
    if (phase == kPhaseSearch) {
        st->steg = steg;
        st->pending = 1;
#pragma unroll
        for (int i = 0; i < M; i++) {
            st->y[i] = v.y[i];
            st->lam[i] = v.lam[i];
            st->mu[i] = v.mu[i];
            st->s[i] = v.s[i];
        }
        st->z = v.z;
        st->zet = v.zet;
    }
#pragma unroll
    for (int i = 0; i < M; i++) st->gvec[i] = q[1 + i];
    st->residunorm = resinew;
    next_phase(st, m2);
}

// The subproblem's solution becomes the design: xold2 <- xold1 <- x <- solution (mmasub_g,
// mmaOpt.cu:1057-1059), rounded to FP32 for the caller.  out may be v.x0 itself.
template <int M>
__global__ __launch_bounds__(kMmaThreads) void k_mma_finish(MmaVars v, const MmaState* __restrict__ st,
                                                            double* __restrict__ xcur, double* __restrict__ xold1,
                                                            double* __restrict__ xold2, float* out) {
    const long j = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= v.n || st->status) return;
    const double x0 = (double)v.x0[j];
    MmaVar<M> a;
    a.load(v, j);
    double x = a.x;
    if (st->pending) {
        double dx, dxsi, deta, ia, ib;
        a.direction(st->lamo, st->dlam, st->epsd, dx, dxsi, deta, ia, ib);
        x += st->steg * dx;
    }
    xold2[j] = xold1[j];
    xold1[j] = x0;
    xcur[j] = x;
    out[j] = (float)x;
}

__global__ __launch_bounds__(kMmaThreads) void k_f32_to_f64(long n, const float* __restrict__ a,
                                                            double* __restrict__ b) {
    const long j = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < n) b[j] = (double)a[j];
}

__global__ __launch_bounds__(kMmaThreads) void k_fill(long n, double value, double* __restrict__ a) {
    const long j = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < n) a[j] = value;
}

unsigned nblk(long n) { return (unsigned)((n + kMmaThreads - 1) / kMmaThreads); }

}  // namespace

struct homo3d_mma {
    int m = 0;
    long n = 0;
    int nb = 0;  // workgroups of the per-variable passes
    double a0 = 1, a[kMmaMaxM], c[kMmaMaxM], d[kMmaMaxM];
    hipStream_t stream = nullptr;
    double *x = nullptr, *xmin = nullptr, *xmax = nullptr, *xold1 = nullptr, *xold2 = nullptr, *low = nullptr,
           *upp = nullptr, *xs = nullptr, *xsi = nullptr, *eta = nullptr, *part = nullptr;
    float *x0 = nullptr, *df = nullptr, *dg = nullptr;  // this step's design and gradients
    MmaState* st = nullptr;
    MmaState* seen[2] = {nullptr, nullptr};  // pinned copies of the state, one per round in flight
    hipEvent_t ev[2] = {nullptr, nullptr};
    bool initialised = false;
    int last_newton = 0;
    std::string err;
};

namespace {

int mma_err(homo3d_mma* h, int code, const char* msg) {
    if (h) h->err = msg;
    return code;
}

#define MMACHK(h, expr)                                                          \
    do {                                                                         \
        hipError_t e_ = (expr);                                                  \
        if (e_ != hipSuccess) return mma_err(h, HOMO3D_HIP_ERROR, hipGetErrorString(e_)); \
    } while (0)

void fill(homo3d_mma* h, double* a, double value) {
    hipLaunchKernelGGL(k_fill, dim3(nblk(h->n)), dim3(kMmaThreads), 0, h->stream, h->n, value, a);
}

// One round of the interior-point method: a Newton step with its line search's first pass, or a further
// search pass, or the residual of a new epsi; passes that the state does not call for return at once.
template <int M>
void launch_round(homo3d_mma* h, const MmaVars& v) {
    const dim3 g(h->nb), b(kMmaThreads), one(1), c(kMmaCtlThreads);
    const int nbs = std::min(h->nb, kMmaSearchBlocks);
    hipLaunchKernelGGL(k_mma_newton<M>, g, b, 0, h->stream, v, h->st, h->part);
    hipLaunchKernelGGL(k_mma_solve<M>, one, c, 0, h->stream, h->st, h->part, h->nb);
    hipLaunchKernelGGL(k_mma_length<M>, g, b, 0, h->stream, v, h->st, h->part);
    hipLaunchKernelGGL(k_mma_steplen<M>, one, c, 0, h->stream, h->st, h->part, h->nb);
    hipLaunchKernelGGL(k_mma_search<M>, dim3(nbs), b, 0, h->stream, v, h->st, h->part);
    hipLaunchKernelGGL(k_mma_accept<M>, one, c, 0, h->stream, h->st, h->part, nbs);
}

// Rounds queued between two looks at the state.
constexpr int kRounds = 4;

template <int M>
int mma_step(homo3d_mma* h, int itn, float* out) {
    const MmaVars v{h->n, h->x0, h->df, h->dg, h->low, h->upp, h->xmin, h->xmax, h->xs, h->xsi, h->eta};
    hipLaunchKernelGGL(k_mma_setup<M>, dim3(h->nb), dim3(kMmaThreads), 0, h->stream, v, itn, h->xold1, h->xold2, h->low,
                       h->upp, h->part);
    hipLaunchKernelGGL(k_mma_begin<M>, dim3(1), dim3(kMmaCtlThreads), 0, h->stream, h->st, h->part, h->nb);
    // The state is read back behind every kRounds rounds while the next ones are already queued (they
    // return at once when the method has ended).  8 values of epsi, at most kMmaNewton Newton steps each and
    // 50 trials a step bound the rounds.
    const int most = 8 * (kMmaNewton * (1 + 50 / kMmaCand + 1) + 1) / kRounds + 2;
    bool done = false;
    for (int k = 0; k < most && !done; k++) {
        for (int r = 0; r < kRounds; r++) launch_round<M>(h, v);
        MMACHK(h, hipGetLastError());
        MMACHK(h, hipMemcpyAsync(h->seen[k & 1], h->st, sizeof(MmaState), hipMemcpyDeviceToHost, h->stream));
        MMACHK(h, hipEventRecord(h->ev[k & 1], h->stream));
        if (k == 0) continue;
        MMACHK(h, hipEventSynchronize(h->ev[(k - 1) & 1]));
        done = h->seen[(k - 1) & 1]->phase == kPhaseDone;
    }
    hipLaunchKernelGGL(k_mma_finish<M>, dim3(nblk(h->n)), dim3(kMmaThreads), 0, h->stream, v, h->st, h->x, h->xold1,
                       h->xold2, out);
    MMACHK(h, hipGetLastError());
    MMACHK(h, hipMemcpyAsync(h->seen[0], h->st, sizeof(MmaState), hipMemcpyDeviceToHost, h->stream));
    return HOMO3D_OK;
}

// on_device < 0: classify the pointer (device or managed memory -> 1, anything else -> 0)
int resolve_on_device(const void* p, int on_device) {
    if (on_device >= 0) return on_device;
    hipPointerAttribute_t attr;
    if (hipPointerGetAttributes(&attr, p) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return (attr.type == hipMemoryTypeDevice || attr.type == hipMemoryTypeManaged) ? 1 : 0;
}

}  // namespace

extern "C" {

int homo3d_mma_create(int m, long n, double a0, double a, double c, double d, int device, homo3d_mma** out) {
    if (!out || m < 1 || m > kMmaMaxM || n < 1) return HOMO3D_BAD_ARG;
    *out = nullptr;
    homo3d_mma* h = new homo3d_mma();
    h->m = m;
    h->n = n;
    h->nb = (int)std::min<long>(kMmaBlocks, nblk(n));
    h->a0 = a0;
    for (int i = 0; i < kMmaMaxM; i++) {
        h->a[i] = a;
        h->c[i] = c;
        h->d[i] = d;
    }
    auto fail = [&](int code) {
        homo3d_mma_destroy(h);
        return code;
    };
    if (hipSetDevice(device) != hipSuccess) return fail(HOMO3D_HIP_ERROR);
    if (hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking) != hipSuccess) return fail(HOMO3D_HIP_ERROR);
    double** vecs[] = {&h->x, &h->xmin, &h->xmax, &h->xold1, &h->xold2, &h->low, &h->upp, &h->xs, &h->xsi, &h->eta};
    for (double** v : vecs)
        if (hipMalloc(v, sizeof(double) * n) != hipSuccess) return fail(HOMO3D_HIP_ERROR);
    if (hipMalloc(&h->x0, sizeof(float) * n) || hipMalloc(&h->df, sizeof(float) * n) ||
        hipMalloc(&h->dg, sizeof(float) * n * m) || hipMalloc(&h->part, sizeof(double) * h->nb * kMmaSums) ||
        hipMalloc(&h->st, sizeof(MmaState)) ||
        hipHostMalloc((void**)&h->seen[0], 2 * sizeof(MmaState), hipHostMallocDefault) ||
        hipEventCreateWithFlags(&h->ev[0], hipEventDisableTiming) ||
        hipEventCreateWithFlags(&h->ev[1], hipEventDisableTiming))
        return fail(HOMO3D_HIP_ERROR);
    h->seen[1] = h->seen[0] + 1;
    fill(h, h->xmin, 0.0);
    fill(h, h->xmax, 1.0);
    double* zeros[] = {h->xold1, h->xold2, h->low, h->upp};
    for (double* z : zeros) fill(h, z, 0.0);
    if (hipStreamSynchronize(h->stream) != hipSuccess) return fail(HOMO3D_HIP_ERROR);
    *out = h;
    return HOMO3D_OK;
}

int homo3d_mma_destroy(homo3d_mma* h) {
    if (!h) return HOMO3D_OK;
    // teardown: errors are not actionable here, so they are ignored
    if (h->stream) (void)hipStreamSynchronize(h->stream);
    void* ptrs[] = {h->x, h->xmin, h->xmax, h->xold1, h->xold2, h->low, h->upp, h->xs, h->xsi, h->eta,
                    h->part, h->x0, h->df, h->dg, h->st};
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    if (h->seen[0]) (void)hipHostFree(h->seen[0]);
    for (hipEvent_t e : h->ev)
        if (e) (void)hipEventDestroy(e);
    if (h->stream) (void)hipStreamDestroy(h->stream);
    delete h;
    return HOMO3D_OK;
}

const char* homo3d_mma_last_error(const homo3d_mma* h) { return h ? h->err.c_str() : "null handle"; }

// MMAOptimizer::setBound(float xmin, float xmax) (mmaOptimizer.cu:53-57)
int homo3d_mma_set_bound(homo3d_mma* h, double xmin, double xmax) {
    if (!h || !(xmax > xmin)) return HOMO3D_BAD_ARG;
    fill(h, h->xmin, xmin);
    fill(h, h->xmax, xmax);
    MMACHK(h, hipStreamSynchronize(h->stream));
    return HOMO3D_OK;
}

// MMAOptimizer::setBound(float* xmin, float* xmax) (mmaOptimizer.h:30): per-variable bounds, n floats
// each, in host (on_device = 0) or device memory (1); -1 classifies the pointers.
int homo3d_mma_set_bounds(homo3d_mma* h, const float* xmin, const float* xmax, int on_device) {
    if (!h || !xmin || !xmax) return HOMO3D_BAD_ARG;
    on_device = resolve_on_device(xmin, on_device);
    if (on_device) {
        hipLaunchKernelGGL(k_f32_to_f64, dim3(nblk(h->n)), dim3(kMmaThreads), 0, h->stream, h->n, xmin, h->xmin);
        hipLaunchKernelGGL(k_f32_to_f64, dim3(nblk(h->n)), dim3(kMmaThreads), 0, h->stream, h->n, xmax, h->xmax);
        MMACHK(h, hipStreamSynchronize(h->stream));
        return HOMO3D_OK;
    }
    std::vector<double> lo(h->n), hi(h->n);
    for (long i = 0; i < h->n; i++) {
        if (!(xmax[i] >= xmin[i])) return mma_err(h, HOMO3D_BAD_ARG, "setBound: xmax < xmin");
        lo[i] = xmin[i];
        hi[i] = xmax[i];
    }
    MMACHK(h, hipMemcpyAsync(h->xmin, lo.data(), sizeof(double) * h->n, hipMemcpyHostToDevice, h->stream));
    MMACHK(h, hipMemcpyAsync(h->xmax, hi.data(), sizeof(double) * h->n, hipMemcpyHostToDevice, h->stream));
    MMACHK(h, hipStreamSynchronize(h->stream));
    return HOMO3D_OK;
}

// One MMA step (MMAOptimizer::update, mmaOptimizer.cu:61-77): x (n floats) is updated in place.
// dfdx: n floats; gval: m floats (host); dgdx: m pointers to n floats.  Arrays are device
// pointers when on_device != 0, host pointers otherwise.
int homo3d_mma_update(homo3d_mma* h, int itn, float* x, const float* dfdx, const float* gval, const float* const* dgdx,
                      int on_device) {
    if (!h || !x || !dfdx || !gval || !dgdx) return HOMO3D_BAD_ARG;
    on_device = resolve_on_device(x, on_device);
    const int m = h->m;
    const long n = h->n;
    hipStream_t s = h->stream;
    const hipMemcpyKind kin = on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice;
    MMACHK(h, hipMemcpyAsync(h->x0, x, sizeof(float) * n, kin, s));
    MMACHK(h, hipMemcpyAsync(h->df, dfdx, sizeof(float) * n, kin, s));
    for (int i = 0; i < m; i++)
        MMACHK(h, hipMemcpyAsync(h->dg + (size_t)i * n, dgdx[i], sizeof(float) * n, kin, s));
    if (!h->initialised) {
        hipLaunchKernelGGL(k_f32_to_f64, dim3(nblk(n)), dim3(kMmaThreads), 0, s, n, h->x0, h->xold1);
        hipLaunchKernelGGL(k_f32_to_f64, dim3(nblk(n)), dim3(kMmaThreads), 0, s, n, h->x0, h->xold2);
        h->initialised = true;
    }
    MmaState st{};
    st.a0 = h->a0;
    for (int i = 0; i < m; i++) {
        st.a[i] = h->a[i];
        st.c[i] = h->c[i];
        st.d[i] = h->d[i];
        st.gval[i] = (double)gval[i];
    }
    *h->seen[0] = st;
    MMACHK(h, hipMemcpyAsync(h->st, h->seen[0], sizeof(MmaState), hipMemcpyHostToDevice, s));
    // the result leaves from x0 when the caller's array is in host memory
    float* out = on_device ? x : h->x0;
    const int rc = m == 1 ? mma_step<1>(h, itn, out)
                          : (m == 2 ? mma_step<2>(h, itn, out) : (m == 3 ? mma_step<3>(h, itn, out) : mma_step<4>(h, itn, out)));
    if (rc) return rc;
    MMACHK(h, hipStreamSynchronize(s));
    h->last_newton = h->seen[0]->itera;
    if (h->seen[0]->status) return mma_err(h, HOMO3D_DIVERGED, "singular MMA Newton system");
    if (!on_device) {
        MMACHK(h, hipMemcpyAsync(x, h->x0, sizeof(float) * n, hipMemcpyDeviceToHost, s));
        MMACHK(h, hipStreamSynchronize(s));
    }
    return HOMO3D_OK;
}

int homo3d_mma_state(homo3d_mma* h, double* x, double* low, double* upp, int* newton_iters) {
    if (!h) return HOMO3D_BAD_ARG;
    const size_t b = sizeof(double) * h->n;
    if (x) MMACHK(h, hipMemcpyAsync(x, h->x, b, hipMemcpyDeviceToHost, h->stream));
    if (low) MMACHK(h, hipMemcpyAsync(low, h->low, b, hipMemcpyDeviceToHost, h->stream));
    if (upp) MMACHK(h, hipMemcpyAsync(upp, h->upp, b, hipMemcpyDeviceToHost, h->stream));
    MMACHK(h, hipStreamSynchronize(h->stream));
    if (newton_iters) *newton_iters = h->last_newton;
    return HOMO3D_OK;
}

}  // extern "C"
