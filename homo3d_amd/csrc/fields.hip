// Density utilities on pitched lexicographic n^3 arrays: radial filters and their adjoint, projection,
// elementwise maps and symmetry projection.  All of them stream a few FP32 fields, so the
// kernels read the caller's arrays where they lie and touch each value once; arithmetic is FP64, rounded
// to FP32, unless noted.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "fields.h"
#include "kernels.h"

namespace homo3d {

namespace {

constexpr int kThreads = 256;

inline unsigned nblk(size_t work, int bs = kThreads) { return (unsigned)((work + bs - 1) / bs); }

// ---------------------------------------------------------------------------------------------
// Elementwise maps.  Unpitched arrays on 16-byte boundaries run four values a thread over the whole
// array (192^3: 10-14 us, 5 TB/s or more; 17-36 us with a 64-bit division of the cell index in each
// thread); others one value a thread, a wave along each row.
// ---------------------------------------------------------------------------------------------
template <typename F>
__global__ __launch_bounds__(kThreads) void k_map4(size_t quads, F f) {
    const size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (i < quads) f.quad(i);
}

template <typename F>
__global__ __launch_bounds__(kThreads) void k_map_rows(int n, int pitch, F f) {
    const int x = (int)(blockIdx.x * 64 + (threadIdx.x & 63));
    if (x >= n) return;
    const int rows = n * n;
    for (int row = (int)(blockIdx.y * 4 + (threadIdx.x >> 6)); row < rows; row += (int)gridDim.y * 4)
        f.one((size_t)x + (size_t)row * pitch);
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

template <typename F>
void launch_map(hipStream_t s, int n, int pitch, bool vec, const F& f) {
    const size_t N = (size_t)n * n * n;
    if (vec && pitch == n && N % 4 == 0)
        hipLaunchKernelGGL(k_map4<F>, dim3(nblk(N / 4)), dim3(kThreads), 0, s, N / 4, f);
    else
        hipLaunchKernelGGL(k_map_rows<F>, dim3((n + 63) / 64, std::min((n * n + 3) / 4, 32768)), dim3(kThreads), 0, s, n,
                           pitch, f);
}

__device__ __forceinline__ float4 ld4(const float* p, size_t i) { return reinterpret_cast<const float4*>(p)[i]; }
__device__ __forceinline__ void st4(float* p, size_t i, float4 v) { reinterpret_cast<float4*>(p)[i] = v; }

// out = op(a), or op(a, b); the arrays may be one and the same (each value is read before it is written)
template <typename Op>
struct Map1 {
    const float* a;
    float* out;
    Op op;
    __device__ void one(size_t i) const { out[i] = op(a[i]); }
    __device__ void quad(size_t i) const {
        const float4 v = ld4(a, i);
        st4(out, i, make_float4(op(v.x), op(v.y), op(v.z), op(v.w)));
    }
};
template <typename Op>
struct Map2 {
    const float *a, *b;
    float* out;
    Op op;
    __device__ void one(size_t i) const { out[i] = op(a[i], b[i]); }
    __device__ void quad(size_t i) const {
        const float4 v = ld4(a, i), w = ld4(b, i);
        st4(out, i, make_float4(op(v.x, w.x), op(v.y, w.y), op(v.z, w.z), op(v.w, w.w)));
    }
};

// sgm projection (sgm_exp_t, AutoDiff.h:808-823): y = 1 / (1 + exp(-k (x - c))); backward gx = gy k y (1 - y).
struct SgmOp {
    double k, c;
    __device__ float operator()(float x) const { return (float)(1.0 / (1.0 + exp(-k * ((double)x - c)))); }
};
struct SgmBackOp {
    double k;
    __device__ float operator()(float y, float gy) const {
        const double yv = y;
        return (float)((double)gy * k * yv * (1.0 - yv));
    }
};

// x = rho^p and its chain rule (rho.pow(p) of the reference's expression templates), FP32.  p = 3 is
// evaluated as r * r * r and 3 r r d, the products the host loops of the drivers form.
struct PowOp {
    float p;
    __device__ float operator()(float r) const { return p == 3.f ? r * r * r : powf(r, p); }
};
struct PowGradOp {
    float p;
    __device__ float operator()(float r, float d) const {
        return p == 3.f ? 3.f * r * r * d : p * powf(r, p - 1.f) * d;
    }
};

// ---------------------------------------------------------------------------------------------
// Radial filters over the (2h+1)^3 box with normalised weights w:
//   conv       out(i) = sum_off w(off) in(i + off) / W(i)            (TensorExpression.cuh:288-330)
//   adjoint    out(j) = sum_off w(off) in(j - off) / W(j - off)      (TensorExpression.cuh:331-366)
//   sensitivity filter  out(i) = sum_off w(off) sens rho (i + off) / (W(i) rho(i))
//                                                                   (filterSens_kernel, OCOptimizer.cu:76-153)
// W(i): the sum of w over the neighbours inside the grid (all of them when periodic).  FP64 sums.
//
// The taps, not the bytes, bound a filter that reads its neighbours from memory (125 gathers a cell for
// h = 2: 2.33 ms at 192^3, 0.06 ms of traffic).  Here a workgroup stages the FP64 source values of a
// 32 x 8 x 8 tile and its halo in LDS (41 KB for h = 2: three workgroups a CU; 60 KB for h = 3) and each
// thread forms four x-neighbouring cells at two z, so a row of 4 + 2h staged values serves 4 (2h + 1)
// products.  The taps are added in the order of the box, as the general kernel does.  Periodic, h = 2,
// 192^3: conv 0.108 ms (2.33), adjoint 0.110 ms (2.66, and 2.33 more for the W of every cell, which now
// comes from one value, or a table of (2h + 1)^3 at a wall): 885 M FP64 products at 8.2 G a ms.
// ---------------------------------------------------------------------------------------------
constexpr int kBoxTX = 32, kBoxTY = 8, kBoxTZ = 8;

enum { kBoxConv = 0, kBoxAdjoint = 1, kBoxSens = 2 };

template <int H>
struct BoxWeights {
    double w[(2 * H + 1) * (2 * H + 1) * (2 * H + 1)];
};

// The position classes of a non-periodic axis: distance to the nearer wall, capped at h on both sides
// (2h + 1 classes; with fewer cells than that, the position itself).
__device__ __forceinline__ int box_class(int p, int n, int h) {
    if (n < 2 * h + 1) return p;
    return p < h ? p : (p >= n - h ? 2 * h - (n - 1 - p) : h);
}

// W of every class triple, summed over the in-grid taps in box order: table[(cz (2h+1) + cy) (2h+1) + cx].
template <int H>
__global__ __launch_bounds__(64) void k_box_wsum(int n, BoxWeights<H> bw, double* __restrict__ table) {
    constexpr int S = 2 * H + 1;
    const int t = (int)(blockIdx.x * 64 + threadIdx.x);
    if (t >= S * S * S) return;
    const int c[3] = {t % S, t / S % S, t / (S * S)};
    int p[3];
    bool used = true;
    for (int k = 0; k < 3; k++) {
        p[k] = n < S ? c[k] : (c[k] <= H ? c[k] : n - 1 - (2 * H - c[k]));
        used = used && p[k] < n;
    }
    double ws = 0.0;
    if (used)
        for (int i = 0; i < S * S * S; i++) {
            const int x = p[0] + i % S - H, y = p[1] + i / S % S - H, z = p[2] + i / (S * S) - H;
            if (x >= 0 && x < n && y >= 0 && y < n && z >= 0 && z < n) ws += bw.w[i];
        }
    table[t] = ws;
}

template <int H, int MODE, bool PERIODIC>
__global__ __launch_bounds__(kThreads, H == 3 ? 2 : 3) void k_box_filter(int n, int pitch, BoxWeights<H> bw, double wtotal,
                                                         const double* __restrict__ table,
                                                         const float* __restrict__ in, const float* __restrict__ rho,
                                                         float* __restrict__ out) {
    constexpr int S = 2 * H + 1, BX = kBoxTX + 2 * H, BY = kBoxTY + 2 * H, BZ = kBoxTZ + 2 * H;
    __shared__ double v[BZ * BY * BX];
    const int x0 = (int)blockIdx.x * kBoxTX, y0 = (int)blockIdx.y * kBoxTY, z0 = (int)blockIdx.z * kBoxTZ;
    for (int t = threadIdx.x; t < BX * BY * BZ; t += kThreads) {
        int x = x0 + t % BX - H, y = y0 + t / BX % BY - H, z = z0 + t / (BX * BY) - H;
        // positions further than h outside the grid belong to cells past its end only
        if (PERIODIC) {
            x = x < 0 ? x + n : (x >= n && x < n + H ? x - n : x);
            y = y < 0 ? y + n : (y >= n && y < n + H ? y - n : y);
            z = z < 0 ? z + n : (z >= n && z < n + H ? z - n : z);
        }
        double val = 0.0;
        if (x >= 0 && x < n && y >= 0 && y < n && z >= 0 && z < n) {
            const size_t id = (size_t)x + ((size_t)y + (size_t)z * n) * pitch;
            val = (double)in[id];
            if constexpr (MODE == kBoxSens) val *= (double)rho[id];
            if constexpr (MODE == kBoxAdjoint)
                val /= PERIODIC ? (double)(float)wtotal
                                : (double)(float)table[(box_class(z, n, H) * S + box_class(y, n, H)) * S +
                                                       box_class(x, n, H)];
        }
        v[t] = val;
    }
    __syncthreads();
    const int tx = 4 * ((int)threadIdx.x & 7), ty = ((int)threadIdx.x >> 3) & 7;
    const int y = y0 + ty;
#pragma unroll 1
    for (int tz = (int)threadIdx.x >> 6; tz < kBoxTZ; tz += 4) {
        const int z = z0 + tz;
        double sum[4] = {0.0, 0.0, 0.0, 0.0};
        // tap (dx, dy, dz) in box order; the adjoint reads at minus the offset
#pragma unroll 1
        for (int dz = 0; dz < S; dz++) {
            const double* w = bw.w + dz * S * S;
#pragma unroll
            for (int dy = 0; dy < S; dy++) {
                const double* row = MODE == kBoxAdjoint ? v + ((tz + 2 * H - dz) * BY + (ty + 2 * H - dy)) * BX + tx
                                                        : v + ((tz + dz) * BY + (ty + dy)) * BX + tx;
                double a[4 + 2 * H];
#pragma unroll
                for (int k = 0; k < 4 + 2 * H; k++) a[k] = row[k];
#pragma unroll
                for (int dx = 0; dx < S; dx++)
#pragma unroll
                    for (int k = 0; k < 4; k++)
                        sum[k] = fma(w[dy * S + dx], a[MODE == kBoxAdjoint ? k + 2 * H - dx : k + dx], sum[k]);
            }
        }
        if (y >= n || z >= n) continue;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int x = x0 + tx + k;
            if (x >= n) continue;
            const size_t id = (size_t)x + ((size_t)y + (size_t)z * n) * pitch;
            double r = sum[k];
            if constexpr (MODE != kBoxAdjoint) {
                const double ws = PERIODIC ? wtotal
                                           : table[(box_class(z, n, H) * S + box_class(y, n, H)) * S +
                                                   box_class(x, n, H)];
                r = MODE == kBoxSens ? sum[k] / (ws * (double)rho[id]) : sum[k] / ws;
            }
            out[id] = (float)r;
        }
    }
}

// Boxes wider than the staged kernels take (h = 0, h > 3, or a grid smaller than the half-width): one
// cell a thread, the neighbours from memory.
__global__ __launch_bounds__(kThreads) void k_oc_filter(int n, int pitch, int h, int periodic,
                                                        const float* __restrict__ wk, const float* __restrict__ sens,
                                                        const float* __restrict__ rho, float* __restrict__ out) {
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long N = (long)n * n * n;
    if (e >= N) return;
    const int p[3] = {(int)(e % n), (int)((e / n) % n), (int)(e / ((long)n * n))};
    const int side = 2 * h + 1;
    double sum = 0.0, ws = 0.0;
    for (int i = 0; i < side * side * side; i++) {
        int q[3] = {p[0] + i % side - h, p[1] + (i / side) % side - h, p[2] + i / (side * side) - h};
        bool inb = true;
        for (int k = 0; k < 3; k++) {
            if (periodic) q[k] = ((q[k] % n) + n) % n;
            if (q[k] < 0 || q[k] >= n) inb = false;
        }
        if (!inb) continue;
        const size_t id = q[0] + ((size_t)q[1] + (size_t)q[2] * n) * pitch;
        sum += (double)sens[id] * (double)rho[id] * (double)wk[i];
        ws += (double)wk[i];
    }
    const size_t me = p[0] + ((size_t)p[1] + (size_t)p[2] * n) * pitch;
    out[me] = (float)(sum / (ws * (double)rho[me]));
}

// conv; W is written when wsum is not null.
__global__ __launch_bounds__(kThreads) void k_conv_filter(int n, int pitch, int h, int periodic,
                                                          const float* __restrict__ wk, const float* __restrict__ in,
                                                          float* __restrict__ out, float* __restrict__ wsum) {
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long N = (long)n * n * n;
    if (e >= N) return;
    const int p[3] = {(int)(e % n), (int)((e / n) % n), (int)(e / ((long)n * n))};
    const int side = 2 * h + 1;
    double sum = 0.0, ws = 0.0;
    for (int i = 0; i < side * side * side; i++) {
        int q[3] = {p[0] + i % side - h, p[1] + (i / side) % side - h, p[2] + i / (side * side) - h};
        bool inb = true;
        for (int k = 0; k < 3; k++) {
            if (periodic) q[k] = ((q[k] % n) + n) % n;
            if (q[k] < 0 || q[k] >= n) inb = false;
        }
        if (!inb) continue;
        sum += (double)wk[i] * (double)in[q[0] + ((size_t)q[1] + (size_t)q[2] * n) * pitch];
        ws += (double)wk[i];
    }
    const size_t me = p[0] + ((size_t)p[1] + (size_t)p[2] * n) * pitch;
    out[me] = (float)(sum / ws);
    if (wsum) wsum[me] = (float)ws;
}

// its adjoint; wsum from k_conv_filter
__global__ __launch_bounds__(kThreads) void k_conv_filter_back(int n, int pitch, int h, int periodic,
                                                               const float* __restrict__ wk,
                                                               const float* __restrict__ dout,
                                                               const float* __restrict__ wsum,
                                                               float* __restrict__ din) {
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long N = (long)n * n * n;
    if (e >= N) return;
    const int p[3] = {(int)(e % n), (int)((e / n) % n), (int)(e / ((long)n * n))};
    const int side = 2 * h + 1;
    double sum = 0.0;
    for (int i = 0; i < side * side * side; i++) {
        int q[3] = {p[0] - (i % side - h), p[1] - ((i / side) % side - h), p[2] - (i / (side * side) - h)};
        bool inb = true;
        for (int k = 0; k < 3; k++) {
            if (periodic) q[k] = ((q[k] % n) + n) % n;
            if (q[k] < 0 || q[k] >= n) inb = false;
        }
        if (!inb) continue;
        const size_t id = q[0] + ((size_t)q[1] + (size_t)q[2] * n) * pitch;
        sum += (double)wk[i] * (double)dout[id] / (double)wsum[id];
    }
    din[p[0] + ((size_t)p[1] + (size_t)p[2] * n) * pitch] = (float)sum;
}

template <int H, int MODE>
void box_filter(hipStream_t s, int n, int pitch, int periodic, const float* wk, double* table, const float* in,
                const float* rho, float* out) {
    constexpr int S = 2 * H + 1;
    BoxWeights<H> bw;
    double total = 0.0;
    for (int i = 0; i < S * S * S; i++) total += bw.w[i] = (double)wk[i];
    const dim3 g((n + kBoxTX - 1) / kBoxTX, (n + kBoxTY - 1) / kBoxTY, (n + kBoxTZ - 1) / kBoxTZ);
    if (periodic) {
        hipLaunchKernelGGL((k_box_filter<H, MODE, true>), g, dim3(kThreads), 0, s, n, pitch, bw, total, table, in, rho, out);
        return;
    }
    hipLaunchKernelGGL(k_box_wsum<H>, dim3(nblk(S * S * S, 64)), dim3(64), 0, s, n, bw, table);
    hipLaunchKernelGGL((k_box_filter<H, MODE, false>), g, dim3(kThreads), 0, s, n, pitch, bw, total, table, in, rho, out);
}

template <int MODE>
void box_filter_pick(hipStream_t s, int n, int pitch, int h, int periodic, const float* wk, double* table,
                     const float* in, const float* rho, float* out) {
    switch (h) {
        case 1: box_filter<1, MODE>(s, n, pitch, periodic, wk, table, in, rho, out); break;
        case 2: box_filter<2, MODE>(s, n, pitch, periodic, wk, table, in, rho, out); break;
        default: box_filter<3, MODE>(s, n, pitch, periodic, wk, table, in, rho, out); break;
    }
}

// Symmetry projection (symetrize_tensor_kernel, TensorExpression.cuh:72-262): every cell of an orbit
// receives the FP64 average over the group applied to the orbit's smallest-index member.  The thread of that
// member reads the orbit and writes it, in place (orbits do not meet); the others find a smaller image and
// stop, half of them at each mirror axis.  Bound by the scattered images of the permuted axes.  Every cell
// finding its smallest member and gathering the orbit itself (48 times the reads, out of place, copied back)
// took 217 us a call at 128^3 and 45 at 64^3, and the copies; 58 and 18 now.
__global__ __launch_bounds__(kThreads) void k_symmetrize(int n, int pitch, uint64_t group, double count,
                                                         float* __restrict__ field) {
    const int x = (int)blockIdx.x * 64 + ((int)threadIdx.x & 63), y = (int)blockIdx.y * 4 + ((int)threadIdx.x >> 6);
    const int z = (int)blockIdx.z;
    if (x >= n || y >= n) return;
    const int p[3] = {x, y, z}, m[3] = {n - 1 - x, n - 1 - y, n - 1 - z};
    const uint64_t row = (uint64_t)n, slab = row * row, self = x + row * y + slab * z;
    const uint64_t prow = (uint64_t)pitch, pslab = prow * row;
    // index of image (k, f) with rows of r and slabs of s elements
    auto image = [&](int k, int f, uint64_t r, uint64_t sl) {
        const int *a = kSymPerm[k];
        return (uint64_t)(f & 1 ? m : p)[a[0]] + r * (uint64_t)(f & 2 ? m : p)[a[1]] + sl * (uint64_t)(f & 4 ? m : p)[a[2]];
    };
    bool first = true;
#pragma unroll
    for (int k = 0; k < 6; k++) {
        if (!(group >> (8 * k) & 255)) continue;
#pragma unroll
        for (int f = 0; f < 8; f++) first = first && (!(group >> (8 * k + f) & 1) || image(k, f, row, slab) >= self);
        if (!first) return;
    }
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < 6; k++) {
        if (!(group >> (8 * k) & 255)) continue;
        float v[8];
#pragma unroll
        for (int f = 0; f < 8; f++) v[f] = field[image(k, f, prow, pslab)];
#pragma unroll
        for (int f = 0; f < 8; f++)
            if (group >> (8 * k + f) & 1) s += (double)v[f];
    }
    const float mean = (float)(s / count);
#pragma unroll
    for (int k = 0; k < 6; k++) {
        if (!(group >> (8 * k) & 255)) continue;
#pragma unroll
        for (int f = 0; f < 8; f++)
            if (group >> (8 * k + f) & 1) field[image(k, f, prow, pslab)] = mean;
    }
}

}  // namespace

int box_filter_ok(int n, int h) { return h >= 1 && h <= 3 && n >= h; }

void launch_box_conv(hipStream_t s, int n, int pitch, int h, int periodic, const float* wk, double* table,
                     const float* in, float* out) {
    box_filter_pick<kBoxConv>(s, n, pitch, h, periodic, wk, table, in, nullptr, out);
}

void launch_box_adjoint(hipStream_t s, int n, int pitch, int h, int periodic, const float* wk, double* table,
                        const float* in, float* out) {
    box_filter_pick<kBoxAdjoint>(s, n, pitch, h, periodic, wk, table, in, nullptr, out);
}

void launch_box_sens(hipStream_t s, int n, int pitch, int h, int periodic, const float* wk, double* table,
                     const float* sens, const float* rho, float* out) {
    box_filter_pick<kBoxSens>(s, n, pitch, h, periodic, wk, table, sens, rho, out);
}

void launch_oc_filter(hipStream_t s, int n, int pitch, int h, int periodic, const float* wk, const float* sens,
                      const float* rho, float* out) {
    const size_t N = (size_t)n * n * n;
    hipLaunchKernelGGL(k_oc_filter, dim3(nblk(N)), dim3(kThreads), 0, s, n, pitch, h, periodic, wk, sens, rho, out);
}

void launch_conv_filter(hipStream_t s, int n, int pitch, int h, int periodic, const float* wk, const float* in,
                        float* out, float* wsum) {
    const size_t N = (size_t)n * n * n;
    hipLaunchKernelGGL(k_conv_filter, dim3(nblk(N)), dim3(kThreads), 0, s, n, pitch, h, periodic, wk, in, out, wsum);
}

void launch_conv_filter_back(hipStream_t s, int n, int pitch, int h, int periodic, const float* wk, const float* dout,
                             const float* wsum, float* din) {
    const size_t N = (size_t)n * n * n;
    hipLaunchKernelGGL(k_conv_filter_back, dim3(nblk(N)), dim3(kThreads), 0, s, n, pitch, h, periodic, wk, dout, wsum, din);
}

void launch_sgm(hipStream_t s, int n, int pitch, double k, double c, const float* x, float* y) {
    launch_map(s, n, pitch, aligned16(x) && aligned16(y), Map1<SgmOp>{x, y, {k, c}});
}

void launch_sgm_back(hipStream_t s, int n, int pitch, double k, const float* y, const float* gy, float* gx) {
    launch_map(s, n, pitch, aligned16(y) && aligned16(gy) && aligned16(gx), Map2<SgmBackOp>{y, gy, gx, {k}});
}

void launch_density_pow(hipStream_t s, int n, int pitch, float p, const float* rho, float* x) {
    launch_map(s, n, pitch, aligned16(rho) && aligned16(x), Map1<PowOp>{rho, x, {p}});
}

void launch_density_pow_grad(hipStream_t s, int n, int pitch, float p, const float* rho, const float* dx, float* drho) {
    launch_map(s, n, pitch, aligned16(rho) && aligned16(dx) && aligned16(drho), Map2<PowGradOp>{rho, dx, drho, {p}});
}

void launch_symmetrize(hipStream_t s, int n, int pitch, uint64_t group, float* field) {
    hipLaunchKernelGGL(k_symmetrize, dim3(nblk(n, 64), nblk(n, 4), n), dim3(kThreads), 0, s, n, pitch, group,
                       (double)__builtin_popcountll(group), field);
}

}  // namespace homo3d
