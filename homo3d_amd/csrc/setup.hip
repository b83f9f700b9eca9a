// What a density update prepares: the Galerkin stencils of the coarse levels
// (restrict_stencil_otf_aos_kernel_1, grid_ex.cu:936-1061; restrict_stencil_aos_kernel_1,
// grid_ex.cu:1065-1160; pinned-origin rows, grid.cpp:1184-1325) and the coarsest level's dense FP64
// inverse and its application (in place of the host solve of grid.cpp:349-424).
//
// All but the first product of a large grid are small: what bounds them is the length of the chain of
// dependent loads in a thread and the number of launches, not bytes or arithmetic.  The kernels split the
// work until each thread has some ten to a hundred independent loads.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.h"
#include "level.h"

namespace homo3d {

namespace {

// Level-1 stencil away from the pinned origin: st[V][D] = sum_{c} w_{2V+c} G[c][D], c in {-2..1}^3.
// G (64 x 27 x 9) is the density-independent table of P-weighted KE blocks.  A thread forms ND of the 27
// directions (blockIdx.y selects them) from the 64 cell weights it loads first: one direction where the
// level is small (27 times the threads: 142 -> 27 us at n = 32), nine or all where the threads fill the GPU.
// T = double: sums of FP64 blocks, rounded once.  A row of the operator sums to zero over its neighbours,
// but a table rounded to FP32 leaves the same small remainder in every row, and all rows' remainders
// together disturb the one weak mode of the coarsest system (its solution was 1e-4 off at 28^3, with
// rounded sums 4e-6).  T = float from level-1 grids above 64^3, where the FP64 table costs more scalar
// loads than the sums hide (n = 256: 0.98 ms, 1.74 in FP64).
template <int ND, typename T, typename SO>
__global__ __launch_bounds__(256) void k_galerkin_fine(Lay Lf, Lay Lc, const T* __restrict__ G,
                                                       const float* __restrict__ w, SO* __restrict__ stc,
                                                       float clamp) {
    const int nf = Lf.n;
    const size_t Nc = (size_t)Lc.n * Lc.n * Lc.n;
    int X, Y, Z;
    uint32_t V;
    if (!coarse_lex_vertex(Lc, X, Y, Z, V)) return;
    float wc[64];
#pragma unroll
    for (int c = 0; c < 64; c++) {
        int cx = 2 * X + (c & 3) - 2, cy = 2 * Y + ((c >> 2) & 3) - 2, cz = 2 * Z + (c >> 4) - 2;
        cx = cx < 0 ? cx + nf : (cx >= nf ? cx - nf : cx);
        cy = cy < 0 ? cy + nf : (cy >= nf ? cy - nf : cy);
        cz = cz < 0 ? cz + nf : (cz >= nf ? cz - nf : cz);
        wc[c] = w[Lf.idx(cx, cy, cz)];
    }
    for (int D = (int)blockIdx.y * ND; D < ((int)blockIdx.y + 1) * ND; D++) {
        const int Dx = D % 3 - 1, Dy = D / 3 % 3 - 1, Dz = D / 9 - 1;
        T S[9];
#pragma unroll
        for (int k = 0; k < 9; k++) S[k] = T(0);
#pragma unroll
        for (int c = 0; c < 64; c++) {
            // cell offset o from 2V per axis (-2..1): G[c][D] is zero unless the cell also touches the
            // support of V + D, i.e. o >= 0 where D is +1 and o < 0 where D is -1 (a wave-uniform test:
            // 8 to 64 of the 64 cells per direction, 512 of 1728 in all)
            const int ox = (c & 3) - 2, oy = ((c >> 2) & 3) - 2, oz = (c >> 4) - 2;
            if ((Dx > 0 && ox < 0) || (Dx < 0 && ox >= 0) || (Dy > 0 && oy < 0) || (Dy < 0 && oy >= 0) ||
                (Dz > 0 && oz < 0) || (Dz < 0 && oz >= 0))
                continue;
            const T* g = G + (c * 27 + D) * 9;
            const T we = (T)wc[c];
#pragma unroll
            for (int k = 0; k < 9; k++) S[k] = fma(we, g[k], S[k]);
        }
        if (D == 13) {
#pragma unroll
            for (int k = 0; k < 9; k += 4)
                if (fabs(S[k]) < (T)clamp) S[k] = (T)clamp;
        }
#pragma unroll
        for (int k = 0; k < 9; k++) StencilIO<SO>::put(stc, Nc, V, D * 9 + k, (float)S[k]);
    }
}

// Level-1 stencil of the 27 coarse vertices around the pinned origin: node pairs touching the origin
// contribute identity when they are the same node and nothing otherwise.  One wave per vertex and
// direction, a lane per cell offset (a thread per pair walked all 64 cells by itself: 405 us).
template <typename SO>
__global__ __launch_bounds__(64) void k_galerkin_fine_pin(Lay Lf, Lay Lc, const double* __restrict__ ke,
                                                          const float* __restrict__ w, SO* __restrict__ stc,
                                                          float clamp) {
    const int nf = Lf.n, nc = Lc.n;
    const size_t Nc = (size_t)nc * nc * nc;
    const int vi = (int)blockIdx.x / 27, D = (int)blockIdx.x % 27;  // (vi%3-1, vi/3%3-1, vi/9-1) around the origin
    const int X = (vi % 3) - 1, Y = (vi / 3 % 3) - 1, Z = (vi / 9) - 1;
    const int Dx = D % 3 - 1, Dy = D / 3 % 3 - 1, Dz = D / 9 - 1;
    const int c = (int)threadIdx.x;
    const int ox = (c & 3) - 2, oy = ((c >> 2) & 3) - 2, oz = (c >> 4) - 2;  // cell offset from 2V
    const int cx = 2 * X + ox, cy = 2 * Y + oy, cz = 2 * Z + oz;
    const double we = (double)w[Lf.idx((cx % nf + nf) % nf, (cy % nf + nf) % nf, (cz % nf + nf) % nf)];
    double S[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    // only the cells in the supports of both V and V + D contribute (as in k_galerkin_fine)
    const bool in = !((Dx > 0 && ox < 0) || (Dx < 0 && ox >= 0) || (Dy > 0 && oy < 0) || (Dy < 0 && oy >= 0) ||
                      (Dz > 0 && oz < 0) || (Dz < 0 && oz >= 0));
    for (int a = 0; in && a < 8; a++) {
        const float wa = hat(ox + (a & 1)) * hat(oy + ((a >> 1) & 1)) * hat(oz + (a >> 2));
        if (wa == 0.f) continue;
        const bool pa = (cx + (a & 1)) % nf == 0 && (cy + ((a >> 1) & 1)) % nf == 0 && (cz + (a >> 2)) % nf == 0;
        for (int b = 0; b < 8; b++) {
            const float wb = hat(ox + (b & 1) - 2 * Dx) * hat(oy + ((b >> 1) & 1) - 2 * Dy) * hat(oz + (b >> 2) - 2 * Dz);
            if (wb == 0.f) continue;
            const bool pb = (cx + (b & 1)) % nf == 0 && (cy + ((b >> 1) & 1)) % nf == 0 && (cz + (b >> 2)) % nf == 0;
            if (pa || pb) {
                if (a == b) {
                    S[0] += (double)(wa * wb);
                    S[4] += (double)(wa * wb);
                    S[8] += (double)(wa * wb);
                }
            } else {
#pragma unroll
                for (int k = 0; k < 9; k++) S[k] += (double)(wa * wb) * we * ke[(3 * a + k / 3) * 24 + 3 * b + k % 3];
            }
        }
    }
#pragma unroll
    for (int k = 0; k < 9; k++)
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) S[k] += __shfl_xor(S[k], off, 64);
    if (D == 13) {
        if (fabs(S[0]) < (double)clamp) S[0] = clamp;
        if (fabs(S[4]) < (double)clamp) S[4] = clamp;
        if (fabs(S[8]) < (double)clamp) S[8] = clamp;
    }
    if (c != 0) return;
    const uint32_t V = Lc.idx((X + nc) % nc, (Y + nc) % nc, (Z + nc) % nc);
#pragma unroll
    for (int k = 0; k < 9; k++) StencilIO<SO>::put(stc, Nc, V, D * 9 + k, (float)S[k]);
}

// Coarser stencil from a stored one: st_c[V][D] = sum_{o,d} hat3(o) A_f[2V+o][d] hat3(o+d-2D), one axis
// after another: the sum over (o, d) of one axis turns its nine blocks into three (13 products instead of
// the 27 of a direct sum), and the axes do not mix.  The x and y axes in one pass over the fine stencil, z
// in a second over T[((dz 3 + Dy) 3 + Dx) 9 + k][X + nc (Y + nc z)] (243 planes, z fine), a row of the
// 3 x 3 blocks per thread in the first pass, an entry in the second (an entry in the first as well read
// every line of the packed stencils from nine workgroups: 430 us on average over a 256^3 solve's levels, 220
// this way).  FP64 sums, rounded once: the coarsest
// system is nearly singular (one node holds the translations), and its solution is as far off as the
// stencil's rounding times that condition.  A direct sum, a thread per
// coarse vertex and plane Dz, took 330-380 us at any small size (567 blocks in a chain) and 2 ms at
// 128^3 -> 64^3; its thread count is what the split multiplies by 9 nf/nc.
template <typename SI>
__global__ __launch_bounds__(256) void k_galerkin_xy(Lay Lf, int nc, const SI* __restrict__ stf,
                                                     double* __restrict__ T) {
    const int nf = Lf.n;
    const uint32_t i = xcd_chunk(blockIdx.x, gridDim.x) * 256u + threadIdx.x, nt = (uint32_t)nc * nc * nf;
    if (i >= nt) return;
    const int X = (int)(i % nc), Y = (int)(i / nc % nc), z = (int)(i / ((uint32_t)nc * nc));
    const int row = (int)blockIdx.y % 3, dz = (int)blockIdx.y / 3;
    const size_t Nf = (size_t)nf * nf * nf;
    const uint32_t xs[3] = {Lf.part(wrap_dec(2 * X, nf), 0), Lf.part(2 * X, 0), Lf.part(2 * X + 1, 0)};
    const uint32_t ys[3] = {Lf.part(wrap_dec(2 * Y, nf), 1), Lf.part(2 * Y, 1), Lf.part(2 * Y + 1, 1)};
    const uint32_t zp = Lf.part(z, 2);
    const Rsrc rf = make_rsrc(stf, (size_t)StencilIO<SI>::words * Nf * 4);
    double S[9][3];  // [(Dy + 1) 3 + Dx + 1][column]
#pragma unroll
    for (int j = 0; j < 9; j++)
#pragma unroll
        for (int c = 0; c < 3; c++) S[j][c] = 0.0;
#pragma unroll
    for (int oy = -1; oy <= 1; oy++)
#pragma unroll
        for (int dy = -1; dy <= 1; dy++) {
            double R[3][3];
#pragma unroll
            for (int j = 0; j < 3; j++)
#pragma unroll
                for (int c = 0; c < 3; c++) R[j][c] = 0.0;
#pragma unroll
            for (int ox = -1; ox <= 1; ox++)
#pragma unroll
                for (int dx = -1; dx <= 1; dx++) {
                    const int d = (dx + 1) + 3 * (dy + 1) + 9 * dz;
                    float e[3];
                    StencilIO<SI>::get3(rf, (xs[ox + 1] + ys[oy + 1] + zp) * 4u, (uint32_t)(Nf * 4), d * 9 + 3 * row, e);
#pragma unroll
                    for (int Dx = -1; Dx <= 1; Dx++) {
                        const int q = ox + dx - 2 * Dx;
                        if (q < -1 || q > 1) continue;
#pragma unroll
                        for (int c = 0; c < 3; c++)
                            R[Dx + 1][c] = fma((ox ? 0.5 : 1.0) * (q ? 0.5 : 1.0), (double)e[c], R[Dx + 1][c]);
                    }
                }
#pragma unroll
            for (int Dy = -1; Dy <= 1; Dy++) {
                const int q = oy + dy - 2 * Dy;
                if (q < -1 || q > 1) continue;
                const double wy = (oy ? 0.5 : 1.0) * (q ? 0.5 : 1.0);
#pragma unroll
                for (int j = 0; j < 3; j++)
#pragma unroll
                    for (int c = 0; c < 3; c++) S[(Dy + 1) * 3 + j][c] = fma(wy, R[j][c], S[(Dy + 1) * 3 + j][c]);
            }
        }
#pragma unroll
    for (int j = 0; j < 9; j++)
#pragma unroll
        for (int c = 0; c < 3; c++) T[(size_t)((dz * 9 + j) * 9 + 3 * row + c) * nt + i] = S[j][c];
}

template <typename SO>
__global__ __launch_bounds__(256) void k_galerkin_z(Lay Lc, int nf, const double* __restrict__ T,
                                                    SO* __restrict__ stc, float clamp) {
    const size_t Nc = (size_t)Lc.n * Lc.n * Lc.n;
    int X, Y, Z;
    uint32_t V;
    if (!coarse_lex_vertex(Lc, X, Y, Z, V)) return;
    const int nc = Lc.n, k = (int)blockIdx.y % 9, j = (int)blockIdx.y / 9;  // j: (Dy + 1) 3 + Dx + 1
    const size_t nt = (size_t)nc * nc * nf, slab = (size_t)nc * nc, xy = (size_t)X + (size_t)nc * Y;
    const size_t zs[3] = {wrap_dec(2 * Z, nf) * slab + xy, 2 * Z * slab + xy, (2 * Z + 1) * slab + xy};
    double S[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int oz = -1; oz <= 1; oz++)
#pragma unroll
        for (int dz = -1; dz <= 1; dz++) {
            const double e = T[(size_t)(((dz + 1) * 9 + j) * 9 + k) * nt + zs[oz + 1]];
#pragma unroll
            for (int Dz = -1; Dz <= 1; Dz++) {
                const int q = oz + dz - 2 * Dz;
                if (q >= -1 && q <= 1) S[Dz + 1] = fma((oz ? 0.5 : 1.0) * (q ? 0.5 : 1.0), e, S[Dz + 1]);
            }
        }
    if (j == 4 && k % 4 == 0 && fabs(S[1]) < (double)clamp) S[1] = clamp;
#pragma unroll
    for (int Dz = 0; Dz < 3; Dz++) StencilIO<SO>::put(stc, Nc, V, (Dz * 9 + j) * 9 + k, (float)S[Dz]);
}

// ---------------------------------------------------------------------------------------------
// Coarsest level: its dense FP64 operator assembled and inverted, and the inverse applied.  Dof order
// 3 v + i, m = 3 n_c^3 <= 1029 (n_c = 4..7: the 27 neighbours of a vertex are distinct).
// ---------------------------------------------------------------------------------------------

// A = (S + S^T) / 2 of the stencil's matrix S (entry k = 9d + 3i + j of vertex v couples (v, i) with
// (v + d, j)), one thread per entry; *status = 0.
__global__ __launch_bounds__(256) void k_coarse_assemble(int nc, const float* __restrict__ st, double* __restrict__ A,
                                                         int* __restrict__ status) {
    const int Nc = nc * nc * nc, m = 3 * Nc;
    const int t = (int)(blockIdx.x * 256 + threadIdx.x);
    if (t == 0) *status = 0;
    if (t >= m * m) return;
    const int row = t / m, col = t - row * m;
    const int v = row / 3, i = row % 3, q = col / 3, j = col % 3;
    int d[3];
    bool near = true;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const int pv = a == 0 ? v % nc : (a == 1 ? v / nc % nc : v / (nc * nc));
        const int pq = a == 0 ? q % nc : (a == 1 ? q / nc % nc : q / (nc * nc));
        int o = pq - pv;
        o = o == nc - 1 ? -1 : (o == 1 - nc ? 1 : o);
        near = near && o >= -1 && o <= 1;
        d[a] = o + 1;
    }
    double val = 0.0;
    if (near) {
        const int e = d[0] + 3 * d[1] + 9 * d[2];
        const double s = (double)st[(size_t)(e * 9 + i * 3 + j) * Nc + v];
        const double r = (double)st[(size_t)((26 - e) * 9 + j * 3 + i) * Nc + q];
        val = row == col ? s : 0.5 * (s + r);
    }
    A[t] = val;
}

// Inverse of the symmetric positive definite A by Gauss-Jordan elimination in blocks of 32, one launch per
// block step K over the whole matrix, from one buffer into another (no launch reads what it writes).  With
// D = A[K][K]^-1:  A'[K][K] = D, A'[K][J] = D A[K][J], A'[I][K] = -A[I][K] D,
// A'[I][J] = A[I][J] - A[I][K] D A[K][J].  Every workgroup inverts the diagonal block itself by scalar
// Gauss-Jordan steps in registers (one barrier a step), whose pivots are the Schur complements: positive
// exactly when A is positive definite (the squares of the Cholesky pivots).  A launch finds in *before 0, or
// 1 + the first step whose pivot was not positive (it then does nothing), and leaves the same after itself
// in *after.  These are two words, as A and B are two buffers: a workgroup that read the word which another
// one of the same launch may set could see it in some of its waves only, and they would part at a barrier.
// Every workgroup forms the same pivots, so they all stop at the same one.  A launch per scalar step took
// 3.2-5 us m times (0.63 ms at m = 192).
constexpr int kGjB = 32;

__global__ __launch_bounds__(256) void k_gj_block(int m, int k0, const double* __restrict__ A, double* __restrict__ B,
                                                  const int* __restrict__ before, int* __restrict__ after) {
    const bool writer = blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0;
    const int failed = *before;
    if (failed != 0) {
        if (writer) *after = failed;
        return;
    }
    __shared__ double Dv[kGjB][kGjB + 1], Ct[kGjB][kGjB + 1], Rt[kGjB][kGjB + 1], prow[2][kGjB], pcol[2][kGjB];
    const int i = (int)(threadIdx.x >> 3), j0 = (int)(threadIdx.x & 7) * 4;
    const int I = (int)blockIdx.y * kGjB, J = (int)blockIdx.x * kGjB;
    // entries past the matrix: the identity
    auto get = [&](int r, int c) { return r < m && c < m ? A[(size_t)r * m + c] : (r == c ? 1.0 : 0.0); };
    double v[4], own[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        v[q] = get(k0 + i, k0 + j0 + q);
        own[q] = get(I + i, J + j0 + q);
        Ct[i][j0 + q] = get(I + i, k0 + j0 + q);
        Rt[i][j0 + q] = get(k0 + i, J + j0 + q);
    }
    for (int kb = 0; kb < kGjB; kb += 4) {
#pragma unroll
        for (int kq = 0; kq < 4; kq++) {
            const int k = kb + kq, buf = kq & 1;
            if (i == k) {
#pragma unroll
                for (int q = 0; q < 4; q++) prow[buf][j0 + q] = v[q];
            }
            if (j0 == kb) pcol[buf][i] = v[kq];
            __syncthreads();
            const double piv = prow[buf][k];
            if (!(piv > 0.0)) {  // the same for every thread
                if (writer) *after = 1 + k0 + k;
                return;
            }
            const double inv = 1.0 / piv, ci = pcol[buf][i];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const double rj = (j0 + q == k ? 1.0 : prow[buf][j0 + q]) * inv;
                v[q] = i == k ? rj : (j0 + q == k ? -ci * inv : fma(-ci, rj, v[q]));
            }
        }
    }
    if (writer) *after = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) Dv[i][j0 + q] = v[q];
    __syncthreads();
    const bool rk = I == k0, ck = J == k0;
    double o[4];
    if (rk && ck) {
#pragma unroll
        for (int q = 0; q < 4; q++) o[q] = v[q];
    } else if (ck) {
#pragma unroll
        for (int q = 0; q < 4; q++) o[q] = 0.0;
        for (int l = 0; l < kGjB; l++)
#pragma unroll
            for (int q = 0; q < 4; q++) o[q] = fma(-Ct[i][l], Dv[l][j0 + q], o[q]);
    } else {
        double r[4] = {0.0, 0.0, 0.0, 0.0};
        for (int l = 0; l < kGjB; l++)
#pragma unroll
            for (int q = 0; q < 4; q++) r[q] = fma(Dv[i][l], Rt[l][j0 + q], r[q]);
#pragma unroll
        for (int q = 0; q < 4; q++) o[q] = r[q];
        if (!rk) {
            __syncthreads();  // rk and ck are the same for the whole workgroup
#pragma unroll
            for (int q = 0; q < 4; q++) Rt[i][j0 + q] = r[q];
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 4; q++) o[q] = own[q];
            for (int l = 0; l < kGjB; l++)
#pragma unroll
                for (int q = 0; q < 4; q++) o[q] = fma(-Ct[i][l], Rt[l][j0 + q], o[q]);
        }
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
        if (I + i < m && J + j0 + q < m) B[(size_t)(I + i) * m + J + j0 + q] = o[q];
}

// u = A^-1 f for the six load cases: a wave per row, so that the inverse is read once, along its rows, for
// all six (a thread per row and workgroup per load case: 14.5 us at m = 192, 48 us at m = 375).
__global__ __launch_bounds__(256) void k_coarse_solve(int m, size_t Nc, const double* __restrict__ Ainv,
                                                      const float* __restrict__ f, float* __restrict__ u) {
    extern __shared__ float fb[];  // [6][m]
    for (int t = threadIdx.x; t < 6 * m; t += 256) {
        const int r = t / m, k = t - r * m, v = k / 3, i = k - 3 * v;
        fb[t] = f[(size_t)(r * 3 + i) * Nc + v];
    }
    __syncthreads();
    const int row = (int)(blockIdx.x * 4 + (threadIdx.x >> 6)), lane = (int)(threadIdx.x & 63);
    if (row >= m) return;
    double s[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    const double* a = Ainv + (size_t)row * m;
    for (int k = lane; k < m; k += 64) {
        const double av = a[k];
#pragma unroll
        for (int r = 0; r < 6; r++) s[r] = fma(av, (double)fb[r * m + k], s[r]);
    }
    const int v = row / 3, i = row % 3;
#pragma unroll
    for (int r = 0; r < 6; r++) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) s[r] += __shfl_xor(s[r], off, 64);
        if (lane == r) u[(size_t)(r * 3 + i) * Nc + v] = (float)s[r];
    }
}

template <typename SO>
void galerkin_fine_case(hipStream_t s, const Lay& Lf, const Lay& Lc, const double* G, const float* G32,
                        const double* ke, const float* w, SO* o, float clamp) {
    const unsigned nb = nblk((size_t)Lc.n * Lc.n * Lc.n);
    if (Lc.n <= 32)
        hipLaunchKernelGGL((k_galerkin_fine<1, double, SO>), dim3(nb, 27), dim3(256), 0, s, Lf, Lc, G, w, o, clamp);
    else if (Lc.n <= 64)
        hipLaunchKernelGGL((k_galerkin_fine<9, double, SO>), dim3(nb, 3), dim3(256), 0, s, Lf, Lc, G, w, o, clamp);
    else
        hipLaunchKernelGGL((k_galerkin_fine<27, float, SO>), dim3(nb), dim3(256), 0, s, Lf, Lc, G32, w, o, clamp);
    hipLaunchKernelGGL(k_galerkin_fine_pin<SO>, dim3(27 * 27), dim3(64), 0, s, Lf, Lc, ke, w, o, clamp);
}

template <typename SI, typename SO>
void galerkin_coarse_case(hipStream_t s, const Lay& Lf, const Lay& Lc, const void* stf, void* stc, double* work,
                          float clamp) {
    const size_t Nc = (size_t)Lc.n * Lc.n * Lc.n;
    hipLaunchKernelGGL(k_galerkin_xy<SI>, dim3(nblk(2 * Nc), 9), dim3(256), 0, s, Lf, Lc.n,
                       static_cast<const SI*>(stf), work);
    hipLaunchKernelGGL(k_galerkin_z<SO>, dim3(nblk(Nc), 81), dim3(256), 0, s, Lc, Lf.n, work, static_cast<SO*>(stc),
                       clamp);
}

}  // namespace

void launch_galerkin_fine(hipStream_t s, int nf, int lexc, const double* G, const float* G32, const double* ke,
                          const float* w, void* stc, int out_half, float clamp) {
    const Lay Lf = make_lay(nf, 0), Lc = make_lay(nf / 2, lexc);
    if (out_half)
        galerkin_fine_case(s, Lf, Lc, G, G32, ke, w, static_cast<half2_t*>(stc), clamp);
    else
        galerkin_fine_case(s, Lf, Lc, G, G32, ke, w, static_cast<float*>(stc), clamp);
}

void launch_galerkin_coarse(hipStream_t s, int nf, int lexc, const void* stf, int in_half, void* stc, int out_half,
                            double* work, float clamp) {
    const Lay Lf = make_lay(nf, 0), Lc = make_lay(nf / 2, lexc);
    if (in_half && out_half)
        galerkin_coarse_case<half2_t, half2_t>(s, Lf, Lc, stf, stc, work, clamp);
    else if (in_half)
        galerkin_coarse_case<half2_t, float>(s, Lf, Lc, stf, stc, work, clamp);
    else if (out_half)
        galerkin_coarse_case<float, half2_t>(s, Lf, Lc, stf, stc, work, clamp);
    else
        galerkin_coarse_case<float, float>(s, Lf, Lc, stf, stc, work, clamp);
}

void launch_coarse_solve(hipStream_t s, int nc, const double* Ainv, const float* f, float* u) {
    const size_t Nc = (size_t)nc * nc * nc;
    const int m = (int)(3 * Nc);
    hipLaunchKernelGGL(k_coarse_solve, dim3((m + 3) / 4), dim3(256), sizeof(float) * 6 * m, s, m, Nc, Ainv, f, u);
}

void launch_coarse_factor(hipStream_t s, int nc, const float* st, double* ainv, double* work, int* status) {
    const int m = 3 * nc * nc * nc, nb = (m + kGjB - 1) / kGjB;
    // the steps alternate between the two buffers and status words and end in ainv and status[0]
    double* buf[2] = {ainv, work};
    hipLaunchKernelGGL(k_coarse_assemble, dim3(nblk((size_t)m * m)), dim3(256), 0, s, nc, st, buf[nb & 1],
                       status + (nb & 1));
    for (int k = 0; k < nb; k++) {
        const int from = (nb - k) & 1, to = 1 - from;
        hipLaunchKernelGGL(k_gj_block, dim3(nb, nb), dim3(256), 0, s, m, k * kGjB, buf[from], buf[to], status + from,
                           status + to);
    }
}

}  // namespace homo3d
