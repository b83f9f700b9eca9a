// C^H and sensitivity (elasticMatrix_kernel_opt, homogenization.cu:208-346; Sensitivity_kernel_opt_2,
// homogenization.cu:697-858): the mutual energies E_ij = (chi0_i - chi_i)^T KE (chi0_j - chi_j) of the six
// load cases in every cell.
//
// A product with the 24 x 24 element matrix costs 3456 FMAs a cell and 504 more for the 21 energies, and
// that, not the 1.3 GB of fields at 256^3, bounded the kernels (2.76 ms).  The energy of the trilinear
// isotropic cube is a sum of 19 squares instead.  A component's nodal values have, beside their mean, seven
// Haar coefficients (differences along x, y, z, xy, xz, yz, xyz), the coefficients of the displacement in
// the basis 1, xi, eta, zeta, xi eta, ... of centred coordinates.  Products of different basis functions
// integrate to zero over the cell, so with lambda, mu:
//   energy = lambda (exx + eyy + ezz)^2 + 2 mu (exx^2 + eyy^2 + ezz^2) + mu (gyz^2 + gxz^2 + gxy^2)  [means]
//     + 1/12 [ (lambda + 3/2 mu) (a + b)^2 + 3/2 mu (a - b)^2  for the three pairs
//              (a, b) = (y_xy, z_xz), (x_xy, z_yz), (x_xz, y_yz)
//            + mu ((y_xz + z_xy)^2 + (x_yz + z_xy)^2 + (x_yz + y_xz)^2) ]
//     + 1/144 (lambda + 4 mu) (x_xyz^2 + y_xyz^2 + z_xyz^2)
// (x_xy: the xi eta coefficient of component x).  That is about 500 additions for the coefficients and
// 27 products per square for the 21 mutual energies: a third of the arithmetic.  The macro displacements
// are linear, so they only enter the six mean strains.  FP32 per cell, C^H summed over the cells in FP64.
//
// The other cost is the gather: 144 values a cell from memory keep the texture addresser busy longer than
// the arithmetic takes.  A workgroup stages the 33 x 5 x 3 nodes of a tile of 32 x 4 x 2 cells, all 18
// components, in LDS (36 KB: three workgroups a CU at the sensitivity's 161 registers, two at C^H's 256 with
// its 21 FP64 sums) with 35 loads a thread.  256^3: sensitivity 2.76 -> 0.81 ms, C^H 2.08 -> 1.13 ms; 1200
// vector instructions a wave are 0.51 ms of that, the rest waits for the tile.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.h"
#include "level.h"

namespace homo3d {

namespace {

constexpr int kEnTX = 32, kEnTY = 4, kEnTZ = 2;
constexpr int kEnThreads = kEnTX * kEnTY * kEnTZ;
constexpr int kEnNX = kEnTX + 1, kEnNY = kEnTY + 1, kEnNZ = kEnTZ + 1;
constexpr int kEnNodes = kEnNX * kEnNY * kEnNZ;
constexpr int kEnModes = 19;

// weights of the 19 squares, with the Haar coefficients' 1/4 (one difference) and 1/2 (two) folded in
struct EnergyWeights {
    float tr, axial, shear, sum, diff, cross, tri;
};

struct CaseWeights {
    float v[21];  // dJ/dC_ij (+ dJ/dC_ji), i <= j
};

// Stage the tile's nodes: u[c][z][y][x], c = 3 r + i.  Rows are read by x parity, as they lie.
__device__ __forceinline__ void stage_nodes(float* u, const Lay& L, size_t N, const float* __restrict__ chi, int x0,
                                            int y0, int z0) {
    const int n = L.n;
    const Rsrc rc = make_rsrc(chi, 18 * N * sizeof(float));
    const uint32_t plane = (uint32_t)(N * sizeof(float));
    constexpr int even = (kEnNX + 1) / 2;
#pragma unroll
    for (int it = 0; it < (kEnNodes + kEnThreads - 1) / kEnThreads; it++) {
        const int t = it * kEnThreads + (int)threadIdx.x;
        const int row = t / kEnNX, k = t - row * kEnNX;
        const int lx = k < even ? 2 * k : 2 * (k - even) + 1, ly = row % kEnNY, lz = row / kEnNY;
        int x = x0 + lx, y = y0 + ly, z = z0 + lz;
        // nodes past the far faces of the grid belong to no cell of it
        if (t >= kEnNodes || x > n || y > n || z > n) continue;
        x = x == n ? 0 : x;
        y = y == n ? 0 : y;
        z = z == n ? 0 : z;
        const uint32_t q = L.idx(x, y, z) * 4u;
        float v[18];
#pragma unroll
        for (int c = 0; c < 18; c++) v[c] = bload<float>(rc, q, (uint32_t)c * plane);
#pragma unroll
        for (int c = 0; c < 18; c++) u[c * kEnNodes + (lz * kEnNY + ly) * kEnNX + lx] = v[c];
    }
}

// The 21 energies of the cell whose first node is u[0].
__device__ __forceinline__ void cell_energies(const float* u, const EnergyWeights& w, float (&E)[21]) {
    float S[kEnModes][6];
#pragma unroll
    for (int s = 0; s < 6; s++) {
        // Haar differences of the three components: dx, dy, dz, dxy, dxz, dyz, dxyz
        float d[3][7];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const float* p = u + (3 * s + c) * kEnNodes;
            float sm[4], df[4];  // over x, for (y, z) = 00, 10, 01, 11
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float* q = p + ((r >> 1) * kEnNY + (r & 1)) * kEnNX;
                sm[r] = q[0] + q[1];
                df[r] = q[1] - q[0];
            }
            const float ss0 = sm[0] + sm[1], ss1 = sm[2] + sm[3], sd0 = sm[1] - sm[0], sd1 = sm[3] - sm[2];
            const float ds0 = df[0] + df[1], ds1 = df[2] + df[3], dd0 = df[1] - df[0], dd1 = df[3] - df[2];
            d[c][0] = ds0 + ds1;
            d[c][1] = sd0 + sd1;
            d[c][2] = ss1 - ss0;
            d[c][3] = dd0 + dd1;
            d[c][4] = ds1 - ds0;
            d[c][5] = sd1 - sd0;
            d[c][6] = dd1 - dd0;
        }
        // mean strains of chi0 - chi, times 4
        const float exx = (s == 0 ? 4.f : 0.f) - d[0][0], eyy = (s == 1 ? 4.f : 0.f) - d[1][1],
                    ezz = (s == 2 ? 4.f : 0.f) - d[2][2];
        S[0][s] = exx + eyy + ezz;
        S[1][s] = exx;
        S[2][s] = eyy;
        S[3][s] = ezz;
        S[4][s] = (s == 3 ? 4.f : 0.f) - (d[1][2] + d[2][1]);
        S[5][s] = (s == 4 ? 4.f : 0.f) - (d[0][2] + d[2][0]);
        S[6][s] = (s == 5 ? 4.f : 0.f) - (d[0][1] + d[1][0]);
        // bilinear terms (chi0 has none; their sign does not matter)
        S[7][s] = d[1][3] + d[2][4];
        S[8][s] = d[0][3] + d[2][5];
        S[9][s] = d[0][4] + d[1][5];
        S[10][s] = d[1][3] - d[2][4];
        S[11][s] = d[0][3] - d[2][5];
        S[12][s] = d[0][4] - d[1][5];
        S[13][s] = d[1][4] + d[2][3];
        S[14][s] = d[0][5] + d[2][3];
        S[15][s] = d[0][5] + d[1][4];
        S[16][s] = d[0][6];
        S[17][s] = d[1][6];
        S[18][s] = d[2][6];
    }
#pragma unroll
    for (int k = 0; k < 21; k++) E[k] = 0.f;
#pragma unroll
    for (int m = 0; m < kEnModes; m++) {
        const float wm = m == 0 ? w.tr
                                : (m < 4 ? w.axial
                                         : (m < 7 ? w.shear
                                                  : (m < 10 ? w.sum : (m < 13 ? w.diff : (m < 16 ? w.cross : w.tri)))));
        int k = 0;
#pragma unroll
        for (int a = 0; a < 6; a++) {
            const float t = wm * S[m][a];
#pragma unroll
            for (int b = a; b < 6; b++) {
                E[k] = fmaf(t, S[m][b], E[k]);
                k++;
            }
        }
    }
}

__device__ __forceinline__ void tile_of(uint32_t tile, uint32_t ntx, uint32_t nty, int& x0, int& y0, int& z0) {
    x0 = (int)(tile % ntx) * kEnTX;
    y0 = (int)(tile / ntx % nty) * kEnTY;
    z0 = (int)(tile / (ntx * nty)) * kEnTZ;
}

// partial[k * gridDim.x + block] = sum of w_e E_k,e over the block's tiles (FP64)
__global__ __launch_bounds__(kEnThreads, 2) void k_elastic_matrix(Lay L, size_t N, uint32_t ntx, uint32_t nty,
                                                                  uint32_t ntiles, EnergyWeights ew,
                                                                  const float* __restrict__ w,
                                                                  const float* __restrict__ chi,
                                                                  double* __restrict__ partial) {
    __shared__ float u[18 * kEnNodes];
    const int tx = (int)(threadIdx.x % kEnTX), ty = (int)(threadIdx.x / kEnTX % kEnTY),
              tz = (int)(threadIdx.x / (kEnTX * kEnTY));
    double acc[21];
#pragma unroll
    for (int k = 0; k < 21; k++) acc[k] = 0.0;
    const uint32_t per = (ntiles + gridDim.x - 1) / gridDim.x;  // consecutive tiles share their nodes in L2
    const uint32_t first = xcd_chunk(blockIdx.x, gridDim.x) * per, last = min(first + per, ntiles);
    for (uint32_t tile = first; tile < last; tile++) {
        int x0, y0, z0;
        tile_of(tile, ntx, nty, x0, y0, z0);
        stage_nodes(u, L, N, chi, x0, y0, z0);
        __syncthreads();
        const int x = x0 + tx, y = y0 + ty, z = z0 + tz;
        if (x < L.n && y < L.n && z < L.n) {
            const double we = (double)w[L.idx(x, y, z)];
            float E[21];
            cell_energies(u + (tz * kEnNY + ty) * kEnNX + tx, ew, E);
#pragma unroll
            for (int k = 0; k < 21; k++) acc[k] = fma(we, (double)E[k], acc[k]);
        }
        __syncthreads();
    }
    __shared__ double sh[kEnThreads / 64][21];
#pragma unroll
    for (int k = 0; k < 21; k++) {
        double t = acc[k];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) t += __shfl_down(t, off, 64);
        if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6][k] = t;
    }
    __syncthreads();
    if (threadIdx.x < 21) {
        double t = 0.0;
        for (int i = 0; i < kEnThreads / 64; i++) t += sh[i][threadIdx.x];
        partial[threadIdx.x * gridDim.x + blockIdx.x] = t;
    }
}

// sens[x + (y + z*n)*pitch] = (1/N) sum_{i<=j} E_ij (dC_ij + [i!=j] dC_ji)
// pitch 0: the level's own (parity-blocked) cell order, unpitched.
__global__ __launch_bounds__(kEnThreads, 2) void k_sensitivity(Lay L, size_t N, int pitch, uint32_t ntx, uint32_t nty,
                                                               EnergyWeights ew, const float* __restrict__ chi,
                                                               CaseWeights wdc, float* __restrict__ sens) {
    __shared__ float u[18 * kEnNodes];
    int x0, y0, z0;
    tile_of(xcd_chunk(blockIdx.x, gridDim.x), ntx, nty, x0, y0, z0);
    stage_nodes(u, L, N, chi, x0, y0, z0);
    __syncthreads();
    const int tx = (int)(threadIdx.x % kEnTX), ty = (int)(threadIdx.x / kEnTX % kEnTY),
              tz = (int)(threadIdx.x / (kEnTX * kEnTY));
    const int x = x0 + tx, y = y0 + ty, z = z0 + tz;
    if (x >= L.n || y >= L.n || z >= L.n) return;
    float E[21];
    cell_energies(u + (tz * kEnNY + ty) * kEnNX + tx, ew, E);
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < 21; k++) s = fmaf(E[k], wdc.v[k], s);
    sens[pitch ? x + ((size_t)y + (size_t)z * L.n) * pitch : (size_t)L.idx(x, y, z)] = s / (float)N;
}

EnergyWeights energy_weights(double lam, double mu) {
    EnergyWeights w;
    w.tr = (float)(lam / 16);
    w.axial = (float)(2 * mu / 16);
    w.shear = (float)(mu / 16);
    w.sum = (float)((lam + 1.5 * mu) / 48);
    w.diff = (float)(1.5 * mu / 48);
    w.cross = (float)(mu / 48);
    w.tri = (float)((lam + 4 * mu) / 144);
    return w;
}

}  // namespace

void launch_elastic_matrix(hipStream_t s, int n, double lam, double mu, const float* w, const float* chi,
                           double* partial, int nblocks, double* out21) {
    const size_t N = (size_t)n * n * n;
    const uint32_t ntx = (n + kEnTX - 1) / kEnTX, nty = (n + kEnTY - 1) / kEnTY, ntz = (n + kEnTZ - 1) / kEnTZ;
    const uint32_t ntiles = ntx * nty * ntz;
    const int nb = (int)std::min<uint32_t>((uint32_t)nblocks, ntiles);
    hipLaunchKernelGGL(k_elastic_matrix, dim3(nb), dim3(kEnThreads), 0, s, make_lay(n, 0), N, ntx, nty, ntiles,
                       energy_weights(lam, mu), w, chi, partial);
    launch_sum_partials(s, 21, nb, partial, out21);
}

void launch_sensitivity(hipStream_t s, int n, int pitch, double lam, double mu, const float* chi, const float* wdc,
                        float* sens) {
    const size_t N = (size_t)n * n * n;
    const uint32_t ntx = (n + kEnTX - 1) / kEnTX, nty = (n + kEnTY - 1) / kEnTY, ntz = (n + kEnTZ - 1) / kEnTZ;
    CaseWeights cw;
    std::copy(wdc, wdc + 21, cw.v);
    hipLaunchKernelGGL(k_sensitivity, dim3(ntx * nty * ntz), dim3(kEnThreads), 0, s, make_lay(n, 0), N, pitch, ntx, nty,
                       energy_weights(lam, mu), chi, cw, sens);
}

}  // namespace homo3d
