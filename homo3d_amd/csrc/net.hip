// Learned warm start: a small periodic 3D U-Net that maps a density field to the six load cases'
// displacement fields, trained and run on the GPU by the kernels in this file.
//
// The reference has no learned component; its warm start is the previous design's stored solutions
// (homogenization.cu:471-477, grid.cpp:459-462).  Here the network's prediction, upsampled to the
// solve grid, takes that place (homo3d_net_warm_start in api.cpp), and the FP64-refined MG-PCG remains
// the solver and the judge of the prediction's error.
//
// Architecture (levels L, channels c_l = C0 2^l, grid g / 2^l at level l; g >= 8 * 2^(L-1)):
//   encoder: E_l = relu(conv3(in_l)), S_l = relu(conv3(E_l)), in_0 = density, in_{l+1} = avgpool2(S_l)
//   decoder: CAT_l = [up2(D_{l+1}) | S_l], D_l = relu(conv3(relu(conv3(CAT_l)))), D_{L-1} = S_{L-1}
//   head:    P = conv1(D_0) (18 channels: u of load case s, component k at channel 3 s + k)
// conv3 is a periodic 3x3x3 correlation, tap t = (dx+1) + 3 (dy+1) + 9 (dz+1) reading X[v + (dx,dy,dz)].
//
// Storage: activations are bf16 in planes of 8 channels, [C/8][B g^3][8] (voxel v = x + g (y + g z) + g^3 b;
// a plane is as long as the largest batch), so a matrix operand, 8 channels of 16 consecutive voxels, is
// 256 bytes in a row.  With the voxels' channels in a row instead it was 16 bytes from each of 16 cache
// lines, and the convolutions were bound by the lines a load touches (some 64 cycles each): 2.0 ms for a
// 64^3 x 4 gradient's 28 of them, 1.1 ms now.  S_l lives inside
// CAT_l (channel offset c_{l+1}), which makes the concatenation free.  Master weights, Adam state and
// gradients are FP32.
//
// Matrix cores: every convolution pass is an implicit GEMM on v_mfma_f32_16x16x32_bf16 (bf16
// operands, FP32 accumulation):
//   forward / input gradient (k_conv):  out[v][co] = sum_{t,ci} W[co][t][ci] X[v + d_t][ci]
//       A = weights (16 output channels x 32 of (t, ci)), B = the 16 voxels' shifted inputs.  The input
//       gradient is the same pass over dZ with the flipped, transposed weights Wb[ci][t][co] = W[co][26-t][ci].
//   weight gradient (k_wgrad):  dW[co][t][ci] = sum_v dZ[v][co] X[v + d_t][ci]
//       the reduction runs over voxels: tiles of dZ and X staged in LDS are read transposed.  Split over
//       voxel ranges, partial sums reduced after (k_wgrad_reduce): deterministic, no atomics.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "../../include/homo3d.h"
#include "net.h"

using namespace homo3d;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kOut = 18;      // output channels
constexpr int kInCh = 8;      // stored input channels (density + 7 zeros): the 8-channel loads stay aligned
constexpr int kPld = 24;      // row stride of the FP32 prediction
constexpr int kDpC = 24;      // channels of the head's output gradient (18 used, zeros after)
constexpr int kPlanes = kDpC / 8;

// 8-channel group of channel c of voxel v; ps: length of a plane
__device__ __forceinline__ size_t group(long v, int c, long ps) { return ((size_t)(c >> 3) * (size_t)ps + (size_t)v) * 8; }

__device__ __forceinline__ bf16x8 load8(const uint16_t* p) {
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(p));
}

// what a convolution reads past its last tap or chunk (selecting the address, not the loaded value, keeps the load
// in flight, and an address in the constant segment would make it a flat one); never written
__device__ __attribute__((aligned(16))) uint16_t kZeros[8] = {};

// ---------------------------------------------------------------------------------------------------
// Convolution (forward and input gradient): implicit GEMM.  A wave computes 16 MB output channels for
// 16 NB voxels; a block holds 4 waves (64 NB consecutive voxels); blockIdx.y selects the channel block.
// cin % 8 == 0; the weights lie as [kpad / 8][rows][8], rows padded to gridDim.y * 16 MB and kpad (a multiple
// of 32) with zeros.
// ---------------------------------------------------------------------------------------------------
template <int MB, int NB, bool TAP27, bool RELU, bool F32OUT>
__global__ __launch_bounds__(256) void k_conv(const uint16_t* __restrict__ in, int cin, const uint16_t* __restrict__ w,
                                              int kpad, int rows, const float* __restrict__ bias,
                                              void* __restrict__ out, int cout, int lg, long nvox, long ps,
                                              const uint16_t* __restrict__ relu) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = lane & 15, grp = lane >> 4;
    const long vb = ((long)blockIdx.x * 4 + wave) * (16 * NB);
    const int cb = blockIdx.y * 16 * MB;
    // the voxels that the taps of the wave's voxels read
    __shared__ uint32_t nbrs[4][TAP27 ? 27 : 1][16 * NB];
    uint32_t(*const nb)[16 * NB] = nbrs[wave];
    const int m = (1 << lg) - 1;
    for (int v = lane; v < 16 * NB; v += 64) {
        const uint32_t g = (uint32_t)(vb + v), x = g & m, y = (g >> lg) & m, z = (g >> (2 * lg)) & m, s0 = (g >> (3 * lg)) << (3 * lg);
        if (TAP27) {
#pragma unroll
            for (int t = 0; t < 27; t++)
                nb[t][v] = s0 | ((z + t / 9 - 1) & m) << (2 * lg) | ((y + t / 3 % 3 - 1) & m) << lg | ((x + t % 3 - 1) & m);
        } else {
            nb[0][v] = g;
        }
    }
    // the wave's lanes read each other's entries below
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (vb >= nvox) return;
    constexpr int D = MB + NB > 6 ? 2 : MB + NB > 3 ? 4 : 6;  // chunks of operands in flight
    f32x4 acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int ntaps = TAP27 ? 27 : 1;
    // (tap, ci) of k0 = 32 kc + 8 grp of the next load, advanced by 32 = dtap cin + dci
    int tap = 8 * grp / cin, ci = 8 * grp - tap * cin;
    const int dtap = 32 / cin, dci = 32 - dtap * cin;
    const int kch = kpad >> 5;
    bf16x8 a[D][MB], b[D][NB];
    const uint16_t* wr = w + ((size_t)grp * rows + cb + col) * 8;
    int next = 0;
    auto load = [&](bf16x8 (&as)[MB], bf16x8 (&bs)[NB]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MB; i++) as[i] = load8(next < kch ? wr + 128 * i : kZeros);
        wr += (size_t)32 * rows;
        next++;
        const int t = min(tap, ntaps - 1);
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const uint16_t* p = in + group(nb[t][16 * j + col], ci, ps);
            bs[j] = load8(tap < ntaps ? p : kZeros);
        }
        tap += dtap;
        ci += dci;
        if (ci >= cin) {
            ci -= cin;
            tap++;
        }
    };
    // D chunks ahead without a branch, whose two sides would have to wait for the same loads: a few chunks of
    // zeros at the end instead
#pragma unroll
    for (int d = 0; d < D; d++) load(a[d], b[d]);
    for (int kc = 0; kc < kch; kc += D) {
#pragma unroll
        for (int d = 0; d < D; d++) {
#pragma unroll
            for (int i = 0; i < MB; i++)
#pragma unroll
                for (int j = 0; j < NB; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[d][i], b[d][j], acc[i][j], 0, 0, 0);
            load(a[d], b[d]);
        }
    }
    // D layout: lane (col, grp) holds voxel vb + 16 j + col, channels cb + 16 i + 4 grp + r
#pragma unroll
    for (int i = 0; i < MB; i++) {
        const int co0 = cb + 16 * i + 4 * grp;
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const long v = vb + 16 * j + col;
            float o[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                o[r] = acc[i][j][r] + (bias ? bias[co0 + r] : 0.f);
                if (RELU) o[r] = fmaxf(o[r], 0.f);
            }
            if (F32OUT) {
                float* dst = reinterpret_cast<float*>(out) + v * kPld + co0;
                if (co0 + 3 < cout) {
                    *reinterpret_cast<float4*>(dst) = make_float4(o[0], o[1], o[2], o[3]);
                } else {
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (co0 + r < cout) dst[r] = o[r];
                }
            } else {
                if (co0 >= cout) continue;
                const size_t at = group(v, co0, ps) + (co0 & 7);
                uint2 q;
                if (!RELU && relu) {  // the layer below's ReLU: no gradient where its output is not positive
                    q = *reinterpret_cast<const uint2*>(relu + at);
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (!(bf2f((uint16_t)((r < 2 ? q.x : q.y) >> (16 * (r & 1)))) > 0.f)) o[r] = 0.f;
                }
                q.x = (uint32_t)f2bf(o[0]) | ((uint32_t)f2bf(o[1]) << 16);
                q.y = (uint32_t)f2bf(o[2]) | ((uint32_t)f2bf(o[3]) << 16);
                *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(out) + at) = q;
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------------
// Weight gradient.  A block stages a tile of TX x TY x TZ voxels in LDS, 16 input channels of X with one row
// more on each side in y and z, and 16 WC output channels of dZ with one voxel more on each side in x, a
// voxel's 16 channels in 32 bytes.  The tap (dx, dy, dz) pairs X at v + (dy, dz)
// with dZ at v - dx, so a tile's 27 products need 9 X and 3 dZ operands.  The reduction over voxels wants a
// channel's voxels in one lane: the transposing LDS reads (four voxels of 16 channels to 16 lanes with a
// channel each) give that from any voxel on, so nothing is copied to channel-major order first.  Bound by
// the tiles' loads, X three times over with its neighbour rows.  The 15 layers of a 64^3 x 4 gradient:
// 0.68 ms with the sums of the partials; with channel-major copies of X (three, shifted in x) and dZ
// through memory, one wave a block on the products and a thread or a block for each sum 7.6 ms.
// Wave w takes output channels 16 (w % WC) and every (4 / WC)th 32-voxel chunk; a block walks a range of
// tiles, adds its waves' sums in LDS and leaves one partial; the bias gradient is a 28th product with ones.
// ---------------------------------------------------------------------------------------------------
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr int kWgTapFloats = 256;  // one 16 x 16 accumulator

// Lane's 8 voxels of channel lane % 16: 4 from each of two 16-voxel reads (p0, p1: the lane's 8-byte piece).
__device__ __forceinline__ bf16x8 read_tr(const uint16_t* p0, const uint16_t* p1) {
    typedef __attribute__((address_space(3))) s16x4 lds4;
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)p0), b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)p1);
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

template <int TX, int TY, int TZ, bool TAP27>
struct WgTile {
    static constexpr int H = TAP27 ? 1 : 0;
    static constexpr int vox = TX * TY * TZ, xvox = TX * (TY + 2 * H) * (TZ + 2 * H), zvox = (TX + 2 * H) * TY * TZ;
    static constexpr int taps = TAP27 ? 27 : 1;
    static size_t lds(int wc) {  // the tile, or the waves' sums on their way to one
        const size_t t = 32 * (size_t)(xvox + wc * zvox), r = sizeof(float) * (size_t)(taps + 1) * kWgTapFloats * 2;
        return wc < 4 && r > t ? r : t;
    }
};

// partial: [splits][czp][taps][cxp], bpartial: [splits][czp]
template <int TX, int TY, int TZ, bool TAP27>
__global__ __launch_bounds__(256, 2) void k_wgrad(const uint16_t* __restrict__ dz, int cz,
                                                  const uint16_t* __restrict__ x, int cx, int lg, long ps, int tiles,
                                                  int per, int wc, int czp, int cxp, float* __restrict__ partial,
                                                  float* __restrict__ bpartial) {
    using W = WgTile<TX, TY, TZ, TAP27>;
    constexpr int H = W::H, YH = TY + 2 * H, XP = TX + 2 * H, NT = W::taps;
    extern __shared__ __attribute__((aligned(16))) uint16_t sh[];
    uint16_t* const xs = sh;
    uint16_t* const zs = sh + 16 * W::xvox;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int cw = wave & (wc - 1), vw = wave / wc, nvw = 4 / wc;
    const int cb = (int)blockIdx.y * 16 * wc, nb = (int)blockIdx.z * 16;
    const int m = (1 << lg) - 1;
    f32x4 acc[NT], accb = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < NT; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    bf16x8 ones;
#pragma unroll
    for (int k = 0; k < 8; k++) ones[k] = (__bf16)1.0f;
    const int tend = min(tiles, ((int)blockIdx.x + 1) * per);
    for (int tile = (int)blockIdx.x * per; tile < tend; tile++) {
        // first voxel of the tile (1x1: the tiles are runs of consecutive voxels)
        int x0 = 0, y0 = 0, z0 = 0;
        long base = (long)tile * W::vox;
        if (TAP27) {
            const int nx = (1 << lg) / TX, ny = (1 << lg) / TY, nz = (1 << lg) / TZ;
            x0 = tile % nx * TX;
            y0 = tile / nx % ny * TY;
            z0 = tile / (nx * ny) % nz * TZ;
            base = (long)(tile / (nx * ny * nz)) << (3 * lg);
        }
        auto voxel = [&](int xx, int yy, int zz) {  // relative to the tile
            if (!TAP27) return base + xx + (long)TX * (yy + TY * zz);
            return base + (((long)((z0 + zz) & m) << (2 * lg)) | (long)(((y0 + yy) & m) << lg) | (long)((x0 + xx) & m));
        };
        if (tile != (int)blockIdx.x * per) __syncthreads();
#pragma unroll
        for (int k = 0; k < (2 * W::xvox + 255) / 256; k++) {
            const int i = (int)threadIdx.x + 256 * k, r = i >> 1, row = r / TX;
            const int c = nb + 8 * (i & 1);
            if (2 * W::xvox % 256 == 0 || i < 2 * W::xvox) {
                uint4 v = make_uint4(0, 0, 0, 0);
                if (c < cx) v = *reinterpret_cast<const uint4*>(x + group(voxel(r % TX, row % YH - H, row / YH - H), c, ps));
                *reinterpret_cast<uint4*>(xs + 8 * i) = v;
            }
        }
        for (int w = 0; w < wc; w++) {
#pragma unroll
            for (int k = 0; k < (2 * W::zvox + 255) / 256; k++) {
                const int i = (int)threadIdx.x + 256 * k, r = i >> 1, row = r / XP;
                const int c = cb + 16 * w + 8 * (i & 1);
                if (2 * W::zvox % 256 == 0 || i < 2 * W::zvox) {
                    uint4 v = make_uint4(0, 0, 0, 0);
                    if (c < cz) v = *reinterpret_cast<const uint4*>(dz + group(voxel(r % XP - H, row % TY, row / TY), c, ps));
                    *reinterpret_cast<uint4*>(zs + 16 * W::zvox * w + 8 * i) = v;
                }
            }
        }
        __syncthreads();
        for (int q = vw; q < W::vox / 32; q += nvw) {
            // the lane's pieces: voxels 32 q + 16 r + lane / 4, channels 4 (lane % 4) ..
            const uint16_t *px[2], *pz[2];
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const int v = 32 * q + 16 * r + (lane >> 2), xx = v % TX, row = v / TX, yy = row % TY, zz = row / TY;
                px[r] = xs + 16 * ((zz + H) * YH * TX + (yy + H) * TX + xx) + 4 * (lane & 3);
                pz[r] = zs + 16 * (cw * W::zvox + row * XP + xx + H) + 4 * (lane & 3);
            }
            bf16x8 a[2 * H + 1];
#pragma unroll
            for (int d = 0; d < 2 * H + 1; d++) a[d] = read_tr(pz[0] - 16 * (d - H), pz[1] - 16 * (d - H));
            accb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[H], ones, accb, 0, 0, 0);
#pragma unroll
            for (int d = 0; d < NT / (2 * H + 1); d++) {
                const int o = TAP27 ? 16 * ((d / 3 - 1) * YH * TX + (d % 3 - 1) * TX) : 0;
                const bf16x8 b = read_tr(px[0] + o, px[1] + o);
#pragma unroll
                for (int e = 0; e < 2 * H + 1; e++)
                    acc[d * (2 * H + 1) + e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[e], b, acc[d * (2 * H + 1) + e], 0, 0, 0);
            }
        }
    }
    // the waves of the same output channels: the upper half to LDS, the lower half adds, until one is left
    float* const fs = reinterpret_cast<float*>(sh);
    for (int half = nvw / 2; half > 0; half /= 2) {
        float* const mine = fs + (size_t)(cw * half + vw % half) * (NT + 1) * kWgTapFloats + 4 * lane;
        __syncthreads();
        if (vw >= half && vw < 2 * half) {
#pragma unroll
            for (int t = 0; t < NT; t++) *reinterpret_cast<f32x4*>(mine + t * kWgTapFloats) = acc[t];
            *reinterpret_cast<f32x4*>(mine + NT * kWgTapFloats) = accb;
        }
        __syncthreads();
        if (vw < half) {
#pragma unroll
            for (int t = 0; t < NT; t++) acc[t] += *reinterpret_cast<const f32x4*>(mine + t * kWgTapFloats);
            accb += *reinterpret_cast<const f32x4*>(mine + NT * kWgTapFloats);
        }
    }
    // lane (col, grp) holds input channel nb + col, output channels cb + 16 cw + 4 grp + r
    const int col = lane & 15, co = cb + 16 * cw + 4 * (lane >> 4);
    if (vw == 0 && co < czp) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const long o = (long)blockIdx.x * czp + co + r;
#pragma unroll
            for (int t = 0; t < NT; t++) partial[(o * NT + t) * cxp + nb + col] = acc[t][r];
            if (nb == 0 && col == 0) bpartial[o] = accb[r];
        }
    }
}

// dW[co][t][ci] (co < cout, ci < cin; the flat parameter layout) and db[co] = sums over the splits: a block
// takes 64 of them, its waves every (blockDim / 64)th split: 12 us on average (one thread a parameter, a chain
// of up to 1024 loads, was 101).
__global__ __launch_bounds__(1024) void k_wgrad_reduce(const float* __restrict__ partial, const float* __restrict__ bpartial,
                                                       int splits, int czp, int taps, int cxp, int cout, int cin,
                                                       float* __restrict__ dW, float* __restrict__ db) {
    __shared__ float sh[1024];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const int i = (int)blockIdx.x * 64 + lane, total = cout * taps * cin;
    const float* p = nullptr;
    long stride = 0;
    if (i < total) {
        const int ci = i % cin, t = i / cin % taps, co = i / (cin * taps);
        p = partial + ((long)co * taps + t) * cxp + ci;
        stride = (long)czp * taps * cxp;
    } else if (i < total + cout) {
        p = bpartial + i - total;
        stride = czp;
    }
    float s = 0.f;
    if (p) {
#pragma unroll 8
        for (int k = w; k < splits; k += nw) s += p[k * stride];
    }
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int k = nw / 2; k > 0; k >>= 1) {
        if (w < k) sh[threadIdx.x] += sh[threadIdx.x + 64 * k];
        __syncthreads();
    }
    if (w == 0 && p) (i < total ? dW[i] : db[i - total]) = sh[lane];
}

// The elementwise passes between levels: a thread takes a group of 8 channels.
__device__ __forceinline__ float group_at(const uint4& q, int k) {
    return bf2f((uint16_t)((k < 2 ? q.x : k < 4 ? q.y : k < 6 ? q.z : q.w) >> (16 * (k & 1))));
}
__device__ __forceinline__ uint4 group_of(const float (&f)[8]) {
    uint32_t w[4];
#pragma unroll
    for (int k = 0; k < 4; k++) w[k] = (uint32_t)f2bf(f[2 * k]) | ((uint32_t)f2bf(f[2 * k + 1]) << 16);
    return make_uint4(w[0], w[1], w[2], w[3]);
}
__device__ __forceinline__ const uint4* groups(const uint16_t* p, int plane, long ps) {
    return reinterpret_cast<const uint4*>(p) + (size_t)plane * ps;
}

// First child (grid 2^(lgc+1)) of voxel vc of grid 2^lgc; the others are + (k & 1), + (k >> 1 & 1) rows, + (k >> 2) planes.
__device__ __forceinline__ long child0(long vc, int lgc) {
    const long mc = (1 << lgc) - 1, x = vc & mc, y = (vc >> lgc) & mc, z = (vc >> (2 * lgc)) & mc;
    const int lg = lgc + 1;
    return (vc >> (3 * lgc) << (3 * lg)) + (2 * z << (2 * lg)) + (2 * y << lg) + 2 * x;
}
__device__ __forceinline__ long parent(long v, int lg) {
    const long m = (1 << lg) - 1, x = v & m, y = (v >> lg) & m, z = (v >> (2 * lg)) & m;
    const int lgc = lg - 1;
    return (v >> (3 * lg) << (3 * lgc)) + (z >> 1 << (2 * lgc)) + (y >> 1 << lgc) + (x >> 1);
}

// s = sum over the eight children of one group
__device__ __forceinline__ void child_sum(const uint4* __restrict__ in, long v0, int lg, float (&s)[8]) {
    uint4 q[8];
#pragma unroll
    for (int k = 0; k < 8; k++) q[k] = in[v0 + ((long)(k >> 2) << (2 * lg)) + ((long)((k >> 1) & 1) << lg) + (k & 1)];
#pragma unroll
    for (int c = 0; c < 8; c++) {
        s[c] = 0.f;
#pragma unroll
        for (int k = 0; k < 8; k++) s[c] += group_at(q[k], c);
    }
}

// avgpool2: out (grid g/2) = mean of the 8 children of in (grid g); blockIdx.y: plane.
__global__ __launch_bounds__(256) void k_pool(const uint16_t* __restrict__ in, int lgc, long nvc, long ps, long psc,
                                              uint16_t* __restrict__ out) {
    const long vc = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (vc >= nvc) return;
    float s[8];
    child_sum(groups(in, blockIdx.y, ps), child0(vc, lgc), lgc + 1, s);
#pragma unroll
    for (int c = 0; c < 8; c++) s[c] *= 0.125f;
    *const_cast<uint4*>(groups(out, blockIdx.y, psc) + vc) = group_of(s);
}

// up2: out (grid g) from in (grid g/2); blockIdx.y: plane.
__global__ __launch_bounds__(256) void k_up(const uint16_t* __restrict__ in, int lg, long nvox, long ps, long psc,
                                            uint16_t* __restrict__ out) {
    const long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nvox) return;
    *const_cast<uint4*>(groups(out, blockIdx.y, ps) + v) = groups(in, blockIdx.y, psc)[parent(v, lg)];
}

// gradient of up2: out (grid g/2) = sum of the children's entries of in (grid g) where the upsampled D (grid
// g/2) is positive, else 0: the gradient before D's ReLU.  blockIdx.y: plane.
__global__ __launch_bounds__(256) void k_up_back(const uint16_t* __restrict__ in, int lgc, long nvc, long ps, long psc,
                                                 const uint16_t* __restrict__ d, uint16_t* __restrict__ out) {
    const long vc = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (vc >= nvc) return;
    float s[8];
    child_sum(groups(in, blockIdx.y, ps), child0(vc, lgc), lgc + 1, s);
    const uint4 y = groups(d, blockIdx.y, psc)[vc];
#pragma unroll
    for (int c = 0; c < 8; c++)
        if (!(group_at(y, c) > 0.f)) s[c] = 0.f;
    *const_cast<uint4*>(groups(out, blockIdx.y, psc) + vc) = group_of(s);
}

// Gradient of the skip tensor S_l (relu applied): out = S > 0 ? dS + dIn[parent] / 8 : 0, dS its part of the
// gradient of CAT_l and dIn (grid g/2) the gradient of in_{l+1} = avgpool2(S_l).  blockIdx.y: plane.
__global__ __launch_bounds__(256) void k_skip_grad(const uint16_t* __restrict__ s, const uint16_t* __restrict__ ds,
                                                   const uint16_t* __restrict__ din, int lg, long nvox, long ps, long psc,
                                                   uint16_t* __restrict__ out) {
    const long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nvox) return;
    const uint4 y = groups(s, blockIdx.y, ps)[v], a = groups(ds, blockIdx.y, ps)[v], b = groups(din, blockIdx.y, psc)[parent(v, lg)];
    float o[8];
#pragma unroll
    for (int c = 0; c < 8; c++) o[c] = group_at(y, c) > 0.f ? group_at(a, c) + 0.125f * group_at(b, c) : 0.f;
    *const_cast<uint4*>(groups(out, blockIdx.y, ps) + v) = group_of(o);
}

// Stiffness weight of voxel v: w = rho^3 of the network input (the cell stiffness of the SIMP law).
__device__ __forceinline__ float net_weight(const uint16_t* in, long v) {
    const float r = bf2f(in[v * kInCh]);
    return r * r * r;
}

// Per (sample, channel) stiffness-weighted mean of the prediction P [v][kPld] over the sample's g^3
// voxels, and the sample's mean weight.  A sum is 256 chains, of the voxels t, t + 256, ..., then a tree
// over them.  A wave takes eight chains, eight lanes each: four channels a lane, so that a row of P is read
// once and not once a channel (109 us and 5 for the trees at 64^3 x 4, 464 with a block a channel); bound by
// the latency of its loads, 16 of them in flight.
constexpr int kChains = 256, kMeanRow = 20;  // kOut channels and the weight, padded to the lanes' fours

__global__ __launch_bounds__(64) void k_chan_chains(const float* __restrict__ P, const uint16_t* __restrict__ in, long nsv,
                                                    float* __restrict__ chains) {
    const int q = threadIdx.x & 7, t = (int)blockIdx.y * 8 + (threadIdx.x >> 3);
    const long base = (long)blockIdx.x * nsv;
    if (q >= kMeanRow / 4) return;
    float s[4] = {0.f, 0.f, 0.f, 0.f}, ws = 0.f;
#pragma unroll 16
    for (long v = t; v < nsv; v += kChains) {
        const float w = net_weight(in, base + v);
        const float4 p = *reinterpret_cast<const float4*>(P + (base + v) * kPld + 4 * q);
        s[0] += w * p.x;
        s[1] += w * p.y;
        s[2] += w * p.z;
        s[3] += w * p.w;
        ws += w;
    }
    if (q == kOut / 4) s[kOut % 4] = ws;
#pragma unroll
    for (int k = 0; k < 4; k++) chains[((long)blockIdx.x * kMeanRow + 4 * q + k) * kChains + t] = s[k];
}

__global__ __launch_bounds__(kChains) void k_chan_mean(const float* __restrict__ chains, long nsv, float* __restrict__ mean,
                                                       float* __restrict__ wbar) {
    __shared__ float sh[2][kChains];
    const int b = blockIdx.x, c = blockIdx.y;
    sh[0][threadIdx.x] = chains[((long)b * kMeanRow + c) * kChains + threadIdx.x];
    sh[1][threadIdx.x] = chains[((long)b * kMeanRow + kOut) * kChains + threadIdx.x];
    __syncthreads();
    for (int k = kChains / 2; k > 0; k >>= 1) {
        if ((int)threadIdx.x < k) {
            sh[0][threadIdx.x] += sh[0][threadIdx.x + k];
            sh[1][threadIdx.x] += sh[1][threadIdx.x + k];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        mean[b * kOut + c] = sh[1][0] > 0.f ? sh[0][0] / sh[1][0] : 0.f;
        if (c == 0) wbar[b] = sh[1][0] / (float)nsv;
    }
}

// Loss terms with stiffness weights (w / mean w per sample): d = P - mean_w P - T;
// dP = 2 (w / wbar) d / count (bf16, channels >= 18 stay 0); per-block FP64 partial sums of
// (w / wbar) d^2.  T is mean-free under the same weights, so the weighted mean needs no gradient term.
// A thread takes a group of 8 channels (blockIdx.y: plane); bound by the prediction, target and gradient
// rows, 190 MB at 64^3 x 4: 50 us (105 with a thread a value).
__global__ __launch_bounds__(256) void k_head_loss(const float* __restrict__ P, const float* __restrict__ mean,
                                                   const float* __restrict__ wbar, const uint16_t* __restrict__ in,
                                                   const uint16_t* __restrict__ T, long nvox, int lgs, double inv_count,
                                                   long ps, uint16_t* __restrict__ dP, double* __restrict__ partial) {
    __shared__ double sh[256];
    const int c0 = 8 * (int)blockIdx.y;
    double s = 0.0;
    for (long v = (long)blockIdx.x * blockDim.x + threadIdx.x; v < nvox; v += (long)gridDim.x * blockDim.x) {
        const long b = v >> (3 * lgs);
        const float wb = wbar[b];
        const float wt = wb > 0.f ? net_weight(in, v) / wb : 0.f;
        const float4 p0 = *reinterpret_cast<const float4*>(P + v * kPld + c0), p1 = *reinterpret_cast<const float4*>(P + v * kPld + c0 + 4);
        const float p[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
        const uint32_t* t = reinterpret_cast<const uint32_t*>(T + v * kOut + c0);  // kOut and c0 are even
        float o[8];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const bool live = c0 + 2 * k < kOut;
            const uint32_t tk = live ? t[k] : 0u;
#pragma unroll
            for (int e = 0; e < 2; e++) {
                o[2 * k + e] = 0.f;
                if (live) {
                    const float d = p[2 * k + e] - mean[b * kOut + c0 + 2 * k + e] - bf2f((uint16_t)(tk >> (16 * e)));
                    o[2 * k + e] = (float)(2.0 * inv_count) * wt * d;
                    s += (double)wt * d * d;
                }
            }
        }
        *reinterpret_cast<uint4*>(dP + group(v, c0, ps)) = group_of(o);
    }
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if ((int)threadIdx.x < k) sh[threadIdx.x] += sh[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.y * gridDim.x + blockIdx.x] = sh[0];
}

// Adam on the FP32 master parameters (c1 = 1 / (1 - b1^t), c2 = 1 / (1 - b2^t)).
__global__ __launch_bounds__(256) void k_adam(long n, const float* __restrict__ g, float* __restrict__ p,
                                              float* __restrict__ m1, float* __restrict__ m2, float lr, float b1, float b2,
                                              float c1, float c2, float eps) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float a = b1 * m1[i] + (1.f - b1) * gi;
    const float b = b2 * m2[i] + (1.f - b2) * gi * gi;
    m1[i] = a;
    m2[i] = b;
    p[i] -= lr * (a * c1) / (sqrtf(b * c2) + eps);
}

// bf16 weight layouts of one layer from the master W[co][t][ci] (cin real input channels):
// forward Wf[k / 8][r][k % 8], k = t cinp + ci (rows r < rows_f, zero outside co < cout, ci < cin, k < taps cinp);
// input-gradient Wb likewise, r = ci, k = t' coutp + co, Wb = W[co][flip t'][ci] (flip t = 26 - t for 3x3x3).
__global__ __launch_bounds__(256) void k_pack(const float* __restrict__ W, const float* __restrict__ bias, int cout,
                                              int cin, int cinp, int taps, int rows_f, int kpad_f,
                                              uint16_t* __restrict__ wf, float* __restrict__ bias_pad, int coutp,
                                              int rows_b, int kpad_b, uint16_t* __restrict__ wb) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long nf = (long)rows_f * kpad_f, nbk = wb ? (long)rows_b * kpad_b : 0;
    if (i < nf) {
        const int r = (int)(i / kpad_f), k = (int)(i % kpad_f);
        const int t = k / cinp, ci = k % cinp;
        float v = 0.f;
        if (r < cout && t < taps && ci < cin) v = W[((long)r * taps + t) * cin + ci];
        wf[((long)(k >> 3) * rows_f + r) * 8 + (k & 7)] = f2bf(v);
        if (k == 0) bias_pad[r] = r < cout ? bias[r] : 0.f;
    } else if (i < nf + nbk) {
        const long j = i - nf;
        const int r = (int)(j / kpad_b), k = (int)(j % kpad_b);
        const int t = k / coutp, co = k % coutp;
        float v = 0.f;
        if (r < cin && t < taps && co < cout) v = W[((long)co * taps + (taps == 27 ? 26 - t : t)) * cin + r];
        wb[((long)(k >> 3) * rows_b + r) * 8 + (k & 7)] = f2bf(v);
    }
}

// density (FP32, [B][g^3]) -> input slots (bf16 [v][8], channel 0)
__global__ __launch_bounds__(256) void k_set_input(const float* __restrict__ rho, long nvox, uint16_t* __restrict__ in) {
    const long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nvox) return;
    uint4 z = make_uint4(f2bf(rho[v]), 0, 0, 0);
    *reinterpret_cast<uint4*>(in + v * kInCh) = z;
}

__global__ __launch_bounds__(256) void k_f32_to_bf16(const float* __restrict__ a, long n, uint16_t* __restrict__ b) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = f2bf(a[i]);
}

// The prediction's 18 channels out of its rows of kPld, contiguous: a strided copy to the host moves each
// 72-byte row by itself (1.73 s at 64^3), a packed one 18.9 MB at once.
__global__ __launch_bounds__(256) void k_pack_pred(const float* __restrict__ P, long count, float* __restrict__ out) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const long v = i / kOut;
    out[i] = P[v * kPld + (i - v * kOut)];
}

inline unsigned nblk(long n, int t = 256) { return (unsigned)((n + t - 1) / t); }

int round_up(int a, int b) { return (a + b - 1) / b * b; }

}  // namespace

// =====================================================================================================
// Host side
// =====================================================================================================
struct NetLayer {
    int cin, cinp, cout, taps;
    bool relu;
    long off_w, off_b;      // into the flat parameter vector
    int mb_f, rows_f, kpad_f;
    int coutp, mb_b, rows_b, kpad_b;
    uint16_t *wf = nullptr, *wb = nullptr;
    float* bias_pad = nullptr;
};

struct NetLevel {
    int g, lg, c;
    long nvox;                   // batch_max g^3, the length of a plane
    uint16_t* in = nullptr;      // level 0: input, 8 channels; else avgpool2(S_{l-1}), c_{l-1}
    uint16_t* e = nullptr;       // E_l
    uint16_t* cat = nullptr;     // CAT_l, c_{l+1} + c channels (S_l at offset c_{l+1}); l < L-1
    uint16_t* s = nullptr;       // S_{L-1} at the bottom level
    uint16_t* d1 = nullptr;      // decoder first conv
    uint16_t* d = nullptr;       // D_l
    uint16_t* ga = nullptr;      // gradient scratch, c channels each
    uint16_t* gb = nullptr;
    uint16_t* dcat = nullptr;    // gradient of CAT_l
    uint16_t* din = nullptr;     // gradient of in_l (l > 0), c_{l-1} channels
};

struct homo3d_net {
    homo3d_net_config cfg{};
    hipStream_t stream = nullptr, copy = nullptr;  // copy: targets from the host during the forward pass
    hipEvent_t copy_start = nullptr, copy_done = nullptr;
    int L = 0;
    std::vector<NetLayer> layers;
    std::vector<NetLevel> lv;
    long nparam = 0;
    float *p = nullptr, *g = nullptr, *m1 = nullptr, *m2 = nullptr;
    long adam_t = 0;
    float* P = nullptr;          // prediction [v][kPld]
    uint16_t* T = nullptr;       // targets [v][18]
    uint16_t* dP = nullptr;      // kDpC channels
    float* mean = nullptr;       // [batch][18]
    float* wbar = nullptr;       // [batch] mean stiffness weight
    float* chains = nullptr;     // [batch][kMeanRow][kChains] their sums in parts
    double* lpart = nullptr;     // loss partial sums
    int lblocks = 512 * kPlanes;
    float* rho = nullptr;        // host-staged densities [batch][g^3]
    float* tstage = nullptr;     // [batch][g^3][18]: host-staged targets, or a prediction on its way to the host
    float* partial = nullptr;    // the weight gradient's partial sums
    size_t partial_elems = 0;
    // dataset (device resident): inputs [count][g^3][8], targets [count][g^3][18]
    uint16_t *ds_in = nullptr, *ds_tg = nullptr;
    int ds_cap = 0, ds_count = 0;
    std::string err;
};

namespace {

int nerr(homo3d_net* n, int code, const char* fmt, ...) {
    if (n) {
        char buf[512];
        va_list ap;
        va_start(ap, fmt);
        vsnprintf(buf, sizeof(buf), fmt, ap);
        va_end(ap);
        n->err = buf;
    }
    return code;
}

#define NETCHK(n, expr)                                                                      \
    do {                                                                                     \
        hipError_t e_ = (expr);                                                              \
        if (e_ != hipSuccess) return nerr(n, HOMO3D_HIP_ERROR, "%s: %s", #expr, hipGetErrorString(e_)); \
    } while (0)

int pick_mb(int cout) { return cout >= 128 ? 8 : cout >= 64 ? 4 : cout >= 32 ? 2 : 1; }

struct ConvArgs {
    const uint16_t* in;
    int cin;
    const uint16_t* w;
    int kpad, rows;
    const float* bias;
    void* out;
    int cout, lg;
    long nvox, ps;
    const uint16_t* relu;
};

template <int MB, int NB, bool TAP27, bool RELU, bool F32OUT>
void conv_tile(hipStream_t s, const ConvArgs& a) {
    const dim3 grid((unsigned)((a.nvox + 64 * NB - 1) / (64 * NB)), (unsigned)((a.cout + 16 * MB - 1) / (16 * MB)));
    hipLaunchKernelGGL((k_conv<MB, NB, TAP27, RELU, F32OUT>), grid, dim3(256), 0, s, a.in, a.cin, a.w, a.kpad, a.rows,
                       a.bias, a.out, a.cout, a.lg, a.nvox, a.ps, a.relu);
}

// A wave's tile: 8 products of 16 x 16 a chunk (mb rows of weights, the layer's padding) where that gives
// every SIMD two waves (2048 waves), else 2, and 1 below that again: a wave walks the whole reduction, and
// it is its latency that the small levels wait for.  64 channels at 16^3 x 4: 21 us with 2 products, and
// 128 channels at 8^3 x 4 13 us with 1, against 58 and 86 with 8 (and operands 64 cache lines a load apart).
template <bool TAP27, bool RELU, bool F32OUT>
void conv_any(hipStream_t s, int mb, const ConvArgs& a) {
    const long products = a.nvox / 16 * ((a.cout + 15) / 16);
    if (products < 2048 * 2)
        conv_tile<1, 1, TAP27, RELU, F32OUT>(s, a);
    else if (products < 2048 * 8 && mb > 1)
        conv_tile<2, 1, TAP27, RELU, F32OUT>(s, a);
    else if (products < 2048 * 8)
        conv_tile<1, 2, TAP27, RELU, F32OUT>(s, a);
    else
        switch (mb) {
            case 1: conv_tile<1, 8, TAP27, RELU, F32OUT>(s, a); break;
            case 2: conv_tile<2, 4, TAP27, RELU, F32OUT>(s, a); break;
            case 4: conv_tile<4, 2, TAP27, RELU, F32OUT>(s, a); break;
            default: conv_tile<8, 1, TAP27, RELU, F32OUT>(s, a); break;
        }
}

// forward pass of one layer at level V: out = act(conv(in) + b)
void layer_fwd(homo3d_net* n, const NetLayer& Ly, const uint16_t* in, void* out, const NetLevel& V, long nvox, bool f32out) {
    const ConvArgs a = {in, Ly.cinp, Ly.wf, Ly.kpad_f, Ly.rows_f, Ly.bias_pad, out, Ly.cout, V.lg, nvox, V.nvox, nullptr};
    if (Ly.taps == 27)
        conv_any<true, true, false>(n->stream, Ly.mb_f, a);
    else if (f32out)
        conv_any<false, false, true>(n->stream, Ly.mb_f, a);
}

// input gradient of one layer at level V: dX = conv(dZ, Wb), where relu (the layer's input, if that is a
// ReLU's output) is positive; cz channels of dZ
void layer_dx(homo3d_net* n, const NetLayer& Ly, const uint16_t* dz, int cz, uint16_t* dx, const NetLevel& V, long nvox,
              const uint16_t* relu) {
    const ConvArgs a = {dz, cz, Ly.wb, Ly.kpad_b, Ly.rows_b, nullptr, dx, Ly.cin, V.lg, nvox, V.nvox, relu};
    if (Ly.taps == 27)
        conv_any<true, false, false>(n->stream, Ly.mb_b, a);
    else
        conv_any<false, false, false>(n->stream, Ly.mb_b, a);
}

// How the weight gradient of a layer is split: wc output-channel tiles a block, `splits` ranges of `per` tiles.
struct WgPlan {
    int czp, cxp, wc, tx, tiles, per, splits;
    size_t partial() const { return (size_t)splits * czp; }  // rows of taps * cxp + 1 floats
};

// Tiles are whole x-rows up to 64 voxels.  Two blocks a compute unit fill the GPU (a block's tile takes 60 KB
// of LDS in the usual layers, up to 117 KB with 64 output channels at 64 voxels), and every split more is a partial of
// czp * taps * cxp sums written and read: 512 blocks over the channel tiles.
WgPlan wgrad_plan(int cz, int cx, int taps, int lg, long nvox) {
    WgPlan w;
    w.czp = round_up(cz, 16);
    w.cxp = round_up(cx, 16);
    w.wc = w.czp >= 64 ? 4 : w.czp >= 32 ? 2 : 1;
    w.czp = round_up(w.czp, 16 * w.wc);
    w.tx = taps == 27 ? std::min(64, 1 << lg) : 64;
    w.tiles = (int)(nvox / (w.tx * 4 * (w.tx == 64 ? 2 : 4)));
    const int groups = w.czp / (16 * w.wc) * (w.cxp / 16);
    w.per = (int)std::max(1L, ((long)w.tiles * groups + 511) / 512);
    w.splits = (w.tiles + w.per - 1) / w.per;
    return w;
}

template <int TX, int TZ, bool TAP27>
void wgrad(hipStream_t s, const WgPlan& w, const uint16_t* dz, int cz, const uint16_t* x, int cx, int lg, long ps,
           float* partial, float* bpartial) {
    using W = WgTile<TX, 4, TZ, TAP27>;
    const dim3 grid((unsigned)w.splits, (unsigned)(w.czp / (16 * w.wc)), (unsigned)(w.cxp / 16));
    hipLaunchKernelGGL((k_wgrad<TX, 4, TZ, TAP27>), grid, dim3(256), W::lds(w.wc), s, dz, cz, x, cx, lg, ps, w.tiles,
                       w.per, w.wc, w.czp, w.cxp, partial, bpartial);
}

// weight and bias gradient of one layer at level V into n->g: X the layer's input (cx stored channels), dZ the
// gradient of its output (cz channels with cz >= cout; both counts multiples of 8).
int layer_dw(homo3d_net* n, const NetLayer& Ly, const uint16_t* x, int cx, const uint16_t* dz, int cz, const NetLevel& V,
             long nvox) {
    const int lg = V.lg;
    const WgPlan w = wgrad_plan(cz, cx, Ly.taps, lg, nvox);
    if (w.partial() * (Ly.taps * w.cxp + 1) > n->partial_elems) return nerr(n, HOMO3D_BAD_ARG, "partial buffer too small");
    float* bp = n->partial + w.partial() * Ly.taps * w.cxp;
    if (Ly.taps != 27)
        wgrad<64, 2, false>(n->stream, w, dz, cz, x, cx, lg, V.nvox, n->partial, bp);
    else if (w.tx == 64)
        wgrad<64, 2, true>(n->stream, w, dz, cz, x, cx, lg, V.nvox, n->partial, bp);
    else if (w.tx == 32)
        wgrad<32, 4, true>(n->stream, w, dz, cz, x, cx, lg, V.nvox, n->partial, bp);
    else if (w.tx == 16)
        wgrad<16, 4, true>(n->stream, w, dz, cz, x, cx, lg, V.nvox, n->partial, bp);
    else
        wgrad<8, 4, true>(n->stream, w, dz, cz, x, cx, lg, V.nvox, n->partial, bp);
    const int tot = Ly.cout * Ly.taps * Ly.cin + Ly.cout;
    int waves = 1;
    while (waves < 16 && 2 * waves <= w.splits) waves *= 2;
    hipLaunchKernelGGL(k_wgrad_reduce, dim3(nblk(tot, 64)), dim3(64 * waves), 0, n->stream, n->partial, bp, w.splits, w.czp,
                       Ly.taps, w.cxp, Ly.cout, Ly.cin, n->g + Ly.off_w, n->g + Ly.off_b);
    return HOMO3D_OK;
}

int pack_weights(homo3d_net* n) {
    for (const NetLayer& Ly : n->layers) {
        const long tot = (long)Ly.rows_f * Ly.kpad_f + (Ly.wb ? (long)Ly.rows_b * Ly.kpad_b : 0);
        hipLaunchKernelGGL(k_pack, dim3(nblk(tot)), dim3(256), 0, n->stream, n->p + Ly.off_w, n->p + Ly.off_b, Ly.cout,
                           Ly.cin, Ly.cinp, Ly.taps, Ly.rows_f, Ly.kpad_f, Ly.wf, Ly.bias_pad, Ly.coutp, Ly.rows_b,
                           Ly.kpad_b, Ly.wb);
    }
    NETCHK(n, hipGetLastError());
    return HOMO3D_OK;
}

// Forward pass over `batch` samples already in lv[0].in; prediction into n->P.
void forward(homo3d_net* n, int batch) {
    const int L = n->L;
    int li = 0;
    for (int l = 0; l < L; l++) {
        NetLevel& V = n->lv[l];
        const long nv = (long)batch << (3 * V.lg);
        const NetLayer& c1 = n->layers[li++];
        const NetLayer& c2 = n->layers[li++];
        layer_fwd(n, c1, V.in, V.e, V, nv, false);
        if (l < L - 1) {
            const NetLevel& W = n->lv[l + 1];
            uint16_t* S = V.cat + W.c * V.nvox;
            layer_fwd(n, c2, V.e, S, V, nv, false);
            hipLaunchKernelGGL(k_pool, dim3(nblk(nv / 8), V.c / 8), dim3(256), 0, n->stream, S, W.lg, nv / 8, V.nvox, W.nvox,
                               W.in);
        } else {
            layer_fwd(n, c2, V.e, V.s, V, nv, false);
        }
    }
    // decoder
    for (int l = L - 2; l >= 0; l--) {
        NetLevel& V = n->lv[l];
        const NetLevel& W = n->lv[l + 1];
        const long nv = (long)batch << (3 * V.lg);
        hipLaunchKernelGGL(k_up, dim3(nblk(nv), W.c / 8), dim3(256), 0, n->stream, l == L - 2 ? W.s : W.d, V.lg, nv, V.nvox,
                           W.nvox, V.cat);
        const NetLayer& c1 = n->layers[li++];
        const NetLayer& c2 = n->layers[li++];
        layer_fwd(n, c1, V.cat, V.d1, V, nv, false);
        layer_fwd(n, c2, V.d1, V.d, V, nv, false);
    }
    const NetLayer& hd = n->layers[li];
    const NetLevel& V0 = n->lv[0];
    layer_fwd(n, hd, L > 1 ? V0.d : V0.s, n->P, V0, (long)batch << (3 * V0.lg), true);
}

// Loss of the prediction against n->T and the full parameter gradient into n->g.
int loss_backward(homo3d_net* n, int batch, double* loss) {
    const int L = n->L;
    const NetLevel& V0 = n->lv[0];
    const long nv0 = (long)batch << (3 * V0.lg);
    const long nsv = 1L << (3 * V0.lg);
    hipLaunchKernelGGL(k_chan_chains, dim3(batch, kChains / 8), dim3(64), 0, n->stream, n->P, V0.in, nsv, n->chains);
    hipLaunchKernelGGL(k_chan_mean, dim3(batch, kOut), dim3(kChains), 0, n->stream, n->chains, nsv, n->mean, n->wbar);
    const double inv = 1.0 / ((double)nv0 * kOut);
    hipLaunchKernelGGL(k_head_loss, dim3(n->lblocks / kPlanes, kPlanes), dim3(256), 0, n->stream, n->P, n->mean, n->wbar, V0.in, n->T, nv0,
                       V0.lg, inv, V0.nvox, n->dP, n->lpart);
    int li = (int)n->layers.size() - 1;
    int rc;
    // head
    {
        const NetLayer& hd = n->layers[li--];
        const uint16_t* top = L > 1 ? V0.d : V0.s;
        if ((rc = layer_dw(n, hd, top, V0.c, n->dP, kDpC, V0, nv0))) return rc;
        layer_dx(n, hd, n->dP, kDpC, V0.ga, V0, nv0, top);  // dZ of dec 0.c2 (L = 1: of enc 0.c2)
    }
    // decoder levels, top down in the parameter list (level 0 first)
    for (int l = 0; l <= L - 2; l++) {
        NetLevel& V = n->lv[l];
        NetLevel& W = n->lv[l + 1];
        const long nv = (long)batch << (3 * V.lg);
        const NetLayer& c2 = n->layers[li--];
        const NetLayer& c1 = n->layers[li--];
        // ga: dZ of dec l.c2, gb: of dec l.c1
        if ((rc = layer_dw(n, c2, V.d1, V.c, V.ga, V.c, V, nv))) return rc;
        layer_dx(n, c2, V.ga, V.c, V.gb, V, nv, V.d1);
        if ((rc = layer_dw(n, c1, V.cat, W.c + V.c, V.gb, V.c, V, nv))) return rc;
        layer_dx(n, c1, V.gb, V.c, V.dcat, V, nv, nullptr);
        // dZ of D_{l+1} (or S_{L-1}): up2^T of the first W.c channels
        hipLaunchKernelGGL(k_up_back, dim3(nblk(nv / 8), W.c / 8), dim3(256), 0, n->stream, V.dcat, W.lg, nv / 8, V.nvox,
                           W.nvox, l + 1 == L - 1 ? W.s : W.d, W.ga);
    }
    // encoder, bottom up; lv[L-1].ga holds dZ of S_{L-1}
    for (int l = L - 1; l >= 0; l--) {
        NetLevel& V = n->lv[l];
        const long nv = (long)batch << (3 * V.lg);
        const NetLayer& c2 = n->layers[2 * l + 1];
        const NetLayer& c1 = n->layers[2 * l];
        if (l < L - 1) {
            const NetLevel& W = n->lv[l + 1];
            const long o = W.c * V.nvox;  // S_l's planes of CAT_l
            hipLaunchKernelGGL(k_skip_grad, dim3(nblk(nv), V.c / 8), dim3(256), 0, n->stream, V.cat + o, V.dcat + o, W.din,
                               V.lg, nv, V.nvox, W.nvox, V.ga);
        }
        if ((rc = layer_dw(n, c2, V.e, V.c, V.ga, V.c, V, nv))) return rc;
        layer_dx(n, c2, V.ga, V.c, V.gb, V, nv, V.e);  // dZ of enc l.c1
        if ((rc = layer_dw(n, c1, V.in, c1.cinp, V.gb, V.c, V, nv))) return rc;
        if (l > 0) layer_dx(n, c1, V.gb, V.c, V.din, V, nv, nullptr);
    }
    NETCHK(n, hipGetLastError());
    if (loss) {
        std::vector<double> part(n->lblocks);
        NETCHK(n, hipMemcpyAsync(part.data(), n->lpart, sizeof(double) * n->lblocks, hipMemcpyDeviceToHost, n->stream));
        NETCHK(n, hipStreamSynchronize(n->stream));
        double s = 0;
        for (double v : part) s += v;
        *loss = s * inv;
    }
    return HOMO3D_OK;
}

int adam_step(homo3d_net* n, double lr) {
    n->adam_t++;
    const double b1 = 0.9, b2 = 0.999;
    const float c1 = (float)(1.0 / (1.0 - std::pow(b1, (double)n->adam_t)));
    const float c2 = (float)(1.0 / (1.0 - std::pow(b2, (double)n->adam_t)));
    hipLaunchKernelGGL(k_adam, dim3(nblk(n->nparam)), dim3(256), 0, n->stream, n->nparam, n->g, n->p, n->m1, n->m2,
                       (float)lr, (float)b1, (float)b2, c1, c2, 1e-8f);
    return pack_weights(n);
}

int stage_inputs(homo3d_net* n, const float* rho, int batch) {
    const long nsv = 1L << (3 * n->lv[0].lg);
    NETCHK(n, hipMemcpyAsync(n->rho, rho, sizeof(float) * nsv * batch, hipMemcpyHostToDevice, n->stream));
    hipLaunchKernelGGL(k_set_input, dim3(nblk(nsv * batch)), dim3(256), 0, n->stream, n->rho, nsv * batch, n->lv[0].in);
    return HOMO3D_OK;
}

// On the copy stream, after what the network's stream held before: the 75 MB of a 64^3 x 4 batch (3 ms from
// pageable memory, the host copying) arrive while the forward pass runs.  The caller has enqueued that pass,
// and goes on behind copy_done.
int stage_targets(homo3d_net* n, const float* t, int batch) {
    const long cnt = (1L << (3 * n->lv[0].lg)) * batch * kOut;
    NETCHK(n, hipMemcpyAsync(n->tstage, t, sizeof(float) * cnt, hipMemcpyHostToDevice, n->copy));
    hipLaunchKernelGGL(k_f32_to_bf16, dim3(nblk(cnt)), dim3(256), 0, n->copy, n->tstage, cnt, n->T);
    NETCHK(n, hipEventRecord(n->copy_done, n->copy));
    NETCHK(n, hipStreamWaitEvent(n->stream, n->copy_done, 0));
    return HOMO3D_OK;
}

void destroy(homo3d_net* n) {
    if (n->stream) (void)hipStreamSynchronize(n->stream);
    if (n->copy) (void)hipStreamSynchronize(n->copy);
    for (NetLayer& Ly : n->layers) {
        (void)hipFree(Ly.wf);
        (void)hipFree(Ly.wb);
        (void)hipFree(Ly.bias_pad);
    }
    for (NetLevel& V : n->lv) {
        void* ptrs[] = {V.in, V.e, V.cat, V.s, V.d1, V.d, V.ga, V.gb, V.dcat, V.din};
        for (void* q : ptrs)
            if (q) (void)hipFree(q);
    }
    void* ptrs[] = {n->p, n->g, n->m1, n->m2, n->P, n->T, n->dP, n->mean, n->wbar, n->chains, n->lpart, n->rho, n->tstage, n->partial, n->ds_in, n->ds_tg};
    for (void* q : ptrs)
        if (q) (void)hipFree(q);
    if (n->copy_start) (void)hipEventDestroy(n->copy_start);
    if (n->copy_done) (void)hipEventDestroy(n->copy_done);
    if (n->copy) (void)hipStreamDestroy(n->copy);
    if (n->stream) (void)hipStreamDestroy(n->stream);
    delete n;
}

}  // namespace

// ---------------------------------------------------------------------------------------------------
// Internal interface for api.cpp
// ---------------------------------------------------------------------------------------------------
namespace homo3d {
int net_grid(const homo3d_net* n) { return n->cfg.grid; }
int net_pred_ld(const homo3d_net*) { return kPld; }
float net_target_scale(const homo3d_net* n) { return (float)n->cfg.target_scale; }
hipStream_t net_stream(const homo3d_net* n) { return n->stream; }
uint16_t* net_input_slot(homo3d_net* n) { return n->lv[0].in; }
int net_forward_one(homo3d_net* n, const float** pred) {
    forward(n, 1);
    NETCHK(n, hipGetLastError());
    *pred = n->P;
    return HOMO3D_OK;
}
int net_dataset_push(homo3d_net* n, uint16_t** input, uint16_t** target) {
    if (n->ds_count >= n->ds_cap) return nerr(n, HOMO3D_BAD_ARG, "dataset full (%d pairs)", n->ds_cap);
    const long nsv = (long)n->cfg.grid * n->cfg.grid * n->cfg.grid;
    *input = n->ds_in + (long)n->ds_count * nsv * kInCh;
    *target = n->ds_tg + (long)n->ds_count * nsv * kOut;
    n->ds_count++;
    return HOMO3D_OK;
}
int net_set_error(homo3d_net* n, int code, const char* msg) { return nerr(n, code, "%s", msg); }
}  // namespace homo3d

// ---------------------------------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------------------------------
extern "C" {

void homo3d_net_default_config(homo3d_net_config* c) {
    if (!c) return;
    std::memset(c, 0, sizeof(*c));
    c->grid = 64;
    c->levels = 4;
    c->base_channels = 16;
    c->batch = 4;
    c->target_scale = 8.0;
    c->seed = 0;
    c->device = 0;
}

int homo3d_net_create(const homo3d_net_config* cfg, homo3d_net** out) {
    if (!cfg || !out) return HOMO3D_BAD_ARG;
    *out = nullptr;
    const int g = cfg->grid, L = cfg->levels, c0 = cfg->base_channels, B = cfg->batch;
    int lg = 0;
    while ((1 << lg) < g) lg++;
    if ((1 << lg) != g || L < 1 || L > 6 || (g >> (L - 1)) < 8 || c0 < 8 || c0 % 8 || (c0 << (L - 1)) > 256 || B < 1 ||
        B > 64 || !(cfg->target_scale > 0))
        return HOMO3D_NO_SUPPORT;
    homo3d_net* n = new homo3d_net();
    n->cfg = *cfg;
    n->L = L;
    auto fail = [&](int code) {
        destroy(n);
        return code;
    };
    if (hipSetDevice(cfg->device) != hipSuccess) return fail(HOMO3D_HIP_ERROR);
    if (hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking) != hipSuccess ||
        hipStreamCreateWithFlags(&n->copy, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&n->copy_start, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&n->copy_done, hipEventDisableTiming) != hipSuccess)
        return fail(HOMO3D_HIP_ERROR);
    // layers (parameter order: enc0.c1, enc0.c2, ..., enc{L-1}.c2, dec{L-2}.c1, dec{L-2}.c2, ..., dec0.c2, head)
    auto add = [&](int cin, int cinp, int cout, int taps, bool relu, bool need_dx) {
        NetLayer Ly;
        Ly.cin = cin;
        Ly.cinp = cinp;
        Ly.cout = cout;
        Ly.taps = taps;
        Ly.relu = relu;
        Ly.off_w = n->nparam;
        n->nparam += (long)cout * taps * cin;
        Ly.off_b = n->nparam;
        n->nparam += cout;
        Ly.mb_f = pick_mb(cout);
        Ly.rows_f = round_up(cout, 16 * Ly.mb_f);
        Ly.kpad_f = round_up(taps * cinp, 32);
        Ly.coutp = round_up(cout, 8);
        Ly.mb_b = pick_mb(cin);
        Ly.rows_b = round_up(cin, 16 * Ly.mb_b);
        Ly.kpad_b = round_up(taps * Ly.coutp, 32);
        n->layers.push_back(Ly);
        NetLayer& Q = n->layers.back();
        return !(hipMalloc(&Q.wf, sizeof(uint16_t) * Q.rows_f * Q.kpad_f) ||
                 hipMalloc(&Q.bias_pad, sizeof(float) * Q.rows_f) ||
                 (need_dx && hipMalloc(&Q.wb, sizeof(uint16_t) * Q.rows_b * Q.kpad_b)));
    };
    std::vector<int> ch(L);
    for (int l = 0; l < L; l++) ch[l] = c0 << l;
    bool ok = true;
    for (int l = 0; l < L && ok; l++) {
        ok = add(l == 0 ? 1 : ch[l - 1], l == 0 ? kInCh : ch[l - 1], ch[l], 27, true, l > 0) &&
             add(ch[l], ch[l], ch[l], 27, true, true);
    }
    for (int l = L - 2; l >= 0 && ok; l--)
        ok = add(ch[l + 1] + ch[l], ch[l + 1] + ch[l], ch[l], 27, true, true) && add(ch[l], ch[l], ch[l], 27, true, true);
    ok = ok && add(ch[0], ch[0], kOut, 1, false, true);
    if (!ok) return fail(HOMO3D_HIP_ERROR);
    // activations
    n->lv.resize(L);
    size_t max_part = 0;
    for (int l = 0; l < L; l++) {
        NetLevel& V = n->lv[l];
        V.g = g >> l;
        V.lg = lg - l;
        V.c = ch[l];
        V.nvox = (long)B << (3 * V.lg);
        const long nv = V.nvox;
        const int cin = l == 0 ? kInCh : ch[l - 1];
        const int cu = l < L - 1 ? ch[l + 1] : 0;
        auto mal = [&](uint16_t** q, long elems) { return hipMalloc((void**)q, sizeof(uint16_t) * elems) == hipSuccess; };
        ok = mal(&V.in, nv * cin) && mal(&V.e, nv * V.c) && mal(&V.ga, nv * std::max(V.c, 1)) && mal(&V.gb, nv * V.c);
        if (l > 0) ok = ok && mal(&V.din, nv * cin);
        if (l < L - 1)
            ok = ok && mal(&V.cat, nv * (cu + V.c)) && mal(&V.dcat, nv * (cu + V.c)) && mal(&V.d1, nv * V.c) &&
                 mal(&V.d, nv * V.c);
        else
            ok = ok && mal(&V.s, nv * V.c);
        if (!ok) return fail(HOMO3D_HIP_ERROR);
        if (l == 0 && hipMemset(V.in, 0, sizeof(uint16_t) * nv * kInCh)) return fail(HOMO3D_HIP_ERROR);
    }
    // weight-gradient partials, for every layer (in the parameters' order) and every batch size up to B
    for (size_t i = 0; i < n->layers.size(); i++) {
        const NetLayer& Ly = n->layers[i];
        const bool head = i + 1 == n->layers.size();
        const int l = head ? 0 : (int)i < 2 * L ? (int)i / 2 : L - 2 - ((int)i - 2 * L) / 2;
        for (int b = 1; b <= B; b++) {
            const WgPlan w = wgrad_plan(head ? kDpC : Ly.cout, Ly.cinp, Ly.taps, n->lv[l].lg, (long)b << (3 * n->lv[l].lg));
            max_part = std::max(max_part, w.partial() * (Ly.taps * w.cxp + 1));
        }
    }
    n->partial_elems = max_part;
    const long nv0 = n->lv[0].nvox;
    if (hipMalloc(&n->p, sizeof(float) * n->nparam) || hipMalloc(&n->g, sizeof(float) * n->nparam) ||
        hipMalloc(&n->m1, sizeof(float) * n->nparam) || hipMalloc(&n->m2, sizeof(float) * n->nparam) ||
        hipMalloc(&n->P, sizeof(float) * nv0 * kPld) || hipMalloc(&n->T, sizeof(uint16_t) * nv0 * kOut) ||
        hipMalloc(&n->dP, sizeof(uint16_t) * nv0 * kDpC) || hipMalloc(&n->mean, sizeof(float) * B * kOut) || hipMalloc(&n->wbar, sizeof(float) * B) ||
        hipMalloc(&n->chains, sizeof(float) * B * kMeanRow * kChains) ||
        hipMalloc(&n->lpart, sizeof(double) * n->lblocks) || hipMalloc(&n->rho, sizeof(float) * nv0) ||
        hipMalloc(&n->tstage, sizeof(float) * nv0 * kOut) ||
        hipMalloc(&n->partial, sizeof(float) * max_part))
        return fail(HOMO3D_HIP_ERROR);
    if (hipMemset(n->dP, 0, sizeof(uint16_t) * nv0 * kDpC) || hipMemset(n->m1, 0, sizeof(float) * n->nparam) ||
        hipMemset(n->m2, 0, sizeof(float) * n->nparam) || hipMemset(n->P, 0, sizeof(float) * nv0 * kPld))
        return fail(HOMO3D_HIP_ERROR);
    // He-normal initial weights (head: sqrt(1 / cin) / 4), zero biases
    std::vector<float> hp(n->nparam, 0.f);
    std::mt19937_64 rng(cfg->seed);
    std::normal_distribution<double> nd(0.0, 1.0);
    for (const NetLayer& Ly : n->layers) {
        const double sd = Ly.relu ? std::sqrt(2.0 / (Ly.taps * Ly.cin)) : std::sqrt(1.0 / Ly.cin) / 4;
        for (long i = 0; i < (long)Ly.cout * Ly.taps * Ly.cin; i++) hp[Ly.off_w + i] = (float)(nd(rng) * sd);
    }
    if (hipMemcpy(n->p, hp.data(), sizeof(float) * n->nparam, hipMemcpyHostToDevice)) return fail(HOMO3D_HIP_ERROR);
    if (pack_weights(n)) return fail(HOMO3D_HIP_ERROR);
    if (hipStreamSynchronize(n->stream)) return fail(HOMO3D_HIP_ERROR);
    *out = n;
    return HOMO3D_OK;
}

int homo3d_net_destroy(homo3d_net* n) {
    if (n) destroy(n);
    return HOMO3D_OK;
}

const char* homo3d_net_last_error(const homo3d_net* n) { return n ? n->err.c_str() : "null network"; }

long homo3d_net_num_params(const homo3d_net* n) { return n ? n->nparam : -1; }

int homo3d_net_params(homo3d_net* n, float* host, int to_device) {
    if (!n || !host) return HOMO3D_BAD_ARG;
    if (to_device) {
        NETCHK(n, hipMemcpyAsync(n->p, host, sizeof(float) * n->nparam, hipMemcpyHostToDevice, n->stream));
        NETCHK(n, hipMemsetAsync(n->m1, 0, sizeof(float) * n->nparam, n->stream));
        NETCHK(n, hipMemsetAsync(n->m2, 0, sizeof(float) * n->nparam, n->stream));
        n->adam_t = 0;
        int rc = pack_weights(n);
        if (rc) return rc;
    } else {
        NETCHK(n, hipMemcpyAsync(host, n->p, sizeof(float) * n->nparam, hipMemcpyDeviceToHost, n->stream));
    }
    NETCHK(n, hipStreamSynchronize(n->stream));
    return HOMO3D_OK;
}

int homo3d_net_forward(homo3d_net* n, const float* rho, int batch, float* out) {
    if (!n || !rho || !out) return HOMO3D_BAD_ARG;
    if (batch < 1 || batch > n->cfg.batch) return nerr(n, HOMO3D_BAD_ARG, "batch %d outside [1, %d]", batch, n->cfg.batch);
    int rc = stage_inputs(n, rho, batch);
    if (rc) return rc;
    forward(n, batch);
    const long count = ((long)batch << (3 * n->lv[0].lg)) * kOut;
    hipLaunchKernelGGL(k_pack_pred, dim3(nblk(count)), dim3(256), 0, n->stream, n->P, count, n->tstage);
    NETCHK(n, hipGetLastError());
    NETCHK(n, hipMemcpyAsync(out, n->tstage, sizeof(float) * count, hipMemcpyDeviceToHost, n->stream));
    NETCHK(n, hipStreamSynchronize(n->stream));
    return HOMO3D_OK;
}

int homo3d_net_loss_grad(homo3d_net* n, const float* rho, const float* target, int batch, double* loss, float* grad) {
    if (!n || !rho || !target || !loss) return HOMO3D_BAD_ARG;
    if (batch < 1 || batch > n->cfg.batch) return nerr(n, HOMO3D_BAD_ARG, "batch %d outside [1, %d]", batch, n->cfg.batch);
    NETCHK(n, hipEventRecord(n->copy_start, n->stream));
    NETCHK(n, hipStreamWaitEvent(n->copy, n->copy_start, 0));
    int rc = stage_inputs(n, rho, batch);
    if (rc) return rc;
    forward(n, batch);
    if ((rc = stage_targets(n, target, batch))) return rc;
    rc = loss_backward(n, batch, loss);
    if (rc) return rc;
    if (grad) NETCHK(n, hipMemcpyAsync(grad, n->g, sizeof(float) * n->nparam, hipMemcpyDeviceToHost, n->stream));
    NETCHK(n, hipStreamSynchronize(n->stream));
    return HOMO3D_OK;
}

int homo3d_net_train_step(homo3d_net* n, const float* rho, const float* target, int batch, double lr, double* loss) {
    double l = 0;
    int rc = homo3d_net_loss_grad(n, rho, target, batch, &l, nullptr);
    if (rc) return rc;
    rc = adam_step(n, lr);
    if (rc) return rc;
    NETCHK(n, hipStreamSynchronize(n->stream));
    if (loss) *loss = l;
    return HOMO3D_OK;
}

int homo3d_net_dataset_reserve(homo3d_net* n, int count) {
    if (!n || count < 1) return HOMO3D_BAD_ARG;
    NETCHK(n, hipStreamSynchronize(n->stream));
    if (n->ds_in) (void)hipFree(n->ds_in);
    if (n->ds_tg) (void)hipFree(n->ds_tg);
    n->ds_in = n->ds_tg = nullptr;
    n->ds_cap = n->ds_count = 0;
    const long nsv = (long)n->cfg.grid * n->cfg.grid * n->cfg.grid;
    NETCHK(n, hipMalloc(&n->ds_in, sizeof(uint16_t) * nsv * kInCh * count));
    NETCHK(n, hipMalloc(&n->ds_tg, sizeof(uint16_t) * nsv * kOut * count));
    n->ds_cap = count;
    return HOMO3D_OK;
}

int homo3d_net_dataset_size(const homo3d_net* n) { return n ? n->ds_count : -1; }

// Adam epochs over the first `count` pairs of the device-resident dataset (all when count <= 0): each epoch
// visits them in a seeded random order in batches of the configured size (the last partial batch is
// dropped).  losses[e] = mean batch loss of epoch e.
int homo3d_net_train(homo3d_net* n, int epochs, int count, double lr, uint64_t seed, double* losses) {
    if (!n || epochs < 0) return HOMO3D_BAD_ARG;
    const int B = n->cfg.batch;
    if (count <= 0 || count > n->ds_count) count = n->ds_count;
    if (count < B) return nerr(n, HOMO3D_BAD_ARG, "training on %d pairs, fewer than one batch", count);
    const long nsv = (long)n->cfg.grid * n->cfg.grid * n->cfg.grid;
    std::mt19937_64 rng(seed);
    std::vector<int> order(count);
    for (int i = 0; i < count; i++) order[i] = i;
    for (int e = 0; e < epochs; e++) {
        std::shuffle(order.begin(), order.end(), rng);
        double sum = 0;
        int steps = 0;
        for (int s = 0; s + B <= count; s += B) {
            for (int b = 0; b < B; b++) {
                const long k = order[s + b];
                NETCHK(n, hipMemcpyAsync(n->lv[0].in + b * nsv * kInCh, n->ds_in + k * nsv * kInCh,
                                         sizeof(uint16_t) * nsv * kInCh, hipMemcpyDeviceToDevice, n->stream));
                NETCHK(n, hipMemcpyAsync(n->T + b * nsv * kOut, n->ds_tg + k * nsv * kOut, sizeof(uint16_t) * nsv * kOut,
                                         hipMemcpyDeviceToDevice, n->stream));
            }
            forward(n, B);
            double l = 0;
            int rc = loss_backward(n, B, &l);
            if (rc) return rc;
            rc = adam_step(n, lr);
            if (rc) return rc;
            sum += l;
            steps++;
        }
        if (losses) losses[e] = steps ? sum / steps : 0.0;
    }
    NETCHK(n, hipStreamSynchronize(n->stream));
    return HOMO3D_OK;
}

// Mean loss of the network over dataset pairs [first, first + count) (no update).
int homo3d_net_eval(homo3d_net* n, int first, int count, double* loss) {
    if (!n || !loss || first < 0 || count < 1 || first + count > n->ds_count) return HOMO3D_BAD_ARG;
    const long nsv = (long)n->cfg.grid * n->cfg.grid * n->cfg.grid;
    double sum = 0;
    for (int k = first; k < first + count; k++) {
        NETCHK(n, hipMemcpyAsync(n->lv[0].in, n->ds_in + (long)k * nsv * kInCh, sizeof(uint16_t) * nsv * kInCh,
                                 hipMemcpyDeviceToDevice, n->stream));
        NETCHK(n, hipMemcpyAsync(n->T, n->ds_tg + (long)k * nsv * kOut, sizeof(uint16_t) * nsv * kOut,
                                 hipMemcpyDeviceToDevice, n->stream));
        forward(n, 1);
        double l = 0;
        int rc = loss_backward(n, 1, &l);
        if (rc) return rc;
        sum += l;
    }
    *loss = sum / count;
    return HOMO3D_OK;
}

}  // extern "C"
