// Smoothing on the small coarse levels (stored 27-point stencils), where a colour pass is too little work
// for a launch of its own.
//
// A pass over one of the eight colours of a level of at most 32^3 vertices has 4096 of them at most, and
// one thread a vertex and load case walked 27 neighbours in a chain of loads: 6 us a launch and 2 us
// between launches, eight launches a sweep, whatever the size.  Here a launch does four colours.  The
// colours c and c + 1, c + 2, c + 3 of one z-parity differ in x- and y-parity only, so a vertex of one
// depends on the others through neighbours in its own z-plane, and planes of the same parity do not meet: a
// workgroup owns a z-plane for one load case, keeps that plane and its two neighbours
// of u in LDS, and updates the four colours in turn between barriers.  Three threads share a vertex, one per
// neighbour plane: each has its 9 stencil blocks (11 st of words) in flight at once, those of the next
// colour before the barriers of this one.  Bound by that load latency and the barriers: a sweep takes two
// launches of 8 us at 8^3 to 16^3 and 12 us at 32^3, where eight of 6 us each took 65 us with their gaps.
// Levels above 32^3 fill the GPU with one or two colours a launch and stream their stencils; FP32 stencils
// are twice the registers (both sets in flight spilled some 70 of them), so those levels keep the
// one-colour kernels as well.
#include <hip/hip_runtime.h>

#include "kernels.h"
#include "level.h"

namespace homo3d {

namespace {

constexpr int kPlaneVerts = 256;  // most vertices a workgroup updates at a time

// The nine blocks of a neighbour plane g = dz + 1: entries 81 g .. 81 g + 80 of the stencil, which start g
// entries into quad first(g).
struct PlaneBlocks {
    typedef uint32_t Quad __attribute__((ext_vector_type(4)));
    static constexpr int st = 11;
    Quad w[st];
    __device__ __forceinline__ void load(Rsrc rs, uint32_t N, int g, uint32_t v, bool live) {
        const uint32_t q0 = (uint32_t)(81 * g / 8);
#pragma unroll
        for (int q = 0; q < st; q++) {
            if (live)
                w[q] = __builtin_bit_cast(Quad, __builtin_amdgcn_raw_buffer_load_b128(
                                                    rs, (int)(v * 16u), (int)((q0 + (uint32_t)q) * N * 16u), 0));
        }
    }
    template <int G>
    __device__ __forceinline__ float get(int e) const {
        return (float)__builtin_bit_cast(half2_t, (uint32_t)w[(e + G) >> 3][((e + G) >> 1) & 3])[(e + G) & 1];
    }
};

// acc += the blocks of plane G times its u (pl: the plane's three components in LDS, cs words apart); the
// vertex itself left out.
template <int G>
__device__ __forceinline__ void plane_sum(const PlaneBlocks& w, const float* pl, int cs, const int (&xo)[3],
                                          const int (&yo)[3], float (&acc)[3]) {
#pragma unroll
    for (int d = 0; d < 9; d++) {
        if (d == 4 && G == 1) continue;
        float S[9];
#pragma unroll
        for (int k = 0; k < 9; k++) S[k] = w.template get<G>(9 * d + k);
        const float* q = pl + yo[d / 3] + xo[d % 3];
        const float u0 = q[0], u1 = q[cs], u2 = q[2 * cs];
#pragma unroll
        for (int i = 0; i < 3; i++)
            acc[i] = fmaf(S[3 * i], u0, fmaf(S[3 * i + 1], u1, fmaf(S[3 * i + 2], u2, acc[i])));
    }
}

// Stage plane z of load case r of u in LDS: natural (y, x) order, n2 words a component.
__device__ __forceinline__ void stage_plane(float* dst, const Lay& L, size_t N, const float* __restrict__ u, int r,
                                            int z) {
    const int n = L.n, h = L.h, h2 = h * h, n2 = n * n;
    const uint32_t zp = L.part(z, 2);
    for (int t = threadIdx.x; t < n2; t += blockDim.x) {
        const int b = t / h2, l = t - b * h2, yy = l / h, xx = l - yy * h;
        const uint32_t v = zp + (uint32_t)(b & 1) * L.h3 + (uint32_t)(b >> 1) * 2u * L.h3 + (uint32_t)l;
        float* q = dst + (2 * yy + (b >> 1)) * n + 2 * xx + (b & 1);
#pragma unroll
        for (int i = 0; i < 3; i++) q[i * n2] = u[(size_t)(r * 3 + i) * N + v];
    }
}

// Colours 4 (1 - pz) .. + 3 of a sweep (in falling order when REVERSE) on the planes z of parity pz, load
// case blockIdx.y.  zero: 0 an ordinary sweep; u = 0 before the sweep whatever it holds, and
// this is its first (1: the neighbouring planes are zero too) or second launch (2).  The blocks of the next
// colour are loaded while this one's are used.
template <bool REVERSE>
__global__ __launch_bounds__(3 * kPlaneVerts) void k_plane_gs(Lay L, size_t N, int pz, float omega, int zero,
                                                              const uint4* __restrict__ st, float* __restrict__ u,
                                                              const float* __restrict__ f) {
    constexpr int NM = 32;
    __shared__ float us[3 * 3 * NM * NM];
    __shared__ float red[2][kPlaneVerts][3];
    const int n = L.n, h = L.h, n2 = n * n, h2 = h * h;
    const int vb = (int)blockDim.x / 3, g = __builtin_amdgcn_readfirstlane((int)threadIdx.x / vb);
    const int lv = (int)threadIdx.x - g * vb;
    const int kz = (int)blockIdx.x, z = 2 * kz + pz, r = (int)blockIdx.y;
    const Rsrc rs = make_rsrc(st, (size_t)StencilIO<half2_t>::words * N * 4);
    const bool live = lv < h2, load = live && !(zero == 1 && g != 1);  // the neighbour planes may be zero
    const int yy = lv / h, xx = lv - yy * h;
    const uint32_t v0 = (uint32_t)pz * 4u * L.h3 + (uint32_t)lv + (uint32_t)h2 * (uint32_t)kz;
    auto colour = [&](int s) { return REVERSE ? 3 - s : s; };
    auto vertex = [&](int s) {
        const int c = colour(s);
        return v0 + (uint32_t)((1 - (c & 1)) + 2 * (1 - (c >> 1))) * L.h3;
    };
    auto load_f = [&](int s, float (&ff)[3]) __attribute__((always_inline)) {
        if (g == 1 && live && s < 4) {
#pragma unroll
            for (int i = 0; i < 3; i++) ff[i] = f[(size_t)(r * 3 + i) * N + vertex(s)];
        }
    };
    PlaneBlocks cur;
    float ff[3];
    cur.load(rs, (uint32_t)N, g, vertex(0), load);
    load_f(0, ff);
    if (zero) {
        for (int t = threadIdx.x; t < 3 * n2; t += blockDim.x) us[3 * n2 + t] = 0.f;
    } else {
        stage_plane(us + 3 * n2, L, N, u, r, z);
    }
    if (zero != 1) {
        stage_plane(us, L, N, u, r, z == 0 ? n - 1 : z - 1);
        stage_plane(us + 6 * n2, L, N, u, r, z == n - 1 ? 0 : z + 1);
    }
    __syncthreads();
#pragma unroll 1
    for (int s = 0; s < 4; s++) {
        PlaneBlocks nxt;
        float fn[3];
        nxt.load(rs, (uint32_t)N, g, vertex(s + 1), load && s < 3);
        load_f(s + 1, fn);
        float acc[3] = {0.f, 0.f, 0.f}, Ks[9];
        const int c4 = colour(s), x = 2 * xx + 1 - (c4 & 1), y = 2 * yy + 1 - (c4 >> 1), me = y * n + x;
        if (load) {
            const int xo[3] = {x == 0 ? n - 1 : x - 1, x, x == n - 1 ? 0 : x + 1};
            const int yo[3] = {(y == 0 ? n - 1 : y - 1) * n, y * n, (y == n - 1 ? 0 : y + 1) * n};
            const float* pl = us + 3 * n2 * g;
            if (g == 1) {
                plane_sum<1>(cur, pl, n2, xo, yo, acc);
#pragma unroll
                for (int k = 0; k < 9; k++) Ks[k] = cur.template get<1>(36 + k);
            } else {
                if (g == 0)
                    plane_sum<0>(cur, pl, n2, xo, yo, acc);
                else
                    plane_sum<2>(cur, pl, n2, xo, yo, acc);
#pragma unroll
                for (int i = 0; i < 3; i++) red[g >> 1][lv][i] = acc[i];
            }
        }
        __syncthreads();
        if (g == 1 && live) {
            const float inv[3] = {1.f / Ks[0], 1.f / Ks[4], 1.f / Ks[8]};
            float* own = us + 3 * n2 + me;
            float uu[3];
#pragma unroll
            for (int i = 0; i < 3; i++) {
                uu[i] = own[i * n2];
                if (zero != 1) acc[i] += red[0][lv][i] + red[1][lv][i];
            }
            block_update<REVERSE>(uu, ff, acc, Ks, inv, omega);
#pragma unroll
            for (int i = 0; i < 3; i++) {
                own[i * n2] = uu[i];
                u[(size_t)(r * 3 + i) * N + vertex(s)] = uu[i];
            }
        }
        __syncthreads();
        cur = nxt;
#pragma unroll
        for (int i = 0; i < 3; i++) ff[i] = fn[i];
    }
}

// ---------------------------------------------------------------------------------------------
// The bottom of a V-cycle in one launch: the last smoothed level (8 to 14 points an axis) and the coarsest
// (4 to 7), one workgroup per load case with every field in LDS.  Pre-smoothing from zero, residual,
// restriction, the coarsest solve, prolongation and post-smoothing were 20 launches of 5 to 15 us, some
// 160 us with their gaps; 51 us at 8^3 and 74 us at 10^3 now.  A colour is one or two steps of 256 vertices
// between barriers, bounded by the latency of its stencil words, which are loaded a step ahead.
// ---------------------------------------------------------------------------------------------
constexpr int kTailN = 14;
constexpr int kTailV = kTailN * kTailN * kTailN, kTailVc = 7 * 7 * 7;
constexpr int kTailOneM = 375;  // most unknowns of a coarsest system solved in the same launch
enum { kTailForward = 0, kTailReverse = 1, kTailResidual = 2 };

// Vertices of a colour taken at a time: its h^3 = 64 .. 343, in one step up to 256, else in two.
__device__ __forceinline__ int tail_verts(int h3) { return h3 <= 256 ? (h3 + 63) / 64 * 64 : 192; }

// One pass over the level's vertices colour by colour: a GS sweep of u, or r = f - A u.
template <int MODE>
__device__ __forceinline__ void tail_pass(const Lay& L, size_t N, float omega, const uint4* __restrict__ st, float* u,
                                          const float* f, float* r, float (*red)[kPlaneVerts][3]) {
    const int n = L.n, h = L.h, n2 = n * n, n3 = n2 * n, h3 = (int)L.h3, vb = tail_verts(h3);
    const int g = __builtin_amdgcn_readfirstlane((int)threadIdx.x / vb), lv = (int)threadIdx.x - g * vb;
    const Rsrc rs = make_rsrc(st, (size_t)StencilIO<half2_t>::words * N * 4);
    const int nch = h3 <= vb ? 1 : 2, steps = 8 * nch;
    int pos[2];  // half coordinates of the thread's vertex in each chunk, 4 bits each; -1: none
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const int i = k * vb + lv, zz = i / (h * h), yy = (i - zz * h * h) / h, xx = i - (zz * h + yy) * h;
        pos[k] = g < 3 && k < nch && i < h3 ? xx | yy << 4 | zz << 8 : -1;
    }
    auto colour = [&](int s) {
        const int q = nch == 1 ? s : s >> 1;
        return MODE == kTailReverse ? 7 - q : q;
    };
    auto chunk = [&](int s) { return nch == 1 ? 0 : s & 1; };
    auto vertex = [&](int s) { return (uint32_t)((7 - colour(s)) * h3 + chunk(s) * vb + lv); };
    PlaneBlocks cur;
    cur.load(rs, (uint32_t)N, g, vertex(0), pos[0] >= 0);
#pragma unroll 1
    for (int s = 0; s < steps; s++) {
        const int nk = s + 1 < steps ? (chunk(s + 1) ? pos[1] : pos[0]) : -1;
        PlaneBlocks nxt;
        nxt.load(rs, (uint32_t)N, g, vertex(s + 1), nk >= 0);
        float acc[3] = {0.f, 0.f, 0.f}, Ks[9];
        const int me3 = chunk(s) ? pos[1] : pos[0];
        int me = 0;
        if (me3 >= 0) {
            const int c = 7 - colour(s);  // the block: its coordinate parities
            const int x = 2 * (me3 & 15) + (c & 1), y = 2 * (me3 >> 4 & 15) + (c >> 1 & 1), z = 2 * (me3 >> 8) + (c >> 2);
            me = x + n * y + n2 * z;
            const int xo[3] = {x == 0 ? n - 1 : x - 1, x, x == n - 1 ? 0 : x + 1};
            const int yo[3] = {(y == 0 ? n - 1 : y - 1) * n, y * n, (y == n - 1 ? 0 : y + 1) * n};
            if (g == 1) {
                plane_sum<1>(cur, u + n2 * z, n3, xo, yo, acc);
#pragma unroll
                for (int k = 0; k < 9; k++) Ks[k] = cur.template get<1>(36 + k);
            } else {
                if (g == 0)
                    plane_sum<0>(cur, u + n2 * (z == 0 ? n - 1 : z - 1), n3, xo, yo, acc);
                else
                    plane_sum<2>(cur, u + n2 * (z == n - 1 ? 0 : z + 1), n3, xo, yo, acc);
#pragma unroll
                for (int i = 0; i < 3; i++) red[g >> 1][lv][i] = acc[i];
            }
        }
        __syncthreads();
        if (g == 1 && me3 >= 0) {
            float uu[3], ff[3];
#pragma unroll
            for (int i = 0; i < 3; i++) {
                uu[i] = u[me + i * n3];
                ff[i] = f[me + i * n3];
                acc[i] += red[0][lv][i] + red[1][lv][i];
            }
            if constexpr (MODE == kTailResidual) {
#pragma unroll
                for (int i = 0; i < 3; i++)
                    r[me + i * n3] = ff[i] - acc[i] -
                                     fmaf(Ks[3 * i], uu[0], fmaf(Ks[3 * i + 1], uu[1], Ks[3 * i + 2] * uu[2]));
            } else {
                const float inv[3] = {1.f / Ks[0], 1.f / Ks[4], 1.f / Ks[8]};
                block_update<MODE == kTailReverse>(uu, ff, acc, Ks, inv, omega);
#pragma unroll
                for (int i = 0; i < 3; i++) u[me + i * n3] = uu[i];
            }
        }
        __syncthreads();
        cur = nxt;
    }
}

// down: from f to the coarsest right-hand side; solve: the coarsest system; up: back to u.  A part that is
// not run leaves or finds its fields in memory (u, f, residual of the level; uc, fc of the lexicographic
// coarsest); the fields a run of the separate passes would leave there are written too.
__global__ __launch_bounds__(3 * kPlaneVerts) void k_tail(Lay L, size_t N, float omega, int reverse, int down, int solve,
                                                          int up, const uint4* __restrict__ st, float* __restrict__ u,
                                                          const float* __restrict__ f, float* __restrict__ res,
                                                          int nc, float* __restrict__ uc, float* __restrict__ fc,
                                                          const double* __restrict__ Ainv) {
    __shared__ float su[3 * kTailV], sf[3 * kTailV], sr[3 * kTailV], sc[2][3 * kTailVc], red[2][kPlaneVerts][3];
    const int n = L.n, n3 = n * n * n, Nc = nc * nc * nc, m = 3 * Nc, r = (int)blockIdx.x, nt = (int)blockDim.x;
    for (int t = threadIdx.x; t < n3; t += nt) {
        int x, y, z;
        L.pos((uint32_t)t, x, y, z);
        const int q = x + n * (y + n * z);
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const size_t o = (size_t)(r * 3 + i) * N + t;
            sf[q + i * n3] = f[o];
            su[q + i * n3] = down ? 0.f : u[o];
        }
    }
    __syncthreads();
    if (down) {
        tail_pass<kTailForward>(L, N, omega, st, su, sf, sr, red);
        tail_pass<kTailResidual>(L, N, omega, st, su, sf, sr, red);
        for (int t = threadIdx.x; t < m; t += nt) {
            const int i = t / Nc, V = t - i * Nc, X = V % nc, Y = V / nc % nc, Z = V / (nc * nc);
            float a = 0.f;
            for (int o = 0; o < 27; o++) {
                const int ox = o % 3 - 1, oy = o / 3 % 3 - 1, oz = o / 9 - 1;
                int x = 2 * X + ox, y = 2 * Y + oy, z = 2 * Z + oz;
                x = x < 0 ? n - 1 : x;
                y = y < 0 ? n - 1 : y;
                z = z < 0 ? n - 1 : z;
                a = fmaf(hat(ox) * hat(oy) * hat(oz), sr[x + n * (y + n * z) + i * n3], a);
            }
            sc[0][3 * V + i] = a;
            fc[(size_t)(r * 3 + i) * Nc + V] = a;
        }
    }
    if (solve) {
        __syncthreads();
        // a wave takes four rows at a time and has all their loads in flight together
        constexpr int KM = (kTailOneM + 63) / 64;
        const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6), nw = nt / 64;
        for (int row0 = 4 * wave; row0 < m; row0 += 4 * nw) {
            double a[4][KM], sum[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int k = 0; k < KM; k++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    a[q][k] = lane + 64 * k < m && row0 + q < m ? Ainv[(size_t)(row0 + q) * m + lane + 64 * k] : 0.0;
#pragma unroll
            for (int k = 0; k < KM; k++) {
                const double fk = lane + 64 * k < m ? (double)sc[0][lane + 64 * k] : 0.0;
#pragma unroll
                for (int q = 0; q < 4; q++) sum[q] = fma(a[q][k], fk, sum[q]);
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
#pragma unroll
                for (int off = 32; off > 0; off >>= 1) sum[q] += __shfl_xor(sum[q], off, 64);
                if (lane == q && row0 + q < m) {
                    sc[1][row0 + q] = (float)sum[q];
                    uc[(size_t)(r * 3 + (row0 + q) % 3) * Nc + (row0 + q) / 3] = (float)sum[q];
                }
            }
        }
    } else if (up) {
        for (int t = threadIdx.x; t < m; t += nt) {
            const int i = t / Nc, V = t - i * Nc;
            sc[1][3 * V + i] = uc[(size_t)(r * 3 + i) * Nc + V];
        }
    }
    __syncthreads();
    if (up) {
        for (int t = threadIdx.x; t < n3; t += nt) {
            const int x = t % n, y = t / n % n, z = t / (n * n);
            // the coarse neighbours below and above along each axis (one and the same at even points)
            const int cx[2] = {x >> 1, (x + 1) / 2 == nc ? 0 : (x + 1) / 2}, cy[2] = {y >> 1, (y + 1) / 2 == nc ? 0 : (y + 1) / 2},
                      cz[2] = {z >> 1, (z + 1) / 2 == nc ? 0 : (z + 1) / 2};
            float a[3] = {0.f, 0.f, 0.f};
#pragma unroll
            for (int b = 0; b < 8; b++) {
                const float* q = &sc[1][3 * (cx[b & 1] + nc * (cy[b >> 1 & 1] + nc * cz[b >> 2]))];
#pragma unroll
                for (int i = 0; i < 3; i++) a[i] += q[i];
            }
#pragma unroll
            for (int i = 0; i < 3; i++) su[t + i * n3] = fmaf(0.125f, a[i], su[t + i * n3]);
        }
        __syncthreads();
        if (reverse)
            tail_pass<kTailReverse>(L, N, omega, st, su, sf, sr, red);
        else
            tail_pass<kTailForward>(L, N, omega, st, su, sf, sr, red);
    }
    for (int t = threadIdx.x; t < n3; t += nt) {
        int x, y, z;
        L.pos((uint32_t)t, x, y, z);
#pragma unroll
        for (int i = 0; i < 3; i++) {
            u[(size_t)(r * 3 + i) * N + t] = su[x + n * (y + n * z) + i * n3];
            if (down) res[(size_t)(r * 3 + i) * N + t] = sr[x + n * (y + n * z) + i * n3];
        }
    }
}

}  // namespace

int small_level_ok(int n, int lex, int st_half) { return st_half && !lex && n % 2 == 0 && n >= 4 && n <= 32; }

int vcycle_tail_ok(int n, int lex, int st_half) { return small_level_ok(n, lex, st_half) && n >= 8 && n <= kTailN; }

void launch_vcycle_tail(hipStream_t s, int n, float omega, int reverse, const void* st, float* u, const float* f,
                        float* res, float* uc, float* fc, const double* Ainv) {
    const size_t N = (size_t)n * n * n;
    const Lay L = make_lay(n, 0);
    // one workgroup reads the whole inverse (8 m^2 bytes at some 150 GB/s): up to 375 unknowns that is
    // less than the two launches it saves, beyond it the solve is a launch of its own over the whole GPU
    const bool one = 3 * (n / 2) * (n / 2) * (n / 2) <= kTailOneM;
    for (int part = one ? 0 : 1; part <= (one ? 0 : 2); part++) {
        if (part == 2) launch_coarse_solve(s, n / 2, Ainv, fc, uc);
        hipLaunchKernelGGL(k_tail, dim3(6), dim3(3 * kPlaneVerts), 0, s, L, N, omega, reverse, part != 2 ? 1 : 0,
                           part == 0 ? 1 : 0, part != 1 ? 1 : 0, static_cast<const uint4*>(st), u, f, res, n / 2, uc,
                           fc, Ainv);
    }
}

void launch_plane_sweep(hipStream_t s, int n, float omega, int reverse, int zero_start, const void* st, float* u,
                        const float* f) {
    const size_t N = (size_t)n * n * n;
    const Lay L = make_lay(n, 0);
    const uint4* q = static_cast<const uint4*>(st);
    const int vb = (L.h * L.h + 63) / 64 * 64;
    const dim3 g(L.h, 6), b(3 * vb);
    for (int k = 0; k < 2; k++) {
        const int pz = reverse ? k : 1 - k;  // colours 0..3 are the odd planes
        if (reverse)
            hipLaunchKernelGGL((k_plane_gs<true>), g, b, 0, s, L, N, pz, omega, 0, q, u, f);
        else
            hipLaunchKernelGGL((k_plane_gs<false>), g, b, 0, s, L, N, pz, omega, zero_start ? k + 1 : 0, q, u, f);
    }
}

}  // namespace homo3d
