// gfx950 kernels of the periodic homogenization solve path.
//
// Grid convention: a cubic periodic level of n^3 vertices; vertex/cell id v = x + n*(y + n*z); cell
// (x,y,z) has its minimum corner at vertex (x,y,z); node b of a cell sits at corner +
// (b&1, b>>1&1, b>>2) (homogenization/templateMatrix.cpp:79-93).  Fields hold R = 6 load cases:
// component c of load case r of vertex v lives at (r*3 + c)*N + v.  Coarse stencils are stored
// structure-of-arrays: entry k = d*9 + i*3 + j (d = (dx+1) + 3(dy+1) + 9(dz+1)) of vertex v at k*N + v.
//
// The finest level is matrix-free: the 27 3x3 blocks of a vertex row are rebuilt from the 8 cell
// weights w_e = Emin + x_e and the element matrix KE, which is read with wave-uniform indices so
// the compiler keeps it in scalar registers.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

#include "../../include/homo3d.h"
#include "kernels.h"
#include "level.h"
#include "net.h"

namespace homo3d {

namespace {

// The FP64 iterate of the refinement loop stores its 18 components as nine planes of 16-byte pairs
// (u64_index), so a neighbour of all six load cases is nine 16-byte loads rather than eighteen
// 8-byte ones: the gather's cost is per load instruction.
typedef double double2_t __attribute__((ext_vector_type(2)));
template <>
__device__ __forceinline__ double2_t bload<double2_t>(Rsrc r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(double2_t, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0));
}

__device__ __forceinline__ void bstore(float v, Rsrc r, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, (int)voff, (int)soff, 0);
}

// the nine words of vertex idx of a packed FP16 field through a buffer resource over it (plane = 4 N
// bytes; the byte offsets stay below 36 N)
__device__ __forceinline__ void hload9(uint32_t (&wv)[9], Rsrc r, uint32_t idx, uint32_t plane) {
    const auto a = __builtin_amdgcn_raw_buffer_load_b128(r, (int)(idx * 16u), 0, 0);
    const auto b = __builtin_amdgcn_raw_buffer_load_b128(r, (int)(idx * 16u), (int)(4u * plane), 0);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        wv[k] = (uint32_t)a[k];
        wv[4 + k] = (uint32_t)b[k];
    }
    wv[8] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, (int)(idx * 4u), (int)(8u * plane), 0);
}

// The FP64 element matrix staged in LDS: KE (576 entries) followed by 243 block constants (kBlockConsts).
constexpr int kBlockConsts = 576;
constexpr int kKeStaged = 832;

// Sum over the cells that contain both v and v + d of the cell weights w_e, each with the sign
// prod over the axes m in SM of (e_m ? -1 : +1).  Cell e (0..7) sits at offset (e&1, e>>1&1, e>>2) - 1
// from v; it holds v + d iff e_m = (d_m + 1) / 2 on every axis with d_m != 0.
template <int D, int SM, typename T, typename W>
__device__ __forceinline__ T cell_form(const W wc[8]) {
    constexpr int dm[3] = {D % 3 - 1, D / 3 % 3 - 1, D / 9 - 1};
    T s = T(0);
    bool first = true;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        bool in = true;
#pragma unroll
        for (int m = 0; m < 3; m++)
            if (dm[m] != 0 && ((e >> m) & 1) != (dm[m] + 1) / 2) in = false;
        if (!in) continue;
        const bool neg = (__builtin_popcount(e & SM) & 1) != 0;
        const T we = (T)wc[e];
        s = first ? (neg ? -we : we) : (neg ? s - we : s + we);
        first = false;
    }
    return s;
}

// 3x3 block of the assembled fine operator between vertex v and its neighbour v+d:
// S = sum over the cells e containing both of w_e * KE[node(v)][node(v+d)], v being node 7-e of cell e.
// For the isotropic cube element, entry (i, j) of KE[a][b] over those cells is one constant times
// s_i s_j (i != j; s_m = +1 at the upper node of axis m, the sign of every axis along which d is
// non-zero being the same for all the cells) and one constant (i = j), so
// S_ij = C_d,ij * (sum of w_e, with the sign s_m(e) for each axis m in {i, j} along which d is zero).
// C_d,ij (BlockConsts) is the entry of the cell with e_m = 1 exactly where d_m = +1.  Four signed sums of
// two to eight weights and nine products per block, instead of nine FMAs per cell.
//
// The constants are wave-uniform and come through the scalar cache (kKeBlocks floats into ke, 12 a block,
// set when the operator is made), loaded a neighbour ahead: they cost neither vector loads, nor
// registers, nor the staging of KE at the start of a workgroup.  At 256^3 the CG pass takes 1.80 ms (1.87
// with the constants read from LDS) and a reverse colour pair 0.376 ms (0.389 with that and with its
// neighbours loaded one ahead instead of three).
struct BlockConsts {
    float v[9];
};
typedef const __attribute__((address_space(4))) float* KeBlocks;

__device__ __forceinline__ KeBlocks ke_blocks(const float* ke) { return (KeBlocks)(uintptr_t)(ke + kKeBlocks); }

template <int D>
__device__ __forceinline__ BlockConsts block_consts(KeBlocks kb) {
    BlockConsts c;
#pragma unroll
    for (int k = 0; k < 9; k++) c.v[k] = kb[12 * D + k];
    return c;
}

template <int D>
__device__ __forceinline__ void fine_block(const float wc[8], const BlockConsts& c, float S[9]) {
    constexpr int fm = (D % 3 == 1 ? 1 : 0) | (D / 3 % 3 == 1 ? 2 : 0) | (D / 9 == 1 ? 4 : 0);  // axes with d_m = 0
    const float* cb = c.v;
    const float w0 = cell_form<D, 0, float>(wc);
    const float fxy = cell_form<D, fm & 3, float>(wc), fxz = cell_form<D, fm & 5, float>(wc), fyz = cell_form<D, fm & 6, float>(wc);
    S[0] = cb[0] * w0;
    S[4] = cb[4] * w0;
    S[8] = cb[8] * w0;
    S[1] = cb[1] * fxy;
    S[3] = cb[3] * fxy;
    S[2] = cb[2] * fxz;
    S[6] = cb[6] * fxz;
    S[5] = cb[5] * fyz;
    S[7] = cb[7] * fyz;
}

struct FineCtx {
    uint32_t X[3], Y[3], Z[3];  // index parts of the coordinates -1, 0, +1 per axis
    float wc[8];
    double wd[8];  // FP64 weights Emin + x (refinement residual only)
    __device__ __forceinline__ uint32_t nb(int d) const { return X[d % 3] + Y[d / 3 % 3] + Z[d / 9]; }
    // cell at offset (ex-1, ey-1, ez-1) from the vertex
    __device__ __forceinline__ uint32_t cell(int e) const { return X[e & 1] + Y[(e >> 1) & 1] + Z[e >> 2]; }
};

__device__ __forceinline__ void fine_parts(FineCtx& c, int x, int y, int z, const Lay& L) {
    c.X[0] = L.part(wrap_dec(x, L.n), 0); c.X[1] = L.part(x, 0); c.X[2] = L.part(wrap_inc(x, L.n), 0);
    c.Y[0] = L.part(wrap_dec(y, L.n), 1); c.Y[1] = L.part(y, 1); c.Y[2] = L.part(wrap_inc(y, L.n), 1);
    c.Z[0] = L.part(wrap_dec(z, L.n), 2); c.Z[1] = L.part(z, 2); c.Z[2] = L.part(wrap_inc(z, L.n), 2);
}

__device__ __forceinline__ void fine_ctx(FineCtx& c, int x, int y, int z, const Lay& L, const float* __restrict__ w) {
    fine_parts(c, x, y, z, L);
    const Rsrc rw = make_rsrc(w, (size_t)L.n * L.n * L.n * sizeof(float));
#pragma unroll
    for (int e = 0; e < 8; e++) c.wc[e] = bload<float>(rw, c.cell(e) * 4u, 0);
}

// FP64 cell weights w = Emin + x from the raw cell values x (FP32 input data, exact in FP64).
__device__ __forceinline__ void fine_ctx64(FineCtx& c, int x, int y, int z, const Lay& L, const float* __restrict__ xc,
                                           double emin) {
    fine_parts(c, x, y, z, L);
    const Rsrc rw = make_rsrc(xc, (size_t)L.n * L.n * L.n * sizeof(float));
#pragma unroll
    for (int e = 0; e < 8; e++) {
        c.wd[e] = emin + (double)bload<float>(rw, c.cell(e) * 4u, 0);
        c.wc[e] = (float)c.wd[e];
    }
}

// Neighbour masks: bit d (d = 0..26, offset (d%3-1, d/3%3-1, d/9-1)) selects the neighbours a row
// gathers.  kRowAll is the whole row, kRowOffDiag the row without the vertex itself (d = 13).
constexpr uint32_t kRowAll = (1u << 27) - 1u;
constexpr int kSumThreads = 1024;       // workgroup of k_sum_partials
constexpr uint32_t kRowOffDiag = kRowAll & ~(1u << 13);

// Colour c of a sweep that starts from u = 0: the neighbours of colours above c still hold zero, so
// only those of colours below c are gathered.  A neighbour at offset d has colour c ^ flip(d), where
// flip sets bit k when the offset is odd along axis k.
__host__ __device__ constexpr uint32_t zero_start_mask(int c) {
    uint32_t m = 0;
    for (int d = 0; d < 27; d++) {
        const int f = (d % 3 != 1 ? 1 : 0) | (d / 3 % 3 != 1 ? 2 : 0) | (d / 9 != 1 ? 4 : 0);
        if ((c ^ f) < c) m |= 1u << d;
    }
    return m;
}

// first selected neighbour after d (27 when none)
constexpr int next_nb(uint32_t mask, int d) {
    for (int k = d + 1; k < 27; k++)
        if ((mask >> k) & 1u) return k;
    return 27;
}

// zero-start colour of a GS pass (-1: ordinary pass) -> gathered neighbours
constexpr uint32_t gs_mask(int zc) { return zc < 0 ? kRowOffDiag : zero_start_mask(zc); }

// neighbours of a colour-c vertex whose colour comes after c in a forward sweep
__host__ __device__ constexpr uint32_t later_mask(int c) {
    uint32_t m = 0;
    for (int d = 0; d < 27; d++) {
        const int f = (d % 3 != 1 ? 1 : 0) | (d / 3 % 3 != 1 ? 2 : 0) | (d / 9 != 1 ? 4 : 0);
        if ((c ^ f) > c) m |= 1u << d;
    }
    return m;
}

// the stored words of one neighbour: W = R / (load cases per word) words per component; r0 counts
// load cases (a multiple of the cases per word)
// (qo = 4 * vertex index; plane = 4 N bytes)
template <int W, typename A>
__device__ __forceinline__ void load_nb(A (&dst)[W][3], Rsrc ru, uint32_t qo, uint32_t plane, int r0) {
    constexpr int cpw = CasesPerWord<A>::value;
    if constexpr (cpw == 2 && W == 3) {  // all six load cases (r0 = 0): the vertex's nine words
        uint32_t wv[9];
        hload9(wv, ru, qo >> 2, plane);
#pragma unroll
        for (int p = 0; p < 3; p++)
#pragma unroll
            for (int i = 0; i < 3; i++) dst[p][i] = __builtin_bit_cast(A, wv[p * 3 + i]);
    } else if constexpr (cpw == 2) {
#pragma unroll
        for (int p = 0; p < W; p++)
#pragma unroll
            for (int i = 0; i < 3; i++) {
                const int q = (r0 / 2 + p) * 3 + i;
                dst[p][i] = q < 8 ? bload<A>(ru, 4u * qo + 4u * (uint32_t)(q & 3), (uint32_t)(q >> 2) * 4u * plane)
                                  : bload<A>(ru, qo, 8u * plane);
            }
    } else {
#pragma unroll
        for (int p = 0; p < W; p++)
#pragma unroll
            for (int i = 0; i < 3; i++) dst[p][i] = bload<A>(ru, qo, (uint32_t)((r0 / cpw + p) * 3 + i) * plane);
    }
}

// The two x-neighbours (d = 12, 14) of a vertex taken from LDS instead of memory: `base` holds 3W word
// planes of 256 slots (one per thread of the workgroup), slot[0] / slot[1] the x-1 / x+1 neighbour.
template <typename A>
struct XNbLds {
    const A* base = nullptr;
    int slot[2] = {0, 0};
};

template <int W, typename A>
__device__ __forceinline__ void load_nb_lds(A (&dst)[W][3], const XNbLds<A>& xl, int k) {
#pragma unroll
    for (int p = 0; p < W; p++)
#pragma unroll
        for (int i = 0; i < 3; i++) dst[p][i] = xl.base[(p * 3 + i) * 256 + xl.slot[k]];
}

// the stored words of neighbour d: from memory, or from LDS for the x-neighbours when XL
template <int W, typename A, bool XL, int D>
__device__ __forceinline__ void load_nb_at(A (&dst)[W][3], const FineCtx& c, Rsrc ru, uint32_t plane, int r0,
                                           const XNbLds<A>& xl) {
    if constexpr (XL && (D == 12 || D == 14))
        load_nb_lds<W, A>(dst, xl, D == 12 ? 0 : 1);
    else
        load_nb<W, A>(dst, ru, c.nb(D) * (uint32_t)sizeof(A), plane, r0);
}

// acc[r] += S u_r for the load cases of one stored word triple
template <int W, typename T, typename A>
__device__ __forceinline__ void block_fma(const T (&S)[9], const A (&cur)[W][3], T (&acc)[W * CasesPerWord<A>::value][3]) {
#pragma unroll
    for (int p = 0; p < W; p++) {
        if constexpr (CasesPerWord<A>::value == 2) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const float u0 = (float)cur[p][0][h], u1 = (float)cur[p][1][h], u2 = (float)cur[p][2][h];
                T(&a)[3] = acc[2 * p + h];
                a[0] = fmaf(S[0], u0, fmaf(S[1], u1, fmaf(S[2], u2, a[0])));
                a[1] = fmaf(S[3], u0, fmaf(S[4], u1, fmaf(S[5], u2, a[1])));
                a[2] = fmaf(S[6], u0, fmaf(S[7], u1, fmaf(S[8], u2, a[2])));
            }
        } else {
            const T u0 = (T)cur[p][0], u1 = (T)cur[p][1], u2 = (T)cur[p][2];
            acc[p][0] = fma(S[0], u0, fma(S[1], u1, fma(S[2], u2, acc[p][0])));
            acc[p][1] = fma(S[3], u0, fma(S[4], u1, fma(S[5], u2, acc[p][1])));
            acc[p][2] = fma(S[6], u0, fma(S[7], u1, fma(S[8], u2, acc[p][2])));
        }
    }
}

// Keep a neighbour's products at its step: the products read values loaded one step earlier, and without
// this the instruction selector may sink all of them below the last scheduling barrier, keeping every
// neighbour's operands live (hundreds of spilled registers).  The empty volatile statement emits nothing.
template <int R, typename T>
__device__ __forceinline__ void pin_acc(T (&acc)[R][3]) {
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int i = 0; i < 3; i++) __asm__ volatile("" : "+v"(acc[r][i]));
}

// One neighbour of the row, the loads PF neighbours ahead (buf: a ring of the neighbours in flight, this
// one, the K-th, in slot K % PF) and the next block's constants (k: this one's) in flight: build the 3x3
// block from the cell weights, accumulate, recurse.
template <int R, uint32_t MASK, int PF, int D, int DA, int K, typename A, bool XL>
__device__ __forceinline__ void gather_step(const FineCtx& c, KeBlocks kb, Rsrc ru, uint32_t plane, int r0,
                                            const BlockConsts& k, A (&buf)[PF][R / CasesPerWord<A>::value][3],
                                            float (&acc)[R][3], const XNbLds<A>& xl) {
    constexpr int W = R / CasesPerWord<A>::value;
    constexpr int DN = next_nb(MASK, D), DAN = DA < 27 ? next_nb(MASK, DA) : 27;
    // keep each neighbour's block build next to its use (bounds register pressure)
    __builtin_amdgcn_sched_barrier(0);
    pin_acc<R, float>(acc);
    A nxt[W][3];
    BlockConsts kn = {};
    if constexpr (DN < 27) kn = block_consts<DN>(kb);
    if constexpr (DA < 27) load_nb_at<W, A, XL, DA>(nxt, c, ru, plane, r0, xl);
    float S[9];
    fine_block<D>(c.wc, k, S);
    block_fma<W, float, A>(S, buf[K % PF], acc);
    if constexpr (DA < 27) {
#pragma unroll
        for (int p = 0; p < W; p++)
#pragma unroll
            for (int i = 0; i < 3; i++) buf[K % PF][p][i] = nxt[p][i];
    }
    if constexpr (DN < 27) gather_step<R, MASK, PF, DN, DAN, K + 1, A, XL>(c, kb, ru, plane, r0, kn, buf, acc, xl);
}

// the first PF neighbours' loads
template <int W, uint32_t MASK, int PF, int D, int K, typename A, bool XL>
__device__ __forceinline__ void gather_fill(const FineCtx& c, Rsrc ru, uint32_t plane, int r0, A (&buf)[PF][W][3],
                                            const XNbLds<A>& xl) {
    if constexpr (K < PF && D < 27) {
        load_nb_at<W, A, XL, D>(buf[K], c, ru, plane, r0, xl);
        gather_fill<W, MASK, PF, next_nb(MASK, D), K + 1, A, XL>(c, ru, plane, r0, buf, xl);
    }
}
constexpr int nth_nb(uint32_t mask, int k) {
    int d = next_nb(mask, -1);
    for (int i = 0; i < k && d < 27; i++) d = next_nb(mask, d);
    return d;
}

// acc[r][i] = sum_d S_d u_{v+d} over the neighbours d selected by MASK, load cases r0..r0+R-1.
// The pinned origin's entries of u are zero by construction (every entry point zeroes them before the
// fine operator reads u).  XL: the two x-neighbours come from LDS (xl).
template <int R, uint32_t MASK, typename A, bool XL = false, int PF = 1>
__device__ __forceinline__ void fine_gather(const FineCtx& c, size_t N, KeBlocks kb, const A* __restrict__ u,
                                            float (&acc)[R][3], int r0 = 0, const XNbLds<A>& xl = XNbLds<A>()) {
    constexpr int W = R / CasesPerWord<A>::value;
    const Rsrc ru = make_rsrc(u, (size_t)(18 / CasesPerWord<A>::value) * N * sizeof(A));
    const uint32_t plane = (uint32_t)(N * sizeof(A));
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int i = 0; i < 3; i++) acc[r][i] = 0.f;
    constexpr int D0 = next_nb(MASK, -1);
    if constexpr (D0 < 27) {
        A buf[PF][W][3];
        const BlockConsts k = block_consts<D0>(kb);
        gather_fill<W, MASK, PF, D0, 0, A, XL>(c, ru, plane, r0, buf, xl);
        gather_step<R, MASK, PF, D0, nth_nb(MASK, PF), 0, A, XL>(c, kb, ru, plane, r0, k, buf, acc, xl);
    }
}

// The same sum for FP32 u where every 64 consecutive vertices are whole grid rows (64 % (n/2) == 0): of a
// vertex's two x-neighbours, which alternate in the other x-parity's block, one sits at the vertex's own
// position (x - 1 for PXP = 1, the odd vertices, x + 1 for 0) and the other is that of the next lane of the
// row, so one load and a lane exchange (through LDS, byte address `lane`) serve both: 324 loads of single words
// instead of 486, which the texture addresser was busy with (a colour pair at 128^3 81 us for 90, at 64^3 21
// for 24; the residual 206 for 270 and 27 for 34).  Unit U: row U / 2, its middle or its sides.
constexpr bool unit_in(uint32_t mask, int u) { return mask >> (3 * (u / 2) + (u & 1 ? 0 : 1)) & 1u; }
constexpr int next_unit(uint32_t mask, int u) {
    for (int k = u + 1; k < 18; k++)
        if (unit_in(mask, k)) return k;
    return 18;
}

template <int R, int PXP, bool XL, int U>
__device__ __forceinline__ void load_unit(float (&dst)[R][3], const FineCtx& c, Rsrc ru, uint32_t plane, int r0,
                                          const XNbLds<float>& xl) {
    constexpr int D = 3 * (U / 2) + (U & 1 ? (PXP ? 0 : 2) : 1);
    load_nb_at<R, float, XL, D>(dst, c, ru, plane, r0, xl);
}

template <int R, uint32_t MASK, int PXP, bool XL, int U>
__device__ __forceinline__ void gather_unit(const FineCtx& c, KeBlocks kb, Rsrc ru, uint32_t plane, int r0, int lane,
                                            const BlockConsts& k, const float (&cur)[R][3], float (&acc)[R][3],
                                            const XNbLds<float>& xl) {
    constexpr int row = U / 2, UN = next_unit(MASK, U);
    constexpr bool sides = U & 1;
    constexpr int D = 3 * row + (sides ? (PXP ? 0 : 2) : 1), DS = 3 * row + (PXP ? 2 : 0);
    __builtin_amdgcn_sched_barrier(0);
    pin_acc<R, float>(acc);
    float nxt[R][3], far[R][3];
    if constexpr (UN < 18) load_unit<R, PXP, XL, UN>(nxt, c, ru, plane, r0, xl);
    BlockConsts kn = {}, ks = {};
    if constexpr (UN < 18) kn = block_consts<3 * (UN / 2) + (UN & 1 ? (PXP ? 0 : 2) : 1)>(kb);
    if constexpr (sides) {
        ks = block_consts<DS>(kb);
        if constexpr (XL && row == 4) {
            load_nb_lds<R, float>(far, xl, PXP ? 1 : 0);
        } else {
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int i = 0; i < 3; i++)
                    far[r][i] = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(lane, __builtin_bit_cast(int, cur[r][i])));
        }
    }
    float S[9];
    fine_block<D>(c.wc, k, S);
    block_fma<R, float, float>(S, cur, acc);
    if constexpr (sides) {
        fine_block<DS>(c.wc, ks, S);
        block_fma<R, float, float>(S, far, acc);
    }
    if constexpr (UN < 18) gather_unit<R, MASK, PXP, XL, UN>(c, kb, ru, plane, r0, lane, kn, nxt, acc, xl);
}

template <int R, uint32_t MASK, int PXP, bool XL>
__device__ __forceinline__ void fine_gather_rows(const FineCtx& c, int h, size_t N, KeBlocks kb, const float* __restrict__ u,
                                                 float (&acc)[R][3], int r0, const XNbLds<float>& xl) {
    const Rsrc ru = make_rsrc(u, (size_t)18 * N * sizeof(float));
    const uint32_t plane = (uint32_t)(N * sizeof(float));
    const int l = (int)(threadIdx.x & 63u), lane = 4 * ((l & ~(h - 1)) | ((l + (PXP ? 1 : -1)) & (h - 1)));
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int i = 0; i < 3; i++) acc[r][i] = 0.f;
    constexpr int U0 = next_unit(MASK, -1);
    float first[R][3];
    const BlockConsts k = block_consts<3 * (U0 / 2) + (U0 & 1 ? (PXP ? 0 : 2) : 1)>(kb);
    load_unit<R, PXP, XL, U0>(first, c, ru, plane, r0, xl);
    gather_unit<R, MASK, PXP, XL, U0>(c, kb, ru, plane, r0, lane, k, first, acc, xl);
}

// Stage the FP64 element matrix in LDS (all threads of the block take part), followed by the block
// constants of fine_block: C_d,ij = KE[7 - e0][b0](i, j)
// for the cell e0 with e0_m = 1 exactly where d_m = +1 and b0_m = d_m + 1 - e0_m.
template <typename T>
__device__ __forceinline__ void stage_ke(T* ke_s, const T* __restrict__ ke) {
    for (int i = threadIdx.x; i < 576; i += blockDim.x) ke_s[i] = ke[i];
    __syncthreads();
    for (int t = threadIdx.x; t < 243; t += blockDim.x) {
        const int d = t / 9, i = t / 3 % 3, j = t % 3;
        int e0 = 0, b0 = 0;
        for (int m = 0; m < 3; m++) {
            const int dm = (m == 0 ? d % 3 : (m == 1 ? d / 3 % 3 : d / 9)) - 1;
            const int em = dm > 0 ? 1 : 0;
            e0 |= em << m;
            b0 |= (dm + 1 - em) << m;
        }
        ke_s[kBlockConsts + t] = ke_s[(3 * (7 - e0) + i) * 24 + 3 * b0 + j];
    }
    __syncthreads();
}

// GS colour c covers the vertices with coordinate parity (1-c&1, 1-c>>1&1, 1-c>>2): the reference
// colours by the parity of the ghost-padded position (grid.cpp:155-198) and sweeps colours 0..7.
// In the parity-blocked order that is block 7 - c.
__device__ __forceinline__ uint32_t colour_block(int colour) { return (uint32_t)(7 - colour); }

// ---------------------------------------------------------------------------------------------
// Finest level (matrix-free)
// ---------------------------------------------------------------------------------------------

// MODE 0: out = K u; MODE 1: out = f - K u.  Pinned origin row is zero.
// (update_residual_otf_kernel_1 grid.cu:1277-1461; v3_stencilOnLeft_kernel grid.cu:3686-3857)
// MODE 0: out = K u, or with beta (per load case) out = K u + beta out_old, the CG recurrence
// K p = K z + beta K p_old that applies K to the (cheaper to gather) preconditioned vector z.
// DOT (MODE 0): also the per-workgroup FP64 partial sums of dotv . out per load case (the p . Kp of a
// CG step) in partial[r * gridDim.x + block].  The launcher uses it only when every lane of the grid
// holds a vertex (64 | (n/2)^3), so no thread leaves before the workgroup reduction.
// A: storage of u (float, or half2_t pairs of load cases).  BETA selects the recurrence form at compile
// time (a run-time test in the epilogue makes the compiler spill the gather pipeline).
// PX (with DOT, u = z): the CG vector updates of the step, fused: p = z (PX 1, first step) or
// x += alpha p_old, p = z + beta p_old (PX 2), per load case with alpha, beta from the device; the dot
// is then p . out with the new p (dotv unused).  Load cases that have converged carry alpha = beta = 0.
template <int R, int MODE, bool DOT, typename A, bool BETA = false, int PX = 0, int PF = 1, bool LANES = false>
__global__ __launch_bounds__(kFullThreads, 4) void k_fine_apply(Lay L, size_t N, const float* __restrict__ ke,
                                                                const float* __restrict__ w,
                                                                const A* __restrict__ u,
                                                                const float* __restrict__ f, float* __restrict__ out,
                                                                double* __restrict__ partial,
                                                                const float* __restrict__ dotv,
                                                                const double* __restrict__ beta,
                                                                float* __restrict__ pp = nullptr,
                                                                float* __restrict__ xx = nullptr,
                                                                const double* __restrict__ alpha = nullptr) {
    const KeBlocks kb = ke_blocks(ke);
    uint32_t v;
    if (!full_vertex(L, xcd_chunk(blockIdx.x, gridDim.x), v)) return;
    int x, y, z;
    L.pos(v, x, y, z);
    FineCtx c;
    fine_ctx(c, x, y, z, L, w);
    float acc[R][3];
    if constexpr (LANES) {  // a wave is in one parity block
        if (__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) & 1)
            fine_gather_rows<R, kRowAll, 1, false>(c, L.h, N, kb, u, acc, 0, XNbLds<A>());
        else
            fine_gather_rows<R, kRowAll, 0, false>(c, L.h, N, kb, u, acc, 0, XNbLds<A>());
    } else {
        fine_gather<R, kRowAll, A, false, PF>(c, N, kb, u, acc);
    }
    double dot[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        float b = 0.f, a = 0.f;
        if constexpr (BETA) b = (float)beta[r];
        if constexpr (PX == 2) a = (float)alpha[r];
        dot[r] = 0.0;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const size_t o = (size_t)(r * 3 + i) * N + v;
            float val = (MODE == 1) ? f[o] - acc[r][i] : acc[r][i];
            if constexpr (BETA) val = fmaf(b, out[o], val);
            val = (v == 0) ? 0.f : val;
            out[o] = val;
            float dv = 0.f;
            if constexpr (PX != 0) {
                float zc;  // z of the vertex itself
                if constexpr (CasesPerWord<A>::value == 2)
                    zc = (float)u[hw_index((r >> 1) * 3 + i, v, N)][r & 1];
                else
                    zc = (float)u[o];
                dv = zc;
                if constexpr (PX == 2) {
                    const float po = pp[o];
                    xx[o] = fmaf(a, po, xx[o]);
                    dv = fmaf(b, po, zc);
                }
                pp[o] = dv;
            } else if constexpr (DOT) {
                dv = dotv[o];
            }
            if constexpr (DOT) dot[r] = fma((double)dv, (double)val, dot[r]);
        }
    }
    if constexpr (DOT) {
        __shared__ double sh[kFullThreads / 64];
#pragma unroll
        for (int r = 0; r < R; r++) {
            const double d = block_sum<kFullThreads>(dot[r], sh);
            if (threadIdx.x == 0) partial[r * gridDim.x + blockIdx.x] = d;
        }
    }
}

// ---------------------------------------------------------------------------------------------
// CG pass with each workgroup's node box of z staged in LDS
// ---------------------------------------------------------------------------------------------
// The step of k_fine_apply<6, 0, true, half2_t, BETA, PX> on the same 128 x 2 x 2 vertex tiles, with the
// same arithmetic in the same order (so the same results bit for bit), for a parity-blocked level with
// 64 | n/2.  The row form gathers 243 single words per vertex from memory, and on gfx950 it is the texture
// addresser that those gathers keep busy, not HBM; here the workgroup loads the 130 x 4 x 4 node box of
// the packed-FP16 z (9 word planes) once, row by row with coalesced loads (about 37 per thread), and
// reads the 27 neighbours of each vertex from LDS.
// Box layout: word plane q, then z row lz and y row ly (coordinate - (2 by - 1), bz alike), then x
// parity s, then the half-x position k = (x >> 1) - (bx0 - s).  A row of one parity is contiguous in
// memory and in LDS, so the 64 lanes of a wave (consecutive x >> 1) read 64 consecutive words.
constexpr int kStK = 65;                    // half-x positions per staged row: 64 owned + 1 halo
constexpr int kStRow = 2 * kStK;            // both x parities of one (y, z) row
constexpr int kStRows = 16;                 // 4 z rows x 4 y rows
constexpr int kStPlane = 2112;              // 16 x 130 words padded to a multiple of 64 (256-byte steps)
constexpr int kStPos = kStRows * kStRow;   // staged positions per word plane
constexpr int kStIter = (kStPos + kFullThreads - 1) / kFullThreads;
static_assert(kStPlane >= kStRows * kStRow && kStPlane % 64 == 0, "staged plane stride");

// neighbour d of the vertex: its 9 words from the staged box; xb[dx + 1] holds the thread's word index of
// the x-neighbour dx in row (py, pz) of every plane
template <int D>
__device__ __forceinline__ void staged_nb(half2_t (&dst)[3][3], const uint32_t* zs, const int (&xb)[3]) {
    constexpr int dx = D % 3, dy = D / 3 % 3, dz = D / 9;
    const uint32_t* a = zs + xb[dx] + (dz * 4 + dy) * kStRow;
#pragma unroll
    for (int p = 0; p < 3; p++)
#pragma unroll
        for (int i = 0; i < 3; i++) dst[p][i] = __builtin_bit_cast(half2_t, a[(p * 3 + i) * kStPlane]);
}

template <int D>
__device__ __forceinline__ void staged_step(const FineCtx& c, KeBlocks kb, const BlockConsts& k, const uint32_t* zs,
                                            const int (&xb)[3], const half2_t (&cur)[3][3], float (&acc)[6][3]) {
    __builtin_amdgcn_sched_barrier(0);
    half2_t nxt[3][3];
    BlockConsts kn = {};
    if constexpr (D < 26) kn = block_consts<D + 1>(kb);
    if constexpr (D < 26) staged_nb<D + 1>(nxt, zs, xb);
    float S[9];
    fine_block<D>(c.wc, k, S);
    block_fma<3, float, half2_t>(S, cur, acc);
    if constexpr (D < 26) staged_step<D + 1>(c, kb, kn, zs, xb, nxt, acc);
}

// Load the workgroup's node box of the packed-FP16 z (tile of chunk t0: half-x bx0.. bx0 + 63, half-y by,
// half-z bz) into zs: position pos = ((lz * 4 + ly) * 2 + s) * 65 + k of the box, one address and its
// nine words per position.  The caller publishes it with a workgroup barrier.
__device__ __forceinline__ void stage_z_box(uint32_t* zs, const uint32_t* __restrict__ z, const Lay& L, size_t N,
                                            int bx0, int by, int bz) {
    const int h = L.h;
    const Rsrc rz = make_rsrc(z, 9 * N * sizeof(uint32_t));
    const uint32_t plane = (uint32_t)(N * sizeof(uint32_t));
    uint32_t tmp[kStIter][9];
#pragma unroll
    for (int it = 0; it < kStIter; it++) {
        const int pos = it * kFullThreads + (int)threadIdx.x;
        if (kStPos % kFullThreads == 0 || pos < kStPos) {
            const int row = pos / kStK, k = pos - row * kStK;
            const int s = row & 1, ly = (row >> 1) & 3, lz = row >> 3;
            int hx = bx0 - s + k;
            hx = hx < 0 ? hx + h : (hx >= h ? hx - h : hx);
            const int yy = L.wrap(2 * by - 1 + ly), zz = L.wrap(2 * bz - 1 + lz);
            const uint32_t blk = (uint32_t)(s | (yy & 1) << 1 | (zz & 1) << 2);
            const uint32_t id = blk * L.h3 + (uint32_t)hx +
                                (uint32_t)h * ((uint32_t)(yy >> 1) + (uint32_t)h * (uint32_t)(zz >> 1));
            hload9(tmp[it], rz, id, plane);
        }
    }
#pragma unroll
    for (int it = 0; it < kStIter; it++) {
        const int pos = it * kFullThreads + (int)threadIdx.x;
        if (kStPos % kFullThreads == 0 || pos < kStPos) {
#pragma unroll
            for (int q = 0; q < 9; q++) zs[q * kStPlane + pos] = tmp[it][q];
        }
    }
}

// word index of the x-neighbours dx = -1, 0, 1 of a thread's vertex in the staged box (row (py, pz) of
// every plane): parity s' = (px + dx) & 1, half-x position k = lane + (px + dx - s') / 2 + s'
__device__ __forceinline__ void staged_xb(int (&xb)[3], int lane, int px, int py, int pz) {
#pragma unroll
    for (int dx = -1; dx <= 1; dx++) {
        const int sp = (px + dx) & 1;
        xb[dx + 1] = lane + (pz * 4 + py) * kStRow + sp * kStK + (px + dx - sp) / 2 + sp;
    }
}

template <bool BETA, int PX>
__global__ __launch_bounds__(kFullThreads, 4) void k_fine_cg_staged(Lay L, size_t N, const float* __restrict__ ke,
                                                                    const float* __restrict__ w,
                                                                    const uint32_t* __restrict__ z,
                                                                    float* __restrict__ out,
                                                                    double* __restrict__ partial,
                                                                    const double* __restrict__ beta,
                                                                    float* __restrict__ pp, float* __restrict__ xx,
                                                                    const double* __restrict__ alpha) {
    static_assert(BETA == (PX == 2), "the first pass (PX 1) has no beta; later passes (PX 2) have both");
    __shared__ uint32_t zs[9 * kStPlane];
    const KeBlocks kb = ke_blocks(ke);
    const int h = L.h;
    const uint32_t t0 = xcd_chunk(blockIdx.x, gridDim.x) * 64u;
    const int bx0 = (int)(t0 % (uint32_t)h), by = (int)((t0 / (uint32_t)h) % (uint32_t)h);
    const int bz = (int)(t0 / ((uint32_t)h * h));
    const int b = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = (int)(threadIdx.x & 63u);
    const uint32_t v = (uint32_t)b * L.h3 + t0 + (uint32_t)lane;
    // PX 2: the vertex's p_old and x are loaded with the box and q_old right after it, so their latency
    // overlaps the staging and the neighbour loop; x += alpha p_old is stored before the loop, q_old and
    // p_old stay in registers
    // (buffer accesses: one 32-bit offset v * 4 per thread, the (load case, component) plane in an SGPR)
    const uint32_t vo = v * 4u, fplane = (uint32_t)(N * sizeof(float));
    const size_t fbytes = 18 * N * sizeof(float);
    const Rsrc rq = make_rsrc(out, fbytes), rp = make_rsrc(pp, fbytes), rx = make_rsrc(xx, fbytes);
    float qo[6][3], po[6][3];
    {
        float xo[6][3];
        if constexpr (PX == 2) {
#pragma unroll
            for (int r = 0; r < 6; r++)
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    po[r][i] = bload<float>(rp, vo, (uint32_t)(r * 3 + i) * fplane);
                    xo[r][i] = bload<float>(rx, vo, (uint32_t)(r * 3 + i) * fplane);
                }
        }
        stage_z_box(zs, z, L, N, bx0, by, bz);
        if constexpr (PX == 2) {
#pragma unroll
            for (int r = 0; r < 6; r++) {
                const float a = (float)alpha[r];
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    const uint32_t so = (uint32_t)(r * 3 + i) * fplane;
                    bstore(fmaf(a, po[r][i], xo[r][i]), rx, vo, so);
                    qo[r][i] = bload<float>(rq, vo, so);
                }
            }
        }
    }
    __syncthreads();  // the staged box
    const int px = b & 1, py = (b >> 1) & 1, pz = b >> 2;
    const int x = 2 * (bx0 + lane) + px, y = 2 * by + py, zc = 2 * bz + pz;
    FineCtx c;
    fine_ctx(c, x, y, zc, L, w);
    int xb[3];
    staged_xb(xb, lane, px, py, pz);
    float acc[6][3];
#pragma unroll
    for (int r = 0; r < 6; r++)
#pragma unroll
        for (int i = 0; i < 3; i++) acc[r][i] = 0.f;
    {
        half2_t first[3][3];
        staged_nb<0>(first, zs, xb);
        staged_step<0>(c, kb, block_consts<0>(kb), zs, xb, first, acc);
    }
    half2_t zv[3][3];  // z of the vertex itself (d = 13)
    staged_nb<13>(zv, zs, xb);
    double dot[6];
#pragma unroll
    for (int r = 0; r < 6; r++) {
        float bt = 0.f;
        if constexpr (BETA) bt = (float)beta[r];
        dot[r] = 0.0;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const uint32_t so = (uint32_t)(r * 3 + i) * fplane;
            float val = acc[r][i];
            if constexpr (BETA) val = fmaf(bt, qo[r][i], val);
            val = (v == 0) ? 0.f : val;
            bstore(val, rq, vo, so);
            const float zr = (float)zv[r >> 1][i][r & 1];
            float dv = zr;
            if constexpr (PX == 2) dv = fmaf(bt, po[r][i], zr);
            bstore(dv, rp, vo, so);
            dot[r] = fma((double)dv, (double)val, dot[r]);
        }
    }
    __shared__ double sh[kFullThreads / 64];
#pragma unroll
    for (int r = 0; r < 6; r++) {
        const double d = block_sum<kFullThreads>(dot[r], sh);
        if (threadIdx.x == 0) partial[r * gridDim.x + blockIdx.x] = d;
    }
}

// ---------------------------------------------------------------------------------------------
// Finest-level operator in element form on the matrix cores (packed-FP16 u, n % 32 == 0)
// ---------------------------------------------------------------------------------------------
// K u = sum over cells e of w_e KE u_e (the per-cell form of grid.cu:1277-1461).  A workgroup owns a
// tile of 32 x 4 x 4 vertices.  For one load-case pair at a time it stages the 34 x 6 x 6 node box
// of u in LDS, forms KE u_e for the 33 x 5 x 5 cells that touch the tile with
// v_mfma_f32_16x16x32_f16 and adds w_e KE u_e into the tile's vertices in LDS.  KE enters through its
// Lame tables, KE = lambda/72 Kl + mu/72 Km with small-integer Kl, Km (templateMatrix.cpp:8-61),
// which FP16 holds exactly: every product is exact, the sums are FP32, and a constant (rigid
// translation) field gives exactly zero, as it must; CG on this operator relies on that.
//
// Lanes: column c = lane % 16 of a wave is one cell; lane group g = lane / 16 carries the cell's two
// nodes (ox, g & 1, g >> 1), ox = 0, 1.  B holds their 6 words (3 components x 2 nodes) as K entries
// 8g .. 8g + 5, and the three 16-row output tiles return to the lane the same 6 rows of Kl u_e and of
// Km u_e (table layout: ke_mfma_table).  The 16 cells of a group are consecutive cells of one grid
// row, so the face shared by cells c and c + 1 is summed across lanes (DPP row shift).
//
// Sums without atomics: a vertex row (y, z) receives from the four cell rows (ey, ez) in
// {y-1, y} x {z-1, z}, one of each (ey, ez) parity class.  Each class writes its own LDS plane, and
// every vertex of a plane is written exactly once per load case: plain stores, no clearing, no
// ordering between waves.  The few contributions that meet on a plane at the x-seams of the row
// groups (x = 0, 16: first lane of a group; x = 0 also from the cells at x = -1, which form
// separate groups) go to small per-class arrays of their own.  The epilogue adds it all up.
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

constexpr int kEfTX = 16, kEfTY = 2, kEfTZ = 2;                                     // parity positions
constexpr int kEfVX = 2 * kEfTX, kEfVY = 2 * kEfTY, kEfVZ = 2 * kEfTZ;              // owned vertices
constexpr int kEfVerts = kEfVX * kEfVY * kEfVZ;
constexpr int kEfBX = kEfVX + 2, kEfBY = kEfVY + 2, kEfBZ = kEfVZ + 2;              // node box
constexpr int kEfNodes = kEfBX * kEfBY * kEfBZ;
constexpr int kEfCX = kEfVX + 1, kEfCY = kEfVY + 1, kEfCZ = kEfVZ + 1;              // cells, from -1
constexpr int kEfCells = kEfCX * kEfCY * kEfCZ;
constexpr int kEfRows = kEfCY * kEfCZ;
constexpr int kEfRowGroups = kEfVX / 16;                 // groups of cells x = 0 .. VX-1 per row
constexpr int kEfFull = kEfRows * kEfRowGroups;
constexpr int kEfGroups = kEfFull + (kEfRows + 15) / 16;  // + groups of the x = -1 cells
constexpr int kEfYZ = kEfVY * kEfVZ;                      // vertex rows of the tile
// one LDS row per (cell-row class, case of the pair, component): the tile's vertices, the x-seam and
// x = 0 contributions, and a slot per lane that absorbs the stores of lanes with nothing for the tile
// (stores stay unconditional: no exec-mask branches in the cell loop)
constexpr int kEfSeam = kEfVerts, kEfHalo = kEfSeam + 2 * kEfYZ, kEfDummy = kEfHalo + kEfYZ;
constexpr int kEfSlots = kEfDummy + 64;
constexpr int kEfThreads = 512;
constexpr int kEfStage = (3 * kEfNodes + kEfThreads - 1) / kEfThreads;  // staged words per thread and pair
static_assert(kEfVerts == kEfThreads, "epilogue maps one vertex per thread and plane");
static_assert(kEfRowGroups == 2, "x-seams at x = 0 and x = 16");

// row shift of a 16-lane row: lane c reads lane c + 1, lane 15 reads 0
__device__ __forceinline__ float dpp_next(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x101, 0xf, 0xf, true));
}

// One group of 16 cells and the two load cases of a packed word pair: the B operands (the lane's 6 node
// words, split into the two load cases) from the node box ...
__device__ __forceinline__ void ef_load_b(const uint32_t* nodes, int nb0, half8_t (&b)[2]) {
    half2_t wv[6];
#pragma unroll
    for (int k = 0; k < 6; k++) wv[k] = __builtin_bit_cast(half2_t, nodes[(k % 3) * kEfNodes + nb0 + k / 3]);
#pragma unroll
    for (int k = 0; k < 6; k++) {
        b[0][k] = wv[k].x;
        b[1][k] = wv[k].y;
    }
    b[0][6] = b[0][7] = b[1][6] = b[1][7] = (_Float16)0.f;
}

// ... and NT + 1 output tiles per case (NT = 1: one exact table T; NT = 2: Kl and Km), giving the lane's
// 6 rows of w_e KE u_e per case in val[case][k] (k = 3 ox + component); w0, w1 = w_e c0, w_e c1.
template <int NT>
__device__ __forceinline__ void ef_mma(const half8_t (&b)[2], half8_t a0, half8_t a1, half8_t a2, float w0, float w1,
                                       float (&val)[2][6]) {
    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int hh = 0; hh < 2; hh++) {
        const float4_t d0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, b[hh], zero, 0, 0, 0);
        const float4_t d1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, b[hh], zero, 0, 0, 0);
        if constexpr (NT == 1) {
            // rows k = 0..3 in tile 0, k = 4, 5 in tile 1
            val[hh][0] = w0 * d0[0];
            val[hh][1] = w0 * d0[1];
            val[hh][2] = w0 * d0[2];
            val[hh][3] = w0 * d0[3];
            val[hh][4] = w0 * d1[0];
            val[hh][5] = w0 * d1[1];
        } else {
            // Kl rows in tiles 0/1, Km rows in tiles 1/2
            const float4_t d2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(a2, b[hh], zero, 0, 0, 0);
            val[hh][0] = fmaf(w0, d0[0], w1 * d1[2]);
            val[hh][1] = fmaf(w0, d0[1], w1 * d1[3]);
            val[hh][2] = fmaf(w0, d0[2], w1 * d2[0]);
            val[hh][3] = fmaf(w0, d0[3], w1 * d2[1]);
            val[hh][4] = fmaf(w0, d1[0], w1 * d2[2]);
            val[hh][5] = fmaf(w0, d1[1], w1 * d2[3]);
        }
    }
}

// A group of cells x = 16 half .. 16 half + 15 of cell row gi / 2 and where its lanes' results go
struct EfRowGroup {
    int nb0;   // node box index of the lane's node (0, gy, gz)
    int wi;    // cell weight index
    int v1;    // tile vertex of the lane's node (1, gy, gz): x = 16 half + col + 1
    int yz;    // vertex row of the lane's nodes
    int cls;   // parity class of the cell row
    int half;
    bool own;  // the lane's vertex row lies in the tile
};

__device__ __forceinline__ EfRowGroup ef_row_group(int gi, int col, int gy, int gz, int lane_nb, int lane_v) {
    EfRowGroup G;
    const int row = gi >> 1;
    G.half = gi & 1;
    const int ey = row % kEfCY - 1, ez = row / kEfCY - 1;
    G.cls = ((ey + 1) & 1) | (((ez + 1) & 1) << 1);
    G.wi = ((ez + 1) * kEfCY + (ey + 1)) * kEfCX + 16 * G.half + 1 + col;
    G.nb0 = ((ez + 1) * kEfBY + (ey + 1)) * kEfBX + 16 * G.half + 1 + lane_nb;
    const int vy = ey + gy, vz = ez + gz;
    G.own = vy >= 0 && vy < kEfVY && vz >= 0 && vz < kEfVZ;
    G.v1 = (ez * kEfVY + ey) * kEfVX + 16 * G.half + 1 + lane_v;
    G.yz = vz * kEfVY + vy;
    return G;
}

// MODE 0: out = K u (BETA: + beta out_old); MODE 1: out = f - K u.  DOT (MODE 0): per-workgroup FP64
// partial sums of dotv . out per load case in partial[r * gridDim.x + block].  Pinned origin row zero.
// PX: the CG vector updates fused as in k_fine_apply (z of the vertex read from the staged node box).
// KE = c0 T (NT = 1) or c0 Kl + c1 Km (NT = 2).  Needs 72 n^3 < 2^32 (32-bit buffer offsets).
template <int MODE, bool DOT, bool BETA, int NT, int PX = 0>
__global__ __launch_bounds__(kEfThreads, 2) void k_fine_apply_ef(Lay L, size_t N, const half8_t* __restrict__ amat,
                                                              float c0, float c1, const float* __restrict__ w,
                                                              const uint32_t* __restrict__ u,
                                                              const float* __restrict__ f, float* __restrict__ out,
                                                              double* __restrict__ partial,
                                                              const float* __restrict__ dotv,
                                                              const double* __restrict__ beta,
                                                              float* __restrict__ pp, float* __restrict__ xx,
                                                              const double* __restrict__ alpha) {
    __shared__ uint32_t nodes[3 * kEfNodes];       // packed words of the node box, one load-case pair
    __shared__ float acc[4][6][kEfSlots];          // per cell-row class, (case of the pair, component)
    __shared__ float wcell[kEfCells];              // w_e of the cells from -1
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, col = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: group loops stay scalar
    const int gy = g & 1, gz = g >> 1;
    const uint32_t wg = xcd_chunk(blockIdx.x, gridDim.x);
    const uint32_t ntx = (uint32_t)(L.h / kEfTX), nty = (uint32_t)(L.h / kEfTY);
    const int x0 = kEfVX * (int)(wg % ntx), y0 = kEfVY * (int)((wg / ntx) % nty), z0 = kEfVZ * (int)(wg / (ntx * nty));
    const half8_t a0 = amat[lane], a1 = amat[64 + lane], a2 = NT == 2 ? amat[128 + lane] : a1;
    const Rsrc ru = make_rsrc(u, 9 * N * sizeof(uint32_t));
    const Rsrc ro = make_rsrc(out, 18 * N * sizeof(float));
    const Rsrc rf = make_rsrc(f, f ? 18 * N * sizeof(float) : 0);
    const Rsrc rd = make_rsrc(PX ? pp : dotv, (PX ? pp != nullptr : dotv != nullptr) ? 18 * N * sizeof(float) : 0);
    const Rsrc rx = make_rsrc(xx, xx ? 18 * N * sizeof(float) : 0);
    for (int c = tid; c < kEfCells; c += kEfThreads) {
        const int ex = c % kEfCX - 1, ey = (c / kEfCX) % kEfCY - 1, ez = c / (kEfCX * kEfCY) - 1;
        wcell[c] = w[L.idx(L.wrap(x0 + ex), L.wrap(y0 + ey), L.wrap(z0 + ez))];
    }
    // node-box words of this thread: component i and vertex index of each (~0u: none).  The next pair's
    // words (q = 3 p + i, hw_index) are fetched into registers before the current pair is computed.
    uint32_t nidx[kEfStage], pre[kEfStage];
    int ncomp[kEfStage];
#pragma unroll
    for (int k = 0; k < kEfStage; k++) {
        const int s = tid + k * kEfThreads, i = s / kEfNodes, b = s - i * kEfNodes;
        const int bx = b % kEfBX, by = (b / kEfBX) % kEfBY, bz = b / (kEfBX * kEfBY);
        ncomp[k] = i;
        nidx[k] = s < 3 * kEfNodes ? L.idx(L.wrap(x0 - 1 + bx), L.wrap(y0 - 1 + by), L.wrap(z0 - 1 + bz)) : ~0u;
    }
    auto fetch = [&](int p) {
#pragma unroll
        for (int k = 0; k < kEfStage; k++)
            if (nidx[k] != ~0u)
                pre[k] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(
                    ru, (int)(4u * (uint32_t)hw_index(3 * p + ncomp[k], nidx[k], N)), 0, 0);
    };
    auto put = [&]() {
#pragma unroll
        for (int k = 0; k < kEfStage; k++)
            if (nidx[k] != ~0u) nodes[tid + k * kEfThreads] = pre[k];
    };
    fetch(0);
    put();
    __syncthreads();
    // epilogue vertex of this thread
    const int vx = tid % kEfVX, vyz = tid / kEfVX;
    const uint32_t vg = L.idx(x0 + vx, y0 + vyz % kEfVY, z0 + vyz / kEfVY), vb = 4u * vg;
    const int nb_self = ((vyz / kEfVY + 1) * kEfBY + (vyz % kEfVY + 1)) * kEfBX + vx + 1;  // the vertex in the node box
    const uint32_t plane_bytes = (uint32_t)(N * sizeof(float));
    // lane offsets of the full-row groups: node (0, gy, gz) of cell (col, 0, 0) in the node box; vertex
    // (col + 1, gy, gz) in the tile
    const int lane_nb = (gz * kEfBY + gy) * kEfBX + col, lane_v = (gz * kEfVY + gy) * kEfVX + col;
    double dot[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int p = 0; p < 3; p++) {
        if (p < 2) fetch(p + 1);
        // epilogue inputs of this pair, in flight during the cell products
        float fin[6], oin[6], din[6], xin[6];
#pragma unroll
        for (int pl = 0; pl < 6; pl++) {
            const uint32_t so = (uint32_t)(6 * p + pl) * plane_bytes;
            if constexpr (MODE == 1) fin[pl] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rf, (int)vb, (int)so, 0));
            if constexpr (BETA) oin[pl] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ro, (int)vb, (int)so, 0));
            if constexpr ((DOT && PX == 0) || PX == 2)  // dotv, or p_old
                din[pl] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rd, (int)vb, (int)so, 0));
            if constexpr (PX == 2) xin[pl] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, (int)vb, (int)so, 0));
        }
        // cells x = 0 .. VX-1 of every cell row, 16 per group
        for (int gi = wave; gi < kEfFull; gi += kEfThreads / 64) {
            const EfRowGroup g = ef_row_group(gi, col, gy, gz, lane_nb, lane_v);
            half8_t b[2];
            ef_load_b(nodes, g.nb0, b);
            const float wc = wcell[g.wi];
            float val[2][6];
            ef_mma<NT>(b, a0, a1, a2, wc * c0, wc * c1, val);
            // vertex x = 16 half + col + 1 (all lanes but the last of the second half), and the seam x = 16 half
            // of the first lane
            float* row = &acc[g.cls][0][0];
            const int s1 = g.own && (g.half == 0 || col < 15) ? g.v1 : kEfDummy + lane;
            const int sm = g.own && col == 0 ? kEfSeam + g.half * kEfYZ + g.yz : kEfDummy + lane;
#pragma unroll
            for (int hh = 0; hh < 2; hh++)
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    // node ox = 1 of cell c is node ox = 0 of cell c + 1
                    row[(hh * 3 + i) * kEfSlots + s1] = val[hh][3 + i] + dpp_next(val[hh][i]);
                    row[(hh * 3 + i) * kEfSlots + sm] = val[hh][i];
                }
        }
        // cells x = -1 of the cell rows, 16 rows per group
        for (int gi = kEfFull + wave; gi < kEfGroups; gi += kEfThreads / 64) {
            const int k = 16 * (gi - kEfFull) + col;
            const bool valid = k < kEfRows;
            const int kk = valid ? k : 0, ey = kk % kEfCY - 1, ez = kk / kEfCY - 1;
            const int cls = ((ey + 1) & 1) | (((ez + 1) & 1) << 1);
            const float wc = wcell[((ez + 1) * kEfCY + (ey + 1)) * kEfCX];
            half8_t b[2];
            ef_load_b(nodes, ((ez + 1 + gz) * kEfBY + (ey + 1 + gy)) * kEfBX, b);
            float val[2][6];
            ef_mma<NT>(b, a0, a1, a2, wc * c0, wc * c1, val);
            const int vy = ey + gy, vz = ez + gz;
            const int hs = valid && vy >= 0 && vy < kEfVY && vz >= 0 && vz < kEfVZ ? kEfHalo + vz * kEfVY + vy
                                                                                   : kEfDummy + lane;
            float* row = &acc[cls][0][0];
#pragma unroll
            for (int hh = 0; hh < 2; hh++)
#pragma unroll
                for (int i = 0; i < 3; i++) row[(hh * 3 + i) * kEfSlots + hs] = val[hh][3 + i];  // node x = 0
        }
        // z of this thread's vertex for the fused CG update, read before the barrier: after it, the node
        // box is refilled with the next pair while other threads may still be in the epilogue
        uint32_t zself[3];
        if constexpr (PX != 0) {
#pragma unroll
            for (int i = 0; i < 3; i++) zself[i] = nodes[i * kEfNodes + nb_self];
        }
        __syncthreads();
#pragma unroll
        for (int pl = 0; pl < 6; pl++) {
            const int r = 2 * p + pl / 3;
            float val = 0.f;
            if (vx != 0) val = (acc[0][pl][tid] + acc[1][pl][tid]) + (acc[2][pl][tid] + acc[3][pl][tid]);
            if (vx == 0 || vx == 16) {
                const int sl = kEfSeam + (vx >> 4) * kEfYZ + vyz;
                val += (acc[0][pl][sl] + acc[1][pl][sl]) + (acc[2][pl][sl] + acc[3][pl][sl]);
            }
            if (vx == 0) {
                const int sl = kEfHalo + vyz;
                val += (acc[0][pl][sl] + acc[1][pl][sl]) + (acc[2][pl][sl] + acc[3][pl][sl]);
            }
            const uint32_t so = (uint32_t)(6 * p + pl) * plane_bytes;
            if constexpr (MODE == 1) val = fin[pl] - val;
            if constexpr (BETA) val = fmaf((float)beta[r], oin[pl], val);
            if (vg == 0) val = 0.f;
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, val), ro, (int)vb, (int)so, 0);
            float dv = 0.f;
            if constexpr (PX != 0) {
                const half2_t zw = __builtin_bit_cast(half2_t, zself[pl % 3]);
                const float zc = (float)zw[pl / 3];
                dv = zc;
                if constexpr (PX == 2) {
                    __builtin_amdgcn_raw_buffer_store_b32(
                        __builtin_bit_cast(uint32_t, fmaf((float)alpha[r], din[pl], xin[pl])), rx, (int)vb, (int)so, 0);
                    dv = fmaf((float)beta[r], din[pl], zc);
                }
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, dv), rd, (int)vb, (int)so, 0);
            } else if constexpr (DOT) {
                dv = din[pl];
            }
            if constexpr (DOT) dot[r] = fma((double)dv, (double)val, dot[r]);
        }
        if (p < 2) put();
        __syncthreads();
    }
    if constexpr (DOT) {
        __shared__ double sh[kEfThreads / 64];
#pragma unroll
        for (int r = 0; r < 6; r++) {
            const double t = block_sum<kEfThreads>(dot[r], sh);
            if (threadIdx.x == 0) partial[r * gridDim.x + blockIdx.x] = t;
        }
    }
}

// neighbours whose loads are in flight ahead of the smoother's block products
template <typename A>
constexpr int kGsAhead = CasesPerWord<A>::value == 2 ? 3 : 1;

// GS / SOR update of the colour vertex v (load cases r0 .. r0 + R - 1), in place.  A: storage of u
// (float, or half2_t pairs of load cases); f is FP32.  ZC >= 0: colour ZC of a forward sweep that
// starts from u = 0 (colours above ZC are never read, so u needs no clearing beforehand; the old value
// of the vertex itself is zero).  XL: the x-neighbours come from LDS; TO_LDS: the new words are also
// stored to slot threadIdx.x of out_lds.  DOT: dot[r] += f . u_new over the vertex (stored values;
// FP32 over the vertex's 3 components, FP64 across vertices).  ROWN (ZC >= 0): also
// rown = f - sum over the neighbours of colours up to ZC and the vertex itself of K_vj u_j, with the
// stored values; once the sweep is complete, subtracting the later colours' terms gives f - K u.
// The pinned origin keeps u = 0 (and rown = 0).
// PXP: the vertex's x-parity where its row is whole in the wave and u is FP32 (fine_gather_rows), else -1.
template <int R, bool REVERSE, int ZC, typename A, bool XL, bool TO_LDS, bool DOT = false, bool ROWN = false, int PXP = -1>
__device__ __forceinline__ void gs_vertex(const Lay& L, size_t N, uint32_t v, float omega, KeBlocks kb,
                                          const float* __restrict__ w, A* __restrict__ u,
                                          const float* __restrict__ f, int r0, const XNbLds<A>& xl, A* out_lds,
                                          float* dot = nullptr, float* __restrict__ rown = nullptr) {
    static_assert(!ROWN || ZC >= 0, "the own-colour residual needs a zero-start forward pass");
    constexpr int cpw = CasesPerWord<A>::value;
    int x, y, z;
    L.pos(v, x, y, z);
    FineCtx c;
    fine_ctx(c, x, y, z, L, w);
    float acc[R][3];
    if constexpr (PXP >= 0)
        fine_gather_rows<R, gs_mask(ZC), PXP, XL>(c, L.h, N, kb, u, acc, r0, xl);
    else
        fine_gather<R, gs_mask(ZC), A, XL, kGsAhead<A>>(c, N, kb, u, acc, r0, xl);
    float Ks[9];
    fine_block<13>(c.wc, block_consts<13>(kb), Ks);
    const float inv[3] = {1.f / Ks[0], 1.f / Ks[4], 1.f / Ks[8]};
    const bool pin = v == 0;
#pragma unroll
    for (int p = 0; p < R / cpw; p++) {
        float uu[cpw][3], ff[cpw][3];
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const size_t o = fw_index<A>((r0 / cpw + p) * 3 + i, v, N);
            if constexpr (cpw == 2) {
                const half2_t wv = ZC >= 0 ? half2_t{0, 0} : u[o];
                uu[0][i] = (float)wv.x;
                uu[1][i] = (float)wv.y;
            } else {
                uu[0][i] = ZC >= 0 ? 0.f : u[o];
            }
#pragma unroll
            for (int h = 0; h < cpw; h++) ff[h][i] = f[(size_t)((r0 + p * cpw + h) * 3 + i) * N + v];
        }
#pragma unroll
        for (int h = 0; h < cpw; h++) block_update<REVERSE>(uu[h], ff[h], acc[p * cpw + h], Ks, inv, omega);
        float us[cpw][3];  // the stored values
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const size_t o = fw_index<A>((r0 / cpw + p) * 3 + i, v, N);
            A word;
            if constexpr (cpw == 2)
                word = half2_t{(_Float16)uu[0][i], (_Float16)uu[1][i]};
            else
                word = uu[0][i];
            if (pin) word = A(0);
            if constexpr (cpw == 2) {
                us[0][i] = (float)word.x;
                us[1][i] = (float)word.y;
            } else {
                us[0][i] = word;
            }
            u[o] = word;
            if constexpr (TO_LDS) out_lds[(p * 3 + i) * 256 + threadIdx.x] = word;
            if constexpr (DOT) {
                if constexpr (cpw == 2) {
                    dot[p * 2] = fmaf(ff[0][i], (float)word.x, dot[p * 2]);
                    dot[p * 2 + 1] = fmaf(ff[1][i], (float)word.y, dot[p * 2 + 1]);
                } else {
                    dot[p] = fmaf(ff[0][i], word, dot[p]);
                }
            }
        }
        if constexpr (ROWN) {
#pragma unroll
            for (int hh = 0; hh < cpw; hh++)
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    const float kv = fmaf(Ks[3 * i], us[hh][0], fmaf(Ks[3 * i + 1], us[hh][1], Ks[3 * i + 2] * us[hh][2]));
                    const float ro = (ff[hh][i] - acc[p * cpw + hh][i]) - kv;
                    rown[(size_t)((r0 + p * cpw + hh) * 3 + i) * N + v] = pin ? 0.f : ro;
                }
        }
    }
}

// Two consecutive colours of a fine block GS / SOR sweep in one launch, in place
// (gs_relaxation_otf_kernel, grid.cu:323-551): cfirst, then cfirst + 1 (forward) or cfirst - 1
// (REVERSE), cfirst even resp. odd.  DOT: per-workgroup FP64 sums of f . u_new over the pair's vertices
// per load case to partial[r * pstride + blockIdx.x] (over the four pair launches of a sweep that is
// the last to write u, this is the r . z of the CG step).  The two colours differ only in x-parity, and a vertex of the
// second depends on the first only through its x-neighbours, which lie in the same grid row.  Each
// workgroup owns as many whole rows of n/2 as 256 threads hold (pair_rows; n <= 512, the rest of the
// threads and of the last workgroup idle): it updates the first colour of its rows, keeps the new values
// in LDS, and updates the second colour reading those x-neighbours from LDS.  Other workgroups never read the rows' first-colour values
// before they are final, so the result equals the two colour passes in sequence.
// ROWN (zero-start passes): both colours also store their own-colour residuals to rown (gs_vertex).
// LANES: gs_vertex's PXP (colour c lies in block 7 - c).
template <int R, bool REVERSE, int ZC, typename A, bool DOT = false, bool ROWN = false, bool LANES = false>
__global__ __launch_bounds__(256, 4) void k_fine_gs2(Lay L, size_t N, int cfirst, float omega,
                                                     const float* __restrict__ ke, const float* __restrict__ w,
                                                     A* __restrict__ u, const float* __restrict__ f,
                                                     double* __restrict__ partial, int pstride,
                                                     float* __restrict__ rown) {
    constexpr int W = R / CasesPerWord<A>::value;
    __shared__ A xs[3 * W * 256];
    const KeBlocks kb = ke_blocks(ke);
    const int h = L.h, span = pair_rows(h) * h;
    const uint32_t t = xcd_chunk(blockIdx.x, gridDim.x) * (uint32_t)span + threadIdx.x;
    const bool live = (int)threadIdx.x < span && t < L.h3;
    const int c2 = REVERSE ? cfirst - 1 : cfirst + 1;
    float dot[R];
#pragma unroll
    for (int r = 0; r < R; r++) dot[r] = 0.f;
    if (live)
        gs_vertex<R, REVERSE, ZC, A, false, true, DOT, ROWN, LANES ? (REVERSE ? 0 : 1) : -1>(L, N, colour_block(cfirst) * L.h3 + t, omega, kb, w, u,
                                                            f, 0, XNbLds<A>(), xs, dot, rown);
    __syncthreads();
    if (live) {
        XNbLds<A> xl;
        xl.base = xs;
        const int lx = (int)(t % (uint32_t)h), row0 = (int)threadIdx.x - lx;
        const bool odd = (colour_block(c2) & 1u) != 0;  // x-parity of the second colour
        xl.slot[0] = row0 + (odd ? lx : (lx == 0 ? h - 1 : lx - 1));
        xl.slot[1] = row0 + (odd ? (lx + 1 == h ? 0 : lx + 1) : lx);
        gs_vertex<R, REVERSE, (ZC < 0 ? -1 : ZC + 1), A, true, false, DOT, ROWN, LANES ? (REVERSE ? 1 : 0) : -1>(
            L, N, colour_block(c2) * L.h3 + t, omega, kb, w, u, f, 0, xl, nullptr, dot, rown);
    }
    if constexpr (DOT) {
        __shared__ double sh[4];
#pragma unroll
        for (int r = 0; r < R; r++) {
            const double sdot = block_sum<256>((double)dot[r], sh);
            if (threadIdx.x == 0) partial[(size_t)r * pstride + blockIdx.x] = sdot;
        }
    }
}

// The residual f - K u after a zero-start forward sweep whose colour passes stored their own-colour
// residuals in r (gs_vertex ROWN): r -= sum over the neighbours of colours after C of K_vj u_j, for
// a vertex v of colour C (C < 7; colour 7 has no later neighbours, so its r is final).  About half
// the neighbour terms of a full residual pass, averaged over the colours.
// zero is 0 at run time: chaining the three components through it keeps the compiler converting the
// gathered FP16 words inside the FMAs (v_fma_mix); with independent components it converts every word
// up front and spills.
template <int R, int C, typename A>
__device__ __forceinline__ void later_vertex(const Lay& L, size_t N, uint32_t v, KeBlocks kb,
                                             const float* __restrict__ w, const A* __restrict__ u,
                                             float* __restrict__ r, float zero) {
    int x, y, z;
    L.pos(v, x, y, z);
    FineCtx c;
    fine_ctx(c, x, y, z, L, w);
    float acc[R][3];
    fine_gather<R, later_mask(C), A>(c, N, kb, u, acc);
#pragma unroll
    for (int q = 0; q < R; q++) {
        float ro[3], rn[3];
#pragma unroll
        for (int i = 0; i < 3; i++) ro[i] = r[(size_t)(q * 3 + i) * N + v];
        rn[0] = ro[0] - acc[q][0];
        rn[1] = fmaf(-zero, rn[0], ro[1] - acc[q][1]);
        rn[2] = fmaf(-zero, rn[1], ro[2] - acc[q][2]);
#pragma unroll
        for (int i = 0; i < 3; i++) r[(size_t)(q * 3 + i) * N + v] = (v == 0) ? 0.f : rn[i];
    }
}

// Colours 0..6 in one launch, on the 128 x 2 x 2 vertex tiles of full_vertex (64 positions t of the
// eight parity blocks; colour c is block 7 - c) with four waves per tile: wave w takes colours w and
// 7 - w at the tile's positions in turn (a wave-uniform branch).  Colour c has 26, 24, 20, 18, 8, 6, 2,
// 0 later neighbours for c = 0..7, so each wave gathers 26 (one wave per colour left the colour-0
// wave to finish alone).  The tile's blocks share their neighbour rows in L1/L2, so the gathered u is
// fetched from HBM about once.  Parity-blocked levels only (make_lay(n, 0)).
template <int R, typename A>
__global__ __launch_bounds__(256) void k_fine_resid_later(Lay L, size_t N, const float* __restrict__ ke,
                                                          const float* __restrict__ w, const A* __restrict__ u,
                                                          float* __restrict__ r, float zero) {
    const KeBlocks kb = ke_blocks(ke);
    const uint32_t t = xcd_chunk(blockIdx.x, gridDim.x) * 64u + (threadIdx.x & 63u);
    if (t >= L.h3) return;
    const uint32_t h3 = L.h3;
    switch (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) {
        case 0: later_vertex<R, 0, A>(L, N, 7 * h3 + t, kb, w, u, r, zero); break;  // colour 7: none
        case 1:
            later_vertex<R, 1, A>(L, N, 6 * h3 + t, kb, w, u, r, zero);
            later_vertex<R, 6, A>(L, N, 1 * h3 + t, kb, w, u, r, zero);
            break;
        case 2:
            later_vertex<R, 2, A>(L, N, 5 * h3 + t, kb, w, u, r, zero);
            later_vertex<R, 5, A>(L, N, 2 * h3 + t, kb, w, u, r, zero);
            break;
        default:
            later_vertex<R, 3, A>(L, N, 4 * h3 + t, kb, w, u, r, zero);
            later_vertex<R, 4, A>(L, N, 3 * h3 + t, kb, w, u, r, zero);
            break;
    }
}

// Macro-strain right-hand sides f_s = sum_e w_e KE chi0_s for the 6 strains (grid.cu:1818-1919).
// kchi: 6 x 24 table of KE * chi0_s.  Pinned row zero.
__global__ __launch_bounds__(kFullThreads) void k_macro_rhs(Lay L, size_t N, const float* __restrict__ kchi,
                                                            const float* __restrict__ w, float* __restrict__ f) {
    uint32_t v;
    if (!full_vertex(L, xcd_chunk(blockIdx.x, gridDim.x), v)) return;
    int x, y, z;
    L.pos(v, x, y, z);
    FineCtx c;
    fine_ctx(c, x, y, z, L, w);
#pragma unroll
    for (int s = 0; s < 6; s++)
#pragma unroll
        for (int i = 0; i < 3; i++) {
            float a = 0.f;
#pragma unroll
            for (int e = 0; e < 8; e++) a = fmaf(c.wc[e], kchi[s * 24 + 3 * (7 - e) + i], a);
            f[(size_t)(s * 3 + i) * N + v] = (v == 0) ? 0.f : a;
        }
}

// Iterative-refinement residual in FP64 (the row of grid.cu:1277-1461 in FP64): r = f(w) - K u with u
// the FP64 solution, f the macro-strain loads rebuilt from the cell weights in FP64 (kchi64 = KE chi0
// in FP64) and every product accumulated in FP64.  Writes r rounded to FP32 (the inner solve's
// right-hand side) and per-block FP64 partial sums of |r|^2 per load case.  DO_K = false gives r = f
// (u = 0, nothing read from u).  All six load cases in one pass:
// the 27 FP64 blocks are built once per vertex and applied to every load case.  The neighbour loop
// stays rolled (d is uniform over the wave): fully unrolled, the FP64 gather spills.  At most 128
// VGPRs, so that two 512-thread workgroups share a CU (the FP64 gather is latency-bound).
template <bool DO_K>
__global__ __launch_bounds__(kFullThreads) __attribute__((amdgpu_waves_per_eu(4))) void k_fine_residual64(
    Lay L, size_t N, const double* __restrict__ ke, const double* __restrict__ kchi, const float* __restrict__ xc,
    double emin, const double* __restrict__ u, float* __restrict__ r32, double* __restrict__ partial) {
    constexpr int R = 6;
    __shared__ double sh[kFullThreads / 64];
    __shared__ double ke_s[kKeStaged];
    stage_ke(ke_s, ke);
    uint32_t v;
    const bool live = full_vertex(L, xcd_chunk(blockIdx.x, gridDim.x), v);
    double nrm[R];
#pragma unroll
    for (int r = 0; r < R; r++) nrm[r] = 0.0;
    if (live) {
        int x, y, z;
        L.pos(v, x, y, z);
        FineCtx c;
        fine_ctx64(c, x, y, z, L, xc, emin);
        double acc[R][3];
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int i = 0; i < 3; i++) acc[r][i] = 0.0;
        if (DO_K) {
            const Rsrc ru = make_rsrc(u, 18 * N * sizeof(double));
            const uint32_t plane = (uint32_t)(2 * N * sizeof(double));  // one plane of component pairs
            // cell weights and index parts as plain scalars: the loop below runs over a run-time d
            double wd[8];
#pragma unroll
            for (int e = 0; e < 8; e++) wd[e] = c.wd[e];
            const uint32_t X0 = c.X[0], X1 = c.X[1], X2 = c.X[2], Y0 = c.Y[0], Y1 = c.Y[1], Y2 = c.Y[2], Z0 = c.Z[0],
                           Z1 = c.Z[1], Z2 = c.Z[2];
#pragma unroll 1
            for (int d = 0; d < 27; d++) {
                const int dx = d % 3 - 1, dy = d / 3 % 3 - 1, dz = d / 9 - 1;
                const uint32_t qo = ((dx < 0 ? X0 : (dx == 0 ? X1 : X2)) + (dy < 0 ? Y0 : (dy == 0 ? Y1 : Y2)) +
                                     (dz < 0 ? Z0 : (dz == 0 ? Z1 : Z2))) *
                                    (uint32_t)sizeof(double2_t);
                double un[R][3];
#pragma unroll
                for (int q = 0; q < 9; q++) {
                    const double2_t w = bload<double2_t>(ru, qo, (uint32_t)q * plane);
                    un[(2 * q) / 3][(2 * q) % 3] = w.x;
                    un[(2 * q + 1) / 3][(2 * q + 1) % 3] = w.y;
                }
                // the block from signed sums of the weights of the cells holding v and v + d
                // (fine_block's form, with d known only at run time): cell e at offset
                // (e&1, e>>1&1, e>>2) - 1 holds v + d iff e_m = (d_m + 1) / 2 wherever d_m != 0; the sign
                // of axis m is -1 for e_m = 1 where d_m = 0
                double w0 = 0.0, fxy = 0.0, fxz = 0.0, fyz = 0.0;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int ex = e & 1, ey = (e >> 1) & 1, ez = e >> 2;
                    if ((dx == 0 || ex == (dx + 1) / 2) && (dy == 0 || ey == (dy + 1) / 2) &&
                        (dz == 0 || ez == (dz + 1) / 2)) {
                        const double sx = (dx == 0 && ex) ? -1.0 : 1.0, sy = (dy == 0 && ey) ? -1.0 : 1.0,
                                     sz = (dz == 0 && ez) ? -1.0 : 1.0;
                        w0 += wd[e];
                        fxy = fma(sx * sy, wd[e], fxy);
                        fxz = fma(sx * sz, wd[e], fxz);
                        fyz = fma(sy * sz, wd[e], fyz);
                    }
                }
                const double* cb = ke_s + kBlockConsts + 9 * d;
                const double S[9] = {cb[0] * w0,  cb[1] * fxy, cb[2] * fxz, cb[3] * fxy, cb[4] * w0,
                                     cb[5] * fyz, cb[6] * fxz, cb[7] * fyz, cb[8] * w0};
#pragma unroll
                for (int r = 0; r < R; r++)
#pragma unroll
                    for (int i = 0; i < 3; i++)
                        acc[r][i] = fma(S[i * 3], un[r][0], fma(S[i * 3 + 1], un[r][1], fma(S[i * 3 + 2], un[r][2], acc[r][i])));
            }
        }
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int i = 0; i < 3; i++) {
                double f = 0.0;
#pragma unroll
                for (int e = 0; e < 8; e++) f = fma(c.wd[e], kchi[r * 24 + 3 * (7 - e) + i], f);
                const double val = (v == 0) ? 0.0 : f - acc[r][i];
                r32[(size_t)(r * 3 + i) * N + v] = (float)val;
                nrm[r] = fma(val, val, nrm[r]);
            }
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        const double s = block_sum<kFullThreads>(nrm[r], sh);
        if (threadIdx.x == 0) partial[r * gridDim.x + blockIdx.x] = s;
    }
}

// |f|^2 per load case of the FP64 macro-strain loads (pinned row excluded).
__global__ __launch_bounds__(kFullThreads) void k_rhs_norm64(Lay L, size_t N, const double* __restrict__ kchi,
                                                             const float* __restrict__ xc, double emin,
                                                             double* __restrict__ partial) {
    __shared__ double sh[kFullThreads / 64];
    uint32_t v;
    const bool live = full_vertex(L, xcd_chunk(blockIdx.x, gridDim.x), v);
    double nrm[6] = {0, 0, 0, 0, 0, 0};
    if (live && v != 0) {
        int x, y, z;
        L.pos(v, x, y, z);
        FineCtx c;
        fine_ctx64(c, x, y, z, L, xc, emin);
#pragma unroll
        for (int s = 0; s < 6; s++)
#pragma unroll
            for (int i = 0; i < 3; i++) {
                double f = 0.0;
#pragma unroll
                for (int e = 0; e < 8; e++) f = fma(c.wd[e], kchi[s * 24 + 3 * (7 - e) + i], f);
                nrm[s] = fma(f, f, nrm[s]);
            }
    }
#pragma unroll
    for (int s = 0; s < 6; s++) {
        const double t = block_sum<kFullThreads>(nrm[s], sh);
        if (threadIdx.x == 0) partial[s * gridDim.x + blockIdx.x] = t;
    }
}

// u (+)= x + alpha p for all six load cases (x, p FP32 planes [18][N], N % 2 == 0; u in pairs,
// u64_index; alpha of load case r = sc[12 + r], taken as 0 unless pending): the last CG step's x
// update, rounded to FP32 as the CG pass rounds it, added to the FP64 iterate (add) or copied into
// it, in one pass.  Grid row q covers the pair plane of components 2q and 2q + 1.
__global__ __launch_bounds__(256) void k_refine_accumulate(size_t N, const double* __restrict__ sc, int pending,
                                                           const float* __restrict__ x, const float* __restrict__ p,
                                                           double* __restrict__ u, int add) {
    const int q = blockIdx.y, c0 = 2 * q, c1 = 2 * q + 1;
    const float a0 = pending ? (float)sc[12 + c0 / 3] : 0.f, a1 = pending ? (float)sc[12 + c1 / 3] : 0.f;
    const float2* x0 = reinterpret_cast<const float2*>(x + (size_t)c0 * N);
    const float2* x1 = reinterpret_cast<const float2*>(x + (size_t)c1 * N);
    const float2* p0 = reinterpret_cast<const float2*>(p + (size_t)c0 * N);
    const float2* p1 = reinterpret_cast<const float2*>(p + (size_t)c1 * N);
    double2* u2 = reinterpret_cast<double2*>(u + (size_t)q * 2 * N);
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < N / 2; i += (size_t)gridDim.x * blockDim.x) {
        float2 xa = x0[i], xb = x1[i];
        if (a0 != 0.f) {
            const float2 pa = p0[i];
            xa.x = fmaf(a0, pa.x, xa.x);
            xa.y = fmaf(a0, pa.y, xa.y);
        }
        if (a1 != 0.f) {
            const float2 pb = p1[i];
            xb.x = fmaf(a1, pb.x, xb.x);
            xb.y = fmaf(a1, pb.y, xb.y);
        }
        // vertices 2i and 2i + 1: pairs (c0, c1) of each
        double2 lo = make_double2((double)xa.x, (double)xb.x), hi = make_double2((double)xa.y, (double)xb.y);
        if (add) {
            const double2 ulo = u2[2 * i], uhi = u2[2 * i + 1];
            lo.x += ulo.x;
            lo.y += ulo.y;
            hi.x += uhi.x;
            hi.y += uhi.y;
        }
        u2[2 * i] = lo;
        u2[2 * i + 1] = hi;
    }
}

// FP64 iterate (pairs) -> FP32 planes [18][N], and back; one thread per (pair plane, vertex)
__global__ __launch_bounds__(256) void k_round_f32(size_t N, const double* __restrict__ u, float* __restrict__ x) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 9 * N) return;
    const size_t q = t / N, v = t - q * N;
    const double2 w = reinterpret_cast<const double2*>(u)[t];
    x[2 * q * N + v] = (float)w.x;
    x[(2 * q + 1) * N + v] = (float)w.y;
}

__global__ __launch_bounds__(256) void k_widen_f64(size_t N, const float* __restrict__ x, double* __restrict__ u) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 9 * N) return;
    const size_t q = t / N, v = t - q * N;
    reinterpret_cast<double2*>(u)[t] = make_double2((double)x[2 * q * N + v], (double)x[(2 * q + 1) * N + v]);
}

// zero the components of load case r (3 r .. 3 r + 2) of the FP64 iterate, every vertex
__global__ __launch_bounds__(256) void k_zero_case64(size_t N, int r, double* __restrict__ u) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 3 * N) return;
    const size_t k = t / N, v = t - k * N;
    u[u64_index(3 * r + (int)k, v, N)] = 0.0;
}

// zero the pinned origin's components of the FP64 iterate
__global__ void k_zero_pin64(size_t N, double* __restrict__ u) {
    if (threadIdx.x < 18) u[u64_index((int)threadIdx.x, 0, N)] = 0.0;
}

// zero the pinned origin's entries of a 6-load-case field of `planes` word planes
// FP32 planes [6][3][N] <-> packed FP16 words (word q = p * 3 + i: cases 2p, 2p + 1; hw_index)
__global__ __launch_bounds__(256) void k_pack_half(size_t N, const float* __restrict__ u, half2_t* __restrict__ z) {
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= 9 * N) return;
    const size_t q = t / N, v = t - q * N, p = q / 3, i = q - 3 * p;
    half2_t h;
    h.x = (_Float16)u[((2 * p) * 3 + i) * N + v];
    h.y = (_Float16)u[((2 * p + 1) * 3 + i) * N + v];
    z[hw_index((int)q, v, N)] = h;
}
__global__ __launch_bounds__(256) void k_unpack_half(size_t N, const half2_t* __restrict__ z, float* __restrict__ u) {
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= 9 * N) return;
    const size_t q = t / N, v = t - q * N, p = q / 3, i = q - 3 * p;
    const half2_t h = z[hw_index((int)q, v, N)];
    u[((2 * p) * 3 + i) * N + v] = (float)h.x;
    u[((2 * p + 1) * 3 + i) * N + v] = (float)h.y;
}

// (half: the 9 words of a packed FP16 field)
template <typename T, bool HALF = false>
__global__ void k_zero_pin(size_t N, int planes, T* __restrict__ u) {
    if ((int)threadIdx.x < planes) u[HALF ? hw_index((int)threadIdx.x, 0, N) : (size_t)threadIdx.x * N] = T(0);
}

// ---------------------------------------------------------------------------------------------
// Coarse levels (stored 27-point stencils)
// ---------------------------------------------------------------------------------------------

// One neighbour of a coarse row: issue the loads of the next selected neighbour (its stencil block and
// words), accumulate this one, recurse.  The barrier keeps the loads one neighbour ahead: with the whole
// row unrolled freely the compiler issues every neighbour's loads at once and needs 256 VGPRs.
struct StencilRow {
    Rsrc rs, ru;
    uint32_t X[3], Y[3], Z[3], vo, plane;
};
// The entries of a vertex's stencil, each loaded with the neighbour that first needs it (DP: the one loaded
// before, -1 none): packed FP16 in quads of eight, which the wave's loads fetch whole.  A word a load kept
// the texture addresser busy: a colour pair took 20.5 us at 40^3 and 22.4 at 64^3 (55 on average at 64^3 and
// 128^3), 17.8 and 19 (52) with quads and the vertex's own values loaded first.
template <typename SA>
struct StencilEntries;
template <>
struct StencilEntries<float> {
    float e[243];
    template <int DP, int D>
    __device__ __forceinline__ void load(Rsrc rs, uint32_t vo, uint32_t plane) {
#pragma unroll
        for (int k = 9 * D; k < 9 * D + 9; k++) e[k] = StencilIO<float>::get(rs, vo, plane, k);
    }
    __device__ __forceinline__ float get(int k) const { return e[k]; }
};
template <>
struct StencilEntries<half2_t> {
    typedef uint32_t Quad __attribute__((ext_vector_type(4)));
    Quad q[31];
    template <int DP, int D>
    __device__ __forceinline__ void load(Rsrc rs, uint32_t vo, uint32_t plane) {
        constexpr int before = DP < 0 ? 0 : (9 * DP + 8) / 8 + 1, first = 9 * D / 8 > before ? 9 * D / 8 : before;
#pragma unroll
        for (int k = first; k <= (9 * D + 8) / 8; k++)
            q[k] = __builtin_bit_cast(Quad, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(4u * vo), (int)((uint32_t)k * 4u * plane), 0));
    }
    __device__ __forceinline__ float get(int k) const {
        return (float)__builtin_bit_cast(half2_t, (uint32_t)q[k >> 3][k >> 1 & 3])[k & 1];
    }
};

template <typename A, int W, bool XL, int D>
__device__ __forceinline__ void stencil_nb(A (&cur)[W][3], const StencilRow& c, int r0, const XNbLds<A>& xl) {
    if constexpr (XL && (D == 12 || D == 14)) {
        load_nb_lds<W, A>(cur, xl, D == 12 ? 0 : 1);
    } else {
        const uint32_t qo = (c.X[D % 3] + c.Y[D / 3 % 3] + c.Z[D / 9]) * 4u;
        load_nb<W, A>(cur, c.ru, qo, c.plane, r0);
    }
}
template <int R, uint32_t MASK, int D, typename SA, typename A, bool XL>
__device__ __forceinline__ void stencil_step(const StencilRow& c, int r0, const XNbLds<A>& xl, StencilEntries<SA>& S,
                                             const A (&cur)[R / CasesPerWord<A>::value][3], float (&acc)[R][3]) {
    constexpr int W = R / CasesPerWord<A>::value;
    constexpr int DN = next_nb(MASK, D);
    __builtin_amdgcn_sched_barrier(0);
    pin_acc<R, float>(acc);
    A nxt[W][3];
    if constexpr (DN < 27) {
        S.template load<D, DN>(c.rs, c.vo, c.plane);
        stencil_nb<A, W, XL, DN>(nxt, c, r0, xl);
    }
    float e[9];
#pragma unroll
    for (int k = 0; k < 9; k++) e[k] = S.get(9 * D + k);
    block_fma<W, float, A>(e, cur, acc);
    if constexpr (DN < 27) stencil_step<R, MASK, DN, SA, A, XL>(c, r0, xl, S, nxt, acc);
}

// acc = sum over the neighbours selected by MASK of the stored 3x3 blocks times u, load cases r0 .. r0 + R - 1.
// A: storage of u (float planes, or half2_t words of load-case pairs; r0 then even).  XL: the two
// x-neighbours (d = 12, 14) come from LDS (xl).
template <int R, uint32_t MASK, typename SA, typename A = float, bool XL = false>
__device__ __forceinline__ void stencil_gather(int x, int y, int z, const Lay& L, size_t N, uint32_t v,
                                               const SA* __restrict__ st, const A* __restrict__ u,
                                               float (&acc)[R][3], int r0, const XNbLds<A>& xl = XNbLds<A>()) {
    constexpr int W = R / CasesPerWord<A>::value;
    StencilRow c;
    c.X[0] = L.part(wrap_dec(x, L.n), 0); c.X[1] = L.part(x, 0); c.X[2] = L.part(wrap_inc(x, L.n), 0);
    c.Y[0] = L.part(wrap_dec(y, L.n), 1); c.Y[1] = L.part(y, 1); c.Y[2] = L.part(wrap_inc(y, L.n), 1);
    c.Z[0] = L.part(wrap_dec(z, L.n), 2); c.Z[1] = L.part(z, 2); c.Z[2] = L.part(wrap_inc(z, L.n), 2);
    c.rs = make_rsrc(st, (size_t)StencilIO<SA>::words * N * 4);
    c.ru = make_rsrc(u, (size_t)(18 / CasesPerWord<A>::value) * N * sizeof(A));
    c.plane = (uint32_t)(N * sizeof(float));  // stencil and u words are 4 bytes
    c.vo = v * 4u;
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int i = 0; i < 3; i++) acc[r][i] = 0.f;
    constexpr int D0 = next_nb(MASK, -1);
    if constexpr (D0 < 27) {
        StencilEntries<SA> S;
        A cur[W][3];
        S.template load<-1, D0>(c.rs, c.vo, c.plane);
        stencil_nb<A, W, XL, D0>(cur, c, r0, xl);
        stencil_step<R, MASK, D0, SA, A, XL>(c, r0, xl, S, cur, acc);
    }
}

// MODE 0: out = A u; MODE 1: out = f - A u (update_residual_kernel_1, grid.cu:1465-1564).  A: u storage.
template <int R, int MODE, typename SA, typename A = float>
__global__ __launch_bounds__(kFullThreads) void k_stencil_apply(Lay L, size_t N, const SA* __restrict__ st,
                                                                const A* __restrict__ u,
                                                                const float* __restrict__ f, float* __restrict__ out) {
    uint32_t v;
    if (!full_vertex(L, xcd_chunk(blockIdx.x, gridDim.x), v)) return;
    int x, y, z;
    L.pos(v, x, y, z);
    float acc[R][3];
    const int r0 = blockIdx.y * R;
    stencil_gather<R, kRowAll, SA, A>(x, y, z, L, N, v, st, u, acc, r0);
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const size_t o = (size_t)((r0 + r) * 3 + i) * N + v;
            out[o] = (MODE == 1) ? f[o] - acc[r][i] : acc[r][i];
        }
}

// GS / SOR update of the colour vertex v of a coarse level (load cases r0 .. r0 + R - 1), in place.
// ZC as in k_fine_gs2.  A: u storage (float, or half2_t load-case pairs with FP32 arithmetic).  XL: the
// x-neighbours come from LDS; TO_LDS: the new words also go to slot threadIdx.x of out_lds.  ROWN
// (ZC >= 0): also the own-colour residual f - (A u)_{colours <= ZC} to rown, as gs_vertex does.
template <int R, bool REVERSE, int ZC, typename SA, typename A, bool XL, bool TO_LDS, bool ROWN = false>
__device__ __forceinline__ void stencil_gs_vertex(const Lay& L, size_t N, uint32_t v, float omega,
                                                  const SA* __restrict__ st, A* __restrict__ u,
                                                  const float* __restrict__ f, int r0, const XNbLds<A>& xl,
                                                  A* out_lds, float* __restrict__ rown = nullptr) {
    static_assert(!ROWN || ZC >= 0, "the own-colour residual needs a zero-start forward pass");
    int x, y, z;
    L.pos(v, x, y, z);
    constexpr int cpw = CasesPerWord<A>::value;
    // the vertex's own values are loaded before the gather: after it, their latency would be the wave's
    constexpr bool own = cpw == 2 && ZC < 0;
    float fv[R][3];
    A old[own ? R / cpw : 1][3];
    StencilEntries<SA> diag;
    diag.template load<-1, 13>(make_rsrc(st, (size_t)StencilIO<SA>::words * N * 4), v * 4u, (uint32_t)(N * 4));
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int i = 0; i < 3; i++) fv[r][i] = f[(size_t)((r0 + r) * 3 + i) * N + v];
    if constexpr (own) {
#pragma unroll
        for (int p = 0; p < R / cpw; p++)
#pragma unroll
            for (int i = 0; i < 3; i++) old[p][i] = u[fw_index<A>((r0 / cpw + p) * 3 + i, v, N)];
    }
    float acc[R][3];
    stencil_gather<R, gs_mask(ZC), SA, A, XL>(x, y, z, L, N, v, st, u, acc, r0, xl);
    float Ks[9];
#pragma unroll
    for (int k = 0; k < 9; k++) Ks[k] = diag.get(13 * 9 + k);
    const float inv[3] = {1.f / Ks[0], 1.f / Ks[4], 1.f / Ks[8]};
#pragma unroll
    for (int p = 0; p < R / cpw; p++) {
        A wd[3];
#pragma unroll
        for (int i = 0; i < 3; i++)
            wd[i] = ZC >= 0 ? A(0) : own ? old[own ? p : 0][i] : u[fw_index<A>((r0 / cpw + p) * 3 + i, v, N)];
#pragma unroll
        for (int hh = 0; hh < cpw; hh++) {
            const int r = p * cpw + hh;
            float uu[3], ff[3];
#pragma unroll
            for (int i = 0; i < 3; i++) {
                if constexpr (cpw == 2)
                    uu[i] = (float)wd[i][hh];
                else
                    uu[i] = (float)wd[i];
                ff[i] = fv[r][i];
            }
            block_update<REVERSE>(uu, ff, acc[r], Ks, inv, omega);
#pragma unroll
            for (int i = 0; i < 3; i++) {
                if constexpr (cpw == 2)
                    wd[i][hh] = (_Float16)uu[i];
                else
                    wd[i] = uu[i];
            }
            if constexpr (ROWN) {
                float us[3];  // the stored values
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    if constexpr (cpw == 2)
                        us[i] = (float)wd[i][hh];
                    else
                        us[i] = (float)wd[i];
                }
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    const float kv = fmaf(Ks[3 * i], us[0], fmaf(Ks[3 * i + 1], us[1], Ks[3 * i + 2] * us[2]));
                    rown[(size_t)((r0 + r) * 3 + i) * N + v] = (ff[i] - acc[r][i]) - kv;
                }
            }
        }
#pragma unroll
        for (int i = 0; i < 3; i++) {
            u[fw_index<A>((r0 / cpw + p) * 3 + i, v, N)] = wd[i];
            if constexpr (TO_LDS) out_lds[(p * 3 + i) * 256 + threadIdx.x] = wd[i];
        }
    }
}

// One colour of the coarse block GS sweep (gs_relaxation_kernel, grid.cu:556-689) on a level of at most 32^3
// with FP32 stencils, a load case per thread; no pin on coarse levels.
template <bool REVERSE, int ZC>
__global__ __launch_bounds__(256) void k_stencil_gs(Lay L, size_t N, int colour, float omega, const float* __restrict__ st,
                                                    float* __restrict__ u, const float* __restrict__ f) {
    const uint32_t t = xcd_chunk(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (t >= L.h3) return;
    stencil_gs_vertex<1, REVERSE, ZC, float, float, false, false>(L, N, colour_block(colour) * L.h3 + t, omega, st, u, f,
                                                                  blockIdx.y, XNbLds<float>(), nullptr);
}

// Two consecutive colours of a coarse sweep in one launch, as k_fine_gs2 does at the finest level
// (whole grid rows per workgroup; the first colour's new words stay in LDS for the second colour's
// x-neighbours).
template <int R, bool REVERSE, int ZC, typename SA, typename A, bool ROWN = false>
__global__ __launch_bounds__(256) void k_stencil_gs2(Lay L, size_t N, int cfirst, float omega,
                                                     const SA* __restrict__ st, A* __restrict__ u,
                                                     const float* __restrict__ f, float* __restrict__ rown) {
    constexpr int W = R / CasesPerWord<A>::value;
    __shared__ A xs[3 * W * 256];
    const int h = L.h, span = pair_rows(h) * h;
    const uint32_t t = xcd_chunk(blockIdx.x, gridDim.x) * (uint32_t)span + threadIdx.x;
    const bool live = (int)threadIdx.x < span && t < L.h3;
    const int c2 = REVERSE ? cfirst - 1 : cfirst + 1;
    const int r0 = blockIdx.y * R;
    if (live)
        stencil_gs_vertex<R, REVERSE, ZC, SA, A, false, true, ROWN>(L, N, colour_block(cfirst) * L.h3 + t, omega, st, u,
                                                                    f, r0, XNbLds<A>(), xs, rown);
    __syncthreads();
    if (!live) return;
    XNbLds<A> xl;
    xl.base = xs;
    const int lx = (int)(t % (uint32_t)h), row0 = (int)threadIdx.x - lx;
    const bool odd = (colour_block(c2) & 1u) != 0;  // x-parity of the second colour
    xl.slot[0] = row0 + (odd ? lx : (lx == 0 ? h - 1 : lx - 1));
    xl.slot[1] = row0 + (odd ? (lx + 1 == h ? 0 : lx + 1) : lx);
    stencil_gs_vertex<R, REVERSE, (ZC < 0 ? -1 : ZC + 1), SA, A, true, false, ROWN>(
        L, N, colour_block(c2) * L.h3 + t, omega, st, u, f, r0, xl, nullptr, rown);
}

// The coarse-level counterpart of k_fine_resid_later: r = r_own - the later-colour terms, on the same
// parity tiles with four waves (wave w takes colours w and 7 - w; colour 7 is final).  Load cases
// r0 .. r0 + R - 1 with r0 = blockIdx.y R.  zero as in k_fine_resid_later.
template <int R, int C, typename SA, typename A>
__device__ __forceinline__ void stencil_later_vertex(const Lay& L, size_t N, uint32_t v, const SA* __restrict__ st,
                                                     const A* __restrict__ u, float* __restrict__ r, int r0,
                                                     float zero) {
    int x, y, z;
    L.pos(v, x, y, z);
    float acc[R][3];
    stencil_gather<R, later_mask(C), SA, A>(x, y, z, L, N, v, st, u, acc, r0);
#pragma unroll
    for (int q = 0; q < R; q++) {
        float ro[3], rn[3];
#pragma unroll
        for (int i = 0; i < 3; i++) ro[i] = r[(size_t)((r0 + q) * 3 + i) * N + v];
        rn[0] = ro[0] - acc[q][0];
        rn[1] = fmaf(-zero, rn[0], ro[1] - acc[q][1]);
        rn[2] = fmaf(-zero, rn[1], ro[2] - acc[q][2]);
#pragma unroll
        for (int i = 0; i < 3; i++) r[(size_t)((r0 + q) * 3 + i) * N + v] = rn[i];
    }
}

template <int R, typename SA, typename A>
__global__ __launch_bounds__(256) void k_stencil_resid_later(Lay L, size_t N, const SA* __restrict__ st,
                                                             const A* __restrict__ u, float* __restrict__ r,
                                                             float zero) {
    const uint32_t t = xcd_chunk(blockIdx.x, gridDim.x) * 64u + (threadIdx.x & 63u);
    if (t >= L.h3) return;
    const uint32_t h3 = L.h3;
    const int r0 = blockIdx.y * R;
    switch (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) {
        case 0: stencil_later_vertex<R, 0, SA, A>(L, N, 7 * h3 + t, st, u, r, r0, zero); break;
        case 1:
            stencil_later_vertex<R, 1, SA, A>(L, N, 6 * h3 + t, st, u, r, r0, zero);
            stencil_later_vertex<R, 6, SA, A>(L, N, 1 * h3 + t, st, u, r, r0, zero);
            break;
        case 2:
            stencil_later_vertex<R, 2, SA, A>(L, N, 5 * h3 + t, st, u, r, r0, zero);
            stencil_later_vertex<R, 5, SA, A>(L, N, 2 * h3 + t, st, u, r, r0, zero);
            break;
        default:
            stencil_later_vertex<R, 3, SA, A>(L, N, 4 * h3 + t, st, u, r, r0, zero);
            stencil_later_vertex<R, 4, SA, A>(L, N, 3 * h3 + t, st, u, r, r0, zero);
            break;
    }
}


// ---------------------------------------------------------------------------------------------
// Grid transfers (restrict_residual_kernel_1 grid.cu:917-994; prolongate_correction_kernel_1
// grid.cu:1120-1190).  Weights prod_k (2-|o_k|)/2; R = P^T.
// ---------------------------------------------------------------------------------------------
template <int R>
__global__ __launch_bounds__(256) void k_restrict(Lay Lf, Lay Lc, const float* __restrict__ rf,
                                                  float* __restrict__ fc) {
    const size_t Nc = (size_t)Lc.n * Lc.n * Lc.n, Nf = (size_t)Lf.n * Lf.n * Lf.n;
    int X, Y, Z;
    uint32_t V;
    if (!coarse_lex_vertex(Lc, X, Y, Z, V)) return;
    const uint32_t xs[3] = {Lf.part(wrap_dec(2 * X, Lf.n), 0), Lf.part(2 * X, 0), Lf.part(2 * X + 1, 0)};
    const uint32_t ys[3] = {Lf.part(wrap_dec(2 * Y, Lf.n), 1), Lf.part(2 * Y, 1), Lf.part(2 * Y + 1, 1)};
    const uint32_t zs[3] = {Lf.part(wrap_dec(2 * Z, Lf.n), 2), Lf.part(2 * Z, 2), Lf.part(2 * Z + 1, 2)};
    float acc[R][3];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int i = 0; i < 3; i++) acc[r][i] = 0.f;
    const int r0 = blockIdx.y * R;
#pragma unroll
    for (int o = 0; o < 27; o++) {
        const int ox = o % 3, oy = o / 3 % 3, oz = o / 9;
        const float wgt = (float)((ox == 1 ? 2 : 1) * (oy == 1 ? 2 : 1) * (oz == 1 ? 2 : 1)) * 0.125f;
        const uint32_t q = xs[ox] + ys[oy] + zs[oz];
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int i = 0; i < 3; i++)
                acc[r][i] = fmaf(wgt, rf[(size_t)((r0 + r) * 3 + i) * Nf + q], acc[r][i]);
    }
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int i = 0; i < 3; i++) fc[(size_t)((r0 + r) * 3 + i) * Nc + V] = acc[r][i];
}

template <int R>
__global__ __launch_bounds__(kFullThreads) void k_prolong(Lay Lf, Lay Lc, const float* __restrict__ uc,
                                                          float* __restrict__ uf, int pin) {
    const size_t Nc = (size_t)Lc.n * Lc.n * Lc.n, Nf = (size_t)Lf.n * Lf.n * Lf.n;
    uint32_t v;
    if (!full_vertex(Lf, xcd_chunk(blockIdx.x, gridDim.x), v)) return;
    if (pin && v == 0) return;
    const int nc = Lc.n;
    int x, y, z;
    Lf.pos(v, x, y, z);
    // per axis: even -> one parent weight 1, odd -> two parents weight 1/2
    int ix[2], iy[2], iz[2];
    float wx[2], wy[2], wz[2];
    ix[0] = x >> 1; ix[1] = (x & 1) ? ((x >> 1) + 1 == nc ? 0 : (x >> 1) + 1) : ix[0];
    wx[0] = (x & 1) ? 0.5f : 1.f; wx[1] = (x & 1) ? 0.5f : 0.f;
    iy[0] = y >> 1; iy[1] = (y & 1) ? ((y >> 1) + 1 == nc ? 0 : (y >> 1) + 1) : iy[0];
    wy[0] = (y & 1) ? 0.5f : 1.f; wy[1] = (y & 1) ? 0.5f : 0.f;
    iz[0] = z >> 1; iz[1] = (z & 1) ? ((z >> 1) + 1 == nc ? 0 : (z >> 1) + 1) : iz[0];
    wz[0] = (z & 1) ? 0.5f : 1.f; wz[1] = (z & 1) ? 0.5f : 0.f;
    float acc[R][3];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int i = 0; i < 3; i++) acc[r][i] = 0.f;
    const int r0 = blockIdx.y * R;
#pragma unroll
    for (int p = 0; p < 8; p++) {
        const float wgt = wx[p & 1] * wy[(p >> 1) & 1] * wz[p >> 2];
        if (wgt == 0.f) continue;
        const uint32_t q = Lc.idx(ix[p & 1], iy[(p >> 1) & 1], iz[p >> 2]);
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int i = 0; i < 3; i++)
                acc[r][i] = fmaf(wgt, uc[(size_t)((r0 + r) * 3 + i) * Nc + q], acc[r][i]);
    }
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int i = 0; i < 3; i++) uf[(size_t)((r0 + r) * 3 + i) * Nf + v] += acc[r][i];
}

// Vectorised transfers for nf % 8 == 0 (so nc = nf / 2 and the fine local row length are multiples of
// 4): each thread handles four consecutive x of one load case (r = blockIdx.y) with float4 / float2
// accesses.  Same weights and sums as k_restrict / k_prolong.
//
// Restriction: coarse X = 4j..4j+3 of row (Y, Z).  Along x the fine taps are 2X (even block, local X),
// 2X+1 (odd block, local X) and 2X-1 (odd block, local X-1): two float4 rows and one scalar.
__global__ __launch_bounds__(256) void k_restrict4(Lay Lf, Lay Lc, const float* __restrict__ rf,
                                                   float* __restrict__ fc) {
    const int nf = Lf.n, nc = Lc.n, q = nc / 4;
    const uint32_t i = xcd_chunk(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (i >= (uint32_t)q * nc * nc) return;
    const int j = (int)(i % q), Y = (int)((i / q) % nc), Z = (int)(i / ((uint32_t)q * nc));
    const size_t Nf = (size_t)nf * nf * nf, Nc = (size_t)nc * nc * nc;
    const int r = blockIdx.y;
    const uint32_t xe = Lf.part(8 * j, 0), xo = Lf.part(8 * j + 1, 0), xp = Lf.part(wrap_dec(8 * j, nf), 0);
    const uint32_t ys[3] = {Lf.part(wrap_dec(2 * Y, nf), 1), Lf.part(2 * Y, 1), Lf.part(2 * Y + 1, 1)};
    const uint32_t zs[3] = {Lf.part(wrap_dec(2 * Z, nf), 2), Lf.part(2 * Z, 2), Lf.part(2 * Z + 1, 2)};
    const float wt[3] = {0.5f, 1.f, 0.5f};
#pragma unroll
    for (int c = 0; c < 3; c++) {
        const float* pl = rf + (size_t)(r * 3 + c) * Nf;
        float a[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int oz = 0; oz < 3; oz++)
#pragma unroll
            for (int oy = 0; oy < 3; oy++) {
                const uint32_t base = ys[oy] + zs[oz];
                const float4 e = *reinterpret_cast<const float4*>(pl + base + xe);
                const float4 o = *reinterpret_cast<const float4*>(pl + base + xo);
                const float op = pl[base + xp];
                const float w = wt[oy] * wt[oz];
                a[0] = fmaf(w, e.x + 0.5f * (o.x + op), a[0]);
                a[1] = fmaf(w, e.y + 0.5f * (o.y + o.x), a[1]);
                a[2] = fmaf(w, e.z + 0.5f * (o.z + o.y), a[2]);
                a[3] = fmaf(w, e.w + 0.5f * (o.w + o.z), a[3]);
            }
        float* out = fc + (size_t)(r * 3 + c) * Nc;
        if (Lc.lex) {
            *reinterpret_cast<float4*>(out + Lc.idx(4 * j, Y, Z)) = make_float4(a[0], a[1], a[2], a[3]);
        } else {
            const uint32_t yz = Lc.part(Y, 1) + Lc.part(Z, 2);
            *reinterpret_cast<float2*>(out + yz + Lc.part(4 * j, 0)) = make_float2(a[0], a[2]);
            *reinterpret_cast<float2*>(out + yz + Lc.part(4 * j + 1, 0)) = make_float2(a[1], a[3]);
        }
    }
}

// Prolongation: the 8 waves of a workgroup take the 8 fine parity blocks; a lane adds P u_c to four
// consecutive local x (fine x = 2lx + px) of one row.  Parents along x: lx (weight 1) when px = 0;
// lx and lx + 1 (1/2 each) when px = 1.
__global__ __launch_bounds__(kFullThreads) void k_prolong4(Lay Lf, Lay Lc, const float* __restrict__ uc,
                                                           float* __restrict__ uf, int pin) {
    const uint32_t hf = (uint32_t)Lf.h, q = hf / 4;
    const uint32_t t4 = xcd_chunk(blockIdx.x, gridDim.x) * 64u + (threadIdx.x & 63u);
    if (t4 >= Lf.h3 / 4) return;
    const uint32_t b = threadIdx.x >> 6;
    const int px = b & 1, py = (b >> 1) & 1, pz = (int)(b >> 2);
    const uint32_t j = t4 % q, row = t4 / q;
    const int ly = (int)(row % hf), lz = (int)(row / hf);
    const int nc = Lc.n;
    const int Ys[2] = {ly, ly + 1 == nc ? 0 : ly + 1}, Zs[2] = {lz, lz + 1 == nc ? 0 : lz + 1};
    const float wy[2] = {py ? 0.5f : 1.f, 0.5f}, wz[2] = {pz ? 0.5f : 1.f, 0.5f};
    const int X4 = (int)(4 * j + 4) == nc ? 0 : (int)(4 * j + 4);
    const size_t Nf = (size_t)Lf.n * Lf.n * Lf.n, Nc = (size_t)nc * nc * nc;
    const int r = blockIdx.y;
    const bool skip0 = pin && b == 0 && row == 0 && j == 0;  // pinned origin
#pragma unroll
    for (int c = 0; c < 3; c++) {
        const float* cp = uc + (size_t)(r * 3 + c) * Nc;
        float a[4] = {0.f, 0.f, 0.f, 0.f};
        for (int iz = 0; iz <= pz; iz++)
            for (int iy = 0; iy <= py; iy++) {
                float cv[5];
                if (Lc.lex) {
                    const uint32_t base = (uint32_t)nc * (Ys[iy] + (uint32_t)nc * Zs[iz]);
                    const float4 v4 = *reinterpret_cast<const float4*>(cp + base + 4 * j);
                    cv[0] = v4.x; cv[1] = v4.y; cv[2] = v4.z; cv[3] = v4.w;
                    cv[4] = px ? cp[base + X4] : 0.f;
                } else {
                    const uint32_t yz = Lc.part(Ys[iy], 1) + Lc.part(Zs[iz], 2);
                    const float2 ev = *reinterpret_cast<const float2*>(cp + yz + Lc.part(4 * j, 0));
                    const float2 od = *reinterpret_cast<const float2*>(cp + yz + Lc.part(4 * j + 1, 0));
                    cv[0] = ev.x; cv[1] = od.x; cv[2] = ev.y; cv[3] = od.y;
                    cv[4] = px ? cp[yz + Lc.part(X4, 0)] : 0.f;
                }
                const float w = wy[iy] * wz[iz];
#pragma unroll
                for (int k = 0; k < 4; k++) a[k] = fmaf(w, px ? 0.5f * (cv[k] + cv[k + 1]) : cv[k], a[k]);
            }
        float4* dst = reinterpret_cast<float4*>(uf + (size_t)(r * 3 + c) * Nf + b * Lf.h3 + row * hf + 4 * j);
        float4 u4 = *dst;
        u4.x += skip0 ? 0.f : a[0];
        u4.y += a[1];
        u4.z += a[2];
        u4.w += a[3];
        *dst = u4;
    }
}

// Prolongation into a packed FP16 fine field (hw_index words): uf += P uc, one thread per fine vertex
// and all nine of its words (two 16-byte and one 4-byte read-modify-write), on the 512-thread parity
// tiles of full_vertex.  Per axis an even fine coordinate has one coarse parent (weight 1) and an odd one
// two (weight 1/2 each): the x parents are averaged first, then the (y, z) parents accumulate with their
// weights.  CT: coarse storage, FP32 planes (lexicographic or parity-blocked) or packed FP16 words
// (parity-blocked).  The pinned origin (pin) keeps its value.
template <typename CT>
__device__ __forceinline__ void coarse_words(float (&c)[9][2], const CT* __restrict__ uc, uint32_t idx, size_t Nc) {
    if constexpr (CasesPerWord<CT>::value == 2) {
        const uint32_t* w = reinterpret_cast<const uint32_t*>(uc);
        const uint4 a = *reinterpret_cast<const uint4*>(w + 4 * (size_t)idx);
        const uint4 b = *reinterpret_cast<const uint4*>(w + 4 * Nc + 4 * (size_t)idx);
        const uint32_t wv[9] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w, w[8 * Nc + idx]};
#pragma unroll
        for (int q = 0; q < 9; q++) {
            const half2_t hv = __builtin_bit_cast(half2_t, wv[q]);
            c[q][0] = (float)hv.x;
            c[q][1] = (float)hv.y;
        }
    } else {
#pragma unroll
        for (int q = 0; q < 9; q++)
#pragma unroll
            for (int h = 0; h < 2; h++) c[q][h] = uc[(size_t)((2 * (q / 3) + h) * 3 + q % 3) * Nc + idx];
    }
}

template <typename CT>
__global__ __launch_bounds__(kFullThreads) void k_prolong_h(Lay Lf, Lay Lc, const CT* __restrict__ uc,
                                                           half2_t* __restrict__ uf, int pin) {
    uint32_t v;
    if (!full_vertex(Lf, xcd_chunk(blockIdx.x, gridDim.x), v)) return;
    if (pin && v == 0) return;
    int x, y, z;
    Lf.pos(v, x, y, z);
    const int nc = Lc.n;
    const int px = x & 1, py = y & 1, pz = z & 1;
    const int X0 = x >> 1, X1 = X0 + 1 == nc ? 0 : X0 + 1;
    const int Ys[2] = {y >> 1, (y >> 1) + 1 == nc ? 0 : (y >> 1) + 1};
    const int Zs[2] = {z >> 1, (z >> 1) + 1 == nc ? 0 : (z >> 1) + 1};
    const float wy[2] = {py ? 0.5f : 1.f, 0.5f}, wz[2] = {pz ? 0.5f : 1.f, 0.5f};
    const size_t Nf = (size_t)Lf.n * Lf.n * Lf.n, Nc = (size_t)nc * nc * nc;
    float a[9][2];
#pragma unroll
    for (int q = 0; q < 9; q++) a[q][0] = a[q][1] = 0.f;
    for (int iz = 0; iz <= pz; iz++)
        for (int iy = 0; iy <= py; iy++) {
            const float w = wy[iy] * wz[iz];
            float c0[9][2], c1[9][2];
            coarse_words<CT>(c0, uc, Lc.idx(X0, Ys[iy], Zs[iz]), Nc);
            if (px) coarse_words<CT>(c1, uc, Lc.idx(X1, Ys[iy], Zs[iz]), Nc);
#pragma unroll
            for (int q = 0; q < 9; q++)
#pragma unroll
                for (int h = 0; h < 2; h++) a[q][h] = fmaf(w, px ? 0.5f * (c0[q][h] + c1[q][h]) : c0[q][h], a[q][h]);
        }
    uint32_t* fw = reinterpret_cast<uint32_t*>(uf);
    uint4* f0 = reinterpret_cast<uint4*>(fw + 4 * (size_t)v);
    uint4* f1 = reinterpret_cast<uint4*>(fw + 4 * Nf + 4 * (size_t)v);
    const uint4 o0 = *f0, o1 = *f1;
    uint32_t wv[9] = {o0.x, o0.y, o0.z, o0.w, o1.x, o1.y, o1.z, o1.w, fw[8 * Nf + v]};
#pragma unroll
    for (int q = 0; q < 9; q++) {
        half2_t hv = __builtin_bit_cast(half2_t, wv[q]);
        hv.x = (_Float16)((float)hv.x + a[q][0]);
        hv.y = (_Float16)((float)hv.y + a[q][1]);
        wv[q] = __builtin_bit_cast(uint32_t, hv);
    }
    *f0 = make_uint4(wv[0], wv[1], wv[2], wv[3]);
    *f1 = make_uint4(wv[4], wv[5], wv[6], wv[7]);
    fw[8 * Nf + v] = wv[8];
}

// ---------------------------------------------------------------------------------------------
// FP64 reductions and vector updates (per load case)
// ---------------------------------------------------------------------------------------------
// partial[r * gridDim.x + b] = block b's grid-stride share of a_r . b_r, r = blockIdx.y (3N values
// per load case); products are exact in FP64 and summed in FP64.
__global__ __launch_bounds__(256) void k_dot(size_t M, const float* __restrict__ a, const float* __restrict__ b,
                                             double* __restrict__ partial) {
    __shared__ double sh[4];
    const int r = blockIdx.y;
    const float* ar = a + (size_t)r * M;
    const float* br = b + (size_t)r * M;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    double s = 0.0;
    if ((M & 3) == 0) {
        const float4* a4 = reinterpret_cast<const float4*>(ar);
        const float4* b4 = reinterpret_cast<const float4*>(br);
        for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < M / 4; i += stride) {
            const float4 x = a4[i], y = b4[i];
            s += ((double)x.x * y.x + (double)x.y * y.y) + ((double)x.z * y.z + (double)x.w * y.w);
        }
    } else {
        for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < M; i += stride) s += (double)ar[i] * br[i];
    }
    s = block_sum<256>(s, sh);
    if (threadIdx.x == 0) partial[r * gridDim.x + blockIdx.x] = s;
}

// out[r] = sum of partial[r * nb + i] over i < nb; one workgroup per row, four independent loads in
// flight per thread.
//
// What a CG step derives from a sum is formed by the workgroup that has it (a launch of its own is 4 us and a
// gap): sc = [rz | pq | alpha | rz_new | beta | active], six each; kSumPq: out is pq, alpha = rz / pq;
// kSumRz: out is rz_new, beta = rz_new / rz, then rz = rz_new.  Zero for load cases no longer active.
template <int THEN>
__global__ __launch_bounds__(kSumThreads) void k_sum_partials(int nb, const double* __restrict__ partial, double* out,
                                                              double* sc) {
    __shared__ double sh[kSumThreads / 64];
    const double* p = partial + (size_t)blockIdx.x * nb;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    int i = threadIdx.x;
    for (; i + 3 * kSumThreads < nb; i += 4 * kSumThreads) {
        s0 += p[i];
        s1 += p[i + kSumThreads];
        s2 += p[i + 2 * kSumThreads];
        s3 += p[i + 3 * kSumThreads];
    }
    for (; i < nb; i += kSumThreads) s0 += p[i];
    const double s = block_sum<kSumThreads>((s0 + s1) + (s2 + s3), sh);
    if (threadIdx.x == 0) {
        const int r = (int)blockIdx.x;
        out[r] = s;
        if constexpr (THEN == kSumPq) sc[12 + r] = sc[30 + r] != 0.0 && s != 0.0 ? sc[r] / s : 0.0;
        if constexpr (THEN == kSumRz) {
            const double rz = sc[r];
            sc[24 + r] = sc[30 + r] != 0.0 && rz != 0.0 ? s / rz : 0.0;
            sc[r] = s;
        }
    }
}

// CG vector updates, one grid row per load case k = blockIdx.y, grid-stride over the M values of a
// load case in float4 steps (M % 4 == 0; the caller checks it).
//
// r -= alpha q, with per-block FP64 partial sums of |r|^2 in partial[k * gridDim.x + block].
__global__ __launch_bounds__(256) void k_pcg_update_r(int R, size_t M, const double* __restrict__ sc,
                                                      const float* __restrict__ q, float* __restrict__ r,
                                                      double* __restrict__ partial) {
    __shared__ double sh[4];
    const int k = blockIdx.y;
    const float a = (float)sc[2 * R + k];
    const float4* q4 = reinterpret_cast<const float4*>(q + (size_t)k * M);
    float4* r4 = reinterpret_cast<float4*>(r + (size_t)k * M);
    double s = 0.0;
    typedef float v4f __attribute__((ext_vector_type(4)));
    const v4f* qn = reinterpret_cast<const v4f*>(q4);
    v4f* rn = reinterpret_cast<v4f*>(r4);
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < M / 4; i += (size_t)gridDim.x * blockDim.x) {
        const v4f qv = __builtin_nontemporal_load(qn + i);
        v4f rv = __builtin_nontemporal_load(rn + i);
        rv.x = fmaf(-a, qv.x, rv.x);
        rv.y = fmaf(-a, qv.y, rv.y);
        rv.z = fmaf(-a, qv.z, rv.z);
        rv.w = fmaf(-a, qv.w, rv.w);
        __builtin_nontemporal_store(rv, rn + i);
        s += ((double)rv.x * rv.x + (double)rv.y * rv.y) + ((double)rv.z * rv.z + (double)rv.w * rv.w);
    }
    s = block_sum<256>(s, sh);
    if (threadIdx.x == 0) partial[k * gridDim.x + blockIdx.x] = s;
}

// x += alpha p (the step of this iteration, all load cases: alpha is zero for finished ones), then,
// when do_p, p = z + beta p for the active load cases.
__global__ __launch_bounds__(256) void k_pcg_update_px(int R, size_t M, const double* __restrict__ sc,
                                                       const float* __restrict__ z, float* __restrict__ p,
                                                       float* __restrict__ x, int do_p) {
    const int k = blockIdx.y;
    const float a = (float)sc[2 * R + k];
    const float b = (float)sc[4 * R + k];
    const bool upd = do_p && sc[5 * R + k] != 0.0;
    const float4* z4 = reinterpret_cast<const float4*>(z + (size_t)k * M);
    float4* p4 = reinterpret_cast<float4*>(p + (size_t)k * M);
    float4* x4 = reinterpret_cast<float4*>(x + (size_t)k * M);
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < M / 4; i += (size_t)gridDim.x * blockDim.x) {
        float4 pv = p4[i];
        if (a != 0.f) {
            float4 xv = x4[i];
            xv.x = fmaf(a, pv.x, xv.x);
            xv.y = fmaf(a, pv.y, xv.y);
            xv.z = fmaf(a, pv.z, xv.z);
            xv.w = fmaf(a, pv.w, xv.w);
            x4[i] = xv;
        }
        if (upd) {
            const float4 zv = z4[i];
            pv.x = fmaf(b, pv.x, zv.x);
            pv.y = fmaf(b, pv.y, zv.y);
            pv.z = fmaf(b, pv.z, zv.z);
            pv.w = fmaf(b, pv.w, zv.w);
            p4[i] = pv;
        }
    }
}

// The same CG steps with the preconditioned vector z in packed FP16 (hw_index words; load-case pair
// pr = blockIdx.y holds cases 2pr (.x) and 2pr + 1 (.y); M = 3 N values per load case, N % 4 == 0).
//
// words q = pr * 3 + c (c = e / N, the entry e = 4 i of the pair's M = 3 N values) of the four vertices
// e % N .. e % N + 3 of a packed FP16 field (hw_index; N % 4 == 0)
__device__ __forceinline__ void hwords4(half2_t (&o)[4], const half2_t* __restrict__ z, int pr, size_t i, size_t N) {
    const size_t e = 4 * i, c = e / N, v0 = e - c * N;
    const int q = pr * 3 + (int)c;
    if (q == 8) {
        const uint4 w = *reinterpret_cast<const uint4*>(z + 8 * N + v0);
        o[0] = __builtin_bit_cast(half2_t, w.x);
        o[1] = __builtin_bit_cast(half2_t, w.y);
        o[2] = __builtin_bit_cast(half2_t, w.z);
        o[3] = __builtin_bit_cast(half2_t, w.w);
    } else {
#pragma unroll
        for (int k = 0; k < 4; k++) o[k] = z[hw_index(q, v0 + k, N)];
    }
}

// partial[(2pr + h) * gridDim.x + block] = block's share of r_{2pr+h} . z_{2pr+h}
__global__ __launch_bounds__(256) void k_dot_fh(size_t M, const float* __restrict__ r, const half2_t* __restrict__ z,
                                                double* __restrict__ partial) {
    __shared__ double sh[4];
    const int pr = blockIdx.y;
    const size_t N = M / 3;
    const float4* r0 = reinterpret_cast<const float4*>(r + (size_t)(2 * pr) * M);
    const float4* r1 = reinterpret_cast<const float4*>(r + (size_t)(2 * pr + 1) * M);
    double s0 = 0.0, s1 = 0.0;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < M / 4; i += (size_t)gridDim.x * blockDim.x) {
        const float4 a = r0[i], b = r1[i];
        half2_t zq[4];
        hwords4(zq, z, pr, i, N);
        const half2_t h0 = zq[0], h1 = zq[1], h2 = zq[2], h3 = zq[3];
        s0 += ((double)a.x * (double)h0.x + (double)a.y * (double)h1.x) +
              ((double)a.z * (double)h2.x + (double)a.w * (double)h3.x);
        s1 += ((double)b.x * (double)h0.y + (double)b.y * (double)h1.y) +
              ((double)b.z * (double)h2.y + (double)b.w * (double)h3.y);
    }
    s0 = block_sum<256>(s0, sh);
    if (threadIdx.x == 0) partial[(2 * pr) * gridDim.x + blockIdx.x] = s0;
    s1 = block_sum<256>(s1, sh);
    if (threadIdx.x == 0) partial[(2 * pr + 1) * gridDim.x + blockIdx.x] = s1;
}

// k_pcg_update_px with z in packed FP16; set_p: p = z (start of the iteration, x untouched).
__global__ __launch_bounds__(256) void k_pcg_update_px_h(int R, size_t M, const double* __restrict__ sc,
                                                         const half2_t* __restrict__ z, float* __restrict__ p,
                                                         float* __restrict__ x, int do_p, int set_p) {
    const int pr = blockIdx.y;
    float a[2], b[2];
    bool upd[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int k = 2 * pr + h;
        a[h] = set_p ? 0.f : (float)sc[2 * R + k];
        b[h] = set_p ? 0.f : (float)sc[4 * R + k];
        upd[h] = set_p || (do_p && sc[5 * R + k] != 0.0);
    }
    const size_t N = M / 3;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < M / 4; i += (size_t)gridDim.x * blockDim.x) {
        half2_t zh[4];
        hwords4(zh, z, pr, i, N);
#pragma unroll
        for (int h = 0; h < 2; h++) {
            float4* p4 = reinterpret_cast<float4*>(p + (size_t)(2 * pr + h) * M);
            float4* x4 = reinterpret_cast<float4*>(x + (size_t)(2 * pr + h) * M);
            float4 pv = set_p ? make_float4(0.f, 0.f, 0.f, 0.f) : p4[i];
            if (a[h] != 0.f) {
                float4 xv = x4[i];
                xv.x = fmaf(a[h], pv.x, xv.x);
                xv.y = fmaf(a[h], pv.y, xv.y);
                xv.z = fmaf(a[h], pv.z, xv.z);
                xv.w = fmaf(a[h], pv.w, xv.w);
                x4[i] = xv;
            }
            if (upd[h]) {
                pv.x = fmaf(b[h], pv.x, (float)zh[0][h]);
                pv.y = fmaf(b[h], pv.y, (float)zh[1][h]);
                pv.z = fmaf(b[h], pv.z, (float)zh[2][h]);
                pv.w = fmaf(b[h], pv.w, (float)zh[3][h]);
                p4[i] = pv;
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Density utilities
// ---------------------------------------------------------------------------------------------

// OC update of one cell for multiplier g (update_kernel, OCOptimizer.cu:12-34), FP64 arithmetic rounded
// to FP32.
__device__ __forceinline__ float oc_cell(double r0, double sv, double g, double min_rho, double step, double damp) {
    double B = -sv / g;
    if (B < 0) B = 0.01;
    double xv = (damp == 0.5 ? sqrt(B) : pow(B, damp)) * r0;
    if (xv - r0 < -step) xv = r0 - step;
    if (xv - r0 > step) xv = r0 + step;
    if (xv < min_rho) xv = min_rho;
    if (xv > 1.0) xv = 1.0;
    return (float)xv;
}

// OC trial for multiplier g: per-block FP64 partial sums of the new density; the new density is written
// to out unless out is null (sum only).
__global__ __launch_bounds__(256) void k_oc_trial(int n, int pitch, double g, double min_rho, double step,
                                                  double damp, const float* __restrict__ sens,
                                                  const float* __restrict__ rho, float* __restrict__ out,
                                                  double* __restrict__ partial) {
    __shared__ double sh[4];
    const long N = (long)n * n * n;
    double s = 0.0;
    for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < N; e += (long)gridDim.x * blockDim.x) {
        const int x = (int)(e % n), y = (int)((e / n) % n), z = (int)(e / ((long)n * n));
        const size_t id = x + ((size_t)y + (size_t)z * n) * pitch;
        const float o = oc_cell(rho[id], sens[id], g, min_rho, step, damp);
        if (out) out[id] = o;
        s += (double)o;
    }
    s = block_sum<256>(s, sh);
    if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// The OC update for the final multiplier, in place (rho is read and written by the same thread).
__global__ __launch_bounds__(256) void k_oc_apply(int n, int pitch, double g, double min_rho, double step, double damp,
                                                  const float* __restrict__ sens, float* rho) {
    const long N = (long)n * n * n;
    for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < N; e += (long)gridDim.x * blockDim.x) {
        const int x = (int)(e % n), y = (int)((e / n) % n), z = (int)(e / ((long)n * n));
        const size_t id = x + ((size_t)y + (size_t)z * n) * pitch;
        rho[id] = oc_cell(rho[id], sens[id], g, min_rho, step, damp);
    }
}

// index of live cell e in a pitched lexicographic array
__device__ __forceinline__ size_t pitched(long e, int n, int pitch) {
    const int x = (int)(e % n), y = (int)((e / n) % n), z = (int)(e / ((long)n * n));
    return x + ((size_t)y + (size_t)z * n) * pitch;
}
__global__ __launch_bounds__(256) void k_field_sum(int n, int pitch, const float* __restrict__ a,
                                                   double* __restrict__ partial) {
    __shared__ double sh[4];
    const long N = (long)n * n * n;
    double s = 0.0;
    for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < N; e += (long)gridDim.x * blockDim.x)
        s += (double)a[pitched(e, n, pitch)];
    s = block_sum<256>(s, sh);
    if (threadIdx.x == 0) partial[blockIdx.x] = s;
}
__global__ __launch_bounds__(256) void k_field_fill(int n, int pitch, float value, float* __restrict__ a) {
    const long N = (long)n * n * n;
    for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < N; e += (long)gridDim.x * blockDim.x)
        a[pitched(e, n, pitch)] = value;
}

__global__ __launch_bounds__(256) void k_absmax(long N, int n, int pitch, const float* __restrict__ a,
                                                float* __restrict__ partial) {
    __shared__ float sh[256];
    float m = 0.f;
    for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < N; e += (long)gridDim.x * blockDim.x) {
        const int x = (int)(e % n), y = (int)((e / n) % n), z = (int)(e / ((long)n * n));
        m = fmaxf(m, fabsf(a[x + ((size_t)y + (size_t)z * n) * pitch]));
    }
    sh[threadIdx.x] = m;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) sh[threadIdx.x] = fmaxf(sh[threadIdx.x], sh[threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = sh[0];
}

// pitched lexicographic density -> dense cell weights w = emin + x
// pitched lexicographic density -> cell weights w = emin + x and raw x in level storage order
__global__ __launch_bounds__(256) void k_set_weights(Lay L, int pitch, double emin, const float* __restrict__ x,
                                                     float* __restrict__ w, float* __restrict__ xc) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t n = (uint32_t)L.n;
    if (i >= n * n * n) return;
    const int xx = (int)(i % n), y = (int)((i / n) % n), z = (int)(i / (n * n));
    const uint32_t e = L.idx(xx, y, z);
    const float xv = x[xx + ((size_t)y + (size_t)z * L.n) * pitch];
    xc[e] = xv;
    w[e] = (float)(emin + (double)xv);
}

__global__ __launch_bounds__(256) void k_copy_pitched(int n, int pitch_in, int pitch_out, const float* __restrict__ in,
                                                      float* __restrict__ out) {
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long N = (long)n * n * n;
    if (e >= N) return;
    const int x = (int)(e % n), y = (int)((e / n) % n), z = (int)(e / ((long)n * n));
    out[x + ((size_t)y + (size_t)z * n) * pitch_out] = in[x + ((size_t)y + (size_t)z * n) * pitch_in];
}


}  // namespace

// ---------------------------------------------------------------------------------------------
// Launch wrappers
// ---------------------------------------------------------------------------------------------
int ke_mfma_table(const double* kl, const double* km, double lam, double mu, void* table, float* c0, float* c1) {
    // One exact table T = r Kl + Km (KE = mu/72 T) when r = lambda / mu is a short binary fraction
    // (nu = 0.3 gives r = 3/2) and every entry of T is an FP16 value; else Kl and Km separately.
    std::vector<double> T(576);
    const double r = std::nearbyint(lam / mu * 256.0) / 256.0;
    bool one = std::fabs(r - lam / mu) <= 1e-12 * std::fabs(lam / mu);
    for (int e = 0; one && e < 576; e++) {
        T[e] = r * kl[e] + km[e];
        one = (double)(_Float16)T[e] == T[e];
    }
    // lane l of tile t holds row 16t + l % 16, K entries 8(l / 16) .. + 7.  Row 16t + 4g + j is slot
    // 4t + j of lane group g: one table: slots 0..5 its rows k = 0..5 of the group; two tables: slots
    // 0..5 the Kl rows, 6..11 the Km rows.  Row k of group g is component k % 3 of node
    // (k / 3, g & 1, g >> 1).  K entry 8g' + e (e < 6) is component e % 3 of node (e / 3, g' & 1, g' >> 1);
    // entries 6 and 7 are zero.
    _Float16* A = static_cast<_Float16*>(table);
    for (int t = 0; t < 3; t++)
        for (int l = 0; l < 64; l++) {
            const int m = l % 16, gp = l / 16, g = m / 4, slot = 4 * t + m % 4;
            const double* src = one ? (slot < 6 ? T.data() : nullptr) : (slot < 6 ? kl : km);
            const int k = slot % 6, o = k / 3 + 2 * (g & 1) + 4 * (g >> 1), i = k % 3;
            for (int e = 0; e < 8; e++) {
                const int op = e / 3 + 2 * (gp & 1) + 4 * (gp >> 1), ip = e % 3;
                A[(t * 64 + l) * 8 + e] = (_Float16)(src && e < 6 ? src[(3 * o + i) * 24 + 3 * op + ip] : 0.0);
            }
        }
    *c0 = (float)((one ? mu : lam) / 72.0);
    *c1 = one ? 0.f : (float)(mu / 72.0);
    return one ? 1 : 2;
}

void fine_block_consts(float* ke) {
    for (int t = 0; t < 243; t++) {
        const int d = t / 9, i = t / 3 % 3, j = t % 3;
        int e0 = 0, b0 = 0;
        for (int m = 0; m < 3; m++) {
            const int dm = (m == 0 ? d % 3 : (m == 1 ? d / 3 % 3 : d / 9)) - 1, em = dm > 0 ? 1 : 0;
            e0 |= em << m;
            b0 |= (dm + 1 - em) << m;
        }
        ke[kKeBlocks + 12 * d + 3 * i + j] = ke[(3 * (7 - e0) + i) * 24 + 3 * b0 + j];
    }
}

int fine_apply_mfma_ok(int n) { return n % 32 == 0 && 72.0 * n * n * n < 4294967296.0; }

static unsigned ef_grid(int n) {
    const unsigned h = (unsigned)n / 2;
    return (h / kEfTX) * (h / kEfTY) * (h / kEfTZ);
}

template <int MODE, bool DOT, bool BETA, int PX = 0>
static void fine_apply_ef(hipStream_t s, int n, const FineMfma* mf, const float* w, const void* u, const float* f,
                          float* out, double* partial, const float* dotv, const double* beta, float* pp = nullptr,
                          float* xx = nullptr, const double* alpha = nullptr) {
    const size_t N = (size_t)n * n * n;
    const Lay L = make_lay(n, 0);
    const half8_t* am = static_cast<const half8_t*>(mf->table);
    const uint32_t* uw = static_cast<const uint32_t*>(u);
    if (mf->nt == 1)
        hipLaunchKernelGGL((k_fine_apply_ef<MODE, DOT, BETA, 1, PX>), dim3(ef_grid(n)), dim3(kEfThreads), 0, s, L, N,
                           am, mf->c0, mf->c1, w, uw, f, out, partial, dotv, beta, pp, xx, alpha);
    else
        hipLaunchKernelGGL((k_fine_apply_ef<MODE, DOT, BETA, 2, PX>), dim3(ef_grid(n)), dim3(kEfThreads), 0, s, L, N,
                           am, mf->c0, mf->c1, w, uw, f, out, partial, dotv, beta, pp, xx, alpha);
}

void launch_fine_apply(hipStream_t s, int n, const float* ke, const FineMfma* mf, const float* w, const void* u,
                       int u_half, const float* f, float* out) {
    const size_t N = (size_t)n * n * n;
    const Lay L = make_lay(n, 0);
    const dim3 g(full_grid(L)), b(kFullThreads);
    if (u_half && mf && fine_apply_mfma_ok(n)) {
        if (f)
            fine_apply_ef<1, false, false>(s, n, mf, w, u, f, out, nullptr, nullptr, nullptr);
        else
            fine_apply_ef<0, false, false>(s, n, mf, w, u, f, out, nullptr, nullptr, nullptr);
        return;
    }
    if (u_half) {
        const half2_t* uh = static_cast<const half2_t*>(u);
        if (f)
            hipLaunchKernelGGL((k_fine_apply<6, 1, false, half2_t>), g, b, 0, s, L, N, ke, w, uh, f, out, nullptr,
                               nullptr, nullptr, nullptr, nullptr, nullptr);
        else
            hipLaunchKernelGGL((k_fine_apply<6, 0, false, half2_t>), g, b, 0, s, L, N, ke, w, uh, f, out, nullptr,
                               nullptr, nullptr, nullptr, nullptr, nullptr);
        return;
    }
    const float* uf = static_cast<const float*>(u);
    if (f && 64 % L.h == 0)
        hipLaunchKernelGGL((k_fine_apply<6, 1, false, float, false, 0, 1, true>), g, b, 0, s, L, N, ke, w, uf, f, out,
                           nullptr, nullptr, nullptr, nullptr, nullptr, nullptr);
    else if (f)
        hipLaunchKernelGGL((k_fine_apply<6, 1, false, float>), g, b, 0, s, L, N, ke, w, uf, f, out, nullptr, nullptr,
                           nullptr, nullptr, nullptr, nullptr);
    else
        hipLaunchKernelGGL((k_fine_apply<6, 0, false, float>), g, b, 0, s, L, N, ke, w, uf, f, out, nullptr, nullptr,
                           nullptr, nullptr, nullptr, nullptr);
}

// neighbours whose loads are in flight ahead of the CG pass's block products (FP32 z: one, as two
// spill there)
template <typename A>
constexpr int kCgPrefetch = CasesPerWord<A>::value == 2 ? 2 : 1;
template <typename A, bool FIRST>
static void fine_apply_cg_row(hipStream_t s, const Lay& L, size_t N, const float* ke, const float* w, const A* z,
                              float* p, float* x, const double* sc, float* q, double* partial) {
    constexpr int R = 6;
    hipLaunchKernelGGL((k_fine_apply<R, 0, true, A, !FIRST, FIRST ? 1 : 2, kCgPrefetch<A>>), dim3(full_grid(L)),
                       dim3(kFullThreads), 0, s, L, N, ke, w, z, nullptr, q, partial, nullptr, sc + 4 * R, p, x,
                       sc + 2 * R);
}

int fine_cg_staged_ok(int n) { return n % 128 == 0; }

void launch_fine_apply_cg(hipStream_t s, int n, const float* ke, const FineMfma* mf, const float* w, const void* z,
                          int z_half, int staged, float* p, float* x, double* sc, int first, float* q,
                          double* partial, int dot_blocks) {
    constexpr int R = 6;
    const size_t N = (size_t)n * n * n, M = 3 * N;
    const Lay L = make_lay(n, 0);
    unsigned nb = full_grid(L);
    if (z_half && mf && fine_apply_mfma_ok(n)) {
        if (first)
            fine_apply_ef<0, true, false, 1>(s, n, mf, w, z, nullptr, q, partial, nullptr, nullptr, p, x, nullptr);
        else
            fine_apply_ef<0, true, true, 2>(s, n, mf, w, z, nullptr, q, partial, nullptr, sc + 4 * R, p, x, sc + 2 * R);
        nb = ef_grid(n);
    } else if (L.h3 % 64) {
        // partial waves (FP32 z only: packed FP16 needs n % 8 == 0): the same step from separate passes
        if (first) {
            (void)launch_set_p(s, M, z, 0, p, dot_blocks);
        } else {
            launch_pcg_update_px(s, M, sc, z, 0, p, x, 1, dot_blocks);
        }
        launch_fine_apply(s, n, ke, nullptr, w, p, 0, nullptr, q);
        launch_dot6(s, M, p, q, partial, dot_blocks, sc + R, kSumPq, sc);
        return;
    } else if (z_half && staged && fine_cg_staged_ok(n)) {
        const uint32_t* zw = static_cast<const uint32_t*>(z);
        if (first)
            hipLaunchKernelGGL((k_fine_cg_staged<false, 1>), dim3(nb), dim3(kFullThreads), 0, s, L, N, ke, w, zw, q,
                               partial, nullptr, p, x, nullptr);
        else
            hipLaunchKernelGGL((k_fine_cg_staged<true, 2>), dim3(nb), dim3(kFullThreads), 0, s, L, N, ke, w, zw, q,
                               partial, sc + 4 * R, p, x, sc + 2 * R);
    } else if (z_half) {
        const half2_t* zh = static_cast<const half2_t*>(z);
        if (first)
            fine_apply_cg_row<half2_t, true>(s, L, N, ke, w, zh, p, x, sc, q, partial);
        else
            fine_apply_cg_row<half2_t, false>(s, L, N, ke, w, zh, p, x, sc, q, partial);
    } else {
        const float* zf = static_cast<const float*>(z);
        if (first)
            fine_apply_cg_row<float, true>(s, L, N, ke, w, zf, p, x, sc, q, partial);
        else
            fine_apply_cg_row<float, false>(s, L, N, ke, w, zf, p, x, sc, q, partial);
    }
    launch_sum_partials(s, R, (int)nb, partial, sc + R, kSumPq, sc);
}

// a multiple of 8, so that each XCD gets a contiguous run (workgroups past the last row do nothing)
int gs_pair_blocks(int n) {
    const int h = n / 2;
    return (int)((nblk((size_t)h * h, pair_rows(h)) + 7) / 8 * 8);
}

template <bool REV, int ZC, typename A, bool DOT = false, bool ROWN = false>
static void fine_gs2_pair(hipStream_t s, const Lay& L, size_t N, int cfirst, float omega, const float* ke,
                          const float* w, A* u, const float* f, double* partial = nullptr, int pstride = 0,
                          float* rown = nullptr) {
    if constexpr (CasesPerWord<A>::value == 1 && ZC < 0) {
        if (64 % L.h == 0) {
            hipLaunchKernelGGL((k_fine_gs2<6, REV, ZC, A, DOT, ROWN, true>), dim3(gs_pair_blocks(L.n)), dim3(256), 0, s, L, N,
                               cfirst, omega, ke, w, u, f, partial, pstride, rown);
            return;
        }
    }
    hipLaunchKernelGGL((k_fine_gs2<6, REV, ZC, A, DOT, ROWN>), dim3(gs_pair_blocks(L.n)), dim3(256), 0, s, L, N, cfirst, omega,
                       ke, w, u, f, partial, pstride, rown);
}

template <int ZC, typename A>
static void fine_gs2_zero(hipStream_t s, const Lay& L, size_t N, float omega, const float* ke, const float* w, A* u,
                          const float* f, float* rown) {
    if (rown)
        fine_gs2_pair<false, ZC, A, false, true>(s, L, N, ZC, omega, ke, w, u, f, nullptr, 0, rown);
    else
        fine_gs2_pair<false, ZC>(s, L, N, ZC, omega, ke, w, u, f);
}

template <typename A>
static void fine_gs2_pick(hipStream_t s, const Lay& L, size_t N, int cfirst, float omega, int reverse,
                          int zero_start, const float* ke, const float* w, A* u, const float* f, float* rown) {
    if (reverse) {
        fine_gs2_pair<true, -1>(s, L, N, cfirst, omega, ke, w, u, f);
        return;
    }
    switch (zero_start ? cfirst : -1) {
        case 0: fine_gs2_zero<0>(s, L, N, omega, ke, w, u, f, rown); break;
        case 2: fine_gs2_zero<2>(s, L, N, omega, ke, w, u, f, rown); break;
        case 4: fine_gs2_zero<4>(s, L, N, omega, ke, w, u, f, rown); break;
        case 6: fine_gs2_zero<6>(s, L, N, omega, ke, w, u, f, rown); break;
        default: fine_gs2_pair<false, -1>(s, L, N, cfirst, omega, ke, w, u, f); break;
    }
}

void launch_fine_gs2(hipStream_t s, int n, int cfirst, float omega, int reverse, int zero_start, const float* ke,
                     const float* w, void* u, int u_half, const float* f, double* partial, int pstride, float* rown) {
    const size_t N = (size_t)n * n * n;
    const Lay L = make_lay(n, 0);
    if (reverse || !zero_start) rown = nullptr;  // own-colour residuals only for zero-start passes
    if (partial && reverse && u_half) {  // f . u_new per workgroup (the r . z of a CG step)
        fine_gs2_pair<true, -1, half2_t, true>(s, L, N, cfirst, omega, ke, w, static_cast<half2_t*>(u), f, partial,
                                               pstride);
        return;
    }
    if (u_half)
        fine_gs2_pick(s, L, N, cfirst, omega, reverse, zero_start, ke, w, static_cast<half2_t*>(u), f, rown);
    else
        fine_gs2_pick(s, L, N, cfirst, omega, reverse, zero_start, ke, w, static_cast<float*>(u), f, rown);
}

void launch_fine_residual_later(hipStream_t s, int n, const float* ke, const float* w, const void* u, int u_half,
                                float* r) {
    const size_t N = (size_t)n * n * n;
    const Lay L = make_lay(n, 0);
    const dim3 g(nblk(L.h3, 64)), b(256);
    if (u_half)
        hipLaunchKernelGGL((k_fine_resid_later<6, half2_t>), g, b, 0, s, L, N, ke, w, static_cast<const half2_t*>(u),
                           r, 0.f);
    else
        hipLaunchKernelGGL((k_fine_resid_later<6, float>), g, b, 0, s, L, N, ke, w, static_cast<const float*>(u), r,
                           0.f);
}

void launch_macro_rhs(hipStream_t s, int n, const float* kchi, const float* w, float* f) {
    const size_t N = (size_t)n * n * n;
    const Lay L = make_lay(n, 0);
    hipLaunchKernelGGL(k_macro_rhs, dim3(full_grid(L)), dim3(kFullThreads), 0, s, L, N, kchi, w, f);
}

// One load case per FP64 residual launch: with two, the FP64 gather pipeline no longer fits the
// register file.
void launch_fine_residual64(hipStream_t s, int n, const double* ke, const double* kchi, const float* xc, double emin,
                            const double* u, float* r32, double* partial, double* out6, int do_k) {
    const size_t N = (size_t)n * n * n;
    const Lay L = make_lay(n, 0);
    const dim3 g(full_grid(L)), b(kFullThreads);
    if (!do_k)
        hipLaunchKernelGGL((k_fine_residual64<false>), g, b, 0, s, L, N, ke, kchi, xc, emin, u, r32, partial);
    else
        hipLaunchKernelGGL((k_fine_residual64<true>), g, b, 0, s, L, N, ke, kchi, xc, emin, u, r32, partial);
    launch_sum_partials(s, 6, (int)full_grid(L), partial, out6);
}

void launch_rhs_norm64(hipStream_t s, int n, const double* kchi, const float* xc, double emin, double* partial,
                       double* out6) {
    const size_t N = (size_t)n * n * n;
    const Lay L = make_lay(n, 0);
    const unsigned nb = full_grid(L);
    hipLaunchKernelGGL(k_rhs_norm64, dim3(nb), dim3(kFullThreads), 0, s, L, N, kchi, xc, emin, partial);
    launch_sum_partials(s, 6, (int)nb, partial, out6);
}

void launch_refine_accumulate(hipStream_t s, size_t N, const double* sc, int pending, const float* x, const float* p,
                              double* u, int add) {
    hipLaunchKernelGGL(k_refine_accumulate, dim3(2048, 9), dim3(256), 0, s, N, sc, pending, x, p, u, add);
}

void launch_round_f32(hipStream_t s, size_t N, const double* u, float* x) {
    hipLaunchKernelGGL(k_round_f32, dim3(nblk(9 * N)), dim3(256), 0, s, N, u, x);
}

void launch_widen_f64(hipStream_t s, size_t N, const float* x, double* u) {
    hipLaunchKernelGGL(k_widen_f64, dim3(nblk(9 * N)), dim3(256), 0, s, N, x, u);
}

void launch_pack_half(hipStream_t s, size_t N, const float* u, void* z) {
    hipLaunchKernelGGL(k_pack_half, dim3(nblk(9 * N)), dim3(256), 0, s, N, u, static_cast<half2_t*>(z));
}

void launch_unpack_half(hipStream_t s, size_t N, const void* z, float* u) {
    hipLaunchKernelGGL(k_unpack_half, dim3(nblk(9 * N)), dim3(256), 0, s, N, static_cast<const half2_t*>(z), u);
}

void launch_zero_pin(hipStream_t s, size_t N, void* u, int u_half) {
    if (u_half)
        hipLaunchKernelGGL((k_zero_pin<uint32_t, true>), dim3(1), dim3(64), 0, s, N, 9, static_cast<uint32_t*>(u));
    else
        hipLaunchKernelGGL((k_zero_pin<float>), dim3(1), dim3(64), 0, s, N, 18, static_cast<float*>(u));
}

void launch_zero_pin64(hipStream_t s, size_t N, double* u) {
    hipLaunchKernelGGL(k_zero_pin64, dim3(1), dim3(64), 0, s, N, u);
}

void launch_zero_case64(hipStream_t s, size_t N, int r, double* u) {
    hipLaunchKernelGGL(k_zero_case64, dim3(nblk(3 * N)), dim3(256), 0, s, N, r, u);
}

// Levels up to this size run the coarse-stencil kernels with one load case per thread (six grid
// rows): their stencils sit in cache, and the extra threads hide the gather latency that dominates
// there.  Larger levels keep all six load cases per thread so the stored stencil is read once.
constexpr int kSplitLoadCasesMaxN = 32;

template <int R, typename SA, typename A>
static void stencil_apply_case(hipStream_t s, const Lay& L, size_t N, const SA* st, const A* u, const float* f,
                               float* out) {
    const dim3 g(full_grid(L), 6 / R), b(kFullThreads);
    if (f)
        hipLaunchKernelGGL((k_stencil_apply<R, 1, SA, A>), g, b, 0, s, L, N, st, u, f, out);
    else
        hipLaunchKernelGGL((k_stencil_apply<R, 0, SA, A>), g, b, 0, s, L, N, st, u, f, out);
}

template <typename SA>
static void stencil_apply_pick(hipStream_t s, const Lay& L, size_t N, bool split, const SA* st, const void* u,
                               int u_half, const float* f, float* out) {
    if (u_half)
        stencil_apply_case<6>(s, L, N, st, static_cast<const half2_t*>(u), f, out);
    else if (split)
        stencil_apply_case<1>(s, L, N, st, static_cast<const float*>(u), f, out);
    else
        stencil_apply_case<6>(s, L, N, st, static_cast<const float*>(u), f, out);
}

int stencil_u_half_ok(int n, int lex) { return !lex && n > kSplitLoadCasesMaxN && n % 8 == 0; }

void launch_stencil_apply(hipStream_t s, int n, int lex, const void* st, int st_half, const void* u, int u_half,
                          const float* f, float* out) {
    const size_t N = (size_t)n * n * n;
    const Lay L = make_lay(n, lex);
    const bool split = n <= kSplitLoadCasesMaxN;
    if (u_half && !stencil_u_half_ok(n, lex)) return;  // the caller checks stencil_u_half_ok
    if (st_half)
        stencil_apply_pick(s, L, N, split, static_cast<const half2_t*>(st), u, u_half, f, out);
    else
        stencil_apply_pick(s, L, N, split, static_cast<const float*>(st), u, u_half, f, out);
}

template <bool REV, int ZC>
static void stencil_gs_colour(hipStream_t s, const Lay& L, size_t N, int colour, float omega, const float* st, float* u,
                              const float* f) {
    hipLaunchKernelGGL((k_stencil_gs<REV, ZC>), dim3(nblk(L.h3), 6), dim3(256), 0, s, L, N, colour, omega, st, u, f);
}

template <int R, bool REV, int ZC, typename SA, typename A, bool ROWN = false>
static void stencil_gs2_colour(hipStream_t s, const Lay& L, size_t N, int cfirst, float omega, const SA* st, A* u,
                               const float* f, float* rown = nullptr) {
    hipLaunchKernelGGL((k_stencil_gs2<R, REV, ZC, SA, A, ROWN>), dim3(gs_pair_blocks(L.n), 6 / R), dim3(256), 0, s, L, N, cfirst,
                       omega, st, u, f, rown);
}

template <int R, int ZC, typename SA, typename A>
static void stencil_gs2_zero(hipStream_t s, const Lay& L, size_t N, float omega, const SA* st, A* u, const float* f,
                             float* rown) {
    if (rown)
        stencil_gs2_colour<R, false, ZC, SA, A, true>(s, L, N, ZC, omega, st, u, f, rown);
    else
        stencil_gs2_colour<R, false, ZC>(s, L, N, ZC, omega, st, u, f);
}

template <int R, typename SA, typename A>
static void stencil_gs2_pick(hipStream_t s, const Lay& L, size_t N, int cfirst, float omega, int reverse,
                             int zero_start, const SA* st, A* u, const float* f, float* rown) {
    if (reverse) {
        stencil_gs2_colour<R, true, -1>(s, L, N, cfirst, omega, st, u, f);
        return;
    }
    switch (zero_start ? cfirst : -1) {
        case 0: stencil_gs2_zero<R, 0>(s, L, N, omega, st, u, f, rown); break;
        case 2: stencil_gs2_zero<R, 2>(s, L, N, omega, st, u, f, rown); break;
        case 4: stencil_gs2_zero<R, 4>(s, L, N, omega, st, u, f, rown); break;
        case 6: stencil_gs2_zero<R, 6>(s, L, N, omega, st, u, f, rown); break;
        default: stencil_gs2_colour<R, false, -1>(s, L, N, cfirst, omega, st, u, f); break;
    }
}

template <typename SA>
static void stencil_gs2_st(hipStream_t s, const Lay& L, size_t N, int cfirst, float omega, int reverse,
                           int zero_start, const SA* st, void* u, int u_half, const float* f, float* rown) {
    if (u_half)
        stencil_gs2_pick<6>(s, L, N, cfirst, omega, reverse, zero_start, st, static_cast<half2_t*>(u), f, rown);
    else
        stencil_gs2_pick<6>(s, L, N, cfirst, omega, reverse, zero_start, st, static_cast<float*>(u), f, rown);
}

// pairs only where a launch runs six load cases per thread: on the one-case levels (<= 32^3) the
// launch is latency-bound and two colours in one cost more than two launches (14 vs 11 us at 32^3)
int stencil_gs_pairs_ok(int n, int lex) { return !lex && n > kSplitLoadCasesMaxN; }

void launch_stencil_gs2(hipStream_t s, int n, int cfirst, float omega, int reverse, int zero_start, const void* st,
                        int st_half, void* u, int u_half, const float* f, float* rown) {
    const size_t N = (size_t)n * n * n;
    const Lay L = make_lay(n, 0);
    if (!stencil_gs_pairs_ok(n, 0)) return;            // the caller checks stencil_gs_pairs_ok
    if (u_half && !stencil_u_half_ok(n, 0)) return;    // ... and stencil_u_half_ok
    if (reverse || !zero_start) rown = nullptr;        // own-colour residuals only for zero-start passes
    if (st_half)
        stencil_gs2_st(s, L, N, cfirst, omega, reverse, zero_start, static_cast<const half2_t*>(st), u, u_half,
                       f, rown);
    else
        stencil_gs2_st(s, L, N, cfirst, omega, reverse, zero_start, static_cast<const float*>(st), u, u_half, f,
                       rown);
}

template <int R, typename SA, typename A>
static void stencil_resid_later(hipStream_t s, const Lay& L, size_t N, const SA* st, const A* u, float* r) {
    hipLaunchKernelGGL((k_stencil_resid_later<R, SA, A>), dim3(nblk(L.h3, 64), 6 / R), dim3(256), 0, s, L, N, st, u,
                       r, 0.f);
}

template <typename SA>
static void stencil_resid_later_st(hipStream_t s, const Lay& L, size_t N, const SA* st, const void* u, int u_half,
                                   float* r) {
    if (u_half)
        stencil_resid_later<6>(s, L, N, st, static_cast<const half2_t*>(u), r);
    else
        stencil_resid_later<6>(s, L, N, st, static_cast<const float*>(u), r);
}

void launch_stencil_residual_later(hipStream_t s, int n, const void* st, int st_half, const void* u, int u_half,
                                   float* r) {
    const size_t N = (size_t)n * n * n;
    const Lay L = make_lay(n, 0);
    if (!stencil_gs_pairs_ok(n, 0)) return;          // the caller checks stencil_gs_pairs_ok
    if (u_half && !stencil_u_half_ok(n, 0)) return;  // ... and stencil_u_half_ok
    if (st_half)
        stencil_resid_later_st(s, L, N, static_cast<const half2_t*>(st), u, u_half, r);
    else
        stencil_resid_later_st(s, L, N, static_cast<const float*>(st), u, u_half, r);
}

void launch_stencil_gs(hipStream_t s, int n, int colour, float omega, int reverse, int zero_start, const float* st,
                       float* u, const float* f) {
    const size_t N = (size_t)n * n * n;
    const Lay L = make_lay(n, 0);
    if (reverse) {
        stencil_gs_colour<true, -1>(s, L, N, colour, omega, st, u, f);
        return;
    }
    switch (zero_start ? colour : -1) {
        case 0: stencil_gs_colour<false, 0>(s, L, N, colour, omega, st, u, f); break;
        case 1: stencil_gs_colour<false, 1>(s, L, N, colour, omega, st, u, f); break;
        case 2: stencil_gs_colour<false, 2>(s, L, N, colour, omega, st, u, f); break;
        case 3: stencil_gs_colour<false, 3>(s, L, N, colour, omega, st, u, f); break;
        case 4: stencil_gs_colour<false, 4>(s, L, N, colour, omega, st, u, f); break;
        case 5: stencil_gs_colour<false, 5>(s, L, N, colour, omega, st, u, f); break;
        case 6: stencil_gs_colour<false, 6>(s, L, N, colour, omega, st, u, f); break;
        case 7: stencil_gs_colour<false, 7>(s, L, N, colour, omega, st, u, f); break;
        default: stencil_gs_colour<false, -1>(s, L, N, colour, omega, st, u, f); break;
    }
}

// Transfers take one load case per thread (six grid rows): the load cases' planes are disjoint, so
// this costs no extra traffic and shortens each thread's chain of dependent loads.
void launch_restrict(hipStream_t s, int nf, int lexc, const float* rf, float* fc) {
    const size_t Nc = (size_t)(nf / 2) * (nf / 2) * (nf / 2);
    const Lay Lf = make_lay(nf, 0), Lc = make_lay(nf / 2, lexc);
    if (nf % 8 == 0)
        hipLaunchKernelGGL(k_restrict4, dim3(nblk(Nc / 4), 6), dim3(256), 0, s, Lf, Lc, rf, fc);
    else
        hipLaunchKernelGGL((k_restrict<1>), dim3(nblk(Nc), 6), dim3(256), 0, s, Lf, Lc, rf, fc);
}

void launch_prolong(hipStream_t s, int nf, int lexc, const void* uc, int uc_half, void* uf, int u_half, int pin) {
    const Lay Lf = make_lay(nf, 0), Lc = make_lay(nf / 2, lexc);
    if (uc_half && (!u_half || lexc)) return;  // packed FP16 coarse u: parity-blocked, into a packed FP16 fine u
    if (u_half && uc_half)
        hipLaunchKernelGGL((k_prolong_h<half2_t>), dim3(full_grid(Lf)), dim3(kFullThreads), 0, s, Lf, Lc,
                           static_cast<const half2_t*>(uc), static_cast<half2_t*>(uf), pin);
    else if (u_half)  // packed FP16 fine fields are only used with nf % 8 == 0
        hipLaunchKernelGGL((k_prolong_h<float>), dim3(full_grid(Lf)), dim3(kFullThreads), 0, s, Lf, Lc,
                           static_cast<const float*>(uc), static_cast<half2_t*>(uf), pin);
    else if (nf % 8 == 0)
        hipLaunchKernelGGL(k_prolong4, dim3(nblk(Lf.h3 / 4, 64), 6), dim3(kFullThreads), 0, s, Lf, Lc,
                           static_cast<const float*>(uc), static_cast<float*>(uf), pin);
    else
        hipLaunchKernelGGL((k_prolong<1>), dim3(full_grid(Lf), 6), dim3(kFullThreads), 0, s, Lf, Lc,
                           static_cast<const float*>(uc), static_cast<float*>(uf), pin);
}

void launch_dot6(hipStream_t s, size_t M, const float* a, const float* b, double* partial, int nblocks,
                 double* out, int then, double* sc) {
    hipLaunchKernelGGL(k_dot, dim3(nblocks, 6), dim3(256), 0, s, M, a, b, partial);
    launch_sum_partials(s, 6, nblocks, partial, out, then, sc);
}

void launch_sum_partials(hipStream_t s, int R, int nblocks, const double* partial, double* out, int then, double* sc) {
    if (then == kSumPq)
        hipLaunchKernelGGL(k_sum_partials<kSumPq>, dim3(R), dim3(kSumThreads), 0, s, nblocks, partial, out, sc);
    else if (then == kSumRz)
        hipLaunchKernelGGL(k_sum_partials<kSumRz>, dim3(R), dim3(kSumThreads), 0, s, nblocks, partial, out, sc);
    else
        hipLaunchKernelGGL(k_sum_partials<kSumOnly>, dim3(R), dim3(kSumThreads), 0, s, nblocks, partial, out, nullptr);
}


void launch_pcg_update_r(hipStream_t s, size_t M, const double* sc, const float* q, float* r, double* partial,
                         int nblocks, double* out6) {
    hipLaunchKernelGGL(k_pcg_update_r, dim3(nblocks, 6), dim3(256), 0, s, 6, M, sc, q, r, partial);
    launch_sum_partials(s, 6, nblocks, partial, out6);
}

void launch_pcg_update_px(hipStream_t s, size_t M, const double* sc, const void* z, int z_half, float* p, float* x,
                          int do_p, int nblocks) {
    if (z_half)
        hipLaunchKernelGGL(k_pcg_update_px_h, dim3(nblocks, 3), dim3(256), 0, s, 6, M, sc,
                           static_cast<const half2_t*>(z), p, x, do_p, 0);
    else
        hipLaunchKernelGGL(k_pcg_update_px, dim3(nblocks, 6), dim3(256), 0, s, 6, M, sc, static_cast<const float*>(z),
                           p, x, do_p);
}

hipError_t launch_set_p(hipStream_t s, size_t M, const void* z, int z_half, float* p, int nblocks) {
    if (!z_half) return hipMemcpyAsync(p, z, sizeof(float) * 6 * M, hipMemcpyDeviceToDevice, s);
    hipLaunchKernelGGL(k_pcg_update_px_h, dim3(nblocks, 3), dim3(256), 0, s, 6, M, nullptr,
                       static_cast<const half2_t*>(z), p, nullptr, 0, 1);
    return hipGetLastError();
}

void launch_dot_rz(hipStream_t s, size_t M, const float* r, const void* z, int z_half, double* partial, int nblocks,
                   double* out6, int then, double* sc) {
    if (!z_half) {
        launch_dot6(s, M, r, static_cast<const float*>(z), partial, nblocks, out6, then, sc);
        return;
    }
    hipLaunchKernelGGL(k_dot_fh, dim3(nblocks, 3), dim3(256), 0, s, M, r, static_cast<const half2_t*>(z), partial);
    launch_sum_partials(s, 6, nblocks, partial, out6, then, sc);
}

void launch_oc_trial(hipStream_t s, int n, int pitch, double g, double min_rho, double step, double damp,
                     const float* sens, const float* rho, float* out, double* partial, int nblocks, double* sum) {
    hipLaunchKernelGGL(k_oc_trial, dim3(nblocks), dim3(256), 0, s, n, pitch, g, min_rho, step, damp, sens, rho, out,
                       partial);
    launch_sum_partials(s, 1, nblocks, partial, sum);
}

void launch_field_sum(hipStream_t s, int n, int pitch, const float* a, double* partial, int nblocks) {
    hipLaunchKernelGGL(k_field_sum, dim3(nblocks), dim3(256), 0, s, n, pitch, a, partial);
}
void launch_field_fill(hipStream_t s, int n, int pitch, float value, float* a) {
    hipLaunchKernelGGL(k_field_fill, dim3(1024), dim3(256), 0, s, n, pitch, value, a);
}

void launch_absmax(hipStream_t s, int n, int pitch, const float* a, float* partial, int nblocks) {
    const long N = (long)n * n * n;
    hipLaunchKernelGGL(k_absmax, dim3(nblocks), dim3(256), 0, s, N, n, pitch, a, partial);
}

void launch_set_weights(hipStream_t s, int n, int pitch, double emin, const float* x, float* w, float* xc) {
    const size_t N = (size_t)n * n * n;
    hipLaunchKernelGGL(k_set_weights, dim3(nblk(N)), dim3(256), 0, s, make_lay(n, 0), pitch, emin, x, w, xc);
}

// ---------------------------------------------------------------------------------------------
// Bridges between the solver's fields and the learned warm-start network (net.hip): the network runs
// on a g^3 grid (g | n) with bf16 channels-last tensors.
// ---------------------------------------------------------------------------------------------
namespace {

// Network input: channel 0 of cell (i, j, k) = mean of rho = x^(1/3) over the f^3 fine cells it covers
// (f = n / g), channels 1..7 = 0.  x holds the raw x = rho^3 per cell in level storage order.
__global__ __launch_bounds__(256) void k_net_input(Lay L, int g, const float* __restrict__ x, uint16_t* __restrict__ in) {
    const long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long g3 = (long)g * g * g;
    if (v >= g3) return;
    const int f = L.n / g;
    const int i = (int)(v % g), j = (int)((v / g) % g), k = (int)(v / ((long)g * g));
    float s = 0.f;
    for (int c = 0; c < f * f * f; c++) {
        const int xx = i * f + c % f, yy = j * f + (c / f) % f, zz = k * f + c / (f * f);
        s += cbrtf(fmaxf(x[L.idx(xx, yy, zz)], 0.f));
    }
    *reinterpret_cast<uint4*>(in + v * 8) = make_uint4(f2bf(s / (float)(f * f * f)), 0u, 0u, 0u);
}

// Per-channel mean of the solution sampled at the coarse vertices (i f, j f, k f), weighted by the
// stiffness rho^3 of the network input at the same index (the network's loss weights).
__global__ __launch_bounds__(256) void k_net_target_mean(Lay L, int g, const double* __restrict__ u,
                                                         const uint16_t* __restrict__ in, double* __restrict__ mean) {
    __shared__ double sh[2][256];
    const int c = blockIdx.x;
    const long g3 = (long)g * g * g;
    const size_t N = (size_t)L.n * L.n * L.n;
    const int f = L.n / g;
    double s = 0.0, ws = 0.0;
    for (long v = threadIdx.x; v < g3; v += blockDim.x) {
        const int i = (int)(v % g), j = (int)((v / g) % g), k = (int)(v / ((long)g * g));
        const double r = bf2f(in[v * 8]);
        s += r * r * r * u[u64_index(c, L.idx(i * f, j * f, k * f), N)];
        ws += r * r * r;
    }
    sh[0][threadIdx.x] = s;
    sh[1][threadIdx.x] = ws;
    __syncthreads();
    for (int t = 128; t > 0; t >>= 1) {
        if ((int)threadIdx.x < t) {
            sh[0][threadIdx.x] += sh[0][threadIdx.x + t];
            sh[1][threadIdx.x] += sh[1][threadIdx.x + t];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) mean[c] = sh[1][0] > 0 ? sh[0][0] / sh[1][0] : 0.0;
}

// Network target: channel 3 s + k of coarse vertex v = scale (u_sk(i f, j f, k f) - mean) / n.
__global__ __launch_bounds__(256) void k_net_target(Lay L, int g, const double* __restrict__ u,
                                                    const double* __restrict__ mean, double scale,
                                                    uint16_t* __restrict__ tg) {
    const long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long g3 = (long)g * g * g;
    if (v >= g3) return;
    const size_t N = (size_t)L.n * L.n * L.n;
    const int f = L.n / g;
    const int i = (int)(v % g), j = (int)((v / g) % g), k = (int)(v / ((long)g * g));
    const uint32_t e = L.idx(i * f, j * f, k * f);
    const double sc = scale / (double)L.n;
    for (int c = 0; c < 18; c++) tg[v * 18 + c] = f2bf((float)(sc * (u[u64_index(c, e, N)] - mean[c])));
}

// Warm start from the prediction P ([g^3][ldp], channel 3 s + k = scale u_sk / n): periodic trilinear
// interpolation to the n^3 vertices, minus the value at vertex 0 (the pinned vertex keeps u = 0),
// times n / scale, into the FP64 iterate U64 and its FP32 copy X (level storage order).
__global__ __launch_bounds__(256) void k_net_warm_start(Lay L, int g, const float* __restrict__ P, int ldp, double inv,
                                                        double* __restrict__ U64, float* __restrict__ X) {
    const size_t N = (size_t)L.n * L.n * L.n;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= N) return;
    int x, y, z;
    L.pos((uint32_t)t, x, y, z);
    const int f = L.n / g;
    const int i0 = x / f, j0 = y / f, k0 = z / f;
    const float tx = (float)(x - i0 * f) / f, ty = (float)(y - j0 * f) / f, tz = (float)(z - k0 * f) / f;
    long cv[8];
    float wt[8];
    for (int c = 0; c < 8; c++) {
        const int i = (i0 + (c & 1)) % g, j = (j0 + ((c >> 1) & 1)) % g, k = (k0 + (c >> 2)) % g;
        cv[c] = i + (long)g * (j + (long)g * k);
        wt[c] = ((c & 1) ? tx : 1.f - tx) * (((c >> 1) & 1) ? ty : 1.f - ty) * ((c >> 2) ? tz : 1.f - tz);
    }
    for (int ch = 0; ch < 18; ch++) {
        float s = 0.f;
        for (int c = 0; c < 8; c++) s += wt[c] * P[cv[c] * ldp + ch];
        const double u = ((double)s - (double)P[ch]) * inv;
        U64[u64_index(ch, t, N)] = u;
        X[ch * N + t] = (float)u;
    }
}

}  // namespace

void launch_net_input(hipStream_t s, int n, int g, const float* x, uint16_t* in) {
    const long g3 = (long)g * g * g;
    hipLaunchKernelGGL(k_net_input, dim3(nblk(g3)), dim3(256), 0, s, make_lay(n, 0), g, x, in);
}

void launch_net_target(hipStream_t s, int n, int g, const double* u64, const uint16_t* in, double scale, double* mean18,
                       uint16_t* tg) {
    const long g3 = (long)g * g * g;
    hipLaunchKernelGGL(k_net_target_mean, dim3(18), dim3(256), 0, s, make_lay(n, 0), g, u64, in, mean18);
    hipLaunchKernelGGL(k_net_target, dim3(nblk(g3)), dim3(256), 0, s, make_lay(n, 0), g, u64, mean18, scale, tg);
}

void launch_net_warm_start(hipStream_t s, int n, int g, const float* P, int ldp, double scale, double* u64, float* x) {
    const size_t N = (size_t)n * n * n;
    hipLaunchKernelGGL(k_net_warm_start, dim3(nblk(N)), dim3(256), 0, s, make_lay(n, 0), g, P, ldp, (double)n / scale,
                       u64, x);
}

void launch_copy_pitched(hipStream_t s, int n, int pitch_in, int pitch_out, const float* in, float* out) {
    const size_t N = (size_t)n * n * n;
    hipLaunchKernelGGL(k_copy_pitched, dim3(nblk(N)), dim3(256), 0, s, n, pitch_in, pitch_out, in, out);
}

}  // namespace homo3d

// =============================================================================================
// OC update without allocation: homo3d_oc_update_noalloc
// =============================================================================================
// The bisection's reduction scratch (|s| maxima of kOcBlocks workgroups, kOcBlocks FP64 partial volume
// sums and their total) lives in this file-scope device array: every GPU the library runs on holds one
// copy until the process ends.  Its device address is looked up once per device and used for every
// launch; every launch rewrites what it reads, so nothing needs clearing between calls.  Calls that
// overlap on one GPU share the array and race.
namespace {
constexpr int kOcBlocks = 1024;
constexpr int kOcMaxReso = 1024;  // largest grid accepted (as the density-only handle)
constexpr int kOcScratchDoubles = kOcBlocks + kOcBlocks / 2 + 8;  // partials, float maxima, total
constexpr int kOcMaxDevices = 64;
static __device__ __align__(256) double scratch[kOcScratchDoubles];
double* g_scratch[kOcMaxDevices] = {};
std::mutex g_scratch_mu;

int scratch_ptr(double** out) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kOcMaxDevices) return HOMO3D_HIP_ERROR;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return HOMO3D_HIP_ERROR;
        g_scratch[dev] = static_cast<double*>(p);
    }
    *out = g_scratch[dev];
    return HOMO3D_OK;
}
}  // namespace

extern "C" int homo3d_oc_update_noalloc(const float* sens, float* rho, int n, int pitch, double vol, double min_rho,
                                        double step, double damp, void* stream) {
    using namespace homo3d;
    if (!sens || !rho || n < 1 || pitch < n) return HOMO3D_BAD_ARG;
    if (n > kOcMaxReso) return HOMO3D_BAD_ARG;  // beyond the stated maximum grid
    double* sc = nullptr;
    int rc = scratch_ptr(&sc);
    if (rc) return rc;
    hipStream_t s = static_cast<hipStream_t>(stream);
    double* partial = sc;
    float* pmax = reinterpret_cast<float*>(sc + kOcBlocks);
    double* total = sc + kOcBlocks + kOcBlocks / 2;
    const long N = (long)n * n * n;
    hipLaunchKernelGGL(k_absmax, dim3(kOcBlocks), dim3(256), 0, s, N, n, pitch, sens, pmax);
    std::vector<float> pm(kOcBlocks);
    if (hipMemcpyAsync(pm.data(), pmax, sizeof(float) * kOcBlocks, hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return HOMO3D_HIP_ERROR;
    double hi = 0, lo = 0, g = 0;
    for (float v : pm) hi = std::max(hi, (double)v);
    const double Ne = (double)N;
    // the same bisection as homo3d_oc_update (OCOptimizer.cu:218-247): the trials only sum, and the
    // last trial's multiplier is applied in place at the end
    for (int it = 0; it < 20; it++) {
        g = (hi + lo) / 2;
        double sum = 0;
        hipLaunchKernelGGL(k_oc_trial, dim3(kOcBlocks), dim3(256), 0, s, n, pitch, g, min_rho, step, damp, sens,
                           (const float*)rho, (float*)nullptr, partial);
        launch_sum_partials(s, 1, kOcBlocks, (const double*)partial, total);
        if (hipMemcpyAsync(&sum, total, sizeof(double), hipMemcpyDeviceToHost, s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess)
            return HOMO3D_HIP_ERROR;
        const double cur = sum / Ne;
        if (cur < vol - 1e-4)
            hi = g;
        else if (cur > vol + 1e-4)
            lo = g;
        else
            break;
    }
    hipLaunchKernelGGL(k_oc_apply, dim3(kOcBlocks), dim3(256), 0, s, n, pitch, g, min_rho, step, damp, sens, rho);
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s) != hipSuccess) return HOMO3D_HIP_ERROR;
    return HOMO3D_OK;
}
