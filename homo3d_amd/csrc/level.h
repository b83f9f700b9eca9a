// Device helpers shared by the kernels that work on a grid level: storage order, workgroup order, buffer
// loads and workgroup sums.  Included inside each kernel file; everything has internal linkage.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace homo3d {
namespace {

__device__ __forceinline__ int wrap_dec(int a, int n) { return a == 0 ? n - 1 : a - 1; }
__device__ __forceinline__ int wrap_inc(int a, int n) { return a == n - 1 ? 0 : a + 1; }

// Storage order of a level's vertices (and of the cells, which share the vertex index).  Even levels
// are parity-blocked: the 8 coordinate-parity classes are contiguous (n/2)^3 blocks, block
// b = (x&1) | (y&1)<<1 | (z&1)<<2, and inside a block (x>>1) + h((y>>1) + h(z>>1)).  A GS colour is
// one block, so colour passes read their own vertices and every neighbour class contiguously.
// The coarsest level (possibly odd) is lexicographic.  Vertex (0,0,0) has index 0 in both orders.
struct Lay {
    int n;        // points per axis
    int h;        // n / 2
    uint32_t h3;  // h^3
    int lex;      // 1: x + n(y + n z)
    // index contribution of (already wrapped) coordinate a on axis k
    __device__ __forceinline__ uint32_t part(int a, int k) const {
        if (lex) return k == 0 ? (uint32_t)a : (k == 1 ? (uint32_t)a * n : (uint32_t)a * n * n);
        const uint32_t stride = k == 0 ? 1u : (k == 1 ? (uint32_t)h : (uint32_t)h * h);
        return ((uint32_t)(a & 1) << k) * h3 + (uint32_t)(a >> 1) * stride;
    }
    __device__ __forceinline__ uint32_t idx(int x, int y, int z) const { return part(x, 0) + part(y, 1) + part(z, 2); }
    __device__ __forceinline__ void pos(uint32_t t, int& x, int& y, int& z) const {
        if (lex) {
            x = (int)(t % n);
            y = (int)((t / n) % n);
            z = (int)(t / ((uint32_t)n * n));
            return;
        }
        const uint32_t b = t / h3, l = t - b * h3;
        x = 2 * (int)(l % h) + (int)(b & 1);
        y = 2 * (int)((l / h) % h) + (int)((b >> 1) & 1);
        z = 2 * (int)(l / ((uint32_t)h * h)) + (int)(b >> 2);
    }
    __device__ __forceinline__ int wrap(int a) const { return a < 0 ? a + n : (a >= n ? a - n : a); }
};

// Workgroup id -> work chunk.  The hardware deals workgroup g to XCD g % 8; this gives each XCD a
// contiguous run of chunks, so the neighbour rows that adjacent chunks share stay in one L2.
__device__ __forceinline__ uint32_t xcd_chunk(uint32_t g, uint32_t G) {
    if (G & 7u) return g;
    return (g & 7u) * (G >> 3) + (g >> 3);
}

// Rows of n/2 = h vertices that a workgroup of a fused colour pair takes: as many as 256 threads hold.
__host__ __device__ inline int pair_rows(int h) { return h < 256 ? 256 / h : 1; }

// Full-level kernels run 512-thread workgroups.  On a parity-blocked level the 8 waves of a
// workgroup take the same 64 local positions in the 8 parity blocks, so a workgroup covers a
// 128 x 2 x 2 vertex tile and the neighbour reads of its waves overlap in L1/L2; on a
// lexicographic level the 512 threads take consecutive vertices.  False past the end of the level.
constexpr int kFullThreads = 512;
__device__ __forceinline__ bool full_vertex(const Lay& L, uint32_t chunk, uint32_t& v) {
    if (L.lex) {
        v = chunk * (uint32_t)kFullThreads + threadIdx.x;
        return v < (uint32_t)L.n * L.n * L.n;
    }
    const uint32_t t = chunk * 64u + (threadIdx.x & 63u);
    v = (threadIdx.x >> 6) * L.h3 + t;
    return t < L.h3;
}

// Buffer-resource loads: one SGPR descriptor per array, a 32-bit VGPR byte offset per element and an
// SGPR byte offset per (load case, component) plane.  Offsets past the array read as zero.
typedef __amdgpu_buffer_rsrc_t Rsrc;
__device__ __forceinline__ Rsrc make_rsrc(const void* p, size_t bytes) {
    const uint32_t nrec = bytes > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)bytes;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)nrec, 0x00020000);
}
template <typename T>
__device__ __forceinline__ T bload(Rsrc r, uint32_t voff, uint32_t soff);
template <>
__device__ __forceinline__ float bload<float>(Rsrc r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)voff, (int)soff, 0));
}

// Packed FP16 storage of a 6-load-case field: word plane (p * 3 + i) holds components i of load cases
// 2p (.x) and 2p + 1 (.y), so a neighbour of all six load cases is 9 32-bit words.
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
template <>
__device__ __forceinline__ half2_t bload<half2_t>(Rsrc r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(half2_t, __builtin_amdgcn_raw_buffer_load_b32(r, (int)voff, (int)soff, 0));
}

// load cases per stored word of a field type
template <typename A>
struct CasesPerWord {
    static constexpr int value = 1;
};
template <>
struct CasesPerWord<half2_t> {
    static constexpr int value = 2;
};

// Packed FP16 six-load-case fields (half2_t words): word q = p * 3 + i of vertex v (component i of load
// cases 2p (.x) and 2p + 1 (.y)) is word hw_index(q, v, N) of the field.  Words 0-3 and 4-7 form two
// planes of 16-byte quads and word 8 a plane of single words, so the nine words of a vertex are two
// 16-byte loads and one 4-byte load: a 27-neighbour gather costs the texture addresser per load
// instruction, not per byte (nine 4-byte loads per neighbour take about four times as long).
__host__ __device__ __forceinline__ size_t hw_index(int q, size_t v, size_t N) {
    return q < 8 ? (size_t)(q >> 2) * 4 * N + 4 * v + (size_t)(q & 3) : 8 * N + v;
}
// word q of vertex v in a field of A words: packed FP16 as above, FP32 planes q * N + v
template <typename A>
__device__ __forceinline__ size_t fw_index(int q, size_t v, size_t N) {
    if constexpr (CasesPerWord<A>::value == 2)
        return hw_index(q, v, N);
    else
        return (size_t)q * N + v;
}

// A stored coarse stencil: FP32 entries [243][N] (entry e = 9d + 3i + j), or packed FP16 [31][N] quads of
// four words, quad q holding the entries 8q .. 8q + 7 (so that one load brings 16 bytes).  words: 4-byte
// words a vertex; vo: 4 times the vertex, plane: 4 N.
template <typename SA>
struct StencilIO;
template <>
struct StencilIO<float> {
    static constexpr int words = 243;
    __device__ static float get(Rsrc rs, uint32_t vo, uint32_t plane, int e) {
        return bload<float>(rs, vo, (uint32_t)e * plane);
    }
    // entries e .. e + 2 (e the same in every lane)
    __device__ static void get3(Rsrc rs, uint32_t vo, uint32_t plane, int e, float (&out)[3]) {
#pragma unroll
        for (int j = 0; j < 3; j++) out[j] = get(rs, vo, plane, e + j);
    }
    __device__ static void put(float* st, size_t N, uint32_t v, int e, float val) { st[(size_t)e * N + v] = val; }
};
template <>
struct StencilIO<half2_t> {
    static constexpr int words = 124;
    __device__ static float get(Rsrc rs, uint32_t vo, uint32_t plane, int e) {
        return (float)bload<half2_t>(rs, 4u * vo + 4u * (uint32_t)(e >> 1 & 3), (uint32_t)(e >> 3) * 4u * plane)[e & 1];
    }
    __device__ static void get3(Rsrc rs, uint32_t vo, uint32_t plane, int e, float (&out)[3]) {
        const uint32_t w0 = (uint32_t)e >> 1, w1 = w0 + 1, odd = 16u * (uint32_t)(e & 1);
        const auto word = [&](uint32_t w) {
            return __builtin_bit_cast(uint32_t, bload<half2_t>(rs, 4u * vo, (w >> 2) * 4u * plane + 4u * (w & 3u)));
        };
        const uint32_t a = word(w0), b = word(w1);
        const half2_t lo = __builtin_bit_cast(half2_t, __builtin_amdgcn_alignbit(b, a, odd));
        out[0] = (float)lo[0];
        out[1] = (float)lo[1];
        out[2] = (float)__builtin_bit_cast(half2_t, b >> odd)[0];
    }
    // one 16-bit store per entry: the halves of a word may come from different threads
    __device__ static void put(half2_t* st, size_t N, uint32_t v, int e, float val) {
        reinterpret_cast<_Float16*>(st)[((size_t)(e >> 3) * N + v) * 8 + (size_t)(e & 7)] = (_Float16)val;
    }
};

// Coarse-vertex kernels that read the fine level around 2V take coarse vertices in lexicographic
// order whatever the coarse storage, so that consecutive lanes read consecutive fine local positions.
__device__ __forceinline__ bool coarse_lex_vertex(const Lay& Lc, int& X, int& Y, int& Z, uint32_t& V) {
    const uint32_t i = xcd_chunk(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    const uint32_t n = (uint32_t)Lc.n;
    if (i >= n * n * n) return false;
    X = (int)(i % n);
    Y = (int)((i / n) % n);
    Z = (int)(i / (n * n));
    V = Lc.idx(X, Y, Z);
    return true;
}

// weight of fine offset o in the 1-D prolongation
__device__ __forceinline__ float hat(int o) { return o == 0 ? 1.f : ((o == 1 || o == -1) ? 0.5f : 0.f); }

// Block Gauss-Seidel / SOR update of one vertex: x, y, z in turn (z, y, x when REVERSE)
// (gs_relaxation_otf_kernel update formula, grid.cu:530-541).
// inv holds 1 / Ks[0], 1 / Ks[4], 1 / Ks[8] (shared by all load cases of the vertex).
template <bool REVERSE>
__device__ __forceinline__ void block_update(float u[3], const float f[3], const float KeU[3], const float Ks[9],
                                             const float inv[3], float omega) {
    if (!REVERSE) {
        u[0] = omega * (f[0] - KeU[0] - Ks[1] * u[1] - Ks[2] * u[2]) * inv[0] + (1.f - omega) * u[0];
        u[1] = omega * (f[1] - KeU[1] - Ks[3] * u[0] - Ks[5] * u[2]) * inv[1] + (1.f - omega) * u[1];
        u[2] = omega * (f[2] - KeU[2] - Ks[6] * u[0] - Ks[7] * u[1]) * inv[2] + (1.f - omega) * u[2];
    } else {
        u[2] = omega * (f[2] - KeU[2] - Ks[6] * u[0] - Ks[7] * u[1]) * inv[2] + (1.f - omega) * u[2];
        u[1] = omega * (f[1] - KeU[1] - Ks[3] * u[0] - Ks[5] * u[2]) * inv[1] + (1.f - omega) * u[1];
        u[0] = omega * (f[0] - KeU[0] - Ks[1] * u[1] - Ks[2] * u[2]) * inv[0] + (1.f - omega) * u[0];
    }
}

template <int BS>
__device__ __forceinline__ double block_sum(double v, double* sh) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) sh[wid] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0) {
        for (int i = 0; i < BS / 64; i++) s += sh[i];
    }
    __syncthreads();
    return s;
}

inline unsigned nblk(size_t work, int bs = 256) { return (unsigned)((work + bs - 1) / bs); }

inline Lay make_lay(int n, int lex) {
    Lay L;
    L.n = n;
    L.h = n / 2;
    L.h3 = (uint32_t)L.h * L.h * L.h;
    L.lex = lex;
    return L;
}

inline unsigned full_grid(const Lay& L) {
    const size_t N = (size_t)L.n * L.n * L.n;
    return L.lex ? nblk(N, kFullThreads) : nblk(L.h3, 64);
}

}  // namespace
}  // namespace homo3d
