// Launch wrappers of the gfx950 kernels (kernels.hip).  All fields carry 6 load cases.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace homo3d {

// Fine-level kernels take u as FP32 planes ([6][3][n^3]) or, with u_half, as packed FP16 load-case
// pairs ([3][3][n^3] words of two halves, cases 2p and 2p + 1; only with n % 8 == 0).
// Element matrix for the matrix-core form of the fine operator, built from the integer Lame tables
// Kl = 72 KE(1, 0), Km = 72 KE(0, 1): either one FP16-exact table T = (lambda / mu) Kl + Km with
// KE = c0 T (nt = 1), or Kl and Km with KE = c0 Kl + c1 Km (nt = 2), laid out as the A operands of
// 16x16x32 tiles (kKeMfmaBytes).  ke_mfma_table returns nt.
constexpr int kKeMfmaBytes = 3 * 64 * 8 * 2;
int ke_mfma_table(const double* kl, const double* km, double lam, double mu, void* table, float* c0, float* c1);
struct FineMfma {
    const void* table;  // device copy of the ke_mfma_table output
    float c0, c1;
    int nt;
};
// The FP32 element matrix as the fine-level kernels take it: KE (576 floats), then from kKeBlocks on the
// block constants C_d,ij = KE[7 - e0][b0](i, j) of each neighbour offset d at 12 d + 3 i + j, for the cell e0
// with e0_m = 1 exactly where d_m = +1 and b0_m = d_m + 1 - e0_m.
constexpr int kKeBlocks = 576, kKeFloats = kKeBlocks + 27 * 12;
void fine_block_consts(float* ke);  // fills them from KE, on the host
// n for which packed-FP16 fine operators run in element form on the matrix cores
int fine_apply_mfma_ok(int n);
// out = K u (f == nullptr) or f - K u.  With mf, packed-FP16 u and fine_apply_mfma_ok(n) the operator
// runs in element form on the matrix cores.
void launch_fine_apply(hipStream_t s, int n, const float* ke, const FineMfma* mf, const float* w, const void* u,
                       int u_half, const float* f, float* out);
// One CG step's operator pass with the vector updates fused (z the preconditioned residual, FP32 or
// packed FP16 by z_half; sc the device CG scalars, alpha at sc + 12, beta at sc + 24):
//   first: p = z, q = K p;  else: x += alpha p_old, p = z + beta p_old, q = K z + beta q_old (= K p),
// and the per-load-case FP64 dot p . q -> out6.  partial holds 6 * n^3 / 512 doubles (and at least
// 6 * dot_blocks).
// staged (packed FP16 z, fine_cg_staged_ok(n)): each workgroup stages its z node box in LDS instead of
// gathering the neighbours from memory; the results are the same bit for bit.
int fine_cg_staged_ok(int n);
void launch_fine_apply_cg(hipStream_t s, int n, const float* ke, const FineMfma* mf, const float* w, const void* z,
                          int z_half, int staged, float* p, float* x, double* sc, int first, float* q,
                          double* partial, int dot_blocks);
// Colours cfirst and cfirst + 1 (cfirst even; REVERSE: cfirst and cfirst - 1, cfirst odd) in one launch,
// the second colour reading the first one's new values.  zero_start: part of a forward sweep that starts from
// u = 0 (u need not be cleared).  n even, at most 512.  With partial (reverse sweeps of
// a packed-FP16 u only), each of the gs_pair_blocks(n) workgroups also writes its FP64 sums of f . u_new per
// load case to partial[r * pstride + workgroup].
int gs_pair_blocks(int n);
// rown (zero-start forward passes; ignored otherwise): both colours also store, per vertex, f minus the
// K u terms of the colours swept so far (the vertex itself included); after the sweep,
// launch_fine_residual_later turns these into the residual f - K u.
void launch_fine_gs2(hipStream_t s, int n, int cfirst, float omega, int reverse, int zero_start, const float* ke,
                     const float* w, void* u, int u_half, const float* f, double* partial = nullptr,
                     int pstride = 0, float* rown = nullptr);
// r -= the K u terms of later-colour neighbours, colours 0..6 (one launch): with the own-colour
// residuals of a complete zero-start forward sweep (launch_fine_gs2 rown) in r, leaves r = f - K u.
void launch_fine_residual_later(hipStream_t s, int n, const float* ke, const float* w, const void* u, int u_half,
                                float* r);
void launch_macro_rhs(hipStream_t s, int n, const float* kchi, const float* w, float* f);
void launch_fine_residual64(hipStream_t s, int n, const double* ke, const double* kchi, const float* xc, double emin,
                            const double* u, float* r32, double* partial, double* out6, int do_k);
void launch_rhs_norm64(hipStream_t s, int n, const double* kchi, const float* xc, double emin, double* partial,
                       double* out6);
// The FP64 refinement iterate u of N vertices is nine planes of component pairs: component c = 3 r + i
// (component i of load case r) of vertex v is u[u64_index(c, v, N)].  x, p are FP32 planes [18][N].
__host__ __device__ inline size_t u64_index(int c, size_t v, size_t N) {
    return (size_t)(c >> 1) * 2 * N + 2 * v + (size_t)(c & 1);
}
void launch_round_f32(hipStream_t s, size_t N, const double* u, float* x);
// u (+)= x + alpha p for the 6 load cases (N % 2 == 0; alpha = sc + 12, only when pending): the last
// CG step's x update fused into the FP64 refinement iterate (add) or its first value.
void launch_refine_accumulate(hipStream_t s, size_t N, const double* sc, int pending, const float* x, const float* p,
                              double* u, int add);
void launch_widen_f64(hipStream_t s, size_t N, const float* x, double* u);
// zero load case r (all its components, every vertex) of the FP64 iterate
void launch_zero_case64(hipStream_t s, size_t N, int r, double* u);
void launch_zero_pin(hipStream_t s, size_t N, void* u, int u_half);
// FP32 field [6][3][N] <-> packed FP16 field [3][3][N] words (round to nearest)
void launch_pack_half(hipStream_t s, size_t N, const float* u, void* z);
void launch_unpack_half(hipStream_t s, size_t N, const void* z, float* u);
void launch_zero_pin64(hipStream_t s, size_t N, double* u);
// The coarsest level's dense FP64 inverse on the GPU (setup.hip): assembled from its FP32 stencil
// (lexicographic n_c^3 level, m = 3 n_c^3), symmetrised and inverted into ainv (m x m) by Gauss-Jordan
// elimination on the diagonal; work is another m x m doubles.  status (two words of device memory):
// status[0] = 0, or 1 + the first step whose pivot is not positive (the system is not positive definite;
// ainv is then not an inverse).
void launch_coarse_factor(hipStream_t s, int nc, const float* st, double* ainv, double* work, int* status);
// Coarse stencils: FP32 [243][n^3] or, with *_half, packed FP16 in quads of eight entries [31][n^3].
// u FP32 planes, or (u_half, only where stencil_u_half_ok: six load cases per launch) packed FP16 pairs.
int stencil_u_half_ok(int n, int lex);
void launch_stencil_apply(hipStream_t s, int n, int lex, const void* st, int st_half, const void* u, int u_half,
                          const float* f, float* out);
void launch_stencil_gs(hipStream_t s, int n, int colour, float omega, int reverse, int zero_start, const float* st,
                       float* u, const float* f);  // FP32, n <= 32
// Small coarse levels (smallgrid.hip; parity-blocked, n <= 32, packed FP16 stencils, FP32 fields).
int small_level_ok(int n, int lex, int st_half);
// A whole sweep in two launches of four colours each.
void launch_plane_sweep(hipStream_t s, int n, float omega, int reverse, int zero_start, const void* st, float* u,
                        const float* f);
// The bottom of a V(1,1) cycle from the last smoothed level (n points an axis, vcycle_tail_ok: 8 to 14) with
// right-hand side f to its corrected and post-smoothed u (zero before): smoothing, residual (res), transfers
// and the coarsest solve (uc, fc, ainv of the lexicographic coarsest level, n / 2 points an axis).
int vcycle_tail_ok(int n, int lex, int st_half);
void launch_vcycle_tail(hipStream_t s, int n, float omega, int reverse, const void* st, float* u, const float* f,
                        float* res, float* uc, float* fc, const double* Ainv);
// Colours cfirst and cfirst + 1 (cfirst even; reverse: cfirst and cfirst - 1, cfirst odd) of a coarse
// parity-blocked level in one launch, the second colour reading the first one's new values; only when
// stencil_gs_pairs_ok(n, lex) (levels above 32^3 whose grid rows fit a workgroup).
// rown (zero-start forward passes; ignored otherwise): the own-colour residuals, as launch_fine_gs2
// stores them; launch_stencil_residual_later completes them to f - A u after the sweep.
int stencil_gs_pairs_ok(int n, int lex);
void launch_stencil_gs2(hipStream_t s, int n, int cfirst, float omega, int reverse, int zero_start, const void* st,
                        int st_half, void* u, int u_half, const float* f, float* rown = nullptr);
void launch_stencil_residual_later(hipStream_t s, int n, const void* st, int st_half, const void* u, int u_half,
                                   float* r);
void launch_restrict(hipStream_t s, int nf, int lexc, const float* rf, float* fc);
// uf += P uc.  uc FP32, or packed FP16 (uc_half: parity-blocked coarse level, packed FP16 fine u).
void launch_prolong(hipStream_t s, int nf, int lexc, const void* uc, int uc_half, void* uf, int u_half, int pin);
// G: the 64 x 27 x 9 table of P-weighted element blocks, and G32 the same in FP32
void launch_galerkin_fine(hipStream_t s, int nf, int lexc, const double* G, const float* G32, const double* ke,
                          const float* w, void* stc, int out_half, float clamp);
// work: 243 nf^3 / 4 doubles
void launch_galerkin_coarse(hipStream_t s, int nf, int lexc, const void* stf, int in_half, void* stc, int out_half,
                            double* work, float clamp);
void launch_coarse_solve(hipStream_t s, int nc, const double* Ainv, const float* f, float* u);
// then: what else the sums' workgroups form from them for a CG step, in sc = [rz | pq | alpha | rz_new | beta |
// active], six doubles each.  kSumPq (out = sc + 6): alpha = rz / pq; kSumRz (out = sc + 18): beta = rz_new / rz,
// rz = rz_new.
enum { kSumOnly = 0, kSumPq = 1, kSumRz = 2 };
void launch_dot6(hipStream_t s, size_t M, const float* a, const float* b, double* partial, int nblocks, double* out,
                 int then = kSumOnly, double* sc = nullptr);
void launch_sum_partials(hipStream_t s, int R, int nblocks, const double* partial, double* out, int then = kSumOnly,
                         double* sc = nullptr);
// CG updates over 6 load cases of M floats each (M % 4 == 0): r -= alpha q with |r|^2 -> out6;
// x += alpha p and, when do_p, p = z + beta p for the active load cases.
void launch_pcg_update_r(hipStream_t s, size_t M, const double* sc, const float* q, float* r, double* partial,
                         int nblocks, double* out6);
// z FP32 or packed FP16 (z_half); p and x FP32
void launch_pcg_update_px(hipStream_t s, size_t M, const double* sc, const void* z, int z_half, float* p, float* x,
                          int do_p, int nblocks);
// p = z
hipError_t launch_set_p(hipStream_t s, size_t M, const void* z, int z_half, float* p, int nblocks);
// per-load-case r . z -> out6 (z FP32 or packed FP16)
void launch_dot_rz(hipStream_t s, size_t M, const float* r, const void* z, int z_half, double* partial, int nblocks,
                   double* out6, int then = kSumOnly, double* sc = nullptr);
// C^H sums and sensitivity of the fields chi (energy.hip); lam, mu the Lame parameters, wdc 21 host floats
void launch_elastic_matrix(hipStream_t s, int n, double lam, double mu, const float* w, const float* chi,
                           double* partial, int nblocks, double* out21);
void launch_sensitivity(hipStream_t s, int n, int pitch, double lam, double mu, const float* chi, const float* wdc,
                        float* sens);
void launch_oc_trial(hipStream_t s, int n, int pitch, double g, double min_rho, double step, double damp,
                     const float* sens, const float* rho, float* out, double* partial, int nblocks, double* sum);
void launch_absmax(hipStream_t s, int n, int pitch, const float* a, float* partial, int nblocks);
// FP64 block sums of a (nblocks partials); a = value
void launch_field_sum(hipStream_t s, int n, int pitch, const float* a, double* partial, int nblocks);
void launch_field_fill(hipStream_t s, int n, int pitch, float value, float* a);
void launch_set_weights(hipStream_t s, int n, int pitch, double emin, const float* x, float* w, float* xc);
void launch_copy_pitched(hipStream_t s, int n, int pitch_in, int pitch_out, const float* in, float* out);
// Bridges to the learned warm-start network (g | n; network tensors bf16 channels-last, see net.hip):
// input channel 0 = mean of x^(1/3) over each coarse cell; target = scale (u - mean) / n sampled at the
// coarse vertices, the mean weighted by the input's rho^3 (mean18: 18 doubles of device scratch); warm start = periodic trilinear upsampling of
// the prediction P ([g^3][ldp]) minus its value at vertex 0, times n / scale, into U64 and x.
void launch_net_input(hipStream_t s, int n, int g, const float* x, uint16_t* in);
void launch_net_target(hipStream_t s, int n, int g, const double* u64, const uint16_t* in, double scale, double* mean18,
                       uint16_t* tg);
void launch_net_warm_start(hipStream_t s, int n, int g, const float* P, int ldp, double scale, double* u64, float* x);

}  // namespace homo3d
