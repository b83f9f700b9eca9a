// Launch wrappers of the density utilities (fields.hip).  Arrays are n^3 floats, lexicographic, row pitch
// `pitch` (only the n live columns are touched).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace homo3d {

// Radial filters with the normalised (2h+1)^3 box weights wk: conv (Spline4 / linear), its adjoint and the
// OC sensitivity filter.  box_filter_ok(n, h): the staged kernels take the box; wk is then a host array,
// table holds (2h+1)^3 doubles of device scratch, and out must not overlap the inputs.  Other boxes: wk in
// device memory, and the adjoint needs the forward pass's in-grid weight sums (wsum).
int box_filter_ok(int n, int h);
constexpr int kBoxTable = 343;
void launch_box_conv(hipStream_t s, int n, int pitch, int h, int periodic, const float* wk, double* table,
                     const float* in, float* out);
void launch_box_adjoint(hipStream_t s, int n, int pitch, int h, int periodic, const float* wk, double* table,
                        const float* in, float* out);
void launch_box_sens(hipStream_t s, int n, int pitch, int h, int periodic, const float* wk, double* table,
                     const float* sens, const float* rho, float* out);
void launch_oc_filter(hipStream_t s, int n, int pitch, int h, int periodic, const float* wk, const float* sens,
                      const float* rho, float* out);
void launch_conv_filter(hipStream_t s, int n, int pitch, int h, int periodic, const float* wk, const float* in,
                        float* out, float* wsum);
void launch_conv_filter_back(hipStream_t s, int n, int pitch, int h, int periodic, const float* wk, const float* dout,
                             const float* wsum, float* din);

// Elementwise maps (outputs may be the inputs): sgm projection and its backward, x = rho^p and
// drho = p rho^(p - 1) dx.
void launch_sgm(hipStream_t s, int n, int pitch, double k, double c, const float* x, float* y);
void launch_sgm_back(hipStream_t s, int n, int pitch, double k, const float* y, const float* gy, float* gx);
void launch_density_pow(hipStream_t s, int n, int pitch, float p, const float* rho, float* x);
void launch_density_pow_grad(hipStream_t s, int n, int pitch, float p, const float* rho, const float* dx, float* drho);

// Symmetry projection in place over the elements 8 p + f set in `group`: axis permutation p (kSymPerm) after
// which the axes in f are mirrored, q[a] = coordinate kSymPerm[p][a], or n - 1 minus it.
constexpr int kSymPerm[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};
void launch_symmetrize(hipStream_t s, int n, int pitch, uint64_t group, float* field);

}  // namespace homo3d
