// mg.hpp -- launchers of the multigrid kernels (mg_kernels.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/mfx.h"

namespace mfx {

// operator applications with vmult semantics (zero, apply, identity rows)
void vmult64(mfx_op &op, double *dst, const double *src, hipStream_t s);
void vmult32(mfx_op &op, float *dst, const float *src, hipStream_t s);
// `degree` Chebyshev(Jacobi) steps towards A x = b in FP32 on [lmin, lmax]
// (t, d: scratch vectors of the operator's size).  started: t already holds
// the start value of A x (x on the constrained rows, 0 elsewhere); leave_start: t is left as the
// start value of A x for the final x.  Both only where
// cheb_starts(op): the apply then adds to t without a start pass of its own.
void chebyshev(mfx_op &op, float *x, const float *b, const float *dinv, float *t, float *d,
               int degree, double lmin, double lmax, bool zero_initial, hipStream_t s,
               bool started = false, bool leave_start = false);
bool cheb_starts(const mfx_op &op);
// largest eigenvalue of D^-1 A from `iters` CG (Lanczos) steps, FP64
double estimate_lambda_max(mfx_op &op, const double *inv_diag, int iters, hipStream_t s);

// A 1D transfer matrix (device arrays), applied along one axis of a
// lexicographic (x fastest) node grid: row i has span[i].y entries val[i width
// ...] in the consecutive columns from span[i].x.
template <typename T>
struct AxisMatrix {
  int rows = 0, cols = 0, width = 0;
  const int2 *span = nullptr;
  const T *val = nullptr;
};

// Operands of one pass: out = M in, or M (minuend - in); the rows of zero_rows
// (bitmask) are set to zero; add: out += instead; start: beside out, out on
// the rows of start_rows and 0 elsewhere.
template <typename T>
struct AxisIO {
  const T *in = nullptr;
  T *out = nullptr;
  const T *minuend = nullptr;
  const uint32_t *zero_rows = nullptr;
  bool add = false;
  T *start = nullptr;
  const uint32_t *start_rows = nullptr;
};

// out[i0,i1,i2] (+)= sum_k M[i_axis][k] in[..k..]: `out_dims` are the output
// grid's node counts, the input has M.cols nodes along `axis`.
template <typename T>
void launch_axis_pass(const AxisMatrix<T> &M, int axis, const uint32_t out_dims[3],
                      const AxisIO<T> &io, hipStream_t s);

// All three axes in one launch (out = M_z x M_y x M_x in); false, and nothing
// done, unless every row has 2 (or every row 3) entries at most.
template <typename T>
bool launch_axis_all(const AxisMatrix<T> M[3], const AxisIO<T> &io, hipStream_t s);

// An assembled Q_1 operator on a node grid whose boundary rows are constrained
// (identity rows, in the bitmask): 27 entries per row, val[k n + i].
struct Stencil {
  const float *val = nullptr;
  const uint32_t *mask = nullptr;
  uint32_t dims[3] = {0, 0, 0};
};
// x = 1 on the nodes of one of 27 colours, 0 elsewhere; y = A x to the stencil
void launch_colour(double *x, const uint32_t dims[3], uint32_t colour, hipStream_t s);
void launch_take_colour(const double *y, float *val, const uint32_t dims[3], uint32_t colour,
                        hipStream_t s);
// kStep: launch_cheb_step with t = A x, result in xo; kFromZero: the first two
// steps from zero, with x = c0 dinv b after the first; kResidual: xo = b - A x
enum class StencilMode { kStep, kFromZero, kResidual };
void launch_stencil_step(const Stencil &A, StencilMode mode, const float *x, float *xo, float *d,
                         const float *b, const float *dinv, float c0, float c1, float c2,
                         hipStream_t s);

// One Chebyshev step on FP32 vectors:
//   r = b - t (r = b without has_t), d = c1 d + c2 dinv r, x = x + d
// (x = d when x_zero: the iterate was zero).  c1 = 0 starts the recurrence.
// start (bitmask, optional): t = the new x on its rows, 0 elsewhere.
void launch_cheb_step(float *x, float *d, const float *b, float *t, const float *dinv, float c1,
                      float c2, bool has_t, bool x_zero, const uint32_t *start, uint64_t n,
                      hipStream_t s);
// b = r, 0 on the rows of the bitmask; z = x, r on the rows of the bitmask
void launch_to_float_free(const double *r, float *b, const uint32_t *mask, uint64_t n,
                          hipStream_t s);
// (part, optional: pcg_blocks(n) partial sums of r z)
void launch_to_double_free(const float *x, const double *r, double *z, const uint32_t *mask,
                           uint64_t n, hipStream_t s, double *part = nullptr);
// x += alpha p, r -= alpha ap, b = r on the free rows and 0 on the masked ones;
// pcg_blocks(n) partial sums of r r
void launch_pcg_update_fused(double *x, double *r, const double *p, const double *ap, double alpha,
                             float *b, const uint32_t *mask, uint64_t n, double *part,
                             hipStream_t s);
// p = z + beta p; ap = p on the masked rows and 0 elsewhere (the start of A p);
// pcg_blocks(n) partial sums of p p over the masked rows
void launch_pcg_direction_start(double *p, const double *z, double beta, double *ap,
                                const uint32_t *mask, uint64_t n, double *part, hipStream_t s);
uint32_t pcg_blocks(uint64_t n);
// r = b - t
void launch_residual_f32(float *r, const float *b, const float *t, uint64_t n, hipStream_t s);
void launch_to_double(const float *in, double *out, uint64_t n, hipStream_t s);
void launch_set_listed_f32(float *dst, float v, const uint32_t *list, uint64_t n, hipStream_t s);
// x[free[i]] = sum_j Ainv[i][j] b[free[j]] in FP64 (the other entries of x are
// left alone)
void launch_dense_solve(const double *Ainv, const uint32_t *free_idx, uint32_t n_free,
                        const float *b, float *x, hipStream_t s);
// x += alpha p, r -= alpha ap
void launch_pcg_update(double *x, double *r, const double *p, const double *ap, double alpha,
                       uint64_t n, hipStream_t s);
// z = dinv * r (elementwise)
void launch_scale(double *z, const double *r, const double *dinv, uint64_t n, hipStream_t s);
// r = b - t
void launch_residual_f64(double *r, const double *b, const double *t, uint64_t n, hipStream_t s);
// y += a x
void launch_axpy_f64(double *y, double a, const double *x, uint64_t n, hipStream_t s);
// p = z + beta p
void launch_pcg_direction(double *p, const double *z, double beta, uint64_t n, hipStream_t s);

}  // namespace mfx
