// mg_kernels.hip -- kernels of the multigrid preconditioner: separable grid
// transfers, fused Chebyshev steps, precision conversion, the dense FP64
// coarse solve and the vector updates of the outer preconditioned CG.
//
// Transfers.  On a structured box with lexicographic node numbering, both
// the p-transfer (same cells, degree p_f -> p_c) and the h-transfer (Q_p on
// n cells -> n/2 cells) are tensor products of 1D interpolation matrices,
// P = P_z (x) P_y (x) P_x, so prolongation is three passes of a 1D matrix
// along one axis each, and restriction R = P^T is the same three passes with
// the transposed 1D matrices.  Each pass reads its input once per stencil
// entry from a neighbourhood of consecutive threads (coalesced along x for
// every axis) and writes its output once.
#include <algorithm>

#include "mfx_internal.hpp"
#include "mg.hpp"

namespace mfx {
namespace {

constexpr int kBlock = 256;

inline unsigned grid_for(uint64_t n) {
  return (unsigned)std::max<uint64_t>(1, std::min<uint64_t>((n + kBlock - 1) / kBlock, 65536));
}

// One thread per output; the row's entries are consecutive inputs along the
// axis (begin, count), so the loads of the inputs wait for one load only.
// The fused ends of a V-cycle's transfers (AxisIO): the input as a residual
// minuend - in, rows of the output set to zero, the output added to and the
// start of the next A x written beside it.
template <typename T>
__global__ void __launch_bounds__(kBlock)
k_axis_pass(AxisIO<T> io, uint32_t n0, uint32_t n1, uint32_t total, int axis, uint32_t in_len,
            const int2 *__restrict__ span, const T *__restrict__ val, int width) {
  const T *__restrict__ in = io.in;
  const T *__restrict__ minuend = io.minuend;
  for (uint32_t t = blockIdx.x * kBlock + threadIdx.x; t < total; t += gridDim.x * kBlock) {
    const uint32_t q = t / n0, i0 = t - q * n0;
    const uint32_t i2 = q / n1, i1 = q - i2 * n1;
    uint32_t row, base, stride;
    if (axis == 0) {
      row = i0;
      base = in_len * q;
      stride = 1;
    } else if (axis == 1) {
      row = i1;
      base = i0 + n0 * in_len * i2;
      stride = n0;
    } else {
      row = i2;
      base = i0 + n0 * i1;
      stride = n0 * n1;
    }
    const int2 sp = span[row];
    const T *w = val + (size_t)row * width;
    base += stride * (uint32_t)sp.x;
    T acc = 0;
    for (int k = 0; k < sp.y; ++k) {
      const uint32_t at = base + stride * (uint32_t)k;
      acc += w[k] * (minuend ? minuend[at] - in[at] : in[at]);
    }
    if (io.zero_rows && (io.zero_rows[t >> 5] >> (t & 31) & 1)) acc = 0;
    if (io.add) acc += io.out[t];
    io.out[t] = acc;
    if (io.start) io.start[t] = (io.start_rows[t >> 5] >> (t & 31) & 1) ? acc : T(0);
  }
}

// All three axes in one launch, for rows of at most W entries: every thread
// loads its W^3 inputs at once.  A pass costs a launch and a chain of loads
// whatever its size (4.5 us of a V-cycle's each); the two launches saved
// outweigh the loads the passes share up to the largest grids measured.  V-cycle of
// Q_4 on 32^3 cells 698 -> 664 us, of Q_1 on 64^3 cells 197 -> 165, on 128^3
// cells 750 -> 700.
template <typename T, int W>
__global__ void __launch_bounds__(kBlock)
k_axis_all(AxisIO<T> io, AxisMatrix<T> X, AxisMatrix<T> Y, AxisMatrix<T> Z) {
  const T *__restrict__ in = io.in;
  const T *__restrict__ minuend = io.minuend;
  const uint32_t total = (uint32_t)X.rows * Y.rows * Z.rows;
  for (uint32_t t = blockIdx.x * kBlock + threadIdx.x; t < total; t += gridDim.x * kBlock) {
    const uint32_t q = t / X.rows, i0 = t - q * X.rows, i2 = q / Y.rows, i1 = q - i2 * Y.rows;
    const int2 sx = X.span[i0], sy = Y.span[i1], sz = Z.span[i2];
    T v[W][W][W], wx[W], wy[W], wz[W];
#pragma unroll
    for (int k = 0; k < W; ++k) {
      wx[k] = X.val[(size_t)i0 * W + k];
      wy[k] = Y.val[(size_t)i1 * W + k];
      wz[k] = Z.val[(size_t)i2 * W + k];
    }
#pragma unroll
    for (int c = 0; c < W; ++c)
#pragma unroll
      for (int b = 0; b < W; ++b)
#pragma unroll
        for (int a = 0; a < W; ++a) {
          v[c][b][a] = T(0);
          if (a >= sx.y || b >= sy.y || c >= sz.y) continue;
          const uint32_t at =
              sx.x + a + (uint32_t)X.cols * (sy.x + b + (uint32_t)Y.cols * (sz.x + c));
          v[c][b][a] = minuend ? minuend[at] - in[at] : in[at];
        }
    T acc = 0;
#pragma unroll
    for (int c = 0; c < W; ++c) {
      T ay = 0;
#pragma unroll
      for (int b = 0; b < W; ++b) {
        T ax = 0;
#pragma unroll
        for (int a = 0; a < W; ++a) ax += wx[a] * v[c][b][a];
        ay += wy[b] * ax;
      }
      acc += wz[c] * ay;
    }
    if (io.zero_rows && (io.zero_rows[t >> 5] >> (t & 31) & 1)) acc = 0;
    if (io.add) acc += io.out[t];
    io.out[t] = acc;
    if (io.start) io.start[t] = (io.start_rows[t >> 5] >> (t & 31) & 1) ? acc : T(0);
  }
}

// ---- Q_1 levels with an assembled operator ----
// Row i of A couples the 3 x 3 x 3 nodes around node i: entry k = 9 dz + 3 dy + dx
// (each 0..2, offset -1) at st[k n + i].  The constrained rows (bitmask) are
// identity rows; every node of the grid's boundary is one.

// x = 1 on the nodes of one of the 27 colours (indices modulo 3), 0 elsewhere
__global__ void k_colour(double *__restrict__ x, uint32_t n0, uint32_t n1, uint32_t total,
                         uint32_t c) {
  for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < total; i += gridDim.x * kBlock) {
    const uint32_t q = i / n0, ix = i - q * n0, iz = q / n1, iy = q - iz * n1;
    x[i] = ix % 3 + 3 * (iy % 3) + 9 * (iz % 3) == c ? 1.0 : 0.0;
  }
}
// y = A x for x of colour c: the entry of each row's only neighbour of the colour
__global__ void k_take_colour(const double *__restrict__ y, float *__restrict__ st, uint32_t n0,
                              uint32_t n1, uint32_t total, uint32_t c) {
  for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < total; i += gridDim.x * kBlock) {
    const uint32_t q = i / n0, ix = i - q * n0, iz = q / n1, iy = q - iz * n1;
    const uint32_t dx = (c % 3 + 4 - ix % 3) % 3, dy = (c / 3 % 3 + 4 - iy % 3) % 3,
                   dz = (c / 9 + 4 - iz % 3) % 3;
    st[(size_t)(9 * dz + 3 * dy + dx) * total + i] = (float)y[i];
  }
}

// A Chebyshev step (launch_cheb_step) with r = b - A x formed in place:
// xo = x + d.  FROM_ZERO: x is the first iterate, x = c0 dinv b (not stored),
// and d_0 = x.  RESIDUAL: xo = r only.  At 33^3 rows it is bound by its launch
// and one batch of loads, 3.2 us in place of a matrix-free apply (5.6 us) and a
// step on vectors (4.5 us); at 2M rows by the bytes of the entries, which are
// more than the apply's vertices but need no atomics and no zeroed result: V-cycle of
// Q_1 on 64^3 cells 419 -> 197 us, on 128^3 cells 1746 -> 750.
template <bool FROM_ZERO, bool RESIDUAL>
__global__ void __launch_bounds__(kBlock)
k_stencil_step(const float *__restrict__ st, const uint32_t *__restrict__ mask,
               const float *__restrict__ x, float *__restrict__ xo, float *__restrict__ d,
               const float *__restrict__ b, const float *__restrict__ dinv, float c0, float c1,
               float c2, int n0, int n01, uint32_t total) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= total) return;
  const bool cons = mask[i >> 5] >> (i & 31) & 1;
  float s[3] = {0.0f, 0.0f, 0.0f};
  const float xi = FROM_ZERO ? c0 * dinv[i] * b[i] : x[i];
  if (cons) {
    s[0] = xi;
  } else {
    // all loads before the first use
    float a[27], v[27], w[FROM_ZERO ? 27 : 1];
#pragma unroll
    for (int k = 0; k < 27; ++k) {
      const uint32_t j = (uint32_t)((int)i + (k / 9 - 1) * n01 + (k / 3 % 3 - 1) * n0 + k % 3 - 1);
      a[k] = st[(size_t)k * total + i];
      v[k] = FROM_ZERO ? b[j] : x[j];
      if (FROM_ZERO) w[k] = dinv[j];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < 27; ++k) s[k / 9] += a[k] * (FROM_ZERO ? c0 * w[k] * v[k] : v[k]);
  }
  const float r = b[i] - ((s[0] + s[1]) + s[2]);
  if constexpr (RESIDUAL) {
    xo[i] = r;
  } else {
    const float dn = (FROM_ZERO ? c1 * xi : c1 != 0.0f ? c1 * d[i] : 0.0f) + c2 * dinv[i] * r;
    d[i] = dn;
    xo[i] = xi + dn;
  }
}

// start (optional): also the start value of the next A x in t -- the new x on
// the rows of the bitmask (identity rows), 0 elsewhere -- which spares the
// apply its own start pass over x and t.
__global__ void k_cheb_step(float *__restrict__ x, float *__restrict__ d,
                            const float *__restrict__ b, float *__restrict__ t,
                            const float *__restrict__ dinv, float c1, float c2, int has_t,
                            int x_zero, const uint32_t *__restrict__ start, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const float r = has_t ? b[i] - t[i] : b[i];
    const float dn = (c1 != 0.0f ? c1 * d[i] : 0.0f) + c2 * dinv[i] * r;
    d[i] = dn;
    const float xn = x_zero ? dn : x[i] + dn;
    x[i] = xn;
    if (start) t[i] = (start[i >> 5] >> (i & 31) & 1) ? xn : 0.0f;
  }
}

__global__ void k_residual_f32(float *__restrict__ r, const float *__restrict__ b,
                               const float *__restrict__ t, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    r[i] = b[i] - t[i];
}

__global__ void k_to_double(const float *__restrict__ in, double *__restrict__ out, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    out[i] = (double)in[i];
}

// part[workgroup] = the workgroup's sum of v
__device__ __forceinline__ void block_partial(double v, double *__restrict__ part) {
  __shared__ double red[kBlock / 64];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) s += red[w];
    part[blockIdx.x] = s;
  }
}

// FP64 <-> FP32 ends of the V-cycle: b = r with the constrained rows
// (bitmask) zero; z = x with the constrained rows of r
__global__ void k_to_float_free(const double *__restrict__ r, float *__restrict__ b,
                                const uint32_t *__restrict__ mask, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    b[i] = (mask[i >> 5] >> (i & 31) & 1) ? 0.0f : (float)r[i];
}
// part: partial sums of r z (see launch_to_double_free)
__global__ void __launch_bounds__(kBlock)
k_to_double_free(const float *__restrict__ x, const double *__restrict__ r, double *__restrict__ z,
                 const uint32_t *__restrict__ mask, uint64_t n, double *__restrict__ part) {
  double rz = 0.0;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const double ri = r[i];
    const double zi = (mask[i >> 5] >> (i & 31) & 1) ? ri : (double)x[i];
    z[i] = zi;
    rz += ri * zi;
  }
  if (part) block_partial(rz, part);
}

__global__ void k_set_listed_f32(float *__restrict__ dst, float v, const uint32_t *__restrict__ list,
                                 uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    dst[list[i]] = v;
}

// one workgroup per row of the coarse inverse
__global__ void __launch_bounds__(kBlock)
k_dense_solve(const double *__restrict__ Ainv, const uint32_t *__restrict__ free_idx,
              uint32_t n_free, const float *__restrict__ b, float *__restrict__ x) {
  __shared__ double red[kBlock / 64];
  const uint32_t row = blockIdx.x;
  double acc = 0.0;
  for (uint32_t j = threadIdx.x; j < n_free; j += kBlock)
    acc += Ainv[(size_t)row * n_free + j] * (double)b[free_idx[j]];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) s += red[w];
    x[free_idx[row]] = (float)s;
  }
}

__global__ void k_pcg_update(double *__restrict__ x, double *__restrict__ r,
                             const double *__restrict__ p, const double *__restrict__ ap,
                             double alpha, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    x[i] += alpha * p[i];
    r[i] -= alpha * ap[i];
  }
}

__global__ void k_pcg_direction(double *__restrict__ p, const double *__restrict__ z, double beta,
                                uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = z[i] + beta * p[i];
}

// The vector passes of the preconditioned CG with what follows them: a step's own
// dot products, conversion and start pass took 35 us of its ~120 us outside the
// V-cycle at 2.1M rows (a solve 6.03 -> 5.87 ms with them in).  r r goes to part, and b = r in FP32 with the
// constrained rows (bitmask) zero.
__global__ void __launch_bounds__(kBlock)
k_pcg_update_fused(double *__restrict__ x, double *__restrict__ r, const double *__restrict__ p,
                   const double *__restrict__ ap, double alpha, float *__restrict__ b,
                   const uint32_t *__restrict__ mask, uint64_t n, double *__restrict__ part) {
  double rr = 0.0;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    x[i] += alpha * p[i];
    const double ri = r[i] - alpha * ap[i];
    r[i] = ri;
    b[i] = (mask[i >> 5] >> (i & 31) & 1) ? 0.0f : (float)ri;
    rr += ri * ri;
  }
  block_partial(rr, part);
}

// p = z + beta p (p = z for beta = 0) and the start of A p: p on the constrained
// rows, whose p p goes to part, 0 elsewhere
__global__ void __launch_bounds__(kBlock)
k_pcg_direction_start(double *__restrict__ p, const double *__restrict__ z, double beta,
                      double *__restrict__ ap, const uint32_t *__restrict__ mask, uint64_t n,
                      double *__restrict__ part) {
  double c = 0.0;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const double pi = beta != 0.0 ? z[i] + beta * p[i] : z[i];
    const bool cons = mask[i >> 5] >> (i & 31) & 1;
    p[i] = pi;
    ap[i] = cons ? pi : 0.0;
    c += cons ? pi * pi : 0.0;
  }
  block_partial(c, part);
}

__global__ void k_axpy_f64(double *__restrict__ y, double a, const double *__restrict__ x, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    y[i] += a * x[i];
}

__global__ void k_scale(double *__restrict__ z, const double *__restrict__ r,
                        const double *__restrict__ dinv, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    z[i] = dinv[i] * r[i];
}

__global__ void k_residual_f64(double *__restrict__ r, const double *__restrict__ b,
                               const double *__restrict__ t, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    r[i] = b[i] - t[i];
}

}  // namespace

template <typename T>
void launch_axis_pass(const AxisMatrix<T> &M, int axis, const uint32_t out_dims[3],
                      const AxisIO<T> &io, hipStream_t s) {
  MFX_REQUIRE(axis >= 0 && axis < 3, "axis must be 0, 1 or 2");
  MFX_REQUIRE(M.span && M.val && io.in && io.out, "transfer pass: null pointer");
  MFX_REQUIRE((uint32_t)M.rows == out_dims[axis], "transfer pass: matrix rows != output length");
  MFX_REQUIRE(!io.start || io.start_rows, "transfer pass: start value without its rows");
  const uint64_t n = (uint64_t)out_dims[0] * out_dims[1] * out_dims[2];
  const uint64_t n_in = n / out_dims[axis] * (uint64_t)M.cols;
  MFX_REQUIRE(n < (1ull << 31) && n_in < (1ull << 31), "transfer pass: grid too large");
  if (n == 0) return;
  hipLaunchKernelGGL((k_axis_pass<T>), dim3(grid_for(n)), dim3(kBlock), 0, s, io, out_dims[0],
                     out_dims[1], (uint32_t)n, axis, (uint32_t)M.cols, M.span, M.val, M.width);
  MFX_HIP(hipGetLastError());
}
template void launch_axis_pass<float>(const AxisMatrix<float> &, int, const uint32_t[3],
                                      const AxisIO<float> &, hipStream_t);
template void launch_axis_pass<double>(const AxisMatrix<double> &, int, const uint32_t[3],
                                       const AxisIO<double> &, hipStream_t);

template <typename T>
bool launch_axis_all(const AxisMatrix<T> M[3], const AxisIO<T> &io, hipStream_t s) {
  const int w = M[0].width;
  if ((w != 2 && w != 3) || M[1].width != w || M[2].width != w) return false;
  uint64_t n = 1, n_in = 1;
  for (int a = 0; a < 3; ++a) {
    MFX_REQUIRE(M[a].span && M[a].val, "transfer: null pointer");
    n *= (uint64_t)M[a].rows;
    n_in *= (uint64_t)M[a].cols;
  }
  MFX_REQUIRE(io.in && io.out && io.in != io.out, "transfer: bad input or output");
  MFX_REQUIRE(!io.start || io.start_rows, "transfer: start value without its rows");
  MFX_REQUIRE(n < (1ull << 31) && n_in < (1ull << 31), "transfer: grid too large");
  if (n == 0) return true;
  if (w == 2)
    hipLaunchKernelGGL((k_axis_all<T, 2>), dim3(grid_for(n)), dim3(kBlock), 0, s, io, M[0], M[1],
                       M[2]);
  else
    hipLaunchKernelGGL((k_axis_all<T, 3>), dim3(grid_for(n)), dim3(kBlock), 0, s, io, M[0], M[1],
                       M[2]);
  MFX_HIP(hipGetLastError());
  return true;
}
template bool launch_axis_all<float>(const AxisMatrix<float>[3], const AxisIO<float> &, hipStream_t);

void launch_colour(double *x, const uint32_t dims[3], uint32_t colour, hipStream_t s) {
  const uint32_t n = dims[0] * dims[1] * dims[2];
  hipLaunchKernelGGL(k_colour, dim3(grid_for(n)), dim3(kBlock), 0, s, x, dims[0], dims[1], n,
                     colour);
  MFX_HIP(hipGetLastError());
}
void launch_take_colour(const double *y, float *st, const uint32_t dims[3], uint32_t colour,
                        hipStream_t s) {
  const uint32_t n = dims[0] * dims[1] * dims[2];
  hipLaunchKernelGGL(k_take_colour, dim3(grid_for(n)), dim3(kBlock), 0, s, y, st, dims[0], dims[1],
                     n, colour);
  MFX_HIP(hipGetLastError());
}
void launch_stencil_step(const Stencil &A, StencilMode mode, const float *x, float *xo, float *d,
                         const float *b, const float *dinv, float c0, float c1, float c2,
                         hipStream_t s) {
  const uint32_t n = A.dims[0] * A.dims[1] * A.dims[2];
  MFX_REQUIRE(A.val && A.mask && xo != x, "stencil step: bad arguments");
  const dim3 grid((n + kBlock - 1) / kBlock), block(kBlock);
  const int n0 = (int)A.dims[0], n01 = (int)(A.dims[0] * A.dims[1]);
#define MFX_STEP(Z, R)                                                                          \
  hipLaunchKernelGGL((k_stencil_step<Z, R>), grid, block, 0, s, A.val, A.mask, x, xo, d, b, dinv, \
                     c0, c1, c2, n0, n01, n)
  if (mode == StencilMode::kFromZero)
    MFX_STEP(true, false);
  else if (mode == StencilMode::kResidual)
    MFX_STEP(false, true);
  else
    MFX_STEP(false, false);
#undef MFX_STEP
  MFX_HIP(hipGetLastError());
}

void launch_cheb_step(float *x, float *d, const float *b, float *t, const float *dinv, float c1,
                      float c2, bool has_t, bool x_zero, const uint32_t *start, uint64_t n,
                      hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_cheb_step, dim3(grid_for(n)), dim3(kBlock), 0, s, x, d, b, t, dinv, c1, c2,
                     (int)has_t, (int)x_zero, start, n);
  MFX_HIP(hipGetLastError());
}

void launch_residual_f32(float *r, const float *b, const float *t, uint64_t n, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_residual_f32, dim3(grid_for(n)), dim3(kBlock), 0, s, r, b, t, n);
  MFX_HIP(hipGetLastError());
}

void launch_to_double(const float *in, double *out, uint64_t n, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_to_double, dim3(grid_for(n)), dim3(kBlock), 0, s, in, out, n);
  MFX_HIP(hipGetLastError());
}

void launch_to_float_free(const double *r, float *b, const uint32_t *mask, uint64_t n,
                          hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_to_float_free, dim3(grid_for(n)), dim3(kBlock), 0, s, r, b, mask, n);
  MFX_HIP(hipGetLastError());
}

uint32_t pcg_blocks(uint64_t n) {
  return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((n + kBlock - 1) / kBlock, 2048));
}
void launch_to_double_free(const float *x, const double *r, double *z, const uint32_t *mask,
                           uint64_t n, hipStream_t s, double *part) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_to_double_free, dim3(part ? pcg_blocks(n) : grid_for(n)), dim3(kBlock), 0, s,
                     x, r, z, mask, n, part);
  MFX_HIP(hipGetLastError());
}
void launch_pcg_update_fused(double *x, double *r, const double *p, const double *ap, double alpha,
                             float *b, const uint32_t *mask, uint64_t n, double *part,
                             hipStream_t s) {
  hipLaunchKernelGGL(k_pcg_update_fused, dim3(pcg_blocks(n)), dim3(kBlock), 0, s, x, r, p, ap, alpha,
                     b, mask, n, part);
  MFX_HIP(hipGetLastError());
}
void launch_pcg_direction_start(double *p, const double *z, double beta, double *ap,
                                const uint32_t *mask, uint64_t n, double *part, hipStream_t s) {
  hipLaunchKernelGGL(k_pcg_direction_start, dim3(pcg_blocks(n)), dim3(kBlock), 0, s, p, z, beta, ap,
                     mask, n, part);
  MFX_HIP(hipGetLastError());
}

void launch_set_listed_f32(float *dst, float v, const uint32_t *list, uint64_t n, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_set_listed_f32, dim3(grid_for(n)), dim3(kBlock), 0, s, dst, v, list, n);
  MFX_HIP(hipGetLastError());
}

void launch_dense_solve(const double *Ainv, const uint32_t *free_idx, uint32_t n_free,
                        const float *b, float *x, hipStream_t s) {
  if (n_free == 0) return;
  hipLaunchKernelGGL(k_dense_solve, dim3(n_free), dim3(kBlock), 0, s, Ainv, free_idx, n_free, b,
                     x);
  MFX_HIP(hipGetLastError());
}

void launch_pcg_update(double *x, double *r, const double *p, const double *ap, double alpha,
                       uint64_t n, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_pcg_update, dim3(grid_for(n)), dim3(kBlock), 0, s, x, r, p, ap, alpha, n);
  MFX_HIP(hipGetLastError());
}

void launch_axpy_f64(double *y, double a, const double *x, uint64_t n, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_axpy_f64, dim3(grid_for(n)), dim3(kBlock), 0, s, y, a, x, n);
  MFX_HIP(hipGetLastError());
}

void launch_scale(double *z, const double *r, const double *dinv, uint64_t n, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_scale, dim3(grid_for(n)), dim3(kBlock), 0, s, z, r, dinv, n);
  MFX_HIP(hipGetLastError());
}

void launch_residual_f64(double *r, const double *b, const double *t, uint64_t n, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_residual_f64, dim3(grid_for(n)), dim3(kBlock), 0, s, r, b, t, n);
  MFX_HIP(hipGetLastError());
}

void launch_pcg_direction(double *p, const double *z, double beta, uint64_t n, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_pcg_direction, dim3(grid_for(n)), dim3(kBlock), 0, s, p, z, beta, n);
  MFX_HIP(hipGetLastError());
}

}  // namespace mfx
