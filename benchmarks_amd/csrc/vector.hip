// vector.hip -- vector kernels and the device-resident conjugate-gradient
// steps.  All reductions are two-stage and deterministic: every workgroup
// writes one partial (fixed association inside the group), and a single
// workgroup sums the partials in index order.  CG scalars (alpha, beta,
// gamma, the convergence test) never leave the GPU; a `done` flag makes
// every CG kernel return at once after convergence, so the host can enqueue
// iterations in batches and check the flag once per batch.
#include <type_traits>

#include "mfx_internal.hpp"
#include "cg_state.hpp"

namespace mfx {
namespace {

constexpr int kBlock = 256;

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Workgroup sum of up to two values; results valid in thread 0.
__device__ __forceinline__ void block_sum2(double &a, double &b) {
  __shared__ double ra[kBlock / 64], rb[kBlock / 64];
  a = wave_sum(a);
  b = wave_sum(b);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) {
    ra[w] = a;
    rb[w] = b;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double sa = 0.0, sb = 0.0;
#pragma unroll
    for (int i = 0; i < kBlock / 64; ++i) {
      sa += ra[i];
      sb += rb[i];
    }
    a = sa;
    b = sb;
  }
}

// Sum partials[0..n) in a fixed order with one workgroup.
__device__ __forceinline__ double sum_partials(const double *__restrict__ part, uint32_t n) {
  double s = 0.0, unused = 0.0;
  for (uint32_t i = threadIdx.x; i < n; i += kBlock) s += part[i];
  block_sum2(s, unused);
  return s;  // valid in thread 0
}

__global__ void k_fill(double *x, double v, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    x[i] = v;
}
__global__ void k_fill_f32(float *x, float v, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    x[i] = v;
}

template <typename T>
__global__ void k_copy_listed(T *__restrict__ dst, const T *__restrict__ src,
                              const uint32_t *__restrict__ list, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t j = list[i];
    dst[j] = src[j];
  }
}

// dst = the start of an apply that accumulates: src on the rows of the
// bitmask (constrained rows, whose result is src), 0 elsewhere; src is read
// on the masked rows only.  kStartUnroll mask words of a lane are in flight.
constexpr int kStartUnroll = 4;
template <typename T>
__global__ void __launch_bounds__(kBlock)
k_start(T *__restrict__ dst, const T *__restrict__ src, const uint32_t *__restrict__ mask,
        uint64_t n) {
  const uint64_t step = (uint64_t)gridDim.x * (kBlock * kStartUnroll);
  for (uint64_t i0 = (uint64_t)blockIdx.x * (kBlock * kStartUnroll) + threadIdx.x; i0 < n;
       i0 += step) {
    uint32_t w[kStartUnroll];
    T v[kStartUnroll];
#pragma unroll
    for (int k = 0; k < kStartUnroll; ++k) {
      const uint64_t i = i0 + k * kBlock;
      w[k] = i < n ? mask[i >> 5] : 0;
    }
#pragma unroll
    for (int k = 0; k < kStartUnroll; ++k) {
      const uint64_t i = i0 + k * kBlock;
      v[k] = T(0);
      if (w[k] >> (i & 31) & 1) v[k] = src[i];
    }
#pragma unroll
    for (int k = 0; k < kStartUnroll; ++k) {
      const uint64_t i = i0 + k * kBlock;
      if (i < n) dst[i] = v[k];
    }
  }
}

// bit i of the mask for every listed i (words zeroed before)
__global__ void k_mark_bits(const uint32_t *__restrict__ list, uint64_t n,
                            uint32_t *__restrict__ mask) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    atomicOr(mask + (list[i] >> 5), 1u << (list[i] & 31));
}

__global__ void k_any_masked(const uint32_t *__restrict__ map, uint64_t n,
                             const uint32_t *__restrict__ mask, uint32_t *__restrict__ found) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t j = map[i];
    if (j != kInvalid && (mask[j >> 5] >> (j & 31) & 1)) *found = 1;
  }
}

__global__ void k_zero_words(uint32_t *__restrict__ w, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    w[i] = 0;
}

__global__ void k_set_listed(double *__restrict__ dst, double v,
                             const uint32_t *__restrict__ list, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    dst[list[i]] = v;
}

__global__ void k_invert_diagonal(double *d, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    d[i] = d[i] > 0.0 ? 1.0 / d[i] : 1.0;
}

// SplitMix64 stream, element i uses state seed + (i+1) * golden gamma.
__global__ void k_random(double *x, uint64_t n, uint64_t seed) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    uint64_t z = seed + (i + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z = z ^ (z >> 31);
    x[i] = (double)(z >> 11) * 0x1.0p-53 * 2.0 - 1.0;
  }
}

// Sum of sine modes at given points (x, y, z interleaved):
// out_i = sum_m a_m sin(pi k0_m x_i) sin(pi k1_m y_i) sin(pi k2_m z_i),
// the modes summed in index order.
__global__ void k_sine_modes(const double *__restrict__ xyz, uint64_t n, SineModes m,
                             double *__restrict__ out) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const double x = xyz[3 * i], y = xyz[3 * i + 1], z = xyz[3 * i + 2];
    double f = 0.0;
    for (int k = 0; k < m.n; ++k)
      f += m.a[k] * (sinpi(m.k[3 * k] * x) * sinpi(m.k[3 * k + 1] * y) * sinpi(m.k[3 * k + 2] * z));
    out[i] = f;
  }
}

__global__ void k_gather(const uint32_t *__restrict__ map, uint64_t n,
                         const double *__restrict__ src, double *__restrict__ evec) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t j = map[i];
    evec[i] = (j == kInvalid) ? 0.0 : src[j];
  }
}

__global__ void k_scatter_add(const uint32_t *__restrict__ map, uint64_t n,
                              const double *__restrict__ evec, double *__restrict__ dst) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t j = map[i];
    if (j != kInvalid) unsafeAtomicAdd(dst + j, evec[i]);
  }
}

__global__ void k_dot_partials(const double *__restrict__ x, const double *__restrict__ y,
                               uint64_t n, double *__restrict__ part) {
  double s = 0.0, unused = 0.0;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    s += x[i] * y[i];
  block_sum2(s, unused);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ void k_dot_final(const double *__restrict__ part, uint32_t n, double *result) {
  const double s = sum_partials(part, n);
  if (threadIdx.x == 0) *result = s;
}

// ---------------------------------------------------------------------------
// CG (deal.II SolverCG semantics, see cg_state.hpp)
// ---------------------------------------------------------------------------

// r = b - r (r holds A x0 on entry); partials of r.r and r.(P r).
__global__ void k_cg_init(CgState *st, const double *__restrict__ b, double *__restrict__ r,
                          const double *__restrict__ invd, uint64_t n, double *__restrict__ part) {
  double rr = 0.0, rz = 0.0;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const double ri = b[i] - r[i];
    r[i] = ri;
    rr += ri * ri;
    rz += ri * (invd ? invd[i] * ri : ri);
  }
  block_sum2(rr, rz);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = rr;
    part[gridDim.x + blockIdx.x] = rz;
  }
}

// ||r_0||, tolerance, step-0 check.
__global__ void k_cg_start(CgState *st, const double *__restrict__ part, uint32_t nb,
                           double abs_tol, double rel_tol, int max_steps) {
  const double rr = sum_partials(part, nb);
  __syncthreads();
  const double rz = sum_partials(part + nb, nb);
  if (threadIdx.x == 0) {
    const double rn = sqrt(rr);
    st->initial = rn;
    st->last = rn;
    st->tol = fmax(abs_tol, rel_tol * rn);
    st->gamma = rz;
    st->beta = 0.0;
    st->first = 1;
    st->steps = 0;
    st->max_steps = max_steps;
    st->breakdown = 0;
    if (st->history && st->history_len > 0) st->history[0] = rn;
    // deal.II's SolverControl::check fails at step 0 when max_steps <= 0
    st->done = (rn <= st->tol) ? 1 : ((isnan(rn) || max_steps <= 0) ? 2 : 0);
  }
}

// x += alpha p (the previous step's update, which needs the old p this
// kernel reads anyway), then p = P r + beta p (p = P r on the first step);
// Ap = 0.
__global__ void k_cg_direction(const CgState *st, const double *__restrict__ r,
                               const double *__restrict__ invd, double *__restrict__ p,
                               double *__restrict__ ap, double *__restrict__ x, uint64_t n) {
  if (st->done) return;
  const double beta = st->beta, alpha = st->alpha;
  const bool first = st->first != 0;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const double v = invd ? invd[i] * r[i] : r[i];
    if (first) {
      p[i] = v;
    } else {
      const double pi = p[i];
      x[i] += alpha * pi;
      p[i] = v + beta * pi;
    }
    ap[i] = 0.0;
  }
}

// The last step's x += alpha p, after the iteration has stopped; alpha from
// `sa` (the state the update pass wrote it to).
__global__ void k_cg_finish(const CgState *st, const CgState *sa, double *__restrict__ x,
                            const double *__restrict__ p, uint64_t n) {
  if (st->steps == 0) return;
  const double alpha = sa->alpha;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    x[i] += alpha * p[i];
}

// Identity rows: Ap_c = p_c, partial sum of p_c^2 (the constrained part of p.Ap).
__global__ void k_cg_constrained(const CgState *st, const uint32_t *__restrict__ list,
                                 uint64_t nc, const double *__restrict__ p,
                                 double *__restrict__ ap, double *__restrict__ part) {
  if (st->done) return;
  double s = 0.0, unused = 0.0;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nc;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t j = list[i];
    const double v = p[j];
    ap[j] = v;
    s += v * v;
  }
  block_sum2(s, unused);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// alpha = gamma / p.Ap
// sums of chunks of the partials: chunk b = part[b chunk, (b + 1) chunk)
__global__ void k_cg_chunks(const CgState *st, const double *__restrict__ part, uint32_t n,
                            uint32_t chunk, double *__restrict__ out) {
  if (st->done) return;
  const uint32_t b0 = blockIdx.x * chunk, b1 = min(n, b0 + chunk);
  double s = 0.0, unused = 0.0;
  for (uint32_t i = b0 + threadIdx.x; i < b1; i += kBlock) s += part[i];
  block_sum2(s, unused);
  if (threadIdx.x == 0) out[blockIdx.x] = s;
}

__global__ void k_cg_alpha(CgState *st, const double *__restrict__ part, uint32_t n) {
  if (st->done) return;
  const double pap = sum_partials(part, n);
  if (threadIdx.x == 0) {
    st->alpha = st->gamma / pap;
    if (!(pap > 0.0) && !(pap < 0.0)) st->breakdown = 1;
  }
}

// r -= alpha Ap; partials of r.r and r.(P r).  (x += alpha p is applied by
// the next direction update, or by k_cg_finish after the last step.)
__global__ void k_cg_update(const CgState *st, double *__restrict__ r,
                            const double *__restrict__ ap, const double *__restrict__ invd,
                            uint64_t n, double *__restrict__ part) {
  if (st->done) return;
  const double alpha = st->alpha;
  double rr = 0.0, rz = 0.0;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const double ri = r[i] - alpha * ap[i];
    r[i] = ri;
    rr += ri * ri;
    rz += ri * (invd ? invd[i] * ri : ri);
  }
  block_sum2(rr, rz);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = rr;
    part[gridDim.x + blockIdx.x] = rz;
  }
}

// Convergence test of step k and beta for step k+1.
__global__ void k_cg_check(CgState *st, const double *__restrict__ part, uint32_t nb) {
  if (st->done) return;
  const double rr = sum_partials(part, nb);
  __syncthreads();
  const double rz = sum_partials(part + nb, nb);
  if (threadIdx.x == 0) {
    const double rn = sqrt(rr);
    const int it = st->steps + 1;
    st->steps = it;
    st->last = rn;
    if (st->history && it < st->history_len) st->history[it] = rn;
    if (rn <= st->tol) {
      st->done = 1;
    } else if (it >= st->max_steps || isnan(rn) || st->breakdown) {
      st->done = 2;
    } else {
      st->beta = rz / st->gamma;
      st->gamma = rz;
      st->first = 0;
    }
  }
}

// ---------------------------------------------------------------------------
// Small systems: a step in three launches instead of six.  The scalar work of
// a step (alpha, the convergence test, beta) and the identity rows move into
// the vector passes: every workgroup sums the few hundred partials itself, in
// the same order, and workgroup 0 records the result.  Two states alternate,
// so that no kernel reads what it writes: the direction pass reads `sa` and
// writes `sb`, the apply reads sb->done, the update pass reads `sb` and writes
// `sa`.  A step of 114k DoFs (BP3 Q4, q = 6): 27 -> 21 us.
// ---------------------------------------------------------------------------

// Each lane holds its kRows rows in registers, requested before the sums.
constexpr int kRows = 4;  // rows per lane: vec_grid's workgroups cover 4 kBlock rows

// Sums of two sets of n partials, in every thread of the workgroup.
__device__ __forceinline__ void sum_partials_all(const double *__restrict__ pa,
                                                 const double *__restrict__ pb, uint32_t n,
                                                 double &a, double &b) {
  __shared__ double total[2];
  a = b = 0.0;
  for (uint32_t i = threadIdx.x; i < n; i += kBlock) {
    a += pa[i];
    if (pb) b += pb[i];
  }
  block_sum2(a, b);
  if (threadIdx.x == 0) {
    total[0] = a;
    total[1] = b;
  }
  __syncthreads();
  a = total[0];
  b = total[1];
  __syncthreads();
}

// Convergence test of the step whose update left `sa` and the partials of r.r
// and r.(P r): returns the done flag, beta for the next step, and with
// `record` writes the state of the next step.
__device__ __forceinline__ int cg_next(const CgState *sa, CgState *sb,
                                       const double *__restrict__ part, uint32_t nb, bool record,
                                       double &beta) {
  const double tol = sa->tol, gamma = sa->gamma;
  const int steps = sa->steps + 1, max_steps = sa->max_steps, breakdown = sa->breakdown;
  double rr, rz;
  sum_partials_all(part, part + nb, nb, rr, rz);
  const double rn = sqrt(rr);
  const int done = rn <= tol ? 1 : (steps >= max_steps || isnan(rn) || breakdown) ? 2 : 0;
  beta = rz / gamma;
  if (record) {
    CgState s = *sa;
    s.steps = steps;
    s.last = rn;
    s.done = done;
    if (!done) {
      s.beta = beta;
      s.gamma = rz;
      s.first = 0;
    }
    *sb = s;
  }
  return done;
}

// The test alone, before the host reads sb->done; the next direction pass
// repeats it with the same result.
__global__ void __launch_bounds__(kBlock)
k_cg_test(const CgState *sa, CgState *sb, const double *__restrict__ part, uint32_t nb) {
  if (sa->done) return;
  double beta;
  cg_next(sa, sb, part, nb, threadIdx.x == 0, beta);
}

// Convergence test (not on the first step), x += alpha p of the previous step,
// p = P r + beta p, and the start of Ap: p on the constrained rows (bitmask),
// 0 elsewhere, with partial sums of p^2 over the constrained rows.
template <bool FIRST>
__global__ void __launch_bounds__(kBlock)
k_cg_direction_small(const CgState *sa, CgState *sb, const double *__restrict__ part, uint32_t nb,
                     const double *__restrict__ r, const double *__restrict__ invd,
                     const uint32_t *__restrict__ mask, double *__restrict__ p,
                     double *__restrict__ ap, double *__restrict__ x,
                     double *__restrict__ part_c, uint64_t n) {
  if (FIRST ? sb->done : sa->done) return;  // (sb is not written on the first step)
  const uint64_t i0 = (uint64_t)blockIdx.x * (kBlock * kRows) + threadIdx.x;
  double v[kRows], pv[kRows], xv[kRows];
  uint32_t w[kRows];
#pragma unroll
  for (int k = 0; k < kRows; ++k) {
    const uint64_t i = i0 + k * kBlock;
    if (i >= n) continue;
    v[k] = invd ? invd[i] * r[i] : r[i];
    w[k] = mask[i >> 5] >> (i & 31) & 1;
    if (!FIRST) {
      pv[k] = p[i];
      xv[k] = x[i];
    }
  }
  double alpha = 0.0, beta = 0.0;
  if (!FIRST) {
    alpha = sa->alpha;
    if (cg_next(sa, sb, part, nb, blockIdx.x == 0 && threadIdx.x == 0, beta)) return;
  }
  double c = 0.0, unused = 0.0;
#pragma unroll
  for (int k = 0; k < kRows; ++k) {
    const uint64_t i = i0 + k * kBlock;
    if (i >= n) continue;
    if (!FIRST) {
      x[i] = xv[k] + alpha * pv[k];
      v[k] += beta * pv[k];
    }
    p[i] = v[k];
    ap[i] = w[k] ? v[k] : 0.0;
    c += w[k] ? v[k] * v[k] : 0.0;
  }
  block_sum2(c, unused);
  if (threadIdx.x == 0) part_c[blockIdx.x] = c;
}

// alpha = gamma / p.Ap (n_pap partials), r -= alpha Ap, partials of r.r and
// r.(P r)
__global__ void __launch_bounds__(kBlock)
k_cg_update_small(const CgState *sb, CgState *sa, const double *__restrict__ pap, uint32_t n_pap,
                  double *__restrict__ r, const double *__restrict__ ap,
                  const double *__restrict__ invd, uint64_t n, double *__restrict__ part) {
  if (sb->done) {
    if (blockIdx.x == 0 && threadIdx.x == 0) sa->done = sb->done;
    return;
  }
  const uint64_t i0 = (uint64_t)blockIdx.x * (kBlock * kRows) + threadIdx.x;
  double rv[kRows], av[kRows], dv[kRows];
#pragma unroll
  for (int k = 0; k < kRows; ++k) {
    const uint64_t i = i0 + k * kBlock;
    rv[k] = av[k] = 0.0;
    dv[k] = 1.0;
    if (i >= n) continue;
    rv[k] = r[i];
    av[k] = ap[i];
    if (invd) dv[k] = invd[i];
  }
  const double gamma = sb->gamma;
  double s, unused;
  sum_partials_all(pap, nullptr, n_pap, s, unused);
  const double alpha = gamma / s;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    CgState a = *sb;
    a.alpha = alpha;
    if (!(s > 0.0) && !(s < 0.0)) a.breakdown = 1;
    *sa = a;
  }
  double rr = 0.0, rz = 0.0;
#pragma unroll
  for (int k = 0; k < kRows; ++k) {
    const uint64_t i = i0 + k * kBlock;
    if (i >= n) continue;
    const double ri = rv[k] - alpha * av[k];
    r[i] = ri;
    rr += ri * ri;
    rz += ri * (dv[k] * ri);
  }
  block_sum2(rr, rz);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = rr;
    part[gridDim.x + blockIdx.x] = rz;
  }
}

inline unsigned vec_grid(uint64_t n) {
  const uint64_t g = (n + kBlock * 4 - 1) / (kBlock * 4);
  return (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(g, 4096));
}

}  // namespace

void launch_fill(double *x, double v, uint64_t n, hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_fill, dim3(vec_grid(n)), dim3(kBlock), 0, s, x, v, n);
  MFX_HIP(hipGetLastError());
}
void launch_fill_f32(float *x, float v, uint64_t n, hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_fill_f32, dim3(vec_grid(n)), dim3(kBlock), 0, s, x, v, n);
  MFX_HIP(hipGetLastError());
}
template <typename T>
void launch_copy_listed(T *dst, const T *src, const uint32_t *list, uint64_t n, hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_copy_listed<T>, dim3(vec_grid(n)), dim3(kBlock), 0, s, dst, src, list, n);
  MFX_HIP(hipGetLastError());
}
template void launch_copy_listed<double>(double *, const double *, const uint32_t *, uint64_t,
                                         hipStream_t);
template void launch_copy_listed<float>(float *, const float *, const uint32_t *, uint64_t,
                                        hipStream_t);
// Up to kStartRows rows one k_start; above, a fill and a copy of the listed
// rows.  The single launch saves the second one's ~2.5 us (a vmult of 36k
// DoFs 14.7 -> 11.4 us) and, in FP32 at 7.2M rows, still takes 8.2 us against
// 6.8 + 5.0; but its stores wait for the mask and the masked rows' values:
// 57 us against 38 + 10 at 33M rows in FP64, 115 against 78 + 15 at 68M.
constexpr uint64_t kStartRows = 1u << 23;
template <typename T>
void launch_start(T *dst, const T *src, const uint32_t *mask, const uint32_t *list,
                  uint64_t n_list, uint64_t n, hipStream_t s) {
  if (!n) return;
  if (n <= kStartRows) {
    hipLaunchKernelGGL(k_start<T>, dim3(vec_grid(n)), dim3(kBlock), 0, s, dst, src, mask, n);
    MFX_HIP(hipGetLastError());
    return;
  }
  if constexpr (std::is_same<T, double>::value)
    launch_fill(dst, 0.0, n, s);
  else
    launch_fill_f32(dst, 0.0f, n, s);
  launch_copy_listed<T>(dst, src, list, n_list, s);
}
template void launch_start<double>(double *, const double *, const uint32_t *, const uint32_t *,
                                   uint64_t, uint64_t, hipStream_t);
template void launch_start<float>(float *, const float *, const uint32_t *, const uint32_t *,
                                  uint64_t, uint64_t, hipStream_t);
void launch_bitmask(const uint32_t *list, uint64_t n_list, uint32_t *mask, uint64_t n,
                    hipStream_t s) {
  const uint64_t words = (n + 31) / 32;
  if (!words) return;
  hipLaunchKernelGGL(k_zero_words, dim3(vec_grid(words)), dim3(kBlock), 0, s, mask, words);
  if (n_list)
    hipLaunchKernelGGL(k_mark_bits, dim3(vec_grid(n_list)), dim3(kBlock), 0, s, list, n_list, mask);
  MFX_HIP(hipGetLastError());
}
bool any_masked(const uint32_t *map, uint64_t n, const uint32_t *mask, uint32_t *found,
                hipStream_t s) {
  if (!n) return false;
  uint32_t h = 0;
  hipLaunchKernelGGL(k_zero_words, dim3(1), dim3(kBlock), 0, s, found, (uint64_t)1);
  hipLaunchKernelGGL(k_any_masked, dim3(vec_grid(n)), dim3(kBlock), 0, s, map, n, mask, found);
  MFX_HIP(hipMemcpyAsync(&h, found, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
  MFX_HIP(hipStreamSynchronize(s));
  return h != 0;
}
void launch_set_listed(double *dst, double v, const uint32_t *list, uint64_t n, hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_set_listed, dim3(vec_grid(n)), dim3(kBlock), 0, s, dst, v, list, n);
  MFX_HIP(hipGetLastError());
}
void launch_invert_diagonal(double *d, uint64_t n, hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_invert_diagonal, dim3(vec_grid(n)), dim3(kBlock), 0, s, d, n);
  MFX_HIP(hipGetLastError());
}
void launch_random(double *x, uint64_t n, uint64_t seed, hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_random, dim3(vec_grid(n)), dim3(kBlock), 0, s, x, n, seed);
  MFX_HIP(hipGetLastError());
}
void launch_gather(const uint32_t *map, uint64_t n, const double *src, double *evec,
                   hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_gather, dim3(vec_grid(n)), dim3(kBlock), 0, s, map, n, src, evec);
  MFX_HIP(hipGetLastError());
}
void launch_scatter_add(const uint32_t *map, uint64_t n, const double *evec, double *dst,
                        hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_scatter_add, dim3(vec_grid(n)), dim3(kBlock), 0, s, map, n, evec, dst);
  MFX_HIP(hipGetLastError());
}
void launch_sine_modes(const double *xyz, uint64_t n, const SineModes &m, double *out,
                       hipStream_t s) {
  MFX_REQUIRE(m.n >= 0 && m.n <= SineModes::kMax, "sine modes: count out of range");
  if (!n) return;
  hipLaunchKernelGGL(k_sine_modes, dim3(vec_grid(n)), dim3(kBlock), 0, s, xyz, n, m, out);
  MFX_HIP(hipGetLastError());
}
uint32_t dot_n_blocks(uint64_t n) { return vec_grid(n); }
void launch_dot(const double *x, const double *y, uint64_t n, double *partials, double *result,
                hipStream_t s) {
  const unsigned g = vec_grid(n);
  hipLaunchKernelGGL(k_dot_partials, dim3(g), dim3(kBlock), 0, s, x, y, n, partials);
  hipLaunchKernelGGL(k_dot_final, dim3(1), dim3(kBlock), 0, s, partials, g, result);
  MFX_HIP(hipGetLastError());
}

void launch_sum(const double *part, uint32_t n, double *result, hipStream_t s) {
  hipLaunchKernelGGL(k_dot_final, dim3(1), dim3(kBlock), 0, s, part, n, result);
  MFX_HIP(hipGetLastError());
}

// ---- CG launchers ----
uint32_t cg_vec_blocks(uint64_t n) { return vec_grid(n); }
uint32_t cg_cons_blocks(uint64_t nc) { return nc ? std::min<uint32_t>(vec_grid(nc), 256) : 0; }

void cg_init(CgState *st, const double *b, double *r, const double *invd, uint64_t n,
             double *part, double abs_tol, double rel_tol, int max_steps, hipStream_t s) {
  const unsigned g = vec_grid(n);
  hipLaunchKernelGGL(k_cg_init, dim3(g), dim3(kBlock), 0, s, st, b, r, invd, n, part);
  hipLaunchKernelGGL(k_cg_start, dim3(1), dim3(kBlock), 0, s, st, part, g, abs_tol, rel_tol,
                     max_steps);
  MFX_HIP(hipGetLastError());
}
void cg_direction(const CgState *st, const double *r, const double *invd, double *p, double *ap,
                  double *x, uint64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_cg_direction, dim3(vec_grid(n)), dim3(kBlock), 0, s, st, r, invd, p, ap, x,
                     n);
}
void cg_test(const CgState *sa, CgState *sb, const double *part, uint64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_cg_test, dim3(1), dim3(kBlock), 0, s, sa, sb, part, vec_grid(n));
}
void cg_direction_small(const CgState *sa, CgState *sb, const double *part, bool first,
                        const double *r, const double *invd, const uint32_t *mask, double *p,
                        double *ap, double *x, double *part_c, uint64_t n, hipStream_t s) {
  const unsigned g = vec_grid(n);
  MFX_REQUIRE((uint64_t)g * kBlock * kRows >= n, "small CG step: too many rows");
  if (first)
    hipLaunchKernelGGL(k_cg_direction_small<true>, dim3(g), dim3(kBlock), 0, s, sa, sb, part, g, r,
                       invd, mask, p, ap, x, part_c, n);
  else
    hipLaunchKernelGGL(k_cg_direction_small<false>, dim3(g), dim3(kBlock), 0, s, sa, sb, part, g,
                       r, invd, mask, p, ap, x, part_c, n);
}
void cg_update_small(const CgState *sb, CgState *sa, const double *pap, uint32_t n_pap, double *r,
                     const double *ap, const double *invd, uint64_t n, double *part,
                     hipStream_t s) {
  hipLaunchKernelGGL(k_cg_update_small, dim3(vec_grid(n)), dim3(kBlock), 0, s, sb, sa, pap, n_pap,
                     r, ap, invd, n, part);
}
void cg_finish(const CgState *st, const CgState *sa, double *x, const double *p, uint64_t n,
               hipStream_t s) {
  hipLaunchKernelGGL(k_cg_finish, dim3(vec_grid(n)), dim3(kBlock), 0, s, st, sa, x, p, n);
  MFX_HIP(hipGetLastError());
}
void cg_constrained(const CgState *st, const uint32_t *list, uint64_t nc, const double *p,
                    double *ap, double *part, hipStream_t s) {
  if (!nc) return;
  hipLaunchKernelGGL(k_cg_constrained, dim3(cg_cons_blocks(nc)), dim3(kBlock), 0, s, st, list,
                     nc, p, ap, part);
}
// More partials than one workgroup sums quickly (the cell-wise Gauss apply
// writes one per workgroup: ~1.6e5 at 67M DoFs, 0.23 ms in k_cg_alpha
// alone): chunks of kAlphaChunk are summed in parallel first, each in a
// fixed order, into the slots after the partials, and alpha sums those.
constexpr uint32_t kAlphaDirect = 4096, kAlphaChunk = 2048;
uint32_t cg_alpha_extra(uint32_t n) {
  return n > kAlphaDirect ? (n + kAlphaChunk - 1) / kAlphaChunk : 0;
}
void cg_alpha(CgState *st, double *part, uint32_t n, hipStream_t s) {
  const uint32_t r = cg_alpha_extra(n);
  if (r) {
    hipLaunchKernelGGL(k_cg_chunks, dim3(r), dim3(kBlock), 0, s, st, part, n, kAlphaChunk,
                       part + n);
    hipLaunchKernelGGL(k_cg_alpha, dim3(1), dim3(kBlock), 0, s, st, part + n, r);
  } else {
    hipLaunchKernelGGL(k_cg_alpha, dim3(1), dim3(kBlock), 0, s, st, part, n);
  }
}
void cg_update(const CgState *st, double *r, const double *ap, const double *invd, uint64_t n,
               double *part, hipStream_t s) {
  hipLaunchKernelGGL(k_cg_update, dim3(vec_grid(n)), dim3(kBlock), 0, s, st, r, ap, invd, n, part);
}
void cg_check(CgState *st, const double *part, uint32_t nb, hipStream_t s) {
  hipLaunchKernelGGL(k_cg_check, dim3(1), dim3(kBlock), 0, s, st, part, nb);
}

}  // namespace mfx
