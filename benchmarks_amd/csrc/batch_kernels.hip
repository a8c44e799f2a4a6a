// batch_kernels.hip -- vector and scalar steps of the batched CG: many
// independent problems concatenated into one DoF vector, each with its own
// CG scalars and convergence state.
//
// Vector kernels run one workgroup per segment (a contiguous range inside
// one instance), skip segments of converged instances, and write one partial
// per segment.  Their segment loops are unrolled by 4 so that each thread has
// several independent loads in flight.  The scalar kernels run one workgroup per instance, which sums
// that instance's segment partials in a fixed order, so every reduction is
// deterministic.
#include <algorithm>

#include "batch.hpp"
#include "mfx_internal.hpp"
#include "tables.hpp"

namespace mfx {
namespace {

constexpr int kBlock = 256;

template <int BLOCK = kBlock>
__device__ __forceinline__ void block_sum2(double &a, double &b) {
  __shared__ double ra[BLOCK / 64], rb[BLOCK / 64];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    a += __shfl_xor(a, o, 64);
    b += __shfl_xor(b, o, 64);
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) {
    ra[w] = a;
    rb[w] = b;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double sa = 0.0, sb = 0.0;
#pragma unroll
    for (int i = 0; i < BLOCK / 64; ++i) {
      sa += ra[i];
      sb += rb[i];
    }
    a = sa;
    b = sb;
  }
}

__global__ void __launch_bounds__(kBlock)
k_b_residual(const Seg *__restrict__ segs, double *__restrict__ r, const double *__restrict__ b,
             const double *__restrict__ t, const double *__restrict__ dinv,
             double *__restrict__ part_rr, double *__restrict__ part_rz) {
  const Seg sg = segs[blockIdx.x];
  double rr = 0.0, rz = 0.0;
#pragma unroll 4
  for (uint64_t i = sg.begin + threadIdx.x; i < sg.end; i += kBlock) {
    const double v = b[i] - t[i];
    r[i] = v;
    rr += v * v;
    rz += v * dinv[i] * v;
  }
  block_sum2(rr, rz);
  if (threadIdx.x == 0) {
    part_rr[blockIdx.x] = rr;
    part_rz[blockIdx.x] = rz;
  }
}

// Sums of an instance's segment partials: one workgroup per instance,
// threads stride over the segments, fixed-order tree within the workgroup.
__device__ __forceinline__ void instance_sums(const uint32_t *__restrict__ inst_seg, uint32_t i,
                                              const double *__restrict__ pa,
                                              const double *__restrict__ pb, double &a,
                                              double &b) {
  a = 0.0;
  b = 0.0;
  for (uint32_t k = inst_seg[i] + threadIdx.x; k < inst_seg[i + 1]; k += kBlock) {
    a += pa[k];
    if (pb) b += pb[k];
  }
  block_sum2(a, b);  // valid in thread 0
}

__global__ void __launch_bounds__(kBlock)
k_b_init(BatchCg *__restrict__ st, const uint32_t *__restrict__ inst_seg,
         const double *__restrict__ part_rr, const double *__restrict__ part_rz, double abs_tol,
         double rel_tol, int max_steps, int *__restrict__ flags) {
  const uint32_t i = blockIdx.x;
  double rr, rz;
  instance_sums(inst_seg, i, part_rr, part_rz, rr, rz);
  if (threadIdx.x == 0) {
    BatchCg c{};
    c.initial = sqrt(rr);
    c.last = c.initial;
    c.tol = fmax(abs_tol, rel_tol * c.initial);
    c.gamma = rz;
    c.max_steps = max_steps;
    c.first = 1;
    if (c.initial <= c.tol) {
      c.done = 1;
      c.converged = 1;
    } else if (max_steps <= 0) {
      c.done = 1;
    }
    st[i] = c;
    flags[i] = c.done;
  }
}

// number of instances still iterating
__global__ void __launch_bounds__(kBlock)
k_b_count(const int *__restrict__ flags, uint32_t n_inst, int *__restrict__ n_active) {
  double a = 0.0, unused = 0.0;
  for (uint32_t i = threadIdx.x; i < n_inst; i += kBlock) a += flags[i] ? 0.0 : 1.0;
  block_sum2(a, unused);
  if (threadIdx.x == 0) *n_active = (int)a;
}

// x += alpha p of the previous step (it needs the p read here anyway), then
// p = dinv r + beta p; ap = 0 on the free rows (the apply accumulates
// there) and ap = p on the constrained rows (the identity rows of the
// operator), whose share of p.ap, the sum of p^2 over them, goes to one
// partial per segment
__global__ void __launch_bounds__(kBlock)
k_b_direction(const Seg *__restrict__ segs, const BatchCg *__restrict__ st,
              const double *__restrict__ r, const double *__restrict__ dinv,
              const uint8_t *__restrict__ cmask, double *__restrict__ p, double *__restrict__ ap,
              double *__restrict__ x, double *__restrict__ part_c) {
  const Seg sg = segs[blockIdx.x];
  const BatchCg &c = st[sg.inst];
  if (c.done) return;
  const bool first = c.first != 0;
  const double beta = first ? 0.0 : c.beta, alpha = c.alpha;
  double pc = 0.0, unused = 0.0;
#pragma unroll 4
  for (uint64_t i = sg.begin + threadIdx.x; i < sg.end; i += kBlock) {
    const double pi = p[i];
    if (!first) x[i] += alpha * pi;
    const double pn = dinv[i] * r[i] + (beta != 0.0 ? beta * pi : 0.0);
    p[i] = pn;
    const bool cons = cmask[i] != 0;
    ap[i] = cons ? pn : 0.0;
    pc += cons ? pn * pn : 0.0;
  }
  block_sum2(pc, unused);
  if (threadIdx.x == 0) part_c[blockIdx.x] = pc;
}

// the last step's x += alpha p of every instance that took a step
__global__ void __launch_bounds__(kBlock)
k_b_finish(const Seg *__restrict__ segs, const BatchCg *__restrict__ st, double *__restrict__ x,
           const double *__restrict__ p) {
  const Seg sg = segs[blockIdx.x];
  const BatchCg &c = st[sg.inst];
  if (c.steps == 0) return;
  const double alpha = c.alpha;
#pragma unroll 4
  for (uint64_t i = sg.begin + threadIdx.x; i < sg.end; i += kBlock) x[i] += alpha * p[i];
}

__global__ void __launch_bounds__(kBlock)
k_b_pap(const Seg *__restrict__ segs, const BatchCg *__restrict__ st,
        const double *__restrict__ p, const double *__restrict__ ap, double *__restrict__ part) {
  const Seg sg = segs[blockIdx.x];
  if (st[sg.inst].done) return;
  double s = 0.0, unused = 0.0;
#pragma unroll 4
  for (uint64_t i = sg.begin + threadIdx.x; i < sg.end; i += kBlock) s += p[i] * ap[i];
  block_sum2(s, unused);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ void __launch_bounds__(kBlock)
k_b_alpha(BatchCg *__restrict__ st, const uint32_t *__restrict__ inst_seg,
          const double *__restrict__ part) {
  const uint32_t i = blockIdx.x;
  if (st[i].done) return;
  double pap, unused;
  instance_sums(inst_seg, i, part, nullptr, pap, unused);
  if (threadIdx.x == 0) {
    BatchCg &c = st[i];
    if (!(pap > 0.0)) {
      c.breakdown = 1;
      c.alpha = 0.0;
    } else {
      c.alpha = c.gamma / pap;
    }
  }
}

__global__ void __launch_bounds__(kBlock)
k_b_alpha_fused(BatchCg *__restrict__ st, const PapRange *__restrict__ ranges,
                const uint32_t *__restrict__ inst_seg, const double *__restrict__ part_c) {
  const uint32_t i = blockIdx.x;
  if (st[i].done) return;
  const PapRange rg = ranges[i];
  double a = 0.0, b = 0.0;
  for (uint64_t k = threadIdx.x; k < rg.n; k += kBlock) {
    a += rg.part[k];
    rg.part[k] = 0.0;  // the patch kernel writes only the slots it uses
  }
  for (uint32_t k = inst_seg[i] + threadIdx.x; k < inst_seg[i + 1]; k += kBlock) b += part_c[k];
  block_sum2(a, b);
  if (threadIdx.x == 0) {
    BatchCg &c = st[i];
    const double pap = a + b;
    if (!(pap > 0.0)) {
      c.breakdown = 1;
      c.alpha = 0.0;
    } else {
      c.alpha = c.gamma / pap;
    }
  }
}

// r -= alpha ap (x += alpha p follows in the next direction pass or k_b_finish)
__global__ void __launch_bounds__(kBlock)
k_b_update(const Seg *__restrict__ segs, const BatchCg *__restrict__ st, double *__restrict__ r,
           const double *__restrict__ ap, const double *__restrict__ dinv,
           double *__restrict__ part_rr, double *__restrict__ part_rz) {
  const Seg sg = segs[blockIdx.x];
  const BatchCg &c = st[sg.inst];
  if (c.done) return;
  const double alpha = c.alpha;
  double rr = 0.0, rz = 0.0;
#pragma unroll 4
  for (uint64_t i = sg.begin + threadIdx.x; i < sg.end; i += kBlock) {
    const double v = r[i] - alpha * ap[i];
    r[i] = v;
    rr += v * v;
    rz += v * dinv[i] * v;
  }
  block_sum2(rr, rz);
  if (threadIdx.x == 0) {
    part_rr[blockIdx.x] = rr;
    part_rz[blockIdx.x] = rz;
  }
}

// the state after a step whose new residual has the sums rr and rz
__device__ __forceinline__ BatchCg next_state(BatchCg c, double rr, double rz) {
  c.steps += 1;
  c.last = sqrt(rr);
  if (c.breakdown) {
    c.done = 1;
  } else if (c.last <= c.tol) {
    c.done = 1;
    c.converged = 1;
  } else if (c.steps >= c.max_steps) {
    c.done = 1;
  } else {
    c.beta = rz / c.gamma;
    c.gamma = rz;
    c.first = 0;
  }
  return c;
}

// from state sa to sb, which may be the same
__global__ void __launch_bounds__(kBlock)
k_b_check(const BatchCg *sa, BatchCg *sb, const uint32_t *__restrict__ inst_seg,
          const double *__restrict__ part_rr, const double *__restrict__ part_rz,
          int *__restrict__ flags) {
  const uint32_t i = blockIdx.x;
  if (sa[i].done) {
    if (threadIdx.x == 0 && sa != sb) sb[i] = sa[i];
    return;
  }
  double rr, rz;
  instance_sums(inst_seg, i, part_rr, part_rz, rr, rz);
  if (threadIdx.x == 0) {
    const BatchCg c = next_state(sa[i], rr, rz);
    sb[i] = c;
    flags[i] = c.done;
  }
}

// ---- a step of a small batch in three launches ----
//
// Where a step is a few microseconds of work, launches bound it: direction,
// one apply per degree, p.Ap, alpha, update, check and count take 3-23 us each
// (16 problems of degrees 2..6, 1.1M DoFs: 73 us per step, 37 in this form).  Here the vector
// passes run on segments of kSegSmall rows, four per thread and all loaded
// before anything waits, every workgroup sums its instance's partials itself in
// place of the alpha and check launches, and one launch applies the operators
// of all degrees and sums p.Ap.  The states alternate between two arrays: the
// workgroups of the direction pass read one while the instance's first
// segment writes the other.

constexpr int kRows = kSegSmall / kBlock;
constexpr int kTile = 256;  // threads of a tile

__device__ __forceinline__ void cross(const double (&a)[3], const double (&b)[3], double (&c)[3]) {
  c[0] = a[1] * b[2] - a[2] * b[1];
  c[1] = a[2] * b[0] - a[0] * b[2];
  c[2] = a[0] * b[1] - a[1] * b[0];
}

// a and b summed over the workgroup, for every thread
__device__ __forceinline__ void block_sum2_all(double &a, double &b) {
  __shared__ double ra[kBlock / 64], rb[kBlock / 64];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    a += __shfl_xor(a, o, 64);
    b += __shfl_xor(b, o, 64);
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) {
    ra[w] = a;
    rb[w] = b;
  }
  __syncthreads();
  a = b = 0.0;
#pragma unroll
  for (int i = 0; i < kBlock / 64; ++i) {
    a += ra[i];
    b += rb[i];
  }
}

// As k_b_check (not on a round's first step, whose state k_b_check or k_b_init
// left), then as k_b_direction.
template <bool CHECK>
__global__ void __launch_bounds__(kBlock)
k_b_direction_small(const Seg *__restrict__ segs, const BatchCg *sa, BatchCg *sb,
                    const uint32_t *__restrict__ inst_seg, const double *__restrict__ part_rr,
                    const double *__restrict__ part_rz, const double *__restrict__ r,
                    const double *__restrict__ dinv, const uint8_t *__restrict__ cmask,
                    double *__restrict__ p, double *__restrict__ ap, double *__restrict__ x,
                    double *__restrict__ part_c, int *__restrict__ flags) {
  const Seg sg = segs[blockIdx.x];
  const uint32_t s0 = inst_seg[sg.inst], s1 = inst_seg[sg.inst + 1];
  const bool lead = blockIdx.x == s0 && threadIdx.x == 0;
  const BatchCg *c = sa + sg.inst;
  if (c->done) {
    if (CHECK && lead) sb[sg.inst] = *c;
    return;
  }
  double z[kRows], pv[kRows], xv[kRows];
  bool cons[kRows];
#pragma unroll
  for (int k = 0; k < kRows; ++k) {
    const uint64_t i = sg.begin + threadIdx.x + k * kBlock;
    z[k] = pv[k] = xv[k] = 0.0;
    cons[k] = false;
    if (i >= sg.end) continue;
    z[k] = dinv[i] * r[i];
    pv[k] = p[i];
    xv[k] = x[i];
    cons[k] = cmask[i] != 0;
  }
  const double alpha = c->alpha;
  double beta = c->beta;
  bool first = c->first != 0;
  if constexpr (CHECK) {
    double rr = 0.0, rz = 0.0;
    for (uint32_t k = s0 + threadIdx.x; k < s1; k += kBlock) {
      rr += part_rr[k];
      rz += part_rz[k];
    }
    block_sum2_all(rr, rz);
    const BatchCg n = next_state(*c, rr, rz);
    if (lead) {
      sb[sg.inst] = n;
      flags[sg.inst] = n.done;
    }
    if (n.done) return;
    beta = n.beta;
    first = false;
  }
  if (first) beta = 0.0;
  double pc = 0.0, unused = 0.0;
#pragma unroll
  for (int k = 0; k < kRows; ++k) {
    const uint64_t i = sg.begin + threadIdx.x + k * kBlock;
    if (i >= sg.end) continue;
    if (!first) x[i] = xv[k] + alpha * pv[k];
    const double pn = z[k] + (beta != 0.0 ? beta * pv[k] : 0.0);
    p[i] = pn;
    ap[i] = cons[k] ? pn : 0.0;
    pc += cons[k] ? pn * pn : 0.0;
  }
  block_sum2(pc, unused);
  if (threadIdx.x == 0) part_c[blockIdx.x] = pc;
}

// As k_b_alpha (p.Ap from the tiles' partials and the constrained rows'), then
// as k_b_update.
__global__ void __launch_bounds__(kBlock)
k_b_update_small(const Seg *__restrict__ segs, BatchCg *st, const uint32_t *__restrict__ inst_seg,
                 const uint32_t *__restrict__ inst_tile, const double *__restrict__ part_t,
                 const double *__restrict__ part_c, double *__restrict__ r,
                 const double *__restrict__ ap, const double *__restrict__ dinv,
                 double *__restrict__ part_rr, double *__restrict__ part_rz) {
  const Seg sg = segs[blockIdx.x];
  if (st[sg.inst].done) return;
  const uint32_t s0 = inst_seg[sg.inst], s1 = inst_seg[sg.inst + 1];
  const uint32_t t0 = inst_tile[sg.inst], t1 = inst_tile[sg.inst + 1];
  double rv[kRows], av[kRows], dv[kRows];
#pragma unroll
  for (int k = 0; k < kRows; ++k) {
    const uint64_t i = sg.begin + threadIdx.x + k * kBlock;
    rv[k] = av[k] = dv[k] = 0.0;
    if (i >= sg.end) continue;
    rv[k] = r[i];
    av[k] = ap[i];
    dv[k] = dinv[i];
  }
  double pt = 0.0, pc = 0.0;
  for (uint32_t k = t0 + threadIdx.x; k < t1; k += kBlock) pt += part_t[k];
  for (uint32_t k = s0 + threadIdx.x; k < s1; k += kBlock) pc += part_c[k];
  const double gamma = st[sg.inst].gamma;
  block_sum2_all(pt, pc);
  const double pap = pt + pc;
  const bool ok = pap > 0.0;
  const double alpha = ok ? gamma / pap : 0.0;
  if (blockIdx.x == s0 && threadIdx.x == 0) {  // no workgroup of this launch reads these
    st[sg.inst].alpha = alpha;
    if (!ok) st[sg.inst].breakdown = 1;
  }
  double rr = 0.0, rz = 0.0;
#pragma unroll
  for (int k = 0; k < kRows; ++k) {
    const uint64_t i = sg.begin + threadIdx.x + k * kBlock;
    if (i >= sg.end) continue;
    const double v = rv[k] - alpha * av[k];
    r[i] = v;
    rr += v * v;
    rz += v * dv[k] * v;
  }
  block_sum2(rr, rz);
  if (threadIdx.x == 0) {
    part_rr[blockIdx.x] = rr;
    part_rz[blockIdx.x] = rz;
  }
}

// One tile (batch_tile_cells(p) consecutive cells of one instance) of the
// batched apply: one thread per (x, y) column of a cell.  x and y contractions
// run on whole lines in the LDS (each operand is read once) with the even-odd
// split and the derivative matrix as compile-time constants, z contractions in
// registers; the metric comes from the cell's vertices, the rows from the box.
// Faces between cells of a mesh row are summed in the LDS and consecutive
// lanes add consecutive rows: adding each cell's columns through the DoF map took
// 28 us against 20 on 16 problems of 1.8M points (19 without its adds).  On the
// same points: metric terms stored and contractions per point 31 us (30 with the
// metric from the vertices, so its bytes were not the bound), one launch per
// degree with the tuned kernels 35 us.  128 threads instead of 256 (shorter rows)
// 23 us.  What is left at the one problem that takes the most steps (0.49M rows,
// 12 us) is a launch and its chain of loads, four barriers and adds.
template <int NQ>
struct TileCfg {
  static constexpr int NQ2 = NQ * NQ, EPB = kTile / NQ2;
  // an odd row stride spreads the lanes of x-line accesses over the banks
  static constexpr int RS = NQ | 1, PS = RS * NQ, CS = PS * NQ, LDS = 3 * EPB * CS;
};
// boundary bits of a cell (its mesh faces) and whether its x neighbours are in the tile
constexpr uint32_t kX0 = 1, kX1 = 2, kY0 = 4, kY1 = 8, kZ0 = 16, kZ1 = 32, kLeft = 64, kRight = 128;

template <int NQ>
__device__ __forceinline__ void
tile_apply(double *__restrict__ lds, uint2 *__restrict__ info, const BatchTile &m,
           const BatchTiles::Degree &t, const double *__restrict__ src, double *__restrict__ dst,
           double &dot) {
  using C = TileCfg<NQ>;
  constexpr int P = NQ - 1, NQ2 = C::NQ2, EPB = C::EPB, RS = C::RS, PS = C::PS;
  constexpr GllD<NQ> kD{};
  auto dm = [&](int i, int a) { return kD.D[i][a]; };
  auto dmt = [&](int i, int a) { return kD.D[a][i]; };
  const int el = threadIdx.x / NQ2, col = threadIdx.x - el * NQ2;
  const int l0 = col % NQ, l1 = col / NQ;
  const bool active = (uint32_t)el < m.n;  // m.n <= EPB
  double *su = lds + (active ? el : 0) * C::CS, *A = su + EPB * C::CS, *B = A + EPB * C::CS;
  const int xline = l0 * RS + l1 * PS;  // y = l0, z = l1
  const int yline = l0 + l1 * PS;       // x = l0, z = l1
  const int zline = l0 + l1 * RS;       // x = l0, y = l1: the thread's column
  const uint32_t NX = m.n0 * P + 1, NXY = NX * (m.n1 * P + 1);
  double u[NQ], ln[NQ], r[NQ], vz[NQ];
  // the column's Jacobian: J0 = a0 + zeta da, J1 = b0 + zeta db, J2 = jz
  double a0[3], da[3], b0[3], db[3], jz[3], wxy = 0.0;
  if (active) {
    const double *X = t.cellX + (size_t)(m.cell + el) * 24;  // vertex v, coordinate d at X[3v + d]
    const uint32_t e = m.first + el, ex = e % m.n0, ey = e / m.n0 % m.n1, ez = e / m.n0 / m.n1;
    const uint32_t base = m.off + ez * P * NXY + ey * P * NX + ex * P;
    const uint32_t bits = (ex == 0 ? kX0 : 0) | (ex + 1 == m.n0 ? kX1 : 0) | (ey == 0 ? kY0 : 0) |
                          (ey + 1 == m.n1 ? kY1 : 0) | (ez == 0 ? kZ0 : 0) |
                          (ez + 1 == m.n2 ? kZ1 : 0) | (ex > 0 && el > 0 ? kLeft : 0) |
                          (ex + 1 < m.n0 && (uint32_t)el + 1 < m.n ? kRight : 0);
    const bool in = !((l0 == 0 && bits & kX0) || (l0 == P && bits & kX1) ||
                      (l1 == 0 && bits & kY0) || (l1 == P && bits & kY1));
    const double *sc = src + base + l1 * NX + l0;
#pragma unroll
    for (int z = 0; z < NQ; ++z)
      u[z] = in && !(z == 0 && bits & kZ0) && !(z == P && bits & kZ1) ? sc[z * NXY] : 0.0;
    if (col == 0) info[el] = uint2{base, bits};
    const double xi = t.xq[l0], eta = t.xq[l1];
    wxy = t.w[l0] * t.w[l1];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double k0 = X[12 + d] - X[d], k1 = X[15 + d] - X[3 + d], k2 = X[18 + d] - X[6 + d],
                   k3 = X[21 + d] - X[9 + d];
      const double e = X[3 + d] - X[d], f = X[6 + d] - X[d];
      const double ef = (X[9 + d] - X[6 + d]) - e;
      a0[d] = e + eta * ef;
      b0[d] = f + xi * ef;
      da[d] = (k1 - k0) + eta * ((k3 - k2) - (k1 - k0));
      db[d] = (k2 - k0) + xi * ((k3 - k2) - (k1 - k0));
      jz[d] = (1 - xi) * (1 - eta) * k0 + xi * (1 - eta) * k1 + (1 - xi) * eta * k2 +
              xi * eta * k3;
    }
#pragma unroll
    for (int z = 0; z < NQ; ++z) su[zline + z * PS] = u[z];
  }
  __syncthreads();
  if (active) {
#pragma unroll
    for (int a = 0; a < NQ; ++a) ln[a] = su[xline + a];
    eo_mat<NQ, NQ, -1>(dm, ln, r);
#pragma unroll
    for (int a = 0; a < NQ; ++a) A[xline + a] = r[a];
#pragma unroll
    for (int a = 0; a < NQ; ++a) ln[a] = su[yline + a * RS];
    eo_mat<NQ, NQ, -1>(dm, ln, r);
#pragma unroll
    for (int a = 0; a < NQ; ++a) B[yline + a * RS] = r[a];
  }
  __syncthreads();
  if (active) {
    double dz[NQ], fz[NQ];
    eo_mat<NQ, NQ, -1>(dm, u, dz);
#pragma unroll
    for (int z = 0; z < NQ; ++z) {
      const double gx = A[zline + z * PS], gy = B[zline + z * PS];
      const double zeta = t.xq[z];
      double J0[3], J1[3], C0[3], C1[3], C2[3], W[3];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        J0[d] = a0[d] + zeta * da[d];
        J1[d] = b0[d] + zeta * db[d];
      }
      cross(J1, jz, C0);
      cross(jz, J0, C1);
      cross(J0, J1, C2);
      const double det = jz[0] * C2[0] + jz[1] * C2[1] + jz[2] * C2[2];
      const double sc = wxy * t.w[z] * recip(det);
#pragma unroll
      for (int d = 0; d < 3; ++d) W[d] = sc * (gx * C0[d] + gy * C1[d] + dz[z] * C2[d]);
      const double fx = C0[0] * W[0] + C0[1] * W[1] + C0[2] * W[2];
      const double fy = C1[0] * W[0] + C1[1] * W[1] + C1[2] * W[2];
      fz[z] = C2[0] * W[0] + C2[1] * W[1] + C2[2] * W[2];
      A[zline + z * PS] = fx;
      B[zline + z * PS] = fy;
      // p.Ap as the cells' energies: u is 0 on the constrained rows
      dot += gx * fx + gy * fy + dz[z] * fz[z];
    }
    eo_mat<NQ, NQ, -1>(dmt, fz, vz);
  }
  __syncthreads();
  if (active) {
#pragma unroll
    for (int a = 0; a < NQ; ++a) ln[a] = A[xline + a];
    eo_mat<NQ, NQ, -1>(dmt, ln, r);
#pragma unroll
    for (int a = 0; a < NQ; ++a) A[xline + a] = r[a];
#pragma unroll
    for (int a = 0; a < NQ; ++a) ln[a] = B[yline + a * RS];
    eo_mat<NQ, NQ, -1>(dmt, ln, r);
#pragma unroll
    for (int a = 0; a < NQ; ++a) B[yline + a * RS] = r[a];
  }
  __syncthreads();
  if (active) {
#pragma unroll
    for (int z = 0; z < NQ; ++z) su[zline + z * PS] = A[zline + z * PS] + B[zline + z * PS] + vz[z];
  }
  __syncthreads();
  // one lane per (cell, x) of a mesh line, all lines of the tile
#pragma unroll
  for (int k = 0; k < (EPB * NQ * NQ2 + kTile - 1) / kTile; ++k) {
    const int i = threadIdx.x + k * kTile;
    const int line = i / (EPB * NQ), c = i % (EPB * NQ) / NQ, x = i % NQ;
    const int y = line % NQ, z = line / NQ;
    if (line >= NQ2 || (uint32_t)c >= m.n) continue;
    const uint2 f = info[c];
    if ((x == 0 && f.y & kX0) || (x == P && f.y & (kX1 | kRight)) || (y == 0 && f.y & kY0) ||
        (y == P && f.y & kY1) || (z == 0 && f.y & kZ0) || (z == P && f.y & kZ1))
      continue;
    const double *v = lds + c * C::CS + z * PS + y * RS;
    double s = v[x];
    if (x == 0 && f.y & kLeft) s += v[P - C::CS];
    unsafeAtomicAdd(dst + f.x + z * NXY + y * NX + x, s);
  }
}

constexpr int kTileLds = std::max({TileCfg<3>::LDS, TileCfg<4>::LDS, TileCfg<5>::LDS,
                                   TileCfg<6>::LDS, TileCfg<7>::LDS});

__global__ void __launch_bounds__(kTile)
k_b_apply(BatchTiles t, const double *__restrict__ src, double *__restrict__ dst,
          const int *__restrict__ done, double *__restrict__ part) {
  __shared__ double lds[kTileLds];
  __shared__ uint2 info[TileCfg<3>::EPB];
  const BatchTile m = t.tiles[blockIdx.x];
  if (done[m.inst]) return;
  const BatchTiles::Degree &g = t.degree[m.p - 2];
  double dot = 0.0, unused = 0.0;
  switch (m.p) {
    case 2: tile_apply<3>(lds, info, m, g, src, dst, dot); break;
    case 3: tile_apply<4>(lds, info, m, g, src, dst, dot); break;
    case 4: tile_apply<5>(lds, info, m, g, src, dst, dot); break;
    case 5: tile_apply<6>(lds, info, m, g, src, dst, dot); break;
    default: tile_apply<7>(lds, info, m, g, src, dst, dot); break;
  }
  block_sum2<kTile>(dot, unused);
  if (threadIdx.x == 0) part[blockIdx.x] = dot;
}

__global__ void k_offset_map(const uint32_t *__restrict__ src, uint32_t *__restrict__ dst,
                             uint64_t n, uint32_t offset) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t v = src[i];
    dst[i] = v == kInvalid ? kInvalid : v + offset;
  }
}

__global__ void k_fill_u16(uint16_t *__restrict__ dst, uint16_t v, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    dst[i] = v;
}

__global__ void k_mark_u8(const uint32_t *__restrict__ list, uint64_t n, uint8_t *__restrict__ mask) {
  for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n;
       k += (uint64_t)gridDim.x * blockDim.x)
    mask[list[k]] = 1;
}

inline unsigned grid_for(uint64_t n) {
  return (unsigned)std::max<uint64_t>(1, std::min<uint64_t>((n + kBlock - 1) / kBlock, 65536));
}

}  // namespace

void launch_b_residual(const Seg *segs, uint32_t n_segs, double *r, const double *b,
                       const double *t, const double *dinv, double *part_rr, double *part_rz,
                       hipStream_t s) {
  if (!n_segs) return;
  hipLaunchKernelGGL(k_b_residual, dim3(n_segs), dim3(kBlock), 0, s, segs, r, b, t, dinv,
                     part_rr, part_rz);
  MFX_HIP(hipGetLastError());
}

void launch_b_init(BatchCg *st, const uint32_t *inst_seg, uint32_t n_inst, const double *part_rr,
                   const double *part_rz, double abs_tol, double rel_tol, int max_steps,
                   int *flags, int *n_active, hipStream_t s) {
  hipLaunchKernelGGL(k_b_init, dim3(n_inst), dim3(kBlock), 0, s, st, inst_seg, part_rr, part_rz,
                     abs_tol, rel_tol, max_steps, flags);
  hipLaunchKernelGGL(k_b_count, dim3(1), dim3(kBlock), 0, s, flags, n_inst, n_active);
  MFX_HIP(hipGetLastError());
}

void launch_b_direction(const Seg *segs, uint32_t n_segs, const BatchCg *st, const double *r,
                        const double *dinv, const uint8_t *cmask, double *p, double *ap, double *x,
                        double *part_c, hipStream_t s) {
  if (!n_segs) return;
  hipLaunchKernelGGL(k_b_direction, dim3(n_segs), dim3(kBlock), 0, s, segs, st, r, dinv, cmask, p,
                     ap, x, part_c);
  MFX_HIP(hipGetLastError());
}

void launch_b_finish(const Seg *segs, uint32_t n_segs, const BatchCg *st, double *x,
                     const double *p, hipStream_t s) {
  if (!n_segs) return;
  hipLaunchKernelGGL(k_b_finish, dim3(n_segs), dim3(kBlock), 0, s, segs, st, x, p);
  MFX_HIP(hipGetLastError());
}

void launch_b_pap(const Seg *segs, uint32_t n_segs, const BatchCg *st, const double *p,
                  const double *ap, double *part, hipStream_t s) {
  if (!n_segs) return;
  hipLaunchKernelGGL(k_b_pap, dim3(n_segs), dim3(kBlock), 0, s, segs, st, p, ap, part);
  MFX_HIP(hipGetLastError());
}

void launch_b_alpha(BatchCg *st, const uint32_t *inst_seg, uint32_t n_inst, const double *part,
                    hipStream_t s) {
  hipLaunchKernelGGL(k_b_alpha, dim3(n_inst), dim3(kBlock), 0, s, st, inst_seg, part);
  MFX_HIP(hipGetLastError());
}

void launch_b_alpha_fused(BatchCg *st, const PapRange *ranges, const uint32_t *inst_seg,
                          uint32_t n_inst, const double *part_c, hipStream_t s) {
  hipLaunchKernelGGL(k_b_alpha_fused, dim3(n_inst), dim3(kBlock), 0, s, st, ranges, inst_seg,
                     part_c);
  MFX_HIP(hipGetLastError());
}

void launch_mark_u8(const uint32_t *list, uint64_t n, uint8_t *mask, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_mark_u8, dim3(grid_for(n)), dim3(kBlock), 0, s, list, n, mask);
  MFX_HIP(hipGetLastError());
}

void launch_b_update(const Seg *segs, uint32_t n_segs, const BatchCg *st, double *r,
                     const double *ap, const double *dinv, double *part_rr, double *part_rz,
                     hipStream_t s) {
  if (!n_segs) return;
  hipLaunchKernelGGL(k_b_update, dim3(n_segs), dim3(kBlock), 0, s, segs, st, r, ap, dinv, part_rr,
                     part_rz);
  MFX_HIP(hipGetLastError());
}

void launch_b_check(const BatchCg *sa, BatchCg *sb, const uint32_t *inst_seg, uint32_t n_inst,
                    const double *part_rr, const double *part_rz, int *flags, int *n_active,
                    hipStream_t s) {
  hipLaunchKernelGGL(k_b_check, dim3(n_inst), dim3(kBlock), 0, s, sa, sb, inst_seg, part_rr,
                     part_rz, flags);
  hipLaunchKernelGGL(k_b_count, dim3(1), dim3(kBlock), 0, s, flags, n_inst, n_active);
  MFX_HIP(hipGetLastError());
}

uint32_t batch_tile_cells(int p) { return kTile / ((p + 1) * (p + 1)); }

void launch_b_direction_small(const Seg *segs, uint32_t n_segs, const BatchCg *sa, BatchCg *sb,
                              const uint32_t *inst_seg, const double *part_rr,
                              const double *part_rz, const double *r, const double *dinv,
                              const uint8_t *cmask, double *p, double *ap, double *x,
                              double *part_c, int *flags, hipStream_t s) {
  if (sb)
    hipLaunchKernelGGL(k_b_direction_small<true>, dim3(n_segs), dim3(kBlock), 0, s, segs, sa, sb,
                       inst_seg, part_rr, part_rz, r, dinv, cmask, p, ap, x, part_c, flags);
  else
    hipLaunchKernelGGL(k_b_direction_small<false>, dim3(n_segs), dim3(kBlock), 0, s, segs, sa, sb,
                       inst_seg, part_rr, part_rz, r, dinv, cmask, p, ap, x, part_c, flags);
  MFX_HIP(hipGetLastError());
}

void launch_b_update_small(const Seg *segs, uint32_t n_segs, BatchCg *st, const uint32_t *inst_seg,
                           const uint32_t *inst_tile, const double *part_t, const double *part_c,
                           double *r, const double *ap, const double *dinv, double *part_rr,
                           double *part_rz, hipStream_t s) {
  hipLaunchKernelGGL(k_b_update_small, dim3(n_segs), dim3(kBlock), 0, s, segs, st, inst_seg,
                     inst_tile, part_t, part_c, r, ap, dinv, part_rr, part_rz);
  MFX_HIP(hipGetLastError());
}

void launch_b_apply(const BatchTiles &t, uint32_t n_tiles, const double *src, double *dst,
                    const int *done, double *part, hipStream_t s) {
  hipLaunchKernelGGL(k_b_apply, dim3(n_tiles), dim3(kTile), 0, s, t, src, dst, done, part);
  MFX_HIP(hipGetLastError());
}

void launch_offset_map(const uint32_t *src, uint32_t *dst, uint64_t n, uint32_t offset,
                       hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_offset_map, dim3(grid_for(n)), dim3(kBlock), 0, s, src, dst, n, offset);
  MFX_HIP(hipGetLastError());
}

void launch_fill_u16(uint16_t *dst, uint16_t v, uint64_t n, hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_fill_u16, dim3(grid_for(n)), dim3(kBlock), 0, s, dst, v, n);
  MFX_HIP(hipGetLastError());
}

}  // namespace mfx
