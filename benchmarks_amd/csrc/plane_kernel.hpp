// plane_kernel.hpp -- operator apply on box meshes with the metric from the cell
// vertices: a lane holds an (x, z) plane of a cell's points in registers.
//
// A wavefront is one workgroup of C = 64 / NQ cells (consecutive in an xy
// layer); lane (c, j) owns the plane y = j of cell c: the x and z contractions
// (interpolation, derivative and their transposes) run in its registers, and
// only the y contractions go through the LDS, line-wise: lane (c, k) then takes
// the y-lines z = k.  No workgroup barrier: the exchanges order within the
// wave.  Against one lane per (x, y) column with its x and y contractions
// through the LDS (the patch kernel and the per-column Gauss kernel) this halves
// the LDS instructions per point (7.5-8.7 instead of 16-20) and drops the 5-9 barriers
// per batch of cells, which bounded those kernels.  It is bound by the vector
// units where the metric is trilinear (busy 76% in FP32, 51% in FP64 at p = 4
// with two waves per SIMD), by the scatter where it is diagonal (without its
// atomics 310 -> 253 us in FP64, 204 -> 123 in FP32).  33M DoFs, collocated
// p = 4: FP64 undeformed 486 -> 310 us, deformed 476 -> 397; FP32 518 -> 204 and
// 219; Gauss q = 6 on 33M DoFs, undeformed: 884 -> 462 and 448 -> 261.
//
// The wave marches through layers of cells along z.  The node plane two layers
// share is read once and its sums are carried to the next layer in registers;
// sums of faces shared along x are added across lanes.  A layer's sums then go
// through the LDS so that consecutive lanes add consecutive nodes of an x-line
// to dst (FP atomics execute beyond the per-XCD L2s, and their requests are
// what a scatter costs).  DoF indices follow from the cell: no map is read.
#pragma once

#include <algorithm>
#include <type_traits>

#include "mfx_internal.hpp"
#include "plane.hpp"
#include "tables.hpp"

namespace mfx {
namespace {

// LDS strides.  Entry (y, x, z) of cell c is at c CS + y YS + x NQ + z with
// CS = NQ YS and YS = 1 modulo the bank period over gcd: the addresses of the
// lanes of one pass (16 doubles, 32 floats) are then in different banks both
// when lane (c, j) accesses plane y = j and when lane (c, k) accesses the lines
// z = k.
constexpr int plane_gcd(int a, int b) { return b ? plane_gcd(b, a % b) : a; }
template <typename T, int NQ>
constexpr int plane_ys() {
  const int period = (sizeof(T) == 8 ? 16 : 32) / plane_gcd(NQ, sizeof(T) == 8 ? 16 : 32);
  int ys = NQ * NQ;
  while (ys % period != 1 % period) ++ys;
  return ys;
}

template <typename T, int NM_, int NQ_, bool COLLOC_>
struct PlaneCfg {
  static constexpr int NM = NM_, NQ = NQ_, P = NM - 1, C = 64 / NQ;
  static constexpr bool COLLOC = COLLOC_;
  static constexpr int YS = plane_ys<T, NQ>(), CS = NQ * YS;
  // register budget: two waves per SIMD where they hold a plane without
  // spilling much (q = 6, affine: 208 against 300 us at p = 5 on 16M DoFs; one
  // wave where they do not: collocated q = 6 254 against 295, q = 7 306 / 336)
  static constexpr int waves(bool ax) {
    return sizeof(T) == 4 || NQ <= 5 || (ax && !COLLOC && NQ == 6) ? 2 : 1;
  }
  // whole lines stored where the addresses' registers are free (not beside the
  // trilinear metric in FP64: 397 -> 422 us at p = 4, q = 5 on 33M DoFs)
  static constexpr bool stores(bool ax) { return sizeof(T) == 4 || ax; }
  // FP32 p = 4, q = 5 with the trilinear metric is the per-column Gauss kernel's at
  // every size (3% ahead up to 20M DoFs)
  static constexpr bool TRILINEAR = sizeof(T) == 8 || COLLOC || NM != 5 || NQ != 5;
  static constexpr int XS = 65;  // row stride of the scatter staging
  static constexpr int LDS = C * CS > NM * NM * XS ? C * CS : NM * NM * XS;
};

template <typename T, class K, bool AX, bool DOT>
__global__ void __launch_bounds__(64, K::waves(AX))
k_plane(const T *__restrict__ eo_, const T *__restrict__ gxq, const T *__restrict__ gwq,
        const double *__restrict__ cellX, const T *__restrict__ src, T *__restrict__ dst,
        PlaneLayout lay, int fresh, double *__restrict__ partials,
        const int *__restrict__ skip) {
  constexpr int NM = K::NM, NQ = K::NQ, P = K::P, C = K::C, YS = K::YS, CS = K::CS, XS = K::XS;
  constexpr bool COLLOC = K::COLLOC;
  static_assert(!COLLOC || NM == NQ, "collocation: points are the nodes");
  __shared__ T S[K::LDS];
  __shared__ T SX[AX ? 1 : C * 24];
  __shared__ T SK[AX ? 1 : C * 21];
  if (skip && *skip) return;
  // lanes past the last cell repeat lanes of cell C - 1 (same values to the
  // same LDS entries); they neither scatter nor count
  const int lane = threadIdx.x, c = min(lane / NQ, C - 1), j = lane % NQ;
  const uint32_t nx = lay.n[0], ny = lay.n[1], nz = lay.n[2], layer = nx * ny;
  const uint32_t g = blockIdx.x % lay.groups, chunk = blockIdx.x / lay.groups;
  const uint32_t z0 = (uint64_t)nz * chunk / lay.chunks, z1 = (uint64_t)nz * (chunk + 1) / lay.chunks;
  // the group's cells s0 .. s0 + m - 1 of the layer (x fastest), evenly split
  const uint32_t s0 = (uint64_t)layer * g / lay.groups,
                 m = (uint32_t)((uint64_t)layer * (g + 1) / lay.groups) - s0;
  const bool cell_ok = (uint32_t)c < m, active = cell_ok && lane < C * NQ;
  const uint32_t sc = s0 + (cell_ok ? c : 0), ey = sc / nx, ex = sc - ey * nx;
  const uint32_t y0 = s0 / nx;
  const bool has_left = active && c > 0 && ex > 0;
  const bool has_right = active && (uint32_t)c + 1 < m && ex + 1 < nx;
  const uint32_t NX = nx * P + 1, NY = ny * P + 1, NZ = nz * P + 1;
  const uint64_t NXY = (uint64_t)NX * NY;
  // the lane's node plane (lanes j < NM)
  const uint32_t gy = ey * P + (j < NM ? j : 0);
  const bool row_in = cell_ok && j < NM && gy > 0 && gy < NY - 1;
  const bool xl_in = ex > 0, xr_in = ex + 1 < nx;
  const T *const psrc = src + (uint64_t)gy * NX + ex * P;
  // node (x, gz) values of the plane as they are: every address is inside the
  // vector, so the loads need no branch and wait for nothing; constrained
  // nodes are set to zero where the values are used, in waves that hold any
  auto load_row = [&](T (&v)[NM], uint32_t gz) {
    const T *q = psrc + gz * NXY;
#pragma unroll
    for (int x = 0; x < NM; ++x) v[x] = q[x];
  };
  const bool edge = !__all(j >= NM || (row_in && xl_in && xr_in));
  auto mask_row = [&](T (&v)[NM], uint32_t gz) {
    const bool in = gz > 0 && gz < NZ - 1;
    if (edge || !in) {
#pragma unroll
      for (int x = 0; x < NM; ++x)
        v[x] = in && row_in && (x > 0 || xl_in) && (x < P || xr_in) ? v[x] : T(0);
    }
  };
  // staging position of the lane's node x = 0
  const int spos = c * P + (int)(ey - y0);

  const T eta = gxq[j], wy = gwq[j];
  constexpr GllD<NQ> kD{};
  auto dm = [&](int i, int a) { return kD.D[i][a]; };
  auto dmt = [&](int i, int a) { return kD.D[a][i]; };
  constexpr int EO_BT = eo_table_size(NQ, NM), EO_D = EO_BT + eo_table_size(NM, NQ),
                EO_DT = EO_D + eo_table_size(NQ, NQ);
  T *const Sp = S + c * CS + j * YS;  // the lane's plane: (x, z) at x NQ + z
  T *const Sl = S + c * CS + j;       // its lines z = j: (x, y) at x NQ + y YS

  double dot = 0.0;
  T un[P][NM], uc[NM], carry[NM];
  // the cell's vertex coordinates: each lane of the cell loads a share (the
  // trilinear form: 24 / NQ each), exchanged through the LDS
  constexpr int XV = AX ? 6 : (24 + NQ - 1) / NQ;
  double xv[XV];
  auto load_cell = [&](uint32_t ez) {
    const double *X = cellX + ((uint64_t)ez * layer + sc) * 24;
    if constexpr (AX) {
      xv[0] = X[0]; xv[1] = X[3];    // x of vertices 0, 1
      xv[2] = X[1]; xv[3] = X[7];    // y of vertices 0, 2
      xv[4] = X[2]; xv[5] = X[14];   // z of vertices 0, 4
    } else {
#pragma unroll
      for (int k = 0; k < XV; ++k) xv[k] = X[min(j + k * NQ, 23)];
    }
  };
  if (z0 < z1) {
    load_cell(z0);
    load_row(uc, z0 * P);
#pragma unroll
    for (int z = 0; z < P; ++z) load_row(un[z], z0 * P + z + 1);
  }
#pragma unroll
  for (int x = 0; x < NM; ++x) carry[x] = T(0);

  for (uint32_t ez = z0; ez < z1; ++ez) {
    T u[NQ][NQ];  // plane values [z][x], later its weak-form sums
    // kept from being hoisted out of the layer loop: products of the weights
    // (a register pair each) and the tables (more than the scalar registers)
    T wyl = wy;
    asm volatile("" : "+v"(wyl));
    typedef const T __attribute__((address_space(4))) *TabPtr;  // read through the scalar cache
    TabPtr eo = (TabPtr)(uintptr_t)eo_;
    asm volatile("" : "+s"(eo));
    auto apply_d = [&](const T *in, T *out) {
      if constexpr (COLLOC)
        eo_mat<NQ, NQ, -1>(dm, in, out);
      else
        eo_tab<NQ, NQ, -1>(eo + EO_D, in, out);
    };
    auto apply_dt = [&](const T *in, T *out) {
      if constexpr (COLLOC)
        eo_mat<NQ, NQ, -1>(dmt, in, out);
      else
        eo_tab<NQ, NQ, -1>(eo + EO_DT, in, out);
    };
    // 1. the cell's metric data
    [[maybe_unused]] T mx = 0, my = 0, mz = 0;
    [[maybe_unused]] T a0[3], da[3], jz0[3];
    if constexpr (AX) {
      const T hx = (T)xv[1] - (T)xv[0], hy = (T)xv[3] - (T)xv[2], hz = (T)xv[5] - (T)xv[4];
      const T H0 = hy * hz, H1 = hz * hx, H2 = hx * hy, hr = recip(hz * H2) * wyl;
      mx = hr * H0 * H0;
      my = hr * H1 * H1;
      mz = hr * H2 * H2;
    } else {
#pragma unroll
      for (int k = 0; k < XV; ++k)
        if (j + k * NQ < 24) SX[c * 24 + j + k * NQ] = (T)xv[k];
      __syncthreads();
      // trilinear coefficients per coordinate d (patch.hip): J0 = (A0 + eta A1)
      // + zeta (K1 + eta K3), J1 = (G0 + zeta K2) + xi (A1 + zeta K3), J2 =
      // (K0 + eta K2) + xi (K1 + eta K3)
      for (int d = j; d < 3; d += NQ) {
        const T *X = SX + c * 24 + d;
        const T x0 = X[0], x1 = X[3], x2 = X[6], x3 = X[9];
        const T x4 = X[12], x5 = X[15], x6 = X[18], x7 = X[21];
        T *Kd = SK + c * 21 + 7 * d;
        const T e0 = x1 - x0, e1 = (x3 - x2) - e0, k0 = x4 - x0;
        Kd[0] = e0;
        Kd[1] = k0;
        Kd[2] = (x5 - x1) - k0;
        Kd[3] = x2 - x0;
        Kd[4] = e1;
        Kd[5] = (x6 - x2) - k0;
        Kd[6] = ((x7 - x6) - (x5 - x4)) - e1;
      }
      __syncthreads();
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const T *Kd = SK + c * 21 + 7 * d;
        a0[d] = Kd[0] + eta * Kd[4];
        da[d] = Kd[2] + eta * Kd[6];
        jz0[d] = Kd[1] + eta * Kd[5];
      }
    }
    // 2. nodal plane -> point plane and y derivative
    if (ez == z0) mask_row(uc, ez * P);
#pragma unroll
    for (int z = 0; z < P; ++z) mask_row(un[z], ez * P + z + 1);
    if constexpr (COLLOC) {
#pragma unroll
      for (int x = 0; x < NQ; ++x) {
        u[0][x] = uc[x];
#pragma unroll
        for (int z = 0; z < P; ++z) u[z + 1][x] = un[z][x];
      }
#pragma unroll
      for (int x = 0; x < NM; ++x) uc[x] = un[P - 1][x];
#pragma unroll
      for (int x = 0; x < NQ; ++x)
#pragma unroll
        for (int z = 0; z < NQ; ++z) Sp[x * NQ + z] = u[z][x];
      __syncthreads();
#pragma unroll
      for (int x = 0; x < NQ; ++x) {
        T ln[NQ], o[NQ];
#pragma unroll
        for (int y = 0; y < NQ; ++y) ln[y] = Sl[x * NQ + y * YS];
        apply_d(ln, o);
#pragma unroll
        for (int y = 0; y < NQ; ++y) Sl[x * NQ + y * YS] = o[y];
      }
      __syncthreads();
    } else {
      T t[NM][NQ];
      eo_tab<NQ, NM, 1>(eo, uc, t[0]);
#pragma unroll
      for (int z = 0; z < P; ++z) eo_tab<NQ, NM, 1>(eo, un[z], t[z + 1]);
#pragma unroll
      for (int x = 0; x < NM; ++x) uc[x] = un[P - 1][x];
#pragma unroll
      for (int x = 0; x < NQ; ++x) {
        T ln[NM], o[NQ];
#pragma unroll
        for (int z = 0; z < NM; ++z) ln[z] = t[z][x];
        eo_tab<NQ, NM, 1>(eo, ln, o);
#pragma unroll
        for (int z = 0; z < NQ; ++z) Sp[x * NQ + z] = o[z];
      }
      __syncthreads();
      asm volatile("" : "+s"(eo));
      T dl[NQ][NQ];  // y derivatives of the lane's lines [x][y]
#pragma unroll
      for (int x = 0; x < NQ; ++x) {
        T ln[NM], o[NQ];
#pragma unroll
        for (int y = 0; y < NM; ++y) ln[y] = Sl[x * NQ + y * YS];
        eo_tab<NQ, NM, 1>(eo, ln, o);
#pragma unroll
        for (int y = 0; y < NQ; ++y) Sl[x * NQ + y * YS] = o[y];
        apply_d(o, dl[x]);
      }
      __syncthreads();
#pragma unroll
      for (int x = 0; x < NQ; ++x)
#pragma unroll
        for (int z = 0; z < NQ; ++z) u[z][x] = Sp[x * NQ + z];
      __syncthreads();
#pragma unroll
      for (int x = 0; x < NQ; ++x)
#pragma unroll
        for (int y = 0; y < NQ; ++y) Sl[x * NQ + y * YS] = dl[x][y];
      __syncthreads();
    }
    asm volatile("" : "+s"(eo));  // (the tables' loads stay with their phase)
    // 3. z derivatives (columns), then per row z the x derivatives, the
    // fluxes and the x flux's transposed derivative in place of u
    T dz[NQ][NQ];  // [z][x], later the z fluxes
#pragma unroll
    for (int x = 0; x < NQ; ++x) {
      T ln[NQ], o[NQ];
#pragma unroll
      for (int z = 0; z < NQ; ++z) ln[z] = u[z][x];
      apply_d(ln, o);
#pragma unroll
      for (int z = 0; z < NQ; ++z) dz[z][x] = o[z];
    }
#pragma unroll
    for (int z = 0; z < NQ; ++z) {
      T dx[NQ], fx[NQ];
      apply_d(u[z], dx);
      T wz = gwq[z];
      // pins the row's work between its neighbours': left to itself the
      // scheduler holds the temporaries of all rows
      asm volatile("" : "+s"(wz));
      [[maybe_unused]] const T wx = wz * mx, wy1 = wz * my, wz1 = wz * mz, wyz = wyl * wz;
      [[maybe_unused]] T J0[3], p0[3], p1[3];
      if constexpr (!AX) {
        T zeta = gxq[z];
        asm volatile("" : "+s"(zeta));
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          J0[d] = a0[d] + zeta * da[d];
          const T *Kd = SK + c * 21 + 7 * d;  // (kept in the LDS for the registers)
          p0[d] = Kd[3] + zeta * Kd[5];
          p1[d] = Kd[4] + zeta * Kd[6];
        }
      }
#pragma unroll
      for (int x = 0; x < NQ; ++x) {
        const T dy = Sp[x * NQ + z];
        T f1, f2;
        if constexpr (AX) {
          const T w = gwq[x];
          fx[x] = (w * wx) * dx[x];
          f1 = (w * wy1) * dy;
          f2 = (w * wz1) * dz[z][x];
        } else {
          const T xi = gxq[x];
          T J1[3], J2[3], C0[3], C1[3], C2[3], W[3];
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            J1[d] = p0[d] + xi * p1[d];
            J2[d] = jz0[d] + xi * da[d];
          }
          C0[0] = J1[1] * J2[2] - J1[2] * J2[1];
          C0[1] = J1[2] * J2[0] - J1[0] * J2[2];
          C0[2] = J1[0] * J2[1] - J1[1] * J2[0];
          C1[0] = J2[1] * J0[2] - J2[2] * J0[1];
          C1[1] = J2[2] * J0[0] - J2[0] * J0[2];
          C1[2] = J2[0] * J0[1] - J2[1] * J0[0];
          C2[0] = J0[1] * J1[2] - J0[2] * J1[1];
          C2[1] = J0[2] * J1[0] - J0[0] * J1[2];
          C2[2] = J0[0] * J1[1] - J0[1] * J1[0];
          const T det = J2[0] * C2[0] + J2[1] * C2[1] + J2[2] * C2[2];
          const T s = wyz * gwq[x] * recip(det);
#pragma unroll
          for (int d = 0; d < 3; ++d) W[d] = dx[x] * C0[d] + dy * C1[d] + dz[z][x] * C2[d];
          fx[x] = s * (C0[0] * W[0] + C0[1] * W[1] + C0[2] * W[2]);
          f1 = s * (C1[0] * W[0] + C1[1] * W[1] + C1[2] * W[2]);
          f2 = s * (C2[0] * W[0] + C2[1] * W[1] + C2[2] * W[2]);
        }
        // p.Ap as the cells' energies (constrained entries are gathered as 0)
        if constexpr (DOT)
          dot += (double)dx[x] * (double)fx[x] + (double)dy * (double)f1 +
                 (double)dz[z][x] * (double)f2;
        Sp[x * NQ + z] = f1;
        dz[z][x] = f2;
      }
      apply_dt(fx, u[z]);
#pragma unroll
      for (int x = 0; x < NQ; ++x) asm volatile("" : "+v"(u[z][x]), "+v"(dz[z][x]));
      if constexpr (DOT) asm volatile("" : "+v"(dot));
    }
    // the next layer's vertices and values, in flight until it begins
    if (ez + 1 < z1) {
      load_cell(ez + 1);
#pragma unroll
      for (int z = 0; z < P; ++z) load_row(un[z], (ez + 1) * P + z + 1);
    }
#pragma unroll
    for (int x = 0; x < NQ; ++x) {
      T ln[NQ], o[NQ];
#pragma unroll
      for (int z = 0; z < NQ; ++z) ln[z] = dz[z][x];
      apply_dt(ln, o);
#pragma unroll
      for (int z = 0; z < NQ; ++z) u[z][x] += o[z];
    }
    __syncthreads();
    asm volatile("" : "+s"(eo));
    // 4. the y flux's transposed derivative along lines, and back to nodes
    T o[NM][NM];  // nodal sums of the plane y = j < NM: [z][x]
    if constexpr (COLLOC) {
#pragma unroll
      for (int x = 0; x < NQ; ++x) {
        T ln[NQ], r[NQ];
#pragma unroll
        for (int y = 0; y < NQ; ++y) ln[y] = Sl[x * NQ + y * YS];
        apply_dt(ln, r);
#pragma unroll
        for (int y = 0; y < NQ; ++y) Sl[x * NQ + y * YS] = r[y];
      }
      __syncthreads();
#pragma unroll
      for (int x = 0; x < NQ; ++x)
#pragma unroll
        for (int z = 0; z < NQ; ++z) o[z][x] = u[z][x] + Sp[x * NQ + z];
    } else {
      T gl[NQ][NQ];
#pragma unroll
      for (int x = 0; x < NQ; ++x) {
        T ln[NQ];
#pragma unroll
        for (int y = 0; y < NQ; ++y) ln[y] = Sl[x * NQ + y * YS];
        apply_dt(ln, gl[x]);
      }
      __syncthreads();
#pragma unroll
      for (int x = 0; x < NQ; ++x)
#pragma unroll
        for (int z = 0; z < NQ; ++z) Sp[x * NQ + z] = u[z][x];
      __syncthreads();
#pragma unroll
      for (int x = 0; x < NQ; ++x) {
        T ln[NQ], r[NM];
#pragma unroll
        for (int y = 0; y < NQ; ++y) ln[y] = Sl[x * NQ + y * YS] + gl[x][y];
        eo_tab<NM, NQ, 1>(eo + EO_BT, ln, r);
#pragma unroll
        for (int y = 0; y < NM; ++y) Sl[x * NQ + y * YS] = r[y];
      }
      __syncthreads();
      T t[NM][NQ];
#pragma unroll
      for (int x = 0; x < NQ; ++x) {
        T ln[NQ], r[NM];
#pragma unroll
        for (int z = 0; z < NQ; ++z) ln[z] = Sp[x * NQ + z];
        eo_tab<NM, NQ, 1>(eo + EO_BT, ln, r);
#pragma unroll
        for (int z = 0; z < NM; ++z) t[z][x] = r[z];
      }
#pragma unroll
      for (int z = 0; z < NM; ++z) eo_tab<NM, NQ, 1>(eo + EO_BT, t[z], o[z]);
    }
    __syncthreads();  // the planes have been read
    // 5. faces shared along x (the right face of the cell before, then the
    // left one) and with the layer below; scatter
#pragma unroll
    for (int z = 0; z < NM; ++z) {
      const T r = __shfl_up(o[z][P], NQ, 64);
      if (has_left) o[z][0] += r;
    }
#pragma unroll
    for (int x = 0; x < NM; ++x) {
      o[0][x] += carry[x];
      carry[x] = o[P][x];
    }
    const bool last = ez + 1 == z1;
    if (active && j < NM) {
#pragma unroll
      for (int z = 0; z < NM; ++z) {
        if (z == P && !last) continue;
        T *row = S + (z * NM + j) * XS + spos;
#pragma unroll
        for (int x = 0; x < P; ++x) row[x] = o[z][x];
        if (!has_right) row[P] = o[z][P];
      }
    }
    __syncthreads();
    // scatter lane i: node i of the group's x-lines laid end to end (a row of
    // cells continues the line, a new row starts its own).  Formed per layer:
    // kept, these values would cost the flux phase its second wave.
    uint32_t li = lane;
    asm volatile("" : "+v"(li));
    const uint32_t xg = li + (s0 - y0 * nx) * P, rr = xg / NX, gx = xg - rr * NX;
    const uint32_t n_nodes = m * P + (s0 + m - 1) / nx - y0 + 1;
    const bool snode = li < n_nodes && gx > 0 && gx < NX - 1;
    const bool s_first = snode && y0 + rr > 0, s_last = snode && y0 + rr + 1 < ny;
    // nodes of the lane's x-line before and after it that no other wave has
    const int before = min((int)li - (s0 == y0 * nx ? 0 : 1), (int)gx - 1);
    const int after = min((int)n_nodes - 1 - (int)li - ((s0 + m) % nx == 0 ? 0 : 1),
                          (int)NX - 2 - (int)gx);
    T *const pdst = dst + (uint64_t)(snode ? (y0 + rr) * P : 0) * NX + (snode ? gx : 0);
    constexpr int LINE = 128 / sizeof(T);
#pragma unroll
    for (int z = 0; z < NM; ++z) {
      const uint32_t gz = ez * P + z;
      if ((z == P && !last) || gz == 0 || gz == NZ - 1) continue;
      // planes shared with the chunk below or above
      const bool own = K::stores(AX) && fresh && !(z == 0 && ez == z0) && z < P;
      T *q = pdst + gz * NXY;
#pragma unroll
      for (int y = 0; y < NM; ++y, q += NX) {
        const T v = S[(z * NM + y) * XS + li];
        if (y > 0 && y < P && own) {
          // a 128-byte line that only this wave writes: stored whole
          const int at = (int)((uintptr_t)q / sizeof(T)) & (LINE - 1);
          if (snode) {
            if (at <= before && LINE - 1 - at <= after)
              *q = v;
            else
              unsafeAtomicAdd(q, v);
          }
        } else if (y == 0 ? s_first : y == P ? s_last : snode) {
          unsafeAtomicAdd(q, v);
        }
      }
    }
    __syncthreads();  // the staging has been read
  }
  if constexpr (DOT) {
    dot = active ? dot : 0.0;  // idle lanes repeat other lanes' or cells' work
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) dot += __shfl_xor(dot, o, 64);
    if (lane == 0) partials[blockIdx.x] = dot;
  }
}

template <typename T, class K>
void launch_cfg(const PlaneOp<T> &o, const T *src, T *dst, bool fresh, hipStream_t s,
                double *partials, const int *skip) {
  const PlaneLayout &lay = o.lay;
  const dim3 grid(lay.groups * lay.chunks), block(64);
  MFX_REQUIRE(o.axes || K::TRILINEAR, "plane kernel: no instance");
  if (partials) {
    if constexpr (std::is_same<T, double>::value) {
      if (o.axes)
        hipLaunchKernelGGL((k_plane<T, K, true, true>), grid, block, 0, s, o.eo, o.xq, o.wq,
                           o.cellX, src, dst, lay, (int)fresh, partials, skip);
      else
        hipLaunchKernelGGL((k_plane<T, K, false, true>), grid, block, 0, s, o.eo, o.xq, o.wq,
                           o.cellX, src, dst, lay, (int)fresh, partials, skip);
    } else {
      throw Error{MFX_ERR_UNSUPPORTED, "p.Ap partials are computed in FP64 only"};
    }
  } else if (o.axes) {
    hipLaunchKernelGGL((k_plane<T, K, true, false>), grid, block, 0, s, o.eo, o.xq, o.wq, o.cellX,
                       src, dst, lay, (int)fresh, nullptr, nullptr);
  } else if constexpr (K::TRILINEAR) {
    hipLaunchKernelGGL((k_plane<T, K, false, false>), grid, block, 0, s, o.eo, o.xq, o.wq, o.cellX,
                       src, dst, lay, (int)fresh, nullptr, nullptr);
  }
  MFX_HIP(hipGetLastError());
}

// f(PlaneCfg) of the instance for (p, nq, colloc); false if there is none
template <typename T, typename F>
bool with_plane(int p, int nq, bool colloc, F &&f) {
#define MFX_PLANE(NM, NQ, COL)                                        \
  if (p + 1 == NM && nq == NQ && colloc == COL) {                     \
    f(PlaneCfg<T, NM, NQ, COL>{});                                    \
    return true;                                                      \
  }
  MFX_PLANE(2, 2, true)
  MFX_PLANE(3, 3, true)
  MFX_PLANE(4, 4, true)
  MFX_PLANE(5, 5, true)
  MFX_PLANE(6, 6, true)
  MFX_PLANE(2, 2, false)
  MFX_PLANE(2, 3, false)
  MFX_PLANE(3, 3, false)
  MFX_PLANE(3, 4, false)
  MFX_PLANE(4, 4, false)
  MFX_PLANE(4, 5, false)
  MFX_PLANE(5, 5, false)
  MFX_PLANE(5, 6, false)
  MFX_PLANE(6, 6, false)
  MFX_PLANE(6, 7, false)
  MFX_PLANE(7, 7, false)
  MFX_PLANE(7, 7, true)
  if constexpr (sizeof(T) == 4) {
    MFX_PLANE(8, 8, true)
    MFX_PLANE(7, 8, false)
    MFX_PLANE(8, 8, false)
  }
#undef MFX_PLANE
  return false;
}

}  // namespace

template <typename T>
bool plane_instance(int p, int nq, bool colloc, bool axes) {
  bool ok = false;
  with_plane<T>(p, nq, colloc, [&](auto k) { ok = axes || decltype(k)::TRILINEAR; });
  return ok;
}

template <typename T>
void launch_plane(const PlaneOp<T> &o, const T *src, T *dst, bool fresh, hipStream_t s,
                  double *partials, const int *skip) {
  MFX_REQUIRE(o.xq && o.wq && o.cellX && (o.colloc || o.eo), "plane kernel: arrays missing");
  MFX_REQUIRE(o.lay.groups > 0 && o.lay.chunks > 0 &&
                  (uint64_t)o.lay.groups * (64 / o.nq) >= (uint64_t)o.lay.n[0] * o.lay.n[1],
              "plane kernel: layout does not cover the mesh");
  const bool ok = with_plane<T>(o.p, o.nq, o.colloc, [&](auto k) {
    launch_cfg<T, decltype(k)>(o, src, dst, fresh, s, partials, skip);
  });
  MFX_REQUIRE(ok, "plane kernel: no instance");
}

}  // namespace mfx
