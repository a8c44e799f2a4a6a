// patch.hip -- BK5 (GLL collocation) operator apply on patches of cells with
// the metric terms computed on the fly from the cell vertices.
//
// A patch is BX x BY x BZ cells of a structured mesh and the
// (BX p + 1)(BY p + 1)(BZ p + 1) DoFs they touch, numbered patch-locally
// (x fastest).  The patch DoF map (uint32, 0xFFFFFFFF = constrained or
// outside the mesh; bit 31 = DoF also touched by another patch) replaces the
// per-cell map of the reference kernel (CEED_bp/include/bk3_kokkos_kernel.h:
// 113-143, 356-382) for meshes generated by mfx_op_create_box.
//
// The kernel is persistent: the grid is what the device holds at once and
// every workgroup walks its patches (blockIdx, blockIdx + gridDim, ...) in a
// software pipeline, so that the dependent global loads of one patch (map,
// then values) are in flight while the previous patch computes:
//   1. stage: values, indices and vertices of patch k (loaded during patch
//      k-1) go to LDS; the map and vertices of patch k+1 are requested;
//   2. per cell, NQ^2 threads; thread (l0, l1) owns the x-line (y = l0,
//      z = l1), the y-line (x = l0, z = l1) and the z-column (x, y) = (l0,
//      l1) of the cell, each held whole in registers (one LDS read per
//      operand): x and y derivatives along the lines into two per-cell LDS
//      arrays; then per column the z derivative, the metric of the
//      trilinear cell evaluated per quadrature point from per-column
//      polynomial coefficients (no G array: 24 doubles per cell instead of
//      48 q^3 bytes) and the fluxes, written back in place; the 1D
//      contractions use the even-odd split of the GLL derivative matrix,
//      a compile-time table;
//      then the values of patch k+1 are requested (its map has arrived);
//   3. transposed contractions along the same lines; each column adds its
//      three into a patch array in LDS with LDS atomics (ds_add_f64) --
//      cells of one patch share faces;
//   4. scatter: one hardware FP64 atomic (global_atomic_add_f64) per patch
//      DoF instead of one per cell node.
// The deterministic variant (DET) replaces 3 and 4: each column writes its
// sums into the cell's own LDS array, every patch DoF adds the results of
// the cells holding it in ascending cell order and is stored per patch, and
// k_patch_gather adds the stored patch sums per DoF in patch order.
// Optionally the workgroup also returns sum_i u_i (A u)_i over its patches
// (the p.Ap of a CG step) as a per-workgroup partial.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "mfx_internal.hpp"
#include "patch.hpp"
#include "tables.hpp"

namespace mfx {
namespace {

// Compile-time shape and tuning of one patch-kernel instance: NQ points per
// direction, BX x BY x BZ cells per patch, WPE, the waves per SIMD the
// register allocation must leave room for, and the form of the column metric
// (CELLCOEF: per-cell coefficient vectors and cofactors formed per point, with
// fewer registers; else per-column cofactor polynomials, fewer operations per
// point).
//
// WAVECELL (NQ <= 8): whole cells per wavefront, 64 / NQ^2 of them, the
// rest of the wave's lanes idle; the phases that touch only a cell's own
// LDS arrays then need no workgroup barrier, only the wave's own ordering.
//
// SKEW: the layout of the two per-cell derivative arrays.  Node (x, y, z) of
// cell c sits at c CS + x + NQ y + ZS z.  Unskewed, ZS = NQ^2 and CS = NQ^3.
// Skewed, the strides are padded so that the accesses of 16 consecutive
// lanes (one pass of a 64-bit LDS access over 32 four-byte banks) fall in
// 16 different bank pairs: lane t = col + NQ^2 c reads address t + const
// (mod 16) in every phase.  The x-derivative array is read along x-lines and
// z-columns, so (with the x-line of thread (l0, l1) at y = l1, z = l0) its
// ZS = 1 and CS = NQ^2 (mod 16); the y-derivative array is read along y-lines
// and z-columns, so its ZS = NQ and CS = NQ^2 (mod 16).
constexpr int skew_up(int v, int r) { return v + ((r - v) % 16 + 16) % 16; }
template <int NQ_, int BX_, int BY_, int BZ_, int WPE_, bool CELLCOEF_, bool WAVECELL_ = false,
          bool SKEW_ = false>
struct PatchCfg {
  static constexpr int NQ = NQ_, BX = BX_, BY = BY_, BZ = BZ_, WPE = WPE_;
  static constexpr bool CELLCOEF = CELLCOEF_, WAVECELL = WAVECELL_, SKEW = SKEW_;
  static constexpr int P = NQ - 1, NQ2 = NQ * NQ, NQ3 = NQ2 * NQ;
  static constexpr int AZS = SKEW ? skew_up(NQ2, 1) : NQ2;   // x-derivative array
  static constexpr int BZS = SKEW ? skew_up(NQ2, NQ) : NQ2;  // y-derivative array
  static constexpr int ACS = SKEW ? skew_up(P * (NQ + 1 + AZS) + 1, NQ2) : NQ3;
  static constexpr int BCS = SKEW ? skew_up(P * (NQ + 1 + BZS) + 1, NQ2) : NQ3;
  static constexpr int CPP = BX * BY * BZ;
  static_assert(!WAVECELL || NQ2 <= 64, "a wave-held cell needs NQ^2 <= 64");
  static constexpr int CW = WAVECELL ? 64 / NQ2 : 0;  // cells per wave
  static constexpr int THREADS = WAVECELL ? (CPP + CW - 1) / CW * 64 : CPP * NQ2;
  static constexpr int PX = BX * P + 1, PY = BY * P + 1, PZ = BZ * P + 1;
  static constexpr int P3 = PX * PY * PZ;
  static constexpr int PER = (P3 + THREADS - 1) / THREADS;        // patch DoFs per thread
  static constexpr int VPT = (CPP * 24 + THREADS - 1) / THREADS;  // vertex coordinates per thread
  // stored metric terms in patch order: [patch][6][NQ][GTP], the value of
  // component k at point z of column col of cell c at (k NQ + z) GTP +
  // c NQ^2 + col; GTP rounds the patch's columns up to whole 128-byte lines
  // of doubles
  static constexpr int GTP = (CPP * NQ2 + 15) / 16 * 16;
};

// Configuration per degree, chosen by timing the BP5 operators at ~32M DoFs
// (FP64, deformed box; p = 2, 4, 6, 8 over 8 patch shapes and register
// budgets each, with both metric forms).  Whole cells per wave (WAVECELL)
// measured 2-5% faster at p = 1, 2, 6 (16, 7 and 1 cells per wave), level
// at p = 3, 7, and 40-80% slower at p = 4, 5 (2 cells in 50 lanes, 1 in 36;
// at p = 4 also with the second cell at lane 32, in 5x2x1 and 4x2x1 patches).
// The skewed derivative arrays (SKEW) measured 5% faster at p = 3 and 1-2% at
// p = 6, 7, 8; level at p = 1, 4; slower at p = 2 (18%, its arrays grow
// 2x) and p = 5 (6%, 3 -> 2 workgroups per CU for the LDS).  p = 8 goes
// without: its 1.9 KB would keep the aliased accumulator's kernel (see
// k_patch) at 2 workgroups per CU.
template <typename F>
decltype(auto) with_cfg(int p, F &&f) {
  switch (p) {
    case 1: return f(PatchCfg<2, 4, 4, 4, 1, false, true>{});
    case 2: return f(PatchCfg<3, 7, 2, 2, 1, false, true>{});
    case 3: return f(PatchCfg<4, 4, 2, 2, 1, false, false, true>{});
    case 4: return f(PatchCfg<5, 5, 2, 1, 3, true>{});
    case 5: return f(PatchCfg<6, 7, 1, 1, 1, false>{});
    case 6: return f(PatchCfg<7, 4, 1, 1, 1, false, true, true>{});
    case 7: return f(PatchCfg<8, 2, 1, 1, 2, false, false, true>{});
    case 8: return f(PatchCfg<9, 3, 1, 1, 2, true>{});
    default: throw Error{MFX_ERR_UNSUPPORTED, "patch kernel: degree must be in 1..8"};
  }
}

template <typename T>
__device__ __forceinline__ void cross(const T *a, const T *b, T *r) {
  r[0] = a[1] * b[2] - a[2] * b[1];
  r[1] = a[2] * b[0] - a[0] * b[2];
  r[2] = a[0] * b[1] - a[1] * b[0];
}

__device__ __forceinline__ uint32_t patch_count_d(const PatchLayout &lay) {
  return lay.np[0] * lay.np[1] * lay.np[2];
}

__device__ __forceinline__ void patch_xyz(const PatchLayout &lay, uint32_t pt, uint32_t &px,
                                          uint32_t &py, uint32_t &pz) {
  px = pt % lay.np[0];
  py = (pt / lay.np[0]) % lay.np[1];
  pz = pt / (lay.np[0] * lay.np[1]);
}

// Batch mode (BATCH): patch data of several operators, see PatchBatchOp.
struct BatchArgs {
  const uint4 *meta;
  const uint4 *inst;
  const int *done;
  uint32_t n_patches;
  const uint32_t *slot;  // per instance (batch numbering): its p.Ap slot in this launch's partials
};

// Register budget: the configuration's waves per SIMD; the batch kernel
// with p.Ap partials is held to 3 up to nq = 7 (the batched degrees), where
// the plain batch kernel runs 3 and the partials' bookkeeping would
// otherwise cost a wave (measured 20% slower at p = 5, 6).
template <class C, bool DOT, bool BATCH>
constexpr int kPatchWaves = (BATCH && DOT && C::NQ <= 7 && C::WPE < 3) ? 3 : C::WPE;

//
// STORED: the metric terms come from the stored G = w det J J^-1 J^-T
// (xx, xy, xz, yy, yz, zz) instead of the cell vertices, permuted into
// patch order (PatchCfg::GTP, k_patch_geometry) so that every load of a
// wavefront reads whole 128-byte lines.  Each thread's 6 q values of the
// next patch are requested once the current patch's are used, so the G
// stream has the second half of a patch to arrive.
template <typename T, class C, bool DOT, bool BATCH = false, bool DET = false, bool STORED = false>
__global__ void __attribute__((amdgpu_flat_work_group_size(1, C::THREADS),
                               amdgpu_waves_per_eu(kPatchWaves<C, DOT, BATCH>)))
k_patch(const T *__restrict__ gw, const T *__restrict__ gxq,
        const double *__restrict__ cellX, const T *__restrict__ src, T *__restrict__ dst,
        const uint32_t *__restrict__ pmap, PatchLayout lay, double *__restrict__ partials,
        const int *__restrict__ skip, BatchArgs ba, T *__restrict__ pbuf,
        const T *__restrict__ G) {
  constexpr int NQ = C::NQ, NQ2 = C::NQ2, P = C::P, PX = C::PX, PY = C::PY;
  constexpr int P3 = C::P3, THREADS = C::THREADS, PER = C::PER, VPT = C::VPT, CPP = C::CPP;
  constexpr int BX = C::BX, BY = C::BY, BZ = C::BZ;
  static_assert(!(BATCH && DET), "the deterministic scatter is for single operators");
  static_assert(!(BATCH && STORED), "batched patches carry their vertices");
  constexpr bool VERT = !STORED;  // metric from the cell vertices
  __shared__ T spu[P3];
  // ALIAS: the patch accumulator of the atomic scatter reuses the input
  // array, which is dead once the gradient phase is done (it is zeroed
  // there, between two workgroup barriers).  Not with p.Ap partials (the
  // scatter reads the inputs) nor with whole cells per wave (whose
  // per-cell phases have no workgroup barrier).  The smaller LDS footprint
  // gives p = 8 a third workgroup per CU: 6% faster, p = 7 7.5%.
  constexpr bool ALIAS = !DOT && !DET && !C::WAVECELL;
  __shared__ T spv[(DET || ALIAS) ? 1 : P3];  // patch accumulator of the atomic scatter
  T *const acc = ALIAS ? spu : spv;
  __shared__ uint32_t sidx[DET ? P3 : 1];
  constexpr int AZS = C::AZS, BZS = C::BZS, ACS = C::ACS, BCS = C::BCS;
  __shared__ T sfx[CPP * ACS];
  __shared__ T sfy[CPP * BCS];
  __shared__ T sX[VERT ? CPP * 24 : 1];
  __shared__ T sK[VERT && C::CELLCOEF ? CPP * 21 : 1];  // per cell 7 trilinear coefficient vectors
  __shared__ double red[(THREADS + 63) / 64];

  if (skip && *skip) return;
  const uint32_t npatch = BATCH ? ba.n_patches : lay.np[0] * lay.np[1] * lay.np[2];
  // patch coordinates, cell counts and first cell of patch `pt`; false when
  // the patch is to be skipped (past the end, or its instance has converged)
  auto locate = [&](uint32_t pt, uint32_t &px, uint32_t &py, uint32_t &pz, uint32_t (&n)[3],
                    size_t &c0, uint32_t &inst) -> bool {
    if (pt >= npatch) return false;
    if constexpr (BATCH) {
      const uint4 m = ba.meta[pt];
      inst = m.x;
      const uint4 g = ba.inst[m.x];
      px = m.y;
      py = m.z;
      pz = m.w;
      n[0] = g.x;
      n[1] = g.y;
      n[2] = g.z;
      c0 = g.w;
      return !(ba.done && ba.done[m.x]);
    } else {
      patch_xyz(lay, pt, px, py, pz);
      n[0] = lay.n[0];
      n[1] = lay.n[1];
      n[2] = lay.n[2];
      c0 = 0;
      return true;
    }
  };
  const uint32_t step = gridDim.x;
  const int tid = threadIdx.x;
  // cell c of the patch and column col of the cell that this thread owns
  int c, col;
  bool lane_ok = true;
  if constexpr (C::WAVECELL) {
    const int ln = tid & 63;
    c = (tid >> 6) * C::CW + ln / NQ2;
    col = ln % NQ2;
    // lanes past the wave's last whole cell are idle (they would repeat
    // columns of the next wave's first cell)
    lane_ok = ln < C::CW * NQ2 && c < CPP;
    c = lane_ok ? c : 0;
    col = lane_ok ? col : 0;
  } else {
    c = tid / NQ2;
    col = tid - c * NQ2;
  }
  // between phases that touch only the thread's own cell: a workgroup
  // barrier, or with whole cells per wave the wave's own ordering of its
  // LDS accesses
  auto cell_sync = [&]() {
    if constexpr (C::WAVECELL) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
      __syncthreads();
    }
  };
  const int qx = col % NQ, qy = col / NQ;
  const int cx = c % BX, cy = (c / BX) % BY, cz = c / (BX * BY);
  const T xi = gxq[qx], eta = gxq[qy];
  const T wxy = gw[qx] * gw[qy];

  // With stored geometry (memory-bound) a box operator takes the patch DoF
  // indices from the patch coordinates (the same values as the patch map,
  // whose shared-DoF bit the kernel does not use) instead of reading the map:
  // 4-5% faster at p = 2..8.  With the metric from the vertices the map is
  // read: computing the indices there costs 40-110 VGPRs (the per-thread
  // node offsets stay live across the patch loop) and was level at p = 4,
  // 17% slower at p = 6 and 30% slower at p = 8.
  constexpr bool CALC = STORED && !BATCH;
  const uint32_t NX = lay.n[0] * P + 1, NY = lay.n[1] * P + 1, NZ = lay.n[2] * P + 1;
  // loads of patch `pt` into registers: its map entries and vertex coordinates
  uint32_t gidx[PER];
  // the staged patch's DoF indices for the atomic scatter (the same thread
  // stages and scatters DoF tid + k THREADS); the deterministic scatter
  // reads them from LDS (sidx) in its loop
  uint32_t cidx[PER];
  double xv[VPT];
  auto request = [&](uint32_t pt) {
    uint32_t px = 0, py = 0, pz = 0, n[3] = {0, 0, 0}, inst = 0;
    size_t c0 = 0;
    const bool live = locate(pt, px, py, pz, n, c0, inst);
    if constexpr (CALC) {
      // node (lx, ly, lz) of the patch is node (px SX + lx, ...) of the box's
      // node grid; boundary nodes are constrained
      const uint32_t gx0 = px * (BX * P), gy0 = py * (BY * P), gz0 = pz * (BZ * P);
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const int i = tid + k * THREADS;
        const uint32_t gx = gx0 + i % PX, gy = gy0 + (i / PX) % PY, gz = gz0 + i / (PX * PY);
        const bool in = live && i < P3 && gx - 1 < NX - 2 && gy - 1 < NY - 2 && gz - 1 < NZ - 2;
        gidx[k] = in ? gx + NX * (gy + NY * gz) : kInvalid;
      }
    } else {
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const int i = tid + k * THREADS;
        gidx[k] = (live && i < P3) ? pmap[(size_t)pt * P3 + i] : kInvalid;
      }
    }
#pragma unroll
    for (int k = 0; k < (VERT ? VPT : 0); ++k) {
      const int t = tid + k * THREADS, vc = t / 24, vk = t - vc * 24;
      const uint32_t ex = px * BX + vc % BX, ey = py * BY + (vc / BX) % BY,
                     ez = pz * BZ + vc / (BX * BY);
      xv[k] = 0.0;
      if (live && vc < CPP && ex < n[0] && ey < n[1] && ez < n[2])
        xv[k] = cellX[(c0 + ex + (size_t)n[0] * ((size_t)ey + (size_t)n[1] * ez)) * 24 + vk];
    }
  };
  T vals[PER];
  auto request_values = [&]() {
#pragma unroll
    for (int k = 0; k < PER; ++k)
      vals[k] = gidx[k] != kInvalid ? src[gidx[k] & 0x7FFFFFFFu] : T(0);
  };

  // STORED: the thread's column of G for patch `pt`
  T gq[STORED ? 6 : 1][STORED ? NQ : 1];
  auto request_geo = [&](uint32_t pt) {
    if constexpr (STORED) {
      uint32_t px = 0, py = 0, pz = 0, n[3] = {0, 0, 0}, inst = 0;
      size_t c0 = 0;
      const bool live = locate(pt, px, py, pz, n, c0, inst);
      if (live && lane_ok && px * BX + cx < n[0] && py * BY + cy < n[1] && pz * BZ + cz < n[2]) {
        const T *Gq = G + (size_t)pt * (6 * NQ * C::GTP) + c * NQ2 + col;
#pragma unroll
        for (int k = 0; k < 6; ++k)
#pragma unroll
          for (int z = 0; z < NQ; ++z)
            gq[k][z] = __builtin_nontemporal_load(Gq + (k * NQ + z) * C::GTP);
      }
    }
  };

  uint32_t cur = blockIdx.x;
  request(cur);
  request_geo(cur);
  request_values();
  double dot = 0.0;
  // batch mode with partials: `dot` runs over the workgroup's patches of
  // one instance (consecutive in its patch sequence, since the patches are
  // concatenated in instance order) and is stored per wave when the
  // instance changes, in partials[(slot[inst] * gridDim + workgroup) *
  // waves + wave].  Slots of instances the workgroup has no patch of are not
  // written: the caller keeps them zero.
  constexpr int WAVES = (THREADS + 63) / 64;
  uint32_t run_inst = 0xFFFFFFFFu;
  auto store_run = [&]() {
    double s = dot;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((tid & 63) == 0)
      partials[((size_t)ba.slot[run_inst] * gridDim.x + blockIdx.x) * WAVES + (tid >> 6)] = s;
    dot = 0.0;
  };
  for (; cur < npatch; cur += step) {
    // 1. stage patch `cur`, request the map and vertices of the next one
    __syncthreads();  // the previous patch's readers of the LDS arrays are done
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int i = tid + k * THREADS;
      if (i < P3) {
        spu[i] = vals[k];
        if constexpr (!DET && !ALIAS) spv[i] = T(0);
        if constexpr (DET) sidx[i] = gidx[k];
      }
      cidx[k] = gidx[k];
    }
#pragma unroll
    for (int k = 0; k < (VERT ? VPT : 0); ++k)
      if (tid + k * THREADS < CPP * 24) sX[tid + k * THREADS] = (T)xv[k];
    request(cur + step);
    __syncthreads();

    // 2. gradient, metric, fluxes
    uint32_t px = 0, py = 0, pz = 0, ncell[3] = {0, 0, 0}, inst_now = 0;
    size_t c0 = 0;
    const bool live = locate(cur, px, py, pz, ncell, c0, inst_now);
    if constexpr (BATCH && DOT) {
      if (inst_now != run_inst) {  // uniform: every thread has the same patch
        if (run_inst != 0xFFFFFFFFu) store_run();
        run_inst = inst_now;
      }
    }
    const bool active = lane_ok && live && px * BX + cx < ncell[0] && py * BY + cy < ncell[1] &&
                        pz * BZ + cz < ncell[2];
    const int base = cx * P + PX * (cy * P + PY * cz * P);
    // The trilinear cell x(xi, eta, zeta) = sum_v x_v (bilinear weights) has
    // Jacobian columns, along the (xi, eta) column of a thread,
    //   J0 = a0 + zeta da,  J1 = b0 + zeta db,  J2 = jz (constant),
    //   a0 = A0 + eta A1, da = K1 + eta K3, b0 = G0 + xi A1, db = K2 + xi K3,
    //   jz = K0 + xi K1 + eta db,
    // with the per-cell vectors (vertex v = a + 2b + 4c, bits of xi/eta/zeta)
    //   A0 = x1-x0, A1 = x3-x2-x1+x0, G0 = x2-x0, K0 = x4-x0,
    //   K1 = x5-x1-x4+x0, K2 = x6-x2-x4+x0, K3 = x7-x6-x5+x4-x3+x2+x1-x0.
    // The cofactor columns C0 = J1 x J2, C1 = J2 x J0, C2 = J0 x J1 are rows
    // of det J J^-1, det J = J2 . C2, hence with W = sum_b (du/dxi_b) C_b:
    //   (G grad u)_a = (w / det J) C_a . W,  G = w det J J^-1 J^-T.
    // CELLCOEF forms the cofactors per point from a0, da, b0, db, jz; the
    // other form expands them per column as polynomials in zeta:
    //   C0 = P0 + zeta P1, C1 = Q0 + zeta Q1, C2 = R0 + zeta R1 + zeta^2 R2.
    T a0[3], da[3], b0[3], db[3], jz[3];
    constexpr int NP = C::CELLCOEF ? 1 : 3;
    T P0[NP], P1[NP], Q0[NP], Q1[NP], R0[NP], R1[NP], R2[NP];
    auto column_metric = [&]() {
      if constexpr (C::CELLCOEF) {
        const T *K = sK + c * 21;  // coefficient k of coordinate d at K[7 d + k]
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const T A0 = K[7 * d], A1 = K[7 * d + 1], G0 = K[7 * d + 2], K0 = K[7 * d + 3];
          const T K1 = K[7 * d + 4], K2 = K[7 * d + 5], K3 = K[7 * d + 6];
          a0[d] = A0 + eta * A1;
          da[d] = K1 + eta * K3;
          b0[d] = G0 + xi * A1;
          db[d] = K2 + xi * K3;
          jz[d] = (K0 + xi * K1) + eta * db[d];
        }
      } else {
        const T *X = sX + c * 24;  // vertex v, coordinate d at X[3v + d]
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const T x0 = X[d], x1 = X[3 + d], x2 = X[6 + d], x3 = X[9 + d];
          const T x4 = X[12 + d], x5 = X[15 + d], x6 = X[18 + d], x7 = X[21 + d];
          const T e0 = (1 - eta) * (x1 - x0) + eta * (x3 - x2);
          const T e1 = (1 - eta) * (x5 - x4) + eta * (x7 - x6);
          const T f0 = (1 - xi) * (x2 - x0) + xi * (x3 - x1);
          const T f1 = (1 - xi) * (x6 - x4) + xi * (x7 - x5);
          a0[d] = e0;
          da[d] = e1 - e0;
          b0[d] = f0;
          db[d] = f1 - f0;
          jz[d] = (1 - xi) * (1 - eta) * (x4 - x0) + xi * (1 - eta) * (x5 - x1) +
                  (1 - xi) * eta * (x6 - x2) + xi * eta * (x7 - x3);
        }
        T t1[3], t2[3];
        cross(b0, jz, P0);
        cross(db, jz, P1);
        cross(jz, a0, Q0);
        cross(jz, da, Q1);
        cross(a0, b0, R0);
        cross(a0, db, t1);
        cross(da, b0, t2);
        cross(da, db, R2);
#pragma unroll
        for (int d = 0; d < 3; ++d) R1[d] = t1[d] + t2[d];
      }
    };
    // fluxes (G grad u) at quadrature point z of the column from the
    // reference gradient (dx, dy, dz)
    auto flux = [&](int z, T dx, T dy, T dz, T &fx, T &fy, T &fzz) {
      const T zeta = gxq[z];
      T C0[3], C1[3], C2[3], W[3];
      if constexpr (C::CELLCOEF) {
        T J0[3], J1[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          J0[d] = a0[d] + zeta * da[d];
          J1[d] = b0[d] + zeta * db[d];
        }
        cross(J1, jz, C0);
        cross(jz, J0, C1);
        cross(J0, J1, C2);
      } else {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          C0[d] = P0[d] + zeta * P1[d];
          C1[d] = Q0[d] + zeta * Q1[d];
          C2[d] = R0[d] + zeta * (R1[d] + zeta * R2[d]);
        }
      }
      const T det = jz[0] * C2[0] + jz[1] * C2[1] + jz[2] * C2[2];
      const T sc = wxy * gw[z] * recip(det);
#pragma unroll
      for (int d = 0; d < 3; ++d) W[d] = dx * C0[d] + dy * C1[d] + dz * C2[d];
      fx = sc * (C0[0] * W[0] + C0[1] * W[1] + C0[2] * W[2]);
      fy = sc * (C1[0] * W[0] + C1[1] * W[1] + C1[2] * W[2]);
      fzz = sc * (C2[0] * W[0] + C2[1] * W[1] + C2[2] * W[2]);
    };

    // Line form: every 1D contraction is done by a thread that holds the
    // whole line in registers, so each operand is read from LDS once (not
    // NQ times), with the even-odd split of the derivative matrix and its
    // entries as compile-time constants.  Thread `col` = (l0, l1) of cell c
    // owns the x-line (y = l0, z = l1; skewed layout: y = l1, z = l0), the
    // y-line (x = l0, z = l1) and the z-column (x = qx, y = qy) of the cell;
    // sfx / sfy hold the cell's x / y derivatives, then its x / y fluxes,
    // then their transposed contractions.
    constexpr GllD<NQ> kD{};
    auto dm = [&](int i, int a) { return kD.D[i][a]; };   // D
    auto dmt = [&](int i, int a) { return kD.D[a][i]; };  // D^T
    T *A = sfx + c * ACS, *B = sfy + c * BCS;
    const int l0 = col % NQ, l1 = col / NQ;
    const int xy = C::SKEW ? l1 : l0, xz = C::SKEW ? l0 : l1;  // the thread's x-line
    // CELLCOEF: the per-cell coefficient vectors of the column metric, from
    // the staged vertices (read after the next barrier)
    // (with whole cells per wave, each wave forms those of its own cells,
    // one per lane)
    const int kj = C::WAVECELL ? (tid >> 6) * C::CW * 3 + (tid & 63) : tid;
    const bool kj_ok = C::WAVECELL ? (tid & 63) < C::CW * 3 : true;
    for (int j = kj; VERT && C::CELLCOEF && kj_ok && j < CPP * 3;
         j += C::WAVECELL ? CPP * 3 : THREADS) {  // j = 3 cell + coordinate
      const T *X = sX + (j / 3) * 24 + j % 3;
      const T x0 = X[0], x1 = X[3], x2 = X[6], x3 = X[9];
      const T x4 = X[12], x5 = X[15], x6 = X[18], x7 = X[21];
      T *Kd = sK + (j / 3) * 21 + 7 * (j % 3);
      const T a0 = x1 - x0, a1 = (x3 - x2) - a0, k0 = x4 - x0, k1 = (x5 - x1) - k0;
      Kd[0] = a0;
      Kd[1] = a1;
      Kd[2] = x2 - x0;
      Kd[3] = k0;
      Kd[4] = k1;
      Kd[5] = (x6 - x2) - k0;
      Kd[6] = ((x7 - x6) - (x5 - x4)) - a1;
    }
    if (active) {
      T ln[NQ], r[NQ];
#pragma unroll
      for (int a = 0; a < NQ; ++a) ln[a] = spu[base + a + PX * (xy + PY * xz)];
      eo_mat<NQ, NQ, -1>(dm, ln, r);
#pragma unroll
      for (int i = 0; i < NQ; ++i) A[xz * AZS + xy * NQ + i] = r[i];
#pragma unroll
      for (int a = 0; a < NQ; ++a) ln[a] = spu[base + l0 + PX * (a + PY * l1)];
      eo_mat<NQ, NQ, -1>(dm, ln, r);
#pragma unroll
      for (int i = 0; i < NQ; ++i) B[l1 * BZS + i * NQ + l0] = r[i];
    }
    cell_sync();
    T vz[NQ];
    if (active) {
      if constexpr (VERT) column_metric();
      T u[NQ], dz[NQ], fz[NQ];
#pragma unroll
      for (int z = 0; z < NQ; ++z) u[z] = spu[base + qx + PX * (qy + PY * z)];
      eo_mat<NQ, NQ, -1>(dm, u, dz);
#pragma unroll
      for (int z = 0; z < NQ; ++z) {
        T fx, fy;
        const T gx = A[z * AZS + col], gy = B[z * BZS + col];
        if constexpr (VERT) {
          flux(z, gx, gy, dz[z], fx, fy, fz[z]);
        } else {
          fx = gq[0][z] * gx + gq[1][z] * gy + gq[2][z] * dz[z];
          fy = gq[1][z] * gx + gq[3][z] * gy + gq[4][z] * dz[z];
          fz[z] = gq[2][z] * gx + gq[4][z] * gy + gq[5][z] * dz[z];
        }
        A[z * AZS + col] = fx;
        B[z * BZS + col] = fy;
        // batch mode: p.Ap as the sum of the cells' energies u_c^T A_c u_c
        // (constrained entries gather as zero, so this is the sum over the
        // free rows); the registers are live here, no extra LDS reads
        if constexpr (BATCH && DOT)
          dot += (double)gx * (double)fx + (double)gy * (double)fy + (double)dz[z] * (double)fz[z];
      }
      eo_mat<NQ, NQ, -1>(dmt, fz, vz);
    }
    // the next patch's map has had the gradient phase to arrive: request
    // its values (and G), which then have the rest of this patch to arrive
    request_values();
    request_geo(cur + step);
    cell_sync();
    if constexpr (ALIAS) {
#pragma unroll
      for (int k = 0; k < PER; ++k)
        if (tid + k * THREADS < P3) spu[tid + k * THREADS] = T(0);
    }
    if (active) {
      T ln[NQ], r[NQ];
#pragma unroll
      for (int i = 0; i < NQ; ++i) ln[i] = A[xz * AZS + xy * NQ + i];
      eo_mat<NQ, NQ, -1>(dmt, ln, r);
#pragma unroll
      for (int k = 0; k < NQ; ++k) A[xz * AZS + xy * NQ + k] = r[k];
#pragma unroll
      for (int i = 0; i < NQ; ++i) ln[i] = B[l1 * BZS + i * NQ + l0];
      eo_mat<NQ, NQ, -1>(dmt, ln, r);
#pragma unroll
      for (int k = 0; k < NQ; ++k) B[l1 * BZS + k * NQ + l0] = r[k];
    }
    cell_sync();
    // 3. the column's sum of the three transposed contractions.  Atomic
    // scatter: added into the patch accumulator with LDS atomics (ds_add_f64;
    // cells of one patch share faces).  Deterministic scatter: written in
    // place into the cell's own array, the cell's result at its nodes.
    if (active) {
#pragma unroll
      for (int z = 0; z < NQ; ++z) {
        const T v = A[z * AZS + col] + B[z * BZS + col] + vz[z];
        if constexpr (DET)
          A[z * AZS + col] = v;
        else
          unsafeAtomicAdd(&acc[base + qx + PX * (qy + PY * z)], v);
      }
    }
    __syncthreads();

    // 4. scatter the patch.  Every patch DoF goes out as an atomic add: plain
    // stores to the DoFs no other patch touches were measured 2x slower
    // overall, because they share cache lines with atomically updated ones;
    // adding each cell's points to dst directly (no patch sum) was 2x slower
    // at p = 4, for the ~30% more global atomics.  Summing each patch DoF
    // from the cells' own arrays instead of the LDS accumulator (cell_sum
    // below, no accumulator and the map entries in registers) was slower at
    // p = 4, 6, 8 (26%, 14%, 5%), although it took p = 8 to 3 workgroups
    // per CU.
    //
    // Value of patch DoF i from the cells' own arrays (DET): the
    // results of the (1, 2, 4 or 8) active cells of the patch that hold its
    // node, in ascending cell order.  The node is node (ax, ay, az) of the
    // highest cell (hx, hy, hz) holding it, and also the last node of the
    // cell below along each axis where its index in that cell is 0; a cell
    // past the mesh (partial patch) holds no result.
    auto cell_sum = [&](int i) -> T {
      constexpr int DX = -ACS + P, DY = -BX * ACS + P * NQ, DZ = -BX * BY * ACS + P * AZS;
      const int lx = i % PX, ly = (i / PX) % PY, lz = i / (PX * PY);
      const int hx = min(lx / P, BX - 1), hy = min(ly / P, BY - 1), hz = min(lz / P, BZ - 1);
      const int ax = lx - hx * P, ay = ly - hy * P, az = lz - hz * P;
      const int x0 = (hx > 0 && ax == 0) ? 0 : 1, y0 = (hy > 0 && ay == 0) ? 0 : 1,
                z0 = (hz > 0 && az == 0) ? 0 : 1;
      const int x1 = px * BX + hx < ncell[0] ? 2 : 1, y1 = py * BY + hy < ncell[1] ? 2 : 1,
                z1 = pz * BZ + hz < ncell[2] ? 2 : 1;
      const T *S = sfx + (hx + BX * (hy + BY * hz)) * ACS + az * AZS + ay * NQ + ax;
      T v = T(0);
      for (int iz = z0; iz < z1; ++iz)
        for (int iy = y0; iy < y1; ++iy)
          for (int ix = x0; ix < x1; ++ix) v += S[(iz ? 0 : DZ) + (iy ? 0 : DY) + (ix ? 0 : DX)];
      return v;
    };
    if constexpr (!DET) {
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const int i = tid + k * THREADS;
        if (i < P3) {
          const uint32_t gi = cidx[k];
          if (gi != kInvalid) {
            const T v = acc[i];
            if (DOT && !BATCH) dot += (double)spu[i] * (double)v;
            unsafeAtomicAdd(dst + (gi & 0x7FFFFFFFu), v);
          }
        }
      }
    } else {
      // Deterministic scatter: the patch's sums (cell_sum, a fixed order)
      // are stored whole, in patch order, and k_patch_gather adds them up
      // per DoF in a fixed order.
      T *pb = pbuf + (size_t)cur * P3;
#pragma unroll 1
      for (int k = 0; k < PER; ++k) {
        const int i = tid + k * THREADS;
        if (i < P3 && sidx[i] != kInvalid) {
          const T v = cell_sum(i);
          if (DOT) dot += (double)spu[i] * (double)v;
          pb[i] = v;
        }
      }
    }
  }
  if constexpr (BATCH && DOT) {
    if (run_inst != 0xFFFFFFFFu) store_run();
  }
  if constexpr (DOT && !BATCH) {
    double s = dot;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((tid & 63) == 0) red[tid >> 6] = s;
    __syncthreads();
    if (tid == 0) {
      double t = 0.0;
#pragma unroll
      for (int i = 0; i < (THREADS + 63) / 64; ++i) t += red[i];
      partials[blockIdx.x] = t;
    }
  }
}

// patch DoF map: bit 31 marks DoFs on the patch boundary (shared with a
// neighbouring patch); constrained DoFs and DoFs outside the mesh are invalid.
__global__ void k_patch_map(PatchLayout lay, int p, int bx, int by, int bz, uint32_t *pmap) {
  const int PX = bx * p + 1, PY = by * p + 1, PZ = bz * p + 1;
  const uint64_t P3 = (uint64_t)PX * PY * PZ;
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t npatch = (uint64_t)lay.np[0] * lay.np[1] * lay.np[2];
  if (t >= npatch * P3) return;
  const uint64_t patch = t / P3;
  const int i = (int)(t - patch * P3);
  const int lx = i % PX, ly = (i / PX) % PY, lz = i / (PX * PY);
  const uint64_t ppx = patch % lay.np[0], ppy = (patch / lay.np[0]) % lay.np[1],
                 ppz = patch / ((uint64_t)lay.np[0] * lay.np[1]);
  const uint64_t gx = ppx * bx * p + lx, gy = ppy * by * p + ly, gz = ppz * bz * p + lz;
  const uint64_t Nx = (uint64_t)lay.n[0] * p + 1, Ny = (uint64_t)lay.n[1] * p + 1,
                 Nz = (uint64_t)lay.n[2] * p + 1;
  uint32_t v = kInvalid;
  const bool inside = gx < Nx && gy < Ny && gz < Nz;
  const bool bnd = gx == 0 || gy == 0 || gz == 0 || gx == Nx - 1 || gy == Ny - 1 || gz == Nz - 1;
  if (inside && !bnd) {
    const bool shared = lx == 0 || ly == 0 || lz == 0 || lx == PX - 1 || ly == PY - 1 || lz == PZ - 1;
    v = (uint32_t)(gx + Nx * (gy + Ny * gz)) | (shared ? 0x80000000u : 0u);
  }
  pmap[t] = v;
}

// Deterministic scatter, second half: one thread per node of the box's node
// grid adds the sums the patches containing the node stored for it
// (pbuf[patch][local], from k_patch in deterministic mode) in ascending patch
// order -- up to two patches per direction, the lower one first when the
// node lies on their shared face -- to dst.  Constrained nodes (invalid in
// the patch map) are left alone.  ASSIGN: dst is set instead (constrained
// nodes to src), which spares the vmult its start pass and the read of dst.
// Consecutive lanes take consecutive nodes and every lane's up to eight sums are
// loaded before one is used.  (Workgroups of 128 nodes of one node row left half
// of their lanes idle on 136-node rows and waited for each sum, and for the
// patch map's word, in turn: 23 us at 1.95M nodes, p = 3, now 10.)
template <typename T, int P, int BX, int BY, int BZ, bool ASSIGN>
__global__ void __launch_bounds__(256)
k_patch_gather(PatchLayout lay, const T *__restrict__ pbuf, const T *__restrict__ src,
               T *__restrict__ dst, const int *__restrict__ skip) {
  if (skip && *skip) return;  // converged CG: the patch kernel stored nothing
  constexpr uint32_t SX = BX * P, SY = BY * P, SZ = BZ * P;
  constexpr uint32_t PX = SX + 1, PY = SY + 1, P3 = PX * PY * (SZ + 1);
  const uint32_t Nx = lay.n[0] * P + 1, Ny = lay.n[1] * P + 1, Nz = lay.n[2] * P + 1;
  const uint64_t node = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (node >= (uint64_t)Nx * Ny * Nz) return;
  const uint32_t row = (uint32_t)node / Nx, gx = (uint32_t)node - row * Nx;  // N < 2^32
  const uint32_t gz = row / Ny, gy = row - gz * Ny;
  if (gx == 0 || gx == Nx - 1 || gy == 0 || gy == Ny - 1 || gz == 0 || gz == Nz - 1) {
    if (ASSIGN) dst[node] = src[node];  // the boundary is constrained
    return;
  }
  // highest patch holding the node along each axis, and its local index
  const uint32_t qx = min(gx / SX, lay.np[0] - 1), qy = min(gy / SY, lay.np[1] - 1),
                 qz = min(gz / SZ, lay.np[2] - 1);
  const uint32_t lx = gx - qx * SX, ly = gy - qy * SY, lz = gz - qz * SZ;
  const uint64_t pid = qx + (uint64_t)lay.np[0] * (qy + (uint64_t)lay.np[1] * qz);
  const T *at = pbuf + pid * P3 + lx + PX * (ly + PY * lz);
  // offsets to the same node in the lower patch along x, y, z, which holds it as
  // its last one
  const long dx = -(long)P3 + SX;
  const long dy = -(long)lay.np[0] * P3 + (long)SY * PX;
  const long dz = -(long)lay.np[0] * lay.np[1] * P3 + (long)SZ * PX * PY;
  const bool x0 = qx > 0 && lx == 0, y0 = qy > 0 && ly == 0, z0 = qz > 0 && lz == 0;
  T v[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    v[k] = T(0);
    if ((k & 1 || x0) && (k & 2 || y0) && (k & 4 || z0))
      v[k] = at[(k & 1 ? 0 : dx) + (k & 2 ? 0 : dy) + (k & 4 ? 0 : dz)];
  }
  T sum = T(0);
#pragma unroll
  for (int k = 0; k < 8; ++k) sum += v[k];
  dst[node] = ASSIGN ? sum : dst[node] + sum;
}

template <typename T, class C, bool DOT, bool BATCH = false, bool DET = false, bool STORED = false>
uint32_t resident_grid(uint32_t n_patches) {
  int dev = 0, cus = 0, per_cu = 0;
  MFX_HIP(hipGetDevice(&dev));
  MFX_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  MFX_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(
      &per_cu, k_patch<T, C, DOT, BATCH, DET, STORED>, C::THREADS, 0));
  MFX_REQUIRE(cus > 0 && per_cu > 0, "patch kernel does not fit the device");
  const uint64_t g = (uint64_t)cus * per_cu;
  return (uint32_t)std::min<uint64_t>(g, std::max<uint32_t>(n_patches, 1));
}
template <typename T, class C, bool DOT, bool DET = false, bool STORED = false>
uint32_t grid_of(const PatchLayout &lay) {
  return resident_grid<T, C, DOT, false, DET, STORED>(patch_count(lay));
}

template <typename T, class C, bool STORED>
void launch_patch_v(const PatchOp<T> &o, const T *src, T *dst, hipStream_t s, double *partials,
                    const int *skip) {
  // the kernels that return partials write one per workgroup: their grid
  // is the partial count the caller sized the buffer for
  const bool det = o.pbuf != nullptr;
  if (partials) {
    if constexpr (std::is_same<T, double>::value) {
      const uint32_t g = det ? o.grid.det_dot : o.grid.dot;
      MFX_REQUIRE(g > 0, "patch grid not set up");
      if (det)
        hipLaunchKernelGGL((k_patch<T, C, true, false, true, STORED>), dim3(g), dim3(C::THREADS),
                           0, s, o.w, o.xq, o.cellX, src, dst, o.pmap, o.lay, partials, skip,
                           BatchArgs{}, o.pbuf, o.G);
      else
        hipLaunchKernelGGL((k_patch<T, C, true, false, false, STORED>), dim3(g),
                           dim3(C::THREADS), 0, s, o.w, o.xq, o.cellX, src, dst, o.pmap, o.lay,
                           partials, skip, BatchArgs{}, (T *)nullptr, o.G);
    } else {
      throw Error{MFX_ERR_UNSUPPORTED, "patch kernel: partials need FP64"};
    }
  } else {
    const uint32_t g = det ? o.grid.det_plain : o.grid.plain;
    MFX_REQUIRE(g > 0, "patch grid not set up");
    if (det)
      hipLaunchKernelGGL((k_patch<T, C, false, false, true, STORED>), dim3(g), dim3(C::THREADS),
                         0, s, o.w, o.xq, o.cellX, src, dst, o.pmap, o.lay, nullptr, nullptr,
                         BatchArgs{}, o.pbuf, o.G);
    else
      hipLaunchKernelGGL((k_patch<T, C, false, false, false, STORED>), dim3(g), dim3(C::THREADS),
                         0, s, o.w, o.xq, o.cellX, src, dst, o.pmap, o.lay, nullptr, nullptr,
                         BatchArgs{}, (T *)nullptr, o.G);
  }
}

template <typename T, class C>
void launch_patch_t(const PatchOp<T> &o, const T *src, T *dst, hipStream_t s, double *partials,
                    const int *skip, bool assign) {
  MFX_REQUIRE(!assign || (o.pbuf && !skip), "assigning apply: deterministic scatter only");
  // the kernel indexes the patch map with its compile-time patch size: the
  // map must have been built for exactly this shape
  MFX_REQUIRE(o.shape.bx == C::BX && o.shape.by == C::BY && o.shape.bz == C::BZ,
              "patch shape of the operator does not match the kernel instance");
  const int b[3] = {C::BX, C::BY, C::BZ};
  for (int k = 0; k < 3; ++k)
    MFX_REQUIRE(o.lay.np[k] == (o.lay.n[k] + b[k] - 1) / b[k], "patch layout inconsistent with shape");
  MFX_REQUIRE(o.pmap && o.w && o.xq && (o.cellX || o.G), "patch operator arrays missing");
  if (o.G)
    launch_patch_v<T, C, true>(o, src, dst, s, partials, skip);
  else
    launch_patch_v<T, C, false>(o, src, dst, s, partials, skip);
  MFX_HIP(hipGetLastError());
  if (o.pbuf) {
    // deterministic mode: add the stored patch sums per node, in patch order
    const uint64_t nodes = ((uint64_t)o.lay.n[0] * C::P + 1) * ((uint64_t)o.lay.n[1] * C::P + 1) *
                           ((uint64_t)o.lay.n[2] * C::P + 1);
    const dim3 grid((unsigned)((nodes + 255) / 256)), block(256);
    if (assign)
      hipLaunchKernelGGL((k_patch_gather<T, C::P, C::BX, C::BY, C::BZ, true>), grid, block, 0, s,
                         o.lay, o.pbuf, src, dst, skip);
    else
      hipLaunchKernelGGL((k_patch_gather<T, C::P, C::BX, C::BY, C::BZ, false>), grid, block, 0, s,
                         o.lay, o.pbuf, src, dst, skip);
    MFX_HIP(hipGetLastError());
  }
}

}  // namespace

PatchShape patch_shape(int p) {
  return with_cfg(p, [](auto c) {
    using C = decltype(c);
    return PatchShape{C::BX, C::BY, C::BZ};
  });
}

uint32_t patch_count(const PatchLayout &lay) { return lay.np[0] * lay.np[1] * lay.np[2]; }

template <typename T, bool STORED>
PatchGrid patch_grid_v(int p, const PatchLayout &lay) {
  return with_cfg(p, [&](auto c) {
    using C = decltype(c);
    PatchGrid g;
    g.plain = grid_of<T, C, false, false, STORED>(lay);
    g.det_plain = grid_of<T, C, false, true, STORED>(lay);
    if constexpr (std::is_same<T, double>::value) {
      g.dot = grid_of<T, C, true, false, STORED>(lay);
      g.det_dot = grid_of<T, C, true, true, STORED>(lay);
    }
    return g;
  });
}
template <typename T>
PatchGrid patch_grid(int p, const PatchLayout &lay, bool stored) {
  return stored ? patch_grid_v<T, true>(p, lay) : patch_grid_v<T, false>(p, lay);
}
template PatchGrid patch_grid<double>(int, const PatchLayout &, bool);
template PatchGrid patch_grid<float>(int, const PatchLayout &, bool);

template <typename T>
void launch_patch(const PatchOp<T> &o, const T *src, T *dst, hipStream_t s, double *partials,
                  const int *skip, bool assign) {
  with_cfg(o.p,
           [&](auto c) { launch_patch_t<T, decltype(c)>(o, src, dst, s, partials, skip, assign); });
}
template void launch_patch<double>(const PatchOp<double> &, const double *, double *, hipStream_t,
                                   double *, const int *, bool);
template void launch_patch<float>(const PatchOp<float> &, const float *, float *, hipStream_t,
                                  double *, const int *, bool);

uint32_t patch_batch_grid(int p, uint32_t n_patches, bool dot) {
  return with_cfg(p, [&](auto c) {
    using C = decltype(c);
    return dot ? resident_grid<double, C, true, true>(n_patches)
               : resident_grid<double, C, false, true>(n_patches);
  });
}

void launch_patch_batch(const PatchBatchOp &o, const double *src, double *dst, const int *done,
                        hipStream_t s, double *partials) {
  MFX_REQUIRE(o.pmap && o.meta && o.inst && o.cellX && o.w && o.xq, "batch patch arrays missing");
  if (o.n_patches == 0) return;
  with_cfg(o.p, [&](auto c) {
    using C = decltype(c);
    const BatchArgs ba{o.meta, o.inst, done, o.n_patches, o.slot};
    if (partials) {
      MFX_REQUIRE(o.grid_dot > 0, "batch patch grid not set up");
      hipLaunchKernelGGL((k_patch<double, C, true, true>), dim3(o.grid_dot), dim3(C::THREADS), 0,
                         s, o.w, o.xq, o.cellX, src, dst, o.pmap, PatchLayout{}, partials,
                         nullptr, ba, (double *)nullptr, (const double *)nullptr);
    } else {
      MFX_REQUIRE(o.grid > 0, "batch patch grid not set up");
      hipLaunchKernelGGL((k_patch<double, C, false, true>), dim3(o.grid), dim3(C::THREADS), 0, s,
                         o.w, o.xq, o.cellX, src, dst, o.pmap, PatchLayout{}, nullptr, nullptr,
                         ba, (double *)nullptr, (const double *)nullptr);
    }
  });
  MFX_HIP(hipGetLastError());
}

uint32_t patch_batch_waves(int p) {
  return with_cfg(p, [](auto c) { return (uint32_t)((decltype(c)::THREADS + 63) / 64); });
}

namespace {
// Stored metric terms [cell][6][nq^3] (cells lexicographic) -> patch order
// [patch][6][NQ][GTP] as k_patch<..., STORED> reads them: entry c NQ^2 + col
// of a (patch, k, z) row belongs to column col of cell c of the patch;
// cells past the mesh and the row padding hold zero.
template <typename T, class C>
__global__ void k_patch_geometry(PatchLayout lay, const T *__restrict__ G, T *__restrict__ Gp) {
  constexpr int NQ = C::NQ, NQ2 = C::NQ2, NQ3 = C::NQ3;
  const uint64_t rows = (uint64_t)patch_count_d(lay) * 6 * NQ;
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * C::GTP) return;
  const uint64_t row = i / C::GTP;
  const int t = (int)(i - row * C::GTP);
  const uint32_t pt = (uint32_t)(row / (6 * NQ));
  const int kz = (int)(row - (uint64_t)pt * 6 * NQ), k = kz / NQ, z = kz - k * NQ;
  const int c = t / NQ2, col = t - c * NQ2;
  const bool ok = c < C::CPP;
  uint32_t px, py, pz;
  patch_xyz(lay, pt, px, py, pz);
  const uint32_t ex = px * C::BX + c % C::BX, ey = py * C::BY + (c / C::BX) % C::BY,
                 ez = pz * C::BZ + c / (C::BX * C::BY);
  T v = T(0);
  if (ok && ex < lay.n[0] && ey < lay.n[1] && ez < lay.n[2])
    v = G[(ex + (size_t)lay.n[0] * ((size_t)ey + (size_t)lay.n[1] * ez)) * 6 * NQ3 + k * NQ3 +
          z * NQ2 + col];
  Gp[i] = v;
}
}  // namespace

uint64_t patch_geometry_size(int p, const PatchLayout &lay) {
  return with_cfg(p, [&](auto c) {
    using C = decltype(c);
    return (uint64_t)patch_count(lay) * 6 * C::NQ * C::GTP;
  });
}

template <typename T>
void launch_patch_geometry(int p, const PatchLayout &lay, const T *G, T *Gp, hipStream_t s) {
  with_cfg(p, [&](auto c) {
    using C = decltype(c);
    const uint64_t n = (uint64_t)patch_count(lay) * 6 * C::NQ * C::GTP;
    hipLaunchKernelGGL((k_patch_geometry<T, C>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       s, lay, G, Gp);
  });
  MFX_HIP(hipGetLastError());
}
template void launch_patch_geometry<double>(int, const PatchLayout &, const double *, double *,
                                            hipStream_t);
template void launch_patch_geometry<float>(int, const PatchLayout &, const float *, float *,
                                           hipStream_t);

void launch_patch_map(const PatchLayout &lay, int p, PatchShape sh, uint32_t *pmap,
                      hipStream_t s) {
  const uint64_t P3 = (uint64_t)(sh.bx * p + 1) * (sh.by * p + 1) * (sh.bz * p + 1);
  const uint64_t n = (uint64_t)patch_count(lay) * P3;
  hipLaunchKernelGGL(k_patch_map, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, lay, p,
                     sh.bx, sh.by, sh.bz, pmap);
  MFX_HIP(hipGetLastError());
}

}  // namespace mfx
