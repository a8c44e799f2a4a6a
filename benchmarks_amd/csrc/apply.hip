// apply.hip -- sum-factorized scalar-Laplacian element kernels for gfx950.
//
// One kernel family covers the reference's BK3 (Gauss, interpolation B) and
// BK5 (GLL collocation, B = I) element operators
//   v_e = B^T D^T G_e D B u_e
// (CEED_bp/include/bk3_kokkos_kernel.h:113-382,
//  CEED_BK/include/kernels/BK5/templated_cuda_kernels.cuh:37-125), with the
// DoF-map gather (masked entries read as 0) and the scatter-add (masked
// entries skipped) of CEED_bp/include/bk3_kokkos_kernel.h:113-143, 356-382.
//
// Work decomposition (CDNA4, 64-wide wavefronts):
//   * a workgroup holds EPB elements, one thread per (x,y) quadrature column
//     (EPB * nq^2 <= 256 threads); each thread keeps its z-column in
//     registers, so z contractions are register-local and only the x and y
//     contractions go through LDS (3 LDS cubes per element);
//   * the map and G are read with the column index fastest, so every load
//     instruction of a wavefront touches contiguous 8-byte runs (G layout
//     [cell][6][q^3], x fastest);
//   * collocation kernel: where the registers allow (CollocTile), the 6 q-columns
//     of G a thread needs are loaded into them before the first barrier, so the
//     geometry stream is in flight while the dependent map -> src gather completes;
//   * scatter: hardware FP64/FP32 atomic add in L2 (global_atomic_add_f64).
// Cells per workgroup and the prefetch switch were chosen per nq by timing, at nq =
// 5 on 32M DoFs and at nq = 6 and 7 on 1.5M to 6M of general meshes in FP64, FP32 and the
// E-vector form (a remap of workgroups onto XCD-contiguous cell ranges was
// measured too and did not pay).
#include <type_traits>

#include "mfx_internal.hpp"
#include "tables.hpp"

namespace mfx {
namespace {

// Cells per workgroup (EPB) and G prefetch for the collocation kernel;
// the interpolation kernel keeps EPB = floor(256 / nq^2).
template <int NQ>
struct Tile {
  static constexpr int EPB = (256 / (NQ * NQ)) > 0 ? 256 / (NQ * NQ) : 1;
  static constexpr int THREADS = EPB * NQ * NQ;
};
// Without the prefetch of G (its registers) nq = 6 and 7 run 112 and 104 us instead of
// 134 and 126 on 4M DoFs, nq = 6 with 7 cells (3 with the prefetch); nq = 5 is faster
// with it, 5 cells (142, 174 without) and 10 cells 173.  FP32 needs half the
// registers: nq = 7 is faster with the prefetch (1.5M DoFs 35.0, 38.0 without; 6M 113,
// 122).  The E-vector form keeps it at nq = 6 too, with 3 cells (32.9 / 35.2, 109 / 127):
// it has no faces to join, which is what 7 cells are better for.
template <typename T, int NQ, bool GATHER = true>
struct CollocTile {
  static constexpr int EPB = NQ <= 5   ? 128 / (NQ * NQ)
                             : NQ == 6 ? (GATHER ? 7 : 3)
                             : NQ == 7 ? 1
                             : NQ == 8 ? 2
                                       : 3;
  static constexpr int THREADS = EPB * NQ * NQ;
  static constexpr bool PREFETCH =
      NQ <= 5 || (NQ == 6 && !GATHER) || (NQ == 7 && sizeof(T) == 4);
};

// A metric term.  A row of nq^2 terms that does not end at a 128-byte line shares
// its last line with the next row, which a wave reads later, so streaming it
// past the caches fetches that line twice.  Short rows are therefore kept (the
// default policy): vmult with stored terms, streamed -> kept, on 10M DoFs
// p = 1, q = 2 1554 -> 994 us (FP32 1345 -> 649), p = 2, q = 3 638 -> 504 (404 -> 309),
// p = 3, q = 5 610 -> 570 (391 -> 337), p = 4, q = 5 on 2M DoFs 77 -> 65 (51 -> 41).
// Rows of whole lines are read once (FP64 q = 4 783 kept, 761 streamed), and of
// long rows the shared line is too little to make up for what the stream
// evicts (FP64 q = 6 441 kept, 427 streamed; q = 9 347, 328).
// STREAM: stream whatever the length (kCollocStream).
template <typename T, int NQ, bool STREAM = false>
__device__ __forceinline__ T load_geo(const T *p) {
  constexpr int kRow = NQ * NQ * sizeof(T);
  if constexpr (STREAM || kRow % 128 == 0 || kRow > 256)
    return __builtin_nontemporal_load(p);
  else
    return *p;
}

__device__ __forceinline__ void atomic_add(double *p, double v) { unsafeAtomicAdd(p, v); }
__device__ __forceinline__ void atomic_add(float *p, float v) { unsafeAtomicAdd(p, v); }

// Sum over the workgroup; result valid in thread 0.
template <int THREADS>
__device__ __forceinline__ double block_sum(double v, double *red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  constexpr int NW = (THREADS + 63) / 64;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) red[w] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0) {
#pragma unroll
    for (int i = 0; i < NW; ++i) s += red[i];
  }
  return s;
}

// ---------------------------------------------------------------------------
// GLL collocation (BK5): NM == NQ, B = I.
// ---------------------------------------------------------------------------
// EPB cells per workgroup; PREF: G columns loaded into registers before the
// first barrier.  cell_inst / inst_done (optional): cells whose instance is
// flagged done are skipped (batched solves).
// JOIN: a face node that the map gives to two consecutive cells is added once (see
// k_apply_interp).  Not at nq = 5, where its registers beside the prefetched G cost
// more (68 -> 72 us); at nq = 9 by join_colloc.
template <int NQ, int EPB, bool PREF>
constexpr bool kCollocJoin = EPB > 2 && !(PREF && NQ >= 5);
// The prefetched rows of about 200 bytes, FP32 nq = 7, are streamed at any size (kept:
// 1.5M DoFs 35.7 -> 35.0 us, 3M 61.1 -> 62.5, 6M 109 -> 113); FP64 nq = 5 by stream_colloc.
template <typename T, int NQ>
constexpr bool kCollocStream = sizeof(T) == 4 && NQ == 7;
constexpr uint64_t kMemorySideCache = 256ull << 20;
template <typename T, int NQ, int EPB, bool PREF, bool GATHER, bool DOT,
          bool JOIN = GATHER && kCollocJoin<NQ, EPB, PREF>,
          bool STREAM = kCollocStream<T, NQ>>
__global__ void __launch_bounds__(EPB * NQ * NQ)
k_apply_colloc(const T *__restrict__ gD, const T *__restrict__ G,
               const T *__restrict__ src, T *__restrict__ dst,
               const uint32_t *__restrict__ map, uint32_t n_cells,
               double *__restrict__ partials, const int *__restrict__ skip,
               const uint16_t *__restrict__ cell_inst, const int *__restrict__ inst_done) {
  constexpr int THREADS = EPB * NQ * NQ;
  constexpr int NQ2 = NQ * NQ, NQ3 = NQ2 * NQ;
  __shared__ T sD[NQ * NQ];
  __shared__ T su[EPB][NQ3];
  __shared__ T sfx[EPB][NQ3];
  __shared__ T sfy[EPB][NQ3];
  __shared__ double red[(THREADS + 63) / 64];
  // JOIN: the DoFs of the cells' left and right x faces
  __shared__ uint32_t sL[JOIN ? EPB * NQ2 : 1], sR[JOIN ? EPB * NQ2 : 1];

  if (skip && *skip) return;  // converged CG: nothing left to do
  const int tid = threadIdx.x;
  const int el = tid / NQ2;
  const int col = tid - el * NQ2;
  const int qx = col % NQ, qy = col / NQ;
  const uint32_t e = blockIdx.x * EPB + el;
  bool active = e < n_cells;
  if (active && inst_done) active = inst_done[cell_inst[e]] == 0;

  for (int i = tid; i < NQ * NQ; i += THREADS) sD[i] = gD[i];

  // geometry columns first: independent of the gather, so in flight early
  const T *Ge = G + (size_t)(active ? e : 0) * 6 * NQ3 + col;
  T g[PREF ? 6 : 1][PREF ? NQ : 1];
  if (PREF && active) {
#pragma unroll
    for (int z = 0; z < NQ; ++z)
#pragma unroll
      for (int c = 0; c < 6; ++c) g[c][z] = load_geo<T, NQ, STREAM>(Ge + c * NQ3 + z * NQ2);
  }

  uint32_t idx[NQ];
  T u[NQ];
  if (active) {
    if (GATHER) {
      const uint32_t *me = map + (size_t)e * NQ3 + col;
#pragma unroll
      for (int z = 0; z < NQ; ++z) idx[z] = me[z * NQ2];
#pragma unroll
      for (int z = 0; z < NQ; ++z) u[z] = (idx[z] != kInvalid) ? src[idx[z]] : T(0);
    } else {
      const T *se = src + (size_t)e * NQ3 + col;
#pragma unroll
      for (int z = 0; z < NQ; ++z) u[z] = se[z * NQ2];
    }
#pragma unroll
    for (int z = 0; z < NQ; ++z) su[el][z * NQ2 + col] = u[z];
  }
  if constexpr (JOIN) {  // (cells left out give no DoF)
#pragma unroll
    for (int z = 0; z < NQ; ++z) {
      if (qx == 0) sL[el * NQ2 + z * NQ + qy] = active ? idx[z] : kInvalid;
      if (qx == NQ - 1) sR[el * NQ2 + z * NQ + qy] = active ? idx[z] : kInvalid;
    }
  }
  __syncthreads();

  T fz[NQ];
  if (active) {
#pragma unroll
    for (int z = 0; z < NQ; ++z) {
      T gxx, gxy, gxz, gyy, gyz, gzz;
      if constexpr (PREF) {
        gxx = g[0][z]; gxy = g[1][z]; gxz = g[2][z];
        gyy = g[3][z]; gyz = g[4][z]; gzz = g[5][z];
      } else {
        gxx = load_geo<T, NQ, STREAM>(Ge + 0 * NQ3 + z * NQ2);
        gxy = load_geo<T, NQ, STREAM>(Ge + 1 * NQ3 + z * NQ2);
        gxz = load_geo<T, NQ, STREAM>(Ge + 2 * NQ3 + z * NQ2);
        gyy = load_geo<T, NQ, STREAM>(Ge + 3 * NQ3 + z * NQ2);
        gyz = load_geo<T, NQ, STREAM>(Ge + 4 * NQ3 + z * NQ2);
        gzz = load_geo<T, NQ, STREAM>(Ge + 5 * NQ3 + z * NQ2);
      }
      T dx = 0, dy = 0, dz = 0;
#pragma unroll
      for (int a = 0; a < NQ; ++a) {
        dx += sD[qx * NQ + a] * su[el][z * NQ2 + qy * NQ + a];
        dy += sD[qy * NQ + a] * su[el][z * NQ2 + a * NQ + qx];
        dz += sD[z * NQ + a] * u[a];
      }
      sfx[el][z * NQ2 + col] = gxx * dx + gxy * dy + gxz * dz;
      sfy[el][z * NQ2 + col] = gxy * dx + gyy * dy + gyz * dz;
      fz[z] = gxz * dx + gyz * dy + gzz * dz;
    }
  }
  __syncthreads();

  double dot = 0.0;
  T vj[JOIN ? NQ : 1];
  T *lft = &su[0][0];  // [cell][z][y]: left faces that the cell before adds
  auto joined = [&](int z) {
    return qx == 0 && el > 0 && sR[(el - 1) * NQ2 + z * NQ + qy] == idx[z];
  };
  if (active) {
#pragma unroll
    for (int z = 0; z < NQ; ++z) {
      T v = 0;
#pragma unroll
      for (int a = 0; a < NQ; ++a) {
        v += sD[a * NQ + qx] * sfx[el][z * NQ2 + qy * NQ + a];
        v += sD[a * NQ + qy] * sfy[el][z * NQ2 + a * NQ + qx];
        v += sD[a * NQ + z] * fz[a];
      }
      if (DOT) dot += (double)u[z] * (double)v;
      if constexpr (JOIN) {
        vj[z] = v;
        if (joined(z)) lft[el * NQ2 + z * NQ + qy] = v;
      } else if (GATHER) {
        if (idx[z] != kInvalid) atomic_add(dst + idx[z], v);
      } else {
        dst[(size_t)e * NQ3 + z * NQ2 + col] = v;
      }
    }
  }
  if constexpr (JOIN) {
    __syncthreads();
    if (active) {
#pragma unroll
      for (int z = 0; z < NQ; ++z) {
        if (idx[z] == kInvalid || joined(z)) continue;
        T v = vj[z];
        if (qx == NQ - 1 && el + 1 < EPB && sL[(el + 1) * NQ2 + z * NQ + qy] == idx[z])
          v += lft[(el + 1) * NQ2 + z * NQ + qy];
        atomic_add(dst + idx[z], v);
      }
    }
  }
  if (DOT) {
    const double s = block_sum<THREADS>(dot, red);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
  }
}

// ---------------------------------------------------------------------------
// General tensor-product element (BK3): NM = p+1 nodes, NQ >= NM quadrature
// points, interpolation B[q][m] and collocation derivative D[q][k].
// ---------------------------------------------------------------------------
//
// OTF: the metric terms are computed per quadrature point from the 8
// vertices of the trilinear cell (cellX [E][8][3], Gauss points gxq and
// weights gwq on [0,1]) instead of being read from G: per cell seven
// coefficient vectors of the Jacobian (LDS), per (x,y) column its Jacobian
// columns as functions of zeta, per point the cofactor columns
// C0 = J1 x J2, C1 = J2 x J0, C2 = J0 x J1 (rows of det J J^-1), det J =
// J2 . C2 and (G grad u)_a = (w / det J) C_a . sum_b (du/dxi_b) C_b, with
// G = w det J J^-1 J^-T the stored form.  24 doubles per cell replace
// 48 nq^3 bytes of G.
//
// ROW (box meshes, cells and nodes numbered x fastest, boundary constrained; no map is read):
// each workgroup takes up to EPB consecutive cells of one x-row.  The scatter
// then first sums the cells' shared x-faces in LDS (the right face of cell
// c and the left face of cell c+1, in that order) and adds each node of the
// resulting row segment once, with consecutive lanes on consecutive nodes
// of an x-line: ~(p+1)^2 (EPB p + 1) atomic adds in few wide requests
// instead of EPB (p+1)^3 in requests of about p+1 lanes.  The device-scope
// FP atomics execute beyond the per-XCD L2s, and their request count bounds
// the per-cell scatter (measured: plain stores in their place made the FP32
// q = p+1 apply at 135M DoFs 2.1x faster).
//
// JOIN (a DoF map, any mesh): a face node that the map gives to both of two consecutive
// cells is added once, with the first cell's column: in an adapter's numbering a
// cell's left face lies strided in its neighbour's DoFs, a request per node or two.  On
// 1.75M DoFs, Gauss: p = 2, q = 3 143 -> 94 us, p = 4, q = 6 107 -> 91; p = 1 collocated
// 257 -> 143.  Not where the node columns are under half of the lanes (p = 1, q = 3:
// 374 -> 453 us with the metric from the vertices) or with few cells (q = 9 64 -> 66,
// q = 10 78 -> 84).  It costs a barrier and a pass through the LDS: join_faces.
template <int NM, int NQ>
constexpr bool kJoin = Tile<NQ>::EPB > 3 && 2 * NM * NM >= NQ * NQ;
template <typename T, int NM, int NQ, bool GATHER, bool DOT, bool OTF = false, bool ROW = false,
          bool AX = false, bool JOIN = GATHER && !ROW && kJoin<NM, NQ>>
__global__ void __launch_bounds__(Tile<NQ>::THREADS)
k_apply_interp(const T *__restrict__ gB, const T *__restrict__ gD,
               const T *__restrict__ G, const T *__restrict__ src,
               T *__restrict__ dst, const uint32_t *__restrict__ map,
               uint32_t n_cells, double *__restrict__ partials,
               const int *__restrict__ skip, const double *__restrict__ cellX,
               const T *__restrict__ gxq, const T *__restrict__ gwq, RowMesh rows,
               const T *__restrict__ geo) {
  constexpr int EPB = Tile<NQ>::EPB, NQ2 = NQ * NQ, NQ3 = NQ2 * NQ;
  static_assert(!AX || (OTF && ROW), "axis-aligned cells: a box-mesh form of the vertex metric");
  constexpr int NM2 = NM * NM, NM3 = NM2 * NM;
  constexpr int THREADS = Tile<NQ>::THREADS;
  __shared__ T sB[NQ * NM];
  __shared__ T sD[NQ * NQ];
  __shared__ T s0[EPB][NQ3];
  __shared__ T s1[EPB][NQ3];
  __shared__ T s2[EPB][NQ3];
  __shared__ T sXv[OTF ? EPB * 24 : 1];  // cell vertices, then
  __shared__ T sKc[OTF ? EPB * 21 : 1];  // per cell 7 Jacobian coefficient vectors
  __shared__ double red[(Tile<NQ>::THREADS + 63) / 64];
  // JOIN: the DoFs of the cells' left and right x faces
  static_assert(!JOIN || (GATHER && !ROW && kJoin<NM, NQ>), "faces are joined through a map");
  __shared__ uint32_t sL[JOIN ? EPB * NM2 : 1], sR[JOIN ? EPB * NM2 : 1];

  if (skip && *skip) return;  // converged CG: nothing left to do
  const int tid = threadIdx.x;
  const int el = tid / NQ2;
  const int col = tid - el * NQ2;
  const int qx = col % NQ, qy = col / NQ;
  // the workgroup's cells: e0 .. e0 + m - 1
  uint32_t e0, m;
  if constexpr (ROW) {
    const uint32_t wpr = (rows.n0 + EPB - 1) / EPB;  // workgroups per x-row
    const uint32_t row = blockIdx.x / wpr, xs = (blockIdx.x - row * wpr) * EPB;
    e0 = row * rows.n0 + xs;
    m = min((uint32_t)EPB, rows.n0 - xs);
  } else {
    e0 = blockIdx.x * EPB;
    m = min((uint32_t)EPB, n_cells - e0);
  }
  const uint32_t e = e0 + el;
  const bool active = (uint32_t)el < m;
  const bool node_col = active && qx < NM && qy < NM;

  for (int i = tid; i < NQ * NM; i += Tile<NQ>::THREADS) sB[i] = gB[i];
  for (int i = tid; i < NQ * NQ; i += Tile<NQ>::THREADS) sD[i] = gD[i];
  // wave-uniform entries (the z contractions): through the scalar cache up
  // to nq = 7, from LDS above (their scalar registers would spill)
  auto uB = [&](int i, int j) -> T {
    if constexpr (NQ <= 7) return gB[i * NM + j]; else return sB[i * NM + j];
  };
  auto uD = [&](int i, int j) -> T {
    if constexpr (NQ <= 7) return gD[i * NQ + j]; else return sD[i * NQ + j];
  };

  // nq >= 9 (two or three cells per workgroup): the metric terms are loaded into
  // registers after the x interpolation, so their stream overlaps the y/z
  // interpolation (3-20% faster at p = 7, 8 with q = 9, 10; slower at nq = 7
  // in FP64, no gain below).  Smaller nq loads them in the gradient phase.
  constexpr bool PF = NQ >= 9 && !OTF;
  // LINE: every x and y contraction (interpolation, derivative and their
  // transposes) is taken along whole lines, one line per thread, instead of
  // reading a line per output point, with the metric from the vertices; the
  // line contractions read the even-odd tables of B and D (below) through
  // the scalar cache.  Measured against the per-point form: 25-45% faster in
  // FP32 and 10-40% in FP64 at nq = 5..10 (the gain grows with nq), 1-5% at
  // nq = 3 and in FP32 at nq = 4; FP64 at nq = 4 was 3% slower.  With stored
  // G (memory-bound) level, so not used there.
  constexpr bool LINE =
      OTF && (NQ >= 5 || NQ == 3 || (NQ == 4 && std::is_same<T, float>::value));
  // the line-form contractions apply B, B^T, D, D^T through their even-odd
  // tables (half the multiply-adds; geo holds the four in that order)
  constexpr int EO_BT = eo_table_size(NQ, NM), EO_D = EO_BT + eo_table_size(NM, NQ),
                EO_DT = EO_D + eo_table_size(NQ, NQ);
  const T *Ge = OTF ? nullptr : G + (size_t)(active ? e : 0) * 6 * NQ3 + col;
  T g[PF ? 6 : 1][PF ? NQ : 1];
  if constexpr (OTF) {
    for (int i = tid; i < EPB * 24; i += THREADS) {
      const uint32_t c = (uint32_t)(i / 24);
      sXv[i] = c < m ? (T)cellX[(size_t)(e0 + c) * 24 + i % 24] : T(0);
    }
  }

  // ROW: the segment's first node, the strides of the node grid, and which of its
  // nodes are free: the boundary of the box is constrained
  const uint32_t NX = rows.n0 * (NM - 1) + 1, NXY = NX * (rows.n1 * (NM - 1) + 1);
  uint32_t base = 0, x_first = 0;
  bool y0 = false, y1 = false, z0 = false, z1 = false;
  if constexpr (ROW) {
    const uint32_t row = e0 / rows.n0, ey = row % rows.n1, ez = row / rows.n1;
    x_first = (NM - 1) * (e0 - row * rows.n0);
    base = x_first + (NM - 1) * (ey * NX + ez * NXY);
    y0 = ey == 0;
    y1 = ey + 1 == rows.n1;
    z0 = ez == 0;
    z1 = ez + 1 == rows.n2;
  }
  auto row_free = [&](uint32_t X, int yn, int zn) {  // node X of the segment's row (yn, zn)
    return !(x_first + X == 0 || x_first + X == NX - 1 || (y0 && yn == 0) || (y1 && yn == NM - 1) ||
             (z0 && zn == 0) || (z1 && zn == NM - 1));
  };

  // 1. gather the (x,y) node column
  uint32_t idx[NM];
  T uin[NM];
  if (node_col) {
    const int l0 = qy * NM + qx;
    if constexpr (ROW) {
      const uint32_t X = el * (NM - 1) + qx;
      const T *sc = src + base + X + qy * NX;
#pragma unroll
      for (int z = 0; z < NM; ++z) uin[z] = row_free(X, qy, z) ? sc[z * NXY] : T(0);
    } else if (GATHER) {
      const uint32_t *me = map + (size_t)e * NM3 + l0;
#pragma unroll
      for (int z = 0; z < NM; ++z) idx[z] = me[z * NM2];
#pragma unroll
      for (int z = 0; z < NM; ++z) uin[z] = (idx[z] != kInvalid) ? src[idx[z]] : T(0);
      if constexpr (JOIN) {
#pragma unroll
        for (int z = 0; z < NM; ++z) {
          if (qx == 0) sL[el * NM2 + z * NM + qy] = idx[z];
          if (qx == NM - 1) sR[el * NM2 + z * NM + qy] = idx[z];
        }
      }
    } else {
      const T *se = src + (size_t)e * NM3 + l0;
#pragma unroll
      for (int z = 0; z < NM; ++z) uin[z] = se[z * NM2];
    }
#pragma unroll
    for (int z = 0; z < NM; ++z) s0[el][z * NM2 + l0] = uin[z];
  }
  __syncthreads();

  // per cell the Jacobian coefficient vectors (vertex v = a + 2b + 4c from
  // the bits of (xi, eta, zeta)): A0 = x1-x0, A1 = x3-x2-x1+x0, G0 = x2-x0,
  // K0 = x4-x0, K1 = x5-x1-x4+x0, K2 = x6-x2-x4+x0, K3 = x7-x6-x5+x4-x3+x2+x1-x0
  if constexpr (OTF) {
    for (int j = tid; j < EPB * 3; j += THREADS) {  // j = 3 cell + coordinate
      const T *X = sXv + (j / 3) * 24 + j % 3;
      const T x0 = X[0], x1 = X[3], x2 = X[6], x3 = X[9];
      const T x4 = X[12], x5 = X[15], x6 = X[18], x7 = X[21];
      T *Kd = sKc + (j / 3) * 21 + 7 * (j % 3);
      const T a0 = x1 - x0, a1 = (x3 - x2) - a0, k0 = x4 - x0, k1 = (x5 - x1) - k0;
      Kd[0] = a0;
      Kd[1] = a1;
      Kd[2] = x2 - x0;
      Kd[3] = k0;
      Kd[4] = k1;
      Kd[5] = (x6 - x2) - k0;
      Kd[6] = ((x7 - x6) - (x5 - x4)) - a1;
    }
  }
  // 2. interpolate along x: s1[z][y][qx], z,y < NM (LINE: thread (qx, qy)
  // interpolates the node x-line y = qx, z = qy whole)
  if constexpr (LINE) {
    if (active && qx < NM && qy < NM) {
      T ln[NM];
#pragma unroll
      for (int a = 0; a < NM; ++a) ln[a] = s0[el][qy * NM2 + qx * NM + a];
      T o[NQ];
      eo_tab<NQ, NM, 1>(geo, ln, o);
#pragma unroll
      for (int i = 0; i < NQ; ++i) s1[el][qy * NM * NQ + qx * NQ + i] = o[i];
    }
  } else if (active && qy < NM) {
    T bx[NM];  // this lane's row of B, read from LDS once
#pragma unroll
    for (int a = 0; a < NM; ++a) bx[a] = sB[qx * NM + a];
#pragma unroll
    for (int z = 0; z < NM; ++z) {
      T t = 0;
#pragma unroll
      for (int a = 0; a < NM; ++a) t += bx[a] * s0[el][z * NM2 + qy * NM + a];
      s1[el][z * NM * NQ + qy * NQ + qx] = t;
    }
  }
  __syncthreads();

  // 3./4. interpolate along y (LDS) and z (registers), then 5. gradient
  // OTF: the column's Jacobian columns J0 = a0 + zeta da, J1 = b0 + zeta db,
  // J2 = jz at (xi, eta) = (gxq[qx], gxq[qy])
  T ca0[3], cda[3], cb0[3], cdb[3], cjz[3];
  if (OTF && active) {
    const T xi = gxq[qx], eta = gxq[qy];
    const T *K = sKc + el * 21;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const T A0 = K[7 * d], A1 = K[7 * d + 1], G0 = K[7 * d + 2], K0 = K[7 * d + 3];
      const T K1 = K[7 * d + 4], K2 = K[7 * d + 5], K3 = K[7 * d + 6];
      ca0[d] = A0 + eta * A1;
      cda[d] = K1 + eta * K3;
      cb0[d] = G0 + xi * A1;
      cdb[d] = K2 + xi * K3;
      cjz[d] = (K0 + xi * K1) + eta * cdb[d];
    }
  }
  T uq[NQ];
  if (PF && active) {
#pragma unroll
    for (int z = 0; z < NQ; ++z)
#pragma unroll
      for (int c = 0; c < 6; ++c) g[c][z] = load_geo<T, NQ>(Ge + c * NQ3 + z * NQ2);
  }
  if constexpr (LINE) {
    // thread (qx, qy) interpolates the y-line x = qx, z = qy (< NM) into s0
    if (active && qy < NM) {
      T ln[NM];
#pragma unroll
      for (int c = 0; c < NM; ++c) ln[c] = s1[el][qy * NM * NQ + c * NQ + qx];
      T o[NQ];
      eo_tab<NQ, NM, 1>(geo, ln, o);
#pragma unroll
      for (int yq = 0; yq < NQ; ++yq) s0[el][qy * NQ2 + yq * NQ + qx] = o[yq];
    }
    __syncthreads();
  }
  if (active) {
    T t2[NM], by[LINE ? 1 : NM];
#pragma unroll
    for (int b = 0; b < (LINE ? 0 : NM); ++b) by[b] = sB[qy * NM + b];
#pragma unroll
    for (int z = 0; z < NM; ++z) {
      T t = 0;
      if constexpr (LINE) {
        t = s0[el][z * NQ2 + col];
      } else {
#pragma unroll
        for (int b = 0; b < NM; ++b) t += by[b] * s1[el][z * NM * NQ + b * NQ + qx];
      }
      t2[z] = t;
    }
    if constexpr (LINE) {
      eo_tab<NQ, NM, 1>(geo, t2, uq);
#pragma unroll
      for (int zq = 0; zq < NQ; ++zq) s2[el][zq * NQ2 + col] = uq[zq];
    } else {
#pragma unroll
      for (int zq = 0; zq < NQ; ++zq) {
        T t = 0;
#pragma unroll
        for (int c = 0; c < NM; ++c) t += uB(zq, c) * t2[c];
        uq[zq] = t;
        s2[el][zq * NQ2 + col] = t;
      }
    }
  }
  __syncthreads();

  // p.Ap (DOT): the sum over the cells of u_c^T A_c u_c, formed at the
  // quadrature points as grad u . (G grad u) while both are in registers
  // (constrained entries are gathered as zero, so this is the sum over the
  // free rows of p_i (A p)_i)
  // LINE: the x and y derivatives (and their transposes in 6.) are taken
  // along whole lines first -- thread (l0, l1) = (qx, qy) of a cell
  // differentiates the x-line (y = l0, z = l1) and the y-line (x = l0,
  // z = l1) into s0 / s1, which are free after the interpolation -- so each
  // point's value is read once per line instead of NQ times per point.
  if constexpr (LINE) {
    if (active) {
      T ln[NQ];
#pragma unroll
      for (int a = 0; a < NQ; ++a) ln[a] = s2[el][qy * NQ2 + qx * NQ + a];
      T o[NQ];
      eo_tab<NQ, NQ, -1>(geo + EO_D, ln, o);
#pragma unroll
      for (int i = 0; i < NQ; ++i) s0[el][qy * NQ2 + qx * NQ + i] = o[i];
#pragma unroll
      for (int a = 0; a < NQ; ++a) ln[a] = s2[el][qy * NQ2 + a * NQ + qx];
      eo_tab<NQ, NQ, -1>(geo + EO_D, ln, o);
#pragma unroll
      for (int i = 0; i < NQ; ++i) s1[el][qy * NQ2 + i * NQ + qx] = o[i];
    }
    __syncthreads();
  }
  double dot = 0.0;
  T fz[NQ];
  if (active) {
    T dxr[LINE ? 1 : NQ], dyr[LINE ? 1 : NQ];  // this lane's rows of D
#pragma unroll
    for (int a = 0; a < (LINE ? 0 : NQ); ++a) {
      dxr[a] = sD[qx * NQ + a];
      dyr[a] = sD[qy * NQ + a];
    }
    const T wxy = OTF ? gwq[qx] * gwq[qy] : T(0);
    T dzl[LINE ? NQ : 1];  // LINE: the column's z derivatives
    if constexpr (LINE) eo_tab<NQ, NQ, -1>(geo + EO_D, uq, dzl);
    // the column's points.  AX (cells of an undeformed box, whose Jacobian
    // columns lie along x, y and z): the cofactor columns and det J are the
    // same at every point of the column and diagonal, so they are formed once
    // and the products with their zero entries are left out
    [[maybe_unused]] T H0[3], H1[3], H2[3], hr = T(0);
    if constexpr (OTF && AX) {
      H0[0] = cb0[1] * cjz[2] - cb0[2] * cjz[1];
      H0[1] = cb0[2] * cjz[0] - cb0[0] * cjz[2];
      H0[2] = cb0[0] * cjz[1] - cb0[1] * cjz[0];
      H1[0] = cjz[1] * ca0[2] - cjz[2] * ca0[1];
      H1[1] = cjz[2] * ca0[0] - cjz[0] * ca0[2];
      H1[2] = cjz[0] * ca0[1] - cjz[1] * ca0[0];
      H2[0] = ca0[1] * cb0[2] - ca0[2] * cb0[1];
      H2[1] = ca0[2] * cb0[0] - ca0[0] * cb0[2];
      H2[2] = ca0[0] * cb0[1] - ca0[1] * cb0[0];
      hr = recip(cjz[0] * H2[0] + cjz[1] * H2[1] + cjz[2] * H2[2]);
    }
#pragma unroll
    for (int z = 0; z < NQ; ++z) {
      T dx = 0, dy = 0, dz = 0;
      if constexpr (LINE) {
        dx = s0[el][z * NQ2 + col];
        dy = s1[el][z * NQ2 + col];
        dz = dzl[z];
      } else {
#pragma unroll
        for (int a = 0; a < NQ; ++a) {
          dx += dxr[a] * s2[el][z * NQ2 + qy * NQ + a];
          dy += dyr[a] * s2[el][z * NQ2 + a * NQ + qx];
          dz += uD(z, a) * uq[a];
        }
      }
      if constexpr (OTF) {
        T fx, fy, fzv;
        if constexpr (AX) {
          const T sc = wxy * gwq[z] * hr;
          fx = sc * (H0[0] * (dx * H0[0]));
          fy = sc * (H1[1] * (dy * H1[1]));
          fzv = sc * (H2[2] * (dz * H2[2]));
        } else {
          const T zeta = gxq[z];
          T J0[3], J1[3], C0[3], C1[3], C2[3], W[3];
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            J0[d] = ca0[d] + zeta * cda[d];
            J1[d] = cb0[d] + zeta * cdb[d];
          }
          C0[0] = J1[1] * cjz[2] - J1[2] * cjz[1];
          C0[1] = J1[2] * cjz[0] - J1[0] * cjz[2];
          C0[2] = J1[0] * cjz[1] - J1[1] * cjz[0];
          C1[0] = cjz[1] * J0[2] - cjz[2] * J0[1];
          C1[1] = cjz[2] * J0[0] - cjz[0] * J0[2];
          C1[2] = cjz[0] * J0[1] - cjz[1] * J0[0];
          C2[0] = J0[1] * J1[2] - J0[2] * J1[1];
          C2[1] = J0[2] * J1[0] - J0[0] * J1[2];
          C2[2] = J0[0] * J1[1] - J0[1] * J1[0];
          const T det = cjz[0] * C2[0] + cjz[1] * C2[1] + cjz[2] * C2[2];
          const T sc = wxy * gwq[z] * recip(det);
#pragma unroll
          for (int d = 0; d < 3; ++d) W[d] = dx * C0[d] + dy * C1[d] + dz * C2[d];
          fx = sc * (C0[0] * W[0] + C0[1] * W[1] + C0[2] * W[2]);
          fy = sc * (C1[0] * W[0] + C1[1] * W[1] + C1[2] * W[2]);
          fzv = sc * (C2[0] * W[0] + C2[1] * W[1] + C2[2] * W[2]);
        }
        s0[el][z * NQ2 + col] = fx;
        s1[el][z * NQ2 + col] = fy;
        fz[z] = fzv;
        if (DOT) dot += (double)dx * (double)fx + (double)dy * (double)fy + (double)dz * (double)fz[z];
      } else {
        T gxx, gxy, gxz, gyy, gyz, gzz;
        if constexpr (PF) {
          gxx = g[0][z]; gxy = g[1][z]; gxz = g[2][z];
          gyy = g[3][z]; gyz = g[4][z]; gzz = g[5][z];
        } else {
          gxx = load_geo<T, NQ>(Ge + 0 * NQ3 + z * NQ2);
          gxy = load_geo<T, NQ>(Ge + 1 * NQ3 + z * NQ2);
          gxz = load_geo<T, NQ>(Ge + 2 * NQ3 + z * NQ2);
          gyy = load_geo<T, NQ>(Ge + 3 * NQ3 + z * NQ2);
          gyz = load_geo<T, NQ>(Ge + 4 * NQ3 + z * NQ2);
          gzz = load_geo<T, NQ>(Ge + 5 * NQ3 + z * NQ2);
        }
        const T fx = gxx * dx + gxy * dy + gxz * dz;
        const T fy = gxy * dx + gyy * dy + gyz * dz;
        s0[el][z * NQ2 + col] = fx;
        s1[el][z * NQ2 + col] = fy;
        fz[z] = gxz * dx + gyz * dy + gzz * dz;
        if (DOT) dot += (double)dx * (double)fx + (double)dy * (double)fy + (double)dz * (double)fz[z];
      }
    }
  }
  __syncthreads();

  // 6. transposed gradient, 7. transposed interpolation along z (registers)
  if constexpr (LINE) {
    if (active) {
      T ln[NQ];
#pragma unroll
      for (int i = 0; i < NQ; ++i) ln[i] = s0[el][qy * NQ2 + qx * NQ + i];
      T o[NQ];
      eo_tab<NQ, NQ, -1>(geo + EO_DT, ln, o);
#pragma unroll
      for (int k = 0; k < NQ; ++k) s0[el][qy * NQ2 + qx * NQ + k] = o[k];
#pragma unroll
      for (int i = 0; i < NQ; ++i) ln[i] = s1[el][qy * NQ2 + i * NQ + qx];
      eo_tab<NQ, NQ, -1>(geo + EO_DT, ln, o);
#pragma unroll
      for (int k = 0; k < NQ; ++k) s1[el][qy * NQ2 + k * NQ + qx] = o[k];
    }
    __syncthreads();
  }
  if (active) {
    T w[NQ], dxt[LINE ? 1 : NQ], dyt[LINE ? 1 : NQ];  // this lane's columns of D
#pragma unroll
    for (int a = 0; a < (LINE ? 0 : NQ); ++a) {
      dxt[a] = sD[a * NQ + qx];
      dyt[a] = sD[a * NQ + qy];
    }
    T dzt[LINE ? NQ : 1];  // LINE: D^T of the column's z fluxes
    if constexpr (LINE) eo_tab<NQ, NQ, -1>(geo + EO_DT, fz, dzt);
#pragma unroll
    for (int z = 0; z < NQ; ++z) {
      T v = 0;
      if constexpr (LINE) {
        v = s0[el][z * NQ2 + col] + s1[el][z * NQ2 + col] + dzt[z];
      } else {
#pragma unroll
        for (int a = 0; a < NQ; ++a) {
          v += dxt[a] * s0[el][z * NQ2 + qy * NQ + a];
          v += dyt[a] * s1[el][z * NQ2 + a * NQ + qx];
          v += uD(a, z) * fz[a];
        }
      }
      w[z] = v;
    }
    if constexpr (LINE) {
      T o[NM];
      eo_tab<NM, NQ, 1>(geo + EO_BT, w, o);
#pragma unroll
      for (int zn = 0; zn < NM; ++zn) s2[el][zn * NQ2 + col] = o[zn];
    } else {
#pragma unroll
      for (int zn = 0; zn < NM; ++zn) {
        T t = 0;
#pragma unroll
        for (int c = 0; c < NQ; ++c) t += uB(c, zn) * w[c];
        s2[el][zn * NQ2 + col] = t;
      }
    }
  }
  __syncthreads();

  // 8. transposed interpolation along y: s0[zn][yn][qx] (LINE: thread
  // (qx, qy) takes the y-line x = qx, zn = qy whole)
  if constexpr (LINE) {
    if (active && qy < NM) {
      T ln[NQ];
#pragma unroll
      for (int b = 0; b < NQ; ++b) ln[b] = s2[el][qy * NQ2 + b * NQ + qx];
      T o[NM];
      eo_tab<NM, NQ, 1>(geo + EO_BT, ln, o);
#pragma unroll
      for (int yn = 0; yn < NM; ++yn) s0[el][qy * NM * NQ + yn * NQ + qx] = o[yn];
    }
  } else if (active && qy < NM) {
    T byt[NQ];
#pragma unroll
    for (int b = 0; b < NQ; ++b) byt[b] = sB[b * NM + qy];
#pragma unroll
    for (int zn = 0; zn < NM; ++zn) {
      T t = 0;
#pragma unroll
      for (int b = 0; b < NQ; ++b) t += byt[b] * s2[el][zn * NQ2 + b * NQ + qx];
      s0[el][zn * NM * NQ + qy * NQ + qx] = t;
    }
  }
  __syncthreads();

  // 9. transposed interpolation along x and scatter
  constexpr int P = NM - 1, XW = EPB * P + 1;  // ROW: nodes of a full segment row
  T *acc = &s1[0][0];  // ROW: [zn][yn][X], X = c P + xn, the left faces
  T *rgt = &s2[0][0];  // ROW: [zn][yn][c], right faces of all but the last cell
  T *lft = &s2[0][0];  // JOIN: [c][zn][yn], left faces that the cell before adds
  static_assert(!JOIN || NM * NM <= NQ3, "left faces do not fit s2");
  T vj[JOIN ? NM : 1];  // JOIN: the column's sums
  // JOIN: node zn of this column is the right face node of the cell before
  auto joined = [&](int zn) {
    return qx == 0 && el > 0 && sR[(el - 1) * NM2 + zn * NM + qy] == idx[zn];
  };
  static_assert(!ROW || NM * NM * XW <= EPB * NQ3, "row segment does not fit s1");
  static_assert(!ROW || NM * NM * EPB <= EPB * NQ3, "right faces do not fit s2");
  if constexpr (LINE && ROW) {
    // thread (qx, qy) takes the x-line yn = qx, zn = qy whole
    if (node_col) {
      T ln[NQ];
#pragma unroll
      for (int a = 0; a < NQ; ++a) ln[a] = s0[el][qy * NM * NQ + qx * NQ + a];
      T o[NM];
      eo_tab<NM, NQ, 1>(geo + EO_BT, ln, o);
#pragma unroll
      for (int xn = 0; xn < NM; ++xn) {
        const T v = o[xn];
        if (xn < P || (uint32_t)el + 1 == m)
          acc[(qy * NM + qx) * XW + el * P + xn] = v;
        else
          rgt[(qy * NM + qx) * EPB + el] = v;
      }
    }
  } else if (node_col) {
    T bxt[NQ];
#pragma unroll
    for (int a = 0; a < NQ; ++a) bxt[a] = sB[a * NM + qx];
#pragma unroll
    for (int zn = 0; zn < NM; ++zn) {
      T v = 0;
#pragma unroll
      for (int a = 0; a < NQ; ++a) v += bxt[a] * s0[el][zn * NM * NQ + qy * NQ + a];
      if constexpr (ROW) {
        if (qx < P || (uint32_t)el + 1 == m)
          acc[(zn * NM + qy) * XW + el * P + qx] = v;
        else
          rgt[(zn * NM + qy) * EPB + el] = v;
      } else if constexpr (JOIN) {
        vj[zn] = v;
        if (joined(zn)) lft[el * NM2 + zn * NM + qy] = v;
      } else if (GATHER) {
        if (idx[zn] != kInvalid) atomic_add(dst + idx[zn], v);
      } else {
        dst[(size_t)e * NM3 + zn * NM2 + qy * NM + qx] = v;
      }
    }
  }
  if constexpr (JOIN) {
    // a face node that the map gives to two consecutive cells goes out with the
    // first one's column
    __syncthreads();
    if (node_col) {
#pragma unroll
      for (int zn = 0; zn < NM; ++zn) {
        if (idx[zn] == kInvalid || joined(zn)) continue;
        T v = vj[zn];
        if (qx == NM - 1 && (uint32_t)el + 1 < m && sL[(el + 1) * NM2 + zn * NM + qy] == idx[zn])
          v += lft[(el + 1) * NM2 + zn * NM + qy];
        atomic_add(dst + idx[zn], v);
      }
    }
  }
  if constexpr (ROW) {
    __syncthreads();
    // node X of row r = zn NM + yn of the segment: its left-face value plus,
    // on an inner face, the right face of the cell before it
    const int nx = (int)m * P + 1;
    for (int i = tid; i < NM * NM * nx; i += THREADS) {
      const int r = i / nx, X = i - r * nx;
      const int c = X / P;
      T v = acc[r * XW + X];
      if (X == c * P && c >= 1 && c < (int)m) v += rgt[r * EPB + c - 1];
      const int zn = r / NM, yn = r - zn * NM;
      if (row_free(X, yn, zn)) atomic_add(dst + base + X + yn * NX + zn * NXY, v);
    }
  }
  if (DOT) {
    const double s = block_sum<Tile<NQ>::THREADS>(dot, red);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
  }
}

// Workgroups of an apply: cells in batches of EPB, or (Gauss kernel on a box
// mesh) EPB-cell segments of each x-row.
template <int NQ, bool COLLOC, bool GATHER = true>
uint32_t n_blocks_for(uint32_t n_cells, RowMesh rows = {}) {
  constexpr int EPB = COLLOC ? CollocTile<double, NQ, GATHER>::EPB : Tile<NQ>::EPB;
  if (!COLLOC && rows.n0) return (n_cells / rows.n0) * ((rows.n0 + EPB - 1) / EPB);
  return (n_cells + EPB - 1) / EPB;
}

// Whether the Gauss kernel joins faces, where it can, at nq >= 6.  Without / with it:
// - with at most a workgroup per CU its latency counts: raw applies of 60k DoFs, FP64, p = 4,
//   q = 6 9.8 / 10.5 us, p = 7, q = 8 9.8 / 11.4;
// - at q = 8 (few cells in a workgroup) it pays only where the adds it saves are a request
//   each, not where a cell's x-lines are consecutive DoFs (scattered = false).  In the
//   mesh's order, 6M DoFs: p = 6 FP64 211 / 228 us, FP32 130 / 136, p = 7 166 / 175; in an
//   adapter's order, 1.5M: 75 / 73, 41 / 37, 50 / 47;
// - with stored FP64 terms and q = p + 2 (lanes without a node) not once G's stream bounds
//   the kernel: p = 5, q = 7 in the mesh's order 400k DoFs 20.3 / 18.6, 1.5M 63 / 65, in
//   an adapter's 1.5M 69 / 67, 2.5M 100 / 102, 20M 723 / 747; p = 6, q = 8 4M 160 / 155, 6M
//   228 / 227, 9M 347 / 353, 20M 716 / 743.
// Everywhere else it gains in either order (p = 6, q = 7 170 / 152, p = 5, q = 7 with the
// metric from the vertices 179 / 164, FP32 6M DoFs 142 / 121).
template <typename T, int NM, int NQ, bool OTF>
bool join_faces(uint32_t blocks, bool scattered) {
  if (blocks <= 256 || (NQ == 8 && !scattered)) return false;
  if (OTF || sizeof(T) == 4 || NM == NQ || NQ == 6) return true;
  if (NQ == 7) return blocks <= (scattered ? 2816 : 1024);
  return blocks <= 8192;
}

// The same for the collocation kernel at nq = 9.  FP64: not on a few CUs (27 cells 10.6 ->
// 11.2 us, 125 cells 12.5 -> 11.6).  FP32: on many workgroups in an adapter's order while
// G fits the memory-side cache (1.5M DoFs 30.8 -> 29.4 us; 400k 12.4 -> 14.2, 12M 197 -> 205;
// in the mesh's order 27.9 -> 30.4).
template <typename T, int NQ>
bool join_colloc(uint32_t n_cells, bool scattered) {
  const uint32_t blocks = n_blocks_for<NQ, true>(n_cells);
  if (sizeof(T) == 8) return blocks > 16;
  return scattered && blocks > 512 && (uint64_t)n_cells * 24 * NQ * NQ * NQ <= kMemorySideCache;
}

// Whether the collocation kernel streams G at nq = 5 in FP64: where G exceeds the
// memory-side cache and the vectors do not, which then stay in it.  Kept / streamed: 3M
// DoFs 107.6 / 104.9 us, 6M 197 / 190 (E-vectors 133 / 129); below 1.5M 50 / 52, above
// 18M 488 / 490 (E-vectors of 10M 229 / 258).
template <int NQ, bool GATHER>
bool stream_colloc(uint32_t n_cells) {
  constexpr int NV = GATHER ? NQ - 1 : NQ;  // DoFs of a cell per direction
  return (uint64_t)n_cells * 48 * NQ * NQ * NQ > kMemorySideCache &&
         (uint64_t)n_cells * 16 * NV * NV * NV <= kMemorySideCache;
}

template <typename T, int NQ, bool GATHER, bool DOT, bool JOIN, bool STREAM>
void launch_colloc(const T *D, const T *G, const T *src, T *dst, const uint32_t *map,
                   uint32_t n_cells, hipStream_t s, double *partials, const int *skip) {
  using C = CollocTile<T, NQ, GATHER>;
  const dim3 grid(n_blocks_for<NQ, true, GATHER>(n_cells)), block(C::THREADS);
  hipLaunchKernelGGL((k_apply_colloc<T, NQ, C::EPB, C::PREFETCH, GATHER, DOT, JOIN, STREAM>), grid,
                     block, 0, s, D, G, src, dst, map, n_cells, partials, skip, nullptr, nullptr);
}

template <typename T, int NM, int NQ, bool GATHER, bool DOT, bool OTF>
void launch_mapped(const dim3 grid, const T *B, const T *D, const T *G, const T *src, T *dst,
                   const uint32_t *map, uint32_t n_cells, hipStream_t s, double *partials,
                   const int *skip, const double *cellX, const T *xq, const T *wq, const T *eo,
                   bool scattered) {
  constexpr bool CAN = GATHER && kJoin<NM, NQ>, ALWAYS = CAN && NQ <= 5;
  const dim3 block(Tile<NQ>::THREADS);
  if constexpr (CAN) {
    if (ALWAYS || join_faces<T, NM, NQ, OTF>(grid.x, scattered)) {
      hipLaunchKernelGGL((k_apply_interp<T, NM, NQ, true, DOT, OTF, false, false, true>), grid,
                         block, 0, s, B, D, G, src, dst, map, n_cells, partials, skip, cellX, xq,
                         wq, RowMesh{}, eo);
      return;
    }
  }
  if constexpr (!ALWAYS)
    hipLaunchKernelGGL((k_apply_interp<T, NM, NQ, GATHER, DOT, OTF, false, false, false>), grid,
                       block, 0, s, B, D, G, src, dst, map, n_cells, partials, skip, cellX, xq, wq,
                       RowMesh{}, eo);
}

template <typename T, int NM, int NQ, bool COLLOC, bool GATHER>
void launch_t(const T *B, const T *D, const T *G, const T *src, T *dst,
              const uint32_t *map, uint32_t n_cells, hipStream_t s,
              double *partials, const int *skip, RowMesh rows, bool scattered) {
  if (n_cells == 0) return;
  const bool row = !COLLOC && GATHER && rows.n0 > 0;
  MFX_REQUIRE(!row || (uint64_t)rows.n0 * rows.n1 * rows.n2 == n_cells, "row segments: cells of another mesh");
  if constexpr (COLLOC) {
    static_assert(NM == NQ, "collocation needs nm == nq");
    using C = CollocTile<T, NQ, GATHER>;
    constexpr bool JOIN = GATHER && kCollocJoin<NQ, C::EPB, C::PREFETCH>;
    auto with = [&](auto dot) {
      constexpr bool DOT = decltype(dot)::value;
      if constexpr (JOIN && NQ == 9)
        if (!join_colloc<T, NQ>(n_cells, scattered))
          return launch_colloc<T, NQ, GATHER, DOT, false, false>(D, G, src, dst, map, n_cells, s,
                                                                 partials, skip);
      if constexpr (NQ == 5 && sizeof(T) == 8)
        if (stream_colloc<NQ, GATHER>(n_cells))
          return launch_colloc<T, NQ, GATHER, DOT, JOIN, true>(D, G, src, dst, map, n_cells, s,
                                                               partials, skip);
      launch_colloc<T, NQ, GATHER, DOT, JOIN, kCollocStream<T, NQ>>(D, G, src, dst, map, n_cells,
                                                                    s, partials, skip);
    };
    if (!partials)
      with(std::false_type{});
    else if constexpr (std::is_same<T, double>::value && GATHER)
      with(std::true_type{});
  } else {
    const dim3 grid(n_blocks_for<NQ, false>(n_cells, row ? rows : RowMesh{})),
        block(Tile<NQ>::THREADS);
    auto with = [&](auto dot) {
      constexpr bool DOT = decltype(dot)::value;
      if constexpr (GATHER)
        if (row) {
          hipLaunchKernelGGL((k_apply_interp<T, NM, NQ, GATHER, DOT, false, true>), grid, block, 0,
                             s, B, D, G, src, dst, map, n_cells, partials, skip, nullptr, nullptr,
                             nullptr, rows, (const T *)nullptr);
          return;
        }
      launch_mapped<T, NM, NQ, GATHER, DOT, false>(grid, B, D, G, src, dst, map, n_cells, s,
                                                   partials, skip, nullptr, nullptr, nullptr,
                                                   nullptr, scattered);
    };
    if (!partials)
      with(std::false_type{});
    else if constexpr (std::is_same<T, double>::value && GATHER)
      with(std::true_type{});
  }
  MFX_HIP(hipGetLastError());
}

// Runtime (p, nq, collocation) -> template instance.  Supported: p = 1..8;
// collocation nq = p+1; interpolation nq = p+1 or p+2.
template <typename T, bool GATHER>
void dispatch(int p, int nq, bool colloc, const T *B, const T *D, const T *G,
              const T *src, T *dst, const uint32_t *map, uint32_t n,
              hipStream_t s, double *partials, const int *skip, RowMesh rc, bool scattered) {
#define MFX_CASE_C(P)                                                         \
  case P:                                                                     \
    return launch_t<T, P + 1, P + 1, true, GATHER>(B, D, G, src, dst, map, n, s, partials, skip, rc, scattered);
#define MFX_CASE_I(P)                                                         \
  case P:                                                                     \
    if (nq == P + 1)                                                          \
      return launch_t<T, P + 1, P + 1, false, GATHER>(B, D, G, src, dst, map, n, s, partials, skip, rc, scattered); \
    if (nq == P + 2)                                                          \
      return launch_t<T, P + 1, P + 2, false, GATHER>(B, D, G, src, dst, map, n, s, partials, skip, rc, scattered); \
    break;
  if (colloc) {
    MFX_REQUIRE(nq == p + 1, "collocation requires nq == p+1");
    switch (p) { MFX_CASE_C(1) MFX_CASE_C(2) MFX_CASE_C(3) MFX_CASE_C(4)
                 MFX_CASE_C(5) MFX_CASE_C(6) MFX_CASE_C(7) MFX_CASE_C(8) default: break; }
  } else {
    switch (p) { MFX_CASE_I(1) MFX_CASE_I(2) MFX_CASE_I(3) MFX_CASE_I(4)
                 MFX_CASE_I(5) MFX_CASE_I(6) MFX_CASE_I(7) MFX_CASE_I(8) default: break; }
  }
#undef MFX_CASE_C
#undef MFX_CASE_I
  throw Error{MFX_ERR_UNSUPPORTED,
              "unsupported (degree, n_q_points_1d) = (" + std::to_string(p) + ", " +
                  std::to_string(nq) + ")"};
}

// Tile variants of the collocation kernel the autotuner chooses from: three
// cell counts per workgroup, each with and without the G prefetch.
template <int NQ, int EPB, bool PREF>
void launch_cv(const double *D, const double *G, const double *src, double *dst,
               const uint32_t *map, uint32_t n_cells, const uint16_t *cell_inst,
               const int *inst_done, hipStream_t s) {
  const dim3 grid((n_cells + EPB - 1) / EPB), block(EPB * NQ * NQ);
  hipLaunchKernelGGL((k_apply_colloc<double, NQ, EPB, PREF, true, false>), grid, block, 0, s, D, G,
                     src, dst, map, n_cells, nullptr, nullptr, cell_inst, inst_done);
  MFX_HIP(hipGetLastError());
}
template <int NQ>
constexpr int kVariantCells[3] = {0, 0, 0};
template <>
constexpr int kVariantCells<3>[3] = {7, 14, 28};
template <>
constexpr int kVariantCells<4>[3] = {4, 8, 16};
template <>
constexpr int kVariantCells<5>[3] = {2, 5, 10};
template <>
constexpr int kVariantCells<6>[3] = {1, 3, 7};
template <>
constexpr int kVariantCells<7>[3] = {1, 2, 5};
// variant v: cells [v / 2], with the prefetch for even v
constexpr bool variant_prefetch(int v) { return v % 2 == 0; }

// the variant that is the default tile of launch_apply
template <int NQ>
constexpr int default_variant() {
  for (int v = 0; v < 6; ++v)
    if (kVariantCells<NQ>[v / 2] == CollocTile<double, NQ>::EPB &&
        variant_prefetch(v) == CollocTile<double, NQ>::PREFETCH)
      return v;
  return -1;
}
static_assert(default_variant<3>() >= 0 && default_variant<4>() >= 0 && default_variant<5>() >= 0 &&
                  default_variant<6>() >= 0 && default_variant<7>() >= 0,
              "the default tile is among the variants");

template <int NQ>
void launch_cv_sel(int v, int *epb, int *pref, const double *D, const double *G, const double *src,
                   double *dst, const uint32_t *map, uint32_t n, const uint16_t *ci,
                   const int *done, hipStream_t s) {
  constexpr int E0 = kVariantCells<NQ>[0], E1 = kVariantCells<NQ>[1], E2 = kVariantCells<NQ>[2];
  MFX_REQUIRE(v >= 0 && v < 6, "tile variant out of range");
  *epb = kVariantCells<NQ>[v / 2];
  *pref = variant_prefetch(v);
  if (!src) return;  // description only
  if (n == 0) return;
  switch (v) {
    case 0: return launch_cv<NQ, E0, true>(D, G, src, dst, map, n, ci, done, s);
    case 1: return launch_cv<NQ, E0, false>(D, G, src, dst, map, n, ci, done, s);
    case 2: return launch_cv<NQ, E1, true>(D, G, src, dst, map, n, ci, done, s);
    case 3: return launch_cv<NQ, E1, false>(D, G, src, dst, map, n, ci, done, s);
    case 4: return launch_cv<NQ, E2, true>(D, G, src, dst, map, n, ci, done, s);
    default: return launch_cv<NQ, E2, false>(D, G, src, dst, map, n, ci, done, s);
  }
}

}  // namespace

int colloc_variant_count(int p) { return (p >= 2 && p <= 6) ? 6 : 0; }

int colloc_default_variant(int p) {
  switch (p) {
    case 2: return default_variant<3>();
    case 3: return default_variant<4>();
    case 4: return default_variant<5>();
    case 5: return default_variant<6>();
    case 6: return default_variant<7>();
    default: return 0;
  }
}

void launch_colloc_variant(int p, int v, const double *D, const double *G, const double *src,
                           double *dst, const uint32_t *map, uint32_t n_cells,
                           const uint16_t *cell_inst, const int *inst_done, hipStream_t s,
                           int *epb, int *prefetch) {
  int e = 0, pf = 0;
  switch (p) {
    case 2: launch_cv_sel<3>(v, &e, &pf, D, G, src, dst, map, n_cells, cell_inst, inst_done, s); break;
    case 3: launch_cv_sel<4>(v, &e, &pf, D, G, src, dst, map, n_cells, cell_inst, inst_done, s); break;
    case 4: launch_cv_sel<5>(v, &e, &pf, D, G, src, dst, map, n_cells, cell_inst, inst_done, s); break;
    case 5: launch_cv_sel<6>(v, &e, &pf, D, G, src, dst, map, n_cells, cell_inst, inst_done, s); break;
    case 6: launch_cv_sel<7>(v, &e, &pf, D, G, src, dst, map, n_cells, cell_inst, inst_done, s); break;
    default: throw Error{MFX_ERR_UNSUPPORTED, "tile variants exist for degrees 2..6"};
  }
  if (epb) *epb = e;
  if (prefetch) *prefetch = pf;
}

template <typename T>
void launch_apply(int p, int nq, bool colloc, const T *B, const T *D, const T *G,
                  const T *src, T *dst, const uint32_t *map, uint32_t n_cells,
                  hipStream_t s, double *dot_partials, const int *skip, RowMesh rows,
                  bool scattered) {
  dispatch<T, true>(p, nq, colloc, B, D, G, src, dst, map, n_cells, s, dot_partials, skip,
                    rows, scattered);
}
template <typename T>
void launch_evec(int p, int nq, bool colloc, const T *B, const T *D, const T *G,
                 const T *in, T *out, uint32_t n_cells, hipStream_t s) {
  dispatch<T, false>(p, nq, colloc, B, D, G, in, out, nullptr, n_cells, s, nullptr, nullptr, RowMesh{},
                     false);
}

// Gauss (non-collocated) apply with the metric terms computed from the cell
// vertices (k_apply_interp<..., OTF>).
template <typename T, int NM, int NQ>
void launch_interp_otf(const T *B, const T *D, const T *eo, const T *xq, const T *wq,
                       const double *cellX, const T *src, T *dst, const uint32_t *map,
                       uint32_t n_cells, hipStream_t s, double *partials, const int *skip,
                       RowMesh rows, bool axes, bool scattered) {
  MFX_REQUIRE(!axes || rows.n0, "axis-aligned cells are a box-mesh form");
  if (n_cells == 0) return;
  MFX_REQUIRE(!rows.n0 || (uint64_t)rows.n0 * rows.n1 * rows.n2 == n_cells,
              "row segments: cells of another mesh");
  const dim3 grid(n_blocks_for<NQ, false>(n_cells, rows)), block(Tile<NQ>::THREADS);
  auto with = [&](auto dot) {
    constexpr bool DOT = decltype(dot)::value;
    if (axes)
      hipLaunchKernelGGL((k_apply_interp<T, NM, NQ, true, DOT, true, true, true>), grid, block, 0,
                         s, B, D, nullptr, src, dst, map, n_cells, partials, skip, cellX, xq, wq,
                         rows, eo);
    else if (rows.n0)
      hipLaunchKernelGGL((k_apply_interp<T, NM, NQ, true, DOT, true, true>), grid, block, 0, s, B,
                         D, nullptr, src, dst, map, n_cells, partials, skip, cellX, xq, wq, rows,
                         eo);
    else
      launch_mapped<T, NM, NQ, true, DOT, true>(grid, B, D, nullptr, src, dst, map, n_cells, s,
                                                partials, skip, cellX, xq, wq, eo, scattered);
  };
  if (!partials)
    with(std::false_type{});
  else if constexpr (std::is_same<T, double>::value)
    with(std::true_type{});
  else
    throw Error{MFX_ERR_UNSUPPORTED, "p.Ap partials are computed in FP64 only"};
  MFX_HIP(hipGetLastError());
}

template <typename T>
void launch_apply_otf(int p, int nq, const T *B, const T *D, const T *eo, const T *xq,
                      const T *wq, const double *cellX, const T *src, T *dst,
                      const uint32_t *map, uint32_t n_cells, hipStream_t s, double *partials,
                      const int *skip, RowMesh rows, bool axes, bool scattered) {
  MFX_REQUIRE(B && D && eo && xq && wq && cellX, "on-the-fly apply: missing tables or vertices");
#define MFX_CASE_O(P)                                                                         \
  case P:                                                                                    \
    if (nq == P + 1)                                                                         \
      return launch_interp_otf<T, P + 1, P + 1>(B, D, eo, xq, wq, cellX, src, dst, map,      \
                                                n_cells, s, partials, skip, rows, axes,  \
                                                scattered);                              \
    if (nq == P + 2)                                                                         \
      return launch_interp_otf<T, P + 1, P + 2>(B, D, eo, xq, wq, cellX, src, dst, map,      \
                                                n_cells, s, partials, skip, rows, axes,  \
                                                scattered);                              \
    break;
  switch (p) {
    MFX_CASE_O(1) MFX_CASE_O(2) MFX_CASE_O(3) MFX_CASE_O(4)
    MFX_CASE_O(5) MFX_CASE_O(6) MFX_CASE_O(7) MFX_CASE_O(8) default: break;
  }
#undef MFX_CASE_O
  throw Error{MFX_ERR_UNSUPPORTED,
              "unsupported (degree, n_q_points_1d) = (" + std::to_string(p) + ", " +
                  std::to_string(nq) + ")"};
}

template void launch_apply_otf<double>(int, int, const double *, const double *, const double *,
                                       const double *, const double *, const double *,
                                       const double *, double *, const uint32_t *, uint32_t,
                                       hipStream_t, double *, const int *, RowMesh, bool, bool);
template void launch_apply_otf<float>(int, int, const float *, const float *, const float *,
                                      const float *, const float *, const double *, const float *,
                                      float *, const uint32_t *, uint32_t, hipStream_t, double *,
                                      const int *, RowMesh, bool, bool);

template void launch_apply<double>(int, int, bool, const double *, const double *,
                                   const double *, const double *, double *,
                                   const uint32_t *, uint32_t, hipStream_t, double *,
                                   const int *, RowMesh, bool);
template void launch_apply<float>(int, int, bool, const float *, const float *,
                                  const float *, const float *, float *,
                                  const uint32_t *, uint32_t, hipStream_t, double *,
                                  const int *, RowMesh, bool);
template void launch_evec<double>(int, int, bool, const double *, const double *,
                                  const double *, const double *, double *, uint32_t,
                                  hipStream_t);

uint32_t apply_n_blocks(int p, int nq, bool colloc, uint32_t n_cells, RowMesh rows) {
  (void)p;
#define MFX_NB(Q)                                                                    \
  case Q:                                                                           \
    return colloc ? n_blocks_for<Q, true>(n_cells) : n_blocks_for<Q, false>(n_cells, rows);
  switch (nq) {
    MFX_NB(2) MFX_NB(3) MFX_NB(4) MFX_NB(5) MFX_NB(6) MFX_NB(7) MFX_NB(8) MFX_NB(9) MFX_NB(10)
    default: return 0;
  }
#undef MFX_NB
}

}  // namespace mfx
