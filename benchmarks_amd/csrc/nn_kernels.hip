// nn_kernels.hip -- kernels of the learned preconditioner's 3D U-Net: the
// convolutions of the forward pass on BF16 MFMA with FP32 accumulation, the
// backward pass (data and weight gradients) in FP32, the loss and Adam.
//
// Tensors are channels-last [z][y][x][c] over a level's nodal grid.  A
// convolution is a correlation with zero padding 1 over the 27 taps
// t = tx + 3 ty + 9 tz (offset (tx-1, ty-1, tz-1)):
//   out[p][o] = sum_{t,c} W[o][t][c] in[s p + off_t][c]      (stride s = 1, 2)
// and, with up-sampling, in = up(v), up(v)[i] = v[i >> 1] per direction.
//
// Forward (implicit GEMM on v_mfma_f32_16x16x32_bf16): a wavefront owns 16
// consecutive output nodes and NT tiles of 16 output channels; the K dimension
// (t, c) runs in chunks of 32: lane l gathers 8 consecutive channels of one
// tap of node l % 16 (one 16-byte load, channels-last) as the A operand and
// 8 consecutive k of output channel l % 16 as the B operand, whose weights are
// stored in lane order.  D register r of lane l is node 4 (l / 16) + r,
// channel l % 16.
#include <algorithm>

#include "mfx_internal.hpp"
#include "nn.hpp"

namespace mfx {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

constexpr int kBlock = 256;

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
// round to nearest even
__device__ __forceinline__ uint16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

struct Dims {
  uint32_t x, y, z;
};

// coordinates of node i (node counts stay below 2^32: a grid of that many
// nodes exceeds the device's memory)
__device__ __forceinline__ void decode(uint32_t i, const Dims &d, int &x, int &y, int &z) {
  const uint32_t q = i / d.x;
  x = (int)(i - q * d.x);
  const uint32_t r = q / d.y;
  y = (int)(q - r * d.y);
  z = (int)r;
}

__device__ __forceinline__ bool inside(int x, int y, int z, const Dims &d) {
  return x >= 0 && y >= 0 && z >= 0 && x < (int)d.x && y < (int)d.y && z < (int)d.z;
}

__device__ __forceinline__ uint64_t lin(int x, int y, int z, const Dims &d) {
  return (uint64_t)x + (uint64_t)d.x * ((uint64_t)y + (uint64_t)d.y * (uint64_t)z);
}

// Index of the input node of output node (x,y,z) at tap t, or -1 outside.
// od: output grid, id: input tensor grid (the coarse grid when UP).
template <int STRIDE, bool UP>
__device__ __forceinline__ int64_t tap_source(int x, int y, int z, int t, const Dims &od,
                                              const Dims &id) {
  const int ox = t % 3 - 1, oy = (t / 3) % 3 - 1, oz = t / 9 - 1;
  int qx = STRIDE * x + ox, qy = STRIDE * y + oy, qz = STRIDE * z + oz;
  if (UP) {
    if (!inside(qx, qy, qz, od)) return -1;
    return (int64_t)lin(qx >> 1, qy >> 1, qz >> 1, id);
  }
  if (!inside(qx, qy, qz, id)) return -1;
  return (int64_t)lin(qx, qy, qz, id);
}

// The chunks' operands are loaded in groups of GC, one group ahead of the
// products (the sums keep one accumulator per output and the order of k).  On
// the grids the preconditioner uses a layer has few waves, each a chain of
// 27 CIN / 32 products: what bounds it is the latency of the gathered loads,
// so NT = 1 spreads the channels over waves and the groups keep 2 GC loads
// in flight.  33^3 grid: the six layers take 4.2, 6.3, 10.9, 7.7, 8.3 and 9.9
// us, against 9, 15, 31, 33, 22 and 15 us with all channel tiles in one wave
// and one chunk's loads at a time.
template <int CIN, int COUT, int STRIDE, bool UP, int NT>
__global__ void __launch_bounds__(kBlock)
k_conv_mfma(const uint16_t *__restrict__ in, const uint16_t *__restrict__ W,
            const uint16_t *__restrict__ skip, uint16_t *__restrict__ out, Dims od, Dims id) {
  static_assert(CIN % 16 == 0 && CIN <= 64 && COUT % (16 * NT) == 0, "channel tiles");
  constexpr int NC = (27 * CIN + 31) / 32;           // chunks of 32 k
  constexpr int GC = CIN == 16 ? (NT == 1 ? 7 : 2) : (NT == 1 ? 9 : 3), WPN = COUT / 16 / NT;
  static_assert(NC % GC == 0, "chunk groups");
  const int lane = threadIdx.x & 63, g = lane >> 4, li = lane & 15;
  const uint32_t w = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  const uint32_t P = od.x * od.y * od.z, tile = w / WPN;
  const int nt0 = (int)(w % WPN) * NT;
  if (tile >= (P + 15) / 16) return;
  const uint32_t node = tile * 16 + li;
  // the lane's input rows: element offsets of the three taps per axis and the
  // mask of the taps inside the grid
  const Dims bd = UP ? od : id;
  int xo[3];
  int64_t yo[3], zo[3];
  uint32_t mask = 0;
  {
    int x, y, z;
    decode(node < P ? node : 0, od, x, y, z);
    bool vx[3], vy[3], vz[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int qx = STRIDE * x + k - 1, qy = STRIDE * y + k - 1, qz = STRIDE * z + k - 1;
      vx[k] = qx >= 0 && qx < (int)bd.x;
      vy[k] = qy >= 0 && qy < (int)bd.y;
      vz[k] = qz >= 0 && qz < (int)bd.z;
      xo[k] = (vx[k] ? UP ? qx >> 1 : qx : 0) * CIN;
      yo[k] = (int64_t)(vy[k] ? UP ? qy >> 1 : qy : 0) * id.x * CIN;
      zo[k] = (int64_t)(vz[k] ? UP ? qz >> 1 : qz : 0) * id.x * id.y * CIN;
    }
#pragma unroll
    for (int t = 0; t < 27; ++t)
      mask |= (uint32_t)(vx[t % 3] && vy[t / 3 % 3] && vz[t / 9]) << t;
    if (node >= P) mask = 0;
  }
  auto off = [&](int t) { return xo[t % 3] + yo[t / 3 % 3] + zo[t / 9]; };
  // chunk i of the lane: tap and channels (CIN = 16: two taps per chunk, the
  // upper half of the wave on the second one)
  auto load_a = [&](int i, bool &on) -> uint4 {
    int64_t o;
    if constexpr (CIN == 16) {
      const int t0 = 2 * i, t1 = 2 * i + 1;
      const bool hi = g >> 1;
      const int64_t o0 = off(t0), d = t1 < 27 ? off(t1 < 27 ? t1 : 26) - o0 : 0;
      o = o0 + (hi ? d : 0) + 8 * (g & 1);
      on = hi ? (t1 < 27 && (mask >> t1 & 1)) : (mask >> t0 & 1);
    } else {
      const int t = i * 32 / CIN;
      o = off(t) + i * 32 % CIN + 8 * g;
      on = mask >> t & 1;
    }
    return *reinterpret_cast<const uint4 *>(in + o);
  };
  // weights of chunk i, channel tile n: [chunk][tile][lane][8]
  auto load_b = [&](int i, int n) {
    return *reinterpret_cast<const uint4 *>(
        W + ((size_t)(i * (COUT / 16) + nt0 + n) * 64 + lane) * 8);
  };
  v4f acc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[n] = v4f{0.f, 0.f, 0.f, 0.f};
  uint16_t sk[NT][4];
  if (UP) {
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint32_t o = min(tile * 16 + 4 * g + r, P - 1);
        sk[n][r] = skip[(uint64_t)o * COUT + (nt0 + n) * 16 + li];
      }
  }
  uint4 a[2][GC], b[2][GC][NT];
  bool on[2][GC];
  auto load = [&](int i0, int buf) {
#pragma unroll
    for (int k = 0; k < GC; ++k) {
      a[buf][k] = load_a(i0 + k, on[buf][k]);
#pragma unroll
      for (int n = 0; n < NT; ++n) b[buf][k][n] = load_b(i0 + k, n);
    }
  };
  load(0, 0);
#pragma unroll
  for (int i0 = 0; i0 < NC; i0 += GC) {
    const int cur = i0 / GC & 1;
    if (i0 + GC < NC) load(i0 + GC, cur ^ 1);
    __builtin_amdgcn_sched_barrier(0);  // keeps the loads ahead of the products
#pragma unroll
    for (int k = 0; k < GC; ++k) {
      const uint4 z = a[cur][k];
      const bool v = on[cur][k];
      const uint4 av = make_uint4(v ? z.x : 0, v ? z.y : 0, v ? z.z : 0, v ? z.w : 0);
#pragma unroll
      for (int n = 0; n < NT; ++n)
        acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(v8bf, av), __builtin_bit_cast(v8bf, b[cur][k][n]), acc[n], 0, 0, 0);
    }
  }
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint32_t o = tile * 16 + 4 * g + r;
      if (o >= P) continue;
      float v = acc[n][r];
      if (UP) v += bf2f(sk[n][r]);
      out[(uint64_t)o * COUT + (nt0 + n) * 16 + li] = f2bf(fmaxf(v, 0.f));
    }
}

// first layer: one FP32 input channel -> 16, ReLU; a wave holds 64 nodes and
// four of the channels (one 8-byte store), weights in scalar registers
__global__ void __launch_bounds__(kBlock)
k_conv_first(const float *__restrict__ in, const float *__restrict__ W, uint16_t *__restrict__ out,
             Dims d) {
  const uint32_t P = d.x * d.y * d.z;
  const uint32_t i = blockIdx.x * 64 + (threadIdx.x & 63);
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (i >= P) return;
  int x, y, z;
  decode(i, d, x, y, z);
  float v[27];
#pragma unroll
  for (int t = 0; t < 27; ++t) {
    const int64_t s = tap_source<1, false>(x, y, z, t, d, d);
    v[t] = in[s >= 0 ? s : (int64_t)i];
    v[t] = s >= 0 ? v[t] : 0.f;
  }
  uint16_t o[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    float a = 0.f;
#pragma unroll
    for (int t = 0; t < 27; ++t) a += W[(4 * wv + c) * 27 + t] * v[t];
    o[c] = f2bf(fmaxf(a, 0.f));
  }
  *reinterpret_cast<uint2 *>(out + (uint64_t)i * 16 + 4 * wv) =
      make_uint2((uint32_t)o[0] | (uint32_t)o[1] << 16, (uint32_t)o[2] | (uint32_t)o[3] << 16);
}

// last layer: 16 -> 1 FP32 output, no activation; thread per node, a plane of
// nine taps loaded ahead of its products (one FMA chain over taps and channels;
// taps outside the grid are left out)
__global__ void __launch_bounds__(kBlock)
k_conv_last(const uint16_t *__restrict__ in, const float *__restrict__ W, float *__restrict__ out,
            Dims d) {
  const uint32_t P = d.x * d.y * d.z;
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= P) return;
  int x, y, z;
  decode(i, d, x, y, z);
  float a = 0.f;
  uint4 v[2][9][2];
  auto load = [&](int tz, int buf) {
#pragma unroll
    for (int t = 0; t < 9; ++t) {
      const int64_t s = tap_source<1, false>(x, y, z, 9 * tz + t, d, d);
      const uint4 *src = reinterpret_cast<const uint4 *>(in + (s >= 0 ? s : (int64_t)i) * 16);
      v[buf][t][0] = src[0];
      v[buf][t][1] = src[1];
    }
  };
  load(0, 0);
#pragma unroll
  for (int tz = 0; tz < 3; ++tz) {
    if (tz < 2) load(tz + 1, (tz + 1) & 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 9; ++t) {
      const uint4 lo = v[tz & 1][t][0], hi = v[tz & 1][t][1];
      const uint32_t w32[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      float s = a;
#pragma unroll
      for (int c = 0; c < 16; ++c)
        s += W[(9 * tz + t) * 16 + c] *
             bf2f((uint16_t)(w32[c >> 1] >> (16 * (c & 1))));
      a = tap_source<1, false>(x, y, z, 9 * tz + t, d, d) >= 0 ? s : a;
    }
  }
  out[i] = a;
}

// ---------------------------------------------------------------- backward
// Output gradients G are FP32 channels-last with a node's channels in slot
// order: channel o of C at slot (o % 4) (C / 4) + o / 4, so that the lane
// group g of a wave, which multiplies the channels o = 4 s + g (s = 0, 1, ...)
// in v_mfma_f32_16x16x4_f32, reads its channels of four consecutive steps as
// one 16-byte load.
__device__ __forceinline__ int slot_of(int ch, int C) { return (ch & 3) * (C / 4) + (ch >> 2); }

// one tap of the data gradient: acc[n] += G[rows][o] W[o][t][16 (nt0 + n) ..]
// over the COUT channels in ascending order.  The FP32 MFMA adds its four
// products to the accumulator one after the other with a rounding each (an
// FMA chain, checked on the device), so the sums are those of a scalar loop
// over (tap, channel).
template <int COUT, int NT>
struct AdjTap {
  v4f a[COUT / 16], b[NT][COUT / 16];
  // g: this lane's row at its channel group; w: the packed weights of the tap
  // and of the wave's first 16 input channels
  __device__ __forceinline__ void load(const float *g, const float *w, int lane) {
#pragma unroll
    for (int i = 0; i < COUT / 16; ++i) {
      a[i] = *reinterpret_cast<const v4f *>(g + 4 * i);
#pragma unroll
      for (int n = 0; n < NT; ++n)
        b[n][i] = *reinterpret_cast<const v4f *>(w + ((n * (COUT / 16) + i) * 64 + lane) * 4);
    }
  }
  __device__ __forceinline__ void mac(bool on, v4f *acc) const {
#pragma unroll
    for (int i = 0; i < COUT / 16; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float av = on ? a[i][j] : 0.f;
#pragma unroll
        for (int n = 0; n < NT; ++n)
          acc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, b[n][i][j], acc[n], 0, 0, 0);
      }
  }
};

// Data gradient of a stride-1 convolution over an up-sampled input, summed
// to the coarse grid and masked: out[j][c] = (act[j][c] > 0) sum over the
// fine children q of j of sum_{t,o} W[o][t][c] G[q - off_t][o].
// A wave's 16 rows are the 8 children of 2 coarse nodes, its columns NT tiles
// of 16 input channels; the children's sum is taken in the registers (the
// fine-grid gradient is never stored).  Bound by the FP32 matrix rate on
// large grids and by the chain of 27 COUT / 4 MFMAs on small ones; the taps'
// operands are loaded a group of GT taps ahead.  On a 33^3 grid the three
// layers take 17.5, 12.8 and 17.7 us, against 201 us on average (plus 4.8 us
// for the children's sum) with one thread per output on the vector units.
template <int CIN, int COUT, int NT, int GT>
__global__ void __launch_bounds__(kBlock)
k_adjoint_up(const float *__restrict__ G, const float *__restrict__ wa,
             const uint16_t *__restrict__ act, float *__restrict__ out, Dims fd, Dims cd) {
  static_assert(27 % GT == 0 && CIN % (16 * NT) == 0, "tile shape");
  constexpr int WPN = CIN / 16 / NT;  // waves per node tile
  const int lane = threadIdx.x & 63;
  const uint32_t w = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  const uint32_t tile = w / WPN;
  const int nt0 = (int)(w % WPN) * NT;
  const uint32_t P = cd.x * cd.y * cd.z;
  if (tile >= (P + 1) / 2) return;
  const int g = lane >> 4, m = lane & 15;
  // this lane's row: child m % 8 of coarse node 2 tile + m / 8
  uint32_t mask = 0;
  const float *row = G + g * (COUT / 4);
  {
    const uint32_t j = 2 * tile + (m >> 3);
    int X, Y, Z;
    decode(j, cd, X, Y, Z);
    const int x = 2 * X + (m & 1), y = 2 * Y + ((m >> 1) & 1), z = 2 * Z + ((m >> 2) & 1);
    if (j < P && inside(x, y, z, fd)) {
      row += lin(x, y, z, fd) * COUT;
#pragma unroll
      for (int t = 0; t < 27; ++t)
        if (inside(x - (t % 3 - 1), y - (t / 3 % 3 - 1), z - (t / 9 - 1), fd)) mask |= 1u << t;
    }
  }
  const int64_t sy = (int64_t)fd.x * COUT, sz = sy * fd.y;
  auto src = [&](int t) -> const float * {
    const int64_t off = (t % 3 - 1) * COUT + (t / 3 % 3 - 1) * sy + (t / 9 - 1) * sz;
    return (mask >> t & 1) ? row - off : row;  // an outside tap reads the row itself, unused
  };
  auto wgt = [&](int t) { return wa + (size_t)(t * (CIN / 16) + nt0) * COUT * 16; };
  v4f acc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[n] = v4f{0.f, 0.f, 0.f, 0.f};
  AdjTap<COUT, NT> cur[GT], nxt[GT];
#pragma unroll
  for (int k = 0; k < GT; ++k) cur[k].load(src(k), wgt(k), lane);
#pragma unroll
  for (int t = 0; t < 27; t += GT) {
    if (t + GT < 27) {
#pragma unroll
      for (int k = 0; k < GT; ++k) nxt[k].load(src(t + GT + k), wgt(t + GT + k), lane);
      __builtin_amdgcn_sched_barrier(0);  // keeps the loads ahead of the products
    }
#pragma unroll
    for (int k = 0; k < GT; ++k) cur[k].mac(mask >> (t + k) & 1, acc);
    if (t + GT < 27) {
#pragma unroll
      for (int k = 0; k < GT; ++k) cur[k] = nxt[k];
    }
  }
  // rows 4 g .. 4 g + 3 are children 0-3 (even g) or 4-7 (odd g) of coarse
  // node 2 tile + g / 2: summed in child order, the even group first
  const uint32_t j = 2 * tile + (g >> 1);
  int X, Y, Z;
  decode(j, cd, X, Y, Z);
  const bool xi = 2 * X + 1 < (int)fd.x, yi = 2 * Y + 1 < (int)fd.y;
  const bool zi = !(g & 1) || 2 * Z + 1 < (int)fd.z;
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const bool in[4] = {zi, zi && xi, zi && yi, zi && xi && yi};
    float s = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) s = in[r] ? s + acc[n][r] : s;
    s = __shfl(s, lane & 47, 64);  // odd groups: the even group's sum
#pragma unroll
    for (int r = 0; r < 4; ++r) s = in[r] ? s + acc[n][r] : s;
    const int ch = (nt0 + n) * 16 + m;
    if ((g & 1) && j < P)
      out[(uint64_t)j * CIN + slot_of(ch, CIN)] =
          bf2f(act[(uint64_t)j * CIN + ch]) > 0.f ? s : 0.f;
  }
}

// Data gradient of a stride-2 convolution, added to `add` and masked:
// out[q][c] = (act[q][c] > 0) (add[q][c] + sum_{t,o} W[o][t][c]
// G[(q - off_t) / 2][o]) over the taps whose source lands on q.  A node's
// taps depend on the parity of its coordinates only: even takes the middle
// tap of its axis, odd the two outer ones.  blockIdx.y is the parity class,
// so a wave's 16 rows share their 1, 2, 4 or 8 taps.  On a 33^3 grid 9.7-9.9
// us per layer, against 119 us on average (plus 4.8 us for the masked sum)
// with one thread per output on the vector units.
template <int CIN, int COUT, int NT>
__global__ void __launch_bounds__(kBlock)
k_adjoint_down(const float *__restrict__ G, const float *__restrict__ wa,
               const float *__restrict__ add, const uint16_t *__restrict__ act,
               float *__restrict__ out, Dims od, Dims xd) {
  constexpr int WPN = CIN / 16 / NT;
  const int cx = blockIdx.y & 1, cy = blockIdx.y >> 1 & 1, cz = blockIdx.y >> 2;
  const Dims kd{(xd.x + 1 - cx) / 2, (xd.y + 1 - cy) / 2, (xd.z + 1 - cz) / 2};  // class grid
  const uint32_t P = kd.x * kd.y * kd.z;
  const int lane = threadIdx.x & 63;
  const uint32_t w = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  const uint32_t tile = w / WPN;
  const int nt0 = (int)(w % WPN) * NT;
  if (tile >= (P + 15) / 16) return;
  const int g = lane >> 4, m = lane & 15;
  int ix, iy, iz;
  const bool valid = tile * 16 + m < P;
  decode(valid ? tile * 16 + m : 0, kd, ix, iy, iz);
  const int n_taps = (1 + cx) << (cy + cz);
  // tap i of the class, ascending: along an odd axis first tap 0 (source
  // node i + 1), then tap 2 (source i); along an even one tap 1 (source i)
  bool on_cur, on_nxt = false;
  AdjTap<COUT, NT> cur, nxt;
  auto load = [&](int i, AdjTap<COUT, NT> &v) -> bool {
    const int kx = cx ? i & 1 : 1, ky = cy ? (i >> cx) & 1 : 1, kz = cz ? i >> (cx + cy) : 1;
    const int px = ix + 1 - kx, py = iy + 1 - ky, pz = iz + 1 - kz;
    const int t = (cx ? 2 * kx : 1) + 3 * (cy ? 2 * ky : 1) + 9 * (cz ? 2 * kz : 1);
    const bool on = valid && inside(px, py, pz, od);
    v.load(G + (on ? lin(px, py, pz, od) : 0) * COUT + g * (COUT / 4),
           wa + (size_t)(t * (CIN / 16) + nt0) * COUT * 16, lane);
    return on;
  };
  v4f acc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[n] = v4f{0.f, 0.f, 0.f, 0.f};
  on_cur = load(0, cur);
  for (int i = 0; i < n_taps; ++i) {
    if (i + 1 < n_taps) on_nxt = load(i + 1, nxt);
    __builtin_amdgcn_sched_barrier(0);
    cur.mac(on_cur, acc);
    cur = nxt;
    on_cur = on_nxt;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const uint32_t i = tile * 16 + 4 * g + r;
    if (i >= P) continue;
    decode(i, kd, ix, iy, iz);
    const uint64_t q = lin(2 * ix + cx, 2 * iy + cy, 2 * iz + cz, xd) * CIN;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int ch = (nt0 + n) * 16 + m;
      const uint64_t at = q + slot_of(ch, CIN);
      const float v = add[at] + acc[n][r];
      out[at] = bf2f(act[q + ch]) > 0.f ? v : 0.f;
    }
  }
}

// Weight gradients dW[o][t][c] = sum_p G[p][o] X(s p + off_t)[c] of all layers
// in one launch (WgradArgs: per layer its operands, block range and parts;
// the layers are independent once the data gradients are known, and alone
// none of them has waves enough for the device).  Every unit writes a partial
// [part][o][t][c]; k_wgrad_reduce sums the parts in a fixed order.
struct WgradLayer {
  const uint16_t *in;  // bf16 activations (layer 0: nullptr)
  const float *G;      // output gradients, slot order (layer 7: dy)
  float *part;
  Dims od, id;
  uint32_t n_parts, block0;  // first block of this layer
};
struct WgradArgs {
  WgradLayer l[8];
  const float *x32;  // input of layer 0
};

// Layers 1-6 on MFMA (bf16 operands, FP32 accumulation), one unit per wave: 16
// output channels (rows) x CTW tiles of 16 input channels (columns) for the
// three taps of one x-row of the stencil, K = grid points, 32 per
// v_mfma_f32_16x16x32_bf16.  The output gradients are rounded to bf16 and
// loaded once for the three taps; with an up-sampled input the taps share
// two inputs per point, lo = (x - 1) / 2 and lo + 1.  A lane holds 8
// consecutive points, decoded once.  Bound by the latency of the gathered
// 2-byte and 4-byte loads: 38 us for all eight layers on a 33^3 grid, against
// 430 us in one launch per layer with one tap per workgroup, the loads of each
// tap by themselves and a 64-bit index division per point.
//
// The FP32 sums are taken in blocks of kSumChunks chunks, then over the blocks:
// on large grids a unit has hundreds of chunks, and one chain over all of them
// would round that often (257 x 129 x 129 nodes: 1044 chunks, 16 + 66 roundings
// instead).  The sums over the blocks wait in the LDS: in registers they cost the
// fourth wave per SIMD (33^3 grid 201 -> 205 us, 129^3 3781 -> 3927).  LONG: some unit
// has more than one block; the launch without it keeps the small grids' time (33^3 201 us,
// 202-203 with it).
constexpr uint32_t kSumChunks = 16;
constexpr int kWgradSums = 24;  // of a lane: 3 taps x 2 channel tiles x 4
template <bool LONG, int CIN, int COUT, int STRIDE, bool UP, int CTW>
__device__ __forceinline__ void wgrad_mfma(const WgradLayer &L, uint32_t unit,
                                           float (*blocks)[kBlock]) {
  static_assert(3 * CTW * 4 <= kWgradSums, "block sums");
  static_assert(CIN % (16 * CTW) == 0 && COUT % 16 == 0, "channel tiles");
  static_assert(UP == (STRIDE == 1), "the stride-1 layers read an up-sampled input");
  constexpr int OT = COUT / 16, CG = CIN / 16 / CTW;
  constexpr int NX = UP ? 2 : 3;  // inputs per point
  const int lane = threadIdx.x & 63, g = lane >> 4, li = lane & 15;
  const int ot = unit % OT, cg = unit / OT % CG, zy = unit / (OT * CG) % 9;
  const uint32_t pi = unit / (OT * CG * 9);
  if (pi >= L.n_parts) return;
  const int oy = zy % 3 - 1, oz = zy / 3 - 1;
  const uint32_t P = L.od.x * L.od.y * L.od.z, chunks = (P + 31) / 32;
  const uint32_t k0 = (uint64_t)chunks * pi / L.n_parts,
                 k1 = (uint64_t)chunks * (pi + 1) / L.n_parts;
  const int slot = slot_of(ot * 16 + li, COUT);
  const uint16_t *in = L.in + cg * CTW * 16 + li;
  v4f acc[3][CTW];
#pragma unroll
  for (int t = 0; t < 3; ++t)
#pragma unroll
    for (int b = 0; b < CTW; ++b) acc[t][b] = v4f{0.f, 0.f, 0.f, 0.f};
  for (uint32_t k = k0; k < k1; ++k) {
    if (LONG && k > k0 && (k - k0) % kSumChunks == 0) {
#pragma unroll
      for (int t = 0; t < 3; ++t)
#pragma unroll
        for (int b = 0; b < CTW; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float &s = blocks[(t * CTW + b) * 4 + r][threadIdx.x];
            s = k - k0 == kSumChunks ? acc[t][b][r] : s + acc[t][b][r];
            acc[t][b][r] = 0.f;
          }
    }
    const uint32_t p0 = k * 32 + 8 * g;
    int x, y, z;
    decode(p0 < P ? p0 : 0, L.od, x, y, z);
    uint16_t h[NX][CTW][8];
    float gv[8];
    uint32_t row_on = 0, left = 0, right = 0, odd = 0;  // per point
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const bool live = p0 + q < P;
      gv[q] = L.G[(uint64_t)(live ? p0 + q : 0) * COUT + slot];
      gv[q] = live ? gv[q] : 0.f;
      const int ry = STRIDE * y + oy, rz = STRIDE * z + oz;
      // the grid the taps are bounded by: the fine grid of an up-sampled input
      const Dims bd = UP ? L.od : L.id;
      const bool row = live && ry >= 0 && rz >= 0 && ry < (int)bd.y && rz < (int)bd.z;
      row_on |= (uint32_t)row << q;
      left |= (uint32_t)(STRIDE * x > 0) << q;
      right |= (uint32_t)(STRIDE * x + 1 < (int)bd.x) << q;
      odd |= (uint32_t)(x & 1) << q;
      const uint64_t base = row ? lin(0, UP ? ry >> 1 : ry, UP ? rz >> 1 : rz, L.id) : 0;
      const int lo = UP ? (x - 1) >> 1 : 2 * x - 1;
#pragma unroll
      for (int j = 0; j < NX; ++j) {
        const int xs = min(max(lo + j, 0), (int)L.id.x - 1);  // outside: read, not used
#pragma unroll
        for (int b = 0; b < CTW; ++b) h[j][b][q] = in[(base + xs) * CIN + b * 16];
      }
      if (++x == (int)L.od.x) {
        x = 0;
        if (++y == (int)L.od.y) {
          y = 0;
          ++z;
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // all loads of the chunk are in flight
    uint32_t gw[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      gw[q] = (uint32_t)f2bf(gv[2 * q]) | (uint32_t)f2bf(gv[2 * q + 1]) << 16;
    const v8bf ag = __builtin_bit_cast(v8bf, make_uint4(gw[0], gw[1], gw[2], gw[3]));
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      const uint32_t on = row_on & (t == 0 ? left : t == 2 ? right : ~0u);
#pragma unroll
      for (int b = 0; b < CTW; ++b) {
        uint32_t xw[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          uint32_t v[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const int i = 2 * q + e;
            // up-sampled middle tap: x / 2 is lo for odd x, lo + 1 for even x
            const uint16_t raw = !UP      ? h[t][b][i]
                                 : t == 0 ? h[0][b][i]
                                 : t == 2 ? h[1][b][i]
                                          : (odd >> i & 1 ? h[0][b][i] : h[1][b][i]);
            v[e] = (on >> i & 1) ? raw : 0u;
          }
          xw[q] = v[0] | v[1] << 16;
        }
        acc[t][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            ag, __builtin_bit_cast(v8bf, make_uint4(xw[0], xw[1], xw[2], xw[3])), acc[t][b], 0, 0,
            0);
      }
    }
  }
  // D layout: register r of a lane holds (o, c) = (16 ot + 4 g + r, 16 b + li)
#pragma unroll
  for (int t = 0; t < 3; ++t)
#pragma unroll
    for (int b = 0; b < CTW; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int o = ot * 16 + 4 * g + r, c = (cg * CTW + b) * 16 + li;
        float v = acc[t][b][r];
        if (LONG && k1 - k0 > kSumChunks) v += blocks[(t * CTW + b) * 4 + r][threadIdx.x];
        L.part[(((uint64_t)pi * COUT + o) * 27 + zy * 3 + t) * CIN + c] = v;
      }
}

// The two 1-channel layers (stride 1, FP32 products): the input layer (1 ->
// 16, input x32) and the head (16 -> 1, bf16 input, output gradient with one
// channel).  Per tap only 16 weights, so every thread accumulates all 16 over
// its share of the part's points; the sums go through wave shuffles and LDS.
template <bool HEAD>
__device__ __forceinline__ void wgrad_thin(const WgradLayer &L, const float *x32, uint32_t unit,
                                           float (*red)[16]) {
  const int t = unit % 27;
  const uint32_t pi = unit / 27, P = L.od.x * L.od.y * L.od.z;
  const uint32_t p0 = (uint64_t)P * pi / L.n_parts, p1 = (uint64_t)P * (pi + 1) / L.n_parts;
  float acc[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) acc[k] = 0.f;
  for (uint32_t p = p0 + threadIdx.x; p < p1; p += kBlock) {
    int x, y, z;
    decode(p, L.od, x, y, z);
    const int64_t src = tap_source<1, false>(x, y, z, t, L.od, L.od);
    if (src < 0) continue;
    if constexpr (HEAD) {  // dW[0][t][c] = sum_p dy[p] act[p + off_t][c]
      const float g = L.G[p];
      const uint16_t *a = L.in + (uint64_t)src * 16;
#pragma unroll
      for (int k = 0; k < 16; ++k) acc[k] += g * bf2f(a[k]);
    } else {  // dW[o][t][0] = sum_p G[p][o] x[p + off_t]
      const float xv = x32[src];
      const float *g = L.G + (uint64_t)p * 16;
#pragma unroll
      for (int k = 0; k < 16; ++k) acc[k] += g[slot_of(k, 16)] * xv;
    }
  }
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    float v = acc[k];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    acc[k] = v;
  }
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int k = 0; k < 16; ++k) red[threadIdx.x >> 6][k] = acc[k];
  __syncthreads();
  if (threadIdx.x < 16) {
    const int k = threadIdx.x;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) v += red[w][k];
    // HEAD: cout 1, cin 16 (c = k); else cout 16 (o = k), cin 1
    L.part[HEAD ? ((uint64_t)pi * 27 + t) * 16 + k : ((uint64_t)pi * 16 + k) * 27 + t] = v;
  }
}

// block ranges in the order of the layers below (longest units first)
constexpr int kWgradOrder[8] = {6, 5, 1, 4, 2, 3, 7, 0};

template <bool LONG>
__global__ void __launch_bounds__(kBlock) k_wgrad(WgradArgs a) {
  __shared__ float red[kBlock / 64][16];
  __shared__ float blocks[LONG ? kWgradSums : 1][kBlock];
  const uint32_t b = blockIdx.x;
  auto wave_unit = [&](int l) {
    return (b - a.l[l].block0) * (kBlock / 64) + (threadIdx.x >> 6);
  };
  if (b < a.l[5].block0) return wgrad_mfma<LONG, 32, 16, 1, true, 2>(a.l[6], wave_unit(6), blocks);
  if (b < a.l[1].block0) return wgrad_mfma<LONG, 64, 32, 1, true, 2>(a.l[5], wave_unit(5), blocks);
  if (b < a.l[4].block0) return wgrad_mfma<LONG, 16, 32, 2, false, 1>(a.l[1], wave_unit(1), blocks);
  if (b < a.l[2].block0) return wgrad_mfma<LONG, 64, 64, 1, true, 2>(a.l[4], wave_unit(4), blocks);
  if (b < a.l[3].block0) return wgrad_mfma<LONG, 32, 64, 2, false, 2>(a.l[2], wave_unit(2), blocks);
  if (b < a.l[7].block0) return wgrad_mfma<LONG, 64, 64, 2, false, 2>(a.l[3], wave_unit(3), blocks);
  if (b < a.l[0].block0) return wgrad_thin<true>(a.l[7], nullptr, b - a.l[7].block0, red);
  wgrad_thin<false>(a.l[0], a.x32, b - a.l[0].block0, red);
}

// grad[w] += sum over its layer's parts of part[part][w], in a fixed order:
// four strided sums per weight, then their sum
struct ReduceArgs {
  const float *part[8];
  uint32_t n_parts[8], w0[9];  // first weight of each layer
};
__global__ void __launch_bounds__(kBlock) k_wgrad_reduce(ReduceArgs a, float *__restrict__ grad) {
  __shared__ float red[4][64];
  const int j = threadIdx.x >> 6, i = threadIdx.x & 63;
  const uint32_t w = blockIdx.x * 64 + i;
  float s = 0.f;
  if (w < a.w0[8]) {
    int l = 0;
    while (w >= a.w0[l + 1]) ++l;
    const uint32_t nw = a.w0[l + 1] - a.w0[l];
    const float *p = a.part[l] + (w - a.w0[l]);
#pragma unroll 4
    for (uint32_t k = j; k < a.n_parts[l]; k += 4) s += p[(uint64_t)k * nw];
  }
  red[j][i] = s;
  __syncthreads();
  if (j == 0 && w < a.w0[8]) grad[w] += ((red[0][i] + red[1][i]) + red[2][i]) + red[3][i];
}

// head backward: g[p][c] = (sum_t W[t][c] dy[p - off_t]) * (act[p][c] > 0),
// stored in slot order.  A wave holds 64 nodes and the four channels c = 4 j +
// wave (one 16-byte store), with the weights in scalar registers; the taps
// outside the grid are left out of the sum.
__global__ void __launch_bounds__(kBlock)
k_head_backward(const float *__restrict__ dy, const float *__restrict__ W,
                const uint16_t *__restrict__ act, float *__restrict__ g, Dims d) {
  const uint32_t P = d.x * d.y * d.z;
  const uint32_t i = blockIdx.x * 64 + (threadIdx.x & 63);
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (i >= P) return;
  int x, y, z;
  decode(i, d, x, y, z);
  float v[27];
  uint32_t mask = 0;
#pragma unroll
  for (int t = 0; t < 27; ++t) {
    const int px = x - (t % 3 - 1), py = y - ((t / 3) % 3 - 1), pz = z - (t / 9 - 1);
    const bool on = inside(px, py, pz, d);
    mask |= (uint32_t)on << t;
    v[t] = dy[on ? lin(px, py, pz, d) : i];
  }
  v4f o;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float a = 0.f;
#pragma unroll
    for (int t = 0; t < 27; ++t) a = (mask >> t & 1) ? a + W[t * 16 + 4 * j + wv] * v[t] : a;
    o[j] = bf2f(act[(uint64_t)i * 16 + 4 * j + wv]) > 0.f ? a : 0.f;
  }
  *reinterpret_cast<v4f *>(g + (uint64_t)i * 16 + 4 * wv) = o;
}

// loss pieces: dy = scale (y - target) on free nodes (0 on masked nodes),
// partial sums of (y - target)^2 per block
__global__ void __launch_bounds__(kBlock)
k_mse(const float *__restrict__ y, const float *__restrict__ target,
      const uint8_t *__restrict__ mask, float scale, float *__restrict__ dy,
      double *__restrict__ part, uint64_t n) {
  __shared__ double red[kBlock / 64];
  double s = 0.0;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * kBlock) {
    const float d = (mask && mask[i]) ? 0.f : y[i] - target[i];
    dy[i] = scale * d;
    s += (double)d * d;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double a = 0.0;
    for (int w = 0; w < kBlock / 64; ++w) a += red[w];
    part[blockIdx.x] = a;
  }
}

__global__ void k_adam(float *__restrict__ w, float *__restrict__ m, float *__restrict__ v,
                       const float *__restrict__ g, uint32_t n, float lr, float b1, float b2,
                       float eps, float c1, float c2) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// layer weights [o][t][c] FP32 -> bf16 (k = t cin + c, zero padded to kp) in
// the order k_conv_mfma reads them, [k / 32][o / 16][lane 16 (k / 8 % 4) + o %
// 16][k % 8], and the FP32 value of each bf16 weight in the order AdjTap reads
// it, wa[t][c / 16][o / 16][lane 16 (o % 4) + c % 16][(o / 4) % 4] (both where
// the channel counts are multiples of 16, wa given) and as wr[o][t][c]
__global__ void k_pack_weights(const float *__restrict__ w, uint16_t *__restrict__ wb,
                               float *__restrict__ wr, float *__restrict__ wa, int cin, int cout,
                               int kp) {
  const int n = cout * kp;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const int o = i / kp, k = i - o * kp;
  const int K = 27 * cin;
  uint16_t h = 0;
  if (k < K) {
    h = f2bf(w[o * K + k]);
    wr[o * K + k] = bf2f(h);
    if (wa) {
      const int t = k / cin, c = k - t * cin;
      wa[((((t * (cin / 16) + c / 16) * (cout / 16) + o / 16) * 64 + (o & 3) * 16 + c % 16) * 4) +
         ((o >> 2) & 3)] = bf2f(h);
    }
  }
  if (wa) wb[((size_t)(k / 32 * (cout / 16) + o / 16) * 64 + (k >> 3 & 3) * 16 + o % 16) * 8 + k % 8] = h;
}

__global__ void k_scale_to_f32(const double *__restrict__ r, float *__restrict__ out, double s,
                               uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) out[i] = (float)(r[i] * s);
}

__global__ void k_scale_to_f64(const float *__restrict__ y, double *__restrict__ z, double s,
                               uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) z[i] = (double)y[i] * s;
}

__global__ void k_axpy_f32(float *__restrict__ x, float a, const float *__restrict__ y, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) x[i] += a * y[i];
}

constexpr uint64_t kSpreadWaves = 4096;  // four waves per SIMD

inline unsigned blocks(uint64_t n) { return (unsigned)std::max<uint64_t>(1, (n + kBlock - 1) / kBlock); }
inline Dims D3(const uint32_t *d) { return Dims{d[0], d[1], d[2]}; }

// Channel tiles per wave: one while the waves do not fill the device (each
// then waits for its own loads only), all of them on larger grids, where the
// gathered rows are then loaded once for all channels.  The whole network
// against the form with all tiles in a wave and no loads ahead: 63 us / 146 on
// 33^3 nodes, 145 / 241 on 65^3, 5.6 ms / 7.3 on 257^3.
template <int CIN, int COUT, int STRIDE, bool UP>
void mfma_launch(const uint16_t *in, const uint16_t *W, const uint16_t *skip, uint16_t *out,
                 const uint32_t *od, const uint32_t *id, hipStream_t s) {
  constexpr int NT = COUT / 16;
  const uint64_t tiles = ((uint64_t)od[0] * od[1] * od[2] + 15) / 16;
  if (NT == 1 || tiles * NT <= kSpreadWaves)
    hipLaunchKernelGGL((k_conv_mfma<CIN, COUT, STRIDE, UP, 1>), dim3(blocks(tiles * NT * 64)),
                       dim3(kBlock), 0, s, in, W, skip, out, D3(od), D3(id));
  else
    hipLaunchKernelGGL((k_conv_mfma<CIN, COUT, STRIDE, UP, NT>), dim3(blocks(tiles * 64)),
                       dim3(kBlock), 0, s, in, W, skip, out, D3(od), D3(id));
}

}  // namespace

void nn_conv_forward(int layer, const uint16_t *in, const float *in32, const uint16_t *wb,
                     const float *wr, const uint16_t *skip, uint16_t *out, float *out32,
                     const uint32_t *od, const uint32_t *id, hipStream_t s) {
  const uint64_t P = (uint64_t)od[0] * od[1] * od[2];
  switch (layer) {
    case 0: hipLaunchKernelGGL(k_conv_first, dim3((unsigned)((P + 63) / 64)), dim3(kBlock), 0, s, in32, wr, out, D3(od)); break;
    case 1: mfma_launch<16, 32, 2, false>(in, wb, nullptr, out, od, id, s); break;
    case 2: mfma_launch<32, 64, 2, false>(in, wb, nullptr, out, od, id, s); break;
    case 3: mfma_launch<64, 64, 2, false>(in, wb, nullptr, out, od, id, s); break;
    case 4: mfma_launch<64, 64, 1, true>(in, wb, skip, out, od, id, s); break;
    case 5: mfma_launch<64, 32, 1, true>(in, wb, skip, out, od, id, s); break;
    case 6: mfma_launch<32, 16, 1, true>(in, wb, skip, out, od, id, s); break;
    case 7: hipLaunchKernelGGL(k_conv_last, dim3(blocks(P)), dim3(kBlock), 0, s, in, wr, out32, D3(od)); break;
    default: throw Error{MFX_ERR_INVALID_ARG, "layer out of range"};
  }
  MFX_HIP(hipGetLastError());
}

namespace {
template <int CIN, int COUT, int NT, int GT>
void adjoint_up(const float *G, const float *wa, const uint16_t *act, float *out,
                const uint32_t *fd, const uint32_t *cd, hipStream_t s) {
  const uint64_t tiles = ((uint64_t)cd[0] * cd[1] * cd[2] + 1) / 2;
  hipLaunchKernelGGL((k_adjoint_up<CIN, COUT, NT, GT>), dim3(blocks(tiles * (CIN / 16 / NT) * 64)),
                     dim3(kBlock), 0, s, G, wa, act, out, D3(fd), D3(cd));
}
template <int CIN, int COUT, int NT>
void adjoint_down(const float *G, const float *wa, const float *add, const uint16_t *act,
                  float *out, const uint32_t *od, const uint32_t *xd, hipStream_t s) {
  // the all-even parity class is the largest
  const uint64_t n = (uint64_t)((xd[0] + 1) / 2) * ((xd[1] + 1) / 2) * ((xd[2] + 1) / 2);
  hipLaunchKernelGGL((k_adjoint_down<CIN, COUT, NT>),
                     dim3(blocks((n + 15) / 16 * (CIN / 16 / NT) * 64), 8), dim3(kBlock), 0, s, G,
                     wa, add, act, out, D3(od), D3(xd));
}
}  // namespace

void nn_conv_adjoint(int layer, const float *G, const float *wa, const float *add,
                     const uint16_t *act, float *out, const uint32_t *od, const uint32_t *xd,
                     hipStream_t s) {
  // input-channel tiles per wave (NT): two where the grid has waves enough
  switch (layer) {
    case 1: adjoint_down<16, 32, 1>(G, wa, add, act, out, od, xd, s); break;
    case 2: adjoint_down<32, 64, 1>(G, wa, add, act, out, od, xd, s); break;
    case 3: adjoint_down<64, 64, 1>(G, wa, add, act, out, od, xd, s); break;
    case 4: adjoint_up<64, 64, 1, 1>(G, wa, act, out, od, xd, s); break;
    case 5: adjoint_up<64, 32, 2, 1>(G, wa, act, out, od, xd, s); break;
    case 6: adjoint_up<32, 16, 2, 3>(G, wa, act, out, od, xd, s); break;
    default: throw Error{MFX_ERR_INVALID_ARG, "layer has no data gradient"};
  }
  MFX_HIP(hipGetLastError());
}

uint32_t nn_wgrad_parts(int layer, const uint32_t *od) {
  const uint64_t P = (uint64_t)od[0] * od[1] * od[2];
  // MFMA layers: units of at least four 32-point chunks; the 1-channel ones:
  // blocks of at least four points per thread
  const uint64_t n = (layer == 0 || layer == 7) ? P / (4 * kBlock) : (P + 31) / 32 / 4;
  return (uint32_t)std::min<uint64_t>(std::max<uint64_t>(n, 1), 128);
}

void nn_wgrad(const NnWgrad (&l)[8], const float *x32, float *grad, hipStream_t s) {
  // units (waves) per part of the MFMA layers: 9 x-rows of taps x output tiles
  // x input tile groups, as the instances in k_wgrad split them
  const uint32_t units[8] = {0, 9 * 2, 9 * 4, 9 * 4 * 2, 9 * 4 * 2, 9 * 2 * 2, 9, 0};
  WgradArgs a;
  ReduceArgs r;
  a.x32 = x32;
  uint32_t block = 0;
  bool long_units = false;
  for (int k : kWgradOrder) {
    const bool thin = k == 0 || k == 7;
    const uint64_t chunks = ((uint64_t)l[k].od[0] * l[k].od[1] * l[k].od[2] + 31) / 32;
    long_units = long_units || (!thin && chunks > (uint64_t)kSumChunks * l[k].n_parts);
    a.l[k] = WgradLayer{l[k].in, l[k].G, l[k].part, D3(l[k].od), D3(l[k].id), l[k].n_parts, block};
    block += thin ? 27 * l[k].n_parts
                  : (units[k] * l[k].n_parts + kBlock / 64 - 1) / (kBlock / 64);
  }
  uint32_t w = 0;
  for (int k = 0; k < 8; ++k) {
    r.part[k] = l[k].part;
    r.n_parts[k] = l[k].n_parts;
    r.w0[k] = w;
    w += l[k].n_weights;
  }
  r.w0[8] = w;
  if (long_units)
    hipLaunchKernelGGL(k_wgrad<true>, dim3(block), dim3(kBlock), 0, s, a);
  else
    hipLaunchKernelGGL(k_wgrad<false>, dim3(block), dim3(kBlock), 0, s, a);
  hipLaunchKernelGGL(k_wgrad_reduce, dim3((w + 63) / 64), dim3(kBlock), 0, s, r, grad);
  MFX_HIP(hipGetLastError());
}

void nn_head_backward(const float *dy, const float *W, const uint16_t *act, float *g,
                      const uint32_t *d, hipStream_t s) {
  const uint64_t n = (uint64_t)d[0] * d[1] * d[2];
  hipLaunchKernelGGL(k_head_backward, dim3((unsigned)((n + 63) / 64)), dim3(kBlock), 0, s, dy, W, act, g, D3(d));
  MFX_HIP(hipGetLastError());
}

uint32_t nn_mse_blocks(uint64_t n) {
  return (uint32_t)std::min<uint64_t>(std::max<uint64_t>(1, (n + kBlock - 1) / kBlock), 1024);
}

void nn_mse(const float *y, const float *target, const uint8_t *mask, float scale, float *dy,
            double *part, uint64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_mse, dim3(nn_mse_blocks(n)), dim3(kBlock), 0, s, y, target, mask, scale, dy,
                     part, n);
  MFX_HIP(hipGetLastError());
}

void nn_adam(float *w, float *m, float *v, const float *g, uint32_t n, float lr, float b1, float b2,
             float eps, int step, hipStream_t s) {
  const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
  hipLaunchKernelGGL(k_adam, dim3(blocks(n)), dim3(kBlock), 0, s, w, m, v, g, n, lr, b1, b2, eps,
                     c1, c2);
  MFX_HIP(hipGetLastError());
}

void nn_pack_weights(const float *w, uint16_t *wb, float *wr, float *wa, int cin, int cout, int kp,
                     hipStream_t s) {
  if (cin % 16 || cout % 16) wa = nullptr;
  hipLaunchKernelGGL(k_pack_weights, dim3(blocks((uint64_t)cout * kp)), dim3(kBlock), 0, s, w, wb,
                     wr, wa, cin, cout, kp);
  MFX_HIP(hipGetLastError());
}

void nn_scale_to_f32(const double *r, float *out, double s_, uint64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_scale_to_f32, dim3(blocks(n)), dim3(kBlock), 0, s, r, out, s_, n);
  MFX_HIP(hipGetLastError());
}

void nn_axpy_f32(float *x, float a, const float *y, uint64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_axpy_f32, dim3(blocks(n)), dim3(kBlock), 0, s, x, a, y, n);
  MFX_HIP(hipGetLastError());
}

void nn_scale_to_f64(const float *y, double *z, double s_, uint64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_scale_to_f64, dim3(blocks(n)), dim3(kBlock), 0, s, y, z, s_, n);
  MFX_HIP(hipGetLastError());
}

}  // namespace mfx
