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
// consecutive output nodes and all output channels; the K dimension
// (t, c) runs in chunks of 32: lane l gathers 8 consecutive channels of one
// tap of node l % 16 (one 16-byte load, channels-last) as the A operand and
// 8 consecutive k of output channel l % 16 of the weights [o][k] as the B
// operand.  D register r of lane l is node 4 (l / 16) + r, channel l % 16.
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

__device__ __forceinline__ void decode(uint64_t i, const Dims &d, int &x, int &y, int &z) {
  x = (int)(i % d.x);
  const uint64_t q = i / d.x;
  y = (int)(q % d.y);
  z = (int)(q / d.y);
}

// the same for a 32-bit node index (node counts stay below 2^32: a grid of
// that many nodes exceeds the device's memory)
__device__ __forceinline__ void decode32(uint32_t i, const Dims &d, int &x, int &y, int &z) {
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

template <int CIN, int COUT, int STRIDE, bool UP, bool SKIP>
__global__ void __launch_bounds__(kBlock)
k_conv_mfma(const uint16_t *__restrict__ in, const uint16_t *__restrict__ W,
            const uint16_t *__restrict__ skip, uint16_t *__restrict__ out, Dims od, Dims id) {
  static_assert(CIN % 16 == 0 && COUT % 16 == 0, "channel counts must be multiples of 16");
  constexpr int K = 27 * CIN, KP = (K + 31) / 32 * 32, NT = COUT / 16;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t P = (uint64_t)od.x * od.y * od.z;
  const uint64_t base = ((uint64_t)blockIdx.x * (kBlock / 64) + wave) * 16;
  if (base >= P) return;
  const uint64_t node = base + (lane & 15);
  int x = 0, y = 0, z = 0;
  const bool valid = node < P;
  if (valid) decode(node, od, x, y, z);
  const int kl = 8 * (lane >> 4);
  v4f acc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[n] = v4f{0.f, 0.f, 0.f, 0.f};
  for (int kc = 0; kc < KP; kc += 32) {
    const int k = kc + kl;
    uint4 araw = make_uint4(0, 0, 0, 0);
    if (valid && k < K) {
      const int t = k / CIN, c = k - t * CIN;
      const int64_t src = tap_source<STRIDE, UP>(x, y, z, t, od, id);
      if (src >= 0) araw = *reinterpret_cast<const uint4 *>(in + (uint64_t)src * CIN + c);
    }
    const v8bf a = __builtin_bit_cast(v8bf, araw);
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const uint4 braw =
          *reinterpret_cast<const uint4 *>(W + (uint64_t)(n * 16 + (lane & 15)) * KP + k);
      acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(v8bf, braw), acc[n], 0,
                                                       0, 0);
    }
  }
  // epilogue: node base + 4 (lane / 16) + r, channel n * 16 + lane % 16
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint64_t o = base + 4 * (lane >> 4) + r;
      if (o >= P) continue;
      const int ch = n * 16 + (lane & 15);
      float v = acc[n][r];
      if (SKIP) v += bf2f(skip[o * COUT + ch]);
      out[o * COUT + ch] = f2bf(fmaxf(v, 0.f));
    }
}

// first layer: one FP32 input channel -> 16, ReLU; thread per node
__global__ void __launch_bounds__(kBlock)
k_conv_first(const float *__restrict__ in, const float *__restrict__ W, uint16_t *__restrict__ out,
             Dims d) {
  const uint64_t P = (uint64_t)d.x * d.y * d.z;
  const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= P) return;
  int x, y, z;
  decode(i, d, x, y, z);
  float v[27];
#pragma unroll
  for (int t = 0; t < 27; ++t) {
    const int64_t s = tap_source<1, false>(x, y, z, t, d, d);
    v[t] = s >= 0 ? in[s] : 0.f;
  }
  uint16_t o[16];
#pragma unroll
  for (int c = 0; c < 16; ++c) {
    float a = 0.f;
#pragma unroll
    for (int t = 0; t < 27; ++t) a += W[c * 27 + t] * v[t];
    o[c] = f2bf(fmaxf(a, 0.f));
  }
  uint32_t pk[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) pk[c] = (uint32_t)o[2 * c] | ((uint32_t)o[2 * c + 1] << 16);
  uint4 *dst = reinterpret_cast<uint4 *>(out + i * 16);
  dst[0] = make_uint4(pk[0], pk[1], pk[2], pk[3]);
  dst[1] = make_uint4(pk[4], pk[5], pk[6], pk[7]);
}

// last layer: 16 -> 1 FP32 output, no activation; thread per node
__global__ void __launch_bounds__(kBlock)
k_conv_last(const uint16_t *__restrict__ in, const float *__restrict__ W, float *__restrict__ out,
            Dims d) {
  const uint64_t P = (uint64_t)d.x * d.y * d.z;
  const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= P) return;
  int x, y, z;
  decode(i, d, x, y, z);
  float a = 0.f;
  for (int t = 0; t < 27; ++t) {
    const int64_t s = tap_source<1, false>(x, y, z, t, d, d);
    if (s < 0) continue;
    const uint4 *src = reinterpret_cast<const uint4 *>(in + (uint64_t)s * 16);
    const uint4 lo = src[0], hi = src[1];
    const uint32_t w32[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      const uint16_t h = (uint16_t)(w32[c >> 1] >> (16 * (c & 1)));
      a += W[t * 16 + c] * bf2f(h);
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
    decode32(j, cd, X, Y, Z);
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
  decode32(j, cd, X, Y, Z);
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
  decode32(valid ? tile * 16 + m : 0, kd, ix, iy, iz);
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
    decode32(i, kd, ix, iy, iz);
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

// partial weight gradients: block (t, part) sums over its node range
//   dW[o][t][c] += G[p][o] * in(s p + off_t)[c]
// in: bf16 channels-last (or FP32 when cin == 1 and in32 is set)
template <int STRIDE, bool UP>
__global__ void __launch_bounds__(kBlock)
k_conv_wgrad(const uint16_t *__restrict__ in, const float *__restrict__ in32,
             const float *__restrict__ G, float *__restrict__ part, Dims od, Dims id, int cin,
             int cout, uint32_t n_parts) {
  constexpr int PC = 16;  // nodes staged per round
  __shared__ float sX[PC][64];
  __shared__ float sG[PC][64];
  const int t = blockIdx.x;
  const uint32_t pi = blockIdx.y;
  const uint64_t P = (uint64_t)od.x * od.y * od.z;
  const uint64_t p0 = P * pi / n_parts, p1 = P * (pi + 1) / n_parts;
  const int nout = cin * cout;  // <= 4096: up to 16 per thread
  float acc[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) acc[k] = 0.f;
  for (uint64_t pb = p0; pb < p1; pb += PC) {
    __syncthreads();
    for (int e = threadIdx.x; e < PC * 64; e += kBlock) {
      const int j = e / 64, c = e % 64;
      const uint64_t p = pb + j;
      float xv = 0.f, gv = 0.f;
      if (p < p1) {
        int x, y, z;
        decode(p, od, x, y, z);
        if (c < cin) {
          const int64_t s = tap_source<STRIDE, UP>(x, y, z, t, od, id);
          if (s >= 0) xv = in32 ? in32[s] : bf2f(in[(uint64_t)s * cin + c]);
        }
        if (c < cout) gv = G[p * cout + (cout % 4 ? c : slot_of(c, cout))];
      }
      sX[j][c] = xv;
      sG[j][c] = gv;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int idx = threadIdx.x + k * kBlock;
      if (idx >= nout) break;
      const int o = idx / cin, c = idx - o * cin;
      float s = acc[k];
#pragma unroll
      for (int j = 0; j < PC; ++j) s += sG[j][o] * sX[j][c];
      acc[k] = s;
    }
  }
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const int idx = threadIdx.x + k * kBlock;
    if (idx >= nout) break;
    const int o = idx / cin, c = idx - o * cin;
    part[((uint64_t)pi * cout + o) * 27 * cin + (uint64_t)t * cin + c] = acc[k];
  }
}

// The same weight gradient on MFMA (bf16 inputs, FP32 accumulation), for
// channel counts that are multiples of 16: per tap t an implicit GEMM
// dW_t[o][c] = sum_p G[p][o] X[src(p, t)][c] with M = output channels,
// N = input channels and K = grid points, 32 points per
// v_mfma_f32_16x16x32_bf16.  Each wave owns every (o, c) tile and a
// strided share of the part's 32-point chunks; the output gradients G are
// rounded to bf16 (the activations X are stored in bf16 already).  The four
// waves are summed in LDS into the same per-part partials as k_conv_wgrad.
template <int CIN, int COUT, int STRIDE, bool UP>
__global__ void __launch_bounds__(kBlock)
k_conv_wgrad_mfma(const uint16_t *__restrict__ in, const float *__restrict__ G,
                  float *__restrict__ part, Dims od, Dims id, uint32_t n_parts) {
  static_assert(CIN % 16 == 0 && COUT % 16 == 0, "channel counts must be multiples of 16");
  constexpr int OT = COUT / 16, CT = CIN / 16, NW = kBlock / 64;
  __shared__ float red[NW][OT * CT * 4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int t = blockIdx.x;
  const uint32_t pi = blockIdx.y;
  const uint64_t P = (uint64_t)od.x * od.y * od.z;
  const uint64_t p0 = P * pi / n_parts, p1 = P * (pi + 1) / n_parts;
  const int kq = 8 * (lane >> 4), li = lane & 15;
  v4f acc[OT][CT];
#pragma unroll
  for (int a = 0; a < OT; ++a)
#pragma unroll
    for (int b = 0; b < CT; ++b) acc[a][b] = v4f{0.f, 0.f, 0.f, 0.f};
  for (uint64_t cb = p0 + 32 * (uint64_t)wave; cb < p1; cb += 32 * NW) {
    // this lane's 8 points of the chunk: k = kq .. kq + 7
    int64_t src[8];
    uint64_t pt[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      pt[q] = cb + kq + q;
      src[q] = -1;
      if (pt[q] < p1) {
        int x, y, z;
        decode(pt[q], od, x, y, z);
        src[q] = tap_source<STRIDE, UP>(x, y, z, t, od, id);
      }
    }
    v8bf bx[CT], ag[OT];
#pragma unroll
    for (int b = 0; b < CT; ++b) {
      uint16_t h[8];
#pragma unroll
      for (int q = 0; q < 8; ++q)
        h[q] = src[q] >= 0 ? in[(uint64_t)src[q] * CIN + b * 16 + li] : (uint16_t)0;
      const uint4 raw = make_uint4(h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16,
                                   h[4] | (uint32_t)h[5] << 16, h[6] | (uint32_t)h[7] << 16);
      bx[b] = __builtin_bit_cast(v8bf, raw);
    }
#pragma unroll
    for (int a = 0; a < OT; ++a) {
      uint16_t h[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) h[q] = pt[q] < p1 ? f2bf(G[pt[q] * COUT + slot_of(a * 16 + li, COUT)]) : 0;
      const uint4 raw = make_uint4(h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16,
                                   h[4] | (uint32_t)h[5] << 16, h[6] | (uint32_t)h[7] << 16);
      ag[a] = __builtin_bit_cast(v8bf, raw);
    }
#pragma unroll
    for (int a = 0; a < OT; ++a)
#pragma unroll
      for (int b = 0; b < CT; ++b)
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ag[a], bx[b], acc[a][b], 0, 0, 0);
  }
#pragma unroll
  for (int a = 0; a < OT; ++a)
#pragma unroll
    for (int b = 0; b < CT; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wave][(a * CT + b) * 4 + r][lane] = acc[a][b][r];
  __syncthreads();
  // D layout: register r of lane l holds (o, c) = (16 a + 4 (l / 16) + r, 16 b + l % 16)
  for (int e = threadIdx.x; e < OT * CT * 4 * 64; e += kBlock) {
    const int tr = e / 64, l = e % 64;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) v += red[w][tr][l];
    const int tile = tr / 4, r = tr % 4, a = tile / CT, b = tile % CT;
    const int o = a * 16 + 4 * (l >> 4) + r, c = b * 16 + (l & 15);
    part[((uint64_t)pi * COUT + o) * 27 * CIN + (uint64_t)t * CIN + c] = v;
  }
}

// Weight gradient of the two 1-channel layers (stride 1, no up-sampling):
// the input layer (1 -> 16, FP32 input in32) and the head (16 -> 1, bf16
// input in, output gradient with one channel).  Per tap only 16 weights, so
// every thread accumulates all 16 over its share of the part's points; the
// sums go through wave shuffles and LDS into the same per-part partials.
template <bool HEAD>
__global__ void __launch_bounds__(kBlock)
k_conv_wgrad_thin(const uint16_t *__restrict__ in, const float *__restrict__ in32,
                  const float *__restrict__ G, float *__restrict__ part, Dims od,
                  uint32_t n_parts) {
  __shared__ float red[kBlock / 64][16];
  const int t = blockIdx.x;
  const uint32_t pi = blockIdx.y;
  const uint64_t P = (uint64_t)od.x * od.y * od.z;
  const uint64_t p0 = P * pi / n_parts, p1 = P * (pi + 1) / n_parts;
  float acc[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) acc[k] = 0.f;
  for (uint64_t p = p0 + threadIdx.x; p < p1; p += kBlock) {
    int x, y, z;
    decode(p, od, x, y, z);
    const int64_t src = tap_source<1, false>(x, y, z, t, od, od);
    if (src < 0) continue;
    if constexpr (HEAD) {  // dW[0][t][c] = sum_p dy[p] act[p + off_t][c]
      const float g = G[p];
      const uint16_t *a = in + (uint64_t)src * 16;
#pragma unroll
      for (int k = 0; k < 16; ++k) acc[k] += g * bf2f(a[k]);
    } else {  // dW[o][t][0] = sum_p G[p][o] x[p + off_t]
      const float xv = in32[src];
      const float *g = G + p * 16;
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
    const uint64_t idx = HEAD ? ((uint64_t)pi * 27 + t) * 16 + k
                              : ((uint64_t)pi * 16 + k) * 27 + t;
    part[idx] = v;
  }
}

// grad[w] += sum over parts of part[part][w] (fixed order)
__global__ void k_wgrad_reduce(const float *__restrict__ part, float *__restrict__ grad, uint32_t nw,
                               uint32_t n_parts) {
  const uint32_t w = blockIdx.x * kBlock + threadIdx.x;
  if (w >= nw) return;
  float s = 0.f;
  for (uint32_t k = 0; k < n_parts; ++k) s += part[(uint64_t)k * nw + w];
  grad[w] += s;
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
  decode32(i, d, x, y, z);
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

// layer weights [o][t][c] FP32 -> bf16 [o][KP] (k = t cin + c, zero padded)
// and the FP32 value of each bf16 weight [o][t][c]; with wa (channel counts
// that are multiples of 16) also the FP32 value in the order AdjTap reads it:
// [t][c / 16][o / 16][lane 16 (o % 4) + c % 16][(o / 4) % 4]
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
  wb[i] = h;
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

inline unsigned blocks(uint64_t n) { return (unsigned)std::max<uint64_t>(1, (n + kBlock - 1) / kBlock); }
inline Dims D3(const uint32_t *d) { return Dims{d[0], d[1], d[2]}; }

template <int CIN, int COUT, int STRIDE, bool UP, bool SKIP>
void mfma_launch(const uint16_t *in, const uint16_t *W, const uint16_t *skip, uint16_t *out,
                 const uint32_t *od, const uint32_t *id, hipStream_t s) {
  const uint64_t P = (uint64_t)od[0] * od[1] * od[2];
  const uint64_t waves = (P + 15) / 16;
  hipLaunchKernelGGL((k_conv_mfma<CIN, COUT, STRIDE, UP, SKIP>), dim3(blocks(waves * 64)),
                     dim3(kBlock), 0, s, in, W, skip, out, D3(od), D3(id));
}

}  // namespace

void nn_conv_forward(int layer, const uint16_t *in, const float *in32, const uint16_t *wb,
                     const float *wr, const uint16_t *skip, uint16_t *out, float *out32,
                     const uint32_t *od, const uint32_t *id, hipStream_t s) {
  const uint64_t P = (uint64_t)od[0] * od[1] * od[2];
  switch (layer) {
    case 0: hipLaunchKernelGGL(k_conv_first, dim3(blocks(P)), dim3(kBlock), 0, s, in32, wr, out, D3(od)); break;
    case 1: mfma_launch<16, 32, 2, false, false>(in, wb, nullptr, out, od, id, s); break;
    case 2: mfma_launch<32, 64, 2, false, false>(in, wb, nullptr, out, od, id, s); break;
    case 3: mfma_launch<64, 64, 2, false, false>(in, wb, nullptr, out, od, id, s); break;
    case 4: mfma_launch<64, 64, 1, true, true>(in, wb, skip, out, od, id, s); break;
    case 5: mfma_launch<64, 32, 1, true, true>(in, wb, skip, out, od, id, s); break;
    case 6: mfma_launch<32, 16, 1, true, true>(in, wb, skip, out, od, id, s); break;
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

// the MFMA weight gradient for the layer shapes of the U-Net; false if the
// shape has no MFMA instance (then the VALU kernel runs)
template <int CI, int CO, int ST, bool UPF>
bool wgrad_mfma_if(int stride, bool up, const uint16_t *in, const float *G, float *part,
                   const uint32_t *od, const uint32_t *id, int cin, int cout, uint32_t n_parts,
                   hipStream_t s) {
  if (!(in && cin == CI && cout == CO && stride == ST && up == UPF)) return false;
  hipLaunchKernelGGL((k_conv_wgrad_mfma<CI, CO, ST, UPF>), dim3(27, n_parts), dim3(kBlock), 0, s,
                     in, G, part, D3(od), D3(id), n_parts);
  return true;
}
bool wgrad_mfma(int stride, bool up, const uint16_t *in, const float *G, float *part,
                const uint32_t *od, const uint32_t *id, int cin, int cout, uint32_t n_parts,
                hipStream_t s) {
  return wgrad_mfma_if<32, 16, 1, true>(stride, up, in, G, part, od, id, cin, cout, n_parts, s) ||
         wgrad_mfma_if<64, 32, 1, true>(stride, up, in, G, part, od, id, cin, cout, n_parts, s) ||
         wgrad_mfma_if<64, 64, 1, true>(stride, up, in, G, part, od, id, cin, cout, n_parts, s) ||
         wgrad_mfma_if<64, 64, 2, false>(stride, up, in, G, part, od, id, cin, cout, n_parts, s) ||
         wgrad_mfma_if<32, 64, 2, false>(stride, up, in, G, part, od, id, cin, cout, n_parts, s) ||
         wgrad_mfma_if<16, 32, 2, false>(stride, up, in, G, part, od, id, cin, cout, n_parts, s);
}

void nn_conv_wgrad(int stride, bool up, const uint16_t *in, const float *in32, const float *G,
                   float *part, float *grad, const uint32_t *od, const uint32_t *id, int cin,
                   int cout, uint32_t n_parts, hipStream_t s) {
  MFX_REQUIRE(cin <= 64 && cout <= 64 && cin * cout <= 16 * kBlock, "weight tile too large");
  const dim3 grid(27, n_parts);
  // the U-Net's layers with 16-multiple channel counts run on MFMA, the two
  // 1-channel layers on the thin kernel
  if (stride == 1 && !up && cin == 16 && cout == 1 && in) {
    hipLaunchKernelGGL(k_conv_wgrad_thin<true>, grid, dim3(kBlock), 0, s, in, nullptr, G, part,
                       D3(od), n_parts);
  } else if (stride == 1 && !up && cin == 1 && cout == 16 && in32) {
    hipLaunchKernelGGL(k_conv_wgrad_thin<false>, grid, dim3(kBlock), 0, s, nullptr, in32, G,
                       part, D3(od), n_parts);
  } else if (!wgrad_mfma(stride, up, in, G, part, od, id, cin, cout, n_parts, s)) {
    if (stride == 2)
      hipLaunchKernelGGL((k_conv_wgrad<2, false>), grid, dim3(kBlock), 0, s, in, in32, G, part,
                         D3(od), D3(id), cin, cout, n_parts);
    else if (up)
      hipLaunchKernelGGL((k_conv_wgrad<1, true>), grid, dim3(kBlock), 0, s, in, in32, G, part,
                         D3(od), D3(id), cin, cout, n_parts);
    else
      hipLaunchKernelGGL((k_conv_wgrad<1, false>), grid, dim3(kBlock), 0, s, in, in32, G, part,
                         D3(od), D3(id), cin, cout, n_parts);
  }
  const uint32_t nw = 27u * cin * cout;
  hipLaunchKernelGGL(k_wgrad_reduce, dim3(blocks(nw)), dim3(kBlock), 0, s, part, grad, nw, n_parts);
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
