// plane64.hip -- FP64 instances of the plane-per-lane operator kernel, and the
// choice of its work split.
#include <cmath>

#include "plane_kernel.hpp"

namespace mfx {

template bool plane_instance<double>(int, int, bool, bool);
template void launch_plane<double>(const PlaneOp<double> &, const double *, double *, bool,
                                   hipStream_t, double *, const int *);

// Layers per workgroup.  More chunks keep the device full and its last round
// short; every chunk reads and adds one node plane more (about a third of a
// layer's time).  The estimate: rounds of the resident workgroups times the
// layers of one; within 3% of the best of 4 to 40 chunks on 80^3 cells, and on
// 32^3 cells 16 chunks (one round) instead of 32.
PlaneLayout plane_layout(int nq, const uint32_t n[3]) {
  constexpr double kResident = 2048.0;  // two waves per SIMD
  constexpr double kChunk = 0.35;       // a chunk's extra, in layers
  PlaneLayout lay;
  for (int k = 0; k < 3; ++k) lay.n[k] = n[k];
  const uint64_t layer = (uint64_t)n[0] * n[1];
  const uint32_t C = 64 / nq;
  lay.groups = (uint32_t)((layer + C - 1) / C);
  lay.chunks = 1;
  double best = 0.0;
  for (uint32_t c = 1; c <= n[2]; ++c) {
    const double depth = (double)((n[2] + c - 1) / c);
    double rounds = lay.groups * (double)c / kResident;
    rounds = rounds < 4.0 ? std::ceil(rounds) : rounds + 0.5;
    const double cost = rounds * (depth + kChunk);
    if (c == 1 || cost < best) {
      best = cost;
      lay.chunks = c;
    }
  }
  return lay;
}

}  // namespace mfx
