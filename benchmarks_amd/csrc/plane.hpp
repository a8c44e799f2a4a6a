// plane.hpp -- data of the plane-per-lane operator kernel of box meshes
// (plane_kernel.hpp).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mfx {

// A launch covers `groups` groups of consecutive cells of an xy layer of the
// mesh, each marched through `chunks` parts of the layers.
struct PlaneLayout {
  uint32_t n[3] = {0, 0, 0};
  uint32_t groups = 0, chunks = 0;
  uint32_t blocks() const { return groups * chunks; }  // workgroups, p.Ap partials
};
PlaneLayout plane_layout(int nq, const uint32_t n[3]);

template <typename T>
struct PlaneOp {
  int p = 0, nq = 0;
  bool colloc = false;            // Gauss-Lobatto points on the nodes, B = I
  bool axes = false;              // undeformed box: diagonal metric per cell
  PlaneLayout lay{};
  const T *eo = nullptr;          // even-odd tables of B, B^T, D, D^T (not colloc)
  const T *xq = nullptr, *wq = nullptr;
  const double *cellX = nullptr;  // [cells][8][3]
};

// whether the kernel has an instance for the operator's form
template <typename T>
bool plane_instance(int p, int nq, bool colloc, bool axes);
// dst += A src over the free rows; fresh: dst is zero on the free rows, so that
// sums only one wave forms may be stored instead of added
template <typename T>
void launch_plane(const PlaneOp<T> &o, const T *src, T *dst, bool fresh, hipStream_t s,
                  double *partials = nullptr, const int *skip = nullptr);

}  // namespace mfx
