// Boundary images of the staggered fields (apply_boundary_conditions,
// src/boundary_conditions.f90:20-252, one domain), written by the thread that
// computes an interior value.
//
// Applied in the reference's order (periodic x, periodic z, walls in y),
// every boundary value ends as a copy of an interior value: the periodic
// image in x and z (x faces 1 <- nx-1, nx <- 2; x centres 1 <- nxg-2,
// nxg-1 <- 2, nxg <- 3; z alike) and, in the y ghost rows of U and W, the
// negated value of the first interior row; V's wall rows are 0.  Seen from
// the interior value (unique cells i = 2..nx-1, j, k = 2..nz-1; nx, nz >= 18)
// there is at most one image per direction, and the boundary cells are
// exactly the products of those images.  So a kernel that writes every
// interior value can write the boundary with it: no pass over the fields of
// its own, and the x images, one element per row, go to cache lines that the
// row's wave is writing anyway.
#pragma once

#include "kernels.hpp"

namespace c3d {

// Image index of interior index i (0: none) on faces (n of them) and centres
// (ng of them) of a periodic direction.
__device__ __forceinline__ int face_image(int i, int n) { return i == 2 ? n : (i == n - 1 ? 1 : 0); }
__device__ __forceinline__ int ctr_image(int i, int ng) {
  return i == 2 ? ng - 1 : (i == 3 ? ng : (i == ng - 2 ? 1 : 0));
}

// F(i, j, k) = v and its images: i2, k2 in x and z, and the ghost row j2
// (0: none) with value vy.
__device__ __forceinline__ void put_images(double* __restrict__ F, int n1, int n2, int i, int j, int k,
                                           int i2, int j2, int k2, double v, double vy) {
  F[fidx(i, j, k, n1, n2)] = v;
  if (i2) F[fidx(i2, j, k, n1, n2)] = v;
  if (j2) {
    F[fidx(i, j2, k, n1, n2)] = vy;
    if (i2) F[fidx(i2, j2, k, n1, n2)] = vy;
  }
  if (k2) {
    F[fidx(i, j, k2, n1, n2)] = v;
    if (i2) F[fidx(i2, j, k2, n1, n2)] = v;
    if (j2) {
      F[fidx(i, j2, k2, n1, n2)] = vy;
      if (i2) F[fidx(i2, j2, k2, n1, n2)] = vy;
    }
  }
}

// U(nx, nyg, nzg), V(nxg, ny, nzg) and W(nxg, nyg, nz) at interior (i, j, k).
__device__ __forceinline__ void put_u(const DevGrid& g, double* __restrict__ U, int i, int j, int k,
                                      double u) {
  const int j2 = j == 2 ? 1 : (j == g.nyg - 1 ? g.nyg : 0);
  put_images(U, g.nx, g.nyg, i, j, k, face_image(i, g.nx), j2, ctr_image(k, g.nzg), u, -u);
}
// j = 2..ny-1; the threads next to a wall also write its zero row.
__device__ __forceinline__ void put_v(const DevGrid& g, double* __restrict__ V, int i, int j, int k,
                                      double v) {
  const int i2 = ctr_image(i, g.nxg), k2 = ctr_image(k, g.nzg);
  put_images(V, g.nxg, g.ny, i, j, k, i2, j == 2 ? 1 : 0, k2, v, 0.0);
  if (j == g.ny - 1) put_images(V, g.nxg, g.ny, i, g.ny, k, i2, 0, k2, 0.0, 0.0);
}
__device__ __forceinline__ void put_w(const DevGrid& g, double* __restrict__ W, int i, int j, int k,
                                      double w) {
  const int j2 = j == 2 ? 1 : (j == g.nyg - 1 ? g.nyg : 0);
  put_images(W, g.nxg, g.nyg, i, j, k, ctr_image(i, g.nxg), j2, face_image(k, g.nz), w, -w);
}

}  // namespace c3d
