// RK3 advection-diffusion kernels (src/equations.f90, src/time_integration.f90,
// src/mass_flow.f90) for gfx950, FP64.
//
// Each right-hand side is evaluated pointwise: the reference's whole-array
// passes through term_1/term_2 reduce, at every interior point, to the
// expressions below (same operands, same operation order, same order of
// accumulation: convective x, y, z, viscous, pressure gradient).  FMA
// contraction is disabled so the results round exactly as written.
#include <algorithm>
#include <cstdlib>

#include "bc_images.hpp"
#include "kernels.hpp"

#pragma clang fp contract(off)
#include "rk3_march.hpp"

namespace c3d {

namespace {

constexpr int kB = 256;

#define U_(i, j, k) U[fidx(i, j, k, g.nx, g.nyg)]
#define V_(i, j, k) V[fidx(i, j, k, g.nxg, g.ny)]
#define W_(i, j, k) W[fidx(i, j, k, g.nxg, g.nyg)]

// compute_rhs_u/v/w evaluated together.  Ranges: F_u (2:nx-1, 2:nyg-1,
// 2:nzg-1), F_v (2:nxg-1, 2:ny-1, 2:nzg-1), F_w (2:nxg-1, 2:nyg-1, 2:nz-1);
// the grid covers their union, walked plane by plane (rk3_march.hpp).
template <int KC>
__global__ __launch_bounds__(kB) void k_rhs(DevGrid g, const double* __restrict__ U,
                                            const double* __restrict__ V,
                                            const double* __restrict__ W,
                                            const double* __restrict__ Hu,
                                            const double* __restrict__ Hv,
                                            const double* __restrict__ Hw, double nu, double dPdx,
                                            double dPdy, double dPdz, double* __restrict__ Fu,
                                            double* __restrict__ Fv, double* __restrict__ Fw) {
  auto put = [](double* F, double v, int k, const Spot& s) { cell(F + (size_t)(k - 2) * s.pf, s.f) = v; };
  march<KC>(
      g, U, V, W, [](int, const Spot&, const Spot&, const Spot&) {},
      [&](const MarchAcc& A, const MarchGrid& G, int k, const Spot& su, const Spot& sv, const Spot& sw) {
        const int i = A.i, j = A.j;
        if (su.in) put(Fu, rhs_u_at<false>(G, A, Hu, nu, dPdx, i, j, k), k, su);
        if (sv.in) put(Fv, rhs_v_at<false>(G, A, Hv, nu, dPdy, i, j, k), k, sv);
        if (sw.in && k <= g.nz - 1) put(Fw, rhs_w_at<false>(G, A, Hw, nu, dPdz, i, j, k), k, sw);
      });
}

// RK3 stage update on the interior of one component
// (src/time_integration.f90:105-107, 134-136, 163-168).
__global__ __launch_bounds__(kB) void k_rk_update(int n1, int n2, int i1, int j1, int k1, int stage,
                                                  double dt, const double* __restrict__ F1,
                                                  const double* __restrict__ F2,
                                                  const double* __restrict__ F3,
                                                  const double* __restrict__ Xo,
                                                  double* __restrict__ X) {
#pragma clang fp contract(off)
  unsigned bx, by, bz;
  xcd_tile(bx, by, bz);  // neighbouring tiles on one XCD (shared halo rows)
  const int i = bx * 64 + (threadIdx.x & 63) + 2;
  const int j = by * 4 + (threadIdx.x >> 6) + 2;
  const int k = bz + 2;
  if (i > i1 || j > j1) return;
  const double c11 = 8.0 / 15.0, c21 = 1.0 / 4.0, c22 = 5.0 / 12.0, c31 = 1.0 / 4.0, c32 = 0.0,
               c33 = 3.0 / 4.0;
  const size_t f = (size_t)(i - 2) + (size_t)(i1 - 1) * ((size_t)(j - 2) + (size_t)(j1 - 1) * (size_t)(k - 2));
  const size_t o = fidx(i, j, k, n1, n2);
  double v;
  if (stage == 1) v = Xo[o] + dt * c11 * F1[f];
  else if (stage == 2) v = Xo[o] + dt * (c21 * F1[f] + c22 * F2[f]);
  else v = Xo[o] + dt * (c31 * F1[f] + c32 * F2[f] + c33 * F3[f]);
  X[o] = v;
  (void)k1;
}

// U(2:nx-1, 2:nyg-1, 2:nzg-1) += d  (src/time_integration.f90:190).
__global__ __launch_bounds__(kB) void k_add_u(DevGrid g, double* __restrict__ U, double d) {
  unsigned bx, by, bz;
  xcd_tile(bx, by, bz);  // neighbouring tiles on one XCD (shared halo rows)
  const int i = bx * 64 + (threadIdx.x & 63) + 2;
  const int j = by * 4 + (threadIdx.x >> 6) + 2;
  const int k = bz + 2;
  if (i > g.nx - 1 || j > g.nyg - 1) return;
  const size_t o = fidx(i, j, k, g.nx, g.nyg);
  U[o] = U[o] + d;
}

// The constant-flow correction (src/time_integration.f90:187-190) with U's
// boundary conditions: d = q0 - sums[0]/sums[1] from the flow integral on the
// device (no wait for the host in the middle of a step), added to the unique
// cells, each stored with its boundary images.
__global__ __launch_bounds__(kB) void k_hold_flow(DevGrid g, double* __restrict__ U,
                                                  const double* __restrict__ sums, double q0) {
  unsigned bx, by, bz;
  xcd_tile(bx, by, bz);
  const int i = bx * 64 + (threadIdx.x & 63) + 2;
  const int j = __builtin_amdgcn_readfirstlane((int)(by * 4 + (threadIdx.x >> 6) + 2));
  const int k = bz + 2;
  if (i > g.nx - 1 || j > g.nyg - 1) return;
  const double d = q0 - sums[0] / sums[1];
  put_u(g, U, i, j, k, U[fidx(i, j, k, g.nx, g.nyg)] + d);
}

// compute_dt maxima (src/time_integration.f90:228-239): max over the
// centre range of dx/|u| per component (+Inf where u = 0).  A workgroup takes
// 64 x positions, 4 rows and a run of planes, four planes' loads in flight at
// a time, and leaves one partial per component: an atomic per workgroup onto
// three words took most of the time of a small grid.
constexpr int kDtPlanes = 4;
__global__ __launch_bounds__(kB) void k_dt_max(DevGrid g, const double* __restrict__ U,
                                               const double* __restrict__ V,
                                               const double* __restrict__ W, int run,
                                               double* __restrict__ part) {
  __shared__ double sm[3][kB / 64];
  const int i = blockIdx.x * 64 + (threadIdx.x & 63) + 2;
  const int j = blockIdx.y * 4 + (threadIdx.x >> 6) + 2;
  double m[3] = {0.0, 0.0, 0.0};
  if (i <= g.nxg - 1 && j <= g.nyg - 1) {
    const int ka = blockIdx.z * run + 2, ke = min(ka + run - 1, g.nzg - 1);
    const double dx = g.dxg[i], dy = g.dyg[j];
    for (int k0 = ka; k0 <= ke; k0 += kDtPlanes) {
      double u[kDtPlanes], v[kDtPlanes], w[kDtPlanes];
#pragma unroll
      for (int r = 0; r < kDtPlanes; r++) {
        const int k = min(k0 + r, ke);  // past the run: its last plane again
        u[r] = U_(i, j, k);
        v[r] = V_(i, j, k);
        w[r] = W_(i, j, k);
      }
#pragma unroll
      for (int r = 0; r < kDtPlanes; r++) {
        m[0] = fmax(m[0], dx / fabs(u[r]));
        m[1] = fmax(m[1], dy / fabs(v[r]));
        m[2] = fmax(m[2], g.dzg[min(k0 + r, ke)] / fabs(w[r]));
      }
    }
  }
  for (int c = 0; c < 3; c++) {
    double v = m[c];
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
    if ((threadIdx.x & 63) == 0) sm[c][threadIdx.x >> 6] = v;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    double v = sm[threadIdx.x][0];
    for (int w = 1; w < kB / 64; w++) v = fmax(v, sm[threadIdx.x][w]);
    const size_t b = blockIdx.x + (size_t)gridDim.x * (blockIdx.y + (size_t)gridDim.y * blockIdx.z);
    part[3 * b + threadIdx.x] = v;
  }
}

constexpr int kDtFinal = 1024;
__global__ __launch_bounds__(kDtFinal) void k_dt_final(const double* __restrict__ part, int n,
                                                       double* host3) {
  __shared__ double sm[3][kDtFinal / 64];
  double m[3] = {0.0, 0.0, 0.0};
#pragma unroll 2
  for (int b = threadIdx.x; b < n; b += kDtFinal)
    for (int c = 0; c < 3; c++) m[c] = fmax(m[c], part[3 * (size_t)b + c]);
  for (int c = 0; c < 3; c++) {
    for (int off = 32; off > 0; off >>= 1) m[c] = fmax(m[c], __shfl_xor(m[c], off, 64));
    if ((threadIdx.x & 63) == 0) sm[c][threadIdx.x >> 6] = m[c];
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    double v = sm[threadIdx.x][0];
    for (int w = 1; w < kDtFinal / 64; w++) v = fmax(v, sm[threadIdx.x][w]);
    host3[threadIdx.x] = v;
  }
}

// Bulk-flow integral (src/mass_flow.f90:36-44): sums of (H U + H U(j-1))*dy/2
// and of its norm over i = 2..nx-1, j = 3..nyg-1, k = 2..nzg-1.  One wavefront
// per 64 x positions, z plane and chunk of kFlowJ rows, each row's loads in
// flight together and row j-1 reused: U is read once, in whole rows.  The
// chunks keep short channels from running on a few wavefronts.  Per
// workgroup one pair of partials, added in a fixed order.
constexpr int kFlowJ = 16;
template <bool MASK>
__global__ __launch_bounds__(kB) void k_massflow(DevGrid g, const double* __restrict__ U,
                                                 const double* __restrict__ H, int ni, int nj,
                                                 double* __restrict__ part) {
#pragma clang fp contract(off)
  __shared__ double ss[kB / 64], sn[kB / 64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int w = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (kB / 64)) + wv);
  const int i = (w % ni) * 64 + lane + 2;
  const int jc = (w / ni) % nj, k = w / (ni * nj) + 2;
  double s = 0.0, n = 0.0;
  if (k <= g.nzg - 1 && i <= g.nx - 1) {
    const int j0 = 3 + jc * kFlowJ;
    const size_t row = g.nx;
    const double* u = U + fidx(i, j0 - 1, k, g.nx, g.nyg);
    const double* h = MASK ? H + fidx(i, j0 - 1, k, g.nx, g.nyg) : nullptr;
    double um[kFlowJ + 1], hm[kFlowJ + 1];
#pragma unroll
    for (int r = 0; r <= kFlowJ; r++) {
      const int rr = min(r, g.nyg - j0);  // rows j0-1 .. nyg-1
      um[r] = u[rr * row];
      hm[r] = MASK ? h[rr * row] : 1.0;
    }
#pragma unroll
    for (int r = 1; r <= kFlowJ; r++) {
      const int j = j0 + r - 1;
      if (j <= g.nyg - 1) {
        s = s + (hm[r] * um[r] + hm[r - 1] * um[r - 1]) * 0.5 * g.dyg[j - 1];
        n = n + (hm[r] + hm[r - 1]) * 0.5 * g.dyg[j - 1];
      }
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    s += __shfl_xor(s, off, 64);
    n += __shfl_xor(n, off, 64);
  }
  if (lane == 0) {
    ss[wv] = s;
    sn[wv] = n;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int q = 1; q < kB / 64; q++) {
      s += ss[q];
      n += sn[q];
    }
    part[2 * (size_t)blockIdx.x] = s;
    part[2 * (size_t)blockIdx.x + 1] = n;
  }
}

// Ordered sum of the partials (single workgroup, fixed order) into out and
// host (host memory that the device writes).
constexpr int kSumB = 1024;
__global__ __launch_bounds__(kSumB) void k_sum_pairs(const double* __restrict__ part, int nrow,
                                                     double* __restrict__ out, double* host) {
  __shared__ double ss[kSumB], sn[kSumB];
  double s = 0.0, n = 0.0;
#pragma unroll 4
  for (int r = threadIdx.x; r < nrow; r += kSumB) {
    s += part[2 * (size_t)r];
    n += part[2 * (size_t)r + 1];
  }
  ss[threadIdx.x] = s;
  sn[threadIdx.x] = n;
  __syncthreads();
  for (int w = kSumB / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      ss[threadIdx.x] += ss[threadIdx.x + w];
      sn[threadIdx.x] += sn[threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = host[0] = ss[0];
    out[1] = host[1] = sn[0];
  }
}

// Plane sums of compute_statistics on one domain (src/statistics.f90:41-73,
// last-rank branch): one workgroup per row j = 1..nyg.  term_1 is the
// x-centred U (interpolate_x, src/interpolation.f90:21-36), term_2 the
// y-centred V (interpolate_y, :44-58) with term_2(:,1,:) = -term_2(:,2,:)
// and term_2(:,nyg,:) = -term_2(:,nyg-1,:) (src/statistics.f90:47-49).
// sums[q*nyg + j-1] for q = 0 U, 1 V, 2 W, 3 U^2, 4 V^2, 5 W^2, 6 UV over
// i = 2..nxg-2 and k = 2..nzg-2 (W, W^2: k = 2..nz-1); fixed-order sums.
constexpr int kStats = 7;

// The planes are split into chunks so that 1024 workgroups share them (one
// workgroup per row was 193 of them, 597 us on 384x192x384 cells); the chunks
// are added in order by k_plane_final, a single chunk holds the sums already.
// L: lanes per x row, so that short rows share a wavefront (16 and 32 cells in
// x: 800 rows 9.1 -> 6.9 us, 300 rows 9.5 -> 5.8 us).
template <int L>
__global__ __launch_bounds__(kB) void k_plane_sums(DevGrid g, const double* __restrict__ U,
                                                   const double* __restrict__ V,
                                                   const double* __restrict__ W, int run,
                                                   double* __restrict__ part) {
  __shared__ double sh[kStats][kB / 64];
  const int j = blockIdx.x + 1;
  const int nx = g.nx, ny = g.ny, nxg = g.nxg, nyg = g.nyg;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  // term_2 at row j from V rows jv - 1, jv with sign sg (the wall rows mirror)
  const int jv = (j == 1) ? 2 : ((j == nyg) ? nyg - 1 : j);
  const double sg = (j == 1 || j == nyg) ? -1.0 : 1.0;
  double a[kStats] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  // U, V: k = 2..nzg-2; W: k = 2..nz-1, the same range (nzg = nz + 1)
  const int ka = blockIdx.y * run + 2, ke = min(ka + run - 1, g.nzg - 2);
  for (int k = ka + (L == 64 ? wv : (int)threadIdx.x / L); k <= ke; k += kB / L) {
    const double* u = U + fidx(1, j, k, nx, nyg);
    const double* v = V + fidx(1, jv, k, nxg, ny);
    const double* w = W + fidx(1, j, k, nxg, nyg);
#pragma unroll 2
    for (int i = 1 + lane % L; i <= nxg - 3; i += L) {  // offset of x index i + 1
      const double t1 = 0.5 * (u[i - 1] + u[i]);
      const double t2 = sg * (0.5 * (v[i - nxg] + v[i]));
      const double t3 = w[i];
      a[0] += t1;
      a[1] += t2;
      a[2] += t3;
      a[3] += t1 * t1;
      a[4] += t2 * t2;
      a[5] += t3 * t3;
      a[6] += t1 * t2;
    }
  }
#pragma unroll
  for (int q = 0; q < kStats; q++) {
    for (int off = 32; off > 0; off >>= 1) a[q] += __shfl_xor(a[q], off, 64);
    if (lane == 0) sh[q][wv] = a[q];
  }
  __syncthreads();
  if (threadIdx.x < kStats) {
    const double* t = sh[threadIdx.x];
    part[((size_t)blockIdx.y * kStats + threadIdx.x) * nyg + j - 1] = (t[0] + t[1]) + (t[2] + t[3]);
  }
}

__global__ __launch_bounds__(kB) void k_plane_final(const double* __restrict__ part, int n, int chunks,
                                                    double* __restrict__ sums) {
  const int e = blockIdx.x * kB + threadIdx.x;
  if (e >= n) return;
  double s = 0.0;
#pragma unroll 4
  for (int c = 0; c < chunks; c++) s += part[(size_t)c * n + e];
  sums[e] = s;
}

// output_monitor's field summaries (src/monitor.f90:27-47): per workgroup
// the sums and maxima of U(2:nx-1,2:nyg-1,2:nzg-1), V(2:nxg-1,2:ny-1,2:nzg-1)
// and W(2:nxg-1,2:nyg-1,2:nz-1), and the count of non-finite entries of the
// three (a NaN guard), into part[b*kMon + q]; k_monitor_final reduces the
// partials, up to kMonBlocks, in a fixed order.
constexpr int kMon = 7;  // sum U, V, W; max U, V, W; non-finite count
constexpr int kMonBlocks = 1024;

// Lanes per x row of the field summaries: rows of up to 64 share a unit.
inline int mon_lanes(long long ni) { return ni <= 16 ? 16 : (ni <= 32 ? 32 : (ni <= 64 ? 64 : 256)); }

// Interior (2..i1, 2..j1, 2..k1) of an (n1, n2, *) array: a wavefront takes
// units of four loads per lane, 256 x positions of a row (L = 256) or, of rows
// of up to L positions, 256 / L rows of a plane, so the index arithmetic is
// scalar (a division per element made this 838 us on 384x192x384 cells; a row
// per unit whatever its length 15.9 us on 16x799x16 cells, now 8.0).
template <int L>
__device__ __forceinline__ void mon_field(const double* __restrict__ F, int n1, int n2, int i1, int j1,
                                          int k1, double& sum, double& mx, double& bad) {
  constexpr int R = 256 / L;  // rows of a unit
  const int lane = threadIdx.x & 63;
  const long long ni = i1 - 1, nj = j1 - 1, nseg = (ni + L - 1) / L, nu = (nj + R - 1) / R;
  const long long n = nseg * nu * (k1 - 1);
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  for (long long t = (long long)blockIdx.x * (kB / 64) + wv; t < n; t += gridDim.x * (kB / 64)) {
    const long long r = R == 1 ? t / nseg : t, i0 = R == 1 ? (t - r * nseg) * L : 0;
    const long long k = r / nu, j0 = (r - k * nu) * R;
    const double* row = F + 1 + (size_t)n1 * ((size_t)(j0 + 1) + (size_t)n2 * (size_t)(k + 1)) + i0;
    auto at = [&](int q, bool& in) {  // the lane's q-th element of the unit
      const int e = q * 64 + lane, i = e % L, j = e / L;
      in = i0 + i < ni && (R == 1 || j0 + j < nj);
      return (size_t)j * n1 + i;
    };
    double v[4];
    bool in[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const size_t o = at(q, in[q]);
      if (in[q]) v[q] = row[o];
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
      if (in[q]) {
        sum += v[q];
        mx = fmax(mx, v[q]);
        bad += isfinite(v[q]) ? 0.0 : 1.0;
      }
  }
}

template <int L>
__global__ __launch_bounds__(kB) void k_monitor_part(DevGrid g, const double* __restrict__ U,
                                                     const double* __restrict__ V,
                                                     const double* __restrict__ W,
                                                     double* __restrict__ part) {
  __shared__ double sh[kMon][kB];
  double a[kMon] = {0.0, 0.0, 0.0, -INFINITY, -INFINITY, -INFINITY, 0.0};
  mon_field<L>(U, g.nx, g.nyg, g.nx - 1, g.nyg - 1, g.nzg - 1, a[0], a[3], a[6]);
  mon_field<L>(V, g.nxg, g.ny, g.nxg - 1, g.ny - 1, g.nzg - 1, a[1], a[4], a[6]);
  mon_field<L>(W, g.nxg, g.nyg, g.nxg - 1, g.nyg - 1, g.nz - 1, a[2], a[5], a[6]);
#pragma unroll
  for (int q = 0; q < kMon; q++) sh[q][threadIdx.x] = a[q];
  __syncthreads();
  for (int w = kB / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
#pragma unroll
      for (int q = 0; q < kMon; q++)
        sh[q][threadIdx.x] = (q >= 3 && q < 6) ? fmax(sh[q][threadIdx.x], sh[q][threadIdx.x + w])
                                                : sh[q][threadIdx.x] + sh[q][threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x < kMon) part[(size_t)blockIdx.x * kMon + threadIdx.x] = sh[threadIdx.x][0];
}

__global__ __launch_bounds__(kB) void k_monitor_final(const double* __restrict__ part, int n,
                                                      double* __restrict__ out) {
  __shared__ double sh[kMon][kB];
#pragma unroll
  for (int q = 0; q < kMon; q++) {
    const double none = (q >= 3 && q < 6) ? -INFINITY : 0.0;
    double a = none;
#pragma unroll
    for (int r = 0; r < kMonBlocks / kB; r++) {
      const int b = threadIdx.x + r * kB;
      const double v = b < n ? part[(size_t)b * kMon + q] : none;
      a = (q >= 3 && q < 6) ? fmax(a, v) : a + v;
    }
    sh[q][threadIdx.x] = a;
  }
  __syncthreads();
  for (int w = kB / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
#pragma unroll
      for (int q = 0; q < kMon; q++)
        sh[q][threadIdx.x] = (q >= 3 && q < 6) ? fmax(sh[q][threadIdx.x], sh[q][threadIdx.x + w])
                                                : sh[q][threadIdx.x] + sh[q][threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x < kMon) out[threadIdx.x] = sh[threadIdx.x][0];
}

inline dim3 gpts(int ni, int nj, int nk) { return dim3((ni + 63) / 64, (nj + 3) / 4, nk); }

}  // namespace

// Eight planes (1.25 loaded per plane) where that leaves 4 workgroups for each
// of the 256 CUs, else four or two, so that a small grid is not a few long
// chains of planes.  C3D_RHS_KC (2, 4, 8) overrides it (tuning knob).
int rhs_planes(const DevGrid& g) {
  static const int forced = [] {
    const char* e = getenv("C3D_RHS_KC");
    const int v = e ? atoi(e) : 0;
    return (v == 2 || v == 4 || v == 8) ? v : 0;
  }();
  if (forced) return forced;
  const long long cols = (long long)((g.nxg - 2 + 63) / 64) * ((g.nyg - 2 + 3) / 4);
  int kc = 8;
  while (kc > 2 && cols * ((g.nzg - 2 + kc - 1) / kc) < 1024) kc /= 2;
  return kc;
}

hipError_t launch_rhs(const DevGrid& g, const double* U, const double* V, const double* W,
                      const double* Hu, const double* Hv, const double* Hw, double nu, double dPdx,
                      double dPdy, double dPdz, double* Fu, double* Fv, double* Fw, hipStream_t s) {
  const int kc = rhs_planes(g);
  const dim3 grid = gpts(g.nxg - 2, g.nyg - 2, (g.nzg - 2 + kc - 1) / kc);
  switch (kc) {
    case 2: hipLaunchKernelGGL(k_rhs<2>, grid, dim3(kB), 0, s, g, U, V, W, Hu, Hv, Hw, nu, dPdx, dPdy, dPdz, Fu, Fv, Fw); break;
    case 4: hipLaunchKernelGGL(k_rhs<4>, grid, dim3(kB), 0, s, g, U, V, W, Hu, Hv, Hw, nu, dPdx, dPdy, dPdz, Fu, Fv, Fw); break;
    default: hipLaunchKernelGGL(k_rhs<8>, grid, dim3(kB), 0, s, g, U, V, W, Hu, Hv, Hw, nu, dPdx, dPdy, dPdz, Fu, Fv, Fw); break;
  }
  return hipGetLastError();
}

hipError_t launch_rk_update(const DevGrid& g, int which, int stage, double dt, const double* F1,
                            const double* F2, const double* F3, const double* Xo, double* X,
                            hipStream_t s) {
  int n1, n2, i1, j1, k1;
  if (which == 0) { n1 = g.nx; n2 = g.nyg; i1 = g.nx - 1; j1 = g.nyg - 1; k1 = g.nzg - 1; }
  else if (which == 1) { n1 = g.nxg; n2 = g.ny; i1 = g.nxg - 1; j1 = g.ny - 1; k1 = g.nzg - 1; }
  else { n1 = g.nxg; n2 = g.nyg; i1 = g.nxg - 1; j1 = g.nyg - 1; k1 = g.nz - 1; }
  hipLaunchKernelGGL(k_rk_update, gpts(i1 - 1, j1 - 1, k1 - 1), dim3(kB), 0, s, n1, n2, i1, j1, k1,
                     stage, dt, F1, F2, F3, Xo, X);
  return hipGetLastError();
}

hipError_t launch_add_u(const DevGrid& g, double* U, double d, hipStream_t s) {
  hipLaunchKernelGGL(k_add_u, gpts(g.nx - 2, g.nyg - 2, g.nzg - 2), dim3(kB), 0, s, g, U, d);
  return hipGetLastError();
}

hipError_t launch_hold_flow(const DevGrid& g, double* U, const double* sums, double q0, hipStream_t s) {
  hipLaunchKernelGGL(k_hold_flow, gpts(g.nx - 2, g.nyg - 2, g.nz - 2), dim3(kB), 0, s, g, U, sums, q0);
  return hipGetLastError();
}

// Runs of planes per workgroup: about 2048 workgroups (8 per CU), at least
// kDtPlanes planes each.
static int dt_run(const DevGrid& g) {
  const int cols = ((g.nxg - 2 + 63) / 64) * ((g.nyg - 2 + 3) / 4), nk = g.nzg - 2;
  const int runs = std::max(1, std::min((2048 + cols - 1) / cols, nk / kDtPlanes));
  return (nk + runs - 1) / runs;
}
static dim3 dt_grid(const DevGrid& g) {
  const int run = dt_run(g);
  return gpts(g.nxg - 2, g.nyg - 2, (g.nzg - 2 + run - 1) / run);
}
int dt_parts(const DevGrid& g) {
  const dim3 n = dt_grid(g);
  return (int)(n.x * n.y * n.z);
}

hipError_t launch_dt_max(const DevGrid& g, const double* U, const double* V, const double* W,
                         double* part, double* host3, hipStream_t s) {
  hipLaunchKernelGGL(k_dt_max, dt_grid(g), dim3(kB), 0, s, g, U, V, W, dt_run(g), part);
  hipLaunchKernelGGL(k_dt_final, dim3(1), dim3(kDtFinal), 0, s, (const double*)part, dt_parts(g), host3);
  return hipGetLastError();
}

// Wavefronts of the flow integral: x tiles, row chunks, z planes.
static int flow_ni(const DevGrid& g) { return (g.nx - 2 + 63) / 64; }
static int flow_nj(const DevGrid& g) { return (g.nyg - 3 + kFlowJ - 1) / kFlowJ; }
int massflow_parts(const DevGrid& g) {
  return (flow_ni(g) * flow_nj(g) * (g.nzg - 2) + kB / 64 - 1) / (kB / 64);
}

int monitor_part_size() { return kMonBlocks * kMon; }
static_assert(kMonBlocks * kMon == kMonitorPartDoubles, "partials of the monitor kernels");

namespace {
// c3d_monitor's results from the reduced sums r7 (sums U, V, W; maxima U, V,
// W; non-finite count): maxima, sums / vol, count.
__global__ void k_monitor_finish(const double* __restrict__ r7, double vol, double* __restrict__ out) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  out[0] = r7[3];
  out[1] = r7[4];
  out[2] = r7[5];
  out[3] = r7[0] / vol;
  out[4] = r7[1] / vol;
  out[5] = r7[2] / vol;
  out[6] = r7[6];
}
}  // namespace

hipError_t launch_monitor_finish(const double* r7, double vol, double* out, hipStream_t s) {
  hipLaunchKernelGGL(k_monitor_finish, dim3(1), dim3(64), 0, s, r7, vol, out);
  return hipGetLastError();
}

hipError_t launch_monitor(const DevGrid& g, const double* U, const double* V, const double* W,
                          double* part, double* out7, hipStream_t s) {
  // a unit per wavefront, up to kMonBlocks workgroups: fewer partials of a
  // small grid (18x4x18: final 5.6 -> 2.3 us)
  const long long ni = g.nxg - 2;
  const int lanes = mon_lanes(ni), rows = 256 / lanes;
  const long long units = (ni + lanes - 1) / lanes * ((g.nyg - 2 + rows - 1) / rows) * (g.nzg - 2);
  const int n = (int)std::min<long long>((units + kB / 64 - 1) / (kB / 64), kMonBlocks);
  switch (lanes) {
    case 16: hipLaunchKernelGGL(k_monitor_part<16>, dim3(n), dim3(kB), 0, s, g, U, V, W, part); break;
    case 32: hipLaunchKernelGGL(k_monitor_part<32>, dim3(n), dim3(kB), 0, s, g, U, V, W, part); break;
    case 64: hipLaunchKernelGGL(k_monitor_part<64>, dim3(n), dim3(kB), 0, s, g, U, V, W, part); break;
    default: hipLaunchKernelGGL(k_monitor_part<256>, dim3(n), dim3(kB), 0, s, g, U, V, W, part); break;
  }
  hipLaunchKernelGGL(k_monitor_final, dim3(1), dim3(kB), 0, s, (const double*)part, n, out7);
  return hipGetLastError();
}

// Lanes per x row of the plane sums, and planes per chunk: about 1024
// workgroups, but chunks of at least eight rounds of a workgroup's loads, so
// that small grids need no second launch (32x299x32 cells: the call 34.4 -> 31.1 us).
static int stat_lanes(const DevGrid& g) { return g.nxg - 3 <= 16 ? 16 : (g.nxg - 3 <= 32 ? 32 : 64); }
static int stat_run(const DevGrid& g) {
  const int lanes = stat_lanes(g), once = kB / lanes, nk = g.nzg - 3;
  const int rounds = (nk + once - 1) / once * ((g.nxg - 3 + lanes - 1) / lanes);
  const int chunks = std::max(1, std::min(1024 / g.nyg, rounds / 8));
  return (nk + chunks - 1) / chunks;
}
static int stat_chunks(const DevGrid& g) { return (g.nzg - 3 + stat_run(g) - 1) / stat_run(g); }
size_t plane_sums_part_size(const DevGrid& g) { return (size_t)stat_chunks(g) * kStats * g.nyg; }

hipError_t launch_plane_sums(const DevGrid& g, const double* U, const double* V, const double* W,
                             double* part, double* sums, hipStream_t s) {
  const int n = kStats * g.nyg, c = stat_chunks(g);
  double* out = c == 1 ? sums : part;
  switch (stat_lanes(g)) {
    case 16: hipLaunchKernelGGL(k_plane_sums<16>, dim3(g.nyg, c), dim3(kB), 0, s, g, U, V, W, stat_run(g), out); break;
    case 32: hipLaunchKernelGGL(k_plane_sums<32>, dim3(g.nyg, c), dim3(kB), 0, s, g, U, V, W, stat_run(g), out); break;
    default: hipLaunchKernelGGL(k_plane_sums<64>, dim3(g.nyg, c), dim3(kB), 0, s, g, U, V, W, stat_run(g), out); break;
  }
  if (c > 1)
    hipLaunchKernelGGL(k_plane_final, dim3((n + kB - 1) / kB), dim3(kB), 0, s, (const double*)part, n, c,
                       sums);
  return hipGetLastError();
}

hipError_t launch_massflow(const DevGrid& g, const double* U, const double* H, double* part,
                           double* out2, double* host2, hipStream_t s) {
  const int n = massflow_parts(g), ni = flow_ni(g), nj = flow_nj(g);
  if (H) hipLaunchKernelGGL(k_massflow<true>, dim3(n), dim3(kB), 0, s, g, U, H, ni, nj, part);
  else hipLaunchKernelGGL(k_massflow<false>, dim3(n), dim3(kB), 0, s, g, U, H, ni, nj, part);
  hipLaunchKernelGGL(k_sum_pairs, dim3(1), dim3(kSumB), 0, s, part, n, out2, host2);
  return hipGetLastError();
}

}  // namespace c3d
