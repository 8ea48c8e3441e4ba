// Immersed-boundary kernels for gfx950: stencil set-up, interpolation,
// spreading, Schur-complement pieces and BiCGSTAB vector steps.
//
// Interpolation runs one wavefront per marker: the 125 stencil points are
// spread over the 64 lanes and reduced with a fixed butterfly, so results are
// deterministic.  Spreading is a gather over a node -> entry map built once
// per static body, summing each node's contributions in ascending marker
// order (the order of the reference's serial scatter), with no atomics.
#include <hip/hip_runtime.h>

#include "bc_images.hpp"
#include "ib.hpp"

#pragma clang fp contract(off)

namespace c3d {
namespace ib {

namespace {

constexpr int kBlock = 256;

// deltafnc, src/immersed_boundary_operators.f90:270-294.
__device__ double deltafnc(double r, double dr) {
  const double pi = 4.0 * atan(1.0);
  const double s3 = sqrt(3.0);
  const double r1 = fabs(r) / dr;
  const double r2 = r1 * r1;
  double d;
  if (r1 <= 1.0) {
    d = 17.0 / 48.0 + s3 * pi / 108.0 + r1 / 4.0 - r2 / 4.0 +
        (1.0 - 2.0 * r1) / 16.0 * sqrt(-12.0 * r2 + 12.0 * r1 + 1.0) -
        s3 / 12.0 * asin(s3 / 2.0 * (2.0 * r1 - 1.0));
  } else if (r1 <= 2.0) {
    d = 55.0 / 48.0 - s3 * pi / 108.0 - 13.0 * r1 / 12.0 + r2 / 4.0 +
        (2.0 * r1 - 3.0) / 48.0 * sqrt(-12.0 * r2 + 36.0 * r1 - 23.0) +
        s3 / 36.0 * asin(s3 / 2.0 * (2.0 * r1 - 3.0));
  } else {
    d = 0.0;
  }
  return d / dr;
}

__device__ __forceinline__ int floor_div(int a, int b) {
  return (int)floor((double)a / (double)b);
}

// A wavefront's stencil entries v[15] (axis, position) to `out` (the common
// array of all markers): through LDS, so that 64 markers leave as whole lines
// instead of one line per lane and entry.
constexpr int kSetupMarkers = 64, kSetupPitch = kStencils + 1;
template <typename T>
__device__ __forceinline__ void store_stencils(T* __restrict__ out, const T v[kStencil], T* buf, int s,
                                               int lane, int l0, int nb) {
  __syncthreads();  // the buffer's last user is done
#pragma unroll
  for (int e = 0; e < kStencil; e++) buf[lane * kSetupPitch + s * kStencil + e] = v[e];
  __syncthreads();
  const int n = min(kSetupMarkers, nb - l0) * kStencils;
  for (int e = threadIdx.x; e < n; e += kBlock)
    out[(size_t)l0 * kStencils + e] = buf[e / kStencils * kSetupPitch + e % kStencils];
}

// 64 markers per workgroup, one stencil per wavefront (uniform branches):
// pivots (src/immersed_boundary_operators.f90:28-42) and the per-axis windows
// of the u (:46-98), v (:101-148), w (:151-194) and centre (:197-244) stencils
// on one periodic domain, centre z index nzg-1 stored as its canonical plane 2.
// 24,576 markers: 24 us, 43 us with a lane per (marker, stencil) and its stores
// as they come.
static_assert(kBlock == 4 * kSetupMarkers, "a wavefront per stencil");
__global__ __launch_bounds__(kBlock) void k_setup(DevGrid g, SetupGrid sg, Markers m, int* bad) {
  __shared__ double buf[kSetupMarkers * kSetupPitch];
  const int nb = m.nb;
  const int lane = threadIdx.x & 63, l0 = blockIdx.x * kSetupMarkers;
  const int s = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const bool on = l0 + lane < nb;
  const int l = on ? l0 + lane : nb - 1;  // lanes past the end repeat the last marker
  const int nx = g.nx, nz = g.nz, nzg = g.nzg;
  const double dx = sg.dx, dz = sg.dz, dymin = sg.dymin;
  const double xb = m.xb[l], yb = m.yb[l], zb = m.zb[l];
  const double* x = sg.x;
  const double* y = sg.y;
  const double* z = sg.z;
  const int x_piv = (int)floor(xb / dx) + 1;
  const int xm_piv = (int)floor((xb + 0.5 * dx) / dx);
  const int yr = m.yref ? m.yref[l] : 1;
  const int y_piv = (int)floor((yb - y[yr - 1]) / dymin) + yr;
  const int ym_piv = (int)floor((yb - (y[yr - 1] + 0.5 * dymin)) / dymin) + yr;
  const int ylim = (s == 1) ? g.ny - 1 : g.nyg - 1;
  const int z_piv = (int)floor(zb / dz) + 1;
  const int zm_piv = (int)floor((zb + 0.5 * dz) / dz) + 1;
  int idx[kStencil];
  double dd[kStencil], phi[kStencil];
#pragma unroll
  for (int t = 0; t < 5; t++) {
    const int o = t - 2;
    // x
    int X;
    double xgd;
    if (s == 0) {
      const int ii = x_piv + o;
      const int xs = floor_div(ii - 1, nx - 2);
      const int iip = ii - xs * (nx - 2);
      X = (iip == 1) ? nx - 1 : iip;
      xgd = x[iip - 1] + xs * sg.Lxp;
    } else {
      const int ii = xm_piv + o - (s == 2 ? 1 : 0);
      const int xs = floor_div(ii - 1, nx - 2);
      const int iip = ii - xs * (nx - 2);
      X = iip + 1;
      xgd = 0.5 * (x[iip - 1] + x[iip]) + xs * sg.Lxp;
    }
    // y (a window reaching past the walls is flagged with Y = -1 and
    // rejected by the host before any other IB kernel runs)
    int Y = -1;
    double ygd = 0.0;
    if (s == 1) {
      const int jj = y_piv + o;
      if (jj >= 1 && jj <= g.ny) {
        Y = jj;
        ygd = y[jj - 1];
      }
    } else {
      const int jj = ym_piv + o;
      if (jj >= 1 && jj <= g.ny - 1) {
        Y = jj + 1;
        ygd = 0.5 * (y[jj - 1] + y[jj]);
      }
    }
    // z
    int Z;
    double zgd;
    if (s == 2) {
      const int kk = z_piv + o;
      const int zs = floor_div(kk - 2, nz - 2);
      const int kkp = kk - zs * (nz - 2);
      Z = kkp;
      zgd = z[kkp - 1] + zs * sg.Lzp;
    } else {
      const int kk = zm_piv + o;
      const int zs = floor_div(kk - 2, nz - 1);
      const int kkp = kk - zs * (nz - 2);
      Z = (kkp == nzg - 1) ? 2 : kkp;
      zgd = 0.5 * (z[kkp - 2] + z[kkp - 1]) + zs * sg.Lzp;
    }
    const double ddx = xgd - xb, ddy = ygd - yb, ddz = zgd - zb;
    if (on && bad && (X < 2 || X > nx - 1 || Z < 2 || Z > nz - 1 || Y < 2 || Y > ylim))
      atomicMax(bad, l + 1);
    idx[t] = X;
    idx[5 + t] = Y;
    idx[10 + t] = Z;
    dd[t] = ddx;
    dd[5 + t] = ddy;
    dd[10 + t] = ddz;
    phi[t] = deltafnc(ddx, dx);
    phi[5 + t] = deltafnc(ddy, dymin);
    phi[10 + t] = deltafnc(ddz, dz);
  }
  store_stencils(m.st[0].dd, dd, buf, s, lane, l0, nb);
  store_stencils(m.st[0].phi, phi, buf, s, lane, l0, nb);
  store_stencils(m.st[0].idx, idx, reinterpret_cast<int*>(buf), s, lane, l0, nb);
}

__global__ void k_mark_planes(Markers m, int* live) {
  const int tid = blockIdx.x * blockDim.x + threadIdx.x;
  const int nb = m.nb;
  if (tid >= 20 * nb) return;
  const int l = tid / 20, e = tid - 20 * l, s = e / 5;
  const int jj = m.st[s].idx[sidx(1, e - 5 * s, l)] - 2;
  // every writer stores the same value; a set plane is not stored again
  if (!live[jj]) live[jj] = 1;
  if (s == 1 && !live[jj + 1]) live[jj + 1] = 1;
}

// Wall height of marker i (1-based, x-periodic) of one wall at the time wt
// (src/immersed_boundary_geometry.f90:186-191 standing, :295-299 traveling),
// and x itself.  The standing wave's top wall returns the bottom wall's
// curve: its areas are copied from the bottom wall (:264).
__device__ __forceinline__ void wall_point(const WaveBody& w, const WaveTime& wt, int i, bool top,
                                           double& x, double& y) {
  const double dxb = w.Lxp / (double)w.nxb;
  x = ((double)i - 0.5) * dxb;
  if (w.body == 1) {
    y = w.p1 * sin(2.0 * w.pi * w.p3 * x / w.Lxp) * wt.ct;
  } else {
    const double phase = w.p3 * (x - w.p2 * wt.t);
    y = wt.amp / (w.p2 * w.p3) * sin(top ? phase + w.pi : phase);
  }
}

// One thread per marker: position, velocity, normal, area and y_ref_index of
// the moving walls; the area sb = dzb (a1/2 + a2/2) from the chords to the
// x-periodic neighbours on the same wall (:234-262, :346-378).
__global__ void k_wave_geometry(WaveBody w, WaveTime wt, double* __restrict__ xb,
                                double* __restrict__ yb, double* __restrict__ zb,
                                double* __restrict__ normals, double* __restrict__ sb,
                                double* __restrict__ ub, int* __restrict__ yref, int* bad) {
  const int nxb = w.nxb, nb = 2 * nxb * w.nzb;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nb) return;
  const int j = k / (2 * nxb) + 1, r = k - (j - 1) * 2 * nxb;
  const bool top = r >= nxb;
  const int i = (top ? r - nxb : r) + 1;
  const double dzb = w.Lzp / (double)w.nzb;
  // own point, and the curve the neighbours' chords are measured on
  const bool curve_top = top && w.body == 2;
  double x, yc;
  wall_point(w, wt, i, curve_top, x, yc);
  const double y = top ? w.Lyc + yc : yc;
  double s, vy;
  if (w.body == 1) {
    const double phase = 2.0 * w.pi * w.p3 * x / w.Lxp;
    vy = -(w.p1 * w.p2 * sin(phase) * wt.st);
    s = w.p1 * 2.0 * w.pi * w.p3 / w.Lxp * cos(phase) * wt.ct;
  } else {
    const double phase = w.p3 * (x - w.p2 * wt.t);
    const double ph = top ? phase + w.pi : phase;
    vy = -wt.amp * cos(ph) + (wt.damp / (w.p2 * w.p3)) * sin(ph);
    s = wt.amp / w.p2 * cos(ph);
  }
  const double t1 = 1.0 / sqrt(1.0 + s * s), t2 = s / sqrt(1.0 + s * s);
  // chords on the curve (the top wall of a traveling wave on its own curve)
  double xp, yp, xn, yn;
  wall_point(w, wt, i == 1 ? nxb : i - 1, curve_top, xp, yp);
  wall_point(w, wt, i == nxb ? 1 : i + 1, curve_top, xn, yn);
  const double ys = curve_top ? w.Lyc + yc : yc;
  if (curve_top) {
    yp = w.Lyc + yp;
    yn = w.Lyc + yn;
  }
  if (i == 1) xp = xp - w.Lxp;
  if (i == nxb) xn = xn + w.Lxp;
  const double a1 = sqrt((x - xp) * (x - xp) + (ys - yp) * (ys - yp));
  const double a2 = sqrt((x - xn) * (x - xn) + (ys - yn) * (ys - yn));
  xb[k] = x;
  yb[k] = y;
  zb[k] = ((double)j - 0.5) * dzb;
  sb[k] = dzb * (0.5 * a1 + 0.5 * a2);
  yref[k] = top ? w.ny : 1;
  normals[k] = top ? -t2 : t2;
  normals[nb + k] = top ? t1 : -t1;
  normals[2 * nb + k] = 0.0;
  ub[k] = 0.0;
  ub[nb + k] = vy;
  ub[2 * nb + k] = 0.0;
  if (top ? (y > w.yhi) : (y < w.ylo)) atomicMax(bad, k + 1);
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Sum over the 32 lanes of each half of the wavefront: lane pairs, quads and
// rows of 16 through DPP, the two rows by a cross-lane read.
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xf, 0xf, false);
  const unsigned hi =
      (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, false);
  return v + __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ double half_sum(double v) {
  v = dpp_add<0xB1>(v);   // quad_perm 1,0,3,2
  v = dpp_add<0x4E>(v);   // quad_perm 2,3,0,1
  v = dpp_add<0x141>(v);  // mirrored within 8 (the quads' sums are equal there)
  v = dpp_add<0x140>(v);  // mirrored within 16
  return v + __shfl_xor(v, 16, 64);
}

// The stencil tables and normals as arguments of their own: read-only for the
// whole kernel, so that wave-uniform reads become scalar loads.
#define C3D_STENCIL_ARGS                                                           \
  const int *__restrict__ idx, const double *__restrict__ phi, const double *__restrict__ dd, \
      const double *__restrict__ normals
#define C3D_STENCIL(m) m.st[0].idx, m.st[0].phi, m.st[0].dd, m.normals

// Marker handled by this wavefront (XCD-aware: neighbouring markers, whose
// stencils share nodes, run on the same XCD and L2).
__device__ __forceinline__ int wave_marker(int nb) {
  unsigned bx, by, bz;
  xcd_tile(bx, by, bz);
  return __builtin_amdgcn_readfirstlane((int)bx * (kBlock / 64) + (int)(threadIdx.x >> 6));
}

// Stencil sums of marker l over field FA with stencil CA on lanes 0..31 and FB
// with CB on lanes 32..63 (CB < 0: those lanes idle); every lane of a half
// returns its half's sum.  Lane 5j + i of a half holds window position (i, j)
// and walks the five z positions, whose values are wave-uniform (scalar
// loads): five gathers per lane, each of 5-node runs, and no cross-lane reads
// before the sum.  Spreading the 125 points over the lanes took 70 LDS
// permutations a marker to hand out the per-axis values, which bound it.
// DA, DB: terms times the normal distance n . (x_node - xb).
template <int CA, int CB, bool DA, bool DB>
__device__ __forceinline__ double gather_pair(const DevGrid& g, const Markers& m,
                                              const int* __restrict__ idx,
                                              const double* __restrict__ phi,
                                              const double* __restrict__ dd,
                                              const double* __restrict__ normals, int l, int lane,
                                              const double* __restrict__ FA,
                                              const double* __restrict__ FB) {
  constexpr int C1 = CB < 0 ? CA : CB;
  constexpr int DS = C1 - CA;
  const bool hi = lane >= 32;
  const int p = lane & 31;
  const bool on = p < 25 && (CB >= 0 || !hi);
  const int j = on ? p * 13 >> 6 : 0, i = on ? p - 5 * j : 0;  // p / 5, p % 5 (p < 25)
  // the marker's tables (wave-uniform pointers) and this half's stencil in them
  const int* im = idx + (size_t)l * kStencils + CA * kStencil;
  const double* pm = phi + (size_t)l * kStencils + CA * kStencil;
  const unsigned h = hi ? DS * kStencil : 0;
  // strides of the field (the centre field is rhs_p-shaped, first index 2)
  auto n1 = [&](int c) { return c == 0 ? g.nx : (c == 3 ? g.nxg - 2 : g.nxg); };
  auto n2 = [&](int c) { return c == 1 ? g.ny : (c == 3 ? g.nyg - 2 : g.nyg); };
  const int s1 = hi ? n1(C1) : n1(CA);
  const int s2 = hi ? n1(C1) * n2(C1) : n1(CA) * n2(CA);
  const int first = (hi ? C1 : CA) == 3 ? 2 : 1;
  const double* F = hi && CB >= 0 ? FB : FA;
  const int X = im[h + (unsigned)i], Y = im[h + 5 + (unsigned)j];
  const double px = pm[h + (unsigned)i], py = pm[h + 5 + (unsigned)j];
  int Z[5];
  double pz[5];
#pragma unroll
  for (int k = 0; k < 5; k++) {
    const int za = im[10 + k], zb = im[DS * kStencil + 10 + k];
    const double pa = pm[10 + k], pb = pm[DS * kStencil + 10 + k];
    Z[k] = hi ? zb : za;
    pz[k] = hi ? pb : pa;
  }
  const int o0 = (X - first) + s1 * (Y - first);
  double f[5];
#pragma unroll
  for (int k = 0; k < 5; k++) f[k] = F[o0 + s2 * (Z[k] - first)];
  const double wxy = (m.A * px) * py;
  double acc = 0.0;
  if (DA || DB) {
    const double* dm = dd + (size_t)l * kStencils + CA * kStencil;
    const double dx = dm[h + (unsigned)i], dy = dm[h + 5 + (unsigned)j];
    const double nx = normals[l], ny = normals[m.nb + l], nz = normals[2 * (size_t)m.nb + l];
    const double dxy = nx * dx + ny * dy;
#pragma unroll
    for (int k = 0; k < 5; k++) {
      const double da = dm[10 + k], db = dm[DS * kStencil + 10 + k];
      const double v = (wxy * pz[k]) * f[k];
      const double vd = v * (dxy + nz * (hi ? db : da));
      acc += (hi ? DB : DA) ? vd : v;
    }
  } else {
#pragma unroll
    for (int k = 0; k < 5; k++) acc += (wxy * pz[k]) * f[k];
  }
  return half_sum(on ? acc : 0.0);
}

// E / E1n of U, V, W (src/immersed_boundary_operators.f90:409-501): the sums
// of the three components of marker l, component c < 2 on half c, 2 on half 0.
template <bool DXN>
__device__ __forceinline__ void gather_uvw(const DevGrid& g, const Markers& m, int l, int lane,
                                           const int* __restrict__ idx, const double* __restrict__ phi,
                                           const double* __restrict__ dd,
                                           const double* __restrict__ normals,
                                           const double* __restrict__ U, const double* __restrict__ V,
                                           const double* __restrict__ W, double r[2]) {
  r[0] = gather_pair<0, 1, DXN, DXN>(g, m, idx, phi, dd, normals, l, lane, U, V);
  r[1] = gather_pair<2, -1, DXN, DXN>(g, m, idx, phi, dd, normals, l, lane, W, W);
}

template <bool DXN>
__global__ __launch_bounds__(kBlock) void k_interp_uvw(DevGrid g, Markers m, C3D_STENCIL_ARGS,
                                                       const double* __restrict__ U,
                                                       const double* __restrict__ V,
                                                       const double* __restrict__ W,
                                                       double* __restrict__ out) {
  const int l = wave_marker(m.nb);
  const int lane = threadIdx.x & 63;
  if (l >= m.nb) return;
  double r[2];
  gather_uvw<DXN>(g, m, l, lane, idx, phi, dd, normals, U, V, W, r);
  if ((lane & 31) == 0) out[(lane >> 5) * m.nb + l] = r[0];
  if (lane == 0) out[2 * m.nb + l] = r[1];
}

// E1n of a centre field in rhs_p layout (:503-526).
__global__ __launch_bounds__(kBlock) void k_interp_c(DevGrid g, Markers m, C3D_STENCIL_ARGS,
                                                     const double* __restrict__ P, double sign,
                                                     double* __restrict__ out) {
  const int l = wave_marker(m.nb);
  const int lane = threadIdx.x & 63;
  if (l >= m.nb) return;
  const double r = gather_pair<3, -1, true, true>(g, m, idx, phi, dd, normals, l, lane, P, P);
  if (lane == 0) out[l] = sign * r;
}

// G(dt*phi) - Reg_c of the Schur velocity rows (src/projection.f90:131-142) in
// place of Reg_c, at the support nodes of each component (block row c): each
// node once, where the markers' stencils would evaluate it for every one of
// the (37 on average, two cylinders) entries that share it.  Every node lies
// in the gradient's index ranges (checked at set-up), where
// apply_boundary_conditions does not write.
__global__ __launch_bounds__(kBlock) void k_node_grad(DevGrid g, Spread s0, Spread s1, Spread s2,
                                                      const double* __restrict__ phi, double dt,
                                                      double* __restrict__ F0, double* __restrict__ F1,
                                                      double* __restrict__ F2) {
  const int c = blockIdx.y;
  const int nn = c == 0 ? s0.nnodes : (c == 1 ? s1.nnodes : s2.nnodes);
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nn) return;
  const int* node = c == 0 ? s0.node : (c == 1 ? s1.node : s2.node);
  double* F = c == 0 ? F0 : (c == 1 ? F1 : F2);
  const unsigned n1 = c == 0 ? g.nx : g.nxg, n2 = c == 1 ? g.ny : g.nyg;
  const unsigned o = (unsigned)node[t], r = o / n1;
  const int i = (int)(o - r * n1) + 1, k = (int)(r / n2) + 1, j = (int)(r - (unsigned)(k - 1) * n2) + 1;
  const double p0 = dt * phi[ridx(i, j, k, g.nxg, g.nyg)];
  const double p1 = dt * phi[ridx(i + (c == 0), j + (c == 1), k + (c == 2), g.nxg, g.nyg)];
  const double h = c == 0 ? g.dxg[i] : (c == 1 ? g.dyg[j] : g.dzg[k]);
  F[o] = (p1 - p0) / h - F[o];
}

// The four Schur rows of a marker (src/projection.f90:131-142) on one
// wavefront: u with v, then w with the pressure row -E1n(phi).
__global__ __launch_bounds__(kBlock) void k_schur_rows(DevGrid g, Markers m, C3D_STENCIL_ARGS,
                                                       const double* __restrict__ P,
                                                       const double* __restrict__ Du,
                                                       const double* __restrict__ Dv,
                                                       const double* __restrict__ Dw,
                                                       const double* __restrict__ E1nH,
                                                       const double* __restrict__ dudn,
                                                       double* __restrict__ Sf) {
  const int l = wave_marker(m.nb);
  const int lane = threadIdx.x & 63;
  if (l >= m.nb) return;
  const double r0 = gather_pair<0, 1, false, false>(g, m, idx, phi, dd, normals, l, lane, Du, Dv);
  const double r1 = gather_pair<2, 3, false, true>(g, m, idx, phi, dd, normals, l, lane, Dw, P);
  if ((lane & 31) == 0) {
    const int h = lane >> 5, o0 = h * m.nb + l;
    Sf[o0] = r0 - E1nH[o0] * dudn[o0];
    const int o1 = o0 + 2 * m.nb;
    Sf[o1] = h ? -r1 : r1 - E1nH[o1] * dudn[o1];
  }
}

// -E u + ub (src/projection.f90:51-52).
__global__ __launch_bounds__(kBlock) void k_rhs_u(DevGrid g, Markers m, C3D_STENCIL_ARGS,
                                                  const double* __restrict__ U,
                                                  const double* __restrict__ V,
                                                  const double* __restrict__ W,
                                                  double* __restrict__ out) {
  const int l = wave_marker(m.nb);
  const int lane = threadIdx.x & 63;
  if (l >= m.nb) return;
  double r[2];
  gather_uvw<false>(g, m, l, lane, idx, phi, dd, normals, U, V, W, r);
  const int o = (lane >> 5) * m.nb + l;
  if ((lane & 31) == 0) out[o] = -r[0] + m.ub[o];
  if (lane == 0) out[2 * m.nb + l] = -r[1] + m.ub[2 * m.nb + l];
}

__global__ void k_aux(Markers m, const double* __restrict__ f, double dt, double nu,
                      double* __restrict__ aux) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int nb = m.nb;
  if (t >= 3 * nb) return;
  const int l = t % nb;
  aux[t] = dt * nu * f[t] - dt * f[3 * nb + l] * m.normals[t];
}

// Static coefficients of the spreading entries: w*factor*sb[l] per entry.
__global__ void k_spread_coeffs(int nb, double A, double factor, const double* __restrict__ phi,
                                const double* __restrict__ sb, Spread sp) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= sp.nentries) return;
  const int q = sp.q[e];
  const int l = q / 125, p = q - 125 * l;
  const int i = p % 5, j = (p / 5) % 5, k = p / 25;
  const double w = ((A * phi[sidx(0, i, l)]) * phi[sidx(1, j, l)]) *
                   phi[sidx(2, k, l)];
  sp.ml[e] = l;
  sp.wfs[e] = w * factor * sb[l];
}

// entries per batch (16: 29.4 against 26.7 us per spreading of two cylinders'
// 24,576 markers; 8 with each batch's loads waited for: 30.7 us)
constexpr int kSpreadB = 8;

// R, src/immersed_boundary_operators.f90:544-603: one thread per support node,
// contributions in ascending marker order.
__device__ __forceinline__ void spread_node(const Spread& sp, int t, const double* __restrict__ f,
                                            double* __restrict__ F) {
  double acc = 0.0;
  const int n = sp.cnt[t];
  // The lanes of a wavefront walk the entries together, up to the largest
  // count (the first lane's: ranks descend in it); a lane past its own count
  // reads its first entry and does not add it.  The next batch's coefficients
  // and markers load while this batch's forces are gathered: a node has up to
  // about 100 entries, and the few wavefronts of the longest lists, which run
  // alone in the end, waited for both in turn.  The sum stays in entry order.
  const int nmax = __builtin_amdgcn_readfirstlane(n);
  int ml[kSpreadB];
  double wf[kSpreadB];
  auto load = [&](int i0) {
#pragma unroll
    for (int r = 0; r < kSpreadB; r++) {
      const int i = i0 + r;
      const int e = i < n ? sp.slot[min(i, nmax - 1)] + t : t;
      ml[r] = sp.ml[e];
      wf[r] = sp.wfs[e];
    }
  };
  load(0);
  for (int i0 = 0; i0 < nmax; i0 += kSpreadB) {
    double fv[kSpreadB], wc[kSpreadB];
#pragma unroll
    for (int r = 0; r < kSpreadB; r++) {
      fv[r] = f[ml[r]];
      wc[r] = wf[r];
    }
    if (i0 + kSpreadB < nmax) load(i0 + kSpreadB);
#pragma unroll
    for (int r = 0; r < kSpreadB; r++) acc = i0 + r < n ? acc + wc[r] * fv[r] : acc;
  }
  F[sp.node[t]] = acc;
}

__global__ __launch_bounds__(kBlock) void k_spread(Spread sp, const double* __restrict__ f,
                                                   double* __restrict__ F) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= sp.nnodes) return;
  spread_node(sp, t, f, F);
}

// The three components in one launch, block row c = component c, reading
// f_c = f + c*nb.
__global__ __launch_bounds__(kBlock) void k_spread3(Spread s0, Spread s1, Spread s2,
                                                    const double* __restrict__ f, int nb,
                                                    double* __restrict__ F0, double* __restrict__ F1,
                                                    double* __restrict__ F2) {
  const int c = blockIdx.y;
  const Spread sp = c == 0 ? s0 : (c == 1 ? s1 : s2);
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= sp.nnodes) return;
  spread_node(sp, t, f + (size_t)c * nb, c == 0 ? F0 : (c == 1 ? F1 : F2));
}

// remove_mean_per_body for the two-group slab layout
// (src/immersed_boundary_geometry.f90:400-442), then f -= coef*pj.  Block
// partial sums of the two bodies, then every block re-reduces the partials
// in the same fixed order and applies.
constexpr int kMeanBlocks = 64;  // one partial per lane of a wavefront

__device__ __forceinline__ double block_sum(double v, double* sh) {
  v = wave_sum(v);
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane == 0) sh[w] = v;
  __syncthreads();
  double r = 0.0;
  if (threadIdx.x == 0)
    for (int q = 0; q < kBlock / 64; q++) r += sh[q];
  return r;
}

__global__ __launch_bounds__(kBlock) void k_body_sums(Markers m, const double* __restrict__ f,
                                                      double* __restrict__ part) {
  __shared__ double s1[kBlock / 64], s2[kBlock / 64];
  const int nb = m.nb, nxb = m.nxb, nxb1 = m.nxb1;
  double a = 0.0, b = 0.0;
  for (int l = blockIdx.x * kBlock + threadIdx.x; l < nb; l += kMeanBlocks * kBlock) {
    if (l % nxb < nxb1)
      a += f[l];
    else
      b += f[l];
  }
  a = block_sum(a, s1);
  b = block_sum(b, s2);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = a;
    part[kMeanBlocks + blockIdx.x] = b;
  }
}

// The two bodies' means from the partials: every wavefront sums them in the
// same order.
struct Means {
  double a, b;
};
__device__ __forceinline__ Means body_means(const Markers& m, const double* __restrict__ part) {
  const int lane = threadIdx.x & 63;
  return {wave_sum(part[lane]) / (double)(m.nxb1 * m.nzb),
          wave_sum(part[kMeanBlocks + lane]) / (double)((m.nxb - m.nxb1) * m.nzb)};
}

__global__ __launch_bounds__(kBlock) void k_remove_mean(Markers m, double* __restrict__ f,
                                                        const double* __restrict__ part,
                                                        const double* __restrict__ coef,
                                                        const double* __restrict__ pj) {
  const Means avg = body_means(m, part);
  const int l = blockIdx.x * kBlock + threadIdx.x;
  if (l >= m.nb) return;
  double v = f[l] - ((l % m.nxb < m.nxb1) ? avg.a : avg.b);
  if (coef) v = v - coef[l] * pj[l];
  f[l] = v;
}

// U = U_interim - U_reg - G(dt*(P_interim - phi)) and the boundary conditions
// of the result (src/projection.f90:83-94): the unique cells, each value
// stored with its boundary images.
__global__ __launch_bounds__(kBlock) void k_ib_correct(DevGrid g, const double* __restrict__ Uint,
                                                       const double* __restrict__ Vint,
                                                       const double* __restrict__ Wint,
                                                       const double* __restrict__ Ureg,
                                                       const double* __restrict__ Vreg,
                                                       const double* __restrict__ Wreg,
                                                       const double* __restrict__ Pint,
                                                       const double* __restrict__ phi, double dt,
                                                       double* __restrict__ U,
                                                       double* __restrict__ V,
                                                       double* __restrict__ W) {
  const int i = blockIdx.x * 64 + (threadIdx.x & 63) + 2;
  const int j = blockIdx.y * 4 + (threadIdx.x >> 6) + 2;
  const int k = blockIdx.z + 2;
  const int nx = g.nx, ny = g.ny, nxg = g.nxg, nyg = g.nyg;
  if (i > nx - 1 || j > nyg - 1) return;
  auto q = [&](int a, int b, int c) {
    const size_t o = ridx(a, b, c, nxg, nyg);
    return dt * (Pint[o] - phi[o]);
  };
  const double q0 = q(i, j, k);
  bool bad = false;
  {
    const size_t o = fidx(i, j, k, nx, nyg);
    const double u = Uint[o] - Ureg[o] - (q(i + 1, j, k) - q0) / g.dxg[i];
    put_u(g, U, i, j, k, u);
    bad |= !isfinite(u);
  }
  if (j <= ny - 1) {
    const size_t o = fidx(i, j, k, nxg, ny);
    const double v = Vint[o] - Vreg[o] - (q(i, j + 1, k) - q0) / g.dyg[j];
    put_v(g, V, i, j, k, v);
    bad |= !isfinite(v);
  }
  {
    const size_t o = fidx(i, j, k, nxg, nyg);
    const double w = Wint[o] - Wreg[o] - (q(i, j, k + 1) - q0) / g.dzg[k];
    put_w(g, W, i, j, k, w);
    bad |= !isfinite(w);
  }
  if (bad && g.nonfinite) *g.nonfinite = 1u;  // every writer writes the same
}

__global__ void k_affine(const double* __restrict__ x, double a, double b, double* __restrict__ y,
                         size_t n) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) y[t] = a + b * x[t];
}

// interpolate_x/y/z of src/interpolation.f90 into the heaviside ranges.
__global__ void k_h_interp(DevGrid g, const double* __restrict__ Hc, double* __restrict__ Hu,
                           double* __restrict__ Hv, double* __restrict__ Hw) {
  const int i = blockIdx.x * 64 + (threadIdx.x & 63) + 2;
  const int j = blockIdx.y * 4 + (threadIdx.x >> 6) + 2;
  const int k = blockIdx.z + 2;
  const int nx = g.nx, ny = g.ny, nz = g.nz, nxg = g.nxg, nyg = g.nyg;
  if (i > nxg - 1 || j > nyg - 1) return;
  const double c = Hc[ridx(i, j, k, nxg, nyg)];
  if (i <= nx - 1) Hu[fidx(i, j, k, nx, nyg)] = 0.5 * (c + Hc[ridx(i + 1, j, k, nxg, nyg)]);
  if (j <= ny - 1) Hv[fidx(i, j, k, nxg, ny)] = 0.5 * (c + Hc[ridx(i, j + 1, k, nxg, nyg)]);
  if (k <= nz) Hw[fidx(i, j, k, nxg, nyg)] = 0.5 * (c + Hc[ridx(i, j, k + 1, nxg, nyg)]);
}

// ---- BiCGSTAB ----
__global__ __launch_bounds__(kBlock) void k_dot(const double* __restrict__ a, const double* __restrict__ b,
                                                const double* __restrict__ a2,
                                                const double* __restrict__ b2, size_t n,
                                                double* __restrict__ part, int slot) {
  __shared__ double sh[2][kBlock / 64];
  double s1 = 0.0, s2 = 0.0;
  for (size_t t = (size_t)blockIdx.x * kBlock + threadIdx.x; t < n; t += (size_t)kDotBlocks * kBlock) {
    s1 += a[t] * b[t];
    if (a2) s2 += a2[t] * b2[t];
  }
  const double r1 = block_sum(s1, sh[0]);
  if (threadIdx.x == 0) part[slot * kDotBlocks + blockIdx.x] = r1;
  if (a2) {
    const double r2 = block_sum(s2, sh[1]);
    if (threadIdx.x == 0) part[(slot + 1) * kDotBlocks + blockIdx.x] = r2;
  }
}

// The partials of one slot, summed by a whole wavefront in a fixed order (the
// host repeats it for the residual: residual_of_partials).
static_assert(kDotBlocks == 128, "two partials per lane");
__device__ __forceinline__ double sum_part(const double* part, int slot) {
  const double* p = part + slot * kDotBlocks + (threadIdx.x & 63);
  return wave_sum(p[0] + p[64]);
}

// The pressure rows' mean removal (k_remove_mean) and the dot products of the
// finished Schur product with BiCGSTAB's vector a: <a, Sf> into partial slot
// `slot` and, when two is set, <Sf, Sf> into the next.
__global__ __launch_bounds__(kBlock) void k_mean_dot(Markers m, double* __restrict__ Sf,
                                                     const double* __restrict__ mpart,
                                                     const double* __restrict__ coef,
                                                     const double* __restrict__ pj,
                                                     const double* __restrict__ a, int two,
                                                     double* __restrict__ part, int slot) {
  __shared__ double sh[2][kBlock / 64];
  const Means avg = body_means(m, mpart);
  const int nb = m.nb, n3 = 3 * nb, n = 4 * nb;
  double s1 = 0.0, s2 = 0.0;
  for (int t = blockIdx.x * kBlock + threadIdx.x; t < n; t += kDotBlocks * kBlock) {
    double v = Sf[t];
    if (t >= n3) {
      const int l = t - n3;
      v = v - ((l % m.nxb < m.nxb1) ? avg.a : avg.b);
      v = v - coef[l] * pj[l];
      Sf[t] = v;
    }
    s1 += a[t] * v;
    s2 += v * v;
  }
  const double r1 = block_sum(s1, sh[0]);
  if (threadIdx.x == 0) part[slot * kDotBlocks + blockIdx.x] = r1;
  if (two) {
    const double r2 = block_sum(s2, sh[1]);
    if (threadIdx.x == 0) part[(slot + 1) * kDotBlocks + blockIdx.x] = r2;
  }
}

// Per-solve input normalisation of the learned guess: out[0] = 1/rms of the
// n_r entries whose squares are summed in partial slot sr, out[1] = the
// same for slot sf (0 for a zero vector).
__global__ void k_norm_scales(const double* __restrict__ part, int sr, double n_r, int sf, double n_f,
                              double* __restrict__ out) {
  const double qr = sum_part(part, sr), qf = sum_part(part, sf);  // launched as one wavefront
  if (threadIdx.x != 0) return;
  out[0] = qr > 0.0 ? 1.0 / sqrt(qr / n_r) : 0.0;
  out[1] = qf > 0.0 ? 1.0 / sqrt(qf / n_f) : 0.0;
}

// Scalar slots: 0 rho_o, 1 alpha, 2 om, 3 rho_n, 4 bta, 5 err, 6 line-search
// step, 7 iterations begun, 8 the squared tolerance, 9 set once the solve has
// converged.  The vector kernels compute their scalars from the dot partials
// themselves (every wavefront, the same fixed-order sum) and block 0 stores
// them; no block of a kernel reads a slot that the same kernel writes.
__global__ void k_bicg_scalar(int step, double* sc, const double* __restrict__ part, double eps) {
  const double den = sum_part(part, 3), num = sum_part(part, 2);  // launched as one wavefront
  if (threadIdx.x != 0) return;
  if (step == 0) {
    sc[0] = 1.0;
    sc[1] = 1.0;
    sc[2] = 1.0;
    sc[7] = 0.0;
    sc[8] = eps;
    sc[9] = 0.0;
  } else {  // minimal-residual step along d: a = <r, S d> / <S d, S d>
    sc[6] = den > 0.0 ? num / den : 0.0;
  }
}

// aux of the spreading (k_aux) for the entry (l, c = 0..2) of f, fp its
// pressure entry.
__device__ __forceinline__ double aux_entry(const Markers& m, double dt, double nu, double f, double fp,
                                            int t) {
  return dt * nu * f - dt * fp * m.normals[t];
}

// rho_n = rhat.r (partial slot 0); bta = (rho_n/rho_o)*(alpha/om);
// p = r + bta*(p - om*v), and the next spreading's aux of p; one lane per
// marker.  Writes sc[3] = rho_n, sc[4] = bta and counts the iteration.
// The host queues an iteration before it knows the last one's residual: when
// that one (partial slot 4) met the tolerance, p, k_bicg_hs and k_bicg_xr
// leave every vector as it is.
// Breakdown guards here and in k_bicg_hs / k_bicg_xr: an exactly zero
// denominator gives a zero step instead of the reference's 0/0
// (src/projection.f90:165-172); a zero right-hand side then converges to
// x = 0 in one iteration.  Nonzero denominators are untouched.
__global__ __launch_bounds__(kBlock) void k_bicg_p(Markers m, const double* __restrict__ r,
                                                   const double* __restrict__ v, const double* sc,
                                                   double* scw, const double* __restrict__ part,
                                                   double dt, double nu, double* __restrict__ p,
                                                   double* __restrict__ aux) {
  const double begun = sc[7];
  const bool go = begun == 0.0 || sum_part(part, 4) >= sc[8];
  const bool first = blockIdx.x == 0 && threadIdx.x == 0;
  if (!go) {
    if (first) scw[9] = 1.0;
    return;
  }
  const double rho_n = sum_part(part, 0);
  const double bta = (sc[0] != 0.0 && sc[2] != 0.0) ? (rho_n / sc[0]) * (sc[1] / sc[2]) : 0.0;
  const double om = sc[2];
  if (first) {
    scw[3] = rho_n;
    scw[4] = bta;
    scw[5] = begun + 1.0;  // k_bicg_hs moves it to sc[7], which this kernel reads
  }
  const int l = blockIdx.x * kBlock + threadIdx.x, nb = m.nb;
  if (l >= nb) return;
  double q[4];
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const int t = c * nb + l;
    q[c] = r[t] + bta * (p[t] - om * v[t]);
    p[t] = q[c];
  }
#pragma unroll
  for (int c = 0; c < 3; c++) aux[c * nb + l] = aux_entry(m, dt, nu, q[c], q[3], c * nb + l);
}

// alpha = rho_n / rhat.v (partial slot 1); h = x + alpha*p; s = r - alpha*v,
// and the next spreading's aux of s.
// Writes sc[1] = alpha and sc[0] = rho_n (rho_o of the next iteration).
__global__ __launch_bounds__(kBlock) void k_bicg_hs(Markers m, const double* __restrict__ x,
                                                    const double* __restrict__ p,
                                                    const double* __restrict__ r,
                                                    const double* __restrict__ v, const double* sc,
                                                    double* scw, const double* __restrict__ part,
                                                    double dt, double nu, double* __restrict__ h,
                                                    double* __restrict__ sv,
                                                    double* __restrict__ aux) {
  if (sc[9] != 0.0) return;
  const double rho_n = sc[3];
  const double den = sum_part(part, 1);
  const double alpha = den != 0.0 ? rho_n / den : 0.0;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    scw[1] = alpha;
    scw[0] = rho_n;
    scw[7] = sc[5];
  }
  const int l = blockIdx.x * kBlock + threadIdx.x, nb = m.nb;
  if (l >= nb) return;
  double q[4];
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const int t = c * nb + l;
    h[t] = x[t] + alpha * p[t];
    q[c] = r[t] - alpha * v[t];
    sv[t] = q[c];
  }
#pragma unroll
  for (int c = 0; c < 3; c++) aux[c * nb + l] = aux_entry(m, dt, nu, q[c], q[3], c * nb + l);
}

// om = t.s / t.t (partial slots 2, 3); x = h + om*s; r = s - om*t; partials
// of r.r into slot 4 and of rhat.r into slot 0 (the next iteration's rho_n),
// those of r.r also to host memory, one half of `host` for odd iterations and
// one for even ones (the host reads one while the next iteration may run).
// Writes sc[2] = om.
__global__ __launch_bounds__(kBlock) void k_bicg_xr(const double* __restrict__ h,
                                                    const double* __restrict__ sv,
                                                    const double* __restrict__ tv,
                                                    const double* __restrict__ rhat,
                                                    const double* sc, double* scw, double* part,
                                                    double* __restrict__ x, double* __restrict__ r,
                                                    double* host, size_t n) {
  __shared__ double sh[2][kBlock / 64];
  if (sc[9] != 0.0) return;
  const double tt = sum_part(part, 3);
  const double om = tt != 0.0 ? sum_part(part, 2) / tt : 0.0;
  if (blockIdx.x == 0 && threadIdx.x == 0) scw[2] = om;
  double s4 = 0.0, s0 = 0.0;
  for (size_t t = (size_t)blockIdx.x * kBlock + threadIdx.x; t < n; t += (size_t)kDotBlocks * kBlock) {
    x[t] = h[t] + om * sv[t];
    const double rr = sv[t] - om * tv[t];
    r[t] = rr;
    s4 += rr * rr;
    s0 += rhat[t] * rr;
  }
  const double t4 = block_sum(s4, sh[0]);
  const double t0 = block_sum(s0, sh[1]);
  if (threadIdx.x == 0) {
    part[4 * kDotBlocks + blockIdx.x] = t4;
    part[0 * kDotBlocks + blockIdx.x] = t0;
    host[((int)sc[7] & 1) * kDotBlocks + blockIdx.x] = t4;
  }
}

__global__ void k_bicg_init(const double* __restrict__ b, double* __restrict__ r,
                            double* __restrict__ rhat, double* __restrict__ p,
                            double* __restrict__ v, size_t n) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const double rr = b ? b[t] - r[t] : r[t];  // b == null: r already holds the residual
  r[t] = rr;
  rhat[t] = rr;
  p[t] = 0.0;
  v[t] = 0.0;
}

// x = x + a d;  r = r - a S d  (a = sc[6])
__global__ void k_line_step(double* __restrict__ x, const double* __restrict__ d,
                            double* __restrict__ r, const double* __restrict__ Sd,
                            const double* __restrict__ sc, size_t n) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const double a = sc[6];
  x[t] = x[t] + a * d[t];
  r[t] = r[t] - a * Sd[t];
}

// ---------------------------------------------------------------------------
// History-projection start: block partials of several dot products against
// one vector, their fixed-order sums, linear combinations and the scaling of
// a Gram-Schmidt column.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_mdot(VecSet A, const double* __restrict__ q, size_t n,
                                                 double* __restrict__ part) {
  __shared__ double sh[kHist + 1][kBlock / 64];
  double s[kHist + 1];
#pragma unroll
  for (int j = 0; j <= kHist; j++) s[j] = 0.0;
  for (size_t t = (size_t)blockIdx.x * kBlock + threadIdx.x; t < n; t += (size_t)kDotBlocks * kBlock) {
    const double qt = q[t];
#pragma unroll
    for (int j = 0; j <= kHist; j++)
      if (j < A.k) s[j] += A.v[j][t] * qt;
  }
#pragma unroll
  for (int j = 0; j <= kHist; j++) {
    if (j < A.k) {
      const double r = block_sum(s[j], sh[j]);
      if (threadIdx.x == 0) part[j * kDotBlocks + blockIdx.x] = r;
    }
  }
}

// one wavefront per slot
__global__ void k_mreduce(const double* __restrict__ part, double* __restrict__ coef) {
  const double v = sum_part(part, blockIdx.x);
  if (threadIdx.x == 0) coef[blockIdx.x] = v;
}

// qa = (set ? 0 : qa) + sgn * sum_j coef[j] A_j ; xb likewise with B_j
__global__ void k_combine(VecSet A, VecSet B, const double* __restrict__ coef, double sgn, int set,
                          double* __restrict__ qa, double* __restrict__ xb, size_t n) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  double a = 0.0, b = 0.0;
  for (int j = 0; j < A.k; j++) {
    const double cj = sgn * coef[j];
    if (qa) a += cj * A.v[j][t];
    if (xb) b += cj * B.v[j][t];
  }
  if (qa) qa[t] = set ? a : qa[t] + a;
  if (xb) xb[t] = set ? b : xb[t] + b;
}

// q, x /= ||q|| when ||q||^2 > kHistDrop^2 * raw2 (raw2: the column's squared
// norm before orthogonalisation), else q = x = 0 (a dependent column).
__global__ void k_hscale(double* __restrict__ q, double* __restrict__ x,
                         const double* __restrict__ nrm2, const double* __restrict__ raw2, size_t n) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const double v = *nrm2;
  const bool keep = v > 0.0 && v > (kHistDrop * kHistDrop) * (*raw2);
  const double inv = keep ? 1.0 / sqrt(v) : 0.0;
  q[t] = q[t] * inv;
  x[t] = x[t] * inv;
}

// check_slip, src/monitor.f90:223-231
__global__ __launch_bounds__(kBlock) void k_max_slip(DevGrid g, Markers m, C3D_STENCIL_ARGS,
                                                     const double* __restrict__ U,
                                                     const double* __restrict__ V,
                                                     const double* __restrict__ W,
                                                     const double* __restrict__ E1nH,
                                                     const double* __restrict__ fb,
                                                     unsigned long long* red) {
  const int l = wave_marker(m.nb);
  const int lane = threadIdx.x & 63;
  if (l >= m.nb) return;
  double r[2];
  gather_uvw<false>(g, m, l, lane, idx, phi, dd, normals, U, V, W, r);
  auto slip = [&](double v, int o) { return fabs(v - E1nH[o] * fb[o] - m.ub[o]); };
  double mx = slip(r[0], (lane >> 5) * m.nb + l);
  if (lane < 32) mx = fmax(mx, slip(r[1], 2 * m.nb + l));
  mx = fmax(mx, __shfl_xor(mx, 32, 64));
  if (lane == 0) atomicMax(red, (unsigned long long)__double_as_longlong(mx));
}

inline dim3 blocks_for(size_t n, int b = kBlock) { return dim3((unsigned)((n + b - 1) / b)); }
// one lane per support node, a block row per component
inline dim3 node_blocks(const Spread sp[3]) {
  int mx = 1;
  for (int c = 0; c < 3; c++) mx = sp[c].nnodes > mx ? sp[c].nnodes : mx;
  dim3 grid = blocks_for((size_t)mx);
  grid.y = 3;
  return grid;
}
inline dim3 wave_blocks(int nb) { return dim3((unsigned)((nb + kBlock / 64 - 1) / (kBlock / 64))); }

}  // namespace

hipError_t launch_setup(const DevGrid& g, const SetupGrid& sg, const Markers& m, int* bad,
                        hipStream_t s) {
  hipLaunchKernelGGL(k_setup, blocks_for(m.nb, kSetupMarkers), dim3(kBlock), 0, s, g, sg, m, bad);
  return hipGetLastError();
}

hipError_t launch_mark_planes(const Markers& m, int* live, hipStream_t s) {
  hipLaunchKernelGGL(k_mark_planes, blocks_for((size_t)20 * m.nb), dim3(kBlock), 0, s, m, live);
  return hipGetLastError();
}

hipError_t launch_wave_geometry(const WaveBody& w, const WaveTime& wt, double* xb, double* yb,
                                double* zb, double* normals, double* sb, double* ub, int* yref,
                                int* bad, hipStream_t s) {
  const size_t nb = 2 * (size_t)w.nxb * w.nzb;
  hipLaunchKernelGGL(k_wave_geometry, blocks_for(nb), dim3(kBlock), 0, s, w, wt, xb, yb, zb,
                     normals, sb, ub, yref, bad);
  return hipGetLastError();
}

hipError_t launch_interp_uvw(const DevGrid& g, const Markers& m, const double* U, const double* V,
                             const double* W, bool with_dxn, double* out, hipStream_t s) {
  if (with_dxn)
    hipLaunchKernelGGL(k_interp_uvw<true>, wave_blocks(m.nb), dim3(kBlock), 0, s, g, m, C3D_STENCIL(m), U, V, W, out);
  else
    hipLaunchKernelGGL(k_interp_uvw<false>, wave_blocks(m.nb), dim3(kBlock), 0, s, g, m, C3D_STENCIL(m), U, V, W, out);
  return hipGetLastError();
}

hipError_t launch_interp_c(const DevGrid& g, const Markers& m, const double* P, double sign,
                           double* out, hipStream_t s) {
  hipLaunchKernelGGL(k_interp_c, wave_blocks(m.nb), dim3(kBlock), 0, s, g, m, C3D_STENCIL(m), P, sign, out);
  return hipGetLastError();
}

hipError_t launch_schur_rows(const DevGrid& g, const Markers& m, const Spread sp[3],
                             const double* phi, double dt, double* Ureg, double* Vreg,
                             double* Wreg, const double* E1nH, const double* dudn, double* Sf,
                             hipStream_t s) {
  hipLaunchKernelGGL(k_node_grad, node_blocks(sp), dim3(kBlock), 0, s, g, sp[0], sp[1], sp[2], phi, dt,
                     Ureg, Vreg, Wreg);
  hipLaunchKernelGGL(k_schur_rows, wave_blocks(m.nb), dim3(kBlock), 0, s, g, m, C3D_STENCIL(m), phi,
                     (const double*)Ureg, (const double*)Vreg, (const double*)Wreg, E1nH, dudn, Sf);
  return hipGetLastError();
}

hipError_t launch_rhs_u(const DevGrid& g, const Markers& m, const double* U, const double* V,
                        const double* W, double* out, hipStream_t s) {
  hipLaunchKernelGGL(k_rhs_u, wave_blocks(m.nb), dim3(kBlock), 0, s, g, m, C3D_STENCIL(m), U, V, W, out);
  return hipGetLastError();
}

hipError_t launch_aux(const Markers& m, const double* f, double dt, double nu, double* aux,
                      hipStream_t s) {
  hipLaunchKernelGGL(k_aux, blocks_for((size_t)3 * m.nb), dim3(kBlock), 0, s, m, f, dt, nu, aux);
  return hipGetLastError();
}

hipError_t launch_spread3(const Markers& m, const Spread sp[3], const double* f, double* F0,
                          double* F1, double* F2, hipStream_t s) {
  const dim3 grid = node_blocks(sp);
  hipLaunchKernelGGL(k_spread3, grid, dim3(kBlock), 0, s, sp[0], sp[1], sp[2], f, m.nb, F0, F1, F2);
  return hipGetLastError();
}

hipError_t launch_spread_coeffs(const Markers& m, const Spread& sp, int comp, hipStream_t s) {
  if (sp.nentries == 0) return hipSuccess;
  hipLaunchKernelGGL(k_spread_coeffs, blocks_for(sp.nentries), dim3(kBlock), 0, s, m.nb, m.A,
                     m.factor, (const double*)m.st[comp].phi, m.sb, sp);
  return hipGetLastError();
}

hipError_t launch_spread(const Markers& m, const Spread& sp, int comp, const double* f, double* F,
                         hipStream_t s) {
  (void)m;
  (void)comp;
  if (sp.nnodes == 0) return hipSuccess;
  hipLaunchKernelGGL(k_spread, blocks_for(sp.nnodes), dim3(kBlock), 0, s, sp, f, F);
  return hipGetLastError();
}

hipError_t launch_remove_mean(const Markers& m, double* f, const double* coef, const double* pj,
                              double* part, hipStream_t s) {
  hipLaunchKernelGGL(k_body_sums, dim3(kMeanBlocks), dim3(kBlock), 0, s, m, (const double*)f, part);
  hipLaunchKernelGGL(k_remove_mean, blocks_for(m.nb), dim3(kBlock), 0, s, m, f, (const double*)part,
                     coef, pj);
  return hipGetLastError();
}

hipError_t launch_mean_dot(const Markers& m, double* Sf, const double* coef, const double* pj,
                           const double* a, bool two, double* mpart, double* part, int slot,
                           hipStream_t s) {
  hipLaunchKernelGGL(k_body_sums, dim3(kMeanBlocks), dim3(kBlock), 0, s, m,
                     (const double*)(Sf + 3 * (size_t)m.nb), mpart);
  hipLaunchKernelGGL(k_mean_dot, dim3(kDotBlocks), dim3(kBlock), 0, s, m, Sf, (const double*)mpart, coef,
                     pj, a, two ? 1 : 0, part, slot);
  return hipGetLastError();
}

hipError_t launch_ib_correct(const DevGrid& g, const double* Uint, const double* Vint,
                             const double* Wint, const double* Ureg, const double* Vreg,
                             const double* Wreg, const double* Pint, const double* phi, double dt,
                             double* U, double* V, double* W, hipStream_t s) {
  hipLaunchKernelGGL(k_ib_correct, dim3((g.nx - 2 + 63) / 64, (g.nyg - 2 + 3) / 4, g.nz - 2),
                     dim3(kBlock), 0, s, g, Uint, Vint, Wint, Ureg, Vreg, Wreg, Pint, phi, dt, U, V, W);
  return hipGetLastError();
}

hipError_t launch_affine(const double* x, double a, double b, double* y, size_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_affine, blocks_for(n), dim3(kBlock), 0, s, x, a, b, y, n);
  return hipGetLastError();
}

hipError_t launch_h_interp(const DevGrid& g, const double* Hc, double* Hu, double* Hv, double* Hw,
                           hipStream_t s) {
  hipLaunchKernelGGL(k_h_interp, dim3((g.nxg - 2 + 63) / 64, (g.nyg - 2 + 3) / 4, g.nzg - 1),
                     dim3(kBlock), 0, s, g, Hc, Hu, Hv, Hw);
  return hipGetLastError();
}

hipError_t launch_dot(const double* a, const double* b, const double* a2, const double* b2,
                      size_t n, double* part, int slot, hipStream_t s) {
  hipLaunchKernelGGL(k_dot, dim3(kDotBlocks), dim3(kBlock), 0, s, a, b, a2, b2, n, part, slot);
  return hipGetLastError();
}

hipError_t launch_norm_scales(const double* part, int sr, size_t n_r, int sf, size_t n_f,
                              double* out, hipStream_t s) {
  hipLaunchKernelGGL(k_norm_scales, dim3(1), dim3(64), 0, s, part, sr, (double)n_r, sf, (double)n_f,
                     out);
  return hipGetLastError();
}

hipError_t launch_bicg_scalar(int step, double* sc, const double* part, double eps, hipStream_t s) {
  hipLaunchKernelGGL(k_bicg_scalar, dim3(1), dim3(64), 0, s, step, sc, part, eps);
  return hipGetLastError();
}

hipError_t launch_bicg_p(const Markers& m, const double* r, const double* v, double* sc,
                         const double* part, double dt, double nu, double* p, double* aux,
                         hipStream_t s) {
  hipLaunchKernelGGL(k_bicg_p, blocks_for(m.nb), dim3(kBlock), 0, s, m, r, v, (const double*)sc, sc, part,
                     dt, nu, p, aux);
  return hipGetLastError();
}

hipError_t launch_bicg_hs(const Markers& m, const double* x, const double* p, const double* r,
                          const double* v, double* sc, const double* part, double dt, double nu,
                          double* h, double* sv, double* aux, hipStream_t s) {
  hipLaunchKernelGGL(k_bicg_hs, blocks_for(m.nb), dim3(kBlock), 0, s, m, x, p, r, v, (const double*)sc, sc,
                     part, dt, nu, h, sv, aux);
  return hipGetLastError();
}

hipError_t launch_bicg_xr(const double* h, const double* sv, const double* t, const double* rhat,
                          double* sc, double* part, double* x, double* r, double* host, size_t n,
                          hipStream_t s) {
  hipLaunchKernelGGL(k_bicg_xr, dim3(kDotBlocks), dim3(kBlock), 0, s, h, sv, t, rhat, (const double*)sc,
                     sc, part, x, r, host, n);
  return hipGetLastError();
}

double residual_of_partials(const double* host) {
  double a[64], b[64];
  for (int l = 0; l < 64; l++) a[l] = host[l] + host[l + 64];
  for (int off = 32; off > 0; off >>= 1) {  // wave_sum
    for (int l = 0; l < 64; l++) b[l] = a[l] + a[l ^ off];
    for (int l = 0; l < 64; l++) a[l] = b[l];
  }
  return a[0];
}

hipError_t launch_bicg_init(const double* b, double* r, double* rhat, double* p, double* v,
                            size_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_bicg_init, blocks_for(n), dim3(kBlock), 0, s, b, r, rhat, p, v, n);
  return hipGetLastError();
}

hipError_t launch_line_step(double* x, const double* d, double* r, const double* Sd,
                            const double* sc, size_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_line_step, blocks_for(n), dim3(kBlock), 0, s, x, d, r, Sd, sc, n);
  return hipGetLastError();
}

hipError_t launch_mdot(const VecSet& A, const double* q, size_t n, double* part, hipStream_t s) {
  if (A.k < 1 || A.k > kHist + 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_mdot, dim3(kDotBlocks), dim3(kBlock), 0, s, A, q, n, part);
  return hipGetLastError();
}

hipError_t launch_mreduce(const double* part, int k, double* coef, hipStream_t s) {
  if (k < 1 || k > kHist + 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_mreduce, dim3(k), dim3(64), 0, s, part, coef);
  return hipGetLastError();
}

hipError_t launch_combine(const VecSet& A, const VecSet& B, const double* coef, double sgn, bool set,
                          double* qa, double* xb, size_t n, hipStream_t s) {
  if (A.k < 0 || A.k > kHist + 1 || (xb && B.k != A.k)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_combine, blocks_for(n), dim3(kBlock), 0, s, A, B, coef, sgn, set ? 1 : 0, qa,
                     xb, n);
  return hipGetLastError();
}

hipError_t launch_hscale(double* q, double* x, const double* nrm2, const double* raw2, size_t n,
                         hipStream_t s) {
  hipLaunchKernelGGL(k_hscale, blocks_for(n), dim3(kBlock), 0, s, q, x, nrm2, raw2, n);
  return hipGetLastError();
}

hipError_t launch_max_slip(const DevGrid& g, const Markers& m, const double* U, const double* V,
                           const double* W, const double* E1nH, const double* fb,
                           unsigned long long* red, hipStream_t s) {
  hipLaunchKernelGGL(k_max_slip, wave_blocks(m.nb), dim3(kBlock), 0, s, g, m, C3D_STENCIL(m), U, V, W, E1nH, fb, red);
  return hipGetLastError();
}

}  // namespace ib
}  // namespace c3d
