// The z march of the right-hand-side kernels (rk3.hip, rk3_fast.hip).
//
// A workgroup owns a 64 x 4 column of points and walks KC z planes; U, V, W
// around it lie in LDS as a ring of three planes with a one-cell x/y halo, so
// every neighbour read of the point functions is an LDS read.  What bounds it
// is the vector instruction count (570 integer and 146 FP64 instructions per
// point and plane in stage 2 before, 924 us of which 540 us are the words it
// moves), so a lane computes its offsets once: a global address is a
// wave-uniform plane pointer plus a 32-bit byte offset that stays the same, an
// LDS address one of three ring offsets plus a constant.  The x spacing
// factors stay in registers, the y and z ones are scalar loads, and the loads
// of plane k+2 are in flight while plane k is evaluated.
#pragma once

#include "rk3_point.hpp"

namespace c3d {
namespace {

// A grid table at a wave-uniform index: read-only memory, so a scalar load.
struct ScalarTab {
  const double* p;
  __device__ __forceinline__ double operator[](int i) const {
    return ((const __attribute__((address_space(4))) double*)p)[i];
  }
};
// A grid table read at the lane's own x index only.
struct LaneTab {
  double v;
  __device__ __forceinline__ double operator[](int) const { return v; }
};
struct MarchGrid {
  int nx, ny, nz, nxg, nyg, nzg;
  ScalarTab dyf, dzf, dyg, dzg, rdyf, rdzf, rdyg, rdzg, nudyf, nudzf, nudzg;
  LaneTab dxf, dxg;
};

constexpr int kRing = 3 * kTP;  // LDS doubles of one plane: U, V, W

struct MarchAcc {
  const double* s;   // LDS
  int om, o0, op;    // the lane's cell in planes k-1, k, k+1
  int i, j, k;
  double rdxg, rdxf, nudxf0, nudxf1, nudxg0, nudxgm;  // at i (nudxf1 i+1, nudxgm i-1)
  __device__ __forceinline__ double at(int f, int ii, int jj, int kk) const {
    const int o = kk < k ? om : (kk > k ? op : o0);
    return s[o + (f * kTP + (jj - j) * kTX + (ii - i))];
  }
  template <int T>
  __device__ __forceinline__ double x(int ii) const {
    if constexpr (T == kXrdxg) return rdxg;
    else if constexpr (T == kXrdxf) return rdxf;
    else if constexpr (T == kXnudxf) return ii > i ? nudxf1 : nudxf0;
    else return ii < i ? nudxgm : nudxg0;
  }
  __device__ __forceinline__ double U(int ii, int jj, int kk) const { return at(0, ii, jj, kk); }
  __device__ __forceinline__ double V(int ii, int jj, int kk) const { return at(1, ii, jj, kk); }
  __device__ __forceinline__ double W(int ii, int jj, int kk) const { return at(2, ii, jj, kk); }
};

// Element at a byte offset from a wave-uniform pointer.
__device__ __forceinline__ const double& cell(const double* p, unsigned b) {
  return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(p) + b);
}
__device__ __forceinline__ double& cell(double* p, unsigned b) {
  return *reinterpret_cast<double*>(reinterpret_cast<char*>(p) + b);
}

// The lane's place in one component's arrays: byte offsets in a plane of the
// field (o) and of the interior-shaped right-hand side (f), the planes' sizes
// in elements, and whether the point belongs to the component.
struct Spot {
  unsigned o, f;
  size_t po, pf;
  bool in;
};

// Calls pre(k, spots) before the plane's barrier (loads of the point's own
// words) and eval(A, G, k, spots) after it, for each plane k of the workgroup.
template <int KC, typename Pre, typename Eval>
__device__ __forceinline__ void march(const DevGrid& g, const double* __restrict__ U,
                                      const double* __restrict__ V, const double* __restrict__ W,
                                      Pre pre, Eval eval) {
  __shared__ double tile[3 * kRing];
  unsigned bx, by, bz;
  xcd_tile(bx, by, bz);  // neighbouring tiles on one XCD (shared halo rows)
  const int i0 = bx * 64 + 2, j0 = by * 4 + 2, kb = bz * KC + 2;
  const int lane = threadIdx.x & 63;
  // j is the same on all lanes of a wavefront: wave-uniform, as is k
  const int ty = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int i = i0 + lane, j = j0 + ty;
  const int nx = g.nx, ny = g.ny, nz = g.nz, nxg = g.nxg, nyg = g.nyg, nzg = g.nzg;

  // the two tile cells this lane loads; past the arrays' ends the last cell
  // (such halo cells only feed points outside the ranges)
  unsigned bu[2], bv[2], bw[2];
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const int e = min((int)threadIdx.x + q * 256, kTP - 1);
    const int ii = i0 - 1 + e % kTX, jj = j0 - 1 + e / kTX;
    bu[q] = 8u * (unsigned)(min(ii, nx) - 1 + nx * (min(jj, nyg) - 1));
    bv[q] = 8u * (unsigned)(min(ii, nxg) - 1 + nxg * (min(jj, ny) - 1));
    bw[q] = 8u * (unsigned)(min(ii, nxg) - 1 + nxg * (min(jj, nyg) - 1));
  }
  auto load = [&](int k, PlaneRegs& r) {
    const double* pu = U + (size_t)(min(k, nzg) - 1) * nx * nyg;
    const double* pv = V + (size_t)(min(k, nzg) - 1) * nxg * ny;
    const double* pw = W + (size_t)(min(k, nz) - 1) * nxg * nyg;
#pragma unroll
    for (int q = 0; q < 2; q++) {
      r.u[q] = cell(pu, bu[q]);
      r.v[q] = cell(pv, bv[q]);
      r.w[q] = cell(pw, bw[q]);
    }
  };
  auto store = [&](int o, const PlaneRegs& r) {
    double* t = tile + o + threadIdx.x;
    t[0] = r.u[0];
    t[kTP] = r.v[0];
    t[2 * kTP] = r.w[0];
    if (threadIdx.x < kTP - 256) {
      t[256] = r.u[1];
      t[kTP + 256] = r.v[1];
      t[2 * kTP + 256] = r.w[1];
    }
  };

  const int it = min(i, nxg - 1);  // lanes past the domain read its last entries
  MarchGrid G{nx, ny, nz, nxg, nyg, nzg,
              {g.dyf}, {g.dzf}, {g.dyg}, {g.dzg}, {g.rdyf}, {g.rdzf}, {g.rdyg}, {g.rdzg},
              {g.nudyf}, {g.nudzf}, {g.nudzg}, {g.dxf[min(it, nx)]}, {g.dxg[it]}};
  MarchAcc A;
  A.s = tile;
  A.i = i;
  A.j = j;
  A.rdxg = g.rdxg[it];
  A.rdxf = g.rdxf[it];
  A.nudxf0 = g.nudxf[it];
  A.nudxf1 = g.nudxf[it + 1];
  A.nudxg0 = g.nudxg[it];
  A.nudxgm = g.nudxg[it - 1];

  const bool in = i <= nxg - 1 && j <= nyg - 1;
  auto spot = [&](int n1, int n2, int m1, int m2, bool on) {
    return Spot{8u * (unsigned)(i - 1 + n1 * (j - 1)), 8u * (unsigned)(i - 2 + m1 * (j - 2)),
                (size_t)n1 * n2, (size_t)m1 * m2, on};
  };
  const Spot su = spot(nx, nyg, nx - 2, nyg - 2, in && i <= nx - 1);
  const Spot sv = spot(nxg, ny, nxg - 2, ny - 2, in && j <= ny - 1);
  const Spot sw = spot(nxg, nyg, nxg - 2, nyg - 2, in);

  PlaneRegs nxt;
  {  // the first three planes' loads are all in flight before the first is stored
    PlaneRegs p0, p1;
    load(kb - 1, p0);
    load(kb, p1);
    load(kb + 1, nxt);
    store(0, p0);
    store(kRing, p1);
  }
  const int c = (ty + 1) * kTX + lane + 1;
  int om = 0, o0 = kRing, op = 2 * kRing;
  const int ke = min(kb + KC - 1, nzg - 1);
  for (int k = kb; k <= ke; k++) {  // uniform across the workgroup
    store(op, nxt);  // the slot held plane k-2, done with the last iteration
    pre(k, su, sv, sw);
    __syncthreads();
    load(k + 2, nxt);
    A.om = om + c;
    A.o0 = o0 + c;
    A.op = op + c;
    A.k = k;
    eval(A, G, k, su, sv, sw);
    __syncthreads();  // plane k-1's slot is refilled next
    const int t = om;
    om = o0;
    o0 = op;
    op = t;
  }
}

}  // namespace
}  // namespace c3d
