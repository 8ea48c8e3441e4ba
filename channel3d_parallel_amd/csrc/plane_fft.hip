// Both transforms of a y plane in one kernel, FP64, for planes that fit in a
// workgroup's LDS: the x transform with its input (k_fwd_x) followed by the z
// transform, and the z transform followed by the inverse x transform with its
// output stage (k_inv_x).  The half spectrum of a plane stays in LDS between
// the two, one launch and one pass over the spectrum less each way; small
// grids are bound by the length of the chain of launches.
#include <cstdlib>

#include "fft_lds.hpp"
#include "kernels.hpp"

namespace c3d {

namespace {

constexpr int kPB = 512;  // threads per workgroup (one plane)
constexpr int kNTZ = 8;   // threads per z column

// Threads per x row pair: the largest power of two that fits all pairs.
constexpr int row_threads(int np) {
  int t = 1;
  while (2 * t * np <= kPB) t *= 2;
  return t;
}

template <int N, int NZ>
struct Plane {
  static constexpr int NP = NZ / 2;       // row pairs, one complex row each
  static constexpr int NH = N / 2 + 1;
  static constexpr int LP = lds_row_len(N), ZP = lds_row_len(NZ);
  static constexpr int NT = row_threads(NP);
  static constexpr int BUF = NP * LP > NH * ZP ? NP * LP : NH * ZP;
  static constexpr int ITEMS = (NP * N + kPB - 1) / kPB;   // points of row pairs per thread
  static constexpr int SPLIT = (NP * NH + kPB - 1) / kPB;  // bins of row pairs per thread
};

// Threads beyond the last row or column repeat it: they read what its own
// threads read and, after the pass's barrier, store the same values.
template <int N, int NZ, int SIGN>
__device__ __forceinline__ void rows_fft(cpx<double>* buf, const cpx<double>* __restrict__ tw) {
  using L = Plane<N, NZ>;
  const int r = min((int)threadIdx.x / L::NT, L::NP - 1);
  fft_lds<double, N, L::NT, SIGN>(buf + r * L::LP, tw, threadIdx.x % L::NT);
}
template <int N, int NZ, int SIGN>
__device__ __forceinline__ void cols_fft(cpx<double>* buf, const cpx<double>* __restrict__ tw) {
  using L = Plane<N, NZ>;
#pragma unroll 1
  for (int c0 = 0; c0 < L::NH; c0 += kPB / kNTZ) {
    const int c = min(c0 + (int)threadIdx.x / kNTZ, L::NH - 1);
    fft_lds<double, NZ, kNTZ, SIGN>(buf + c * L::ZP, tw, threadIdx.x % kNTZ);
  }
}

// UVW: the divergence of U, V, W (per: with the boundary values taken from the
// interior), else the rhs_p-shaped array.
template <int N, int NZ, bool UVW>
__global__ __launch_bounds__(kPB) void k_fwd_plane(DevGrid g, const double* __restrict__ U,
                                                   const double* __restrict__ V,
                                                   const double* __restrict__ W,
                                                   const double* __restrict__ rhs,
                                                   cpx<double>* __restrict__ S, int per,
                                                   const int* __restrict__ planes) {
  using L = Plane<N, NZ>;
  __shared__ cpx<double> buf[L::BUF];
  const int tid = threadIdx.x;
  const int js = blockIdx.x;
  const int j = (planes ? planes[js] : js) + 2;
  const int nx = g.nx, ny = g.ny, nxg = g.nxg, nyg = g.nyg;
  const double ry = g.rdyf[j];
  const bool vlo = per && j == 2, vhi = per && j == ny;
  double d0[L::ITEMS], d1[L::ITEMS];
#pragma unroll
  for (int q = 0; q < L::ITEMS; q++) {
    const int e = min(tid + q * kPB, L::NP * N - 1);
    const int p = e / N, n = e % N, k = 2 * p + 2;
    if constexpr (UVW) {
      const int nm = (per && n == 0) ? N : n;
      const int km = (per && p == 0) ? g.nz - 1 : k - 1;
      const double* u = U + fidx(1, j, k, nx, nyg);
      const double* v = V + fidx(1, j, k, nxg, ny) + n + 1;
      const double* w = W + fidx(1, j, k, nxg, nyg) + n + 1;
      const size_t pu = (size_t)nx * nyg, pv = (size_t)nxg * ny, pw = (size_t)nxg * nyg;
      const double rx = g.rdxf[n + 2];
      const double w0 = W[fidx(1, j, km, nxg, nyg) + n + 1], w1 = w[0], w2 = w[pw];
      const double v0 = vhi ? 0.0 : v[0], v1 = vhi ? 0.0 : v[pv];
      const double m0 = vlo ? 0.0 : v[-nxg], m1 = vlo ? 0.0 : v[(ptrdiff_t)pv - nxg];
      d0[q] = (u[n + 1] - u[nm]) * rx + (v0 - m0) * ry + (w1 - w0) * g.rdzf[k];
      d1[q] = (u[pu + n + 1] - u[pu + nm]) * rx + (v1 - m1) * ry + (w2 - w1) * g.rdzf[k + 1];
    } else {
      const double* r = rhs + ridx(2, j, k, nxg, nyg) + n;
      d0[q] = r[0];
      d1[q] = r[(size_t)(nxg - 2) * (nyg - 2)];
    }
  }
#pragma unroll
  for (int q = 0; q < L::ITEMS; q++) {
    const int e = tid + q * kPB;
    if (e < L::NP * N) buf[(e / N) * L::LP + lp(e % N)] = cmk(d0[q], d1[q]);
  }
  __syncthreads();
  rows_fft<N, NZ, -1>(buf, g.twx64);
  // the two real rows of a pair: A_k = (Z_k + conj Z_{N-k})/2, B_k =
  // (Z_k - conj Z_{N-k})/(2i), into the z rows [kx][kz]
  cpx<double> A[L::SPLIT], B[L::SPLIT];
#pragma unroll
  for (int q = 0; q < L::SPLIT; q++) {
    const int e = min(tid + q * kPB, L::NP * L::NH - 1);
    const int p = e / L::NH, kx = e % L::NH;
    const cpx<double> z = buf[p * L::LP + lp(kx)];
    const cpx<double> zc = buf[p * L::LP + lp(kx == 0 ? 0 : N - kx)];
    A[q] = cmk(0.5 * (z.x + zc.x), 0.5 * (z.y - zc.y));
    B[q] = cmk(0.5 * (z.y + zc.y), 0.5 * (zc.x - z.x));
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < L::SPLIT; q++) {
    const int e = tid + q * kPB;
    if (e < L::NP * L::NH) {
      const int p = e / L::NH, kx = e % L::NH;
      buf[kx * L::ZP + lp(2 * p)] = A[q];
      buf[kx * L::ZP + lp(2 * p + 1)] = B[q];
    }
  }
  __syncthreads();
  cols_fft<N, NZ, -1>(buf, g.twz64);
  cpx<double>* out = S + (size_t)js * L::NH * NZ;
  for (int e = tid; e < L::NH * NZ; e += kPB) out[e] = buf[(e / NZ) * L::ZP + lp(e % NZ)];
}

// MODE 0: out = phi, MODE 1: out = phi/dt; rk1: P with its ghosts (k_inv_x).
template <int N, int NZ, int MODE>
__global__ __launch_bounds__(kPB) void k_inv_plane(DevGrid g, const cpx<double>* __restrict__ S,
                                                   double* __restrict__ out, double* __restrict__ P,
                                                   double dt, int rk1,
                                                   const int* __restrict__ planes) {
  using L = Plane<N, NZ>;
  __shared__ cpx<double> buf[L::BUF];
  const int tid = threadIdx.x;
  const int js = blockIdx.x;
  const int j = (planes ? planes[js] : js) + 2;
  const int nxg = g.nxg, nyg = g.nyg, nzg = g.nzg;
  {
    constexpr int LOADS = (L::NH * NZ + kPB - 1) / kPB;
    const cpx<double>* in = S + (size_t)js * L::NH * NZ;
    cpx<double> v[LOADS];
#pragma unroll
    for (int q = 0; q < LOADS; q++) v[q] = in[min(tid + q * kPB, L::NH * NZ - 1)];
#pragma unroll
    for (int q = 0; q < LOADS; q++) {
      const int e = tid + q * kPB;
      if (e < L::NH * NZ) buf[(e / NZ) * L::ZP + lp(e % NZ)] = v[q];
    }
  }
  __syncthreads();
  cols_fft<N, NZ, +1>(buf, g.twz64);
  // Hermitian extension and packing Z = A + iB (the imaginary parts of the DC
  // and Nyquist bins dropped: the real part of the full inverse)
  cpx<double> Z[L::ITEMS];
#pragma unroll
  for (int q = 0; q < L::ITEMS; q++) {
    const int e = min(tid + q * kPB, L::NP * N - 1);
    const int p = e / N, n = e % N, kx = n <= N / 2 ? n : N - n;
    cpx<double> a = buf[kx * L::ZP + lp(2 * p)], b = buf[kx * L::ZP + lp(2 * p + 1)];
    const double s = (n == 0 || n == N / 2) ? 0.0 : (n < N / 2 ? 1.0 : -1.0);
    a.y = s == 0.0 ? 0.0 : s * a.y;
    b.y = s == 0.0 ? 0.0 : s * b.y;
    Z[q] = cmk(a.x - b.y, a.y + b.x);
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < L::ITEMS; q++) {
    const int e = tid + q * kPB;
    if (e < L::NP * N) buf[(e / N) * L::LP + lp(e % N)] = Z[q];
  }
  __syncthreads();
  rows_fft<N, NZ, +1>(buf, g.twx64);

  const double norm = (double)(N * NZ), cP = dt * (8.0 / 15.0);
  // value at x index n + 2 of plane k, with the periodic copies i = nxg-1 and
  // k = nzp+2, and P's ghosts, which repeat their neighbour
  auto put = [&](int n, int k, double phi) {
    const double o = MODE == 1 ? phi / dt : phi;
    double* row = out + ridx(2, j, k, nxg, nyg);
    double* dup = out + ridx(2, j, NZ + 2, nxg, nyg);
    row[n] = o;
    if (n == 0) row[N] = o;
    if (k == 2) {
      dup[n] = o;
      if (n == 0) dup[N] = o;
    }
    if (!rk1) return;
    const double v = phi / cP;
    for (int b = 0; b < 2; b++) {
      if (b == 1 && j != 2 && j != nyg - 1) break;
      const int jb = b == 0 ? j : (j == 2 ? 1 : nyg);
      for (int c = 0; c < (k == 2 ? 4 : 1); c++) {
        const int kc = c == 0 ? k : (c == 1 ? NZ + 2 : (c == 2 ? 1 : nzg));
        double* r = P + fidx(2, jb, kc, nxg, nyg);
        r[n] = v;
        if (n == 0) {
          r[-1] = v;
          r[N] = v;
          r[N + 1] = v;
        }
      }
    }
  };
#pragma unroll
  for (int q = 0; q < L::ITEMS; q++) {
    const int e = tid + q * kPB;
    if (e < L::NP * N) {
      const int p = e / N, n = e % N;
      const cpx<double> z = buf[p * L::LP + lp(n)];
      put(n, 2 * p + 2, z.x / norm);
      put(n, 2 * p + 3, z.y / norm);
    }
  }
  // plane nzg: zero after the divergence; a Poisson solve keeps its input but
  // for the x-periodic copy (src/poisson.f90:110)
  double* last = out + ridx(2, j, nzg, nxg, nyg);
  if constexpr (MODE == 1) {
    for (int n = tid; n <= N; n += kPB) last[n] = 0.0;
  } else if (tid == 0) {
    last[N] = last[0];
  }
}

// Largest plane, in points.  One workgroup per plane pays while a plane is a
// few microseconds of one CU's work: 20 steps of 32x64x32 cells 2.92 against
// 3.54 ms with separate transforms, of 96x100x48 cells 4.76 against 5.19 ms; at
// 128 x 64 points the two kernels of a plane take 17.0 + 13.7 us, the four
// separate ones 26.8 us.  Between the two, planes of 6144 points are mixed:
// projections of 96x64x64 cells 41.0 against 43.2 us, of 64x64x96 41.0 against
// 41.7, of 128x96x48 44.5 against 46.2, but of 48x64x128 46.7 against 38.2 us.
constexpr int kPlaneMax = 4608;

// BODY with N and NZ, the transform lengths; planes above kPlaneMax are not
// built, since plane_fft() never takes them.
#define C3D_PLANE_CASE(NN, M, ...)                      \
  case M:                                               \
    if constexpr (NN * M <= kPlaneMax) {                \
      constexpr int NZ = M;                             \
      __VA_ARGS__;                                      \
    } else {                                            \
      return hipErrorInvalidValue;                      \
    }                                                   \
    break;
#define C3D_PLANE_Z(NN, nz, ...)                        \
  switch (nz) {                                         \
    C3D_PLANE_CASE(NN, 16, __VA_ARGS__)                 \
    C3D_PLANE_CASE(NN, 32, __VA_ARGS__)                 \
    C3D_PLANE_CASE(NN, 48, __VA_ARGS__)                 \
    C3D_PLANE_CASE(NN, 64, __VA_ARGS__)                 \
    C3D_PLANE_CASE(NN, 96, __VA_ARGS__)                 \
    C3D_PLANE_CASE(NN, 128, __VA_ARGS__)                \
    default: return hipErrorInvalidValue;               \
  }
#define C3D_PLANE(nx, nz, ...)                                                                      \
  switch (nx) {                                                                                     \
    case 16: { constexpr int N = 16; C3D_PLANE_Z(N, nz, __VA_ARGS__) } break;                       \
    case 32: { constexpr int N = 32; C3D_PLANE_Z(N, nz, __VA_ARGS__) } break;                       \
    case 48: { constexpr int N = 48; C3D_PLANE_Z(N, nz, __VA_ARGS__) } break;                       \
    case 64: { constexpr int N = 64; C3D_PLANE_Z(N, nz, __VA_ARGS__) } break;                       \
    case 96: { constexpr int N = 96; C3D_PLANE_Z(N, nz, __VA_ARGS__) } break;                       \
    case 128: { constexpr int N = 128; C3D_PLANE_Z(N, nz, __VA_ARGS__) } break;                     \
    default: return hipErrorInvalidValue;                                                           \
  }

// Rows from which a plane's kernels pay: their time is that of a plane's chain
// of passes up to 256 planes, that of the separate transforms grows with the
// rows, and the chain is long where eight threads walk long z columns.
// Projections, us, separate | plane's kernels (a time step in brackets): 32 x 128
// points 33 rows 30.8 | 35.3, 96 rows 40.4 | 42.4 [185 | 188], 128 rows 46.2 |
// 42.5; 16 x 128 points 96 rows 35.2 | 36.0, 128 rows 39.8 | 39.5; 48 x 96 points
// 48 rows 36.3 | 37.8 [156 | 158], 80 rows 41.4 | 41.6 [175 | 171].  All other
// shapes gain from 33 rows on (96 x 48 points, the least: 33 rows 33.0 | 33.3,
// 40 rows [144 | 143], 48 rows 35.6 | 35.4).
int plane_rows(int nxp, int nzp) {
  if (nzp >= 128) return 128;
  return nzp > 64 && nxp * nzp > 4096 ? 64 : 0;
}

}  // namespace

// C3D_PLANE_MAX lowers the largest plane (tuning knob; 0: none).
bool plane_fft(const DevGrid& g) {
  static const int most = [] {
    const char* e = getenv("C3D_PLANE_MAX");
    const int v = e ? atoi(e) : kPlaneMax;
    return v < kPlaneMax ? v : kPlaneMax;
  }();
  // With up to 32 rows the iteration count of an immersed body's solve follows
  // the last bits of the transforms and the elimination (two cylinders in 32
  // rows: 97 iterations with this path, the reference's 114 +- 2 without).
  return g.nxp <= 128 && g.nzp <= 128 && g.nxp * g.nzp <= most &&
         g.nym >= plane_rows(g.nxp, g.nzp) && planes_supported(g);
}

hipError_t launch_fwd_plane(const DevGrid& g, bool from_uvw, const double* U, const double* V,
                            const double* W, const double* rhs, cpx<double>* S, bool per,
                            hipStream_t s, const Planes* pl) {
  const dim3 grid(pl ? pl->n : g.nym);
  const int* list = pl ? pl->list : nullptr;
  const int pr = per ? 1 : 0;
  C3D_PLANE(g.nxp, g.nzp, {
    if (from_uvw)
      hipLaunchKernelGGL((k_fwd_plane<N, NZ, true>), grid, dim3(kPB), 0, s, g, U, V, W, rhs, S, pr, list);
    else
      hipLaunchKernelGGL((k_fwd_plane<N, NZ, false>), grid, dim3(kPB), 0, s, g, U, V, W, rhs, S, pr, list);
  });
  return hipGetLastError();
}

hipError_t launch_inv_plane(const DevGrid& g, int mode, const cpx<double>* S, double* out, double* P,
                            double dt, bool rk1, hipStream_t s, const Planes* pl) {
  if (mode != 0 && mode != 1) return hipErrorInvalidValue;
  const dim3 grid(pl ? pl->n : g.nym);
  const int* list = pl ? pl->list : nullptr;
  const int r = rk1 ? 1 : 0;
  C3D_PLANE(g.nxp, g.nzp, {
    if (mode == 1)
      hipLaunchKernelGGL((k_inv_plane<N, NZ, 1>), grid, dim3(kPB), 0, s, g, S, out, P, dt, r, list);
    else
      hipLaunchKernelGGL((k_inv_plane<N, NZ, 0>), grid, dim3(kPB), 0, s, g, S, out, P, dt, r, list);
  });
  return hipGetLastError();
}

}  // namespace c3d
