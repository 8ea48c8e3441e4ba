// Fused right-hand side and stage update of the RK3 time step
// (src/equations.f90:24-423, src/time_integration.f90:101-107, 130-136,
// 159-168) for gfx950, FP64, to round-off tolerance of the reference's
// operations: the spacing quotients are products with tabulated reciprocals
// and FMA contraction is on (rk3.hip keeps the bitwise form).
//
// One kernel per stage reads the stage's velocity through the LDS ring of
// the z march (rk3_march.hpp), evaluates F_s at each point and writes, in the same pass,
// X_s = X_0 + dt sum_l a_sl F_l into a second set of fields (the stage's
// input is still read by the neighbouring workgroups' halos, so the update
// cannot be in place).  F_s is stored for the later stages that use it.
#include "kernels.hpp"
#include "rk3_march.hpp"

namespace c3d {

namespace {

constexpr int kBf = 256;

// Wray coefficients as the reference writes them (src/time_integration.f90:
// 105-107, 134-136, 163-168): stage 2 uses F1, F2; stage 3 uses F1 and F3
// (the F2 coefficient of stage 3 is zero).
constexpr double kC11 = 8.0 / 15.0, kC21 = 1.0 / 4.0, kC22 = 5.0 / 12.0, kC31 = 1.0 / 4.0,
                 kC33 = 3.0 / 4.0;

// Stages 2 and 3 also read the point's own words, the step-start velocity and
// F1: loaded before the plane's barrier, used after its evaluation.
// MASK: H masks (none otherwise: six pointers less to keep in scalar registers,
// which stage 2 overflowed into 118 lane reads per plane).  96 to 104 VGPRs;
// held to 96 (5 waves per SIMD), stages 2 and 3 reload from scratch and take
// 903 and 731 instead of 817 and 667 us on 384x192x384 cells.
template <int KC, int STAGE, bool MASK>
__global__ __launch_bounds__(kBf) void k_rhs_stage(DevGrid g, RkStage a) {
  double xo[3] = {0.0, 0.0, 0.0}, f1[3] = {0.0, 0.0, 0.0};
  auto own = [&](int c, const double* Xo, const double* F1, int k, const Spot& s) {
    xo[c] = cell(Xo + (size_t)(k - 1) * s.po, s.o);
    f1[c] = cell(F1 + (size_t)(k - 2) * s.pf, s.f);
  };
  auto put = [&](int c, double* F, double* Xn, double x0, double Fv, int k, const Spot& s) {
    double x;
    if constexpr (STAGE == 1) x = x0 + (a.dt * kC11) * Fv;
    else if constexpr (STAGE == 2) x = xo[c] + a.dt * (kC21 * f1[c] + kC22 * Fv);
    else x = xo[c] + a.dt * (kC31 * f1[c] + kC33 * Fv);
    if constexpr (STAGE < 3) cell(F + (size_t)(k - 2) * s.pf, s.f) = Fv;
    cell(Xn + (size_t)(k - 1) * s.po, s.o) = x;
  };
  march<KC>(
      g, a.U, a.V, a.W,
      [&](int k, const Spot& su, const Spot& sv, const Spot& sw) {
        if constexpr (STAGE > 1) {
          if (su.in) own(0, a.Uo, a.F1u, k, su);
          if (sv.in) own(1, a.Vo, a.F1v, k, sv);
          if (sw.in && k <= g.nz - 1) own(2, a.Wo, a.F1w, k, sw);
        }
      },
      [&](const MarchAcc& A, const MarchGrid& G, int k, const Spot& su, const Spot& sv, const Spot& sw) {
        const int i = A.i, j = A.j;
        // U(2:nx-1, 2:nyg-1, 2:nzg-1)
        if (su.in)
          put(0, a.Fu, a.Un, A.U(i, j, k), rhs_u_at<true>(G, A, MASK ? a.Hu : nullptr, a.nu, a.dPdx, i, j, k), k, su);
        // V(2:nxg-1, 2:ny-1, 2:nzg-1)
        if (sv.in)
          put(1, a.Fv, a.Vn, A.V(i, j, k), rhs_v_at<true>(G, A, MASK ? a.Hv : nullptr, a.nu, a.dPdy, i, j, k), k, sv);
        // W(2:nxg-1, 2:nyg-1, 2:nz-1)
        if (sw.in && k <= g.nz - 1)
          put(2, a.Fw, a.Wn, A.W(i, j, k), rhs_w_at<true>(G, A, MASK ? a.Hw : nullptr, a.nu, a.dPdz, i, j, k), k, sw);
      });
}

inline dim3 gpts_f(int ni, int nj, int nk) { return dim3((ni + 63) / 64, (nj + 3) / 4, nk); }

template <int STAGE, int KC>
void launch_stage_kernel(const DevGrid& g, const RkStage& a, hipStream_t s) {
  const dim3 grid = gpts_f(g.nxg - 2, g.nyg - 2, (g.nzg - 2 + KC - 1) / KC);
  if (a.Hu && a.Hv && a.Hw)
    hipLaunchKernelGGL((k_rhs_stage<KC, STAGE, true>), grid, dim3(kBf), 0, s, g, a);
  else
    hipLaunchKernelGGL((k_rhs_stage<KC, STAGE, false>), grid, dim3(kBf), 0, s, g, a);
}

template <int KC>
hipError_t launch_stage(const DevGrid& g, int stage, const RkStage& a, hipStream_t s) {
  switch (stage) {
    case 1: launch_stage_kernel<1, KC>(g, a, s); break;
    case 2: launch_stage_kernel<2, KC>(g, a, s); break;
    case 3: launch_stage_kernel<3, KC>(g, a, s); break;
    default: return hipErrorInvalidValue;
  }
  return hipSuccess;
}

}  // namespace

hipError_t launch_rhs_stage(const DevGrid& g, int stage, const RkStage& a, hipStream_t s) {
  hipError_t e;
  switch (rhs_planes(g)) {
    case 2: e = launch_stage<2>(g, stage, a, s); break;
    case 4: e = launch_stage<4>(g, stage, a, s); break;
    default: e = launch_stage<8>(g, stage, a, s); break;
  }
  if (e != hipSuccess) return e;
  return hipGetLastError();
}

}  // namespace c3d
