// Tridiagonal solves along y of the spectral Poisson solver
// (src/poisson.f90:50-75) for gfx950, one system per mode (kx, kz) of the
// spectrum S[j][kx][kz].
#include "kernels.hpp"

namespace c3d {

namespace {

constexpr int kBlock = 256;

// ---------------------------------------------------------------------------
// Tridiagonal solve along y for every mode (kx, kz): src/poisson.f90:50-75.
// Matrix: D(j) = (Dyy(j,j) + kxx) + kzz, DL(j) = Dyy(j+1,j), DU(j) = Dyy(j,j+1),
// and D(2) *= 3/2 for the (0,0) mode.  Thomas elimination without
// pivoting (rows are diagonally dominant; agrees with partial pivoting to
// round-off).  One lane per mode, lanes along kz; CP holds the forward
// multipliers for the back substitution.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_tri64(DevGrid g, cpx<double>* __restrict__ S,
                                                  double* __restrict__ CP) {
  const int nzp = g.nzp, nym = g.nym;
  const size_t stride = (size_t)g.nxh * nzp;
  const size_t m = (size_t)blockIdx.x * kBlock + threadIdx.x;
  if (m >= stride) return;
  const int kx = (int)(m / nzp), kz = (int)(m % nzp);
  const double lamx = g.kxx[kx], lamz = g.kzz[kz];
  cpx<double>* s = S + m;
  double* cp = CP + m;

  double d0 = (g.dyy_d[0] + lamx) + lamz;
  if (kx == 0 && kz == 0) d0 = 1.5 * d0;
  cpx<double> bprev = s[0];
  double den = d0;
  double cprev = (nym > 1) ? g.dyy_u[0] / den : 0.0;
  bprev = cmk(bprev.x / den, bprev.y / den);
  s[0] = bprev;
  cp[0] = cprev;
  for (int jj = 1; jj < nym; jj++) {
    const double l = g.dyy_l[jj - 1];
    den = ((g.dyy_d[jj] + lamx) + lamz) - l * cprev;
    cpx<double> b = s[(size_t)jj * stride];
    b = cmk((b.x - l * bprev.x) / den, (b.y - l * bprev.y) / den);
    s[(size_t)jj * stride] = b;
    if (jj < nym - 1) {
      cprev = g.dyy_u[jj] / den;
      cp[(size_t)jj * stride] = cprev;
    }
    bprev = b;
  }
  cpx<double> xnext = bprev;
  for (int jj = nym - 2; jj >= 0; jj--) {
    const double c = cp[(size_t)jj * stride];
    cpx<double> b = s[(size_t)jj * stride];
    b = cmk(b.x - c * xnext.x, b.y - c * xnext.y);
    s[(size_t)jj * stride] = b;
    xnext = b;
  }
}

// ---------------------------------------------------------------------------
// Same system partitioned: each mode's rows are split into P (8 unless
// stated) parts of M rows, one lane per part, so every row is read once and
// written once and the whole part stays in registers.  A workgroup holds
// 256/P modes; each wave holds 16 of them for 4 of the parts (lane = part*16
// + mode), so that each row access is a run of 16 consecutive modes (256 bytes
// in FP64, 128 in FP32), and the waves of a mode group exchange interface
// rows through LDS.
//
// All quantities but the right-hand side are sums of non-negative terms.
// With the off-diagonals l, u >= 0 and the excess e = -(Dyy(j,j) + l + u) of
// a row (round-off of the table, from the host in extended precision) the
// system is (l + u + E) x_i = l x_{i-1} + u x_{i+1} - b_i, E = e - (kxx +
// kzz) >= 0.  Eliminating x_{i-1} with a row x = y + s x_a + c x_{i+1},
// d = 1 - s - c its deficit, leaves the pivot u + E + l (s + d): the pivots,
// the couplings and the deficits never come from a difference, where the
// elimination in terms of Dyy(j,j) loses the digits that the nearly singular
// low modes need.  Against an 80-bit solve (16 x 33..193 x 16 cells, random
// right-hand sides) the error is 5e-16, that of the plain elimination 6e-14.
//   pass 1  elimination inside the part with the unknown x_{a-1} above it:
//             x_i = y_i + sp_i x_{a-1} + cp_i x_{i+1}, deficit d_i,
//           and the first row's form x_a = G + V x_{a-1} + W x_{i+1}, deficit F
//   reduced the 2x8 interface equations of a mode, solved by its part-0
//           lane through LDS: L_q = x(first row of q), R_q = x(last row);
//           forward L_q = lam_q + mu_q L_{q+1}, R_q = rho_q + sig_q L_{q+1}
//           (deficits 1 - mu, t = 1 - sig carried), back L_q, then
//           R_{q-1} = rho_{q-1} + sig_{q-1} L_q
//   pass 2  back substitution with the boundary values x_{a-1} = R_{q-1},
//           x_b = L_{q+1}.
// Part 0 (l = 0 in its first row) and the last part (u = 0 in its last row)
// have no outside coupling, so the reduced system has no boundary terms.
// ---------------------------------------------------------------------------
// Mode selection of the partitioned solve (mixed precision runs the solve
// in two launches: FP32 arithmetic for the well-conditioned modes, FP64 for
// the (0,0) mode and the lowest |k|, whose systems are nearly singular).
constexpr int kTriAll = 0;   // every mode
constexpr int kTriHigh = 1;  // modes with |kxx + kzz| >= lam_thr
constexpr int kTriList = 2;  // the modes list[0 .. nlist)

// real: storage of the right-hand side read from S; rout: storage of the
// solution written to Sout (in place when both are the same array).
// P: parts per mode; MWX (when set) overrides the modes per wave.  PAD: the
// P*M rows hold g.nym <= P*M of the system and identity rows after them
// (x = 0, no coupling), which leave the other rows as they are: the last
// part may be short and parts after it empty.
// PLANES: S holds the planes of `Planes` only (slot[row], or -1: the row's
// right-hand side is zero and its solution is not stored).
template <typename real, typename acc, int M, int SEL, typename rout = real, int P = 8, int MWX = 0,
          bool PAD = false, bool PLANES = false>
__global__ __launch_bounds__(kBlock) void k_tri_part(DevGrid g, cpx<real>* S,
                                                     const int* __restrict__ list, int nlist,
                                                     double lam_thr, cpx<rout>* Sout,
                                                     const int* __restrict__ slot) {
  constexpr int N = P * M;        // rows
  // modes per wave: a row access of a wave is MW consecutive modes, 256
  // contiguous bytes of the input spectrum (16 FP64 or 32 FP32 complex)
  constexpr int MW = MWX ? MWX : 256 / (int)sizeof(cpx<real>);
  constexpr int PW = 64 / MW;     // parts per wave
  constexpr int WG = P / PW;      // waves that cover the parts of a mode group
  static_assert(WG * PW == P && kBlock / 64 % WG == 0, "waves must tile the parts");
  constexpr int MB = kBlock / P;  // modes per workgroup
  constexpr int CPT = M + 1;      // padded pitch of the row tables
  constexpr int RP = 10 * P + 1;  // padded pitch of a mode's interface rows
  __shared__ acc te[P * CPT], tl[P * CPT], tu[P * CPT];
  __shared__ acc red[MB * RP];
  const int tid = threadIdx.x;
  const int nrow = PAD ? g.nym : N;
  for (int e = tid; e < N; e += kBlock) {
    // three loads in flight at once: clamped in-bounds indices (dyy_l and
    // dyy_u hold nrow-1 entries), the end rows' zero couplings selected after
    const int q = e / M, r = e % M;
    const double ex = g.dyy_e[PAD ? min(e, nrow - 1) : e];
    const double l = g.dyy_l[e > 0 ? (PAD ? min(e - 1, nrow - 2) : e - 1) : 0];
    const double u = g.dyy_u[e < nrow - 1 ? e : 0];
    te[q * CPT + r] = (acc)ex;
    tl[q * CPT + r] = (e == 0 || (PAD && e >= nrow)) ? (acc)0 : (acc)l;
    tu[q * CPT + r] = (e >= nrow - 1) ? (acc)0 : (acc)u;
  }
  const int lane = tid & 63;
  const int wv = tid >> 6;
  const int p = (wv % WG) * PW + lane / MW;
  const int mb = (wv / WG) * MW + lane % MW;
  const int nzp = g.nzp;
  const size_t stride = (size_t)g.nxh * nzp;
  bool valid;
  size_t mv;
  if constexpr (SEL == kTriList) {
    const int e = blockIdx.x * MB + mb;
    valid = e < nlist;
    mv = valid ? (size_t)list[e] : 0;
  } else {
    const size_t m = (size_t)blockIdx.x * MB + mb;
    valid = m < stride;
    mv = valid ? m : 0;
  }
  const int kx = (int)(mv / nzp), kz = (int)(mv % nzp);
  if constexpr (SEL == kTriHigh) valid = valid && !(fabs(g.kxx[kx] + g.kzz[kz]) < lam_thr);
  const acc lam = (acc)(g.kxx[kx] + g.kzz[kz]);
  const bool zero_first = (kx == 0 && kz == 0 && p == 0);
  const int row0 = p * M;
  cpx<real>* s = S + mv + (PAD || PLANES ? 0 : (size_t)row0 * stride);
  cpx<rout>* so = Sout + mv + (PLANES ? 0 : (size_t)row0 * stride);
  int sl[PLANES ? M : 1];
  if constexpr (PLANES) {
#pragma unroll
    for (int r = 0; r < M; r++) {
      const int v = slot[PAD ? min(row0 + r, nrow - 1) : row0 + r];
      sl[r] = (PAD && row0 + r >= nrow) ? -1 : v;
    }
  }

  // All M rows are loaded unconditionally and converted afterwards: mv is a
  // valid mode for every lane, so the addresses stay in bounds, and without
  // a branch per row (whose FP32 -> FP64 conversion waited for its load) the
  // M loads of a lane are in flight together.
  acc yr[M], yi[M], cp[M], sp[M];
  {
    cpx<real> t[M];
#pragma unroll
    for (int r = 0; r < M; r++) {
      // a row without a plane reads the first plane and does not use it
      if constexpr (PLANES) t[r] = s[(size_t)max(sl[r], 0) * stride];
      else t[r] = s[(size_t)(PAD ? min(row0 + r, nrow - 1) : r) * stride];
    }
#pragma unroll
    for (int r = 0; r < M; r++) {
      bool in = valid && (!PAD || row0 + r < nrow);
      if constexpr (PLANES) in = valid && sl[r] >= 0;
      yr[r] = in ? -(acc)t[r].x : (acc)0;
      yi[r] = in ? -(acc)t[r].y : (acc)0;
    }
  }
  __syncthreads();  // row tables

  // pass 1
  const acc* re = te + p * CPT;
  const acc* rl = tl + p * CPT;
  const acc* ru = tu + p * CPT;
  acc gr = 0, gi = 0, v = 0, w = 0, f = 0, de = 0;
#pragma unroll
  for (int r = 0; r < M; r++) {
    acc E = re[r] - lam;
    if (PAD && row0 + r >= nrow) E = (acc)1;
    const acc l = rl[r], u = ru[r];
    if (r == 0) {
      if (zero_first) E = (acc)(-1.5 * g.dyy_d[0]) - u;  // D(2) *= 3/2
      const acc inv = (acc)1 / ((u + E) + l);
      yr[0] = yr[0] * inv;
      yi[0] = yi[0] * inv;
      sp[0] = l * inv;
      cp[0] = u * inv;
      de = E * inv;
      gr = yr[0];
      gi = yi[0];
      v = sp[0];
      w = cp[0];
      f = de;
    } else {
      const acc inv = (acc)1 / ((u + E) + l * (sp[r - 1] + de));
      yr[r] = (yr[r] + l * yr[r - 1]) * inv;
      yi[r] = (yi[r] + l * yi[r - 1]) * inv;
      sp[r] = (l * sp[r - 1]) * inv;
      cp[r] = u * inv;
      de = (E + l * de) * inv;
      gr += w * yr[r];
      gi += w * yi[r];
      v += w * sp[r];
      f += w * de;
      w = w * cp[r];
    }
  }
  acc* my = red + mb * RP + p * 10;
  my[0] = gr;
  my[1] = gi;
  my[2] = v;
  my[3] = w;
  my[4] = yr[M - 1];
  my[5] = yi[M - 1];
  my[6] = sp[M - 1];
  my[7] = cp[M - 1];
  my[8] = f;
  my[9] = de;
  __syncthreads();
  // reduced system: slot q holds GL(2) VL WL GR(2) VR WR FL FR on entry; the
  // forward sweep leaves lam(2) mu sig_{q-1} rho_{q-1}(2) in it and the
  // back sweep x_{a-1}(2) x_b(2) in positions 4..7
  if (p == 0) {
    acc* rs = red + mb * RP;
    acc rhr = 0, rhi = 0, sig = 0, t = 1;
    for (int q = 0; q < P; q++) {
      acc* e = rs + q * 10;
      const acc glr = e[0], gli = e[1], vl = e[2], wl = e[3];
      const acc grr = e[4], gri = e[5], vr = e[6], wr = e[7];
      const acc fl = e[8], fr = e[9];
      const acc iden = (acc)1 / ((fl + wl) + vl * t);
      const acc lr = (glr + vl * rhr) * iden, li = (gli + vl * rhi) * iden;
      const acc mu = wl * iden;
      e[0] = lr;
      e[1] = li;
      e[2] = mu;
      e[3] = sig;
      e[4] = rhr;
      e[5] = rhi;
      const acc dmu = (fl + vl * t) * iden;  // 1 - mu
      const acc nr = grr + vr * (rhr + sig * lr), ni = gri + vr * (rhi + sig * li);
      t = fr + vr * (t + sig * dmu);
      sig = wr + vr * (sig * mu);
      rhr = nr;
      rhi = ni;
    }
    acc lnr = 0, lni = 0;  // L_{q+1}
    for (int q = P - 1; q >= 0; q--) {
      acc* e = rs + q * 10;
      const acc lr = e[0] + e[2] * lnr, li = e[1] + e[2] * lni;  // L_q
      const acc ar = e[4] + e[3] * lr, ai = e[5] + e[3] * li;     // R_{q-1}
      e[6] = lnr;
      e[7] = lni;
      e[4] = ar;
      e[5] = ai;
      lnr = lr;
      lni = li;
    }
  }
  __syncthreads();
  // pass 2
  const acc xar = my[4], xai = my[5];
  acc xnr = my[6], xni = my[7];
#pragma unroll
  for (int r = M - 1; r >= 0; r--) {
    const acc xr = (yr[r] + sp[r] * xar) + cp[r] * xnr;
    const acc xi = (yi[r] + sp[r] * xai) + cp[r] * xni;
    if constexpr (PLANES) {
      if (valid && sl[r] >= 0) so[(size_t)sl[r] * stride] = cmk((rout)xr, (rout)xi);
    } else if (valid && (!PAD || row0 + r < nrow)) {
      so[(size_t)r * stride] = cmk((rout)xr, (rout)xi);
    }
    xnr = xr;
    xni = xi;
  }
}

}  // namespace

// 16 parts of nym/16 rows (152 VGPRs at nym = 192: 3 waves per SIMD against
// 2 with 8 parts of 24 rows).
#define C3D_DISPATCH_M16(nym, BODY)                  \
  switch (nym) {                                     \
    case 64: { constexpr int MM = 4; BODY; } break;    \
    case 128: { constexpr int MM = 8; BODY; } break;   \
    case 192: { constexpr int MM = 12; BODY; } break;  \
    default: return hipErrorInvalidValue;            \
  }

namespace {
// FP64 solve of every mode in P parts of MM rows, MW modes per wave.
template <int P, int MM, int MW, bool PAD>
void tri64_parts(const DevGrid& g, cpx<double>* S, hipStream_t s, const Planes* pl) {
  constexpr int MB = kBlock / P;
  const size_t nm = (size_t)g.nxh * g.nzp;
  const dim3 grid((unsigned)((nm + MB - 1) / MB));
  if (pl)
    hipLaunchKernelGGL((k_tri_part<double, double, MM, kTriAll, double, P, MW, PAD, true>), grid,
                       dim3(kBlock), 0, s, g, S, nullptr, 0, 0.0, S, pl->slot);
  else
    hipLaunchKernelGGL((k_tri_part<double, double, MM, kTriAll, double, P, MW, PAD>), grid,
                       dim3(kBlock), 0, s, g, S, nullptr, 0, 0.0, S, nullptr);
}
// Row counts of the plain elimination, one lane per mode: above what the
// lanes of a workgroup hold in registers, and up to 32 rows, where the number
// of iterations of an immersed body's solve is held to the reference's: it
// follows the rounding of the elimination (two cylinders in 32 rows: 114
// iterations with the reference's, 84 with the partitioned solve).
constexpr int kTriMinRows = 33, kTriMaxRows = 32 * 24;
}  // namespace

bool tri_needs_scratch(const DevGrid& g) { return g.nym < kTriMinRows || g.nym > kTriMaxRows; }

bool planes_supported(const DevGrid& g) { return !tri_needs_scratch(g); }

hipError_t launch_tri(const DevGrid& g, cpx<double>* S, double* CP, hipStream_t s, const Planes* pl) {
  if (pl && (pl->n < 1 || !planes_supported(g))) return hipErrorInvalidValue;
  const size_t nm = (size_t)g.nxh * g.nzp;
  // 64, 128 and 192 rows fill 8 parts exactly.
  if (g.nym % 64 == 0 && g.nym <= 192) {
    switch (g.nym) {
      case 64: tri64_parts<8, 8, 16, false>(g, S, s, pl); break;
      case 128: tri64_parts<8, 16, 16, false>(g, S, s, pl); break;
      default: tri64_parts<8, 24, 16, false>(g, S, s, pl); break;
    }
    return hipGetLastError();
  }
  if (tri_needs_scratch(g)) {
    hipLaunchKernelGGL(k_tri64, dim3((unsigned)((nm + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, g, S, CP);
    return hipGetLastError();
  }
  // Any other row count: 16 parts of the next row count built, 32 parts above
  // 384 rows (a lane's rows in registers: 24 at most).  100 rows of 49 x 48
  // modes: 6.6 us, one lane per mode 72 us; 96 rows of 65 x 128 modes: 10.3
  // against 68 us.
  const int per = (g.nym + 15) / 16;
  if (per <= 4) tri64_parts<16, 4, 16, true>(g, S, s, pl);
  else if (per <= 5) tri64_parts<16, 5, 16, true>(g, S, s, pl);
  else if (per <= 6) tri64_parts<16, 6, 16, true>(g, S, s, pl);
  else if (per <= 7) tri64_parts<16, 7, 16, true>(g, S, s, pl);
  else if (per <= 8) tri64_parts<16, 8, 16, true>(g, S, s, pl);
  else if (per <= 10) tri64_parts<16, 10, 16, true>(g, S, s, pl);
  else if (per <= 12) tri64_parts<16, 12, 16, true>(g, S, s, pl);
  else if (per <= 16) tri64_parts<16, 16, 16, true>(g, S, s, pl);
  else if (per <= 20) tri64_parts<16, 20, 16, true>(g, S, s, pl);
  else if (per <= 24) tri64_parts<16, 24, 16, true>(g, S, s, pl);
  else if (per <= 32) tri64_parts<32, 16, 8, true>(g, S, s, pl);
  else tri64_parts<32, 24, 8, true>(g, S, s, pl);
  return hipGetLastError();
}

bool tri_part_supported(const DevGrid& g) { return g.nym == 64 || g.nym == 128 || g.nym == 192; }

namespace {
// The FP32 solves of launch_tri32 in P parts of MM rows (16 modes per wave
// when P = 16).
template <int P, int MM>
hipError_t tri32_parts(const DevGrid& g, cpx<float>* S, const int* low, int nlow, double lam_thr,
                       hipStream_t s) {
  constexpr int MWX = P == 16 ? 16 : 0;
  constexpr int MB = kBlock / P;
  const size_t nm = (size_t)g.nxh * g.nzp;
  const dim3 grid((unsigned)((nm + MB - 1) / MB));
  if (!low) {  // FP64 arithmetic on every mode
    hipLaunchKernelGGL((k_tri_part<float, double, MM, kTriAll, float, P, MWX>), grid, dim3(kBlock),
                       0, s, g, S, nullptr, 0, 0.0, S, nullptr);
    return hipGetLastError();
  }
  if (nlow <= 0) return hipErrorInvalidValue;  // the (0,0) mode is always a low mode
  const dim3 gridl((unsigned)((nlow + MB - 1) / MB));
  hipLaunchKernelGGL((k_tri_part<float, float, MM, kTriHigh, float, P, MWX>), grid, dim3(kBlock), 0,
                     s, g, S, nullptr, 0, lam_thr, S, nullptr);
  hipLaunchKernelGGL((k_tri_part<float, double, MM, kTriList, float, P, MWX>), gridl, dim3(kBlock),
                     0, s, g, S, low, nlow, 0.0, S, nullptr);
  return hipGetLastError();
}
}  // namespace

hipError_t launch_tri32(const DevGrid& g, cpx<float>* S, const int* low, int nlow, double lam_thr,
                        hipStream_t s) {
  // 192 rows as 16 parts of 12: 8 parts of 24 with all of a lane's FP32 rows
  // in flight need more than 256 registers (one wave per SIMD)
  switch (g.nym) {
    case 64: return tri32_parts<8, 8>(g, S, low, nlow, lam_thr, s);
    case 128: return tri32_parts<8, 16>(g, S, low, nlow, lam_thr, s);
    case 192: return tri32_parts<16, 12>(g, S, low, nlow, lam_thr, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_tri32to64(const DevGrid& g, cpx<float>* S32, cpx<double>* S64, hipStream_t s) {
  // FP32 right-hand side, FP64 solution: 16 parts of nym/16 rows, 16 modes
  // per wave (94 against 99 us with 8 parts at 384x193x384; the FP64 solve
  // gains nothing from it and keeps 8 parts)
  const size_t nm = (size_t)g.nxh * g.nzp;
  constexpr int MB = kBlock / 16;
  const dim3 grid((unsigned)((nm + MB - 1) / MB));
  C3D_DISPATCH_M16(g.nym, hipLaunchKernelGGL((k_tri_part<float, double, MM, kTriAll, double, 16, 16>),
                                             grid, dim3(kBlock), 0, s, g, S32, nullptr, 0, 0.0, S64, nullptr));
  return hipGetLastError();
}

}  // namespace c3d
