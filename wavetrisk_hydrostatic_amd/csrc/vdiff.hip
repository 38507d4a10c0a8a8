// Vertical diffusion of an ocean column (wtg_vertical_diffusion):
// vertical_diffusion (vert_diffusion.f90:66-86) with the analytic eddy
// coefficients or the one-equation TKE closure (turbulent_diffusion,
// vert_diffusion.f90:88-264, with N_sq, l_scales, Richardson, Prandtl, Kv_tke
// and Kt_tke at 438-573), then the backward-Euler steps of the buoyancy
// (backwards_euler_temp, 266-355) and of the edge velocities
// (backwards_euler_velo, 357-424), each through LAPACK's dgtsv (dgtsv.f90).
//
// Two launches, one thread per column (grid y = ensemble member).  The first
// computes Kt, Kv and the TKE of every owned node and pole master; it reads
// the velocities of the node's six edges (its kinetic energy, io.f90:169-206),
// so it must finish before any velocity changes.  The second steps the
// buoyancy of the same columns and the velocities of each owned node's RT,
// DG and UP edges (with the node's Kv and the layer thicknesses averaged with
// the edge's other node).  Up to 32 layers a column stays in registers (unrolled
// loops, sizes 16, 24, 32); above, and where dgtsv would pivot, its arrays are
// private (up to WTG_REMAP_MAX_LAYERS layers).  FP64 in the reference's
// evaluation order without FMA contraction.  The analytic profiles call exp, whose last bit may
// differ from the host library's; everything else equals the oracle bit for bit.
#include <hip/hip_runtime.h>

#include "ctx.h"
#include "exact_div.h"

namespace {

constexpr int H = wtg::HALO;
constexpr int VMAX = WTG_REMAP_MAX_LAYERS;
constexpr int VT = 64;  // threads per block: one wave, since the column arrays are large

struct VdArgs {
  int n, S, L, istep;
  int64_t NC, spole, npole;
  double dt, rho0, grav;
  wtg_vdiff p;
  const double *len, *ped, *hinv, *topo, *eta;  // topo, eta [members][NC] (eta may be null)
  const double* force;                          // [members][6][NC]
  double *m, *t, *u;                            // the state slot
  double *kt, *kv, *tke;                        // [members][L + 1][NC], [members][L][NC]
  unsigned long long* left;                     // lanes that a register kernel leaves, a word per block
};

// LAPACK dgtsv with one right-hand side on rows 1..n of 1-based arrays.  The
// current row's eliminated diagonal and right-hand side, and the last two
// solution values of the back substitution, ride in registers (the arrays
// live in scratch memory, and a reload of what the previous row just stored
// would put a memory round trip on every step of the sweep); every update is
// also stored, so the arrays hold what the library's would, an early return
// at a zero pivot included.
__device__ void dgtsv(int n, double* __restrict__ dl, double* __restrict__ d, double* __restrict__ du,
                      double* __restrict__ b) {
  double di = d[1], bi = b[1];
  for (int i = 1; i <= n - 1; ++i) {
    const double dli = dl[i], dui = du[i], dn = d[i + 1], bn = b[i + 1];
    if (fabs(di) >= fabs(dli)) {
      if (di == 0.0) return;
      const double fact = dli / di;
      di = dn - fact * dui;
      bi = bn - fact * bi;
      d[i + 1] = di;
      b[i + 1] = bi;
      if (i <= n - 2) dl[i] = 0.0;
    } else {  // interchange rows i and i + 1
      const double fact = di / dli;
      d[i] = dli;
      di = dui - fact * dn;
      d[i + 1] = di;
      if (i <= n - 2) {
        dl[i] = du[i + 1];
        du[i + 1] = -fact * dl[i];
      }
      du[i] = dn;
      b[i] = bn;
      bi = bi - fact * bn;
      b[i + 1] = bi;
    }
  }
  if (di == 0.0) return;  // d(n)
  double x1 = bi / di, x2 = 0.0;
  b[n] = x1;
  if (n > 1) {
    const double x = (b[n - 1] - du[n - 1] * x1) / d[n - 1];
    b[n - 1] = x;
    x2 = x1;
    x1 = x;
  }
  for (int i = n - 2; i >= 1; --i) {
    const double x = (b[i] - du[i] * x1 - dl[i] * x2) / d[i];
    b[i] = x;
    x2 = x1;
    x1 = x;
  }
}

struct SolveWork {
  double dg[VMAX + 2], dl[VMAX + 2], du[VMAX + 2], r[VMAX + 2];  // the rows, built only for the full dgtsv
  double Dp[VMAX + 2], Up[VMAX + 2], X[VMAX + 2];                // the elimination's diagonal, super-diagonal, rhs
};

// Solves the rows with dgtsv's arithmetic: while no row interchange or zero
// pivot occurs, the elimination keeps only its diagonal, super-diagonal and
// right-hand side (what dgtsv's no-interchange branch computes, the zeroed
// sub-diagonal entering the back substitution as 0.0 * x); otherwise the
// rows are built and dgtsv runs in full.  The solution is left in X[1..n].
// Rows gives reset(zs) and next(lo, dg, up, r), row after row from 1.
template <class Rows>
__device__ void solve_rows(int n, Rows& rows, double zs, SolveWork& w) {
  double lo, dg, up, r;
  rows.reset(zs);
  rows.next(lo, dg, up, r);
  double di = dg, xi = r, ui = up;
  w.Dp[1] = di;
  w.X[1] = xi;
  w.Up[1] = ui;
  bool fast = true;
  for (int i = 1; i <= n - 1; ++i) {
    rows.next(lo, dg, up, r);  // row i + 1: lo is dgtsv's dl(i)
    if (!(fabs(di) >= fabs(lo)) || di == 0.0) {
      fast = false;
      break;
    }
    const double fact = lo / di;
    di = dg - fact * ui;
    xi = r - fact * xi;
    ui = up;
    w.Dp[i + 1] = di;
    w.X[i + 1] = xi;
    w.Up[i + 1] = ui;
  }
  if (fast && di != 0.0) {
    double x1 = xi / di, x2 = 0.0;
    w.X[n] = x1;
    if (n > 1) {
      const double x = (w.X[n - 1] - w.Up[n - 1] * x1) / w.Dp[n - 1];
      w.X[n - 1] = x;
      x2 = x1;
      x1 = x;
    }
    for (int i = n - 2; i >= 1; --i) {
      const double x = (w.X[i] - w.Up[i] * x1 - 0.0 * x2) / w.Dp[i];
      w.X[i] = x;
      x2 = x1;
      x1 = x;
    }
    return;
  }
  rows.reset(zs);
  for (int k = 1; k <= n; ++k) {
    rows.next(lo, dg, up, r);
    if (k >= 2) w.dl[k - 1] = lo;
    w.dg[k] = dg;
    if (k <= n - 1) w.du[k] = up;
    w.r[k] = r;
  }
  dgtsv(n, w.dl, w.dg, w.du, w.r);
  for (int k = 1; k <= n; ++k) w.X[k] = w.r[k];
}

// the column of thread tid: owned nodes, then the south and north pole masters
__device__ __forceinline__ int64_t column(const VdArgs& a, int64_t tid, bool& pole) {
  const int64_t nown = (int64_t)10 * a.n * a.n;
  pole = tid >= nown;
  if (pole) return tid == nown ? a.spole : a.npole;
  const int lz = (int)(tid / ((int64_t)a.n * a.n)), r = (int)(tid % ((int64_t)a.n * a.n));
  return (int64_t)lz * a.S * a.S + (int64_t)(r / a.n + H) * a.S + (r % a.n + H);
}

__device__ __forceinline__ double prandtl(double Ri) {
  if (Ri < 0.2) return 1.0;
  if (Ri >= 0.2 && Ri <= 2.0) return 5.0 * Ri;
  return 10.0;
}

__device__ __forceinline__ double kv_tke(const wtg_vdiff& p, double e, double lk) {
  return fmin(p.Kv_max, fmax(p.C_k * lk * sqrt(e), p.Kv_min));
}

__device__ __forceinline__ double kt_tke(const wtg_vdiff& p, double Kv, double Nsq, double Ri) {
  double kt = fmin(p.Kt_max, fmax(Kv / prandtl(Ri), p.Kt_min));
  if (p.enhance_diff && Nsq <= p.Nsq_min) kt = p.Kt_enh;
  return kt;
}

__device__ __forceinline__ double free_surface(const VdArgs& a, const double* m, double zs, int64_t c) {
  double depth = 0.0;
  for (int k = 0; k < a.L; ++k) depth = depth + (0.0 + m[(int64_t)k * a.NC + c]) / (a.rho0 * 1.0);
  return depth + zs;
}

struct TkeWork {
  double dz[VMAX + 2], dU2[VMAX + 2], Nsq[VMAX + 2], e[VMAX + 2], leps[VMAX + 2], lk[VMAX + 2], dn[VMAX + 2];
};

// l_scales (vert_diffusion.f90:502-536) on [0..L]: the upward sweep of the
// mixing length from the bottom, then the downward one from the surface with
// the two length scales taken as it passes; the first-order length
// sqrt(2 e / max(N^2, Neps_sq)) is formed where each sweep needs it, and the
// running minima ride in registers (the same numbers as the reference's
// array passes)
__device__ void l_scales(const VdArgs& a, double tau, TkeWork& w) {
  const wtg_vdiff& p = a.p;
  const int L = a.L;
  double prev = p.l_0;
  w.dn[0] = prev;
  for (int l = 1; l <= L; ++l) {
    const double first = sqrt(2.0 * w.e[l] / fmax(w.Nsq[l], p.Neps_sq));
    w.dn[l] = prev = fmin(first, prev + w.dz[l]);
  }
  prev = fmax(p.l_0, p.kappa_VK * p.C_l / (a.rho0 * a.grav) * tau);  // l_up at the surface
  w.leps[L] = fmax(p.l_min, sqrt(prev * w.dn[L]));
  w.lk[L] = fmax(p.l_min, fmin(prev, w.dn[L]));
  for (int l = L - 1; l >= 0; --l) {
    const double first = sqrt(2.0 * w.e[l] / fmax(w.Nsq[l], p.Neps_sq));
    prev = fmin(first, prev + w.dz[l + 1]);
    w.leps[l] = fmax(p.l_min, sqrt(prev * w.dn[l]));
    w.lk[l] = fmax(p.l_min, fmin(prev, w.dn[l]));
  }
}

// Rows 1..L-1 of the TKE system (turbulent_diffusion), generated in order:
// the sources S1, S2 and the coefficients (coeff reads dzl at the row's own
// l) with the expressions of the reference's arrays
struct TkeRows {
  const VdArgs& a;
  const double *kv, *kt;
  int64_t c;
  const TkeWork& w;
  int l;
  __device__ void reset(double) { l = 0; }
  __device__ void next(double& lo, double& dg, double& up, double& r) {
    const wtg_vdiff& p = a.p;
    const int64_t NC = a.NC;
    const int last = a.L - 1;
    const double dt = a.dt;
    ++l;
    const double KV = kv[(int64_t)l * NC + c], KT = kt[(int64_t)l * NC + c];
    const double turb = w.e[l] == 0.0 ? 0.0 : p.C_eps * sqrt(w.e[l]) / w.leps[l];
    double S1 = KV * w.dU2[l] - KT * w.Nsq[l], S2;
    if (p.patankar && S1 <= 0.0) {
      S1 = KV * w.dU2[l];
      S2 = -turb - KT * w.Nsq[l] / w.e[l];
    } else {
      S2 = -turb;
    }
    const double dzl = 0.5 * (w.dz[l] + w.dz[l + 1]);
    up = l <= last - 1 ? -(dt * p.C_e * (0.5 * (KV + kv[(int64_t)(l + 1) * NC + c])) / (dzl * w.dz[l + 1])) : 0.0;
    lo = l >= 2 ? -(dt * p.C_e * (0.5 * (KV + kv[(int64_t)(l - 1) * NC + c])) / (dzl * w.dz[l])) : 0.0;
    if (l == 1)
      dg = 1.0 - up - dt * S2;
    else if (l < last)
      dg = 1.0 - (up + lo) - dt * S2;
    else
      dg = 1.0 - lo - dt * S2;
    r = w.e[l] + dt * S1;
  }
};

// turbulent_diffusion of one column in private arrays
__device__ __forceinline__ void turbulent_column(const VdArgs& a, int64_t mb, int64_t c) {
  const int L = a.L;
  const int64_t NC = a.NC;
  const double* m = a.m + mb * L * NC;
  const double* t = a.t + mb * L * NC;
  const double* u = a.u + mb * 3 * L * NC;
  double* kt = a.kt + mb * (L + 1) * NC;
  double* kv = a.kv + mb * (L + 1) * NC;
  double* tke = a.tke + mb * L * NC;
  const double zs = a.topo[mb * NC + c];
  const double tau = a.force[(mb * 6 + 2) * NC + c];
  const wtg_vdiff& p = a.p;
  if (!p.tke_closure) {
    const double eta = a.eta ? a.eta[mb * NC + c] : free_surface(a, m, zs, c);
    const double e20 = -20.0;
    double z = zs;
    kt[c] = p.Kt_min + p.Kt_max * exp(e20 * (z - eta) / p.mixed_layer);
    kv[c] = p.Kv_min + p.Kv_max * exp(e20 * (z - eta) / p.mixed_layer);
    for (int l = 1; l <= L; ++l) {
      z = z + (0.0 + m[(int64_t)(l - 1) * NC + c]) / (a.rho0 * 1.0);
      kt[(int64_t)l * NC + c] = p.Kt_min + p.Kt_max * exp(e20 * (z - eta) / p.mixed_layer);
      kv[(int64_t)l * NC + c] = p.Kv_min + p.Kv_max * exp(e20 * (z - eta) / p.mixed_layer);
    }
    return;
  }
  TkeWork w;
  // init_diffuse: dz and |u| (twice the TRiSK kinetic energy) per layer
  const int64_t W = c - 1, SW = c - a.S - 1, Sx = c - a.S;
  double umag = 0.0;  // |u| of the layer below, in a register
  for (int k = 1; k <= L; ++k) {
    w.dz[k] = (0.0 + m[(int64_t)(k - 1) * NC + c]) / (a.rho0 * 1.0);
    const double* uk = u + (int64_t)(k - 1) * 3 * NC;
    const double pRT = uk[c] * a.len[c], pDG = uk[NC + c] * a.len[NC + c], pUP = uk[2 * NC + c] * a.len[2 * NC + c];
    const double dRT = uk[c] * a.ped[c], dDG = uk[NC + c] * a.ped[NC + c], dUP = uk[2 * NC + c] * a.ped[2 * NC + c];
    const double pUPS = uk[2 * NC + Sx] * a.len[2 * NC + Sx], pDGSW = uk[NC + SW] * a.len[NC + SW];
    const double pRTW = uk[W] * a.len[W];
    const double dRTW = uk[W] * a.ped[W], dDGSW = uk[NC + SW] * a.ped[NC + SW], dUPS = uk[2 * NC + Sx] * a.ped[2 * NC + Sx];
    const double ke =
        (pUP * dUP + pDG * dDG + pRT * dRT + pUPS * dUPS + pDGSW * dDGSW + pRTW * dRTW) * a.hinv[c] / 4.0;
    const double um = sqrt(2.0 * ke);
    if (k >= 2) {  // dUdZ_sq at the interface below layer k
      const double q = (um - umag) / (0.5 * (w.dz[k - 1] + w.dz[k]));
      w.dU2[k - 1] = q * q;
    }
    umag = um;
  }
  w.dU2[0] = 0.0;
  w.dU2[L] = 0.0;
  for (int l = 0; l <= L; ++l) {
    const int k = l == 0 ? 1 : l == L ? L - 1 : l;  // N_sq at the interface above layer k
    const double bb = t[(int64_t)(k - 1) * NC + c] / (0.0 + m[(int64_t)(k - 1) * NC + c]);
    const double ba = t[(int64_t)k * NC + c] / (0.0 + m[(int64_t)k * NC + c]);
    w.Nsq[l] = a.grav * (ba - bb) / (0.5 * (w.dz[k] + w.dz[k + 1]));
  }
  w.e[0] = p.e_0;
  for (int l = 1; l <= L; ++l) w.e[l] = fmax(tke[(int64_t)(l - 1) * NC + c], p.e_min);
  l_scales(a, tau, w);
  if (a.istep == 1)
    for (int l = 0; l <= L; ++l) {
      const double Ri = w.Nsq[l] / (w.dU2[l] + p.eps_s);
      const double v = kv_tke(p, w.e[l], w.lk[l]);
      kv[(int64_t)l * NC + c] = v;
      kt[(int64_t)l * NC + c] = kt_tke(p, v, w.Nsq[l], Ri);
    }
  // the TKE system's backward-Euler step
  SolveWork sw;
  TkeRows rows{a, kv, kt, c, w, 0};
  solve_rows(L - 1, rows, 0.0, sw);
  w.e[0] = p.e_0;
  for (int l = 1; l <= L - 1; ++l) w.e[l] = p.patankar ? sw.X[l] : fmax(sw.X[l], p.e_min);
  w.e[L] = fmax(p.C_srf * tau / a.rho0, p.e_min_srf);
  // update_Kv_Kt
  l_scales(a, tau, w);
  for (int l = 0; l <= L; ++l) {
    const double Ri = w.Nsq[l] / (w.dU2[l] + p.eps_s);
    const double v = kv_tke(p, w.e[l], w.lk[l]);
    kv[(int64_t)l * NC + c] = v;
    kt[(int64_t)l * NC + c] = kt_tke(p, v, w.Nsq[l], Ri);
  }
  for (int l = 1; l <= L; ++l) tke[(int64_t)(l - 1) * NC + c] = fmax(w.e[l], p.e_min);
}

// turbulent_diffusion of every owned node and pole master: the analytic
// profiles, and the TKE closure for any number of layers
__global__ __launch_bounds__(VT) void vd_turbulent_kernel(VdArgs a) {
  const int64_t tid = (int64_t)blockIdx.x * VT + threadIdx.x;
  if (tid >= (int64_t)10 * a.n * a.n + 2) return;
  bool pole;
  turbulent_column(a, blockIdx.y, column(a, tid, pole));
}

// What the register kernels left, a lane a system: a wave looks at LEFT words
// together and takes those that are not empty one after another, so that a
// grid whose systems are all left still has VT times its words in flight.
constexpr int LEFT = 8;
template <class F>
__device__ __forceinline__ void each_left(const unsigned long long* left, int nwords, const F& take) {
  const int lane = threadIdx.x, first = blockIdx.x * LEFT;
  const unsigned long long mine = lane < LEFT && first + lane < nwords ? left[first + lane] : 0;
  for (unsigned long long some = __ballot(mine != 0); some; some &= some - 1) {
    const int k = __builtin_ctzll(some);
    if (__shfl(mine, k) >> lane & 1) take(first + k);
  }
}

// the columns that vd_tke_kernel left
__global__ __launch_bounds__(VT) void vd_tke_left_kernel(VdArgs a, int nblocks) {
  each_left(a.left + (int64_t)blockIdx.y * nblocks, nblocks, [&](int word) {
    bool pole;
    turbulent_column(a, blockIdx.y, column(a, (int64_t)word * VT + threadIdx.x, pole));
  });
}

// The TKE closure for at most LM layers (and istep > 1, whose coefficients are
// known before the rows), the column in registers: the loops over levels are
// unrolled and run in four sweeps,
//   down  the length from the surface,
//   up    the length from the bottom, the rows and their elimination,
//   down  the back substitution and the new length from the surface,
//   up    the new length from the bottom and the coefficients,
// with dUdZ^2, N^2, one length or pivot and the right-hand side per level kept
// between them.  Same operations as turbulent_column, to which a system that
// dgtsv would pivot is left (vd_tke_left_kernel), and one with an infinity or
// NaN (a massless layer).  Bound by the latency of its divisions and square roots at
// one or two waves per SIMD.  J8 L30: 1.79 -> 1.07 ms
// (one wave per SIMD); the whole call 3.48 -> 1.85 ms, at J7 L20 0.69 -> 0.30 ms.
template <int LM>
__global__ __launch_bounds__(VT, LM > 24 ? 1 : 2) void vd_tke_kernel(VdArgs a) {
  const int64_t tid = (int64_t)blockIdx.x * VT + threadIdx.x;
  const bool live = tid < (int64_t)10 * a.n * a.n + 2;
  bool pole;
  const int64_t c = column(a, live ? tid : 0, pole);
  const int L = a.L;
  const int64_t NC = a.NC, mb = blockIdx.y;
  const double* m = a.m + mb * L * NC + c;
  const double* t = a.t + mb * L * NC + c;
  const double* u = a.u + mb * 3 * L * NC;
  double* kt = a.kt + mb * (L + 1) * NC + c;
  double* kv = a.kv + mb * (L + 1) * NC + c;
  double* tke = a.tke + mb * L * NC + c;
  const double tau = a.force[(mb * 6 + 2) * NC + c];
  const wtg_vdiff& p = a.p;
  const double rho = a.rho0 * 1.0, rrho = 1.0 / rho, dt = a.dt;
  const int64_t W = c - 1, SW = c - a.S - 1, Sx = c - a.S;
  // dUdZ^2 and N^2 at the interfaces 1 .. L - 1
  double dU2[LM], Nsq[LM], A[LM + 1], X[LM];
  bool fast = true;
  {
    const double l0 = a.len[c], l1 = a.len[NC + c], l2 = a.len[2 * NC + c], p0 = a.ped[c], p1 = a.ped[NC + c];
    const double p2 = a.ped[2 * NC + c], lS = a.len[2 * NC + Sx], pS = a.ped[2 * NC + Sx], lSW = a.len[NC + SW];
    const double pSW = a.ped[NC + SW], lW = a.len[W], pW = a.ped[W], hi = a.hinv[c];
    double umag = 0.0, dzp = 0.0, bp = 0.0;
    constexpr int CH = 4;
#pragma unroll
    for (int k0 = 0; k0 < LM; k0 += CH) {
      if (k0 < L) {
        double v[CH][6], mm[CH], tt[CH];
#pragma unroll
        for (int j = 0; j < CH; ++j) {
          const int64_t k = min(k0 + j, L - 1);
          const double* uk = u + 3 * k * NC;
          v[j][0] = uk[c];
          v[j][1] = uk[NC + c];
          v[j][2] = uk[2 * NC + c];
          v[j][3] = uk[2 * NC + Sx];
          v[j][4] = uk[NC + SW];
          v[j][5] = uk[W];
          mm[j] = m[k * NC];
          tt[j] = t[k * NC];
        }
#pragma unroll
        for (int j = 0; j < CH; ++j) {
          const int k = k0 + j;
          const double dz = div_by(0.0 + mm[j], rho, rrho);
          const double pRT = v[j][0] * l0, pDG = v[j][1] * l1, pUP = v[j][2] * l2;
          const double dRT = v[j][0] * p0, dDG = v[j][1] * p1, dUP = v[j][2] * p2;
          const double pUPS = v[j][3] * lS, pDGSW = v[j][4] * lSW, pRTW = v[j][5] * lW;
          const double dRTW = v[j][5] * pW, dDGSW = v[j][4] * pSW, dUPS = v[j][3] * pS;
          const double ke =
              (pUP * dUP + pDG * dDG + pRT * dRT + pUPS * dUPS + pDGSW * dDGSW + pRTW * dRTW) * hi / 4.0;
          const double um = sqrt(2.0 * ke), b = tt[j] / (0.0 + mm[j]);
          if (k >= 1) {
            const double dzm = 0.5 * (dzp + dz), rz = 1.0 / dzm, q = div_by(um - umag, dzm, rz);
            dU2[k - 1] = q * q;
            Nsq[k - 1] = div_by(a.grav * (b - bp), dzm, rz);
            // div_by gives NaN where a division gives an infinity
            if (k < L) fast = fast && fabs(dU2[k - 1]) < INFINITY && fabs(Nsq[k - 1]) < INFINITY;
          }
          umag = um;
          dzp = dz;
          bp = b;
        }
      }
    }
  }
#define DZ(k) div_by(0.0 + m[(int64_t)((k) - 1) * NC], rho, rrho)
#define E_OLD(l) fmax(tke[(int64_t)((l) - 1) * NC], p.e_min)
#define FIRST(e, nsq) sqrt(2.0 * (e) / fmax(nsq, p.Neps_sq))
  // interface l has dU2[l - 1], Nsq[l - 1]; the ends take their neighbours' N^2
  const double up_top = fmax(p.l_0, p.kappa_VK * p.C_l / (a.rho0 * a.grav) * tau);
  {
    double prev = up_top;
#pragma unroll
    for (int l = LM - 1; l >= 1; --l)
      if (l < L) {
        prev = fmin(FIRST(E_OLD(l), Nsq[l - 1]), prev + DZ(l + 1));
        A[l] = prev;
      }
  }
  double di = 0.0, xi = 0.0, ui = 0.0;
  {
    double dn = p.l_0, dzc = DZ(1), Kvp = 0.0, Kvc = kv[NC];
#pragma unroll
    for (int l = 1; l < LM; ++l)
      if (l < L) {
        const double KT = kt[(int64_t)l * NC], KV = Kvc, Kvn = kv[(int64_t)(l + 1) * NC];
        const double e = E_OLD(l), dzn = DZ(l + 1), N2 = Nsq[l - 1], U2 = dU2[l - 1];
        dn = fmin(FIRST(e, N2), dn + dzc);
        const double leps = fmax(p.l_min, sqrt(A[l] * dn));
        const double turb = e == 0.0 ? 0.0 : p.C_eps * sqrt(e) / leps;
        double S1 = KV * U2 - KT * N2, S2;
        if (p.patankar && S1 <= 0.0) {
          S1 = KV * U2;
          S2 = -turb - KT * N2 / e;
        } else {
          S2 = -turb;
        }
        const double dzl = 0.5 * (dzc + dzn);
        const double up = l <= L - 2 ? -(dt * p.C_e * (0.5 * (KV + Kvn)) / (dzl * dzn)) : 0.0;
        const double lo = l >= 2 ? -(dt * p.C_e * (0.5 * (KV + Kvp)) / (dzl * dzc)) : 0.0;
        const double dg = 1.0 - (up + lo) - dt * S2, r = e + dt * S1;
        if (l == 1) {
          di = dg;
          xi = r;
        } else {
          fast = fast && fabs(di) >= fabs(lo) && di != 0.0;
          const double fact = lo / di;
          di = dg - fact * ui;
          xi = r - fact * xi;
        }
        ui = up;
        A[l] = di;
        X[l] = xi;
        Kvp = KV;
        Kvc = Kvn;
        dzc = dzn;
      }
    fast = fast && di != 0.0;
  }
  const unsigned long long left = __ballot(!fast && live);
  if (threadIdx.x == 0) a.left[mb * gridDim.x + blockIdx.x] = left;
  if (!fast || !live) return;
  const double e_top = fmax(p.C_srf * tau / a.rho0, p.e_min_srf);
  {
    double x1 = 0.0, x2 = 0.0, prev = up_top, dzn = DZ(L), Kvn = 0.0;
#pragma unroll
    for (int l = LM - 1; l >= 1; --l)
      if (l < L) {
        const double dzc = DZ(l), KV = kv[(int64_t)l * NC];
        double x;
        if (l == L - 1) {
          x = X[l] / A[l];
        } else {  // the super-diagonal again, as the rows have it
          const double up = -(dt * p.C_e * (0.5 * (KV + Kvn)) / (0.5 * (dzc + dzn) * dzn));
          x = (X[l] - up * x1 - 0.0 * x2) / A[l];
        }
        x2 = l == L - 1 ? 0.0 : x1;
        x1 = x;
        const double e = p.patankar ? x : fmax(x, p.e_min);
        X[l] = e;
        prev = fmin(FIRST(e, Nsq[l - 1]), prev + dzn);
        A[l] = prev;
        dzn = dzc;
        Kvn = KV;
      }
    A[0] = fmin(FIRST(p.e_0, Nsq[0]), prev + dzn);
  }
  {  // update_Kv_Kt
    auto store = [&](int l, double e, double n2, double u2, double up, double dn) {
      const double Ri = n2 / (u2 + p.eps_s), v = kv_tke(p, e, fmax(p.l_min, fmin(up, dn)));
      kv[(int64_t)l * NC] = v;
      kt[(int64_t)l * NC] = kt_tke(p, v, n2, Ri);
      if (l >= 1) tke[(int64_t)(l - 1) * NC] = fmax(e, p.e_min);
    };
    double dn = p.l_0, n2 = Nsq[0];
    store(0, p.e_0, n2, 0.0, A[0], dn);
#pragma unroll
    for (int l = 1; l < LM; ++l)
      if (l < L) {
        n2 = Nsq[l - 1];
        dn = fmin(FIRST(X[l], n2), dn + DZ(l));
        store(l, X[l], n2, dU2[l - 1], A[l], dn);
      }
    dn = fmin(FIRST(e_top, n2), dn + DZ(L));
    store(L, e_top, n2, 0.0, up_top, dn);
  }
#undef DZ
#undef E_OLD
#undef FIRST
}

__device__ __forceinline__ double irradiance(const wtg_vdiff& p, double depth) {
  return p.Q_sr * (0.58 * exp(-depth / 0.35) + (1.0 - 0.58) * exp(-depth / 23.0));
}

// Rows of the backward-Euler systems, generated in order k = 1..L with the
// previous and next layer thicknesses carried in registers (each is the same
// expression as the reference's array entry, so the rows are identical).
// Buoyancy (backwards_euler_temp): e < 0; an edge's velocity: e = 0, 1, 2.
struct Rows {
  const VdArgs& a;
  const double *m, *t, *u, *K, *f;
  int64_t c, nb;
  int e;
  double eta, dt;
  int k;
  double dzp, dzc, dzn, z0, z1;  // dz(k-1), dz(k), dz(k+1); z(k-1), z(k)
  __device__ double dz(int kk) const {
    const int64_t x = (int64_t)(kk - 1) * a.NC;
    if (e < 0) return (0.0 + m[x + c]) / (a.rho0 * 1.0);
    return 0.5 * ((0.0 + m[x + c]) / (a.rho0 * 1.0) + (0.0 + m[x + nb]) / (a.rho0 * 1.0));
  }
  __device__ void reset(double zs) {
    k = 0;
    dzc = 0.0;
    dzn = dz(1);
    z1 = zs;
  }
  // row k + 1: sub-diagonal lo (k + 1 >= 2), diagonal dg, super-diagonal up (k + 1 <= L - 1), rhs r
  __device__ void next(double& lo, double& dg, double& up, double& r) {
    const int L = a.L;
    const wtg_vdiff& p = a.p;
    ++k;
    dzp = dzc;
    dzc = dzn;
    dzn = k < L ? dz(k + 1) : 0.0;
    z0 = z1;
    z1 = z0 + dzc;
    const double dzl_lo = 0.5 * (dzp + dzc), dzl_up = 0.5 * (dzc + dzn);
    lo = k >= 2 ? -(dt * K[(int64_t)(k - 1) * a.NC + c] / (dzl_lo * dzc)) : 0.0;
    up = k <= L - 1 ? -(dt * K[(int64_t)k * a.NC + c] / (dzl_up * dzc)) : 0.0;
    if (e < 0) {
      const int64_t x = (int64_t)(k - 1) * a.NC + c;
      const double b = t[x] / (0.0 + m[x]);
      if (k == 1) {
        dg = 1.0 - up;
        r = b + dt * (-f[c] + solar()) / dzc;
      } else if (k < L) {
        dg = 1.0 - (up + lo);
        r = b + dt * solar() / dzc;
      } else {
        // the reference's top row takes the row below's super-diagonal entry
        dg = 1.0 - (-(dt * K[(int64_t)(k - 1) * a.NC + c] / (dzl_lo * dzp)));
        r = b + dt * (f[a.NC + c] + p.Q_sr / (a.rho0 * p.c_p)) / dzc;
      }
    } else {
      r = u[((int64_t)(k - 1) * 3 + e) * a.NC + c];
      if (k == 1)
        dg = 1.0 - up + dt * p.bottom_friction / dzc;
      else if (k < L)
        dg = 1.0 - (up + lo);
      else
        dg = 1.0 - lo;
      if (k == L) r = r + dt * f[(3 + e) * a.NC + c] / dzc;
    }
  }
  __device__ double solar() const {
    const wtg_vdiff& p = a.p;
    return p.Q_sr * (irradiance(p, eta - z1) - irradiance(p, eta - z0)) / (a.rho0 * p.c_p);
  }
};

// One system of a column in private arrays: the buoyancy (e = -1) or the
// velocity of the RT, DG or UP edge (0..2)
__device__ void solve_column(const VdArgs& a, int64_t mb, int64_t c, int e, double eta) {
  const int L = a.L;
  const int64_t NC = a.NC;
  const double* m = a.m + mb * L * NC;
  double* t = a.t + mb * L * NC;
  double* u = a.u + mb * 3 * L * NC;
  const bool edge = e >= 0;
  const int64_t nb = e == 0 ? c + 1 : e == 1 ? c + a.S + 1 : e == 2 ? c + a.S : c;
  SolveWork w;
  Rows rows{a, m, t, u, (edge ? a.kv : a.kt) + mb * (L + 1) * NC, a.force + mb * 6 * NC, c, nb, e, eta, a.dt};
  solve_rows(L, rows, a.topo[mb * NC + c], w);
  for (int k = 1; k <= L; ++k) {
    const int64_t x = (int64_t)(k - 1) * NC + c;
    if (edge)
      u[((int64_t)(k - 1) * 3 + e) * NC + c] = w.X[k];
    else
      t[x] = (0.0 + m[x]) * w.X[k];
  }
}

// backwards_euler_temp of every owned node and pole master, then
// backwards_euler_velo of the owned nodes' edges
__global__ __launch_bounds__(VT) void vd_solve_kernel(VdArgs a) {
  const int64_t tid = (int64_t)blockIdx.x * VT + threadIdx.x;
  if (tid >= (int64_t)10 * a.n * a.n + 2) return;
  bool pole;
  const int64_t c = column(a, tid, pole);
  const int L = a.L;
  const int64_t NC = a.NC, mb = blockIdx.y;
  const double* m = a.m + mb * L * NC;
  double* t = a.t + mb * L * NC;
  double* u = a.u + mb * 3 * L * NC;
  const double* f = a.force + mb * 6 * NC;
  SolveWork w;
  const double zs = a.topo[mb * NC + c];
  const double eta = a.eta ? a.eta[mb * NC + c] : free_surface(a, m, zs, c);
  Rows rows{a, m, t, u, a.kt + mb * (L + 1) * NC, f, c, c, -1, eta, a.dt};
  solve_rows(L, rows, zs, w);
  for (int k = 1; k <= L; ++k) {
    const int64_t x = (int64_t)(k - 1) * NC + c;
    t[x] = (0.0 + m[x]) * w.X[k];
  }
  if (pole) return;  // the poles carry no edges of their own
  const int64_t nb[3] = {c + 1, c + a.S + 1, c + a.S};
  for (int e = 0; e < 3; ++e) {
    Rows ru{a, m, t, u, a.kv + mb * (L + 1) * NC, f, c, nb[e], e, eta, a.dt};
    solve_rows(L, ru, zs, w);
    for (int k = 1; k <= L; ++k) u[((int64_t)(k - 1) * 3 + e) * NC + c] = w.X[k];
  }
}

// The same for at most LM layers, a lane one system: the elimination's
// diagonal, super-diagonal and right-hand side stay in registers (the loops
// over layers are unrolled), so that the state's own bytes are what moves.
// A system that dgtsv would pivot and a column with a thickness that is not
// positive are left to vd_solve_left_kernel (a call from here would cost the
// arrays their registers).  Grid x: count systems of every column block, the
// first being `first`.  SOLAR: the buoyancy rows with a solar flux, whose two
// exponentials an interface cost the other systems no registers this way.
// Bound by memory latency at two waves per SIMD (three arrays of 32 doubles are
// 192 registers).  J8 L30: 1.63 -> 0.70 ms; with the arrays in LDS (three waves
// per compute unit) 1.6 ms.
template <int LM, bool SOLAR>
__global__ __launch_bounds__(VT, LM > 16 ? 2 : 3) void vd_solve_reg_kernel(VdArgs a, int ncb, int first, int count) {
  const int L = a.L;
  // consecutive blocks lie on different XCDs: an XCD takes a run of column
  // blocks, the systems of one after another
  const int per = ncb / 8, id = blockIdx.x, e = SOLAR ? -1 : first + id / 8 % count;
  const int cb = id % 8 * per + id / 8 / count;
  const bool edge = !SOLAR && e >= 0;
  const int64_t nown = (int64_t)10 * a.n * a.n, tid = (int64_t)cb * VT + threadIdx.x;
  const bool live = tid < (edge ? nown : nown + 2);  // the poles carry no edges of their own
  bool pole;
  const int64_t c = column(a, live ? tid : 0, pole);
  const int64_t NC = a.NC, mb = blockIdx.y;
  const double* m = a.m + mb * L * NC;
  const double* f = a.force + mb * 6 * NC + c;
  const double* K = (edge ? a.kv : a.kt) + mb * (L + 1) * NC + c;
  const int64_t nb = e == 0 ? c + 1 : e == 1 ? c + a.S + 1 : e == 2 ? c + a.S : c;
  double* const v = edge ? a.u + (mb * 3 * L + e) * NC + c : a.t + mb * L * NC + c;
  const int64_t vs = edge ? 3 * NC : NC;
  const double rho = a.rho0 * 1.0, rrho = 1.0 / rho, dt = a.dt;
  const wtg_vdiff& p = a.p;
  // thickness, coefficient at the upper interface and value of every layer;
  // they become the elimination's super-diagonal, diagonal and right-hand side
  double U[LM], D[LM], X[LM];
  double least = INFINITY, depth = 0.0;
  constexpr int CH = 4;
#pragma unroll
  for (int k0 = 0; k0 < LM; k0 += CH) {
    if (k0 < L) {
      double m0[CH], m1[CH];
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        const int64_t k = min(k0 + j, L - 1);
        m0[j] = m[k * NC + c];
        m1[j] = m[k * NC + nb];
        D[k0 + j] = K[(k + 1) * NC];
        X[k0 + j] = v[k * vs];
      }
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        const double z = div_by(0.0 + m0[j], rho, rrho);
        U[k0 + j] = edge ? 0.5 * (z + div_by(0.0 + m1[j], rho, rrho)) : z;
        least = U[k0 + j] > 0.0 ? least : -1.0;
        if (SOLAR && k0 + j < L) depth = depth + z;
        if (!edge) X[k0 + j] = X[k0 + j] / (0.0 + m0[j]);
      }
    }
  }
  bool fast = least > 0.0;
  if (fast) {
    // the irradiance at the layer's lower interface, of height z0
    double z0 = 0.0, eta = 0.0, below = 0.0;
    if (SOLAR) {
      z0 = a.topo[mb * NC + c];
      eta = a.eta ? a.eta[mb * NC + c] : depth + z0;
      below = irradiance(p, eta - z0);
    }
    const double bot = edge ? 0.0 : f[0], top = edge ? f[(3 + e) * NC] : f[NC];
    double di = 0.0, xi = 0.0, ui = 0.0, Kp = 0.0, dzp = 0.0;
#pragma unroll
    for (int k = 0; k < LM; ++k) {
      if (k < L) {
        const bool last = k == L - 1;
        const double dz = U[k], dzn = k + 1 < LM && !last ? U[k + 1 < LM ? k + 1 : k] : 0.0, Kc = D[k];
        const double lo = k > 0 ? -(dt * Kp / (0.5 * (dzp + dz) * dz)) : 0.0;
        const double up = last ? 0.0 : -(dt * Kc / (0.5 * (dz + dzn) * dz));
        double dg = 1.0 - (up + lo), r = X[k];
        if (edge) {
          if (k == 0) dg = dg + dt * p.bottom_friction / dz;
          if (last) r = r + dt * top / dz;
        } else {
          if (SOLAR && !last) {
            z0 = z0 + dz;
            const double above = irradiance(p, eta - z0);
            const double solar = p.Q_sr * (above - below) / (a.rho0 * p.c_p);
            below = above;
            r = r + dt * (k == 0 ? -bot + solar : solar) / dz;
          } else if (k == 0) {
            r = r + dt * (-bot + 0.0) / dz;
          }
          if (last) {
            // the reference's top row takes the row below's super-diagonal entry
            dg = 1.0 - (-(dt * Kp / (0.5 * (dzp + dz) * dzp)));
            r = X[k] + dt * (top + p.Q_sr / (a.rho0 * p.c_p)) / dz;
          }
        }
        if (k == 0) {
          di = dg;
          xi = r;
        } else {
          fast = fast && fabs(di) >= fabs(lo) && di != 0.0;
          const double fact = lo / di;
          di = dg - fact * ui;
          xi = r - fact * xi;
        }
        ui = up;
        D[k] = di;
        X[k] = xi;
        U[k] = up;
        Kp = Kc;
        dzp = dz;
      }
    }
    fast = fast && di != 0.0;
    if (fast) {
      double x1 = 0.0, x2 = 0.0;
#pragma unroll
      for (int k = LM - 1; k >= 0; --k) {
        if (k < L) {
          const double x = k == L - 1 ? X[k] / D[k] : (X[k] - U[k] * x1 - 0.0 * x2) / D[k];
          x2 = k == L - 1 ? 0.0 : x1;
          x1 = x;
          X[k] = x;
        }
      }
#pragma unroll
      for (int k = 0; k < LM; ++k)
        if (k < L && live) v[k * vs] = edge ? X[k] : (0.0 + m[k * NC + c]) * X[k];
    }
  }
  const unsigned long long left = __ballot(!fast && live);
  if (threadIdx.x == 0) a.left[(mb * 4 + e + 1) * ncb + cb] = left;
}

// the systems that vd_solve_reg_kernel left
__global__ __launch_bounds__(VT) void vd_solve_left_kernel(VdArgs a, int ncb) {
  const int64_t mb = blockIdx.y, NC = a.NC;
  each_left(a.left + mb * 4 * ncb, 4 * ncb, [&](int word) {
    bool pole;
    const int64_t c = column(a, (int64_t)(word % ncb) * VT + threadIdx.x, pole);
    const int e = word / ncb - 1;
    const double zs = a.topo[mb * NC + c];
    const double eta = e >= 0 ? 0.0 : a.eta ? a.eta[mb * NC + c] : free_surface(a, a.m + mb * a.L * NC, zs, c);
    solve_column(a, mb, c, e, eta);
  });
}

// With a solar flux the buoyancy rows are a launch of their own: the call at J8
// L30 takes 1.87 ms (3.48 with every system in private arrays), J6 L20 141 us
// (310), 8 us more than without the flux.
template <int LM>
void launch_solve_reg(const VdArgs& a, int ncb, unsigned members, hipStream_t stream) {
  const bool solar = a.p.Q_sr != 0.0;
  if (solar)
    hipLaunchKernelGGL((vd_solve_reg_kernel<LM, true>), dim3((unsigned)ncb, members), dim3(VT), 0, stream, a, ncb, -1,
                       1);
  const int first = solar ? 0 : -1, count = solar ? 3 : 4;
  hipLaunchKernelGGL((vd_solve_reg_kernel<LM, false>), dim3((unsigned)(count * ncb), members), dim3(VT), 0, stream, a,
                     ncb, first, count);
}

}  // namespace

extern "C" void wtg_vdiff_defaults(wtg_vdiff* p) {
  if (!p) return;
  *p = wtg_vdiff{};
  p->C_e = 1.0;
  p->C_eps = 7.0e-1;
  p->C_l = 2.0e5;
  p->C_k = 1.0e-1;
  p->C_srf = 6.783e1;
  p->e_0 = 1.0e-6 / sqrt(2.0);
  p->e_min = 1.0e-6;
  p->e_min_srf = 1.0e-4;
  p->eps_s = 1.0e-20;
  p->kappa_VK = 4.0e-1;
  p->Kt_enh = 1.0;
  p->Kt_max = 1e-2;
  p->Kt_min = 1.2e-5;
  p->Kv_max = 1e-2;
  p->Kv_min = 1.2e-4;
  p->mixed_layer = -200.0;
  p->l_0 = 4.0e-2;
  p->l_min = 1.0e-2;
  p->Neps_sq = 1.0e-20;
  p->Nsq_min = 1.0e-12;
  p->Q_sr = 0.0;
  p->c_p = 1004.64;
}

extern "C" int wtg_set_vdiff(wtg_ctx* c, const wtg_vdiff* p) {
  if (!c || !p) return WTG_E_ARG;
  const int L = c->params.nlayers, M = c->nmembers;
  if (L > VMAX) return wtg_fail(c, WTG_E_ARG, "the vertical diffusion takes at most %d layers, not %d", VMAX, L);
  // backwards_euler_temp indexes a second layer and the TKE system a third one
  if (L < (p->tke_closure ? 3 : 2))
    return wtg_fail(c, WTG_E_ARG, "the vertical diffusion needs at least %d layers%s, not %d", p->tke_closure ? 3 : 2,
                    p->tke_closure ? " with the TKE closure" : "", L);
  const int64_t NC = c->info.ncells;
  if (!c->vd_kt) {
    if (int rc = wtg_dalloc<double>(c, &c->vd_kt, (size_t)M * (L + 1) * NC)) return rc;
    if (int rc = wtg_dalloc<double>(c, &c->vd_kv, (size_t)M * (L + 1) * NC)) return rc;
    if (int rc = wtg_dalloc<double>(c, &c->vd_tke, (size_t)M * L * NC)) return rc;
    if (int rc = wtg_dalloc<double>(c, &c->vd_force, (size_t)M * 6 * NC)) return rc;
    const size_t nblk = ((size_t)10 * c->info.n * c->info.n + 2 + VT - 1) / VT;
    if (int rc = wtg_dalloc<unsigned long long>(c, &c->vd_left, (size_t)M * 4 * ((nblk + 7) / 8 * 8))) return rc;
    WTG_HIPCHK(c, hipMemsetAsync(c->vd_kt, 0, (size_t)M * (L + 1) * NC * sizeof(double), c->stream));
    WTG_HIPCHK(c, hipMemsetAsync(c->vd_kv, 0, (size_t)M * (L + 1) * NC * sizeof(double), c->stream));
    WTG_HIPCHK(c, hipMemsetAsync(c->vd_tke, 0, (size_t)M * L * NC * sizeof(double), c->stream));
    WTG_HIPCHK(c, hipMemsetAsync(c->vd_force, 0, (size_t)M * 6 * NC * sizeof(double), c->stream));
    WTG_HIPCHK(c, hipStreamSynchronize(c->stream));
  }
  c->vd = *p;
  c->vd_set = true;
  return 0;
}

static int vd_ready(wtg_ctx* c) {
  if (!c) return WTG_E_ARG;
  if (!c->vd_set) return wtg_fail(c, WTG_E_STATE, "wtg_set_vdiff must be called first");
  return 0;
}

extern "C" int wtg_vdiff_set_coefficients(wtg_ctx* c, const double* Kt, const double* Kv, const double* tke) {
  if (int rc = vd_ready(c)) return rc;
  const int L = c->params.nlayers, M = c->nmembers;
  const size_t NC = (size_t)c->info.ncells, ni = (size_t)M * (L + 1) * NC, nl = (size_t)M * L * NC;
  if (Kt) WTG_HIPCHK(c, hipMemcpyAsync(c->vd_kt, Kt, ni * sizeof(double), hipMemcpyHostToDevice, c->stream));
  if (Kv) WTG_HIPCHK(c, hipMemcpyAsync(c->vd_kv, Kv, ni * sizeof(double), hipMemcpyHostToDevice, c->stream));
  if (tke) WTG_HIPCHK(c, hipMemcpyAsync(c->vd_tke, tke, nl * sizeof(double), hipMemcpyHostToDevice, c->stream));
  WTG_HIPCHK(c, hipStreamSynchronize(c->stream));
  return 0;
}

extern "C" int wtg_vdiff_get_coefficients(wtg_ctx* c, double* Kt, double* Kv, double* tke) {
  if (int rc = vd_ready(c)) return rc;
  const int L = c->params.nlayers, M = c->nmembers;
  const size_t NC = (size_t)c->info.ncells, ni = (size_t)M * (L + 1) * NC, nl = (size_t)M * L * NC;
  if (Kt) WTG_HIPCHK(c, hipMemcpyAsync(Kt, c->vd_kt, ni * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  if (Kv) WTG_HIPCHK(c, hipMemcpyAsync(Kv, c->vd_kv, ni * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  if (tke) WTG_HIPCHK(c, hipMemcpyAsync(tke, c->vd_tke, nl * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  WTG_HIPCHK(c, hipStreamSynchronize(c->stream));
  return 0;
}

extern "C" int wtg_vdiff_set_forcing(wtg_ctx* c, const double* bot, const double* top, const double* tau,
                                     const double* wind) {
  if (int rc = vd_ready(c)) return rc;
  const size_t NC = (size_t)c->info.ncells;
  const double* src[4] = {bot, top, tau, wind};
  const size_t off[4] = {0, 1, 2, 3}, cnt[4] = {1, 1, 1, 3};
  for (int mb = 0; mb < c->nmembers; ++mb)
    for (int q = 0; q < 4; ++q)
      if (src[q])
        WTG_HIPCHK(c, hipMemcpyAsync(c->vd_force + ((size_t)mb * 6 + off[q]) * NC, src[q] + (size_t)mb * cnt[q] * NC,
                                     cnt[q] * NC * sizeof(double), hipMemcpyHostToDevice, c->stream));
  WTG_HIPCHK(c, hipStreamSynchronize(c->stream));
  return 0;
}

extern "C" int wtg_vertical_diffusion(wtg_ctx* c, int slot, double dt, int istep) {
  if (int rc = vd_ready(c)) return rc;
  if (slot < 0 || slot >= c->nslots) return wtg_fail(c, WTG_E_ARG, "slot %d out of range [0,%d)", slot, c->nslots);
  if (!c->topo_set) return wtg_fail(c, WTG_E_STATE, "wtg_set_topography must be called first");
  const double* eta = nullptr;
  if (c->vd.mode_split) {
    if (!c->fs[FS_ETA])
      return wtg_fail(c, WTG_E_STATE, "mode_split takes eta from the free surface, which has not been set");
    eta = c->fs[FS_ETA];
  }
  const int L = c->params.nlayers, M = c->nmembers;
  const auto& s = c->slots[slot];
  if (int rc = wtg_ghost_fill_layers(c, L * M, s.m, s.t, s.u)) return rc;
  VdArgs a{c->info.n, c->info.S, L, istep, c->info.ncells, c->info.south_pole, c->info.north_pole, dt,
           c->params.ref_density, c->params.grav, c->vd, c->d_len, c->d_ped, c->d_hinv, c->d_topo, eta, c->vd_force,
           s.m, s.t, s.u, c->vd_kt, c->vd_kv, c->vd_tke, c->vd_left};
  const int64_t cols = (int64_t)10 * c->info.n * c->info.n + 2;
  const dim3 grid((unsigned)((cols + VT - 1) / VT), (unsigned)M);
  // the register kernels hold up to 32 layers; above, the private arrays
  const int nblk = (int)grid.x, ncb = (nblk + 7) / 8 * 8;
  if (!c->vd.tke_closure || istep == 1 || L > 32) {
    hipLaunchKernelGGL(vd_turbulent_kernel, grid, dim3(VT), 0, c->stream, a);
  } else {
    if (L <= 16)
      hipLaunchKernelGGL(vd_tke_kernel<16>, grid, dim3(VT), 0, c->stream, a);
    else if (L <= 24)
      hipLaunchKernelGGL(vd_tke_kernel<24>, grid, dim3(VT), 0, c->stream, a);
    else
      hipLaunchKernelGGL(vd_tke_kernel<32>, grid, dim3(VT), 0, c->stream, a);
    WTG_HIPCHK(c, hipGetLastError());
    hipLaunchKernelGGL(vd_tke_left_kernel, dim3((unsigned)((nblk + LEFT - 1) / LEFT), (unsigned)M), dim3(VT), 0,
                       c->stream, a, nblk);
  }
  WTG_HIPCHK(c, hipGetLastError());
  if (L > 32) {
    hipLaunchKernelGGL(vd_solve_kernel, grid, dim3(VT), 0, c->stream, a);
  } else {
    if (L <= 16)
      launch_solve_reg<16>(a, ncb, (unsigned)M, c->stream);
    else if (L <= 24)
      launch_solve_reg<24>(a, ncb, (unsigned)M, c->stream);
    else
      launch_solve_reg<32>(a, ncb, (unsigned)M, c->stream);
    WTG_HIPCHK(c, hipGetLastError());
    hipLaunchKernelGGL(vd_solve_left_kernel, dim3((unsigned)((4 * ncb + LEFT - 1) / LEFT), (unsigned)M), dim3(VT), 0,
                       c->stream, a, ncb);
  }
  WTG_HIPCHK(c, hipGetLastError());
  if (int rc = wtg_ghost_fill_layers(c, L * M, s.m, s.t, s.u)) return rc;
  WTG_HIPCHK(c, hipStreamSynchronize(c->stream));
  return 0;
}
