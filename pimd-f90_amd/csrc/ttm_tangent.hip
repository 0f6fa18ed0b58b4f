// Derivatives of the TTM energy and gradient with respect to the model's vdW,
// polarisation, Thole and charge-surface parameters, for fitting.  No
// counterpart in the reference, whose parameters are fixed in pot_mod.f90.
//
// Forward (tangent) mode: one workgroup evaluates pot_ttm (pot_ttm.f90:3-630)
// for one configuration with dual numbers along one parameter direction, so
// the value parts reproduce the energy and gradient of the force path and the
// derivative parts are their exact derivatives along that parameter, through
// the SOR dipole iterations as executed (the same iteration count, branch
// decisions on the values).  With ew and gw the loss weights of the energy
// and of the gradient of each configuration, the loss derivative along
// parameter k is sum_b ew_b dE_b/dtheta_k + gw_b . dG_b/dtheta_k.
//
// Parameters (theta, PIMD_TTM_NPARAM = 16): vdwA..vdwE, polarO, polarH,
// polarM, polfacO, polfacH, polfacM, aDD, aCCaCD, dms_param1..3
// (potential.f90:84-113, 152-160).  Geometry (sites, k-space phases) does not
// depend on them and stays plain FP64; charges, dipoles, fields, potentials
// and the screened interaction tensors carry the derivative.  The M-site
// fraction gammaM (pot_mod.f90:12,24) also moves the M sites (pot_ttm.f90:
// 74-79): its direction runs an instance whose site positions and phases are
// dual numbers too (GD = true), with dM/dgammaM = (r_OH1 + r_OH2) / 2.
//
// Work layout: grid (configuration, direction), one 256-lane workgroup each;
// lanes stride over sites, k-vectors or molecules per phase, each lane owns
// what it writes (every site-pair term is evaluated from both ends), so no
// atomics.  Per configuration a preparatory kernel writes the sites and the
// per-axis phase tables once for all directions.
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "dual.h"
#include "ttm_device.h"

namespace pimd {

template <>
struct RM<Dual> {
  static __device__ __forceinline__ Dual sqrt_(Dual x) { return dsqrt(x); }
  static __device__ __forceinline__ Dual rcp(Dual x) { return Dual(1.0) / x; }
  static __device__ __forceinline__ Dual div(Dual a, Dual b) { return a / b; }
  static __device__ __forceinline__ Dual exp_(Dual x) { return dexp(x); }
  static __device__ __forceinline__ Dual log_(Dual x) { return dlog(x); }
  static __device__ __forceinline__ Dual abs_(Dual x) { return dabs(x); }
};

constexpr int TAN_BLOCK = 256;
enum TanMode { TAN_PARAMS = 0, TAN_GAMMA_M = 1, TAN_ADJOINT = 2 };

// Per-configuration FP64 data: sites [4N][3] (O, H1, H2, M blocks, as
// pot_ttm.f90:56-80), then the phase tables exp(2 pi i m x / L) per axis,
// [m][site] as (cos, sin): m = 0..hmax, -kmax..kmax, -lmax..lmax; then the
// sites' derivatives along the geometric direction of the dual-geometry
// instances, [4N][3]: dr/dgammaM (nonzero for the M sites only) or the
// position direction of the adjoint's force-loss term.
static size_t tangent_tab_doubles(const SysConst &c) {
  const size_t ns = 4 * (size_t)c.N;
  return 2 * ns * (size_t)((c.hmax + 1) + (2 * c.kmax + 1) + (2 * c.lmax + 1));
}
size_t tangent_cfg_doubles(const SysConst &c) {
  const size_t ns = 4 * (size_t)c.N;
  return ns * 3 + tangent_tab_doubles(c) + 3 * ns;
}

// Per (configuration, direction) dual workspace: charge, phi [4N], Efq, dR
// [4N][3], dip, olddip, Efd [nd N][3], grdq [N][27], S(k) of the charges and
// of the dipoles [nk][2], the monomer energy [1].
size_t tangent_ws_duals(const SysConst &c) {
  const size_t ns = 4 * (size_t)c.N, nds = (size_t)c.nd * c.N;
  return 8 * ns + 9 * nds + 27 * (size_t)c.N + 4 * (size_t)c.nk + 1;
}

// The workspace arrays of one (configuration, direction).
struct TanWs {
  Dual *q, *phi, *Efq, *dR, *dip, *old, *Efd, *grdq, *Sq, *Sm, *umon;
  __device__ TanWs(Dual *base, const SysConst &c) {
    const int ns = 4 * c.N, nds = c.nd * c.N;
    q = base;
    phi = q + ns;
    Efq = phi + ns;
    dR = Efq + 3 * ns;
    dip = dR + 3 * ns;
    old = dip + 3 * nds;
    Efd = old + 3 * nds;
    grdq = Efd + 3 * nds;
    Sq = grdq + 27 * c.N;
    Sm = Sq + 2 * c.nk;
    umon = Sm + 2 * c.nk;
  }
};

// mode 1: dS = dr/dgammaM; mode 2: dS = the atoms' direction gw [P][3N][3]
// (the M site moving with its atoms, pot_ttm.f90:74-79).
__global__ __launch_bounds__(TAN_BLOCK) void k_tangent_prep(SysConst c, const double *__restrict__ RR,
                                                           double *__restrict__ cfg, size_t stride,
                                                           size_t ds_off, int mode,
                                                           const double *__restrict__ gw) {
  const int b = blockIdx.x, N = c.N, ns = 4 * N;
  double *Rs = cfg + (size_t)b * stride;
  double *dS = Rs + ds_off;
  const double *rr = RR + (size_t)b * 9 * N, *g = gw + (size_t)b * 9 * N;
  const double gM = c.gammaM;
  for (int w = threadIdx.x; w < N; w += TAN_BLOCK) {
    double roh1[3], roh2[3];
    for (int k = 0; k < 3; ++k) {
      Rs[(0 * N + w) * 3 + k] = rr[9 * w + k];
      Rs[(1 * N + w) * 3 + k] = rr[9 * w + 3 + k];
      Rs[(2 * N + w) * 3 + k] = rr[9 * w + 6 + k];
      roh1[k] = rr[9 * w + 3 + k] - rr[9 * w + k];
      roh2[k] = rr[9 * w + 6 + k] - rr[9 * w + k];
    }
    minimg(c, roh1[0], roh1[1], roh1[2]);
    minimg(c, roh2[0], roh2[1], roh2[2]);
    for (int k = 0; k < 3; ++k) {
      Rs[(3 * N + w) * 3 + k] = 0.5 * gM * (roh1[k] + roh2[k]) + rr[9 * w + k];
      if (mode == 1) {
        for (int t = 0; t < 3; ++t) dS[(t * N + w) * 3 + k] = 0.0;
        dS[(3 * N + w) * 3 + k] = 0.5 * (roh1[k] + roh2[k]);
      } else if (mode == 2) {
        for (int t = 0; t < 3; ++t) dS[(t * N + w) * 3 + k] = g[9 * w + 3 * t + k];
        dS[(3 * N + w) * 3 + k] =
            (1.0 - gM) * g[9 * w + k] + 0.5 * gM * (g[9 * w + 3 + k] + g[9 * w + 6 + k]);
      }
    }
  }
  __syncthreads();
  double2 *tab = (double2 *)(Rs + (size_t)ns * 3);
  const int lens[3] = {c.hmax + 1, 2 * c.kmax + 1, 2 * c.lmax + 1};
  const int offs[3] = {0, c.kmax, c.lmax};
  for (int ax = 0; ax < 3; ++ax) {
    const int rows = lens[ax];
    for (int e = threadIdx.x; e < rows * ns; e += TAN_BLOCK) {
      const int m = e / ns - offs[ax], s = e % ns;
      double sv, cv;
      sincos(TWOPI * c.boxi[ax] * Rs[s * 3 + ax] * (double)m, &sv, &cv);
      tab[e] = make_double2(cv, sv);
    }
    tab += (size_t)rows * ns;
  }
}

// Model parameters as duals along one direction.
struct TanPar {
  Dual vdw[5], polar[4], apCC[4][4], raCC[4][4], apDD[4][4], lrc;
};

struct TanArgs {
  const double *RR;      // [P][Natoms][3]
  const double *pes;     // monomer PES parameters
  const double4 *kv;     // [nk] kx, ky, kz, 4 pi Ak / volume
  const int4 *khkl;      // [nk] h, k, l
  const double *cfg;     // per-configuration sites and tables
  size_t cfg_stride;
  Dual *ws;              // per (configuration, direction) workspace
  size_t ws_stride;
  const double *ew;      // [P] energy weights
  const double *gw;      // [P][Natoms][3] gradient weights
  double *out;           // [P][dirs][4]: E, dE/dtheta, loss term, SOR iterations
  double *dG;            // NULL or [P][dirs][Natoms][3] dG/dtheta
  double theta[TTM_NPARAM];
  double lrc_coef[3];    // dUvdw_lrc / d(vdwA, vdwB, vdwC)
  int dms_coef;          // 1: the directions are the DMS coefficients coefD
  int gamma_m;           // 1: the one direction is gammaM
  size_t ds_off;         // offset of the sites' directions dS [4N][3] in a configuration's data
  double *adj;           // adjoint: [P][TTM_ADJ_NPARAM] (dE/dtheta, gw . d(dE/dr)/dtheta)
};

// The derivative of the DMS charges and their gradients with respect to
// dms_param1..3 (which = 0..2), the linear corrections of nasa.f90:245-291,
// in the layout of ps_monomer (gq[disp][charge][xyz], order H1, H2, O).
__device__ inline void dms_tangent(const SysConst &c, const double r[3][3], int which,
                                   double dq3[3], double dgq[3][3][3]) {
  double R1[3], R2[3];
  for (int k = 0; k < 3; ++k) {
    R1[k] = r[1][k] - r[0][k];
    R2[k] = r[2][k] - r[0][k];
  }
  minimg(c, R1[0], R1[1], R1[2]);
  minimg(c, R2[0], R2[1], R2[2]);
  const double d1 = sqrt(R1[0] * R1[0] + R1[1] * R1[1] + R1[2] * R1[2]);
  const double d2 = sqrt(R2[0] * R2[0] + R2[1] * R2[1] + R2[2] * R2[2]);
  const double costh = (R1[0] * R2[0] + R1[1] * R2[1] + R1[2] * R2[2]) / (d1 * d2);
  const double ax = R1[1] * R2[2] - R1[2] * R2[1];
  const double ay = -R1[0] * R2[2] + R1[2] * R2[0];
  const double az = R1[0] * R2[1] - R1[1] * R2[0];
  const double sinth = sqrt(ax * ax + ay * ay + az * az) / (d1 * d2);
  const double ang = atan2(sinth, costh), ath0 = 1.82400520401572996557;
  double P1 = 0, P2 = 0, p1r1 = 0, p2r2 = 0, p1c = 0, p2c = 0;
  if (which == 0) {
    P1 = d1 - c.dms2;
    P2 = d2 - c.dms2;
    p1r1 = 1.0;
    p2r2 = 1.0;
  } else if (which == 1) {
    P1 = -c.dms1;
    P2 = -c.dms1;
  } else {
    P1 = ang - ath0;
    P2 = ang - ath0;
    p1c = -1.0 / sinth;
    p2c = -1.0 / sinth;
  }
  dq3[0] = -(P1 + P2);
  dq3[1] = P1;
  dq3[2] = P2;
  const double f1q1r13 = (p1r1 - (p1c * costh / d1)) / d1, f1q1r23 = p1c / (d1 * d2);
  const double f2q1r23 = -(p1c * costh / d2) / d2, f2q1r13 = p1c / (d2 * d1);
  const double f1q2r13 = -(p2c * costh / d1) / d1, f1q2r23 = p2c / (d1 * d2);
  const double f2q2r23 = (p2r2 - (p2c * costh / d2)) / d2, f2q2r13 = p2c / (d2 * d1);
  for (int k = 0; k < 3; ++k) {
    dgq[0][0][k] = f1q1r13 * R1[k] + f1q1r23 * R2[k];
    dgq[1][0][k] = f2q1r13 * R1[k] + f2q1r23 * R2[k];
    dgq[2][0][k] = -(dgq[0][0][k] + dgq[1][0][k]);
    dgq[0][1][k] = f1q2r13 * R1[k] + f1q2r23 * R2[k];
    dgq[1][1][k] = f2q2r13 * R1[k] + f2q2r23 * R2[k];
    dgq[2][1][k] = -(dgq[0][1][k] + dgq[1][1][k]);
    dgq[0][2][k] = -(dgq[0][0][k] + dgq[0][1][k]);
    dgq[1][2][k] = -(dgq[1][0][k] + dgq[1][1][k]);
    dgq[2][2][k] = -(dgq[2][0][k] + dgq[2][1][k]);
  }
}

// The derivative of the DMS charges and their gradients with respect to the
// DMS coefficient coefD(j+1) (nasa.f90:185-242): the charges are linear in
// the coefficients, so this is the surface of ps_monomer with that one
// coefficient set to 1 and every other term (the others, the constant part
// PC0 and the dms_param corrections) left out.  Layout as ps_monomer's.
__device__ inline void dms_coef_tangent(const SysConst &c, const double r[3][3], int j,
                                        double dq3[3], double dgq[3][3][3]) {
  for (int a = 0; a < 3; ++a)
    for (int q = 0; q < 3; ++q)
      for (int k = 0; k < 3; ++k) dgq[a][q][k] = 0.0;
  if (j == 0) {  // the constant term of both P1 and P2
    dq3[0] = -2.0;
    dq3[1] = 1.0;
    dq3[2] = 1.0;
    return;
  }
  double R1[3], R2[3];
  for (int k = 0; k < 3; ++k) {
    R1[k] = r[1][k] - r[0][k];
    R2[k] = r[2][k] - r[0][k];
  }
  minimg(c, R1[0], R1[1], R1[2]);
  minimg(c, R2[0], R2[1], R2[2]);
  const double d1 = sqrt(R1[0] * R1[0] + R1[1] * R1[1] + R1[2] * R1[2]);
  const double d2 = sqrt(R2[0] * R2[0] + R2[1] * R2[1] + R2[2] * R2[2]);
  const double costh = (R1[0] * R2[0] + R1[1] * R2[1] + R1[2] * R2[2]) / (d1 * d2);
  const double costhe = -.24780227221366464506;
  const double x[3] = {(d1 - PS_REOH) / PS_REOH, (d2 - PS_REOH) / PS_REOH, costh - costhe};
  const int I = c_ps.idxd[j][0], J = c_ps.idxd[j][1], K = c_ps.idxd[j][2];
  // x^(n-1), with x^(-1) := 0
  auto pw = [](double v, int n) {
    if (n <= 0) return 0.0;
    double y = 1.0;
    for (int i = 1; i < n; ++i) y *= v;
    return y;
  };
  const double B2A = 0.529177249, bfac = 1.0 / (double)0.529177249f;
  const double efd = exp(-DMS_B1D * ((d1 - PS_REOH) * (d1 - PS_REOH) + (d2 - PS_REOH) * (d2 - PS_REOH)));
  const double defdr1 = -2.0 * DMS_B1D * (d1 - PS_REOH) * efd * B2A;
  const double defdr2 = -2.0 * DMS_B1D * (d2 - PS_REOH) * efd * B2A;
  const double t1 = pw(x[0], I) * pw(x[1], J) * pw(x[2], K);
  const double t2 = pw(x[0], J) * pw(x[1], I) * pw(x[2], K);
  double p1r1 = (double)(I - 1) * pw(x[0], I - 1) * pw(x[1], J) * pw(x[2], K) / PS_REOH * B2A;
  double p1r2 = (double)(J - 1) * pw(x[0], I) * pw(x[1], J - 1) * pw(x[2], K) / PS_REOH * B2A;
  double p1c = (double)(K - 1) * pw(x[0], I) * pw(x[1], J) * pw(x[2], K - 1);
  double p2r1 = (double)(J - 1) * pw(x[0], J - 1) * pw(x[1], I) * pw(x[2], K) / PS_REOH * B2A;
  double p2r2 = (double)(I - 1) * pw(x[0], J) * pw(x[1], I - 1) * pw(x[2], K) / PS_REOH * B2A;
  double p2c = (double)(K - 1) * pw(x[0], J) * pw(x[1], I) * pw(x[2], K - 1);
  p1r1 = (p1r1 * efd + t1 * defdr1) * bfac;
  p1r2 = (p1r2 * efd + t1 * defdr2) * bfac;
  p1c = p1c * efd;
  p2r1 = (p2r1 * efd + t2 * defdr1) * bfac;
  p2r2 = (p2r2 * efd + t2 * defdr2) * bfac;
  p2c = p2c * efd;
  const double P1 = t1 * efd, P2 = t2 * efd;
  dq3[0] = -(P1 + P2);
  dq3[1] = P1;
  dq3[2] = P2;
  const double f1q1r13 = (p1r1 - (p1c * costh / d1)) / d1, f1q1r23 = p1c / (d1 * d2);
  const double f2q1r23 = (p1r2 - (p1c * costh / d2)) / d2, f2q1r13 = p1c / (d2 * d1);
  const double f1q2r13 = (p2r1 - (p2c * costh / d1)) / d1, f1q2r23 = p2c / (d1 * d2);
  const double f2q2r23 = (p2r2 - (p2c * costh / d2)) / d2, f2q2r13 = p2c / (d2 * d1);
  for (int k = 0; k < 3; ++k) {
    dgq[0][0][k] = f1q1r13 * R1[k] + f1q1r23 * R2[k];
    dgq[1][0][k] = f2q1r13 * R1[k] + f2q1r23 * R2[k];
    dgq[2][0][k] = -(dgq[0][0][k] + dgq[1][0][k]);
    dgq[0][1][k] = f1q2r13 * R1[k] + f1q2r23 * R2[k];
    dgq[1][1][k] = f2q2r13 * R1[k] + f2q2r23 * R2[k];
    dgq[2][1][k] = -(dgq[0][1][k] + dgq[1][1][k]);
    dgq[0][2][k] = -(dgq[0][0][k] + dgq[0][1][k]);
    dgq[1][2][k] = -(dgq[1][0][k] + dgq[1][1][k]);
    dgq[2][2][k] = -(dgq[2][0][k] + dgq[2][1][k]);
  }
}

// exp(i k . r_s) from the per-axis tables (the products of ssincos,
// ewald.f90:403-437 and ewald.f90:20-33).
struct Phases {
  const double2 *tx, *ty, *tz;
  const double *dS;  // the sites' directions [4N][3]
  int ns, kmax, lmax, N;
  __device__ __forceinline__ void at(int s, int4 h, double &ck, double &sk) const {
    const double2 a = tx[(size_t)h.x * ns + s], b = ty[(size_t)(h.y + kmax) * ns + s],
                  z = tz[(size_t)(h.z + lmax) * ns + s];
    const double cxy = a.x * b.x - a.y * b.y, sxy = a.y * b.x + a.x * b.y;
    ck = cxy * z.x - sxy * z.y;
    sk = sxy * z.x + cxy * z.y;
  }
  // with moving sites: d exp(i k.r) = i (k . dr) exp(i k.r)
  __device__ __forceinline__ void at(int s, int4 h, const double4 &kv, Dual &ck, Dual &sk) const {
    double c, sn;
    at(s, h, c, sn);
    const double *d = dS + 3 * s;
    const double kd = kv.x * d[0] + kv.y * d[1] + kv.z * d[2];
    ck = Dual(c, -kd * sn);
    sk = Dual(sn, kd * c);
  }
  __device__ __forceinline__ void at(int s, int4 h, const double4 &, double &ck, double &sk) const {
    at(s, h, ck, sk);
  }
};

// Geometry of the GD = true instance: minimum image on the value part (the
// box shift is constant along gammaM).
__device__ __forceinline__ void minimg(const SysConst &c, Dual &x, Dual &y, Dual &z) {
  minimg(c, x.v, y.v, z.v);
}
__device__ __forceinline__ Dual as_dual(Dual x) { return x; }
__device__ __forceinline__ Dual as_dual(double x) { return Dual(x); }

// self1 / self2 (smear.f90:110-156) of a dual distance, the same steps as
// those of the plain ones.
__device__ __forceinline__ void self1(const SysConst &c, Dual drsq, Dual &ts0, Dual &ts1) {
  const Dual dd = dsqrt(drsq), drsqi = Dual(1.0) / drsq, dri = dsqrt(drsqi);
  const Dual expon = dexp(-(c.a2 * drsq));
  const Dual kr0 = erfc_as<Dual>(c.aewald * dd, expon) * dri;
  const Dual kr1 = (kr0 + c.cts1 * expon) * drsqi;
  const Dual ch0 = -dri, ch1 = ch0 * drsqi;
  ts0 = ch0 + kr0;
  ts1 = kr1 + ch1;
}
__device__ __forceinline__ void self2(const SysConst &c, Dual drsq, Dual &ts1, Dual &ts2) {
  const Dual dd = dsqrt(drsq), drsqi = Dual(1.0) / drsq, dri = dsqrt(drsqi);
  const Dual expon = dexp(-(c.a2 * drsq));
  const Dual kr0 = erfc_as<Dual>(c.aewald * dd, expon) * dri;
  const Dual kr1 = (kr0 + c.cts1 * expon) * drsqi;
  const Dual kr2 = (kr1 + c.cts2 * expon) * drsqi;
  const Dual ch0 = -dri, ch1 = ch0 * drsqi, ch2 = ch1 * drsqi;
  ts1 = kr1 + ch1;
  ts2 = kr2 + ch2;
}

__device__ __forceinline__ double block_sum(double v, double *red) {
  red[threadIdx.x] = v;
  __syncthreads();
  for (int o = TAN_BLOCK / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  const double r = red[0];
  __syncthreads();
  return r;
}

// Lanes per site of a loop over nsites sites whose per-site work is a sum
// over k-vectors: the largest power of two (at most a wave) such that the
// groups of all sites fit in the workgroup.  Each group splits the k-vectors
// of its site and combines its partial sums with group_sum.
__device__ __forceinline__ int site_lanes(int nsites) {
  int g = 1;
  while (g < 64 && 2 * g * nsites <= TAN_BLOCK) g *= 2;
  return g;
}

__device__ __forceinline__ Dual group_sum(Dual x, int G) {
  for (int o = G >> 1; o > 0; o >>= 1) {
    x.v += __shfl_xor(x.v, o);
    x.d += __shfl_xor(x.d, o);
  }
  return x;
}

// (3 t2 r r^T - t1) v, get_dd3 applied (pot_ttm.f90:633-647).
template <class G>
__device__ __forceinline__ void dd3d(const G r[3], Dual t1, Dual t2, const Dual v[3], Dual out[3]) {
  const Dual t = 3.0 * t2;
  const Dual rv = v[0] * r[0] + v[1] * r[1] + v[2] * r[2];
  for (int k = 0; k < 3; ++k) out[k] = t * r[k] * rv - t1 * v[k];
}

// The monomer phase of the tangent evaluation (pot_ttm.f90:84-151): DMS
// charges and their coordinate gradients with their derivatives along the
// direction, the PES gradient and the monomer energy of the configuration,
// into the (configuration, direction) workspace.  A kernel of its own: the
// PES and DMS polynomials hold more registers than any later phase.
template <int MODE>
__global__ __launch_bounds__(TAN_BLOCK) void k_tangent_monomer(SysConst c, TanArgs a) {
  using GT = std::conditional_t<MODE != TAN_PARAMS, Dual, double>;
  const int b = blockIdx.x, dir = blockIdx.y, ndir = gridDim.y, tid = threadIdx.x, N = c.N;
  const TanWs W(a.ws + ((size_t)b * ndir + dir) * a.ws_stride, c);
  Dual *q = W.q, *phi = W.phi, *Efq = W.Efq, *dR = W.dR, *grdq = W.grdq;
  __shared__ double red[TAN_BLOCK];
  // gammaM and the charge placement factors (pot_ttm.f90:134-137)
  GT gM = c.gammaM;
  if constexpr (MODE == TAN_GAMMA_M) gM.d = 1.0;
  const GT tmpq = 0.5 * gM / (1.0 - gM), qMf = GT(1.0) / (1.0 - gM);

  double umon = 0.0;
  for (int w = tid; w < N; w += TAN_BLOCK) {
    double r[3][3], e1, dr1[3][3], q3[3], gq[3][3][3], dq3[3] = {0, 0, 0}, dgq[3][3][3] = {};
    const double *rr = a.RR + ((size_t)b * 3 * N + 3 * w) * 3;
    for (int at = 0; at < 3; ++at)
      for (int k = 0; k < 3; ++k) r[at][k] = rr[3 * at + k];
    ps_monomer<true>(c, r, e1, dr1, q3, gq, a.pes);
    umon += e1;
    if constexpr (MODE == TAN_ADJOINT) {
      // the charges along the atoms' direction gw: dq = sum_atoms gq . gw, with
      // gq[disp][charge] in the order (H1, H2, O) and q3 in (O, H1, H2)
      const double *g = a.gw + ((size_t)b * 3 * N + 3 * w) * 3;
      const int atom[3] = {1, 2, 0};
      for (int i = 0; i < 3; ++i) {
        const int ch = i == 0 ? 2 : i - 1;
        double v = 0.0;
        for (int d = 0; d < 3; ++d)
          for (int k = 0; k < 3; ++k) v += gq[d][ch][k] * g[3 * atom[d] + k];
        dq3[i] = v;
      }
    } else if (MODE == TAN_PARAMS && a.dms_coef) {
      dms_coef_tangent(c, r, dir, dq3, dgq);
    } else if (MODE == TAN_PARAMS && dir >= TP_DMS1) {
      dms_tangent(c, r, dir - TP_DMS1, dq3, dgq);
    }
    Dual qd[3];
    for (int i = 0; i < 3; ++i) qd[i] = Dual(q3[i] * CHARGECON, dq3[i] * CHARGECON);
    q[w] = Dual(0.0);
    q[N + w] = qd[1] + tmpq * (qd[1] + qd[2]);
    q[2 * N + w] = qd[2] + tmpq * (qd[1] + qd[2]);
    q[3 * N + w] = qd[0] * qMf;
    Dual *g = grdq + 27 * w;
    for (int d = 0; d < 3; ++d)
      for (int k = 0; k < 3; ++k) {
        const Dual g0 = Dual(gq[d][0][k] * CHARGECON, dgq[d][0][k] * CHARGECON);
        const Dual g1 = Dual(gq[d][1][k] * CHARGECON, dgq[d][1][k] * CHARGECON);
        const Dual g2 = Dual(gq[d][2][k] * CHARGECON, dgq[d][2][k] * CHARGECON);
        g[d * 9 + 0 * 3 + k] = g0 + tmpq * (g0 + g1);
        g[d * 9 + 1 * 3 + k] = g1 + tmpq * (g0 + g1);
        g[d * 9 + 2 * 3 + k] = g2 - 2.0 * tmpq * (g0 + g1);
      }
    for (int k = 0; k < 3; ++k) {
      dR[(0 * N + w) * 3 + k] = Dual(dr1[0][k]);
      dR[(1 * N + w) * 3 + k] = Dual(dr1[1][k]);
      dR[(2 * N + w) * 3 + k] = Dual(dr1[2][k]);
      dR[(3 * N + w) * 3 + k] = Dual(0.0);
    }
    for (int t = 0; t < 4; ++t) {
      phi[t * N + w] = Dual(0.0);
      for (int k = 0; k < 3; ++k) Efq[(t * N + w) * 3 + k] = Dual(0.0);
    }
  }
  const double u = block_sum(umon, red);
  if (tid == 0) *W.umon = Dual(u);
}

// The adjoint's position derivatives of the screening functions ts_n(r^2)
// follow the chain the gradient of pot_ttm uses, ts_(n+1) = -1/((2n+1) r)
// d ts_n/dr (the erfc-screened and Thole tensors of smear.f90), rather than
// differentiating the A&S erfc polynomial and the truncated Gamma(2/3) series
// themselves: the reference's gradient departs from the exact derivative of
// its energy by ~1e-5 relative there, and the adjoint differentiates the
// gradient as computed.  d ts_n = -(2n+1)/2 ts_(n+1) d(r^2).
__device__ __forceinline__ void chain_d(Dual &ts, int n, double ts_next, double dd2) {
  ts.d = -0.5 * (2 * n + 1) * ts_next * dd2;
}

// MODE TAN_PARAMS: one parameter direction per workgroup, plain FP64
// geometry (GT = double); TAN_GAMMA_M: dual site positions and phases
// (GT = Dual) along dr/dgammaM.  (The adjoint has kernels of its own.)
template <int MODE>
__global__ __launch_bounds__(TAN_BLOCK) void k_ttm_tangent(SysConst c, TanArgs a) {
  constexpr bool GD = MODE != TAN_PARAMS;
  using GT = std::conditional_t<GD, Dual, double>;
  const int b = blockIdx.x, dir = blockIdx.y, ndir = gridDim.y, tid = threadIdx.x;
  const int N = c.N, ns = 4 * N, nd = c.nd, tdip = c.tdip, nds = nd * N, nk = c.nk;
  const int tend = tdip + nd;  // dipole site types [tdip, tend): M (TTM3-F) or O, H1, H2 (TTM2.1-F)
  const double *Rs = a.cfg + (size_t)b * a.cfg_stride;
  Phases ph;
  ph.ns = ns;
  ph.kmax = c.kmax;
  ph.lmax = c.lmax;
  ph.N = N;
  ph.dS = Rs + a.ds_off;
  ph.tx = (const double2 *)(Rs + (size_t)ns * 3);
  ph.ty = ph.tx + (size_t)(c.hmax + 1) * ns;
  ph.tz = ph.ty + (size_t)(2 * c.kmax + 1) * ns;
  // site s's position, with its derivative along the geometric direction in
  // the dual-geometry instances
  auto site = [&](int s, GT r[3]) {
    for (int k = 0; k < 3; ++k) r[k] = Rs[3 * s + k];
    if constexpr (GD)
      for (int k = 0; k < 3; ++k) r[k].d = ph.dS[3 * s + k];
  };
  const TanWs W(a.ws + ((size_t)b * ndir + dir) * a.ws_stride, c);
  Dual *q = W.q, *phi = W.phi, *Efq = W.Efq, *dR = W.dR, *dip = W.dip, *old = W.old,
       *Efd = W.Efd, *grdq = W.grdq, *Sq = W.Sq, *Sm = W.Sm;

  __shared__ TanPar P;
  __shared__ double red[TAN_BLOCK];
  if (tid == 0) {
    const bool seed = MODE == TAN_PARAMS && !a.dms_coef;
    auto par = [&](int i) { return Dual(a.theta[i], (seed && i == dir) ? 1.0 : 0.0); };
    for (int i = 0; i < 5; ++i) P.vdw[i] = par(i);
    P.polar[0] = par(5);
    P.polar[1] = par(6);
    P.polar[2] = par(6);
    P.polar[3] = par(7);
    // polfac = (polfac^(1/6))^-3 (potential.f90:157-160)
    const Dual f6[4] = {dpow(par(8), 1.0 / 6.0), dpow(par(9), 1.0 / 6.0), dpow(par(9), 1.0 / 6.0),
                        dpow(par(10), 1.0 / 6.0)};
    Dual pf[4];
    for (int i = 0; i < 4; ++i) pf[i] = Dual(1.0) / (f6[i] * f6[i] * f6[i]);
    const Dual aDD = par(11), aCC = par(12);
    for (int i = 0; i < 4; ++i)
      for (int j = 0; j < 4; ++j) {
        P.apCC[i][j] = aCC * pf[i] * pf[j];
        P.raCC[i][j] = P.apCC[i][j].v > 0.0 ? dpow(P.apCC[i][j], 1.0 / 3.0) : Dual(0.0);
        P.apDD[i][j] = aDD * pf[i] * pf[j];
      }
    P.lrc = Dual(c.Uvdw_lrc, (seed && dir < 3) ? a.lrc_coef[dir] : 0.0);
  }
  __syncthreads();
  // gammaM, which redistributes the M-site gradient (pot_ttm.f90:597-602)
  GT gM = c.gammaM;
  if constexpr (MODE == TAN_GAMMA_M) gM.d = 1.0;
  // charges, their gradients, the monomer gradients and energy: k_tangent_monomer

  // ---- real space: vdW and charge-charge terms (pot_ttm.f90:159-228), per site
  Dual uvdw = 0.0;
  for (int s = tid; s < ns; s += TAN_BLOCK) {
    const int iw = s % N, ti = s / N;
    const double *ROi = Rs + 3 * iw;
    GT Ri[3];
    site(s, Ri);
    Dual pv = 0.0, ef[3] = {0.0, 0.0, 0.0}, gv[3] = {0.0, 0.0, 0.0};
    for (int jw = 0; jw < N; ++jw) {
      if (jw == iw) continue;
      const double *ROj = Rs + 3 * jw;
      double Rij[3] = {ROi[0] - ROj[0], ROi[1] - ROj[1], ROi[2] - ROj[2]};
      minimg(c, Rij[0], Rij[1], Rij[2]);
      const double d2 = norm2_exact(Rij[0], Rij[1], Rij[2]);
      if (!(d2 < c.rc2)) continue;
      if (ti == 0) {
        const double dRij = sqrt(d2), R2i = 1.0 / d2, R4i = R2i * R2i, R6i = R4i * R2i,
                     R8i = R6i * R2i, x = dRij - c.rc1;
        const Dual ex = P.vdw[3] * dexp(-(P.vdw[4] * dRij));
        const Dual uij = R6i * ((P.vdw[0] * R6i + P.vdw[1] * R4i) + P.vdw[2]) + ex;
        const Dual fsc = -(R8i * 6.0 * P.vdw[2] + ex * P.vdw[4] / dRij +
                           Dual(c.shiftA * (x * x) + c.shiftB * (x * x * x)));
        for (int k = 0; k < 3; ++k) gv[k] += fsc * Rij[k];
        if (iw < jw) uvdw += uij;
      }
      GT Ra[3];
      for (int k = 0; k < 3; ++k) Ra[k] = Ri[k] + (Rij[k] - ROi[k] + ROj[k]);
      for (int tj = ti == 0 ? 1 : 0; tj < 4; ++tj) {
        const int sj = tj * N + jw;
        GT Rj[3];
        site(sj, Rj);
        GT r[3] = {Ra[0] - Rj[0], Ra[1] - Rj[1], Ra[2] - Rj[2]};
        minimg(c, r[0], r[1], r[2]);
        const GT d2s = r[0] * r[0] + r[1] * r[1] + r[2] * r[2];
        Dual ts0, ts1;
        smear01<true, Dual>(c, as_dual(d2s), P.apCC[ti][tj], P.raCC[ti][tj], ts0, ts1);
        const Dual qj = q[sj];
        pv += ts0 * qj;
        const Dual f = ts1 * qj;
        for (int k = 0; k < 3; ++k) ef[k] += f * r[k];
      }
    }
    phi[s] += pv;
    for (int k = 0; k < 3; ++k) {
      Efq[3 * s + k] += ef[k];
      dR[3 * s + k] += gv[k];
    }
  }
  __syncthreads();

  // ---- Ewald self energy and intramolecular exclusions (pot_ttm.f90:232-261)
  for (int w = tid; w < N; w += TAN_BLOCK) {
    for (int t = 1; t < 4; ++t) phi[t * N + w] -= c.self_fac * q[t * N + w];
    for (int ti = 0; ti < 3; ++ti)
      for (int tj = ti + 1; tj < 4; ++tj) {
        const int si = ti * N + w, sj = tj * N + w;
        GT Ri[3], Rj[3];
        site(si, Ri);
        site(sj, Rj);
        GT r[3] = {Ri[0] - Rj[0], Ri[1] - Rj[1], Ri[2] - Rj[2]};
        minimg(c, r[0], r[1], r[2]);
        const GT d2x = r[0] * r[0] + r[1] * r[1] + r[2] * r[2];
        GT ts0, ts1;
        self1(c, d2x, ts0, ts1);
        phi[si] += ts0 * q[sj];
        phi[sj] += ts0 * q[si];
        for (int k = 0; k < 3; ++k) {
          Efq[3 * si + k] += ts1 * q[sj] * r[k];
          Efq[3 * sj + k] -= ts1 * q[si] * r[k];
        }
      }
  }
  __syncthreads();

  // ---- reciprocal space, charges (ewald_std_qq, ewald.f90:1-52)
  for (int k = tid; k < nk; k += TAN_BLOCK) {
    const int4 h = a.khkl[k];
    const double4 kv = a.kv[k];
    Dual rQ = 0.0, iQ = 0.0;
    for (int s = N; s < ns; ++s) {
      GT ck, sk;
      ph.at(s, h, kv, ck, sk);
      rQ += q[s] * ck;
      iQ += q[s] * sk;
    }
    Sq[2 * k] = rQ;
    Sq[2 * k + 1] = iQ;
  }
  __syncthreads();
  const int Gs = site_lanes(ns), Gd = site_lanes(nds);
  for (int s = tid / Gs; s < ns; s += TAN_BLOCK / Gs) {
    Dual ef[3] = {0.0, 0.0, 0.0}, pv = 0.0;
    for (int k = tid % Gs; k < nk; k += Gs) {
      const int4 h = a.khkl[k];
      const double4 kv = a.kv[k];
      const double p4vAk = kv.w;
      GT ck, sk;
      ph.at(s, h, kv, ck, sk);
      const Dual rQ = Sq[2 * k], iQ = Sq[2 * k + 1];
      const Dual t = p4vAk * (ck * iQ - sk * rQ);
      ef[0] -= t * kv.x;
      ef[1] -= t * kv.y;
      ef[2] -= t * kv.z;
      pv += p4vAk * (ck * rQ + sk * iQ);
    }
    for (int k = 0; k < 3; ++k) ef[k] = group_sum(ef[k], Gs);
    pv = group_sum(pv, Gs);
    if (tid % Gs == 0) {
      for (int k = 0; k < 3; ++k) Efq[3 * s + k] += ef[k];
      if (s >= N) phi[s] += pv;
    }
  }
  __syncthreads();

  // ---- Uelec, the charge-field gradient (pot_ttm.f90:273-276), initial dipoles
  Dual uel = 0.0;
  for (int s = N + tid; s < ns; s += TAN_BLOCK) {
    uel += q[s] * phi[s];
    for (int k = 0; k < 3; ++k) dR[3 * s + k] -= q[s] * Efq[3 * s + k];
  }
  for (int i = tid; i < nds; i += TAN_BLOCK) {
    const int t = tdip + i / N, s = t * N + i % N;
    for (int k = 0; k < 3; ++k) {
      dip[3 * i + k] = P.polar[t] * Efq[3 * s + k];
      old[3 * i + k] = Dual(0.0);
    }
  }
  __syncthreads();

  // ---- SOR dipole iterations (pot_ttm.f90:306-392)
  int iters = c.maxiter;
  const double om = c.sor;
  for (int it = 1; it <= c.maxiter; ++it) {
    for (int i = tid; i < nds; i += TAN_BLOCK) {
      const int ti = tdip + i / N, iw = i % N, s = ti * N + iw;
      const double *ROi = Rs + 3 * iw;
      GT Ri[3];
      site(s, Ri);
      Dual e[3] = {0.0, 0.0, 0.0};
      for (int jw = 0; jw < N; ++jw) {
        if (jw == iw) continue;
        const double *ROj = Rs + 3 * jw;
        double Rij[3] = {ROi[0] - ROj[0], ROi[1] - ROj[1], ROi[2] - ROj[2]};
        minimg(c, Rij[0], Rij[1], Rij[2]);
        if (!(norm2_exact(Rij[0], Rij[1], Rij[2]) < c.rc2)) continue;
        double R0[3] = {Rij[0] - ROi[0] + ROj[0], Rij[1] - ROi[1] + ROj[1], Rij[2] - ROi[2] + ROj[2]};
        minimg(c, R0[0], R0[1], R0[2]);
        for (int tj = tdip; tj < tend; ++tj) {
          const int sj = tj * N + jw, j = (tj - tdip) * N + jw;
          GT Rj[3], r[3];
          site(sj, Rj);
          for (int k = 0; k < 3; ++k) r[k] = Ri[k] + R0[k] - Rj[k];
          minimg(c, r[0], r[1], r[2]);
          Dual t1, t2, o[3];
          const GT r2 = r[0] * r[0] + r[1] * r[1] + r[2] * r[2];
          smear2<true, Dual>(c, as_dual(r2), P.apDD[ti][tj], t1, t2);
          dd3d(r, t1, t2, dip + 3 * j, o);
          for (int k = 0; k < 3; ++k) e[k] += o[k];
        }
      }
      // dipole sites of the same molecule (TTM2.1-F, pot_ttm.f90:344-365)
      for (int tj = tdip; tj < tend; ++tj) {
        if (tj == ti) continue;
        const int sj = tj * N + iw, j = (tj - tdip) * N + iw;
        GT Rj[3];
        site(sj, Rj);
        GT r[3] = {Ri[0] - Rj[0], Ri[1] - Rj[1], Ri[2] - Rj[2]};
        minimg(c, r[0], r[1], r[2]);
        Dual t1, t2, o[3];
        const GT r2 = r[0] * r[0] + r[1] * r[1] + r[2] * r[2];
        smear2<true, Dual>(c, as_dual(r2), P.apDD[ti][tj], t1, t2);
        dd3d(r, t1, t2, dip + 3 * j, o);
        for (int k = 0; k < 3; ++k) e[k] += o[k];
      }
      for (int k = 0; k < 3; ++k) Efd[3 * i + k] = e[k];
    }
    // structure factor of the dipoles (ewald_std_dd, ewald.f90:56-119)
    for (int k = tid; k < nk; k += TAN_BLOCK) {
      const int4 h = a.khkl[k];
      const double4 kv = a.kv[k];
      Dual rQ = 0.0, iQ = 0.0;
      for (int i = 0; i < nds; ++i) {
        const int s = (tdip + i / N) * N + i % N;
        GT ck, sk;
        ph.at(s, h, kv, ck, sk);
        const Dual dK = dip[3 * i] * kv.x + dip[3 * i + 1] * kv.y + dip[3 * i + 2] * kv.z;
        rQ -= dK * sk;
        iQ += dK * ck;
      }
      Sm[2 * k] = rQ;
      Sm[2 * k + 1] = iQ;
    }
    __syncthreads();
    double ss = 0.0;
    for (int i = tid / Gd; i < nds; i += TAN_BLOCK / Gd) {
      const int ti = tdip + i / N, s = ti * N + i % N;
      Dual e[3] = {0.0, 0.0, 0.0};
      for (int k = tid % Gd; k < nk; k += Gd) {
        const int4 h = a.khkl[k];
        const double4 kv = a.kv[k];
        GT ck, sk;
        ph.at(s, h, kv, ck, sk);
        const Dual t = kv.w * (ck * Sm[2 * k + 1] - sk * Sm[2 * k]);
        e[0] -= kv.x * t;
        e[1] -= kv.y * t;
        e[2] -= kv.z * t;
      }
      for (int k = 0; k < 3; ++k) e[k] = Efd[3 * i + k] + group_sum(e[k], Gd);
      if (tid % Gd != 0) continue;
      for (int k = 0; k < 3; ++k) {
        const Dual mu = dip[3 * i + k];
        const Dual ek = e[k] + Efq[3 * s + k] + c.fac_dd * mu;
        const Dual nu = (1.0 - om) * mu + (om * P.polar[ti]) * ek;
        const double df = nu.v - old[3 * i + k].v;
        ss += df * df;
        dip[3 * i + k] = nu;
      }
    }
    const double sum = block_sum(ss, red);
    if (c.stath * sqrt(sum) < c.peps) {
      iters = it;
      break;
    }
    for (int i = tid; i < 3 * nds; i += TAN_BLOCK) old[i] = dip[i];
    __syncthreads();
  }
  __syncthreads();

  // ---- Uind (pot_ttm.f90:390) and the final real-space forces (pot_ttm.f90:399-542)
  Dual uind = 0.0;
  for (int i = tid; i < nds; i += TAN_BLOCK) {
    const int s = (tdip + i / N) * N + i % N;
    for (int k = 0; k < 3; ++k) uind += dip[3 * i + k] * Efq[3 * s + k];
  }
  for (int s = tid; s < ns; s += TAN_BLOCK) {
    const int iw = s % N, ti = s / N;
    const bool adip = ti >= tdip && ti < tend;
    const double *ROi = Rs + 3 * iw;
    GT Ri[3];
    site(s, Ri);
    const Dual qi = q[s];
    Dual di[3] = {0.0, 0.0, 0.0};
    if (adip)
      for (int k = 0; k < 3; ++k) di[k] = dip[3 * ((ti - tdip) * N + iw) + k];
    Dual g[3] = {0.0, 0.0, 0.0}, pv = 0.0;
    for (int jw = 0; jw < N; ++jw) {
      const bool same = jw == iw;
      double R0[3] = {0.0, 0.0, 0.0};
      if (!same) {
        const double *ROj = Rs + 3 * jw;
        double Rij[3] = {ROi[0] - ROj[0], ROi[1] - ROj[1], ROi[2] - ROj[2]};
        minimg(c, Rij[0], Rij[1], Rij[2]);
        if (!(norm2_exact(Rij[0], Rij[1], Rij[2]) < c.rc2)) continue;
        for (int k = 0; k < 3; ++k) R0[k] = Rij[k] - ROi[k] + ROj[k];
        minimg(c, R0[0], R0[1], R0[2]);
      }
      for (int tj = 0; tj < 4; ++tj) {
        if (same && tj == ti) continue;
        const int sj = tj * N + jw;
        const bool bdip = tj >= tdip && tj < tend;
        GT Rj[3], r[3];
        site(sj, Rj);
        for (int k = 0; k < 3; ++k) r[k] = same ? Ri[k] - Rj[k] : Ri[k] + R0[k] - Rj[k];
        minimg(c, r[0], r[1], r[2]);
        const GT d2 = r[0] * r[0] + r[1] * r[1] + r[2] * r[2];
        const Dual qj = q[sj];
        Dual dj[3] = {0.0, 0.0, 0.0};
        if (bdip)
          for (int k = 0; k < 3; ++k) dj[k] = dip[3 * ((tj - tdip) * N + jw) + k];
        if (adip && bdip) {
          // dipole-dipole: d_i . T3(r) . d_j with T3 the third-rank tensor of PBCsmear3
          Dual t1, t2, t3;
          smear3<true, Dual>(c, as_dual(d2), P.apDD[ti][tj], t1, t2, t3);
          const Dual dir_ = di[0] * r[0] + di[1] * r[1] + di[2] * r[2];
          const Dual djr = dj[0] * r[0] + dj[1] * r[1] + dj[2] * r[2];
          const Dual dd = di[0] * dj[0] + di[1] * dj[1] + di[2] * dj[2];
          const Dual a15 = 15.0 * t3 * dir_ * djr, a3 = 3.0 * t2;
          for (int k = 0; k < 3; ++k) g[k] += a15 * r[k] - a3 * (dir_ * dj[k] + djr * di[k] + dd * r[k]);
        }
        Dual qdqd[3];
        for (int k = 0; k < 3; ++k) qdqd[k] = qj * di[k] - qi * dj[k];
        Dual ts1 = 0.0, ts2 = 0.0;
        bool qd = true;
        if (same) {
          GT s1, s2;
          self2(c, d2, s1, s2);
          ts1 = s1;
          ts2 = s2;
        } else {
          const double qsq = qdqd[0].v * qdqd[0].v + qdqd[1].v * qdqd[1].v + qdqd[2].v * qdqd[2].v;
          qd = qsq > 1e-9;
          if (qd) smear2<true, Dual>(c, as_dual(d2), P.apCC[ti][tj], ts1, ts2);
        }
        if (qd) {
          Dual o[3];
          dd3d(r, ts1, ts2, qdqd, o);
          for (int k = 0; k < 3; ++k) g[k] += o[k];
        }
        pv += ts1 * (dj[0] * r[0] + dj[1] * r[1] + dj[2] * r[2]);
      }
    }
    for (int k = 0; k < 3; ++k) dR[3 * s + k] += g[k];
    phi[s] += pv;
  }
  __syncthreads();

  // ---- reciprocal space, dipole forces (ewald_std_qd, ewald.f90:123-226); the
  // dipole structure factor is the one of the last SOR iteration's input
  for (int s = tid / Gs; s < ns; s += TAN_BLOCK / Gs) {
    const int iw = s % N, ti = s / N;
    const bool sdip = ti >= tdip && ti < tend, schg = s >= N;
    const Dual qs = q[s];
    Dual mu[3] = {0.0, 0.0, 0.0};
    if (sdip)
      for (int k = 0; k < 3; ++k) mu[k] = dip[3 * ((ti - tdip) * N + iw) + k];
    Dual g[3] = {0.0, 0.0, 0.0}, pv = 0.0;
    for (int k = tid % Gs; k < nk; k += Gs) {
      const int4 h = a.khkl[k];
      const double4 kv = a.kv[k];
      const double p4vAk = kv.w;
      GT ck, sk;
      ph.at(s, h, kv, ck, sk);
      const Dual rQm = Sm[2 * k], iQm = Sm[2 * k + 1];
      if (schg) {
        pv += p4vAk * (ck * rQm + sk * iQm);
        const Dual t = qs * p4vAk * (ck * iQm - sk * rQm);
        g[0] += t * kv.x;
        g[1] += t * kv.y;
        g[2] += t * kv.z;
      }
      if (sdip) {
        const Dual dK = mu[0] * kv.x + mu[1] * kv.y + mu[2] * kv.z;
        const Dual t = dK * p4vAk * (ck * (Sq[2 * k] + rQm) + sk * (Sq[2 * k + 1] + iQm));
        g[0] -= t * kv.x;
        g[1] -= t * kv.y;
        g[2] -= t * kv.z;
      }
    }
    for (int k = 0; k < 3; ++k) g[k] = group_sum(g[k], Gs);
    pv = group_sum(pv, Gs);
    if (tid % Gs == 0) {
      for (int k = 0; k < 3; ++k) dR[3 * s + k] += g[k];
      phi[s] += pv;
    }
  }
  __syncthreads();

  // ---- charge chain rule (pot_ttm.f90:556-584), M-site redistribution
  // (pot_ttm.f90:597-602), loss terms
  double lossg = 0.0;
  for (int w = tid; w < N; w += TAN_BLOCK) {
    const Dual *gq = grdq + 27 * w;
    const Dual p1 = phi[N + w], p2 = phi[2 * N + w], pm = phi[3 * N + w];
    Dual G[3][3];  // atoms O, H1, H2
    for (int k = 0; k < 3; ++k) {
      const Dual dg1 = gq[0 * 9 + 0 * 3 + k] * p1 + gq[0 * 9 + 1 * 3 + k] * p2 + gq[0 * 9 + 2 * 3 + k] * pm;
      const Dual dg2 = gq[1 * 9 + 0 * 3 + k] * p1 + gq[1 * 9 + 1 * 3 + k] * p2 + gq[1 * 9 + 2 * 3 + k] * pm;
      const Dual dg0 = gq[2 * 9 + 0 * 3 + k] * p1 + gq[2 * 9 + 1 * 3 + k] * p2 + gq[2 * 9 + 2 * 3 + k] * pm;
      const Dual dM = dR[(3 * N + w) * 3 + k];
      G[1][k] = (dR[(N + w) * 3 + k] + dg1) + 0.5 * gM * dM;
      G[2][k] = (dR[(2 * N + w) * 3 + k] + dg2) + 0.5 * gM * dM;
      G[0][k] = (dR[w * 3 + k] + dg0) + (1.0 - gM) * dM;
    }
    const size_t a0 = ((size_t)b * 3 * N + 3 * w) * 3;
    for (int at = 0; at < 3; ++at)
      for (int k = 0; k < 3; ++k) {
        lossg += a.gw[a0 + 3 * at + k] * G[at][k].d;
        if (a.dG) a.dG[((size_t)b * ndir + dir) * 9 * N + 9 * w + 3 * at + k] = G[at][k].d;
      }
  }
  const double Ev = W.umon->v + block_sum(uvdw.v, red) + 0.5 * block_sum(uel.v, red) -
                    0.5 * block_sum(uind.v, red) + P.lrc.v;
  const double Ed = block_sum(uvdw.d, red) + 0.5 * block_sum(uel.d, red) - 0.5 * block_sum(uind.d, red) +
                    P.lrc.d;
  const double lg = block_sum(lossg, red);
  if (tid == 0) {
    double *o = a.out + ((size_t)b * ndir + dir) * 4;
    o[0] = Ev;
    o[1] = Ed;
    o[2] = a.ew[b] * Ed + lg;
    o[3] = (double)iters;
  }
}

// ---------------------------------------------------------------------------
// The adjoint.  A configuration's sweep is cut into kernels, each spread over
// as many workgroups as its sites, k-vectors or site pairs fill: one workgroup
// per configuration (64 boxes of 32 H2O: 64 workgroups of a 256-CU device, and
// 32 of 256 lanes busy in the dipole field) took 8.8 ms.  The dipole solve is
// the dense one of the force path, on dual numbers: the matrix and its
// derivative along the positions' direction are formed once (k_adj_build) and
// an iteration is a product with them (k_adj_solve).  64 five-water clusters
// and 64 boxes of 32 H2O side by side: 8.8 -> 0.5 ms.  Larger systems, whose
// matrix grows with the square of the sites, take an iteration pass by pass
// from the positions (k_adj_sfac, k_adj_step, k_adj_test; adjoint_plan).
//
// Values are evaluated in plain FP64 and their position derivatives follow
// chain_d; the Thole derivatives d ts / d a come from duals along a.
// ---------------------------------------------------------------------------
constexpr int ADJ_G = 16;                       // lanes per site of the pair loops
constexpr int ADJ_SPB = TAN_BLOCK / ADJ_G;      // sites per workgroup of them
constexpr int ADJ_NV = 11, ADJ_NA = 10;         // partial sums per workgroup
constexpr int ADJ_BW = 8;                       // waves of k_adj_build
constexpr int ADJ_SOLVE = 1024;

struct AdjArgs {
  TanArgs t;
  Dual *mat;             // [slice][D][D] dipole matrix, D = 3 nd N
  int b0;                // first configuration of the slice
  int2 *state;           // [P] of the pass-by-pass solve: active, iterations done
  double *pv, *pa;       // [P][pair workgroups][ADJ_NV], [ADJ_NA]
  const int4 *cols;      // kz-columns and their first k-vectors
  const int *colk;
  double pf[4], dpf[4];  // polfac^(-1/2) per site type and its derivative by polfac
};

__host__ __device__ inline int adj_pair_blocks(const SysConst &c) {
  return (4 * c.N + ADJ_SPB - 1) / ADJ_SPB;
}

// Configuration b's tables and sites.
struct AdjCfg {
  const double *Rs, *dS;
  Phases ph;
  __device__ AdjCfg(const SysConst &c, const TanArgs &a, int b) {
    const int ns = 4 * c.N;
    Rs = a.cfg + (size_t)b * a.cfg_stride;
    dS = Rs + a.ds_off;
    ph.ns = ns;
    ph.kmax = c.kmax;
    ph.lmax = c.lmax;
    ph.N = c.N;
    ph.dS = dS;
    ph.tx = (const double2 *)(Rs + (size_t)ns * 3);
    ph.ty = ph.tx + (size_t)(c.hmax + 1) * ns;
    ph.tz = ph.ty + (size_t)(2 * c.kmax + 1) * ns;
  }
  // minimum-image vector from site sj to site si, with its derivative
  __device__ __forceinline__ void vec(const SysConst &c, int si, int sj, Dual r[3]) const {
    for (int k = 0; k < 3; ++k)
      r[k] = Dual(Rs[3 * si + k] - Rs[3 * sj + k], dS[3 * si + k] - dS[3 * sj + k]);
    minimg(c, r[0], r[1], r[2]);
  }
  // whether molecules i and j are within the cut-off, and their O-O vector
  __device__ __forceinline__ bool within(const SysConst &c, int i, int j, double v[3]) const {
    for (int k = 0; k < 3; ++k) v[k] = Rs[3 * i + k] - Rs[3 * j + k];
    minimg(c, v[0], v[1], v[2]);
    return norm2_exact(v[0], v[1], v[2]) < c.rc2;
  }
};

// Sums of n values per lane over the workgroup into out (lane 0 writes).
template <int n>
__device__ __forceinline__ void block_sums(double *v, double (*red)[TAN_BLOCK / 64], double *out) {
  for (int i = 0; i < n; ++i) {
    v[i] = group_sum<64>(v[i]);
    if ((threadIdx.x & 63) == 0) red[i][threadIdx.x >> 6] = v[i];
  }
  __syncthreads();
  if (threadIdx.x < n) {
    double s = 0.0;
    for (int w = 0; w < TAN_BLOCK / 64; ++w) s += red[threadIdx.x][w];
    out[threadIdx.x] = s;
  }
}

// Real-space charge terms of a site (pot_ttm.f90:159-261): the potential at
// the charged sites, the field at the dipole sites, the vdW sums at the
// oxygens; ADJ_G lanes per site over the molecules.
__global__ __launch_bounds__(TAN_BLOCK) void k_adj_pair_q(SysConst c, AdjArgs x) {
  __shared__ double red[ADJ_NV][TAN_BLOCK / 64];
  const TanArgs &a = x.t;
  const int b = blockIdx.y, N = c.N, ns = 4 * N;
  const AdjCfg g(c, a, b);
  const TanWs W(a.ws + (size_t)b * a.ws_stride, c);
  const int s0 = blockIdx.x * ADJ_SPB + threadIdx.x / ADJ_G, lane = threadIdx.x % ADJ_G;
  const bool valid = s0 < ns;
  const int s = valid ? s0 : 0, iw = s % N, ti = s / N;
  const bool chg = ti > 0, adip = ti >= c.tdip && ti < c.tdip + c.nd;
  Dual pv = 0.0, ef[3] = {0.0, 0.0, 0.0};
  double v[ADJ_NV] = {0};  // uvdw, d Uvdw / d(vdwA..E), gw . dG / d(vdwA..E)
  for (int jw = lane; valid && jw < N; jw += ADJ_G) {
    const bool same = jw == iw;
    double Rij[3];
    if (!same && !g.within(c, iw, jw, Rij)) continue;
    if (ti == 0 && !same) {
      const double d2 = norm2_exact(Rij[0], Rij[1], Rij[2]);
      const double d = sqrt(d2), R2i = 1.0 / d2, R4i = R2i * R2i, R6i = R4i * R2i, R8i = R6i * R2i;
      const double e = exp(-(c.vdwE * d));
      const double *gO = a.gw + ((size_t)b * 3 * N + 3 * iw) * 3;
      const double gr = gO[0] * Rij[0] + gO[1] * Rij[1] + gO[2] * Rij[2];
      if (iw < jw) {
        v[0] += R6i * ((c.vdwA * R6i + c.vdwB * R4i) + c.vdwC) + c.vdwD * e;
        v[1] += R6i * R6i;
        v[2] += R6i * R4i;
        v[3] += R6i;
        v[4] += e;
        v[5] -= c.vdwD * d * e;
      }
      // the gradient as computed: its vdW force (pot_ttm.f90:176) has no
      // vdwA, vdwB terms
      v[8] -= 6.0 * R8i * gr;
      v[9] -= e * c.vdwE / d * gr;
      v[10] -= c.vdwD * e * (1.0 - c.vdwE * d) / d * gr;
    }
    if (!chg && !adip) continue;
    for (int tj = 0; tj < 4; ++tj) {
      if ((same && tj == ti) || tj == 0) continue;  // the oxygens carry no charge
      const int sj = tj * N + jw;
      Dual r[3];
      g.vec(c, s, sj, r);
      const Dual d2 = r[0] * r[0] + r[1] * r[1] + r[2] * r[2];
      double t0, t1, t2 = 0.0, u1;
      if (same) {
        self1(c, d2.v, t0, t1);
        if (adip) self2(c, d2.v, u1, t2);
      } else {
        smear01(c, d2.v, c.apolCC[ti][tj], c.raCC[ti][tj], t0, t1);
        if (adip) smear2(c, d2.v, c.apolCC[ti][tj], u1, t2);
      }
      const Dual qj = W.q[sj];
      Dual ts0 = t0;
      chain_d(ts0, 0, t1, d2.d);
      pv += ts0 * qj;
      if (adip) {
        Dual ts1 = t1;
        chain_d(ts1, 1, t2, d2.d);
        const Dual f = ts1 * qj;
        for (int k = 0; k < 3; ++k) ef[k] += f * r[k];
      }
    }
  }
  pv = group_sum(pv, ADJ_G);
  for (int k = 0; k < 3; ++k) ef[k] = group_sum(ef[k], ADJ_G);
  if (valid && lane == 0) {
    W.phi[s] = chg ? pv - c.self_fac * W.q[s] : Dual(0.0);
    for (int k = 0; k < 3; ++k) W.Efq[3 * s + k] = ef[k];
  }
  block_sums<ADJ_NV>(v, red, x.pv + ((size_t)b * gridDim.x + blockIdx.x) * ADJ_NV);
}

// Structure factor of the charges, or of the dipoles (ewald.f90:1-119): of
// SOR iteration `it`'s input (odd iterations read dip and write old, even ones
// the other way round), with it = 0 of the last step's input, left in old.
// Four lanes per k-vector share its sites.
template <bool DIP>
__global__ __launch_bounds__(TAN_BLOCK) void k_adj_sfac(SysConst c, AdjArgs x, int it) {
  const TanArgs &a = x.t;
  const int b = blockIdx.y, N = c.N;
  if (it > 1 && !x.state[b].x) return;
  const AdjCfg g(c, a, b);
  const TanWs W(a.ws + (size_t)b * a.ws_stride, c);
  const Dual *dip = it & 1 ? W.dip : W.old;
  const int k = blockIdx.x * (TAN_BLOCK / 4) + threadIdx.x / 4, u = threadIdx.x % 4;
  if (k >= c.nk) return;  // alike over the four lanes
  const int4 h = a.khkl[k];
  const double4 kv = a.kv[k];
  const int s0 = DIP ? c.tdip * N : N, n = DIP ? c.nd * N : 3 * N;
  Dual re = 0.0, im = 0.0;
  for (int i = u; i < n; i += 4) {
    Dual ck, sk;
    g.ph.at(s0 + i, h, kv, ck, sk);
    if (DIP) {
      const Dual *m = dip + 3 * i;
      const Dual dk = m[0] * kv.x + m[1] * kv.y + m[2] * kv.z;
      re -= dk * sk;
      im += dk * ck;
    } else {
      const Dual q = W.q[s0 + i];
      re += q * ck;
      im += q * sk;
    }
  }
  re = group_sum(re, 4);
  im = group_sum(im, 4);
  if (u == 0) {
    Dual *S = DIP ? W.Sm : W.Sq;
    S[2 * k] = re;
    S[2 * k + 1] = im;
  }
}

// Reciprocal-space potential at the charged sites, field at the dipole sites
// and starting dipoles (ewald.f90:45-49, pot_ttm.f90:281-297), a wave per
// site; DIP: the potential of the dipoles (ewald.f90:184-193) onto dR, where
// k_adj_pair_d left its real-space part.
template <bool DIP>
__global__ __launch_bounds__(TAN_BLOCK) void k_adj_field(SysConst c, AdjArgs x) {
  const TanArgs &a = x.t;
  const int b = blockIdx.y, N = c.N;
  const int s = blockIdx.x * (TAN_BLOCK / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (s >= 4 * N) return;
  const int ti = s / N;
  const bool chg = ti > 0, adip = !DIP && ti >= c.tdip && ti < c.tdip + c.nd;
  if (!chg && !adip) return;
  const AdjCfg g(c, a, b);
  const TanWs W(a.ws + (size_t)b * a.ws_stride, c);
  const Dual *S = DIP ? W.Sm : W.Sq;
  Dual ef[3] = {0.0, 0.0, 0.0}, pv = 0.0;
  for (int k = lane; k < c.nk; k += 64) {
    const double4 kv = a.kv[k];
    Dual ck, sk;
    g.ph.at(s, a.khkl[k], kv, ck, sk);
    const Dual re = S[2 * k], im = S[2 * k + 1];
    pv += kv.w * (ck * re + sk * im);
    if (adip) {
      const Dual t = kv.w * (ck * im - sk * re);
      ef[0] -= t * kv.x;
      ef[1] -= t * kv.y;
      ef[2] -= t * kv.z;
    }
  }
  pv = group_sum(pv, 64);
  if (adip)
    for (int k = 0; k < 3; ++k) ef[k] = group_sum(ef[k], 64);
  if (lane != 0) return;
  if (DIP) {
    W.dR[s] += pv;
    return;
  }
  if (chg) W.phi[s] += pv;
  if (adip)
    for (int k = 0; k < 3; ++k) {
      const Dual e = W.Efq[3 * s + k] + ef[k];
      W.Efq[3 * s + k] = e;
      W.dip[3 * (s - c.tdip * N) + k] = c.polar[ti] * e;
    }
}

// The dipole matrix with its derivative along the positions' direction: an
// 8 x 8 tile of dipole-site pairs (i <= j) per workgroup, a lane per pair, the
// kz-columns dealt to the waves (sums added in wave order).  With
// phi = k.(r_i - r_j) the reciprocal part is -sum w k k cos phi and its
// derivative +sum w k k (k.dr) sin phi: along a column kx and ky are fixed, so
// the sums over kz of w kz^n cos phi (n <= 2) and w kz^n sin phi (n <= 3) give
// both.  Bound by FP64 issue: 13 operations per (pair, k); 64 boxes of 32 H2O
// (3450 k) 108 us, 40 % of the FP64 rate.
__global__ __launch_bounds__(64 * ADJ_BW) void k_adj_build(SysConst c, AdjArgs x) {
  __shared__ double part[ADJ_BW][12][64];
  const TanArgs &a = x.t;
  const int b = x.b0 + blockIdx.y, N = c.N, M = c.nd * N, sd = c.tdip * N;
  const AdjCfg g(c, a, b);
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nt = (M + 7) / 8;
  int ti = 0, t = blockIdx.x;
  while (t >= nt - ti) {
    t -= nt - ti;
    ++ti;
  }
  const int i = ti * 8 + lane / 8, j = (ti + t) * 8 + lane % 8;
  const bool valid = i < M && j < M && i <= j;
  const int si = sd + (valid ? i : 0), sj = sd + (valid ? j : 0);
  double dr[3];
  for (int k = 0; k < 3; ++k) dr[k] = g.dS[3 * si + k] - g.dS[3 * sj + k];
  auto diff = [&](const double2 *row) {
    const double2 p = row[si], q = row[sj];
    return make_double2(p.x * q.x + p.y * q.y, p.y * q.x - p.x * q.y);
  };
  auto mul = [](double2 p, double2 q) {
    return make_double2(p.x * q.x - p.y * q.y, p.y * q.x + p.x * q.y);
  };
  const size_t ns = 4 * (size_t)N;
  const double2 z1 =
      c.lmax >= 1 ? diff(g.ph.tz + (size_t)(c.lmax + 1) * ns) : make_double2(1.0, 0.0);
  double K[6] = {0, 0, 0, 0, 0, 0}, L[6] = {0, 0, 0, 0, 0, 0};  // xx, xy, yy, zz, xz, yz
  for (int n = wv; n < c.ncol; n += ADJ_BW) {
    const int4 cl = x.cols[n];
    const int k0 = x.colk[n];
    double2 e = mul(mul(diff(g.ph.tx + (size_t)cl.x * ns),
                        diff(g.ph.ty + (size_t)(cl.y + c.kmax) * ns)),
                    diff(g.ph.tz + (size_t)(cl.z + c.lmax) * ns));
    const double kx = a.kv[k0].x, ky = a.kv[k0].y;
    double C0 = 0, C1 = 0, C2 = 0, S0 = 0, S1 = 0, S2 = 0, S3 = 0;
    for (int m = 0; m < cl.w; ++m) {
      const double kz = a.kv[k0 + m].z, w = a.kv[k0 + m].w;
      const double p = w * e.x, q = w * e.y, pz = kz * p, qz = kz * q, qzz = kz * qz;
      C0 += p;
      C1 += pz;
      C2 = fma(kz, pz, C2);
      S0 += q;
      S1 += qz;
      S2 += qzz;
      S3 = fma(kz, qzz, S3);
      e = mul(e, z1);
    }
    const double D = kx * dr[0] + ky * dr[1];
    const double T0 = D * S0 + dr[2] * S1, T1 = D * S1 + dr[2] * S2, T2 = D * S2 + dr[2] * S3;
    K[0] -= kx * kx * C0;
    K[1] -= kx * ky * C0;
    K[2] -= ky * ky * C0;
    K[3] -= C2;
    K[4] -= kx * C1;
    K[5] -= ky * C1;
    L[0] += kx * kx * T0;
    L[1] += kx * ky * T0;
    L[2] += ky * ky * T0;
    L[3] += T2;
    L[4] += kx * T1;
    L[5] += ky * T1;
  }
  for (int q = 0; q < 6; ++q) {
    part[wv][q][lane] = K[q];
    part[wv][6 + q][lane] = L[q];
  }
  __syncthreads();
  if (wv != 0 || !valid) return;
  Dual E[6];
  for (int q = 0; q < 6; ++q) {
    double k = part[0][q][lane], l = part[0][6 + q][lane];
    for (int w = 1; w < ADJ_BW; ++w) {
      k += part[w][q][lane];
      l += part[w][6 + q][lane];
    }
    E[q] = Dual(k, l);
  }
  const int wi = i % N, wj = j % N, ui = c.tdip + i / N, uj = c.tdip + j / N;
  double R[3];
  if (wi == wj ? i != j : g.within(c, wi, wj, R)) {
    Dual r[3];
    g.vec(c, si, sj, r);
    const Dual d2 = r[0] * r[0] + r[1] * r[1] + r[2] * r[2];
    double u1, u2, u3;
    smear3(c, d2.v, c.apolDD[ui][uj], u1, u2, u3);
    Dual t1 = u1, t2 = u2;
    chain_d(t1, 1, u2, d2.d);
    chain_d(t2, 2, u3, d2.d);
    const Dual t3 = 3.0 * t2;
    E[0] += t3 * r[0] * r[0] - t1;
    E[1] += t3 * r[0] * r[1];
    E[2] += t3 * r[1] * r[1] - t1;
    E[3] += t3 * r[2] * r[2] - t1;
    E[4] += t3 * r[0] * r[2];
    E[5] += t3 * r[1] * r[2];
  }
  const size_t D = 3 * (size_t)M;
  Dual *m = x.mat + (size_t)blockIdx.y * D * D;
  const Dual v[3][3] = {{E[0], E[1], E[4]}, {E[1], E[2], E[5]}, {E[4], E[5], E[3]}};
  for (int p = 0; p < 3; ++p)
    for (int q = 0; q < 3; ++q) {
      m[(3 * i + p) * D + 3 * j + q] = v[p][q];
      if (i != j) m[(3 * j + p) * D + 3 * i + q] = v[p][q];
    }
}

// The SOR iterations (pot_ttm.f90:306-392) on duals, one workgroup per
// configuration: 16 lanes per matrix row, the matrix streamed from L2 (147 KB
// for 32 H2O, about 3 us per iteration: 64 B per clock into one CU), the
// dipoles in LDS.  Leaves the final dipoles in dip and the last step's input in
// old.
__global__ __launch_bounds__(ADJ_SOLVE) void k_adj_solve(SysConst c, AdjArgs x) {
  extern __shared__ Dual lds_mu[];  // [2][D]
  __shared__ double red[2][ADJ_SOLVE / 64];
  const TanArgs &a = x.t;
  const int b = x.b0 + blockIdx.x, N = c.N, D = 3 * c.nd * N, sd = c.tdip * N;
  const TanWs W(a.ws + (size_t)b * a.ws_stride, c);
  const Dual *m = x.mat + (size_t)blockIdx.x * D * D;
  const int g = threadIdx.x >> 4, u = threadIdx.x & 15;
  for (int e = threadIdx.x; e < D; e += ADJ_SOLVE) lds_mu[e] = W.dip[e];
  __syncthreads();
  const double om = c.sor;
  int cur = 0;
  for (int it = 1;; ++it) {
    const Dual *mu = lds_mu + (size_t)cur * D;
    Dual *nu = lds_mu + (size_t)(cur ^ 1) * D;
    double ss = 0.0;
    for (int row = g; row < D; row += ADJ_SOLVE / 16) {
      const Dual *A = m + (size_t)row * D;
      Dual f = 0.0;
#pragma unroll 4
      for (int col = u; col < D; col += 16) f += A[col] * mu[col];
      f = group_sum(f, 16);
      if (u == 0) {
        const Dual mr = mu[row], ek = f + W.Efq[3 * sd + row] + c.fac_dd * mr;
        const Dual nr = (1.0 - om) * mr + (om * c.polar[c.tdip + row / (3 * N)]) * ek;
        const double df = nr.v - (it == 1 ? 0.0 : mr.v);
        ss += df * df;
        nu[row] = nr;
      }
    }
    ss = pimd::group_sum<64>(ss);
    if ((threadIdx.x & 63) == 0) red[it & 1][threadIdx.x >> 6] = ss;
    __syncthreads();
    double sum = 0.0;
    for (int w = 0; w < ADJ_SOLVE / 64; ++w) sum += red[it & 1][w];
    cur ^= 1;
    if (c.stath * sqrt(sum) < c.peps || it >= c.maxiter) break;
  }
  for (int e = threadIdx.x; e < D; e += ADJ_SOLVE) {
    W.dip[e] = lds_mu[(size_t)cur * D + e];
    W.old[e] = lds_mu[(size_t)(cur ^ 1) * D + e];
  }
}

// One SOR iteration from the positions, a wave per dipole site: the
// reciprocal-space field of k_adj_sfac's structure factor (lanes over the
// k-vectors), the real-space one (lanes over the molecules) and the update.
// The squared change of a site's dipole goes into its Efd.
__global__ __launch_bounds__(TAN_BLOCK) void k_adj_step(SysConst c, AdjArgs x, int it) {
  const TanArgs &a = x.t;
  const int b = blockIdx.y, N = c.N, tend = c.tdip + c.nd;
  if (it > 1 && !x.state[b].x) return;
  const int i = blockIdx.x * (TAN_BLOCK / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (i >= c.nd * N) return;
  const int s = c.tdip * N + i, iw = s % N, ti = s / N;
  const AdjCfg g(c, a, b);
  const TanWs W(a.ws + (size_t)b * a.ws_stride, c);
  const Dual *src = it & 1 ? W.dip : W.old;
  Dual *dst = it & 1 ? W.old : W.dip;
  Dual e[3] = {0.0, 0.0, 0.0};
  for (int k = lane; k < c.nk; k += 64) {
    const double4 kv = a.kv[k];
    Dual ck, sk;
    g.ph.at(s, a.khkl[k], kv, ck, sk);
    const Dual t = kv.w * (ck * W.Sm[2 * k + 1] - sk * W.Sm[2 * k]);
    e[0] -= t * kv.x;
    e[1] -= t * kv.y;
    e[2] -= t * kv.z;
  }
  for (int jw = lane; jw < N; jw += 64) {
    const bool same = jw == iw;
    double R[3];
    if (!same && !g.within(c, iw, jw, R)) continue;
    for (int tj = c.tdip; tj < tend; ++tj) {
      if (same && tj == ti) continue;
      const int sj = tj * N + jw;
      Dual r[3], o[3];
      g.vec(c, s, sj, r);
      const Dual d2 = r[0] * r[0] + r[1] * r[1] + r[2] * r[2];
      double u1, u2, u3;
      smear3(c, d2.v, c.apolDD[ti][tj], u1, u2, u3);
      Dual t1 = u1, t2 = u2;
      chain_d(t1, 1, u2, d2.d);
      chain_d(t2, 2, u3, d2.d);
      dd3d(r, t1, t2, src + 3 * (sj - c.tdip * N), o);
      for (int k = 0; k < 3; ++k) e[k] += o[k];
    }
  }
  for (int k = 0; k < 3; ++k) e[k] = group_sum(e[k], 64);
  if (lane != 0) return;
  const double om = c.sor, pol = c.polar[ti];
  double d2 = 0.0;
  for (int k = 0; k < 3; ++k) {
    const Dual mr = src[3 * i + k], ek = e[k] + W.Efq[3 * s + k] + c.fac_dd * mr;
    const Dual nr = (1.0 - om) * mr + (om * pol) * ek;
    const double df = nr.v - (it == 1 ? 0.0 : mr.v);
    d2 += df * df;
    dst[3 * i + k] = nr;
  }
  W.Efd[i].v = d2;
}

// The convergence test of iteration `it`, a workgroup per configuration.  One
// that ends after an odd count exchanges dip and old.
__global__ __launch_bounds__(TAN_BLOCK) void k_adj_test(SysConst c, AdjArgs x, int it) {
  __shared__ double red[1][TAN_BLOCK / 64], sum[1];
  const TanArgs &a = x.t;
  const int b = blockIdx.x, M = c.nd * c.N;
  if (it > 1 && !x.state[b].x) return;
  const TanWs W(a.ws + (size_t)b * a.ws_stride, c);
  double d2[1] = {0.0};
  for (int i = threadIdx.x; i < M; i += TAN_BLOCK) d2[0] += W.Efd[i].v;
  block_sums<1>(d2, red, sum);
  __syncthreads();
  const bool last = c.stath * sqrt(sum[0]) < c.peps || it >= c.maxiter;
  if (threadIdx.x == 0) x.state[b] = make_int2(last ? 0 : 1, it);
  if (!last || !(it & 1)) return;
  for (int e = threadIdx.x; e < 3 * M; e += TAN_BLOCK) {
    const Dual t = W.dip[e];
    W.dip[e] = W.old[e];
    W.old[e] = t;
  }
}

// The dipoles' potential at the charged sites (into dR) and d U / d (aCCaCD,
// aDD, polfacO/H/M) at fixed dipoles, through the Thole factors
// a = a0 polfac_i^(-1/2) polfac_j^(-1/2) of each ordered site pair.  The energy
// is stationary in the converged dipoles, so its derivative is the explicit
// one: 1/2 qi qj dts0/da (Uelec), -qj (di . r) dts1/da (-mu . Efq) and
// -1/2 di . dT/da . dj (-1/2 mu T mu); only the Thole terms (r < 5 A,
// smear.f90:23,57) depend on a.
__global__ __launch_bounds__(TAN_BLOCK) void k_adj_pair_d(SysConst c, AdjArgs x) {
  __shared__ double red[ADJ_NA][TAN_BLOCK / 64];
  const TanArgs &a = x.t;
  const int b = blockIdx.y, N = c.N, ns = 4 * N, tend = c.tdip + c.nd;
  const AdjCfg g(c, a, b);
  const TanWs W(a.ws + (size_t)b * a.ws_stride, c);
  const int s0 = blockIdx.x * ADJ_SPB + threadIdx.x / ADJ_G, lane = threadIdx.x % ADJ_G;
  const bool valid = s0 < ns;
  const int s = valid ? s0 : 0, iw = s % N, ti = s / N;
  const bool chg = ti > 0, adip = ti >= c.tdip && ti < tend;
  Dual accCC = 0.0, accDD = 0.0, accPF[3] = {0.0, 0.0, 0.0}, pv = 0.0;
  auto ptype = [](int t) { return t == 0 ? 0 : t == 3 ? 2 : 1; };
  auto thole_acc = [&](Dual w, bool ddt, int tj) {
    const double pi = x.pf[ti], pj = x.pf[tj];
    if (ddt) accDD += w * (pi * pj);
    else accCC += w * (pi * pj);
    const Dual wa = w * a.theta[ddt ? TP_ADD : TP_ACC];
    const Dual wi = wa * (pj * x.dpf[ti]), wj = wa * (pi * x.dpf[tj]);
    // constant indices: the accumulators stay in registers
    for (int q = 0; q < 3; ++q) {
      if (ptype(ti) == q) accPF[q] += wi;
      if (ptype(tj) == q) accPF[q] += wj;
    }
  };
  const Dual qi = W.q[s];
  Dual di[3] = {0.0, 0.0, 0.0};
  if (adip)
    for (int k = 0; k < 3; ++k) di[k] = W.dip[3 * (s - c.tdip * N) + k];
  for (int jw = lane; valid && (chg || adip) && jw < N; jw += ADJ_G) {
    const bool same = jw == iw;
    double Rij[3];
    if (!same && !g.within(c, iw, jw, Rij)) continue;
    for (int tj = 0; tj < 4; ++tj) {
      if (same && tj == ti) continue;
      const bool bdip = tj >= c.tdip && tj < tend, bchg = tj > 0;
      if (!bdip && !bchg) continue;
      const int sj = tj * N + jw;
      Dual r[3];
      g.vec(c, s, sj, r);
      const Dual d2 = r[0] * r[0] + r[1] * r[1] + r[2] * r[2];
      const Dual qj = W.q[sj];
      Dual dj[3] = {0.0, 0.0, 0.0};
      if (bdip)
        for (int k = 0; k < 3; ++k) dj[k] = W.dip[3 * (sj - c.tdip * N) + k];
      if (bdip && chg) {
        double qsq = 0.0, t1, t2;
        for (int k = 0; k < 3; ++k) {
          const double qd = qj.v * di[k].v - qi.v * dj[k].v;
          qsq += qd * qd;
        }
        if (same || qsq > 1e-9) {
          if (same) self2(c, d2.v, t1, t2);
          else smear2(c, d2.v, c.apolCC[ti][tj], t1, t2);
          Dual ts1 = t1;
          chain_d(ts1, 1, t2, d2.d);
          pv += ts1 * (dj[0] * r[0] + dj[1] * r[1] + dj[2] * r[2]);
        }
      }
      if (!(d2.v < 25.0)) continue;
      const bool cc = !same && qi.v != 0.0 && qj.v != 0.0, cd = !same && adip && qj.v != 0.0;
      const double av = c.apolCC[ti][tj], rav = c.raCC[ti][tj];
      Dual t0, t1, u1, u2, u3;
      if ((cc || cd) && av > 0.0) {
        // duals along a; their position derivatives by the chain
        smear3<true, Dual>(c, Dual(d2.v), Dual(av, 1.0), u1, u2, u3);
        Dual w = 0.0;
        if (cc) {
          smear01<true, Dual>(c, Dual(d2.v), Dual(av, 1.0), Dual(rav, rav / (3.0 * av)), t0, t1);
          Dual da0 = t0.d;
          chain_d(da0, 0, u1.d, d2.d);
          w += 0.5 * qi * qj * da0;
        }
        if (cd) {
          Dual da1 = u1.d;
          chain_d(da1, 1, u2.d, d2.d);
          w -= qj * (di[0] * r[0] + di[1] * r[1] + di[2] * r[2]) * da1;
        }
        thole_acc(w, false, tj);
      }
      if (adip && bdip) {
        smear3<true, Dual>(c, Dual(d2.v), Dual(c.apolDD[ti][tj], 1.0), u1, u2, u3);
        Dual da1 = u1.d, da2 = u2.d;
        chain_d(da1, 1, u2.d, d2.d);
        chain_d(da2, 2, u3.d, d2.d);
        const Dual dir_ = di[0] * r[0] + di[1] * r[1] + di[2] * r[2];
        const Dual djr = dj[0] * r[0] + dj[1] * r[1] + dj[2] * r[2];
        const Dual dd = di[0] * dj[0] + di[1] * dj[1] + di[2] * dj[2];
        thole_acc(-0.5 * (3.0 * da2 * dir_ * djr - da1 * dd), true, tj);
      }
    }
  }
  pv = group_sum(pv, ADJ_G);
  if (valid && lane == 0) W.dR[s] = pv;
  double v[ADJ_NA] = {accCC.v, accCC.d, accDD.v, accDD.d, accPF[0].v, accPF[0].d,
                      accPF[1].v, accPF[1].d, accPF[2].v, accPF[2].d};
  block_sums<ADJ_NA>(v, red, x.pa + ((size_t)b * gridDim.x + blockIdx.x) * ADJ_NA);
}

// The adjoint's outputs for configuration b: per parameter j of the 16 TTM
// parameters and the 84 DMS coefficients, adj[b][j] = (dE/dtheta_j,
// gw . d(dE/dr)/dtheta_j), and the energy.  Beside the Thole and vdW partials
// of the pair kernels: the polarisabilities (-1/2 |mu|^2 / alpha^2 per dipole
// site, the alpha^-1 term of the stationary induction energy) in workgroup 0,
// and the charge parameters (sum of phi dq/dtheta over the charged sites, phi
// the potential of charges and dipoles, which is dE/dq) in the others, eight
// lanes per parameter over the molecules.  (gammaM, the last of
// TTM_ADJ_NPARAM, moves the M sites: its slot is filled by the host from a
// tangent sweep.)
constexpr int ADJ_PPB = TAN_BLOCK / 8;  // charge parameters per workgroup
__global__ __launch_bounds__(TAN_BLOCK) void k_adj_out(SysConst c, AdjArgs x) {
  __shared__ double red[TAN_BLOCK];
  const TanArgs &a = x.t;
  const int b = blockIdx.y, N = c.N, tid = threadIdx.x;
  const TanWs W(a.ws + (size_t)b * a.ws_stride, c);
  double *out = a.adj + (size_t)b * TTM_ADJ_NPARAM * 2;
  if (blockIdx.x == 0) {
    const int nds = c.nd * N, nb = adj_pair_blocks(c);
    Dual pol[3] = {0.0, 0.0, 0.0};  // by site type (O, H, M)
    double ue = 0.0, ui = 0.0;
    for (int i = tid; i < nds; i += TAN_BLOCK) {
      const int t = c.tdip + i / N, pt = t == 0 ? 0 : t == 3 ? 2 : 1;
      const double al = c.polar[t];
      const Dual *mu = W.dip + 3 * i, *e = W.Efq + 3 * (c.tdip * N + i);
      const Dual m2 = mu[0] * mu[0] + mu[1] * mu[1] + mu[2] * mu[2];
      for (int q = 0; q < 3; ++q)
        if (q == pt && al > 0.0) pol[q] -= 0.5 * m2 / (al * al);
      for (int k = 0; k < 3; ++k) ui += mu[k].v * e[k].v;
    }
    for (int s = N + tid; s < 4 * N; s += TAN_BLOCK) ue += W.q[s].v * W.phi[s].v;
    Dual sPol[3];
    for (int i = 0; i < 3; ++i)
      sPol[i] = Dual(block_sum(pol[i].v, red), block_sum(pol[i].d, red));
    ue = block_sum(ue, red);
    ui = block_sum(ui, red);
    if (tid != 0) return;
    double sv[ADJ_NV] = {0}, sa[ADJ_NA] = {0};
    for (int q = 0; q < nb; ++q) {
      for (int i = 0; i < ADJ_NV; ++i) sv[i] += x.pv[((size_t)b * nb + q) * ADJ_NV + i];
      for (int i = 0; i < ADJ_NA; ++i) sa[i] += x.pa[((size_t)b * nb + q) * ADJ_NA + i];
    }
    auto put = [&](int j, double v, double d) {
      out[2 * j] = v;
      out[2 * j + 1] = d;
    };
    for (int i = 0; i < 5; ++i)
      put(TP_VDWA + i, sv[1 + i] + (i < 3 ? a.lrc_coef[i] : 0.0), sv[6 + i]);
    for (int i = 0; i < 3; ++i) put(TP_POLARO + i, sPol[i].v, sPol[i].d);
    for (int i = 0; i < 3; ++i) put(TP_POLFACO + i, sa[4 + 2 * i], sa[5 + 2 * i]);
    put(TP_ADD, sa[2], sa[3]);
    put(TP_ACC, sa[0], sa[1]);
    put(TTM_ADJ_NPARAM - 1, 0.0, 0.0);
    double *o = a.out + (size_t)b * 4;
    o[0] = W.umon->v + sv[0] + 0.5 * ue - 0.5 * ui + c.Uvdw_lrc;
    o[1] = o[2] = o[3] = 0.0;
    return;
  }
  // dms_param1..3, then the 84 coefficients coefD
  const int j = (blockIdx.x - 1) * ADJ_PPB + tid / 8;
  const double gM = c.gammaM, tq = 0.5 * gM / (1.0 - gM);
  Dual acc = 0.0;
  for (int w = tid % 8; j < 3 + DMS_NCOEF && w < N; w += 8) {
    const double *rr = a.RR + ((size_t)b * 3 * N + 3 * w) * 3;
    const double *gw = a.gw + ((size_t)b * 3 * N + 3 * w) * 3;
    double r[3][3], dq3[3], dgq[3][3][3];
    for (int at = 0; at < 3; ++at)
      for (int k = 0; k < 3; ++k) r[at][k] = rr[3 * at + k];
    if (j < 3) dms_tangent(c, r, j, dq3, dgq);
    else dms_coef_tangent(c, r, j - 3, dq3, dgq);
    // dq3 in (O, H1, H2), dgq[disp][charge] in (H1, H2, O); along gw
    const int atom[3] = {1, 2, 0};
    Dual dqd[3];
    for (int i = 0; i < 3; ++i) {
      const int ch = i == 0 ? 2 : i - 1;
      double v = 0.0;
      for (int d = 0; d < 3; ++d)
        for (int k = 0; k < 3; ++k) v += dgq[d][ch][k] * gw[3 * atom[d] + k];
      dqd[i] = Dual(dq3[i] * CHARGECON, v * CHARGECON);
    }
    const Dual sH = dqd[1] + dqd[2];
    const Dual p1 = W.phi[N + w] + W.dR[N + w], p2 = W.phi[2 * N + w] + W.dR[2 * N + w],
               pm = W.phi[3 * N + w] + W.dR[3 * N + w];
    acc += p1 * (dqd[1] + tq * sH) + p2 * (dqd[2] + tq * sH) + pm * dqd[0] * (1.0 / (1.0 - gM));
  }
  acc = group_sum(acc, 8);
  if (tid % 8 == 0 && j < 3 + DMS_NCOEF) {
    out[2 * (TP_DMS1 + j)] = acc.v;
    out[2 * (TP_DMS1 + j) + 1] = acc.d;
  }
}

// The dense solve takes systems of up to ADJ_DENSE_MAX_D dipole components
// (16 D^2 bytes of matrix each, in slices of as many configurations as
// PIMD_ADJ_MAT_MB, default 1024, takes, at least one); larger ones, whose
// matrix one workgroup would stream every iteration, go pass by pass, in
// memory that grows with the sites.  Whole adjoint, dense / passes, ms
// (components x configurations): 96 x 64 0.51 / 1.05, 192 x 16 0.47 / 0.69,
// 384 x 1 0.67 / 0.80, 384 x 64 2.23 / 3.03; 576 x 1 (TTM2.1-F) 0.91 / 0.76,
// 576 x 16 1.40 / 1.15, 768 x 1 1.85 / 1.22, 768 x 32 5.10 / 3.56, 2040 x 8
// 21.0 / 4.0.  1000 TTM3-F waters 3.0 (one workgroup per configuration: 215).
// PIMD_ADJ_DENSE=0: pass by pass at every size.
constexpr size_t ADJ_DENSE_MAX_D = 480;
AdjPlan adjoint_plan(const SysConst &c) {
  AdjPlan p;
  const size_t D = 3 * (size_t)c.nd * c.N, mat = D * D;
  auto env = [](const char *name) {
    const char *e = std::getenv(name);
    return e && *e ? std::strtol(e, nullptr, 10) : -1;
  };
  p.dense = D <= ADJ_DENSE_MAX_D && env("PIMD_ADJ_DENSE") != 0;
  if (p.dense) {
    const long mb = env("PIMD_ADJ_MAT_MB");
    const size_t bytes = (size_t)(mb > 0 ? mb : 1024) << 20;
    p.slice = (int)std::min((size_t)c.P, std::max<size_t>(bytes / (sizeof(Dual) * mat), 1));
  }
  // 16-byte aligned: the dual workspace follows
  p.solve = p.dense ? 2 * p.slice * mat : ((size_t)c.P + 1) & ~(size_t)1;
  p.extra = p.solve + (((size_t)c.P * adj_pair_blocks(c) * (ADJ_NV + ADJ_NA) + 1) & ~(size_t)1);
  return p;
}

static void launch_adjoint(const SysConst &c, const TanLaunch &L, const TanArgs &a, hipStream_t s) {
  AdjArgs x;
  x.t = a;
  x.mat = (Dual *)L.extra;
  x.state = (int2 *)L.extra;
  x.pv = L.extra + L.plan.solve;
  x.pa = x.pv + (size_t)c.P * adj_pair_blocks(c) * ADJ_NV;
  x.cols = L.cols;
  x.colk = L.colk;
  x.b0 = 0;
  for (int i = 0; i < 4; ++i) {
    // polfac^(-1/2) as (polfac^(1/6))^-3 (potential.f90:157-160)
    const double p = L.theta[TP_POLFACO + (i == 0 ? 0 : i == 3 ? 2 : 1)], f6 = std::pow(p, 1.0 / 6.0);
    x.pf[i] = 1.0 / (f6 * f6 * f6);
    x.dpf[i] = -0.5 * x.pf[i] / p;
  }
  const int P = c.P, ns = 4 * c.N, M = c.nd * c.N, D = 3 * M, nt = (M + 7) / 8, wpb = TAN_BLOCK / 64;
  const dim3 B(TAN_BLOCK), gp(adj_pair_blocks(c), P), gs((c.nk + TAN_BLOCK / 4 - 1) / (TAN_BLOCK / 4), P),
      gf((ns + wpb - 1) / wpb, P), gm((M + wpb - 1) / wpb, P);
  hipLaunchKernelGGL(k_tangent_monomer<TAN_ADJOINT>, dim3(P, 1), B, 0, s, c, a);
  hipLaunchKernelGGL(k_adj_pair_q, gp, B, 0, s, c, x);
  hipLaunchKernelGGL(k_adj_sfac<false>, gs, B, 0, s, c, x, 0);
  hipLaunchKernelGGL(k_adj_field<false>, gf, B, 0, s, c, x);
  if (L.plan.dense) {
    for (int b0 = 0; b0 < P; b0 += L.plan.slice) {
      const int n = std::min(L.plan.slice, P - b0);
      x.b0 = b0;
      hipLaunchKernelGGL(k_adj_build, dim3(nt * (nt + 1) / 2, n), dim3(64 * ADJ_BW), 0, s, c, x);
      hipLaunchKernelGGL(k_adj_solve, dim3(n), dim3(ADJ_SOLVE), 2 * sizeof(Dual) * D, s, c, x);
    }
  } else {
    for (int it = 1; it <= c.maxiter; ++it) {
      hipLaunchKernelGGL(k_adj_sfac<true>, gs, B, 0, s, c, x, it);
      hipLaunchKernelGGL(k_adj_step, gm, B, 0, s, c, x, it);
      hipLaunchKernelGGL(k_adj_test, dim3(P), B, 0, s, c, x, it);
    }
  }
  hipLaunchKernelGGL(k_adj_sfac<true>, gs, B, 0, s, c, x, 0);
  hipLaunchKernelGGL(k_adj_pair_d, gp, B, 0, s, c, x);
  hipLaunchKernelGGL(k_adj_field<true>, gf, B, 0, s, c, x);
  hipLaunchKernelGGL(k_adj_out, dim3(1 + (3 + DMS_NCOEF + ADJ_PPB - 1) / ADJ_PPB, P), B, 0, s, c, x);
}

void launch_ttm_tangent(const SysConst &c, const TanLaunch &L, hipStream_t s) {
  const size_t ds_off = 3 * 4 * (size_t)c.N + tangent_tab_doubles(c);
  const int mode = L.adjoint ? 2 : L.gamma_m ? 1 : 0;
  hipLaunchKernelGGL(k_tangent_prep, dim3(c.P), dim3(TAN_BLOCK), 0, s, c, L.RR, L.cfg,
                     tangent_cfg_doubles(c), ds_off, mode, L.gw);
  TanArgs a;
  a.RR = L.RR;
  a.pes = L.pes;
  a.kv = L.kv;
  a.khkl = L.khkl;
  a.cfg = L.cfg;
  a.cfg_stride = tangent_cfg_doubles(c);
  a.ws = (Dual *)L.ws;
  a.ws_stride = tangent_ws_duals(c);
  a.ew = L.ew;
  a.gw = L.gw;
  a.out = L.out;
  a.dG = L.dG;
  for (int i = 0; i < TTM_NPARAM; ++i) a.theta[i] = L.theta[i];
  for (int i = 0; i < 3; ++i) a.lrc_coef[i] = L.lrc_coef[i];
  a.dms_coef = L.dms_coef;
  a.gamma_m = L.gamma_m;
  a.ds_off = ds_off;
  a.adj = L.adj;
  if (mode == TAN_ADJOINT) {
    launch_adjoint(c, L, a, s);
  } else if (mode == TAN_GAMMA_M) {
    hipLaunchKernelGGL(k_tangent_monomer<TAN_GAMMA_M>, dim3(c.P, 1), dim3(TAN_BLOCK), 0, s, c, a);
    hipLaunchKernelGGL(k_ttm_tangent<TAN_GAMMA_M>, dim3(c.P, 1), dim3(TAN_BLOCK), 0, s, c, a);
  } else {
    hipLaunchKernelGGL(k_tangent_monomer<TAN_PARAMS>, dim3(c.P, L.ndir), dim3(TAN_BLOCK), 0, s, c, a);
    hipLaunchKernelGGL(k_ttm_tangent<TAN_PARAMS>, dim3(c.P, L.ndir), dim3(TAN_BLOCK), 0, s, c, a);
  }
}

}  // namespace pimd
