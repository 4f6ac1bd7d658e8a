// Device functions shared by the kernel sources: wave reductions, the
// entropy -> primitive conversion, the subgrid scale models and the
// characteristic-matching-layer source.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace vcp {
namespace {

constexpr double kGam = 1.4;
constexpr double kGm1 = 0.4;
constexpr double kPrLam = 0.72;
constexpr double kPrTurb = 0.90;       // VCP3D_CurviLinear.hpp:176
constexpr double kLamOverMu = -2.0 / 3.0;
constexpr double kInvGm1 = 1.0 / kGm1;

// ------------------------------------------------------------ utilities
constexpr int cmax(int x, int y) { return x > y ? x : y; }
constexpr int cmin(int x, int y) { return x < y ? x : y; }

__device__ inline double wave_sum(double v)
{
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}
__device__ inline double wave_max(double v)
{
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
  return v;
}

// Wave64 reduction through DPP row shifts and row broadcasts (no LDS):
// sum, or max of non-negative values; lanes without a source contribute 0.
// The result (lane 63) is returned to every lane.
template <int CTRL, int ROW_MASK>
__device__ inline double dpp_f64(double v)
{
  const int lo = __double2loint(v), hi = __double2hiint(v);
  const int rlo = __builtin_amdgcn_update_dpp(0, lo, CTRL, ROW_MASK, 0xf, false);
  const int rhi = __builtin_amdgcn_update_dpp(0, hi, CTRL, ROW_MASK, 0xf, false);
  return __hiloint2double(rhi, rlo);
}
// Row shift with every row enabled: lanes shifted in from outside the row
// read 0 (bound_ctrl), so no zeroed destination is needed.
template <int CTRL>
__device__ inline double dpp_shr_f64(double v)
{
  const int lo = __double2loint(v), hi = __double2hiint(v);
  const int rlo = __builtin_amdgcn_mov_dpp(lo, CTRL, 0xf, 0xf, true);
  const int rhi = __builtin_amdgcn_mov_dpp(hi, CTRL, 0xf, 0xf, true);
  return __hiloint2double(rhi, rlo);
}
template <bool MAX>
__device__ inline double wave_reduce_dpp(double v)
{
  auto op = [](double x, double y) { return MAX ? fmax(x, y) : x + y; };
  v = op(v, dpp_shr_f64<0x111>(v));    // row_shr:1
  v = op(v, dpp_shr_f64<0x112>(v));    // row_shr:2
  v = op(v, dpp_shr_f64<0x114>(v));    // row_shr:4
  v = op(v, dpp_shr_f64<0x118>(v));    // row_shr:8   -> lane 15 of each row: row total
  v = op(v, dpp_f64<0x142, 0xa>(v));   // row_bcast:15 into rows 1, 3
  v = op(v, dpp_f64<0x143, 0xc>(v));   // row_bcast:31 into rows 2, 3 -> lane 63: total
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), 63);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), 63);
  return __hiloint2double(hi, lo);
}

// The same over the G = 16 or 32 neighbouring lanes that share a wave, or over
// the wave.
template <int CTRL>
__device__ __forceinline__ double dpp_all_f64(double v)
{
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

template <int G, bool MAX>
__device__ __forceinline__ double lanes_reduce(double v)
{
  if constexpr (G >= 64) return wave_reduce_dpp<MAX>(v);
  auto op = [](double x, double y) { return MAX ? fmax(x, y) : x + y; };
  v = op(v, dpp_all_f64<0xB1>(v));     // quad_perm 1,0,3,2
  v = op(v, dpp_all_f64<0x4E>(v));     // quad_perm 2,3,0,1
  v = op(v, dpp_all_f64<0x141>(v));    // row_half_mirror
  v = op(v, dpp_all_f64<0x140>(v));    // row_mirror
  if constexpr (G == 32) v = op(v, __shfl_xor(v, 16, 64));
  return v;
}

// Orders the LDS accesses of a group of G threads: a workgroup barrier, or
// nothing but program order within a wave.
template <int G>
__device__ __forceinline__ void group_sync()
{
  if constexpr (G > 64) {
    // the wait is written out: at the head of a loop whose body ends with LDS
    // stores, the compiler (ROCm 7.2, gfx950) leaves it out of the barrier
    // on the way back
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __syncthreads();
  } else {
    // one wave: its LDS operations complete in order, so only the compiler
    // has to keep them in program order
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// t^(-1/(gamma-1)) = t^(-5/2) for gamma = 1.4, as 1 / (t^2 sqrt(t)).
__device__ inline double pow_m2p5(double t) { return 1.0 / (t * t * sqrt(t)); }

__device__ inline void ent2prim(const double V[5], double &rho, double &u, double &v, double &w,
                                double &p, double &eKin)
{
  const double V4Inv = 1.0 / V[4];
  u = -V4Inv * V[1]; v = -V4Inv * V[2]; w = -V4Inv * V[3];
  eKin = 0.5 * (u * u + v * v + w * w);
  const double s = kGam - kGm1 * (V[0] - V[4] * eKin);
  rho = pow_m2p5(-V[4] * exp(s));
  p = -rho * V4Inv;
}


// 1 / x and 1 / sqrt(x) to about a unit in the last place: the hardware
// approximation with its error removed by Newton steps, without the scaling and
// exception steps of the IEEE division and square root (fewer than half of their
// instructions). recip holds for x of either sign whose reciprocal is a normal
// number; 0 and infinity give not-a-number, where the division gives infinity
// and 0. rsqrt_exact holds for normal x > 0; 0, negative and infinite x give
// not-a-number.
__device__ __forceinline__ double recip(double x)
{
  double y = __builtin_amdgcn_rcp(x);
  y = fma(fma(-x, y, 1.0), y, y);
  return fma(fma(-x, y, 1.0), y, y);
}
__device__ __forceinline__ double rsqrt_exact(double x)
{
  double y = __builtin_amdgcn_rsq(x);
  double e = fma(-x * y, y, 1.0);
  y = fma(fma(0.375, e, 0.5) * e, y, y);
  e = fma(-x * y, y, 1.0);
  return fma(0.5 * e, y, y);
}

// Primitive state of the entropy variables from one reciprocal square root:
// with x = -V4 = rho / p and y = x^(-1/2), p / rho = y^2,
// rho = (x e^s)^(-5/2) = y^5 e^(-5/2 s) for gamma = 1.4, sqrt(rho / p) = x y
// and sqrt(rho p) = rho y.
struct EntState {
  double rho, u, v, w, p, ek, r, y;   // r = p / rho = -1 / V4
};
__device__ __forceinline__ EntState ent_state(const double V[5])
{
  EntState q;
  const double x = -V[4];
  q.y = rsqrt_exact(x);
  q.r = q.y * q.y;
  q.r = fma(fma(-x, q.r, 1.0), q.r, q.r);
  q.u = q.r * V[1]; q.v = q.r * V[2]; q.w = q.r * V[3];
  q.ek = 0.5 * (q.u * q.u + q.v * q.v + q.w * q.w);
  const double s = kGam - kGm1 * (V[0] + x * q.ek);
  q.rho = q.r * q.r * q.y * exp(-2.5 * s);
  q.p = q.rho * q.r;
  return q;
}

// Eddy viscosity mu_SGS = rho nu_t of the subgrid scale model at one point,
// from the velocity gradient G[i][j] = du_i/dx_j and the LES length scale len.
// WALE (CWALEModel::EddyViscosity, SGSModel.cpp:34-113): with S the
// symmetric part of G and Sd the traceless symmetric part of G^2,
// nu_t = (0.325 len)^2 |Sd|^3 / max(|S|^5 + |Sd|^(5/2), 1e-30), |X|^2 = X_ij X_ij.
// Vreman (CVremanModel::EddyViscosity, :128-210): alpha = G with its trace
// taken off the diagonal, beta = len^2 alpha alpha^T, B the sum of the
// principal 2 x 2 minors of beta (clipped at 0),
// nu_t = 0.07 sqrt(B / max(|alpha|^2, 1e-30)).
__device__ inline double eddy_viscosity(int model, double len, double rho, const double G[3][3])
{
  constexpr double third = 1.0 / 3.0, eps = 1e-30;
  if (model == kSgsWale) {
    double G2[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) G2[i][j] = G[i][0] * G[0][j] + G[i][1] * G[1][j] + G[i][2] * G[2][j];
    const double tr = third * (G2[0][0] + G2[1][1] + G2[2][2]);
    double s2 = 0.0, sd2 = 0.0;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const double d = G2[i][i] - tr;
      s2 += G[i][i] * G[i][i];
      sd2 += d * d;
#pragma unroll
      for (int j = i + 1; j < 3; ++j) {
        const double sij = 0.5 * (G[i][j] + G[j][i]), dij = 0.5 * (G2[i][j] + G2[j][i]);
        s2 += 2.0 * sij * sij;
        sd2 += 2.0 * dij * dij;
      }
    }
    const double sd32 = sd2 * sqrt(sd2);
    const double den = s2 * s2 * sqrt(s2) + sqrt(sd32 * sd2);
    const double l = 0.325 * len;
    return rho * (l * l) * sd32 / fmax(den, eps);
  }
  if (model == kSgsVreman) {
    const double tr = third * (G[0][0] + G[1][1] + G[2][2]);
    double al[3][3], a2 = 0.0;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        al[i][j] = i == j ? G[i][j] - tr : G[i][j];
        a2 += al[i][j] * al[i][j];
      }
    const double l2 = len * len;
    double be[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = i; j < 3; ++j) be[i][j] = l2 * (al[i][0] * al[j][0] + al[i][1] * al[j][1] + al[i][2] * al[j][2]);
    const double B = be[0][0] * be[1][1] - be[0][1] * be[0][1] + be[0][0] * be[2][2] - be[0][2] * be[0][2]
                   + be[1][1] * be[2][2] - be[1][2] * be[1][2];
    return rho * 0.07 * sqrt(fmax(B, 0.0) / fmax(a2, eps));
  }
  return 0.0;
}

// Characteristic-matching-layer source at one point (ElementClass.cpp:
// 3887-4117): wave amplitudes of the Cartesian primitive gradients per
// direction with the outgoing eigenvalues of the layer orientation removed,
// P = S L mapped to the conservative variables. V: entropy variables,
// gx/gy/gz their Cartesian gradients, wgt[d] = -J w sigma_d scale_d,
// nsg[d] the layer orientation. Accumulates into out.
__device__ __forceinline__ void cml_source(const double V[5], const double gx[5], const double gy[5],
                                           const double gz[5], const double wgt[3], const double nsg[3],
                                           double out[5])
{
  const double V4Inv = 1.0 / V[4];
  const double u = -V4Inv * V[1], v = -V4Inv * V[2], w = -V4Inv * V[3];
  const double ek = 0.5 * (u * u + v * v + w * w);
  const double s = kGam - kGm1 * (V[0] - V[4] * ek);
  const double rho = pow_m2p5(-V[4] * exp(s));
  const double p = -rho * V4Inv, rE = p / kGm1 + rho * ek;
  const double H = rE / rho - V4Inv, a2 = -kGam * V4Inv, a = sqrt(a2);
  const double rhoa = rho * a, ovra = 1.0 / rhoa, ova2 = 1.0 / a2, rova = rho / a;
  const double rhou = rho * u, rhov = rho * v, rhow = rho * w;
  const double vel[3] = {u, v, w};
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double *G = d == 0 ? gx : d == 1 ? gy : gz;
    double dq[5];
    dq[0] = rho * G[0] + rhou * G[1] + rhov * G[2] + rhow * G[3] + rE * G[4];
    dq[1] = -V4Inv * G[1] + (-V4Inv * u) * G[4];
    dq[2] = -V4Inv * G[2] + (-V4Inv * v) * G[4];
    dq[3] = -V4Inv * G[3] + (-V4Inv * w) * G[4];
    dq[4] = p * G[0] + (p * u) * G[1] + (p * v) * G[2] + (p * w) * G[3] + (p * H) * G[4];
    double l1 = vel[d] - a, l2 = vel[d], l3 = vel[d] + a;
    if (nsg[d] * l1 > 0.0) l1 = 0.0;
    if (nsg[d] * l2 > 0.0) l2 = 0.0;
    if (nsg[d] * l3 > 0.0) l3 = 0.0;
    const double dun = dq[1 + d];
    const double La = 0.5 * l1 * (ovra * dq[4] - dun);
    const double Lb = 0.5 * l3 * (ovra * dq[4] + dun);
    const double Le = l2 * (dq[0] - ova2 * dq[4]);
    double P[5];
    P[0] = rova * (Lb + La) + Le;
    P[4] = rhoa * (Lb + La);
#pragma unroll
    for (int t = 0; t < 3; ++t) P[1 + t] = (t == d) ? (Lb - La) : l2 * dq[1 + t];
    const double wd = wgt[d];
    out[0] += wd * P[0];
    out[1] += wd * (u * P[0] + rho * P[1]);
    out[2] += wd * (v * P[0] + rho * P[2]);
    out[3] += wd * (w * P[0] + rho * P[3]);
    out[4] += wd * (ek * P[0] + rhou * P[1] + rhov * P[2] + rhow * P[3] + P[4] / kGm1);
  }
}

// Eddy viscosity at a face point (FluxesFace.cpp:1409-1459, :1481-1494): the
// model on the density of the averaged entropy variables and the velocity
// gradients of the averaged state and the averaged Cartesian gradients
// gx, gy, gz, with the face's LES length scale. Evaluated before the fluxes,
// so that its temporaries are dead where those peak in registers.
__device__ __forceinline__ double face_eddy(int sgs, double lenLES, const double VL[5], const double VR[5],
                                            const double gx[5], const double gy[5], const double gz[5])
{
  const double V0a = 0.5 * (VL[0] + VR[0]), V4a = 0.5 * (VL[4] + VR[4]);
  const double V4Inv = 2.0 / (VL[4] + VR[4]);
  const double u = -V4Inv * 0.5 * (VL[1] + VR[1]), v = -V4Inv * 0.5 * (VL[2] + VR[2]),
               w = -V4Inv * 0.5 * (VL[3] + VR[3]);
  const double ek = 0.5 * (u * u + v * v + w * w);
  const double rhoA = pow_m2p5(-V4a * exp(kGam - kGm1 * (V0a - V4a * ek)));
  const double vel[3] = {u, v, w};
  double G[3][3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    G[i][0] = -V4Inv * (gx[1 + i] + vel[i] * gx[4]);
    G[i][1] = -V4Inv * (gy[1 + i] + vel[i] * gy[4]);
    G[i][2] = -V4Inv * (gz[1 + i] + vel[i] * gz[4]);
  }
  return eddy_viscosity(sgs, lenLES, rhoA, G);
}

// Ismail-Roe + viscous + interior-penalty + symmetrising fluxes at one face
// point: VL/VR entropy states (L -> R along nn), gx/gy/gz the averaged
// Cartesian gradients, wA = weight * area factor. fl: normal flux, FX/FY/FZ:
// Cartesian symmetrising fluxes (FluxesFace.cpp:813-975, :1290-1651,
// :1152-1284). BND: the boundary form, where factU (wallPerm, 0 on walls)
// multiplies the convective and dissipation parts of the inviscid flux and a
// prescribed wall heat flux (hf) zeroes the laminar heat-flux factor and adds
// wA * qWall to the energy flux (FluxesFace.cpp:1312-1318, :1586-1593).
// sgs: with a subgrid scale model, its eddy viscosity ev at the point
// (face_eddy) adds to mu in the stresses, the penalty and the symmetrising
// fluxes, with the turbulent Prandtl number in the heat flux
// (FluxesFace.cpp:1537-1554, :1096-1103, :1198-1213).
template <bool BND = false>
__device__ __forceinline__ void point_flux(const double VL[5], const double VR[5], const double gx[5],
                                           const double gy[5], const double gz[5], const double nn[3],
                                           double wA, double tau, double mu, double thetaHalf,
                                           double fl[5], double FX[5], double FY[5], double FZ[5],
                                           double factU = 1.0, bool hf = false, double qWall = 0.0,
                                           double *aux = nullptr, bool sgs = false, double ev = 0.0)
{
  const double factHF = (BND && hf) ? 0.0 : kGam / kPrLam;
  const double factHFT = (BND && hf) ? 0.0 : kGam / kPrTurb;
  // total viscosity, total heat-flux factor and their ratio
  double muT = mu, fhT = mu * factHF, fhR = factHF;
  const double lam = kLamOverMu, lamp1 = lam + 1.0, lamp2 = lam + 2.0;
  {
    const EntState L = ent_state(VL), R = ent_state(VR);
    if (BND && aux) aux[0] = L.p + R.p;   // for the wall forces
    const double dV0 = VR[0] - VL[0], dV1 = VR[1] - VL[1], dV2 = VR[2] - VL[2],
                 dV3 = VR[3] - VL[3], dV4 = VR[4] - VL[4];
    // sqrt(rho / p), sqrt(rho p)
    const double z0L = -VL[4] * L.y, z0R = -VR[4] * R.y;
    const double z4L = L.rho * L.y, z4R = R.rho * R.y;
    const double z0A = 0.5 * (z0L + z0R), z4A = 0.5 * (z4L + z4R);
    const double z1A = 0.5 * (L.u * z0L + R.u * z0R), z2A = 0.5 * (L.v * z0L + R.v * z0R),
                 z3A = 0.5 * (L.w * z0L + R.w * z0R);
    // one reciprocal for both means
    const double inv = recip(z0A * z4A), oz0 = z4A * inv, oz4 = z0A * inv;
    // logarithmic means: F = log(zeta) / (2 f), f = (zeta - 1) / (zeta + 1)
    // = (zL - zR) / (zL + zR), by its series for small f
    constexpr double c3 = 1.0 / 3.0, c5 = 1.0 / 5.0, c7 = 1.0 / 7.0, c9 = 1.0 / 9.0;
    auto log_mean = [](double f, double zL, double zR) {
      const double uu = f * f;
      return (uu < 0.01) ? 1.0 + uu * (c3 + uu * (c5 + uu * (c7 + uu * c9))) : log(zL / zR) / (2.0 * f);
    };
    const double F0 = log_mean(0.5 * (z0L - z0R) * oz0, z0L, z0R);   // z0 mean / log mean
    const double F4 = log_mean(0.5 * (z4L - z4R) * oz4, z4L, z4R);
    const double z4Log = z4A * recip(F4);
    const double rA = z0A * z4Log, p1 = oz0 * z4A, orA = inv * F4;
    const double p2 = 0.5 * ((kGam + 1.0) / kGam * (z4Log * F0 * oz0) + kGm1 / kGam * p1);
    const double uA = oz0 * z1A, vA = oz0 * z2A, wAv = oz0 * z3A;
    const double vn = uA * nn[0] + vA * nn[1] + wAv * nn[2];
    const double kin = 0.5 * (uA * uA + vA * vA + wAv * wAv);
    const double a2 = kGam * p2 * orA, oa = rsqrt_exact(a2), aa = a2 * oa;
    const double H = a2 * kInvGm1 + kin, E = H - p2 * orA;
    double abv1 = rA * (uA * dV1 + vA * dV2 + wAv * dV3);
    double abv2 = abv1 + rA * (dV0 + H * dV4);
    const double dr = abv1 + rA * (dV0 + E * dV4);
    const double dru = uA * abv2 + p2 * dV1, drv = vA * abv2 + p2 * dV2, drw = wAv * abv2 + p2 * dV3;
    const double drE = H * abv1 + rA * E * (dV0 + H * dV4) + p2 * kin * dV4;
    const double fac = 0.5 * (1.0 + 1.0 / 6.0);
    const double lam1 = fabs(vn + aa) * fac, lam2 = fabs(vn - aa) * fac, lam3 = 0.5 * fabs(vn);
    abv1 = 0.5 * (lam1 + lam2); abv2 = 0.5 * (lam1 - lam2);
    const double abv3 = abv1 - lam3;
    const double abv4 = kGm1 * (kin * dr - uA * dru - vA * drv - wAv * drw + drE);
    const double abv5 = nn[0] * dru + nn[1] * drv + nn[2] * drw - vn * dr;
    const double abv6 = abv3 * abv4 * (oa * oa) + abv2 * abv5 * oa;
    const double abv7 = abv2 * abv4 * oa + abv3 * abv5;
    if constexpr (BND) {
      fl[0] = wA * (factU * rA * vn - factU * (lam3 * dr + abv6));
      fl[1] = wA * (factU * rA * vn * uA + p1 * nn[0] - factU * (lam3 * dru + uA * abv6 + nn[0] * abv7));
      fl[2] = wA * (factU * rA * vn * vA + p1 * nn[1] - factU * (lam3 * drv + vA * abv6 + nn[1] * abv7));
      fl[3] = wA * (factU * rA * vn * wAv + p1 * nn[2] - factU * (lam3 * drw + wAv * abv6 + nn[2] * abv7));
      fl[4] = wA * (factU * rA * vn * H - factU * (lam3 * drE + H * abv6 + vn * abv7));
    } else {
      fl[0] = wA * (rA * vn - (lam3 * dr + abv6));
      fl[1] = wA * (rA * vn * uA + p1 * nn[0] - (lam3 * dru + uA * abv6 + nn[0] * abv7));
      fl[2] = wA * (rA * vn * vA + p1 * nn[1] - (lam3 * drv + vA * abv6 + nn[1] * abv7));
      fl[3] = wA * (rA * vn * wAv + p1 * nn[2] - (lam3 * drw + wAv * abv6 + nn[2] * abv7));
      fl[4] = wA * (rA * vn * H - (lam3 * drE + H * abv6 + vn * abv7));
    }
  }
  const double V4Inv = recip(0.5 * (VL[4] + VR[4]));
  const double u = -V4Inv * 0.5 * (VL[1] + VR[1]), vv = -V4Inv * 0.5 * (VL[2] + VR[2]),
               w = -V4Inv * 0.5 * (VL[3] + VR[3]);
  {
    const double dudx = -V4Inv * (gx[1] + u * gx[4]), dvdx = -V4Inv * (gx[2] + vv * gx[4]), dwdx = -V4Inv * (gx[3] + w * gx[4]);
    const double dudy = -V4Inv * (gy[1] + u * gy[4]), dvdy = -V4Inv * (gy[2] + vv * gy[4]), dwdy = -V4Inv * (gy[3] + w * gy[4]);
    const double dudz = -V4Inv * (gz[1] + u * gz[4]), dvdz = -V4Inv * (gz[2] + vv * gz[4]), dwdz = -V4Inv * (gz[3] + w * gz[4]);
    const double fe = V4Inv * V4Inv * kInvGm1;
    const double dedx = fe * gx[4], dedy = fe * gy[4], dedz = fe * gz[4];
    if (sgs) {
      muT = mu + ev;
      fhT = mu * factHF + ev * factHFT;
      fhR = fhT / muT;
    }
    const double nx = wA * nn[0], ny = wA * nn[1], nz = wA * nn[2];
    const double lamDiv = kLamOverMu * (dudx + dvdy + dwdz);
    const double txx = muT * (2.0 * dudx + lamDiv), tyy = muT * (2.0 * dvdy + lamDiv), tzz = muT * (2.0 * dwdz + lamDiv);
    const double txy = muT * (dudy + dvdx), txz = muT * (dudz + dwdx), tyz = muT * (dvdz + dwdy);
    const double qx = -fhT * dedx, qy = -fhT * dedy, qz = -fhT * dedz;
    fl[1] -= txx * nx + txy * ny + txz * nz;
    fl[2] -= txy * nx + tyy * ny + tyz * nz;
    fl[3] -= txz * nx + tyz * ny + tzz * nz;
    fl[4] -= (u * txx + vv * txy + w * txz - qx) * nx + (u * txy + vv * tyy + w * tyz - qy) * ny
           + (u * txz + vv * tyz + w * tzz - qz) * nz;
    if (BND && hf) fl[4] += wA * qWall;
    if (BND && aux) { aux[1] = txx; aux[2] = tyy; aux[3] = tzz; aux[4] = txy; aux[5] = txz; aux[6] = tyz; }
  }
  const double pOvRho = -V4Inv, eInt = pOvRho * kInvGm1;
  const double dV1 = VL[1] - VR[1], dV2 = VL[2] - VR[2], dV3 = VL[3] - VR[3], dV4 = VL[4] - VR[4];
  const double factFlux = pOvRho * wA * muT;
  const double abvE = u * u + vv * vv + w * w + fhR * eInt;
  const double un = u * nn[0] + vv * nn[1] + w * nn[2];
  const double dVn = dV1 * nn[0] + dV2 * nn[1] + dV3 * nn[2];
  const double ttau = tau * factFlux, abvMom = lamp1 * (dVn + un * dV4);
  fl[1] += ttau * (abvMom * nn[0] + dV1 + u * dV4);
  fl[2] += ttau * (abvMom * nn[1] + dV2 + vv * dV4);
  fl[3] += ttau * (abvMom * nn[2] + dV3 + w * dV4);
  fl[4] += ttau * (lamp1 * un * dVn + u * dV1 + vv * dV2 + w * dV3 + (abvE + lamp1 * un * un) * dV4);
  const double sx = thetaHalf * factFlux * nn[0], sy = thetaHalf * factFlux * nn[1], sz = thetaHalf * factFlux * nn[2];
  const double K11_14 = u * lamp2, K11_44 = abvE + u * u * lamp1;
  const double K22_24 = vv * lamp2, K22_44 = abvE + vv * vv * lamp1;
  const double K33_34 = w * lamp2, K33_44 = abvE + w * w * lamp1;
  const double K12_14 = vv * lam, K12_42 = u * lam, K12_44 = u * vv * lamp1;
  const double K13_14 = w * lam, K13_43 = u * lam, K13_44 = u * w * lamp1;
  const double K23_24 = w * lam, K23_43 = vv * lam, K23_44 = vv * w * lamp1;
  FX[0] = 0.0;
  FX[1] = -(lamp2 * dV1 + K11_14 * dV4) * sx - (lam * dV2 + K12_14 * dV4) * sy - (lam * dV3 + K13_14 * dV4) * sz;
  FX[2] = -(dV2 + vv * dV4) * sx - (dV1 + u * dV4) * sy;
  FX[3] = -(dV3 + w * dV4) * sx - (dV1 + u * dV4) * sz;
  FX[4] = -(K11_14 * dV1 + vv * dV2 + w * dV3 + K11_44 * dV4) * sx
          - (vv * dV1 + K12_42 * dV2 + K12_44 * dV4) * sy - (w * dV1 + K13_43 * dV3 + K13_44 * dV4) * sz;
  FY[0] = 0.0;
  FY[1] = -(dV2 + vv * dV4) * sx - (dV1 + u * dV4) * sy;
  FY[2] = -(lam * dV1 + K12_42 * dV4) * sx - (lamp2 * dV2 + K22_24 * dV4) * sy - (lam * dV3 + K23_24 * dV4) * sz;
  FY[3] = -(dV3 + w * dV4) * sy - (dV2 + vv * dV4) * sz;
  FY[4] = -(K12_14 * dV1 + u * dV2 + K12_44 * dV4) * sx
          - (u * dV1 + K22_24 * dV2 + w * dV3 + K22_44 * dV4) * sy - (w * dV2 + K23_43 * dV3 + K23_44 * dV4) * sz;
  FZ[0] = 0.0;
  FZ[1] = -(dV3 + w * dV4) * sx - (dV1 + u * dV4) * sz;
  FZ[2] = -(dV3 + w * dV4) * sy - (dV2 + vv * dV4) * sz;
  FZ[3] = -(lam * dV1 + K13_43 * dV4) * sx - (lam * dV2 + K23_43 * dV4) * sy - (lamp2 * dV3 + K33_34 * dV4) * sz;
  FZ[4] = -(K13_14 * dV1 + u * dV3 + K13_44 * dV4) * sx
          - (K23_24 * dV2 + vv * dV3 + K23_44 * dV4) * sy - (u * dV1 + vv * dV2 + K33_34 * dV3 + K33_44 * dV4) * sz;
}

}  // namespace
}  // namespace vcp
