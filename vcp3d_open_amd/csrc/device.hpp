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

}  // namespace
}  // namespace vcp
