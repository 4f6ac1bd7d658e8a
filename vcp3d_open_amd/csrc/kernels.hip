// gfx950 kernels of the VCP3D explicit DG residual and SSP-RK3 stage beside the
// three that are compiled per shape, and the launches of all of them.
//
// Per shape, in sources of their own:
//   face_kernel          (face.hip) interior (incl. periodic) faces: traces of
//                        both elements, Ismail-Roe + viscous + penalty +
//                        symmetrising fluxes, lifted to both elements into
//                        per-element face slots (no atomics)
//   volume_cols_kernel   (volume.hip) volume residual, gather of the six face
//                        slots, per-element entropy mass-matrix PCG, optional
//                        in-place RK stage update, one thread per column of points
//   volume_kernel        (volume_workgroup.hip) the same with one workgroup per
//                        element: the form of small cases
// Here:
//   mach_kernel          boundary-averaged Mach number partial sums (NSCBC)
//   nscbc_kernel         PC-NSCBC boundary faces: characteristic boundary
//                        state, polynomial-correction reconstruction, flux
//                        and lift into the element's face slot
//   time_step_kernel     per-element stable time step and global minimum
//   stage0_kernel        U <- U0 - dt R (buffers swapped by the host)
//
// Reference behaviour followed (VCP3D_CurviLinear/src/):
//   ElementClass::VolumeResidual          ElementClass.cpp:3809-4443
//   ElementClass::{I,J,K}FaceResiduals    ElementClass.cpp:2582-3400
//   FluxesBoundaryFace + NSCBC states     FluxesFace.cpp:16-214,
//                                         BoundaryState.cpp:829-2241
//   AverageDataNSCBC / AverageMachNSCBC   SolverClass.cpp:2502-2581,
//                                         ElementClass.cpp:365-479
//   sponge layer / CML sources            ElementClass.cpp:3887-4117, :4450-4489
//   FluxesInternalFace / InviscidFluxesFace / ViscousFluxesFace /
//   PenAndSymFluxesSymmVar                FluxesFace.cpp:220-343, :813-975,
//                                         :1290-1651, :1152-1284
//   CG_EntropyVarMassMatrix               CG_MassMatrix.cpp:250-504
//   ElementClass::ComputeTimeStep         ElementClass.cpp:1522-1644
//   SolverClass::ExecuteTimeSynchronizationStep  SolverClass.cpp:2177-2422
#include "device.hpp"
#include "kernels.hpp"

#include <cstdint>
#include <mutex>

// Fixed device array that vcp_residual_static uses for the face-slot buffer
// instead of the context's own (for callers that cannot allocate device
// memory). Host code never names it directly: its per-device address comes
// from hipGetSymbolAddress (static_scratch).
static __device__ __align__(256) double scratch[vcp::kStaticScratchBytes / sizeof(double)];

namespace vcp {
namespace {

enum : int { kBCOutflowNSCBC = 1, kBCInflowStaticNSCBC = 2, kBCInflowTotalNSCBC = 3, kBCInflowSubsonic = 4,
              kBCOutflowSubsonic = 5, kBCWallHeatFlux = 6, kBCWallIsothermal = 7, kBCWallInviscid = 8,
              kBCInflowSupersonic = 9, kBCOutflowSupersonic = 10, kBCFarfield = 11 };

// ================================================= open-boundary kernels
template <int K, int M>
struct BndArgs {
  const double *U, *tables, *econst, *bgeo;   // bgeo: [nBFace][13][nInt2D] own face metric
  const int *bface;
  double *machPart, *faceRes, *forcePart;
  TableOffsets to;
  int bug, monitor;             // monitor: wall forces of this residual into forcePart
  double mu, tauFact, thetaHalf;
  int sgs, nElem;
  double *eddyPart;             // eddy-viscosity maxima (null: no SGS model)
  NscbcParams nb;
};

// Operators and trace of one element face in LDS (runtime direction).
template <int K, int M>
struct BndSmem {
  double A[M * K], D[M * K], F[2][K], P1[M * M], dL[M * M], W2[M * M];
  double B[2][5 * K * K];          // normal contraction: value, normal derivative
  double T[3][5 * K * M];          // fast contraction: A, D (of value), A (of normal derivative)
  double S[4][5 * M * M];          // interior trace: value, d/d(normal), d/d(fast), d/d(slow)
  double Q[4][5 * M * M];          // boundary state: value, d/d(normal), d/d(fast), d/d(slow)
  double X[2][5 * M * M];          // B matrix / PC stage; later flux + spare
  double Sym[3][5 * M * M];        // symmetrising fluxes (normal, fast, slow)
  double red[2];
};

// Trace of element e's face (dir, side): values and parametric derivatives
// in the face-local (normal, fast, slow) slots, [5][slow][fast] layout
// (TensorProductSolAndGrad{I,J,K}Face).
template <int K, int M>
__device__ void bnd_trace(BndSmem<K, M> &sm, const double *Ue, int dir, int side, bool grads)
{
  constexpr int ND = K * K * K, N2 = M * M;
  const int tid = threadIdx.x;
  const int SN = dir == 0 ? 1 : dir == 1 ? K : K * K;
  const int SFA = dir == 0 ? K : 1;
  const int SSL = dir == 2 ? K : K * K;
  const double *Fv = sm.F[0], *dFv = sm.F[1];
  for (int pc = tid; pc < 5 * K * K; pc += 64) {
    const int v = pc / (K * K), sl = (pc / K) % K, f = pc % K;
    const double *u = Ue + v * ND + sl * SSL + f * SFA;
    double b0 = 0.0, b1 = 0.0;
#pragma unroll
    for (int t = 0; t < K; ++t) { const double x = u[t * SN]; b0 += Fv[t] * x; b1 += dFv[t] * x; }
    sm.B[0][pc] = b0; sm.B[1][pc] = b1;
  }
  __syncthreads();
  for (int pc = tid; pc < 5 * K; pc += 64) {
    double x0[K], x1[K];
#pragma unroll
    for (int f = 0; f < K; ++f) { x0[f] = sm.B[0][pc * K + f]; x1[f] = sm.B[1][pc * K + f]; }
    for (int n = 0; n < M; ++n) {
      double tA = 0.0, tD = 0.0, tN = 0.0;
#pragma unroll
      for (int f = 0; f < K; ++f) { tA += sm.A[n * K + f] * x0[f]; tD += sm.D[n * K + f] * x0[f]; tN += sm.A[n * K + f] * x1[f]; }
      sm.T[0][pc * M + n] = tA; sm.T[1][pc * M + n] = tD; sm.T[2][pc * M + n] = tN;
    }
  }
  __syncthreads();
  for (int idx = tid; idx < 5 * N2; idx += 64) {
    const int v = idx / N2, m = idx - v * N2, sp = m / M, fp = m - sp * M;
    double val = 0.0, gN = 0.0, gF = 0.0, gS = 0.0;
#pragma unroll
    for (int sl = 0; sl < K; ++sl) {
      const double a = sm.A[sp * K + sl], xa = sm.T[0][(v * K + sl) * M + fp];
      val += a * xa;
      if (grads) { gS += sm.D[sp * K + sl] * xa; gN += a * sm.T[2][(v * K + sl) * M + fp]; gF += a * sm.T[1][(v * K + sl) * M + fp]; }
    }
    sm.S[0][idx] = val;
    if (grads) { sm.S[1][idx] = gN; sm.S[2][idx] = gF; sm.S[3][idx] = gS; }
  }
  __syncthreads();
}

template <int K, int M>
__device__ void bnd_load_ops(BndSmem<K, M> &sm, const BndArgs<K, M> &a, int side)
{
  const int tid = threadIdx.x;
  const double *T = a.tables;
  for (int i = tid; i < M * K; i += 64) { sm.A[i] = T[a.to.A + i]; sm.D[i] = T[a.to.D + i]; }
  for (int i = tid; i < K; i += 64) {
    sm.F[0][i] = T[(side ? a.to.fmax : a.to.fmin) + i];
    sm.F[1][i] = T[(side ? a.to.dfmax : a.to.dfmin) + i];
  }
  for (int i = tid; i < M * M; i += 64) {
    sm.P1[i] = T[a.to.P1 + i]; sm.dL[i] = T[a.to.dLq + i]; sm.W2[i] = T[a.to.w2 + i];
  }
  __syncthreads();
}

// Weighted face-normal Mach number of one boundary face
// (WeightedMachElement, BoundaryState.cpp:935-994).
template <int K, int M>
__global__ __launch_bounds__(64) void mach_kernel(BndArgs<K, M> a)
{
  constexpr int ND = K * K * K, N2 = M * M;
  __shared__ BndSmem<K, M> sm;
  const int b = blockIdx.x;
  const int e = a.bface[2 * b], f = a.bface[2 * b + 1];
  const int dir = f / 2, side = f % 2;
  if (a.nb.bc[f] > kBCInflowTotalNSCBC) {   // not a characteristic face: no part in the average
    if (threadIdx.x == 0) a.machPart[b] = 0.0;
    return;
  }
  bnd_load_ops(sm, a, side);
  bnd_trace(sm, a.U + (size_t) e * 5 * ND, dir, side, false);
  const double *g = a.bgeo + (size_t) b * 13 * N2;
  double sum = 0.0;
  for (int m = threadIdx.x; m < N2; m += 64) {
    const double *rr = g + (size_t) (4 + 3 * dir) * N2;
    const double rx = rr[m], ry = rr[N2 + m], rz = rr[2 * N2 + m];
    const double mag = sqrt(rx * rx + ry * ry + rz * rz);
    const double V4Inv = 1.0 / sm.S[0][4 * N2 + m];
    const double u = -V4Inv * sm.S[0][N2 + m], v = -V4Inv * sm.S[0][2 * N2 + m], w = -V4Inv * sm.S[0][3 * N2 + m];
    const double c = sqrt(-kGam * V4Inv);
    const double urr = (u * rx + v * ry + w * rz) / mag;
    sum += sm.W2[m] * g[3 * N2 + m] * (urr / c);
  }
  sum = wave_sum(sum);
  if (threadIdx.x == 0) a.machPart[b] = sum;
}

// One wave per physical boundary face: on a PC-NSCBC face the characteristic
// boundary state (BoundaryState.cpp:996-2241) and its polynomial-correction
// reconstruction, on the other faces (subsonic in/outflow, walls) a pointwise
// boundary state; then the boundary flux (FluxesBoundaryFace,
// FluxesFace.cpp:16-214) and its lift into the element's face slot. The
// branch is uniform over the workgroup (one face each).
template <int K, int M>
__global__ __launch_bounds__(64) void nscbc_kernel(BndArgs<K, M> a)
{
  constexpr int ND = K * K * K, N2 = M * M;
  __shared__ BndSmem<K, M> sm;
  const int b = blockIdx.x, tid = threadIdx.x;
  const int e = a.bface[2 * b], f = a.bface[2 * b + 1];
  const int dir = f / 2, side = f % 2;
  const double fn = side ? 1.0 : -1.0;
  const int bc = a.nb.bc[f];
  bnd_load_ops(sm, a, side);
  bnd_trace(sm, a.U + (size_t) e * 5 * ND, dir, side, true);
  const double *g = a.bgeo + (size_t) b * 13 * N2;
  // parametric slot (0 r, 1 s, 2 t) of the normal, fast and slow face axes
  const int pN = dir, pF = dir == 0 ? 1 : 0, pS = dir == 2 ? 1 : 2;
  const bool nscbc = bc <= kBCInflowTotalNSCBC;
  if (nscbc) {
    // boundary-averaged Mach number (fixed summation order)
    double mach = 0.0;
    for (int i = a.nb.begin[f] + tid; i < a.nb.begin[f + 1]; i += 64) mach += a.machPart[i];
    mach = wave_sum(mach) * a.nb.invArea[f];
    const double dell = fn * a.nb.dell0;
    const int iPhi = fn > 0.0 ? 0 : 4, iPsi = iPhi == 0 ? 4 : 0;

    for (int m = tid; m < N2; m += 64) {
      // entropy -> primitive state and derivatives (BoundaryState.cpp:1002-1108)
      double V[5], Q[5], dQ[3][5];
  #pragma unroll
      for (int v = 0; v < 5; ++v) V[v] = sm.S[0][v * N2 + m];
      const double V4Inv = 1.0 / V[4];
      const double u = -V4Inv * V[1], v = -V4Inv * V[2], w = -V4Inv * V[3];
      const double ek = 0.5 * (u * u + v * v + w * w);
      const double sEnt = kGam - kGm1 * (V[0] - V[4] * ek);
      const double a2 = -kGam * V4Inv;
      const double rho = pow_m2p5(-V[4] * exp(sEnt));
      const double p = a2 * rho / kGam;
      const double povrho = -V4Inv;
      const double E = povrho / kGm1 + ek, H = E + povrho;
  #pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double *dV = sm.S[1 + c];
        const double d0 = dV[m], d1 = dV[N2 + m], d2 = dV[2 * N2 + m], d3 = dV[3 * N2 + m], d4 = dV[4 * N2 + m];
        dQ[c][0] = rho * d0 + rho * u * d1 + rho * v * d2 + rho * w * d3 + rho * E * d4;
        dQ[c][1] = povrho * d1 + povrho * u * d4;
        dQ[c][2] = povrho * d2 + povrho * v * d4;
        dQ[c][3] = povrho * d3 + povrho * w * d4;
        dQ[c][4] = p * d0 + p * u * d1 + p * v * d2 + p * w * d3 + p * H * d4;
      }
      Q[0] = rho; Q[1] = u; Q[2] = v; Q[3] = w; Q[4] = p;
      // normal wave amplitudes with the incoming ones replaced
      const double rr[3] = {g[(4 + 3 * pN) * N2 + m], g[(5 + 3 * pN) * N2 + m], g[(6 + 3 * pN) * N2 + m]};
      const double magrr = sqrt(rr[0] * rr[0] + rr[1] * rr[1] + rr[2] * rr[2]);
      const double ovmagrr = 1.0 / magrr;
      const double rn[3] = {rr[0] * ovmagrr, rr[1] * ovmagrr, rr[2] * ovmagrr};
      const double drhodr = dQ[0][0], dudr = dQ[0][1], dvdr = dQ[0][2], dwdr = dQ[0][3], dpdr = dQ[0][4];
      const double ovrho = 1.0 / rho, c2 = kGam * p * ovrho, c = sqrt(c2);
      const double ova2 = 1.0 / c2, rhoa = rho * c, ovrhoa = 1.0 / rhoa, rhova = rho / c;
      const double dsdr = drhodr - ova2 * dpdr;
      const double dw1dr = rn[1] * dwdr - rn[2] * dvdr;
      const double dw2dr = rn[2] * dudr - rn[0] * dwdr;
      const double dw3dr = rn[0] * dvdr - rn[1] * dudr;
      const double durdr = rn[0] * dudr + rn[1] * dvdr + rn[2] * dwdr;
      double LL[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
      double lmb1, lmb3;
      if (bc == kBCOutflowNSCBC) {
        // BoundaryState.cpp:1318-1519
        const double sign = iPhi == 0 ? -1.0 : 1.0;
        const double kk = 0.5 * a.nb.outlet_sigma * (1.0 - mach * mach) / a.nb.outlet_len;
        const double bl = a.nb.outlet_beta_l < 0.0 ? mach : a.nb.outlet_beta_l;
        const double bt = a.nb.outlet_beta_t < 0.0 ? mach : a.nb.outlet_beta_t;
        const double cbl = a.nb.outlet_one_minus_beta ? fmin(1.0, 1.0 - bl) : fmin(1.0, bl);
        const double cbt = a.nb.outlet_one_minus_beta ? fmin(1.0, 1.0 - bt) : fmin(1.0, bt);
        const double ss[3] = {g[(4 + 3 * pF) * N2 + m], g[(5 + 3 * pF) * N2 + m], g[(6 + 3 * pF) * N2 + m]};
        const double tt[3] = {g[(4 + 3 * pS) * N2 + m], g[(5 + 3 * pS) * N2 + m], g[(6 + 3 * pS) * N2 + m]};
        const double duds = dQ[1][1], dudt = dQ[2][1], dvds = dQ[1][2], dvdt = dQ[2][2];
        const double dwds = dQ[1][3], dwdt = dQ[2][3], dpds = dQ[1][4], dpdt = dQ[2][4];
        const double ur = u * rr[0] + v * rr[1] + w * rr[2];
        const double us = u * ss[0] + v * ss[1] + w * ss[2];
        const double ut = u * tt[0] + v * tt[1] + w * tt[2];
        const double arr = c * magrr;
        const double ars = c * (rn[0] * ss[0] + rn[1] * ss[1] + rn[2] * ss[2]);
        const double art = c * (rn[0] * tt[0] + rn[1] * tt[1] + rn[2] * tt[2]);
        lmb1 = ur - arr; lmb3 = ur + arr;
        const double durds = rn[0] * duds + rn[1] * dvds + rn[2] * dwds;
        const double durdt = rn[0] * dudt + rn[1] * dvdt + rn[2] * dwdt;
        LL[0] = 0.5 * lmb1 * (ovrhoa * dpdr - durdr);
        LL[1] = rn[0] * dsdr - dw1dr;
        LL[2] = rn[1] * dsdr - dw2dr;
        LL[3] = rn[2] * dsdr - dw3dr;
        LL[4] = 0.5 * lmb3 * (ovrhoa * dpdr + durdr);
        const double LT = 0.5 * ovrhoa * (us + sign * ars) * dpds + sign * 0.5 * us * durds
                        + 0.5 * ovrhoa * (ut + sign * art) * dpdt + sign * 0.5 * ut * durdt;
        const double TT = -0.5 * c * (ss[0] * duds + ss[1] * dvds + ss[2] * dwds
                                    + tt[0] * dudt + tt[1] * dvdt + tt[2] * dwdt);
        LL[iPhi] = kk * ovrho * magrr * (p - a.nb.data[f][0]) - cbl * LT + cbt * TT;
      } else if (bc == kBCInflowStaticNSCBC) {
        // BoundaryState.cpp:1596-1783
        const double sign = fn > 0.0 ? -1.0 : 1.0;
        const double ka = sign * 0.5 * a.nb.inlet_sigma * (1.0 - mach * mach) / a.nb.inlet_len;
        const double ku = a.nb.inlet_sigma / a.nb.inlet_len;
        const double ur = u * rr[0] + v * rr[1] + w * rr[2];
        const double arr = c * magrr;
        lmb1 = ur - arr; lmb3 = ur + arr;
        if (a.nb.inlet_incoming) {
          LL[0] = 0.5 * lmb1 * (ovrhoa * dpdr - durdr);
          LL[4] = 0.5 * lmb3 * (ovrhoa * dpdr + durdr);
        }
        const double drho = rho - a.nb.data[f][0], du = u - a.nb.data[f][1], dv = v - a.nb.data[f][2],
                     dw = w - a.nb.data[f][3];
        const double kaol = ku * c * (1.0 / ur);
        LL[iPhi] = ka * c * (rr[0] * du + rr[1] * dv + rr[2] * dw);
        LL[1] = kaol * (rr[2] * dv - rr[1] * dw + rr[0] * drho);
        LL[2] = kaol * (rr[0] * dw - rr[2] * du + rr[1] * drho);
        LL[3] = kaol * (rr[1] * du - rr[0] * dv + rr[2] * drho);
      } else {
        // total-condition inflow, BoundaryState.cpp:1866-2184
        const double ovrg = 1.0 / 287.058, ovcp = kGm1 / (kGam * 287.058);
        const double kk = -a.nb.inlet_sigma / a.nb.inlet_len;
        const double ova = 1.0 / c, T = p * ovrho * ovrg;
        const double ur = u * rn[0] + v * rn[1] + w * rn[2];
        const double w1 = rn[1] * w - rn[2] * v, w2 = rn[2] * u - rn[0] * w, w3 = rn[0] * v - rn[1] * u;
        lmb1 = ur - c; lmb3 = ur + c;
        const double ovlmb2 = 1.0 / ur;
        if (a.nb.inlet_incoming) {
          LL[0] = 0.5 * lmb1 * (ovrhoa * dpdr - durdr);
          LL[4] = 0.5 * lmb3 * (ovrhoa * dpdr + durdr);
        }
        const double magU2 = 2.0 * ek, magU = sqrt(magU2);
        const double ff = 1.0 + 0.5 * kGm1 * (magU2 / c2);
        const double Pt = p * pow(ff, kGam / kGm1), Tt = T * ff;
        const double Zt = v / magU, Zp = w / magU;
        const double ka = kk * c;
        const double X1 = ka * (Pt - a.nb.data[f][0]), X2 = ka * (Tt - a.nb.data[f][1]);
        const double X3 = ka * (Zt - a.nb.data[f][3]), X4 = ka * (Zp - a.nb.data[f][4]);
        const double ovrPtovTt = ovrg * (Pt / Tt), Ttovrho = Tt * ovrho;
        const double govaPt = kGam * ova * Pt, ekovrho = ek * ovrho, gm1ekova = kGm1 * ek * ova;
        const double gm1ovaTt = kGm1 * ova * Tt, ovmagU2 = 1.0 / magU2;
        const double gp = gm1ekova + ur, gmn = gm1ekova - ur;
        const double f1 = w1 - rn[0] * ekovrho, f2 = w2 - rn[1] * ekovrho, f3 = w3 - rn[2] * ekovrho;
        const double A1 = gp * ovrPtovTt - govaPt, A2 = f1 * ovrPtovTt, A3 = f2 * ovrPtovTt, A4 = f3 * ovrPtovTt;
        const double A5 = gmn * ovrPtovTt - govaPt;
        const double B1 = gp * ovcp - gm1ovaTt, B2 = f1 * ovcp + rn[0] * Ttovrho, B3 = f2 * ovcp + rn[1] * Ttovrho;
        const double B4 = f3 * ovcp + rn[2] * Ttovrho, B5 = gmn * ovcp - gm1ovaTt;
        const double C1 = (rn[1] * magU - ur * Zt) * ovmagU2, C2 = -(rn[2] * magU + w1 * Zt) * ovmagU2;
        const double C3 = (-w2 * Zt) * ovmagU2, C4 = (rn[0] * magU - w3 * Zt) * ovmagU2, C5 = -C1;
        const double D1 = (rn[2] * magU - ur * Zp) * ovmagU2, D2 = (rn[1] * magU - w1 * Zp) * ovmagU2;
        const double D3 = -(rn[0] * magU + w2 * Zp) * ovmagU2, D4 = (-w3 * Zp) * ovmagU2, D5 = -D1;
        const double Y1 = LL[iPsi] * A1, Y2 = LL[iPsi] * B1, Y3 = LL[iPsi] * C1, Y4 = LL[iPsi] * D1;
        // elimination of the 4 x 4 system for the incoming amplitudes
        const double ovA2 = 1.0 / A2;
        const double E0 = ovA2 * X1, E3 = -ovA2 * A3, E4 = -ovA2 * A4, E5 = -ovA2 * A5, P2 = -ovA2 * Y1;
        const double ovdF = 1.0 / (D3 + D2 * E3);
        const double F0 = ovdF * (X4 - D2 * E0), F4 = -ovdF * (D4 + D2 * E4), F5 = -ovdF * (D5 + D2 * E5);
        const double P3 = -ovdF * (Y4 + D2 * P2);
        const double ovdG = 1.0 / (C4 + C2 * E4 + C3 * F4 + C2 * E3 * F4);
        const double G0 = ovdG * (X3 - C2 * E0 - C3 * F0 - C2 * E3 * F0);
        const double G5 = -ovdG * (C5 + C2 * E5 + C3 * F5 + C2 * E3 * F5);
        const double P4 = -ovdG * (Y3 + C2 * P2 + C3 * P3 + C2 * E3 * P3);
        const double ovdH = 1.0 / (B5 + B2 * E5 + B3 * F5 + B4 * G5 + B2 * E3 * F5 + B2 * E4 * G5 + B3 * F4 * G5
                                   + B2 * E3 * F4 * G5);
        const double H0 = ovdH * (X2 - B2 * E0 - B3 * F0 - B4 * G0 - B2 * E3 * F0 - B2 * E4 * G0 - B3 * F4 * G0
                                  - B2 * E3 * F4 * G0);
        const double P5 = -ovdH * (Y2 + B2 * P2 + B3 * P3 + B4 * P4 + B2 * E3 * P3 + B2 * E4 * P4 + B3 * F4 * P4
                                   + B2 * E3 * F4 * P4);
        LL[iPhi] = H0 + P5;
        LL[3] = G0 + G5 * LL[iPhi] + P4;
        LL[2] = F0 + F4 * LL[3] + F5 * LL[iPhi] + P3;
        LL[1] = E0 + E3 * LL[2] + E4 * LL[3] + E5 * LL[iPhi] + P2;
        LL[1] *= ovlmb2; LL[2] *= ovlmb2; LL[3] *= ovlmb2;
      }
      // target normal derivative of the primitive state and the B matrix
      const double ovlmb1 = 1.0 / lmb1, ovlmb3 = 1.0 / lmb3;
      double t[5];
      t[0] = ovlmb1 * rhova * LL[0] + rn[0] * LL[1] + rn[1] * LL[2] + rn[2] * LL[3] + ovlmb3 * rhova * LL[4];
      t[1] = -ovlmb1 * rn[0] * LL[0] - rn[2] * LL[2] + rn[1] * LL[3] + ovlmb3 * rn[0] * LL[4];
      t[2] = -ovlmb1 * rn[1] * LL[0] + rn[2] * LL[1] - rn[0] * LL[3] + ovlmb3 * rn[1] * LL[4];
      t[3] = -ovlmb1 * rn[2] * LL[0] - rn[1] * LL[1] + rn[0] * LL[2] + ovlmb3 * rn[2] * LL[4];
      t[4] = ovlmb1 * rhoa * LL[0] + ovlmb3 * rhoa * LL[4];
  #pragma unroll
      for (int q = 0; q < 5; ++q) {
        sm.Q[1][q * N2 + m] = t[q];
        sm.X[0][q * N2 + m] = t[q] - (dQ[0][q] - Q[q] * dell);
      }
    }
    __syncthreads();
    // polynomial correction Q_b = (P1 x P1) B / dell (sign of the face):
    // fast axis, then slow axis
    for (int idx = tid; idx < 5 * N2; idx += 64) {
      const int row = idx / M, j = idx - row * M;
      double s = 0.0;
  #pragma unroll
      for (int q = 0; q < M; ++q) s += sm.P1[j * M + q] * sm.X[0][row * M + q];
      sm.X[1][idx] = s;
    }
    __syncthreads();
    const double scale = 1.0 / dell;
    for (int idx = tid; idx < 5 * N2; idx += 64) {
      const int v = idx / N2, m = idx - v * N2, i = m / M, j = m - i * M;
      double s = 0.0;
  #pragma unroll
      for (int q = 0; q < M; ++q) s += sm.P1[i * M + q] * sm.X[1][(v * M + q) * M + j];
      sm.Q[0][idx] = s * scale;
    }
    __syncthreads();
    // primitive -> entropy variables for the state and its normal derivative
    for (int m = tid; m < N2; m += 64) {
      const double rho = sm.Q[0][m], u = sm.Q[0][N2 + m], v = sm.Q[0][2 * N2 + m], w = sm.Q[0][3 * N2 + m],
                   p = sm.Q[0][4 * N2 + m];
      const double dr = sm.Q[1][m], du = sm.Q[1][N2 + m], dv = sm.Q[1][2 * N2 + m], dw = sm.Q[1][3 * N2 + m],
                   dp = sm.Q[1][4 * N2 + m];
      const double sEnt = log(p / pow(rho, kGam));
      const double ovrho = 1.0 / rho, ovp = 1.0 / p, rovp = rho * ovp;
      const double ek = 0.5 * (u * u + v * v + w * w);
      const double W1 = rovp * u, W2 = rovp * v, W3 = rovp * w;
      sm.Q[0][m] = -rovp * ek + (kGam - sEnt) / kGm1;
      sm.Q[0][N2 + m] = W1; sm.Q[0][2 * N2 + m] = W2; sm.Q[0][3 * N2 + m] = W3; sm.Q[0][4 * N2 + m] = -rovp;
      const double q0 = kGam / kGm1 * ovrho - ovp * ek, q4 = ovp * (rovp * ek - 1.0 / kGm1);
      sm.Q[1][m] = q0 * dr - W1 * du - W2 * dv - W3 * dw + q4 * dp;
      sm.Q[1][N2 + m] = u * ovp * dr + rovp * du - ovp * W1 * dp;
      sm.Q[1][2 * N2 + m] = v * ovp * dr + rovp * dv - ovp * W2 * dp;
      sm.Q[1][3 * N2 + m] = w * ovp * dr + rovp * dw - ovp * W3 * dp;
      sm.Q[1][4 * N2 + m] = -ovp * dr + ovp * rovp * dp;
    }
    __syncthreads();
    // transverse derivatives of the reconstructed state on the Gauss points;
    // the reference stores the slow-axis derivative in the fast-axis slot
    // (BoundaryState.cpp:1261-1287)
    double *dSlow = a.bug ? sm.Q[2] : sm.Q[3];
    double *dFast = a.bug ? sm.Q[3] : sm.Q[2];
    for (int idx = tid; idx < 5 * N2; idx += 64) {
      const int v = idx / N2, m = idx - v * N2, i = m / M, j = m - i * M;
      const double *q0 = sm.Q[0] + v * N2;
      double ds = 0.0, dt = 0.0;
  #pragma unroll
      for (int k = 0; k < M; ++k) { ds += sm.dL[i * M + k] * q0[k * M + j]; dt += sm.dL[j * M + k] * q0[i * M + k]; }
      dSlow[idx] = ds; dFast[idx] = dt;
    }
    __syncthreads();
  } else {
    // pointwise boundary state (BoundaryState.cpp:40-118, :156-372,
    // :399-604, :636-792, entropy variables); d: the face's non-dimensional
    // prescribed data
    const double *d = a.nb.data[f];
    for (int m = tid; m < N2; m += 64) {
      double V[5], R[5];
#pragma unroll
      for (int v = 0; v < 5; ++v) V[v] = sm.S[0][v * N2 + m];
      const double n0 = g[m], n1 = g[N2 + m], n2 = g[2 * N2 + m];
      if (bc == kBCWallInviscid) {
        const double Vn = V[1] * n0 + V[2] * n1 + V[3] * n2;
        R[0] = V[0] - 0.5 * Vn * Vn / V[4];
        R[1] = V[1] - Vn * n0; R[2] = V[2] - Vn * n1; R[3] = V[3] - Vn * n2;
        R[4] = V[4];
      } else if (bc == kBCWallHeatFlux || bc == kBCWallIsothermal) {
        R[0] = V[0] - 0.5 * (V[1] * V[1] + V[2] * V[2] + V[3] * V[3]) / V[4];
        R[1] = 0.0; R[2] = 0.0; R[3] = 0.0;
        R[4] = bc == kBCWallHeatFlux ? V[4] : d[1] / d[0];   // d[1] = -pRef / (R rhoRef)
      } else if (bc == kBCInflowSubsonic) {
        const double V4Inv = 1.0 / V[4];
        const double u = -V4Inv * V[1], v = -V4Inv * V[2], w = -V4Inv * V[3];
        const double a2 = -kGam * V4Inv, c = sqrt(a2);
        const double nx = fn * n0, ny = fn * n1, nz = fn * n2;
        const double un = u * nx + v * ny + w * nz;
        double riemann = 2.0 * c * kInvGm1 + un;
        const double H = a2 * kInvGm1 + 0.5 * (u * u + v * v + w * w);
        riemann *= sqrt(d[1] / H);
        const double alpha = nx * d[2] + ny * d[3] + nz * d[4];
        const double aa = 1.0 + 0.5 * kGm1 * alpha * alpha;
        const double bb = -kGm1 * alpha * riemann;
        const double cc = 0.5 * kGm1 * riemann * riemann - 2.0 * d[1];
        double dd = bb * bb - 4.0 * aa * cc; dd = sqrt(fmax(0.0, dd));
        double qR = (-bb + dd) / (2.0 * aa); qR = fmax(0.0, qR);
        double qR2 = qR * qR;
        double aR2 = kGm1 * (d[1] - 0.5 * qR2);
        double MR2 = qR2 / aR2; MR2 = fmin(1.0, MR2);
        const double tmp = 1.0 / (1.0 + 0.5 * kGm1 * MR2);
        aR2 = kGm1 * d[1] * tmp;
        qR2 = MR2 * aR2;
        qR = sqrt(qR2);
        const double pR = d[0] * pow(tmp, kGam * kInvGm1);
        const double rhoR = kGam * pR / aR2;
        const double pRInv = 1.0 / pR;
        const double sR = log(pR / pow(rhoR, kGam));
        R[0] = (kGam - sR) * kInvGm1 - 0.5 * pRInv * rhoR * qR2;
        R[1] = rhoR * pRInv * qR * d[2]; R[2] = rhoR * pRInv * qR * d[3]; R[3] = rhoR * pRInv * qR * d[4];
        R[4] = -rhoR * pRInv;
      } else if (bc == kBCInflowSupersonic || bc == kBCFarfield) {   // the prescribed / free-stream state
#pragma unroll
        for (int v = 0; v < 5; ++v) R[v] = d[v];
      } else if (bc == kBCOutflowSupersonic) {  // the interior state
#pragma unroll
        for (int v = 0; v < 5; ++v) R[v] = V[v];
      } else {   // subsonic outflow
        const double V4Inv = 1.0 / V[4];
        const double u = -V4Inv * V[1], v = -V4Inv * V[2], w = -V4Inv * V[3];
        const double eKin = 0.5 * (u * u + v * v + w * w);
        const double sEnt = kGam - kGm1 * (V[0] - V[4] * eKin);
        const double c = sqrt(-kGam * V4Inv);
        const double nx = fn * n0, ny = fn * n1, nz = fn * n2;
        const double un = u * nx + v * ny + w * nz;
        const double riemann = 2.0 * c * kInvGm1 + un;
        const double pR = d[0];
        const double rhoR = pow(pR / exp(sEnt), 1.0 / kGam);
        const double aR = sqrt(kGam * pR / rhoR);
        const double unR = riemann - 2.0 * aR * kInvGm1;
        const double uR = u + (unR - un) * nx, vR = v + (unR - un) * ny, wR = w + (unR - un) * nz;
        const double pRInv = 1.0 / pR;
        R[0] = (kGam - sEnt) * kInvGm1 - 0.5 * pRInv * rhoR * (uR * uR + vR * vR + wR * wR);
        R[1] = rhoR * pRInv * uR; R[2] = rhoR * pRInv * vR; R[3] = rhoR * pRInv * wR;
        R[4] = -rhoR * pRInv;
      }
#pragma unroll
      for (int v = 0; v < 5; ++v) sm.Q[0][v * N2 + m] = R[v];
    }
    __syncthreads();
  }
  // fluxes with the face normal oriented out of the element
  const double lenScale = a.econst[(size_t) e * kElemConst + dir];
  const double tau = a.tauFact / lenScale;
  // the element's own LES length scale (ElementClass.cpp:2788-2790)
  const double lenLES = a.econst[(size_t) e * kElemConst + kElemLenLES];
  double evMax = 0.0;
  const bool wall = bc >= kBCWallHeatFlux && bc <= kBCWallInviscid;
  const bool forces = a.monitor && wall;
  double frc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  for (int m = tid; m < N2; m += 64) {
    double VL[5], VR[5], gx[5], gy[5], gz[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      VL[v] = sm.S[0][v * N2 + m];
      VR[v] = sm.Q[0][v * N2 + m];
      const int pt = a.bug ? (v < N2 ? v : 0) : m;
      double c[9];
#pragma unroll
      for (int q = 0; q < 9; ++q) c[q] = g[(4 + q) * N2 + pt];
      double pl[3], pr[3];
      pl[pN] = sm.S[1][v * N2 + m]; pl[pF] = sm.S[2][v * N2 + m]; pl[pS] = sm.S[3][v * N2 + m];
      const double xL = pl[0] * c[0] + pl[1] * c[3] + pl[2] * c[6];
      const double yL = pl[0] * c[1] + pl[1] * c[4] + pl[2] * c[7];
      const double zL = pl[0] * c[2] + pl[1] * c[5] + pl[2] * c[8];
      if (nscbc) {
        // the interior and the reconstructed gradients averaged
        pr[pN] = sm.Q[1][v * N2 + m]; pr[pF] = sm.Q[2][v * N2 + m]; pr[pS] = sm.Q[3][v * N2 + m];
        const double xR = pr[0] * c[0] + pr[1] * c[3] + pr[2] * c[6];
        const double yR = pr[0] * c[1] + pr[1] * c[4] + pr[2] * c[7];
        const double zR = pr[0] * c[2] + pr[1] * c[5] + pr[2] * c[8];
        gx[v] = 0.5 * (xL + xR); gy[v] = 0.5 * (yL + yR); gz[v] = 0.5 * (zL + zR);
      } else {
        // the interior gradient (FluxesFace.cpp:60-80)
        gx[v] = xL; gy[v] = yL; gz[v] = zL;
      }
    }
    const double nn[3] = {fn * g[m], fn * g[N2 + m], fn * g[2 * N2 + m]};
    const double wA = sm.W2[m] * g[3 * N2 + m];
    double fl[5], FX[5], FY[5], FZ[5];
    double aux[7], ev = 0.0;
    if (a.sgs) {
      ev = face_eddy(a.sgs, lenLES, VL, VR, gx, gy, gz);
      evMax = fmax(evMax, ev);
    }
    point_flux<true>(VL, VR, gx, gy, gz, nn, wA, tau, a.mu, a.thetaHalf, fl, FX, FY, FZ, wall ? 0.0 : 1.0,
                     bc == kBCWallHeatFlux, a.nb.data[f][0], forces ? aux : nullptr, a.sgs != kSgsNone, ev);
    if (forces) {
      // wall forces (FluxesFace.cpp:999-1013, :1590-1612): the averaged
      // pressure and the viscous stress on the normal into the boundary
      const double abv = 0.5 * fn * sm.W2[m] * g[3 * N2 + m] * aux[0];
      frc[0] += abv * g[m]; frc[1] += abv * g[N2 + m]; frc[2] += abv * g[2 * N2 + m];
      const double area = fn * sm.W2[m] * g[3 * N2 + m];
      const double ax = area * g[m], ay = area * g[N2 + m], az = area * g[2 * N2 + m];
      frc[3] -= aux[1] * ax + aux[4] * ay + aux[5] * az;
      frc[4] -= aux[4] * ax + aux[2] * ay + aux[6] * az;
      frc[5] -= aux[5] * ax + aux[6] * ay + aux[3] * az;
    }
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      const int pt = a.bug ? (v < N2 ? v : 0) : m;
      double c[9];
#pragma unroll
      for (int q = 0; q < 9; ++q) c[q] = g[(4 + q) * N2 + pt];
      double par[3];
      par[0] = FX[v] * c[0] + FY[v] * c[1] + FZ[v] * c[2];
      par[1] = FX[v] * c[3] + FY[v] * c[4] + FZ[v] * c[5];
      par[2] = FX[v] * c[6] + FY[v] * c[7] + FZ[v] * c[8];
      sm.X[0][v * N2 + m] = fl[v];
      sm.Sym[0][v * N2 + m] = par[pN];
      sm.Sym[1][v * N2 + m] = par[pF];
      sm.Sym[2][v * N2 + m] = par[pS];
    }
  }
  if (a.eddyPart) {
    evMax = wave_max(evMax);
    if (tid == 0) a.eddyPart[4 * a.nElem + b] = evMax;
  }
  if (a.monitor) {
    // this face's force sums (zero off the walls), summed in a fixed order
    // over the faces by force_sum_kernel
#pragma unroll
    for (int i = 0; i < 6; ++i) frc[i] = wave_sum(frc[i]);
    if (tid == 0)
#pragma unroll
      for (int i = 0; i < 6; ++i) a.forcePart[(size_t) b * 6 + i] = frc[i];
  }
  __syncthreads();
  // lift: fast axis, slow axis, then the face vectors along the normal
  double *T0 = sm.Q[0], *T1 = sm.Q[1], *T2 = sm.Q[2];
  for (int pc = tid; pc < 5 * M; pc += 64) {
    double xf[M], xF[M], xS[M], xN[M];
#pragma unroll
    for (int q = 0; q < M; ++q) {
      xf[q] = sm.X[0][pc * M + q]; xF[q] = sm.Sym[1][pc * M + q]; xS[q] = sm.Sym[2][pc * M + q]; xN[q] = sm.Sym[0][pc * M + q];
    }
    for (int n = 0; n < K; ++n) {
      double p1 = 0.0, p2 = 0.0, p3 = 0.0;
#pragma unroll
      for (int q = 0; q < M; ++q) {
        p1 += sm.A[q * K + n] * xf[q]; p1 += sm.D[q * K + n] * xF[q];
        p2 += sm.A[q * K + n] * xS[q];
        p3 += sm.A[q * K + n] * xN[q];
      }
      T0[pc * K + n] = p1; T1[pc * K + n] = p2; T2[pc * K + n] = p3;
    }
  }
  __syncthreads();
  // slow axis, straight into the face slot: value and normal-derivative
  // coefficient planes [0|1][v][slow][fast]
  double *out = a.faceRes + ((size_t) e * 6 + f) * 10 * K * K;
  for (int pc = tid; pc < 5 * K; pc += 64) {
    const int v = pc / K, fi = pc - v * K;
    double x1[M], x2[M], x3[M];
#pragma unroll
    for (int q = 0; q < M; ++q) {
      const int j = (v * M + q) * K + fi;
      x1[q] = T0[j]; x2[q] = T1[j]; x3[q] = T2[j];
    }
    for (int n = 0; n < K; ++n) {
      double g1 = 0.0, g2 = 0.0;
#pragma unroll
      for (int q = 0; q < M; ++q) { g1 += sm.A[q * K + n] * x1[q] + sm.D[q * K + n] * x2[q]; g2 += sm.A[q * K + n] * x3[q]; }
      out[(v * K + n) * K + fi] = g1; out[5 * K * K + (v * K + n) * K + fi] = g2;
    }
  }
}

// ======================================================= time-step kernel
struct DtArgs {
  CaseDev c;
  TableOffsets to;
  int P;
};

struct DtBatchArgs {
  const CaseDev *cases;
  const WorkItem *work;
  TableOffsets to;
  int P;
};

// In-place contraction of the 5 K^2 lines of sU along the axis of stride ST
// with the K x K matrix L, by one wave: every lane reads all its lines
// before any lane writes.
template <int K, int ST>
__device__ __forceinline__ void lines_inplace(double *sU, const double *L, int lane)
{
  constexpr int NL = 5 * K * K, PP = (NL + 63) / 64;
  double o[PP][K];
#pragma unroll
  for (int t = 0; t < PP; ++t) {
    const int p = lane + 64 * t;
    if (p < NL) {
      const int b = ST == 1 ? p * K : ST == K ? (p / K) * K * K + p % K : (p / (K * K)) * K * K * K + p % (K * K);
      double x[K];
#pragma unroll
      for (int q = 0; q < K; ++q) x[q] = sU[b + q * ST];
#pragma unroll
      for (int n = 0; n < K; ++n) {
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < K; ++q) s += L[n * K + q] * x[q];
        o[t][n] = s;
      }
    }
  }
#pragma unroll
  for (int t = 0; t < PP; ++t) {
    const int p = lane + 64 * t;
    if (p < NL) {
      const int b = ST == 1 ? p * K : ST == K ? (p / K) * K * K + p % K : (p / (K * K)) * K * K * K + p % (K * K);
#pragma unroll
      for (int n = 0; n < K; ++n) sU[b + n * ST] = o[t][n];
    }
  }
}

// Nodal entropy variables of element e and (GRAD) their parametric
// derivatives along r, s and t, in LDS: sV[q][v][ND], q = 0 the values, 1..3
// the derivatives (the modal basis or its derivative along each axis); one
// wave. sL, sDL: the K x K tables phi_q(r_p), phi'_q(r_p) at the nodal DOFs.
template <int K, bool GRAD>
__device__ __forceinline__ void nodal_state(const double *Ue, const double *sL, const double *sDL, double *sV,
                                            int lane)
{
  constexpr int ND = K * K * K, NQ = GRAD ? 4 : 1;
  // the modal state in chunks of up to 16 loads per lane, each chunk issued
  // before its first load is waited for
  constexpr int NL = 5 * ND, NIT = (NL + 63) / 64, CH = NIT < 16 ? NIT : 16;
  for (int c0 = 0; c0 < NIT; c0 += CH) {
    double u[CH];
#pragma unroll
    for (int t = 0; t < CH; ++t) {
      const int i = lane + 64 * (c0 + t);
      u[t] = Ue[i < NL ? i : 0];
    }
#pragma unroll
    for (int t = 0; t < CH; ++t) {
      const int i = lane + 64 * (c0 + t);
      if (i < NL)
#pragma unroll
        for (int q = 0; q < NQ; ++q) sV[q * NL + i] = u[t];
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NQ; ++q) lines_inplace<K, 1>(sV + q * 5 * ND, q == 1 ? sDL : sL, lane);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NQ; ++q) lines_inplace<K, K>(sV + q * 5 * ND, q == 2 ? sDL : sL, lane);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NQ; ++q) lines_inplace<K, K * K>(sV + q * 5 * ND, q == 3 ? sDL : sL, lane);
  __syncthreads();
}

// Dimensional eddy viscosity at nodal DOF d from nodal_state<K, true>: the
// dimensional density and velocity gradients of the entropy variables with
// the nodal metric vn (ElementClass::ComputeVelocityGradientsNodalDOFs,
// ElementClass.cpp:1649-1790) and the element's LES length scale
// (ElementClass.cpp:1562-1573, :3785-3797).
template <int K>
__device__ __forceinline__ double nodal_eddy(const CaseDev &a, const double *sV, const double *vn, double lenLES,
                                             int d)
{
  constexpr int ND = K * K * K;
  double V[5], rho, u, v, w, p, ek;
#pragma unroll
  for (int l = 0; l < 5; ++l) V[l] = sV[l * ND + d];
  ent2prim(V, rho, u, v, w, p, ek);
  rho *= a.rho_ref; p *= a.p_ref;
  const double V4Inv = -p / (a.u_ref * a.u_ref) / rho;
  const double vel[3] = {u, v, w};
  double gp[3][3];     // [velocity][r | s | t]
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const double *D = sV + (1 + r) * 5 * ND;
      gp[i][r] = -V4Inv * (D[(1 + i) * ND + d] + vel[i] * D[4 * ND + d]);
    }
  double G[3][3];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int x = 0; x < 3; ++x)
      G[i][x] = a.u_ref * (gp[i][0] * vn[(1 + x) * ND + d] + gp[i][1] * vn[(4 + x) * ND + d]
                           + gp[i][2] * vn[(7 + x) * ND + d]);
  return eddy_viscosity(a.sgs, lenLES, rho, G);
}

// Per-element time step (ElementClass::ComputeTimeStep, ElementClass.cpp:
// 1522-1644); SGS: with the eddy viscosity at the nodal DOFs in the viscous
// spectral radius, with the turbulent Prandtl number.
template <int K, bool SGS>
__device__ __forceinline__ void time_step_body(const CaseDev &a, const TableOffsets &to, const int P, const int e)
{
  constexpr int ND = K * K * K;
  __shared__ double sL[K * K], sDL[SGS ? K * K : 1], sU[(SGS ? 20 : 5) * ND];
  const int tid = threadIdx.x;
  for (int i = tid; i < K * K; i += 64) {
    sL[i] = a.tables[to.LD + i];
    if constexpr (SGS) sDL[i] = a.tables[to.DLD + i];
  }
  // modal -> nodal values (and derivatives) along i, j and k, in place
  nodal_state<K, SGS>(a.U + (size_t) e * 5 * ND, sL, sDL, sU, tid);
  const double *sT1 = sU;
  const double *ec = a.econst + (size_t) e * kElemConst;
  const double di = 1.0 / ec[0], dj = 1.0 / ec[1], dk = 1.0 / ec[2];
  const double dl2 = di * di + dj * dj + dk * dk;
  const double rvn = fmax(fmax(1.0, 2.0 + kLamOverMu), kGam / kPrLam) * dl2;
  const double rvnT = fmax(fmax(1.0, 2.0 + kLamOverMu), kGam / kPrTurb) * dl2;
  const double *vn = SGS ? a.vgeoN + (size_t) e * kNodalGeo * ND : nullptr;
  double radInv = 0.0, radVis = 0.0;
  int badA2 = 0;                     // a^2 negative or not a number at a DOF
  for (int d = tid; d < ND; d += 64) {
    double V[5];
#pragma unroll
    for (int l = 0; l < 5; ++l) V[l] = sT1[l * ND + d];
    double rho, u, v, w, p, ek;
    ent2prim(V, rho, u, v, w, p, ek);
    rho *= a.rho_ref; u *= a.u_ref; v *= a.u_ref; w *= a.u_ref; p *= a.p_ref;
    const double ri = 1.0 / rho, a2 = kGam * p * ri;
    const double vI = u * ec[4] + v * ec[5] + w * ec[6];
    const double vJ = u * ec[7] + v * ec[8] + w * ec[9];
    const double vK = u * ec[10] + v * ec[11] + w * ec[12];
    const double c = sqrt(fabs(a2));
    radInv = fmax(radInv, (fabs(vI) + c) * di + (fabs(vJ) + c) * dj + (fabs(vK) + c) * dk);
    if constexpr (SGS) {
      const double ev = nodal_eddy<K>(a, sU, vn, ec[kElemLenLES], d);
      radVis = fmax(radVis, ri * (a.muDim * rvn + ev * rvnT));
    } else {
      radVis = fmax(radVis, ri * a.muDim * rvn);
    }
    badA2 |= !(a2 >= 0.0);
  }
  radInv = wave_max(radInv); radVis = wave_max(radVis);
  const bool anyBad = __any(badA2);
  if (tid == 0) {
    const double f1[] = {2.0, 6.0, 12.0, 20.0, 28.0, 38.0, 50.0, 64.0, 80.0, 98.0};
    const double f2[] = {6.0, 36.0, 150.0, 420.0, 980.0, 1975.0, 3575.0, 7000.0, 14000.0, 28000.0};
    if (anyBad) atomicOr(a.flags, kFlagNegativeA2);
    const double dt = a.cfl * a.u_ref / (f1[P] * radInv + f2[P] * radVis);
    a.dtElem[e] = dt;
  }
}

template <int K, bool SGS>
__global__ __launch_bounds__(64) void time_step_kernel(DtArgs a)
{
  time_step_body<K, SGS>(a.c, a.to, a.P, blockIdx.x);
}

template <int K, bool SGS>
__global__ __launch_bounds__(64) void time_step_batch_kernel(DtBatchArgs b)
{
  const WorkItem w = b.work[blockIdx.x];
  const CaseDev c = b.cases[w.c];
  if (c.flags[kWordActive] == 0) return;
  time_step_body<K, SGS>(c, b.to, b.P, w.e);
}

// Running averages of the dimensional primitive variables and the velocity
// products at the nodal DOFs (ElementClass::UpdateAverageData,
// ElementClass.cpp:3741-3782): avg = factOld avg + factNew q, with q =
// (rho, u, v, w, p, uu, vv, ww, uv, uw, vw) and, with an SGS model, the eddy
// viscosity (:3785-3803); layout [nElem][11 | 12][nDOF].
struct AvgArgs {
  CaseDev c;
  double *avg;
  TableOffsets to;
  double factNew, factOld;
};

template <int K, bool SGS>
__global__ __launch_bounds__(64) void average_kernel(AvgArgs a)
{
  constexpr int ND = K * K * K, NA = SGS ? 12 : 11;
  __shared__ double sL[K * K], sDL[SGS ? K * K : 1], sU[(SGS ? 20 : 5) * ND];
  const CaseDev &c = a.c;
  const int e = blockIdx.x, tid = threadIdx.x;
  for (int i = tid; i < K * K; i += 64) {
    sL[i] = c.tables[a.to.LD + i];
    if constexpr (SGS) sDL[i] = c.tables[a.to.DLD + i];
  }
  nodal_state<K, SGS>(c.U + (size_t) e * 5 * ND, sL, sDL, sU, tid);
  double *av = a.avg + (size_t) e * NA * ND;
  const double *vn = SGS ? c.vgeoN + (size_t) e * kNodalGeo * ND : nullptr;
  for (int d = tid; d < ND; d += 64) {
    double V[5];
#pragma unroll
    for (int l = 0; l < 5; ++l) V[l] = sU[l * ND + d];
    double rho, u, v, w, p, ek;
    ent2prim(V, rho, u, v, w, p, ek);
    rho *= c.rho_ref; u *= c.u_ref; v *= c.u_ref; w *= c.u_ref; p *= c.p_ref;
    const double q[11] = {rho, u, v, w, p, u * u, v * v, w * w, u * v, u * w, v * w};
#pragma unroll
    for (int i = 0; i < 11; ++i) av[i * ND + d] = a.factOld * av[i * ND + d] + a.factNew * q[i];
    if constexpr (SGS) {
      const double ev = nodal_eddy<K>(c, sU, vn, c.econst[(size_t) e * kElemConst + kElemLenLES], d);
      av[11 * ND + d] = a.factOld * av[11 * ND + d] + a.factNew * ev;
    }
  }
}

// Sponge target from the running averages (ElementClass::InitializeDampingState,
// SpongeLayer.cpp:943-997): the averaged nodal primitive variables
// (dimensional, avg[e][0..4]) interpolated to the integration points with the
// Lagrange basis of the nodal DOFs, made non-dimensional and converted to the
// conservative variables, into dampState of the element's sponge slot. One
// wave per element; elements outside the sponge return at once.
struct DampAvgArgs {
  const double *avg, *tables;
  const int *spIdx;
  double *dampState;
  TableOffsets to;
  double u_ref, p_ref, rho_ref;
  int nAvg;                     // averaged quantities per DOF
};

template <int K, int M>
__global__ __launch_bounds__(64) void damping_avg_kernel(DampAvgArgs a)
{
  constexpr int ND = K * K * K, NI = M * M * M;
  __shared__ double sL[M * K], s0[5 * K * K * M], s1[5 * K * M * M], s2[5 * NI];
  const int e = blockIdx.x, tid = threadIdx.x;
  const int sp = a.spIdx[e];
  if (sp < 0) return;
  for (int i = tid; i < M * K; i += 64) sL[i] = a.tables[a.to.Lq + i];
  __syncthreads();
  const double *av = a.avg + (size_t) e * a.nAvg * ND;
  // along i: s0[l][k][j][p]
  for (int o = tid; o < 5 * K * K * M; o += 64) {
    const int p = o % M, r = o / M;          // r = (l k j)
    const double *x = av + (r / (K * K)) * ND + (r % (K * K)) * K;
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < K; ++q) s += sL[p * K + q] * x[q];
    s0[o] = s;
  }
  __syncthreads();
  // along j: s1[l][k][pj][pi]
  for (int o = tid; o < 5 * K * M * M; o += 64) {
    const int pi = o % M, pj = (o / M) % M, lk = o / (M * M);
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < K; ++q) s += sL[pj * K + q] * s0[(lk * K + q) * M + pi];
    s1[o] = s;
  }
  __syncthreads();
  // along k: s2[l][pk][pj][pi]
  for (int o = tid; o < 5 * NI; o += 64) {
    const int pij = o % (M * M), pk = (o / (M * M)) % M, l = o / NI;
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < K; ++q) s += sL[pk * K + q] * s1[((l * K + q) * M * M) + pij];
    s2[o] = s;
  }
  __syncthreads();
  double *ds = a.dampState + (size_t) sp * 5 * NI;
  for (int m = tid; m < NI; m += 64) {
    const double rho = s2[m] / a.rho_ref, u = s2[NI + m] / a.u_ref, v = s2[2 * NI + m] / a.u_ref,
                 w = s2[3 * NI + m] / a.u_ref, pr = s2[4 * NI + m] / a.p_ref;
    ds[m] = rho;
    ds[NI + m] = rho * u;
    ds[2 * NI + m] = rho * v;
    ds[3 * NI + m] = rho * w;
    ds[4 * NI + m] = pr * kInvGm1 + 0.5 * rho * (u * u + v * v + w * w);
  }
}

// Minimum of the per-element time steps into scal[0] (one workgroup; a
// fixed reduction order, no atomics on one address from every element).
__global__ __launch_bounds__(1024) void dt_min_kernel(const double *dtElem, int n, double *scal)
{
  __shared__ double red[16];
  double m = 1e10;
  for (int i = threadIdx.x; i < n; i += 1024) m = fmin(m, dtElem[i]);
  m = -wave_max(-m);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double r = red[0];
    for (int w = 1; w < 16; ++w) r = fmin(r, red[w]);
    scal[0] = r;
  }
}

// Per case of a batch group (one workgroup each): the minimum of the
// per-element time steps as dt_min_kernel forms it, then the step control of
// SolverClass::ExecuteTimeSynchronizationStep (SolverClass.cpp:2356-2365):
// the step that reaches 0.99 of the synchronization time step is clipped to
// end it exactly, and the next step starts a new one. A case with error flags
// or no RK steps left is deactivated, so the batch's launches skip it.
__global__ __launch_bounds__(1024) void batch_sync_kernel(const CaseDev *cases)
{
  __shared__ double red[16];
  const CaseDev c = cases[blockIdx.x];
  if (c.flags[kWordActive] == 0) return;
  double m = 1e10;
  for (int i = threadIdx.x; i < c.nElem; i += 1024) m = fmin(m, c.dtElem[i]);
  m = -wave_max(-m);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double r = red[0];
    for (int w = 1; w < 16; ++w) r = fmin(r, red[w]);
    if (c.flags[kWordFlags] != 0 || c.flags[kWordStepsLeft] <= 0) {
      c.flags[kWordActive] = 0;
      return;
    }
    c.scal[0] = r;
    double dt = r;
    const double el = c.scal[kScalElapsed], dtSync = c.scal[kScalDtSync];
    if (el + dt >= 0.99 * dtSync) {
      dt = dtSync - el;
      c.scal[kScalElapsed] = 0.0;
      c.scal[kScalSyncDone] += 1.0;
    } else {
      c.scal[kScalElapsed] = el + dt;
    }
    c.scal[kScalDt] = dt;
    c.flags[kWordStepsLeft] -= 1;
    c.flags[kWordStepsDone] += 1;
  }
}

// First RK stage of a batch: U0 <- U and U <- U - dt R per element, with the
// case's time step (the same values stage0_kernel forms after its buffer swap).
__global__ __launch_bounds__(256) void stage0_batch_kernel(const CaseDev *cases, const WorkItem *work, int nd5)
{
  const WorkItem w = work[blockIdx.x];
  const CaseDev c = cases[w.c];
  if (c.flags[kWordActive] == 0) return;
  const double dt = c.scal[kScalDt];
  const size_t base = (size_t) w.e * nd5;
  for (int i = threadIdx.x; i < nd5; i += 256) {
    const double u = c.U[base + i];
    c.U0[base + i] = u;
    c.U[base + i] = u - dt * c.R[base + i];
  }
}

// Status words of the cases of a batch group, gathered for one readback. A
// case counts as active while the next RK step of the batch would advance it
// (its own word is cleared only by that step's batch_sync_kernel).
__global__ __launch_bounds__(64) void batch_status_kernel(const CaseDev *cases, int n, int *out)
{
  const int i = blockIdx.x * 64 + threadIdx.x;
  if (i >= n) return;
  const CaseDev c = cases[i];
  out[i * kStatusWords + 0] =
      c.flags[kWordActive] != 0 && c.flags[kWordFlags] == 0 && c.flags[kWordStepsLeft] > 0 ? 1 : 0;
  out[i * kStatusWords + 1] = c.flags[kWordStepsDone];
  out[i * kStatusWords + 2] = c.flags[kWordStepsLeft];
  out[i * kStatusWords + 3] = c.flags[kWordFlags];
  out[i * kStatusWords + 4] = (int) c.scal[kScalSyncDone];
}

// Maximum of n non-negative values into *out (one workgroup).
__global__ __launch_bounds__(1024) void reduce_max_kernel(const double *v, int n, double *out)
{
  __shared__ double red[16];
  double m = 0.0;
  for (int i = threadIdx.x; i < n; i += 1024) m = fmax(m, v[i]);
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double r = red[0];
    for (int w = 1; w < 16; ++w) r = fmax(r, red[w]);
    *out = r;
  }
}

// Sums of the six wall-force components over the n boundary faces into
// out[0..6), in face order (one wave, each lane a fixed stride of faces, then
// the lanes in order).
__global__ __launch_bounds__(64) void force_sum_kernel(const double *part, int n, double *out)
{
  __shared__ double red[64][6];
  double s[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  for (int b = threadIdx.x; b < n; b += 64)
#pragma unroll
    for (int i = 0; i < 6; ++i) s[i] += part[(size_t) b * 6 + i];
#pragma unroll
  for (int i = 0; i < 6; ++i) red[threadIdx.x][i] = s[i];
  __syncthreads();
  if (threadIdx.x < 6) {
    double t = 0.0;
    for (int l = 0; l < 64; ++l) t += red[l][threadIdx.x];
    out[threadIdx.x] = t;
  }
}

// First RK stage: U <- U0 - dt R, where U0 already holds the state of the
// step (the host swaps the two buffers instead of copying). dt is the
// argument, which the first lane also stores to dtOut for the later stages,
// or (dtIn non-null) is read from device memory where the host put it.
__global__ void stage0_kernel(double *U, const double *U0, const double *R, size_t n, double dtArg,
                              const double *dtIn, double *dtOut)
{
  const double dt = dtIn ? *dtIn : dtArg;
  if (dtOut && blockIdx.x == 0 && threadIdx.x == 0) *dtOut = dt;
  for (size_t i = blockIdx.x * (size_t) blockDim.x + threadIdx.x; i < n; i += (size_t) gridDim.x * blockDim.x)
    U[i] = U0[i] - dt * R[i];
}

// p[0, n) = v (a kernel, so that it can be captured in a graph).
__global__ void fill_kernel(double *p, size_t n, double v)
{
  for (size_t i = blockIdx.x * (size_t) blockDim.x + threadIdx.x; i < n; i += (size_t) gridDim.x * blockDim.x)
    p[i] = v;
}

// The time step of the RK step about to run, into device memory (one lane,
// a vector store).
__global__ __launch_bounds__(64) void publish_kernel(const double *scal, const int *flags, double *host, int n,
                                                     int flagsAt)
{
  const int i = threadIdx.x;
  if (i < n) host[i] = scal[i];
  if (i == 0) *(int *) (host + flagsAt) = flags[kWordFlags];
}

__global__ __launch_bounds__(256) void store_kernel(double *dst, const double *src, size_t n)
{
  const size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

__global__ void set_dt_kernel(double *p, double v)
{
  if (threadIdx.x == 0) *p = v;
}

template <int K, int M>
hipError_t boundary_impl(const DeviceCase &dc, hipStream_t s, bool monitor)
{
  if (dc.nBFace == 0) return hipSuccess;
  BndArgs<K, M> a;
  a.U = dc.U; a.tables = dc.tables; a.econst = dc.econst; a.bgeo = dc.bgeo; a.bface = dc.bface;
  a.machPart = dc.machPart; a.faceRes = dc.faceRes; a.forcePart = dc.forcePart; a.to = dc.to;
  a.bug = dc.bug_compat; a.monitor = monitor && dc.monitor_forces;
  a.mu = dc.mu; a.tauFact = (dc.P + 1.0) * (dc.P + 1.0) * dc.rel_penalty; a.thetaHalf = 0.5 * dc.theta_sym;
  a.nb = dc.nscbc;
  a.sgs = dc.sgs; a.nElem = dc.nElem; a.eddyPart = dc.sgs ? dc.eddyPart : nullptr;
  hipLaunchKernelGGL((mach_kernel<K, M>), dim3(dc.nBFace), dim3(64), 0, s, a);
  hipLaunchKernelGGL((nscbc_kernel<K, M>), dim3(dc.nBFace), dim3(64), 0, s, a);
  if (a.monitor)
    hipLaunchKernelGGL(force_sum_kernel, dim3(1), dim3(64), 0, s, dc.forcePart, dc.nBFace, dc.scal + kScalForce);
  return hipGetLastError();
}

template <int K>
hipError_t dt_impl(const DeviceCase &dc, hipStream_t s)
{
  DtArgs a;
  a.c = case_dev(dc); a.to = dc.to; a.P = dc.P;
  if (dc.sgs)
    hipLaunchKernelGGL((time_step_kernel<K, true>), dim3(dc.nElem), dim3(64), 0, s, a);
  else
    hipLaunchKernelGGL((time_step_kernel<K, false>), dim3(dc.nElem), dim3(64), 0, s, a);
  hipLaunchKernelGGL(dt_min_kernel, dim3(1), dim3(1024), 0, s, dc.dtElem, dc.nElem, dc.scal);
  return hipGetLastError();
}

template <int K>
hipError_t batch_dt_impl(const BatchGroup &g, hipStream_t s)
{
  DtBatchArgs b;
  b.cases = g.cases; b.work = g.work; b.to = g.proto->to; b.P = g.proto->P;
  if (g.proto->sgs)
    hipLaunchKernelGGL((time_step_batch_kernel<K, true>), dim3(g.nWork), dim3(64), 0, s, b);
  else
    hipLaunchKernelGGL((time_step_batch_kernel<K, false>), dim3(g.nWork), dim3(64), 0, s, b);
  hipLaunchKernelGGL(batch_sync_kernel, dim3(g.nCase), dim3(1024), 0, s, g.cases);
  return hipGetLastError();
}

}  // namespace

CaseDev case_dev(const DeviceCase &dc)
{
  CaseDev c{};
  c.U = dc.U; c.U0 = dc.U0; c.R = dc.R; c.faceRes = dc.faceRes;
  c.tables = dc.tables; c.vgeo = dc.vgeo; c.fgeo = dc.fgeo; c.econst = dc.econst; c.nbr = dc.nbr;
  c.scal = dc.scal; c.flags = dc.flags; c.cgIter = dc.cgIter; c.dtElem = dc.dtElem;
  c.mach2Elem = dc.mach2Elem;
  c.spIdx = dc.nSponge ? dc.spIdx : nullptr; c.spCoef = dc.spCoef; c.dampFn = dc.dampFn;
  c.dampState = dc.dampState; c.srcBuf = dc.srcBuf;
  c.mu = dc.mu; c.tauFact = (dc.P + 1.0) * (dc.P + 1.0) * dc.rel_penalty; c.thetaHalf = 0.5 * dc.theta_sym;
  c.cfl = dc.cfl; c.u_ref = dc.u_ref; c.p_ref = dc.p_ref; c.rho_ref = dc.rho_ref;
  c.muDim = dc.mu * dc.p_ref / dc.u_ref;
  c.nElem = dc.nElem; c.cml = dc.cml;
  c.sgs = dc.sgs; c.vgeoN = dc.vgeoN; c.eddyPart = dc.sgs ? dc.eddyPart : nullptr;
  c.bfBuf = dc.fbodyOn ? dc.bfBuf : nullptr;
  for (int i = 0; i < 3; ++i) c.fbody[i] = dc.fbody[i];
  return c;
}

#define VCP_PAIRS(X) X(3, 4) X(4, 5) X(4, 6) X(5, 7) X(6, 8) X(7, 9)

bool supported_pair(int K, int M)
{
#define X(k, m) if (K == k && M == m) return true;
  VCP_PAIRS(X)
#undef X
  return false;
}

int volume_tiles(int K, int M, int out[4])
{
  int n = 0;
#define X(k, m, nt) if (K == k && M == m && n < 4) out[n++] = nt;
  VCP_COL_TILES(X)
  VCP_TILES(X)
#undef X
  return n;
}

int column_tile(int K, int M)
{
  int t[4];
  return volume_tiles(K, M, t) > 0 ? t[0] : 0;
}

// Without a given size, the column kernel where the case has enough elements
// to fill the chip with it: one wave per element (or several elements per
// wave) runs longer per element than a workgroup, which is ahead as long as the
// chip holds all workgroups at once (1280 or, in the float form, 1536 of them at
// (4, 5), 768 at (4, 6), (5, 7) and in the float form (6, 8), 256 or 512 at (7, 9)).
// Measured on one box, volume launch in us, workgroup / column kernel,
// Taylor-Green cases:
//   (4, 5) 512 elements 31.8 / 39.4, 1000: 38.6 / 43.5, 1331: 47.2 / 46.2, 1728: 63 / 52
//   float  1000: 24.4 / 32.4, 1331: 28.0 / 33.1, 1728: 40.2 / 34.5
//   (4, 6) 512: 36.0 / 40.7, 1000: 67 / 44;  float 512: 27.0 / 31.2, 1000: 36.2 / 33.7
//   (5, 7) 512: 42.3 / 58.3, 729: 51.5 / 61.0, 1000: 76 / 63, 1728: 99 / 74
//   float  729: 36.6 / 46.0, 1000: 55 / 48
//   (6, 8) 27: 76 / 68, 512: 84 / 70;  float 512: 46.4 / 62.1, 729: 56.9 / 64.6, 1000: 85 / 66
//   (7, 9) 216: 72 / 77, 343: 133 / 92;  float 512: 76 / 74, 729: 113 / 77
// (from (6, 8) on in FP64 a column has two threads). A case with boundaries
// (a pulse, a wall layer) is uneven: the solve of most elements stops early, and
// the launch lasts as long as its longest elements. The workgroup stays ahead up
// to two rounds of them, four in FP64 and three in float at the high degrees:
// open boxes with a pulse,
//   (4, 5) 1280: 52 / 66, 1944: 61 / 66, 2916: 67 / 68;  float 1280: 33 / 43, 2916: 46 / 47
//   (5, 7) 1152: 90 / 107, 1944: 102 / 100, 2916: 126 / 129, 5760: 211 / 192
//   float  1152: 60 / 68, 1944: 74 / 65;  (6, 8) float 1152: 90 / 103, 1944: 110 / 124, 2916: 153 / 144
//   (4, 6) 896: 69 / 62;  (7, 9) 384: 149 / 132
// At (3, 4) the column kernel is ahead at every size, up to 4096 elements with
// the columns in halves, when these still run all at once (workgroup / halves /
// whole: 64 elements 30.0 / 26.0 / 31.7, 1000: 32.3 / 25.4 / 29.9, 4096: 72 / 40 / 43,
// 5832: 85 / 57 / 49; float 64: 22.8 / 18.3 / 23.1, 4096: 38 / 29 / 32).
int volume_kind(const DeviceCase &dc, int nt)
{
  const bool full = dc.sgs != kSgsNone || dc.nSponge > 0 || dc.fbodyOn;
  const int cols = full ? kVolColsFull : kVolCols;
  if (nt) return nt == column_tile(dc.K, dc.M) ? cols : kVolWorkgroup;
  if (dc.K == 3) return dc.nElem > 4096 ? cols : full ? kVolHalvesFull : kVolHalves;
  // most elements for the workgroup kernel: [float][with boundaries]
  struct Most {
    int K, M, n[2][2];
  };
  static constexpr Most most[] = {{4, 5, {{1280, 2560}, {1536, 3072}}}, {4, 6, {{768, 768}, {768, 768}}},
                                  {5, 7, {{768, 3072}, {768, 1536}}},   {6, 8, {{0, 0}, {768, 2304}}},
                                  {7, 9, {{256, 256}, {512, 512}}}};
  for (const Most &m : most)
    if (m.K == dc.K && m.M == dc.M) return dc.nElem > m.n[dc.mixed != 0][dc.nBFace > 0] ? cols : kVolWorkgroup;
  return kVolWorkgroup;
}

namespace {
// the workgroup size of volume_kernel: the given one, or the first instantiated
int workgroup_tile(int K, int M, int nt)
{
  if (nt) return nt;
#define X(k, m, t) if (K == k && M == m && !nt) nt = t;
  VCP_TILES(X)
#undef X
  return nt;
}
}  // namespace

int volume_tile(int kind, int K, int M)
{
  if (kind == kVolWorkgroup) return workgroup_tile(K, M, 0);
  return kind == kVolCols || kind == kVolColsFull ? column_tile(K, M) : 0;
}

hipError_t launch_faces(const DeviceCase &dc, hipStream_t s)
{
  const bool wide = volume_kind(dc, dc.nt) != kVolWorkgroup;
#define X(k, m) if (dc.K == k && dc.M == m) return faces<k, m>(dc, wide, s);
  VCP_PAIRS(X)
#undef X
  return hipErrorInvalidValue;
}

hipError_t launch_boundary(const DeviceCase &dc, hipStream_t s, bool monitor)
{
#define X(k, m) if (dc.K == k && dc.M == m) return boundary_impl<k, m>(dc, s, monitor);
  VCP_PAIRS(X)
#undef X
  return hipErrorInvalidValue;
}

hipError_t launch_volume(const DeviceCase &dc, const StageCtl &ctl, hipStream_t s)
{
  const int kind = volume_kind(dc, dc.nt), nt = workgroup_tile(dc.K, dc.M, dc.nt);
  const hipError_t e = [&]() -> hipError_t {
#define X(k, m) if (kind != kVolWorkgroup && dc.K == k && dc.M == m) return volume_cols<k, m>(dc, kind, ctl, s);
    VCP_PAIRS(X)
#undef X
#define X(k, m) if (dc.K == k && dc.M == m) return volume_workgroup<k, m>(dc, nt, ctl, s);
    VCP_PAIRS(X)
#undef X
    return hipErrorInvalidValue;
  }();
  if (e == hipSuccess && ctl.monitor) {
    hipLaunchKernelGGL(reduce_max_kernel, dim3(1), dim3(1024), 0, s, dc.mach2Elem, dc.nElem, dc.scal + 1);
    // volume, internal-face and boundary-face maxima of the eddy viscosity
    if (dc.sgs)
      hipLaunchKernelGGL(reduce_max_kernel, dim3(1), dim3(1024), 0, s, dc.eddyPart, 4 * dc.nElem + dc.nBFace,
                         dc.scal + kScalEddy);
  }
  return e == hipSuccess ? hipGetLastError() : e;
}

hipError_t launch_time_step(const DeviceCase &dc, hipStream_t s)
{
  switch (dc.K) {
    case 3: return dt_impl<3>(dc, s);
    case 4: return dt_impl<4>(dc, s);
    case 5: return dt_impl<5>(dc, s);
    case 6: return dt_impl<6>(dc, s);
    case 7: return dt_impl<7>(dc, s);
  }
  return hipErrorInvalidValue;
}

template <int K>
hipError_t avg_impl(const DeviceCase &dc, double factNew, hipStream_t s)
{
  AvgArgs a;
  a.c = case_dev(dc); a.avg = dc.avg; a.to = dc.to;
  a.factNew = factNew; a.factOld = 1.0 - factNew;
  if (dc.sgs)
    hipLaunchKernelGGL((average_kernel<K, true>), dim3(dc.nElem), dim3(64), 0, s, a);
  else
    hipLaunchKernelGGL((average_kernel<K, false>), dim3(dc.nElem), dim3(64), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_average(const DeviceCase &dc, double factNew, hipStream_t s)
{
  switch (dc.K) {
    case 3: return avg_impl<3>(dc, factNew, s);
    case 4: return avg_impl<4>(dc, factNew, s);
    case 5: return avg_impl<5>(dc, factNew, s);
    case 6: return avg_impl<6>(dc, factNew, s);
    case 7: return avg_impl<7>(dc, factNew, s);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_damping_from_averages(const DeviceCase &dc, hipStream_t s)
{
  if (!dc.avg || !dc.nSponge) return hipErrorInvalidValue;
  DampAvgArgs a;
  a.avg = dc.avg; a.tables = dc.tables; a.spIdx = dc.spIdx; a.dampState = dc.dampState; a.to = dc.to;
  a.u_ref = dc.u_ref; a.p_ref = dc.p_ref; a.rho_ref = dc.rho_ref; a.nAvg = dc.nAvg;
#define X(k, m)                                                                                    \
  if (dc.K == k && dc.M == m) {                                                                    \
    hipLaunchKernelGGL((damping_avg_kernel<k, m>), dim3(dc.nElem), dim3(64), 0, s, a);             \
    return hipGetLastError();                                                                      \
  }
  VCP_PAIRS(X)
#undef X
  return hipErrorInvalidValue;
}

hipError_t launch_fill(double *p, size_t n, double v, hipStream_t s)
{
  if (n == 0) return hipSuccess;
  const int blocks = (int) ((n + 255) / 256 < 4096 ? (n + 255) / 256 : 4096);
  hipLaunchKernelGGL(fill_kernel, dim3(blocks), dim3(256), 0, s, p, n, v);
  return hipGetLastError();
}

hipError_t static_scratch(void **ptr, size_t *bytes)
{
  // one address per device, looked up once with that device current
  static std::mutex mu;
  static void *addr[kMaxDevices] = {};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[dev]) {
    void *a = nullptr;
    e = hipGetSymbolAddress(&a, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    addr[dev] = a;
  }
  *ptr = addr[dev];
  *bytes = sizeof(scratch);
  return hipSuccess;
}

hipError_t launch_publish(const DeviceCase &dc, double *host, int n, int flagsAt, hipStream_t s)
{
  if (n > 64) return hipErrorInvalidValue;
  hipLaunchKernelGGL(publish_kernel, dim3(1), dim3(64), 0, s, dc.scal, dc.flags, host, n, flagsAt);
  return hipGetLastError();
}

hipError_t launch_store(double *dst, const double *src, size_t n, hipStream_t s)
{
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(store_kernel, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, s, dst, src, n);
  return hipGetLastError();
}

hipError_t launch_set_dt(const DeviceCase &dc, double dt, hipStream_t s)
{
  hipLaunchKernelGGL(set_dt_kernel, dim3(1), dim3(64), 0, s, dc.scal + kScalDt, dt);
  return hipGetLastError();
}

hipError_t launch_stage0(const DeviceCase &dc, const double *dt, hipStream_t s)
{
  const size_t n = (size_t) dc.nElem * 5 * dc.nDOF;
  const int blocks = (int) ((n + 255) / 256 < 65536 ? (n + 255) / 256 : 65536);
  hipLaunchKernelGGL(stage0_kernel, dim3(blocks), dim3(256), 0, s, dc.U, dc.U0, dc.R, n,
                     dt ? *dt : 0.0, dt ? nullptr : dc.scal + kScalDt, dt ? dc.scal + kScalDt : nullptr);
  return hipGetLastError();
}

hipError_t launch_batch_faces(const BatchGroup &g, int kind, int w0, int nw, hipStream_t s)
{
  if (nw <= 0) return hipSuccess;
  const DeviceCase &p = *g.proto;
#define X(k, m) if (p.K == k && p.M == m) return batch_faces<k, m>(g, kind != kVolWorkgroup, w0, nw, s);
  VCP_PAIRS(X)
#undef X
  return hipErrorInvalidValue;
}

hipError_t launch_batch_volume(const BatchGroup &g, int kind, const StageCtl &ctl, int w0, int nw, hipStream_t s)
{
  if (nw <= 0) return hipSuccess;
  const DeviceCase &p = *g.proto;
  const int nt = workgroup_tile(p.K, p.M, g.nt);
#define X(k, m)                                                                                     \
  if (kind != kVolWorkgroup && p.K == k && p.M == m)                                                \
    return batch_volume_cols<k, m>(g, kind, ctl, w0, nw, s);
  VCP_PAIRS(X)
#undef X
#define X(k, m) if (p.K == k && p.M == m) return batch_volume_workgroup<k, m>(g, nt, ctl, w0, nw, s);
  VCP_PAIRS(X)
#undef X
  return hipErrorInvalidValue;
}

hipError_t launch_batch_time_step(const BatchGroup &g, hipStream_t s)
{
  if (g.nWork <= 0) return hipSuccess;
  switch (g.proto->K) {
    case 3: return batch_dt_impl<3>(g, s);
    case 4: return batch_dt_impl<4>(g, s);
    case 5: return batch_dt_impl<5>(g, s);
    case 6: return batch_dt_impl<6>(g, s);
    case 7: return batch_dt_impl<7>(g, s);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_batch_status(const BatchGroup &g, int *out, hipStream_t s)
{
  if (g.nCase <= 0) return hipSuccess;
  hipLaunchKernelGGL(batch_status_kernel, dim3((g.nCase + 63) / 64), dim3(64), 0, s, g.cases, g.nCase, out);
  return hipGetLastError();
}

hipError_t launch_batch_stage0(const BatchGroup &g, hipStream_t s)
{
  if (g.nWork <= 0) return hipSuccess;
  hipLaunchKernelGGL(stage0_batch_kernel, dim3(g.nWork), dim3(256), 0, s, g.cases, g.work,
                     5 * g.proto->nDOF);
  return hipGetLastError();
}

}  // namespace vcp
