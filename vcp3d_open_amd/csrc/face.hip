// Interior (and periodic) face residuals (gfx950). Compiled once per shape
// (VCP_SHAPE_K, VCP_SHAPE_M).
//
// Reference behaviour followed (VCP3D_CurviLinear/src/):
//   ElementClass::{I,J,K}FaceResiduals    ElementClass.cpp:2582-3400
//   FluxesInternalFace / InviscidFluxesFace / ViscousFluxesFace /
//   PenAndSymFluxesSymmVar                FluxesFace.cpp:220-343, :813-975,
//                                         :1290-1651, :1152-1284
#include "device.hpp"
#include "kernels.hpp"
#include "transforms.hpp"

namespace vcp {
namespace {

template <int K, int M, typename T = double>
struct FaceOps {
  EvenOdd<K, M, T> a;          // phi_q(r_p) and phi'_q(r_p), even-odd form
  EvenOddD<K, M, T> d;
  EvenOdd<K, M, double> ad;    // phi_q(r_p) for the wide lift of the float form
  T A[M * K], D[M * K];        // the same, row-major (p, q)
  T F[4][K];                   // phi(-1), phi(+1), phi'(-1), phi'(+1)
  double w[M];                 // 1D Gauss weights
  double c03;                  // phi_0^3, the value of the constant mode
};

// Face kernel arguments: the case part (single-case launch) or the case
// table and work items (batched launch), and the operators (the
// metric-indexing mode is the kernel's BUG parameter).
template <int K, int M, typename T = double>
struct FaceArgs {
  CaseDev c;
  const CaseDev *cases;
  const WorkItem *work;
  int w0, n;                   // first work item (batch), number of elements
  FaceOps<K, M, T> op;
};

// ============================================================ face kernel
// Faces in direction DIR: each lane group of a wave (the wave, or 32 or 16
// lanes where the M^2 points fill only that many; two waves at M = 9) takes
// one element's min face. Side 0 is the element itself (its min face), side 1 the neighbour L
// (its max face); the normal points from L to the element. Every phase reads
// all of its lines before it stores over them. LDS regions:
//   X: normal contraction B -> fast contraction T -> flux and Cartesian
//      symmetrising fluxes at the points
//   Y: the first lift stage of one side: flux + fast slot of five variables,
//      slow slot and normal slot of variables 1..4
//
// What bounds it: instruction issue and latency at three waves per SIMD (LDS),
// not memory. The line contractions use the even-odd operators, the lift
// fills the wave (9 M lines per side), the pointwise fluxes take five
// reciprocals and roots instead of twenty divisions and square roots, and two
// or four faces share a wave at M = 5 and 4: 1570 vector instructions per
// face instead of 2070 at (5, 7). Measured on one box, launch over the three
// directions of a Taylor-Green case, with dense lines and one face per wave /
// as it is, us: (3, 4) 18^3 68 / 38, (4, 5) 16^3 65 / 44, (4, 6) 14^3 51 / 42,
// (5, 7) 32^3 577 / 473, (6, 8) 16^3 187 / 103, (7, 9) 14^3 226 / 125; float
// form, with the flux lifted in float / in double: (3, 4) 36 / 36, (4, 5) 36 / 35,
// (4, 6) 39 / 40, (5, 7) 385 / 401, (6, 8) 74 / 86, (7, 9) 107 / 116. The odd
// pitches and, at M = 9, the two waves per face are a fifth of it at (6, 8) and a third
// at (7, 9) (130 / 106 at 16^3, 98 / 68 at 11^3).
template <int K, int M, typename T, typename TL>
struct FaceSmem {
  // faces per wave and lanes per face: the pointwise fluxes are half of the
  // instructions, and the M^2 points of one face leave most of a wave idle at
  // M = 4 and 5 ((3, 4) 18^3: 57 us with one face per wave, 43 with four)
  static constexpr int NF = M * M <= 16 ? 4 : M * M <= 32 ? 2 : 1;
  // threads of the workgroup, and per face: the 81 points of M = 9 take two
  // waves. (In one wave they take two passes, the second with 17 lanes, and the
  // fast contraction's output a region of its own, which leaves four waves per
  // CU: launch over 3457 elements 240 us, in two waves 155.)
  static constexpr int NT = M * M > 64 ? 128 : 64, G = NT / NF;
  static_assert(M * M <= G, "the points of a face in one pass");
  // traces: the value of five variables, the fast and normal derivatives of
  // variables 1..4 (the fluxes need no gradient of the first); points: the
  // flux of five variables, the symmetrising fluxes of 1..4 (the first's are
  // 0). Lines of K and M values at odd pitches: lanes that take neighbouring
  // lines fall into different banks (at (6, 8) more than half of the LDS cycles
  // were conflicts, and the LDS 80 % busy)
  static constexpr int KP = K | 1, MP = M | 1, NP = M * MP;
  // in units of T; the flux and its first lift stage in TL
  static constexpr int W = (int) (sizeof(TL) / sizeof(T));
  static constexpr int kB = 2 * 2 * 5 * K * KP, kT1 = 13 * K * MP, kT = 2 * kT1, kP = (5 * W + 12) * NP;
  static constexpr int kY = (5 * W + 8) * M * KP;
  // Y behind the fluxes, over T's end, where that lets one more face into a
  // CU's LDS and the face is large ((6, 8) 16^3: 110 us, 114 in a region of its
  // own); at (5, 7) the thirteenth face makes the launch slower (32^3: 554
  // against 542 us)
  static constexpr int kOffY = M > 7 ? kP : (cmax(cmax(kB, kT), kP) + W - 1) / W * W;
  static constexpr int kX = cmax(cmax(kB, kT), kOffY + kY);
  static constexpr int kBytes = (int) sizeof(T) * (2 * M * K + 4 * K + NF * kX) + 8 * (M * M + 1 + NF * 82);
  // waves per SIMD to compile for: three when 12 waves fit a CU's 160 KB
  static constexpr int kWaves = 12 * 64 / NT * kBytes <= 160 * 1024 ? 3 : 2;
  T A[M * K], D[M * K];
  double W2[M * M];
  T F[4][K];                       // phi(-1), phi(+1), phi'(-1), phi'(+1)
  double EvMax;                    // the second wave's eddy-viscosity maximum (two waves per face)
  struct Face {
    double Cm[2][4][9];            // metric of points 1..4 (bug)
    double Mean[2][5];             // float form: mode 0 of both elements
    alignas(8) T X[kX];
  } f[NF];
};

// args: the kernel's argument block, read in place from the kernel-argument
// segment by both forms, so that run-time-indexed operator rows come through
// scalar loads and the single-case and batched kernels do the same
// arithmetic. T: the type of the contractions (double, or float for the
// mixed-precision form, where the traces carry the variation about each
// element's mean, added back at the points in double, and the pointwise
// fluxes stay in double). TL: the type in which the flux is lifted: T, or
// double in the float form beside the column volume kernel, whose planes are in
// double too. A residual is the difference of large interior and face terms,
// and the flux and the operator rounded to float in one of them only leave a
// pattern of their own in every element: after 20 steps of a 16^3 (5, 7) case
// the density is off from the FP64 form's by 2.2e-8 with both in float, 6.0e-8
// with the planes alone in double, 2.2e-9 with both (launch over the faces
// 382 / 401 us at 32^3). SGS: the case has a subgrid scale model (a
// separate instantiation: its eddy-viscosity code raises the register peak).
template <int K, int M, int DIR, bool BUG, bool BATCH, typename T, typename TL, bool SGS>
__device__ __forceinline__ void face_body(const FaceArgs<K, M, T> &args, const CaseDev a, FaceSmem<K, M, T, TL> &sm,
                                          int e, bool live)
{
#define VCP_FOPS (args.op)
  constexpr bool kMixed = sizeof(T) == 4;
  // the element below; a physical boundary face is left to the boundary kernels
  int L = a.nbr[e * 6 + 2 * DIR];
  live = live && L >= 0;
  if (!__any(live)) return;
  if (L < 0) L = e;
  constexpr int ND = K * K * K, N2 = M * M;
  using S = FaceSmem<K, M, T, TL>;
  constexpr bool kWide = sizeof(TL) > sizeof(T);
  constexpr int G = S::G, NT = S::NT, KP = S::KP, MP = S::MP, NP = S::NP;
  constexpr int SB = 5 * K * KP;              // one plane of B
  // strides of the (normal, fast, slow) axes in the [k][j][i] DOF layout
  constexpr int SN = DIR == 0 ? 1 : DIR == 1 ? K : K * K;
  constexpr int SFA = DIR == 0 ? K : 1;
  constexpr int SSL = DIR == 2 ? K : K * K;
  // parametric slot of each axis: r = 0, s = 1, t = 2 -> (normal, fast, slow)
  constexpr int PN = DIR, PF = DIR == 0 ? 1 : 0, PS = DIR == 2 ? 1 : 2;
  T *sA = sm.A, *sD = sm.D;
  double *sW2 = sm.W2;
  const int lane = threadIdx.x, tid = lane % G;   // thread of the workgroup, of the face
  typename S::Face &sf = sm.f[lane / G];
  T *B = sf.X;                                // [side][value|deriv][5][K][KP]
  T *Tb = sf.X;                               // [side][A|D|N][5, 4, 4][K][MP]
  TL *sFlux = (TL *) sf.X;                    // flux [5][M][MP]
  T *sFC = sf.X + 5 * S::W * NP;              // Cartesian sym [x|y|z][4][M][MP] of variables 1..4
  // operators in LDS: read as wave-uniform LDS operands in the contractions
  // (as kernel arguments they would not fit the scalar registers)
  for (int i = lane; i < M * K; i += NT) { sA[i] = VCP_FOPS.A[i]; sD[i] = VCP_FOPS.D[i]; }
  for (int i = lane; i < 4 * K; i += NT) sm.F[i / K][i % K] = VCP_FOPS.F[i / K][i % K];
  // operators of the line contractions, through scalar loads
  auto ops = [&]() { auto p = (cptr<FaceOps<K, M, T>>) (uintptr_t) &args.op; asm volatile("" : "+s"(p)); return p; };
  for (int i = lane; i < N2; i += NT) sW2[i] = VCP_FOPS.w[i % M] * VCP_FOPS.w[i / M];
  const double *g = a.fgeo + ((size_t) e * 3 + DIR) * kFaceGeo * N2;
  // Loads issued here and used after the contractions, so that their latency
  // passes under them: the two length scales and this lane's point
  // metric (normal, area and, unless the metric comes from sm.Cm, both sides'
  // inverse metric).
  const double lenE = a.econst[(size_t) e * kElemConst + DIR], lenL = a.econst[(size_t) L * kElemConst + DIR];
  const bool atPoint = tid < N2;
  const int m = atPoint ? tid : 0;
  double geoCm[2][9], geoN[4];
  if constexpr (!BUG)
#pragma unroll
    for (int q = 0; q < 9; ++q) { geoCm[0][q] = g[(13 + q) * N2 + m]; geoCm[1][q] = g[(4 + q) * N2 + m]; }
#pragma unroll
  for (int q = 0; q < 4; ++q) geoN[q] = g[q * N2 + m];
  if constexpr (BUG)
#pragma unroll
    for (int it = 0; it < (72 + G - 1) / G; ++it) {
      const int i = tid + G * it;
      if (i < 72) {
        const int side = i / 36, l = (i / 9) % 4, q = i % 9;
        sf.Cm[side][l][q] = g[(side ? 4 + q : 13 + q) * N2 + 1 + l];
      }
    }
  if constexpr (kMixed)
    if (tid < 10) sf.Mean[tid / 5][tid % 5] = a.U[(size_t) (tid < 5 ? e : L) * 5 * ND + (tid % 5) * ND];
  group_sync<NT>();
  // normal contraction straight from HBM: B[side][0|1][v][s][f]; the loads of
  // both sides (K <= 6, at most 40 registers) or of one side at a time (K = 7)
  // are issued before the first of them is waited for. In the float form the
  // mean (mode 0) is added at the points.
  constexpr int NIT = (5 * K * K + G - 1) / G;
  constexpr int NS = 2 * NIT * K <= 40 ? 2 : 1;
#pragma unroll
  for (int s0 = 0; s0 < 2; s0 += NS) {
    double xu[NS][NIT][K];
#pragma unroll
    for (int sb = 0; sb < NS; ++sb) {
      const double *Us = a.U + (size_t) (s0 + sb ? L : e) * 5 * ND;
#pragma unroll
      for (int it = 0; it < NIT; ++it) {
        const int pc0 = tid + G * it, pc = pc0 < 5 * K * K ? pc0 : 0;
        const int v = pc / (K * K), sl = (pc / K) % K, f = pc % K;
        const double *u = Us + v * ND + sl * SSL + f * SFA;
#pragma unroll
        for (int t = 0; t < K; ++t) xu[sb][it][t] = u[t * SN];
      }
    }
#pragma unroll
    for (int sb = 0; sb < NS; ++sb) {
      const int side = s0 + sb;
      const T *Fv = sm.F[side], *dFv = sm.F[2 + side];
#pragma unroll
      for (int it = 0; it < NIT; ++it) {
        const int pc = tid + G * it;
        if (pc < 5 * K * K) {
          const int sl = (pc / K) % K, f = pc % K;
          T b0 = 0, b1 = 0;
#pragma unroll
          for (int t = 0; t < K; ++t) {
            const T x = (kMixed && t == 0 && sl == 0 && f == 0) ? T(0) : T(xu[sb][it][t]);
            b0 += Fv[t] * x; b1 += dFv[t] * x;
          }
          B[(side * 2 + 0) * SB + (pc / K) * KP + f] = b0;
          B[(side * 2 + 1) * SB + (pc / K) * KP + f] = b1;
        }
      }
    }
  }
  group_sync<NT>();
  // fast tangential contraction, in place over B:
  // T[side][A|D|N][v][s][f'], f' < M
  constexpr int RF = (2 * 5 * K + G - 1) / G;
  T in[RF][2][K];
#pragma unroll
  for (int r = 0; r < RF; ++r) {
    const int c = tid + r * G;
    if (c < 2 * 5 * K) {
      const int side = c / (5 * K), vs = c - side * 5 * K;
#pragma unroll
      for (int f = 0; f < K; ++f) {
        in[r][0][f] = B[(side * 2 + 0) * SB + vs * KP + f];
        in[r][1][f] = B[(side * 2 + 1) * SB + vs * KP + f];
      }
    }
  }
  group_sync<NT>();
#pragma unroll
  for (int r = 0; r < RF; ++r) {
    T (&x)[2][K] = in[r];
    const int c = tid + r * G;
    if (c >= 2 * 5 * K) continue;
    const int side = c / (5 * K), vs = c - side * 5 * K;
    // [A: 5 variables][D: 4][N: 4][s][f'], D and N of variables 1..4
    T *Ts = Tb + side * S::kT1 + vs * MP;
    const auto op = ops();
    const EvenOdd<K, M, T> A = scalar_op<K, M, T>(&op->a);
    T tA[M], tD[M], tN[M];
    to_points(A, x[0], tA);
    to_points(A, x[1], tN);
    to_points(scalar_op<K, M, T>(&op->d), x[0], tD);
#pragma unroll
    for (int n = 0; n < M; ++n) Ts[n] = tA[n];
    if (vs >= K)
#pragma unroll
      for (int n = 0; n < M; ++n) { Ts[4 * K * MP + n] = tD[n]; Ts[8 * K * MP + n] = tN[n]; }
  }
  group_sync<NT>();
  // per point: traces, averaged Cartesian gradients of the entropy variables
  // and the fluxes (Ismail-Roe, viscous, penalty, symmetrising); the outputs
  // overwrite T once every wave has read it
  const double lenScale = fmin(lenE, lenL);
  const double tau = a.tauFact / lenScale;
  // LES length scale of the face: the mean of the two elements'
  // (ElementClass.cpp:2655)
  const double lenLES = SGS ? 0.5 * (a.econst[(size_t) e * kElemConst + kElemLenLES]
                                     + a.econst[(size_t) L * kElemConst + kElemLenLES]) : 0.0;
  double evMax = 0.0;
  const int sp = m / M, fp = m - sp * M;
  double Vs[2][5], gx[5], gy[5], gz[5];
  auto traces = [&]() {
    T ai[K], di[K];
#pragma unroll
    for (int sl = 0; sl < K; ++sl) { ai[sl] = sA[sp * K + sl]; di[sl] = sD[sp * K + sl]; }
#pragma unroll
    for (int v = 0; v < 5; ++v) { gx[v] = 0.0; gy[v] = 0.0; gz[v] = 0.0; }
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      double cm[9];
      if constexpr (!BUG) {
#pragma unroll
        for (int q = 0; q < 9; ++q) cm[q] = geoCm[side][q];
      }
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        const T *tA = Tb + side * S::kT1 + v * K * MP + fp;
        const T *tD = tA + 4 * K * MP, *tN = tA + 8 * K * MP;
        T val = 0, gN = 0, gF = 0, gS = 0;
#pragma unroll
        for (int sl = 0; sl < K; ++sl) {
          const T xa = tA[sl * MP];
          val += ai[sl] * xa;
          if (v > 0) { gS += di[sl] * xa; gN += ai[sl] * tN[sl * MP]; gF += ai[sl] * tD[sl * MP]; }
        }
        Vs[side][v] = kMixed ? double(val) + VCP_FOPS.c03 * sf.Mean[side][v] : double(val);
        if (v == 0) continue;
        const double gr = DIR == 0 ? gN : gF;
        const double gs = DIR == 0 ? gF : DIR == 1 ? gN : gS;
        const double gt = DIR == 2 ? gN : gS;
        const double *c = cm;
        if constexpr (BUG) c = sf.Cm[side][v - 1];
        gx[v] += 0.5 * (gr * c[0] + gs * c[3] + gt * c[6]);
        gy[v] += 0.5 * (gr * c[1] + gs * c[4] + gt * c[7]);
        gz[v] += 0.5 * (gr * c[2] + gs * c[5] + gt * c[8]);
      }
    }
    // materialise the traces and gradients here: otherwise the compiler sinks
    // their computation into the flux and keeps the LDS operands live
#pragma unroll
    for (int v = 0; v < 5; ++v) asm volatile("" : "+v"(Vs[0][v]), "+v"(Vs[1][v]));
#pragma unroll
    for (int v = 1; v < 5; ++v) asm volatile("" : "+v"(gx[v]), "+v"(gy[v]), "+v"(gz[v]));
  };
  auto fluxes = [&]() {
    const double nn[3] = {geoN[0], geoN[1], geoN[2]};
    const double wA = sW2[m] * geoN[3];
    double fl[5], FX[5], FY[5], FZ[5], ev = 0.0;
    if constexpr (SGS) {
      ev = face_eddy(a.sgs, lenLES, Vs[1], Vs[0], gx, gy, gz);
      evMax = fmax(evMax, ev);
    }
    point_flux(Vs[1], Vs[0], gx, gy, gz, nn, wA, tau, a.mu, a.thetaHalf, fl, FX, FY, FZ, 1.0, false, 0.0, nullptr,
               SGS, ev);
    const int mp = sp * MP + fp;
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      sFlux[v * NP + mp] = TL(fl[v]);
      if (v > 0) {
        sFC[(v - 1) * NP + mp] = T(FX[v]); sFC[(3 + v) * NP + mp] = T(FY[v]); sFC[(7 + v) * NP + mp] = T(FZ[v]);
      }
    }
  };
  if constexpr (NT > 64) {
    if (atPoint) traces();
    group_sync<NT>();
    if (atPoint) fluxes();
  } else if (atPoint) {
    traces();
    fluxes();
  }
  if (SGS && a.eddyPart) {
    // the face's eddy-viscosity maximum for the monitoring data
    // (FluxesFace.cpp:336-342)
    evMax = lanes_reduce<G, true>(evMax);
    if constexpr (NT > 64) {
      if (tid == 64) sm.EvMax = evMax;
      group_sync<NT>();
      evMax = fmax(evMax, sm.EvMax);
    }
    if (tid == 0 && live) a.eddyPart[a.nElem + 3 * e + DIR] = evMax;
  }
  group_sync<NT>();
  // ---- lift, one side at a time. Fast-axis lines into Y: the flux (with A)
  // plus the fast slot (with D) of five variables, and the slow and the normal
  // slot (with A) of variables 1..4; with one face per workgroup and 9 M <= G
  // both kinds of lines share a pass. Then the slow axis, straight into the face
  // slot of that side: the value plane (A of the first, D of the slow slot)
  // and the normal-derivative plane (A of the normal slot) [0|1][v][slow]
  // [fast]; the volume kernel applies the face vectors.
  // A of the wide lift stays in scalar registers over both sides from K = 4 on
  // (32^3 (5, 7): 415 us, 432 with it loaded in each stage; at (3, 4) 36.5 / 36.1)
  constexpr bool kKeep = kWide && K >= 4;
  EvenOdd<K, M, TL> AL;
  if constexpr (kKeep) AL = scalar_op<K, M, TL>(&ops()->ad);
  auto wide_modes = [&](auto op, const TL (&x)[M], TL (&u)[K]) {
    if constexpr (kKeep) to_modes(AL, x, u);
    else to_modes(scalar_op<K, M, TL>(&op->ad), x, u);
  };
  // u += the derivative operator's transpose on x
  auto add_derivs = [&](auto op, const T (&x)[M], TL (&u)[K]) {
    T z[K];
#pragma unroll
    for (int n = 0; n < K; ++n) z[n] = 0;
    add_modes(scalar_op<K, M, T>(&op->d), x, z);
#pragma unroll
    for (int n = 0; n < K; ++n) u[n] += TL(z[n]);
  };
  // a symmetrising slot alone, in T
  auto slot_modes = [&](const EvenOdd<K, M, T> &A, const TL (&x)[M], TL (&u)[K]) {
    T y[M], z[K];
#pragma unroll
    for (int p = 0; p < M; ++p) y[p] = T(x[p]);
    to_modes(A, y, z);
#pragma unroll
    for (int n = 0; n < K; ++n) u[n] = TL(z[n]);
  };
  constexpr bool kShare = S::NF == 1 && 9 * M <= G;
  static_assert(4 * K <= G || S::NF == 1, "the derivative plane's lines in one pass");
#pragma unroll
  for (int side = 0; side < 2; ++side) {
    const TL sign = side ? TL(1) : TL(-1);
    double *out = a.faceRes + ((size_t) (side ? L : e) * 6 + 2 * DIR + side) * 10 * K * K;
    TL *Y0 = (TL *) (sf.X + S::kOffY);
    T *YS = sf.X + S::kOffY + 5 * S::W * M * KP, *YN = YS + 4 * M * KP;
    // Cartesian symmetrising flux mapped to this side's parametric slot P
    auto coef = [&](int v, int m, int P, int x) {
      return BUG ? sf.Cm[side][v][3 * P + x] : g[(side ? 4 + 3 * P + x : 13 + 3 * P + x) * N2 + m];
    };
    // lines [0, 5 M): flux and fast slot; [5 M, 9 M): slow and normal slot
    auto lines = [&](int item, bool first, bool second, bool isSecond) {
      const int idx = isSecond ? item - 5 * M : item;
      const int v = isSecond ? 1 + idx / M : idx / M, sp = idx % M;
      const int vc = v > 0 ? v - 1 : 0, P0 = isSecond ? PN : PF;
      double cb[3], ca[3];
      if constexpr (BUG)
#pragma unroll
        for (int x = 0; x < 3; ++x) { cb[x] = coef(vc, 0, P0, x); ca[x] = coef(vc, 0, PS, x); }
      TL xa[M];
      T xb[M];
#pragma unroll
      for (int q = 0; q < M; ++q) {
        const int m = sp * M + q, mp = sp * MP + q;
        const double fx = sFC[vc * NP + mp], fy = sFC[(4 + vc) * NP + mp], fz = sFC[(8 + vc) * NP + mp];
        if constexpr (!BUG)
#pragma unroll
          for (int x = 0; x < 3; ++x) { cb[x] = coef(vc, m, P0, x); ca[x] = coef(vc, m, PS, x); }
        xb[q] = !isSecond && v == 0 ? T(0) : T(fx * cb[0] + fy * cb[1] + fz * cb[2]);
        if (!second) xa[q] = sign * sFlux[v * NP + mp];
        else if (!first) xa[q] = TL(fx * ca[0] + fy * ca[1] + fz * ca[2]);
        else xa[q] = isSecond ? TL(fx * ca[0] + fy * ca[1] + fz * ca[2]) : sign * sFlux[v * NP + mp];
      }
      const auto op = ops();
      TL u[K], z[K];
      T w[K];
      if constexpr (kWide) {
        if (first) wide_modes(op, xa, u);
        if (second) {
          const EvenOdd<K, M, T> A = scalar_op<K, M, T>(&op->a);
          to_modes(A, xb, w);
          if (!first) slot_modes(A, xa, u);
        }
      } else {
        const EvenOdd<K, M, T> A = scalar_op<K, M, T>(&op->a);
        to_modes(A, xa, u);
        if (second) to_modes(A, xb, w);
      }
      if (first) {
#pragma unroll
        for (int n = 0; n < K; ++n) z[n] = u[n];
        if constexpr (kWide) add_derivs(op, xb, z);
        else add_modes(scalar_op<K, M, T>(&op->d), xb, z);
        if (!isSecond)
#pragma unroll
          for (int n = 0; n < K; ++n) Y0[idx * KP + n] = z[n];
      }
      if (second && isSecond)
#pragma unroll
        for (int n = 0; n < K; ++n) { YS[idx * KP + n] = T(u[n]); YN[idx * KP + n] = w[n]; }
    };
    if constexpr (kShare) {
      if (tid < 9 * M) lines(tid, true, true, tid >= 5 * M);
    } else {
#pragma unroll
      for (int r = 0; r < (5 * M + G - 1) / G; ++r)
        if (tid + r * G < 5 * M) lines(tid + r * G, true, false, false);
#pragma unroll
      for (int r = 0; r < (4 * M + G - 1) / G; ++r)
        if (tid + r * G < 4 * M) lines(5 * M + tid + r * G, false, true, true);
    }
    group_sync<NT>();
    // slow-axis lines [0, 5 K) of the value plane, [5 K, 9 K) of the derivative plane
    auto planes = [&](int item, bool first, bool deriv) {
      const int idx = deriv ? item - 5 * K : item, v = deriv ? 1 + idx / K : idx / K, f = idx % K;
      const TL *y0 = Y0 + v * M * KP + f;
      const T *yn = YN + (v - 1) * M * KP + f, *ya = deriv ? yn : (const T *) y0;
      const T *yb = YS + (v > 0 ? v - 1 : 0) * M * KP + f;
      const bool slow = !deriv && v > 0;
      TL xa[M], u[K];
      T xb[M];
#pragma unroll
      for (int q = 0; q < M; ++q) {
        if constexpr (kWide) xa[q] = deriv ? TL(yn[q * KP]) : y0[q * KP];
        else xa[q] = ya[q * KP];
        xb[q] = first && slow ? yb[q * KP] : T(0);
      }
      const auto op = ops();
      if constexpr (kWide) {
        if (first) {
          wide_modes(op, xa, u);
          add_derivs(op, xb, u);
        } else {
          slot_modes(scalar_op<K, M, T>(&op->a), xa, u);
        }
      } else {
        to_modes(scalar_op<K, M, T>(&op->a), xa, u);
        if (first) add_modes(scalar_op<K, M, T>(&op->d), xb, u);
      }
      if (!live) return;
      double *o = out + (deriv ? 5 * K * K : 0) + v * K * K + f;
#pragma unroll
      for (int n = 0; n < K; ++n) o[n * K] = double(u[n]);
      if (first && item < K)
#pragma unroll
        for (int n = 0; n < K; ++n) out[5 * K * K + n * K + f] = 0.0;
    };
    if constexpr (S::NF == 1) {
      static_assert(9 * K <= 64, "the slow-axis lines in one pass");
      if (tid < 9 * K) planes(tid, true, tid >= 5 * K);
    } else {
#pragma unroll
      for (int r = 0; r < (5 * K + G - 1) / G; ++r)
        if (tid + r * G < 5 * K) planes(tid + r * G, true, false);
      if (tid < 4 * K) planes(5 * K + tid, false, true);
    }
    group_sync<NT>();
  }
#undef VCP_FOPS
}

// The three directions in one launch: blockIdx.y is the direction;
// blockIdx.x the element, or (BATCH) a work item (case, element) of the
// group. The argument block is read through the kernel-argument segment
// pointer: a by-value copy indexed at run time would go to scratch. The SGS
// form is compiled for two waves per SIMD, where its eddy-viscosity code fits
// the registers without spilling.
template <int K, int M, bool BUG, bool BATCH, typename T, typename TL, bool SGS>
__global__ __launch_bounds__((FaceSmem<K, M, T, TL>::NT), (SGS ? cmin(2, FaceSmem<K, M, T, TL>::kWaves) : FaceSmem<K, M, T, TL>::kWaves))
void face_kernel(FaceArgs<K, M, T> a_)
{
  __shared__ FaceSmem<K, M, T, TL> sm;
  (void) a_;
  const FaceArgs<K, M, T> &a = *(const FaceArgs<K, M, T> *) __builtin_amdgcn_kernarg_segment_ptr();
  using S = FaceSmem<K, M, T, TL>;
  const int sub = threadIdx.x / S::G, item = blockIdx.x * S::NF + sub;
  bool live = S::NF == 1 || item < a.n;
  CaseDev c;
  int e;
  if constexpr (BATCH) {
    const WorkItem w = a.work[a.w0 + (live ? item : 0)];
    c = a.cases[w.c];
    e = w.e;
    live = live && c.flags[kWordActive] != 0;
    if (!__any(live)) return;
  } else {
    c = a.c;
    e = live ? item : 0;
  }
  if (blockIdx.y == 0) face_body<K, M, 0, BUG, BATCH, T, TL, SGS>(a, c, sm, e, live);
  else if (blockIdx.y == 1) face_body<K, M, 1, BUG, BATCH, T, TL, SGS>(a, c, sm, e, live);
  else face_body<K, M, 2, BUG, BATCH, T, TL, SGS>(a, c, sm, e, live);
}

template <int K, int M, typename T>
void fill_face_ops(const DeviceCase &dc, FaceOps<K, M, T> &op)
{
  fill_even_odd(dc.opA, op.a);
  fill_even_odd(dc.opD, op.d);
  fill_even_odd(dc.opA, op.ad);
  for (int i = 0; i < M * K; ++i) { op.A[i] = T(dc.opA[i]); op.D[i] = T(dc.opD[i]); }
  for (int q = 0; q < K; ++q)
    for (int t = 0; t < 4; ++t) op.F[t][q] = T(dc.opF[t][q]);
  for (int q = 0; q < M; ++q) op.w[q] = dc.opW[q];
  op.c03 = dc.opC0[0] * dc.opC0[0] * dc.opC0[0];
}

template <int K, int M, bool BATCH, typename T, typename TL, bool SGS>
void launch_face_kernel(bool bug, int n, FaceArgs<K, M, T> &a, hipStream_t s)
{
  using S = FaceSmem<K, M, T, TL>;
  const dim3 grid((n + S::NF - 1) / S::NF, 3), block(S::NT);
  a.n = n;
  if (bug) hipLaunchKernelGGL((face_kernel<K, M, true, BATCH, T, TL, SGS>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((face_kernel<K, M, false, BATCH, T, TL, SGS>), grid, block, 0, s, a);
}

template <int K, int M, typename T, typename TL>
hipError_t faces_impl(const DeviceCase &dc, hipStream_t s)
{
  FaceArgs<K, M, T> a{};
  a.c = case_dev(dc);
  fill_face_ops(dc, a.op);
  if (dc.sgs) launch_face_kernel<K, M, false, T, TL, true>(dc.bug_compat, dc.nElem, a, s);
  else launch_face_kernel<K, M, false, T, TL, false>(dc.bug_compat, dc.nElem, a, s);
  return hipGetLastError();
}

template <int K, int M, typename T, typename TL>
hipError_t batch_faces_impl(const BatchGroup &g, int w0, int nw, hipStream_t s)
{
  FaceArgs<K, M, T> a{};
  a.cases = g.cases; a.work = g.work; a.w0 = w0;
  fill_face_ops(*g.proto, a.op);
  if (g.proto->sgs) launch_face_kernel<K, M, true, T, TL, true>(g.proto->bug_compat, nw, a, s);
  else launch_face_kernel<K, M, true, T, TL, false>(g.proto->bug_compat, nw, a, s);
  return hipGetLastError();
}

}  // namespace

template <int K, int M>
hipError_t faces(const DeviceCase &dc, bool wide, hipStream_t s)
{
  if (!dc.mixed) return faces_impl<K, M, double, double>(dc, s);
  return wide ? faces_impl<K, M, float, double>(dc, s) : faces_impl<K, M, float, float>(dc, s);
}

template <int K, int M>
hipError_t batch_faces(const BatchGroup &g, bool wide, int w0, int nw, hipStream_t s)
{
  if (!g.proto->mixed) return batch_faces_impl<K, M, double, double>(g, w0, nw, s);
  return wide ? batch_faces_impl<K, M, float, double>(g, w0, nw, s)
              : batch_faces_impl<K, M, float, float>(g, w0, nw, s);
}

template hipError_t faces<VCP_SHAPE_K, VCP_SHAPE_M>(const DeviceCase &, bool, hipStream_t);
template hipError_t batch_faces<VCP_SHAPE_K, VCP_SHAPE_M>(const BatchGroup &, bool, int, int, hipStream_t);

}  // namespace vcp
