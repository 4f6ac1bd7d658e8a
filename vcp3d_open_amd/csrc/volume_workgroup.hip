// Volume residual, face-slot gather, entropy mass-matrix solve and RK stage
// update, one workgroup per element (gfx950): the form for cases with too few
// elements to fill the chip with the column form (volume.hip). Compiled once
// per shape (VCP_SHAPE_K, VCP_SHAPE_M).
//
// Reference behaviour followed (VCP3D_CurviLinear/src/):
//   ElementClass::VolumeResidual          ElementClass.cpp:3809-4533
//   sponge layer / CML sources            ElementClass.cpp:3887-4117, :4450-4489
//   CG_EntropyVarMassMatrix               CG_MassMatrix.cpp:250-504
#include "device.hpp"
#include "kernels.hpp"

namespace vcp {
namespace {

// Block reduction with one barrier: partial results go to alternating
// halves of red (2 * 3 * NT/64 doubles); every half starts at the same offset
// whatever NV is, so a half is rewritten only after every thread has passed
// the barrier of the following reduction, also when consecutive reductions
// carry different numbers of values. The max slots (q >= NS) take
// non-negative values. Only waves [W0, W0 + NW) hold contributions; the
// others skip the wave reduction.
template <int NT, int NV, int NS, int NW = NT / 64, int W0 = 0>
__device__ inline void block_reduce1(double (&v)[NV], double *red, int &half)
{
  static_assert(NV >= 1 && NV <= 3, "a half holds at most three values per wave");
  static_assert(W0 >= 0 && W0 + NW <= NT / 64, "contributing waves");
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  double *buf = red + half * 3 * (NT / 64);
  if (wid >= W0 && wid < W0 + NW) {
#pragma unroll
    for (int q = 0; q < NV; ++q) v[q] = (q < NS) ? wave_reduce_dpp<false>(v[q]) : wave_reduce_dpp<true>(v[q]);
    if (lane == 0)
#pragma unroll
      for (int q = 0; q < NV; ++q) buf[wid * NV + q] = v[q];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    double s = buf[W0 * NV + q];
#pragma unroll
    for (int w = W0 + 1; w < W0 + NW; ++w) s = (q < NS) ? s + buf[w * NV + q] : fmax(s, buf[w * NV + q]);
    v[q] = s;
  }
  half ^= 1;
}

// 1D operators of the standard element as kernel arguments: indexed with
// compile-time constants after unrolling, they are read into scalar registers.
template <int K, int M, typename T = double>
struct Ops {
  T A[M * K];   // phi_q(r_p), row-major (p, q)
  T D[M * K];   // phi'_q(r_p)
};

// Volume kernel arguments: the case part (single-case launch) or the case
// table and work items (batched launch), the stage control and what depends
// on (K, M) only.
template <int K, int M, typename T = double>
struct VolArgs {
  CaseDev c;
  const CaseDev *cases;
  const WorkItem *work;
  int w0;
  StageCtl ctl;
  TableOffsets to;
  int bug;
  Ops<K, M, T> op;
  double c0[K];                           // phi_q(0): basis at the element centre
  double fvec[4][K];                      // phi(-1), phi(+1), phi'(-1), phi'(+1)
};

// ========================================================== volume kernel
// One workgroup of NT threads per element. LDS holds the modal state, the
// sum-factorisation intermediates and the primitive state at the points;
// the 1D operators come from the kernel arguments (scalar registers) in the
// pencil stages and from LDS rows in the per-point stages.
// Workgroup size of the volume kernel: 256 threads, or 512 when the two point
// passes or the DOFs do not fit 256 threads (K = 7, M = 9).
constexpr int vol_threads(int K, int M)
{
  return K * K * K <= 256 && M * M * M <= 256 + (256 / M) * M ? 256 : 512;
}

// LDS layout of the volume kernel and the waves per SIMD it is compiled for
// (NT = 256: three workgroups per CU when the LDS fits three times into 160 KB,
// which caps the kernel at 168 VGPRs; NT = 512: one or more workgroups of
// two waves per SIMD, or two workgroups when the LDS allows, which caps the
// kernel at 128 VGPRs; NT = 64, 128: as many workgroups as the LDS allows, at
// most three waves per SIMD).
template <int K, int M, int NT, typename T = double>
struct VolShape {
  static constexpr int ND = K * K * K, NI = M * M * M, NR = M * M;
  // Points go through the pointwise stages in two passes split at a row
  // (jk) boundary: rows [0, R0) in the first, the remaining rows in the second.
  static constexpr int R0 = (NT / M) < NR ? (NT / M) : NR;
  static constexpr int P0 = R0 * M, P1 = NI - P0;
  static constexpr int SZ = 5 * M * K * K;          // one z-stage buffer
  static constexpr int SY = 15 * NR * K;            // y-stage buffers, [jk][3][5][K]
  static constexpr int SF0 = 15 * P0, SF = 15 * NI; // fluxes of the first pass / all
  static constexpr int SI = 15 * NR * K;            // backward i-stage output
  static constexpr int BIG = cmax(cmax(2 * SZ + SY, SF), SI + 10 * M * K * K);
  // variable stride of the modal state in LDS: congruent to K^2 modulo the
  // bank count in elements, so that the (variable, j, i) pencil items of a
  // wave run on across a variable boundary without bank conflicts
  static constexpr int MODB = 256 / (int) sizeof(T);
  static constexpr int SUV = ND + ((K * K - ND) % MODB + MODB) % MODB;
  static constexpr int LDS = (int) sizeof(T) * (2 * M * K + 4 * SUV + ND + BIG + 15) + 8 * (45 + 6 * (NT / 64) + 4 * K + 5);
  static constexpr int WGS = (160 * 1024) / LDS;   // workgroups per CU by LDS
  // FP32 contractions: the smaller LDS allows more waves per SIMD
#ifndef VCP_MIXED_CG_TOL
#define VCP_MIXED_CG_TOL 1e-5
#endif
#ifndef VCP_F32_WAVES
#define VCP_F32_WAVES 3
#endif
  static constexpr int WAVES = NT == 256 ? (sizeof(T) == 4 && WGS >= VCP_F32_WAVES ? VCP_F32_WAVES : WGS >= 3 ? 3 : 2)
                              : NT > 256 ? (NT / 256) * (WGS >= 2 ? 2 : 1)
                                         : cmax(1, WGS * (NT / 64) / 4 < 3 ? WGS * (NT / 64) / 4 : 3);
  static_assert(WGS >= 1, "volume kernel LDS exceeds 160 KB");
  // mass-matrix solve buffers cz, cy, pI, by inside sBig
  static_assert(SZ + 5 * M * M * K + 5 * NI + 5 * M * K * K <= BIG, "CG buffers");
  // A p in the padded state layout runs from cz into the (then dead) cy
  static_assert(4 * SUV + ND <= SZ + 5 * M * M * K, "A p buffer");
};

// blockIdx.x is the element, or (BATCH) a work item (case, element) of the
// group; a is the case part. T is the type of the sum-factorisation
// contractions, the LDS buffers and the mass-matrix solve: double, or float
// for the mixed-precision form, where the state, its element means, the
// pointwise physics, the face-slot gather, the metric and the RK update stay
// in double. In the float form the mean (mode 0) of each variable is taken
// out of the modal state before the contractions and added back at the
// points in double (it contributes the same constant at every point and
// nothing to the gradients), so the float contractions carry only the
// variation about the mean.
template <int K, int M, int NT, bool BATCH, typename T = double>
__global__ __launch_bounds__(NT, (VolShape<K, M, NT, T>::WAVES)) void volume_kernel(VolArgs<K, M, T> args)
{
  using S = VolShape<K, M, NT, T>;
  constexpr bool kMixed = sizeof(T) == 4;
  constexpr int ND = S::ND, NI = S::NI, NR = S::NR, R0 = S::R0, P0 = S::P0, P1 = S::P1;
  constexpr int SZ = S::SZ, SF0 = S::SF0, SI = S::SI, BIG = S::BIG;
  static_assert(P1 <= NT, "two point passes");
  // the second point pass runs on the last waves (from thread T2), which own
  // no DOFs, leaving the first waves free
  constexpr int T2 = NT - ((P1 + 63) / 64) * 64;
  constexpr bool kPrecondLate = P1 > 0 && T2 >= 64;
  // rot() below wraps thread numbers with & (NT - 1)
  static_assert((NT & (NT - 1)) == 0, "NT must be a power of two");
  // the first pass's fluxes must leave the y-stage rows of the second pass intact
  static_assert(P1 == 0 || SF0 <= 2 * SZ + 15 * R0 * K, "flux / y-stage overlap");
  __shared__ T sA[M * K], sD[M * K];
  constexpr int SUV = S::SUV;
  __shared__ T sU[4 * SUV + ND];
  __shared__ T sBig[BIG];
  __shared__ double sCm[5][9];
  __shared__ double sRed[2 * (NT / 64) * 3];
  __shared__ T sDv[15];
  __shared__ double sFv[4 * K];
  __shared__ double sMean[5];     // float form: mode 0 of each variable
  // the case part is read where it is used: from the kernel arguments, or
  // (BATCH) from the group's case table
  const CaseDev *ap;
  int e;
  if constexpr (BATCH) {
    const WorkItem w = args.work[args.w0 + blockIdx.x];
    ap = args.cases + w.c;
    e = w.e;
    if (ap->flags[kWordActive] == 0) return;
  } else {
    ap = &args.c;
    e = blockIdx.x;
  }
  const CaseDev &a = *ap;
  const int tid = threadIdx.x;
  // Operators of the pencil stages: the kernel arguments (scalar registers)
  // while they fit; beyond that the compiler parks them in VGPR lanes and
  // reads them back with v_readlane (28 % of the instructions at K = 7 in
  // FP64), so larger operators come from the LDS copies: both above 800 bytes
  // (K = 7 in FP64: 26 % faster), D alone above 600 (K = 6 in FP64: 3 %
  // faster; both from LDS there, or either at K <= 5, measured slower).
  constexpr bool kArgOpsA = sizeof(args.op) <= 800, kArgOpsD = sizeof(args.op) <= 600;
  const T *A = kArgOpsA ? args.op.A : sA, *D = kArgOpsD ? args.op.D : sD;
  const double *Ue = a.U + (size_t) e * 5 * ND;
  const double *vg = a.vgeo + (size_t) e * kVolGeo * NI;
  const int sp = a.spIdx ? a.spIdx[e] : -1;
  for (int i = tid; i < M * K; i += NT) { sA[i] = args.op.A[i]; sD[i] = args.op.D[i]; }
  for (int i = tid; i < 4 * K; i += NT) sFv[i] = args.fvec[i / K][i % K];
  {
    // the modal state: every load issued before the first is waited for
    constexpr int NIT = (5 * ND + NT - 1) / NT;
    double uu[NIT];
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int i = tid + it * NT;
      uu[it] = Ue[i < 5 * ND ? i : 0];
    }
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int i = tid + it * NT;
      if (i < 5 * ND) {
        if constexpr (kMixed) {
          if (i % ND == 0) sMean[i / ND] = uu[it];
          sU[(i / ND) * SUV + i % ND] = i % ND == 0 ? T(0) : T(uu[it]);
        } else {
          sU[(i / ND) * SUV + i % ND] = uu[it];
        }
      }
    }
  }
  if (args.bug)
    for (int i = tid; i < 45; i += NT) sCm[i / 9][i % 9] = vg[(1 + i % 9) * NI + i / 9];
  // loaded here, used much later, so that their latency passes under the
  // first contractions: the element's Jacobian constant and (K <= 5, where
  // the registers allow it) the metric of this thread's point in the first
  // point pass
  const double elemJac = a.econst[(size_t) e * kElemConst + 3];
  constexpr bool kGeoEarly = K <= 5;
  double geoJ0 = 0.0, geoW0 = 0.0, geoCm0[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  if (kGeoEarly && tid < P0) {
    geoJ0 = vg[tid];
    geoW0 = a.tables[args.to.w3 + tid];
#pragma unroll
    for (int t = 0; t < 9; ++t) geoCm0[t] = vg[(1 + t) * NI + tid];
  }
  __syncthreads();

  // ---------------- step 1: solution and parametric gradients at the points
  // z-stage buffers, then the y-stage buffers row-major: yB[jk][3][5][K] with
  // the (A, A), (D, A), (A, D) contractions of variable v at row jk = k * M + j
  T *zA = sBig, *zD = zA + SZ, *yB = zD + SZ;
  for (int pc = tid; pc < 5 * K * K; pc += NT) {      // pencil (v, j, i) along k
    const int v = pc / (K * K), ji = pc - v * K * K;
    T x[K];
#pragma unroll
    for (int q = 0; q < K; ++q) x[q] = sU[v * SUV + q * K * K + ji];
#pragma unroll
    for (int n = 0; n < M; ++n) {
      T sa = 0, sd = 0;
#pragma unroll
      for (int q = 0; q < K; ++q) { sa += A[n * K + q] * x[q]; sd += D[n * K + q] * x[q]; }
      zA[(v * M + n) * K * K + ji] = sa;
      zD[(v * M + n) * K * K + ji] = sd;
    }
  }
  // element-centre entropy variables -> preconditioner dV/dU / Jbar in sDv,
  // by one whole wave (lane 0 the last part), in a stage where that wave has
  // no other work: the second point pass when it leaves the first wave idle,
  // else the first contraction, beside the pencils (none in the last wave when
  // 5 K^2 <= NT - 64)
  auto precond = [&]() {
    const int lane = tid & 63;
    double Vc[5] = {0, 0, 0, 0, 0};
    for (int i = lane; i < ND; i += 64) {
      const int ii = i % K, jj = (i / K) % K, kk = i / (K * K);
      double b = 0.0, bj = 0.0, bk = 0.0;
#pragma unroll
      for (int q = 0; q < K; ++q) {
        if (q == ii) b = args.c0[q];
        if (q == jj) bj = args.c0[q];
        if (q == kk) bk = args.c0[q];
      }
      b *= bj * bk;
#pragma unroll
      for (int v = 0; v < 5; ++v) Vc[v] += b * sU[v * SUV + i];
    }
#pragma unroll
    for (int v = 0; v < 5; ++v) Vc[v] = wave_sum(Vc[v]);
    if constexpr (kMixed) {
      const double c03 = args.c0[0] * args.c0[0] * args.c0[0];
#pragma unroll
      for (int v = 0; v < 5; ++v) Vc[v] += c03 * sMean[v];
    }
    if (lane == 0) {
      double rho, u, v, w, p, eKin;
      ent2prim(Vc, rho, u, v, w, p, eKin);
      const double JacInv = 8.0 / elemJac;
      const double pInv = 1.0 / p, a1 = kGm1 * rho * pInv * pInv, a2 = eKin * a1;
      sDv[0] = T(JacInv * (kGam / kGm1 / rho + a2 * eKin)); sDv[1] = T(-JacInv * u * a2); sDv[2] = T(-JacInv * v * a2);
      sDv[3] = T(-JacInv * w * a2); sDv[4] = T(JacInv * (a2 - pInv)); sDv[5] = T(JacInv * (a1 * u * u + pInv));
      sDv[6] = T(JacInv * a1 * u * v); sDv[7] = T(JacInv * a1 * u * w); sDv[8] = T(-JacInv * a1 * u);
      sDv[9] = T(JacInv * (a1 * v * v + pInv)); sDv[10] = T(JacInv * a1 * v * w); sDv[11] = T(-JacInv * a1 * v);
      sDv[12] = T(JacInv * (a1 * w * w + pInv)); sDv[13] = T(-JacInv * a1 * w); sDv[14] = T(JacInv * a1);
    }
  };
  if (!kPrecondLate && tid >= NT - 64) precond();
  __syncthreads();
  for (int pc = tid; pc < 5 * M * K; pc += NT) {      // pencil (v, k', i) along j
    const int vk = pc / K, i = pc - vk * K;
    const int v = vk / M, kp = vk - v * M;
    T xa[K], xd[K];
#pragma unroll
    for (int q = 0; q < K; ++q) { xa[q] = zA[(vk * K + q) * K + i]; xd[q] = zD[(vk * K + q) * K + i]; }
    T *yo = yB + (kp * M * 15 + v) * K + i;
#pragma unroll
    for (int n = 0; n < M; ++n) {
      T s0 = 0, s1 = 0, s2 = 0;
#pragma unroll
      for (int q = 0; q < K; ++q) { s0 += A[n * K + q] * xa[q]; s1 += D[n * K + q] * xa[q]; s2 += A[n * K + q] * xd[q]; }
      yo[(n * 15 + 0) * K] = s0;
      yo[(n * 15 + 5) * K] = s1;
      yo[(n * 15 + 10) * K] = s2;
    }
  }
  __syncthreads();

  // ---------------- steps 2, 3, 5, 6: x stage, pointwise fluxes, primitive
  // state, monitoring; in two passes over the points (rows [0, R0), then the
  // rest), each thread one point per pass. The first pass's fluxes F[b][m]
  // (b = 5 d + l) fill [0, SF0) and leave the y-stage rows of the second
  // pass in place; the second pass's fluxes go to SF0 + [b][m - P0].
  const double factHF = a.mu * kGam / kPrLam;
  const double lenLES = a.sgs ? a.econst[(size_t) e * kElemConst + kElemLenLES] : 0.0;
  double mach2 = 0.0, evMax = 0.0;
  // (w J rho, u, v, w, w J p, w J dU/dV_44) at the thread's points, for the
  // weighted dU/dV in the solve
  T prim[2][6];
  // float form: the constant contribution of the element means at every point
  double meanPt[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  if constexpr (kMixed) {
    const double c03 = args.c0[0] * args.c0[0] * args.c0[0];
#pragma unroll
    for (int v = 0; v < 5; ++v) meanPt[v] = c03 * sMean[v];
  }
#pragma unroll
  for (int q = 0; q < (P1 > 0 ? 2 : 1); ++q) {
    const int m = q == 0 ? tid : P0 + tid - T2;
    const bool act = q == 0 ? tid < P0 : (tid >= T2 && tid - T2 < P1);
    double Vp[5], Gr[5], Gs[5], Gt[5];
    // the second pass's metric, loaded before its x stage
    double geoJ1 = 0.0, geoW1 = 0.0, geoCm1[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    if (kGeoEarly && q == 1 && act) {
      geoJ1 = vg[m];
      geoW1 = a.tables[args.to.w3 + m];
#pragma unroll
      for (int t = 0; t < 9; ++t) geoCm1[t] = vg[(1 + t) * NI + m];
    }
    if (act) {
      const int i = m % M, jk = m / M;
      T ai[K], di[K];
#pragma unroll
      for (int ii = 0; ii < K; ++ii) { ai[ii] = sA[i * K + ii]; di[ii] = sD[i * K + ii]; }
      int roff = jk * 15 * K;
      asm volatile("" : "+v"(roff));   // one base register, immediate LDS offsets
      const T *row = yB + roff;
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        const T *ra = row + v * K, *rd = row + (5 + v) * K, *rz = row + (10 + v) * K;
        T s0 = 0, s1 = 0, s2 = 0, s3 = 0;
#pragma unroll
        for (int ii = 0; ii < K; ++ii) {
          const T x = ra[ii];
          s0 += ai[ii] * x; s1 += di[ii] * x; s2 += ai[ii] * rd[ii]; s3 += ai[ii] * rz[ii];
        }
        Vp[v] = kMixed ? double(s0) + meanPt[v] : double(s0);
        Gr[v] = s1; Gs[v] = s2; Gt[v] = s3;
      }
    }
    __syncthreads();
    if (kPrecondLate && q == 1 && tid < 64) precond();
    if (!act) continue;
    T *Fb = q == 0 ? sBig + m : sBig + SF0 + (m - P0);
    const int fstride = q == 0 ? P0 : P1;
    const double J = !kGeoEarly ? vg[m] : q == 0 ? geoJ0 : geoJ1;
    const double wJ = (!kGeoEarly ? a.tables[args.to.w3 + m] : q == 0 ? geoW0 : geoW1) * J;
    double cm[9];                                      // dr/dx .. dt/dz at the point
#pragma unroll
    for (int t = 0; t < 9; ++t) cm[t] = !kGeoEarly ? vg[(1 + t) * NI + m] : q == 0 ? geoCm0[t] : geoCm1[t];
    double gx[5], gy[5], gz[5];
    if (args.bug) {
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        const double *c = sCm[v];
        gx[v] = Gr[v] * c[0] + Gs[v] * c[3] + Gt[v] * c[6];
        gy[v] = Gr[v] * c[1] + Gs[v] * c[4] + Gt[v] * c[7];
        gz[v] = Gr[v] * c[2] + Gs[v] * c[5] + Gt[v] * c[8];
      }
    } else {
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        gx[v] = Gr[v] * cm[0] + Gs[v] * cm[3] + Gt[v] * cm[6];
        gy[v] = Gr[v] * cm[1] + Gs[v] * cm[4] + Gt[v] * cm[7];
        gz[v] = Gr[v] * cm[2] + Gs[v] * cm[5] + Gt[v] * cm[8];
      }
    }
    double rho, u, v, w, p, eKin;
    ent2prim(Vp, rho, u, v, w, p, eKin);
    const double V4Inv = 1.0 / Vp[4];
    const double rE = p * kInvGm1 + rho * eKin;
    prim[q][0] = T(wJ * rho); prim[q][1] = T(u); prim[q][2] = T(v); prim[q][3] = T(w); prim[q][4] = T(wJ * p);
    prim[q][5] = T(wJ * (rE * (rE + p) / rho + p * eKin));
    const double dudx = -V4Inv * (gx[1] + u * gx[4]), dudy = -V4Inv * (gy[1] + u * gy[4]), dudz = -V4Inv * (gz[1] + u * gz[4]);
    const double dvdx = -V4Inv * (gx[2] + v * gx[4]), dvdy = -V4Inv * (gy[2] + v * gy[4]), dvdz = -V4Inv * (gz[2] + v * gz[4]);
    const double dwdx = -V4Inv * (gx[3] + w * gx[4]), dwdy = -V4Inv * (gy[3] + w * gy[4]), dwdz = -V4Inv * (gz[3] + w * gz[4]);
    const double fe = V4Inv * V4Inv * kInvGm1;
    const double dedx = fe * gx[4], dedy = fe * gy[4], dedz = fe * gz[4];
    if (args.ctl.monitor) mach2 = fmax(mach2, rho * (u * u + v * v + w * w) / (kGam * p));
    const double ru = rho * u, rv = rho * v, rw = rho * w;
    // eddy viscosity of the SGS model (ElementClass.cpp:4268-4287, :4305-4306)
    // in the total viscosity and heat-flux factor (:4339-4342)
    double mu = a.mu, fhT = factHF;
    if (a.sgs != kSgsNone) {
      const double G[3][3] = {{dudx, dudy, dudz}, {dvdx, dvdy, dvdz}, {dwdx, dwdy, dwdz}};
      const double ev = eddy_viscosity(a.sgs, lenLES, rho, G);
      evMax = fmax(evMax, ev);
      mu = a.mu + ev;
      fhT = a.mu * (kGam / kPrLam) + ev * (kGam / kPrTurb);
    }
    const double divV = kLamOverMu * (dudx + dvdy + dwdz);
    const double txx = mu * (2.0 * dudx + divV), tyy = mu * (2.0 * dvdy + divV), tzz = mu * (2.0 * dwdz + divV);
    const double txy = mu * (dudy + dvdx), txz = mu * (dudz + dwdx), tyz = mu * (dvdz + dwdy);
    const double qx = -fhT * dedx, qy = -fhT * dedy, qz = -fhT * dedz;
    const double fx[5] = {ru, ru * u - txx + p, rv * u - txy, rw * u - txz, (rE + p) * u - (u * txx + v * txy + w * txz - qx)};
    const double fy[5] = {rv, ru * v - txy, rv * v - tyy + p, rw * v - tyz, (rE + p) * v - (u * txy + v * tyy + w * tyz - qy)};
    const double fz[5] = {rw, ru * w - txz, rv * w - tyz, rw * w - tzz + p, (rE + p) * w - (u * txz + v * tyz + w * tzz - qz)};
    const double weight = -wJ;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double mx = weight * cm[3 * d], my = weight * cm[3 * d + 1], mz = weight * cm[3 * d + 2];
#pragma unroll
      for (int l = 0; l < 5; ++l) Fb[(d * 5 + l) * fstride] = T(fx[l] * mx + fy[l] * my + fz[l] * mz);
    }
    if (sp >= 0) {
      // sponge damping sigma J w (U - U_target) and CML sources
      // (ElementClass.cpp:4450-4489, :3887-4117)
      const double *fn = a.dampFn + (size_t) sp * 3 * NI, *ds = a.dampState + (size_t) sp * 5 * NI;
      const double sigma = wJ * (fn[m] + fn[NI + m] + fn[2 * NI + m]);
      double src[5];
      src[0] = sigma * (rho - ds[m]);
      src[1] = sigma * (ru - ds[NI + m]);
      src[2] = sigma * (rv - ds[2 * NI + m]);
      src[3] = sigma * (rw - ds[3 * NI + m]);
      src[4] = sigma * (rE - ds[4 * NI + m]);
      if (a.cml) {
        const double *cf = a.spCoef + (size_t) sp * 8;
        const double wgt[3] = {weight * cf[0] * fn[m], weight * cf[1] * fn[NI + m], weight * cf[2] * fn[2 * NI + m]};
        const double nsg[3] = {cf[3], cf[4], cf[5]};
        cml_source(Vp, gx, gy, gz, wgt, nsg, src);
      }
      double *sb = a.srcBuf + (size_t) sp * 5 * NI;
#pragma unroll
      for (int l = 0; l < 5; ++l) sb[l * NI + m] = src[l];
    }

  }
  __syncthreads();

  if (a.bfBuf) {
    // body force per unit volume (ElementClass.cpp:4492-4523): -w J f on the
    // momentum and -w J u.f on the energy equation at this thread's points,
    // with the velocities kept for the solve; projected with the sponge source
    const double fx = a.fbody[0], fy = a.fbody[1], fz = a.fbody[2];
    double *bb = a.bfBuf + (size_t) e * 4 * NI;
#pragma unroll
    for (int q = 0; q < (P1 > 0 ? 2 : 1); ++q) {
      const int m = q == 0 ? tid : P0 + tid - T2;
      if (!(q == 0 ? tid < P0 : (tid >= T2 && tid - T2 < P1))) continue;
      const double weight = -(a.tables[args.to.w3 + m] * vg[m]);
      const double u = prim[q][1], v = prim[q][2], w = prim[q][3];
      bb[m] = weight * fx;
      bb[NI + m] = weight * fy;
      bb[2 * NI + m] = weight * fz;
      bb[3 * NI + m] = weight * (u * fx + v * fy + w * fz);
    }
  }

  // the six face contributions at this thread's DOF (DOF-major: thread
  // d < ND owns DOF d of all five variables): each face slot holds the value
  // and normal-derivative coefficient planes over its two tangential axes,
  // times the face vectors phi(r_f), phi'(r_f) at the DOF's normal index
  static_assert(ND <= NT, "one DOF per thread in the mass-matrix solve");
  double racc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  if (tid < ND) {
    const int di = tid % K, dj = (tid / K) % K, dk = tid / (K * K);
    const double *fr = a.faceRes + (size_t) e * 6 * 10 * K * K;
#pragma unroll
    for (int f = 0; f < 6; ++f) {
      const int dir = f >> 1, side = f & 1;
      const int tn = dir == 0 ? di : dir == 1 ? dj : dk;
      const int fa = dir == 0 ? dj : di;
      const int sl = dir == 2 ? dj : dk;
      const double cv = sFv[side * K + tn], cd = sFv[(2 + side) * K + tn];
      const double *b = fr + f * 10 * K * K + sl * K + fa;
#pragma unroll
      for (int l = 0; l < 5; ++l) racc[l] += cv * b[l * K * K] + cd * b[(5 + l) * K * K];
    }
  }

  // ---------------- step 7: transposed contractions of the three fluxes
  // rows (b, jk) along i, compacted to I[b][jk][K] once every row is read
  {
    constexpr int NRW = 15 * NR, RPT = (NRW + NT - 1) / NT;
    T o[RPT][K];
#pragma unroll
    for (int t = 0; t < RPT; ++t) {
      const int r = tid + t * NT;
      if (r < NRW) {
        const int b = r / NR, jk = r - b * NR;
        const T *x = jk < R0 ? sBig + b * P0 + jk * M : sBig + SF0 + b * P1 + (jk - R0) * M;
        T xx[M];
#pragma unroll
        for (int q = 0; q < M; ++q) xx[q] = x[q];
#pragma unroll
        for (int n = 0; n < K; ++n) {
          T s = 0;
          if (b < 5) {
#pragma unroll
            for (int q = 0; q < M; ++q) s += D[q * K + n] * xx[q];
          } else {
#pragma unroll
            for (int q = 0; q < M; ++q) s += A[q * K + n] * xx[q];
          }
          o[t][n] = s;
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < RPT; ++t) {
      const int r = tid + t * NT;
      if (r < NRW)
#pragma unroll
        for (int n = 0; n < K; ++n) sBig[r * K + n] = o[t][n];
    }
  }
  __syncthreads();
  const T *I0 = sBig, *I1 = I0 + 5 * NR * K, *I2 = I1 + 5 * NR * K;
  T *Y01 = sBig + SI, *Y2 = Y01 + 5 * M * K * K;   // after the i-stage block
  for (int pc = tid; pc < 5 * M * K; pc += NT) {      // pencil (v, k, i') along j
    const int vk = pc / K, i = pc - vk * K;
    T x0[M], x1[M], x2[M];
#pragma unroll
    for (int q = 0; q < M; ++q) {
      x0[q] = I0[(vk * M + q) * K + i]; x1[q] = I1[(vk * M + q) * K + i]; x2[q] = I2[(vk * M + q) * K + i];
    }
#pragma unroll
    for (int n = 0; n < K; ++n) {
      T s01 = 0, s2 = 0;
#pragma unroll
      for (int q = 0; q < M; ++q) { s01 += A[q * K + n] * x0[q] + D[q * K + n] * x1[q]; s2 += A[q * K + n] * x2[q]; }
      Y01[(vk * K + n) * K + i] = s01;
      Y2[(vk * K + n) * K + i] = s2;
    }
  }
  __syncthreads();
  for (int pc = tid; pc < 5 * K * K; pc += NT) {      // pencil (v, j', i') along k
    const int v = pc / (K * K), ji = pc - v * K * K;
    T y0[M], y2[M];
#pragma unroll
    for (int q = 0; q < M; ++q) { y0[q] = Y01[(v * M + q) * K * K + ji]; y2[q] = Y2[(v * M + q) * K * K + ji]; }
#pragma unroll
    for (int n = 0; n < K; ++n) {
      T s = 0;
#pragma unroll
      for (int q = 0; q < M; ++q) s += A[q * K + n] * y0[q] + D[q * K + n] * y2[q];
      sU[v * SUV + n * K * K + ji] = s;
    }
  }
  __syncthreads();
  if (sp >= 0 || a.bfBuf) {
    // the sponge element's damping and CML sources and the body force
    // (ElementClass.cpp:4492-4533, on the momentum and energy equations),
    // both from the point pass, summed at the points and projected with the
    // basis functions: rows along i, pencils along j, then along k,
    // accumulated into the residual
    const double *sb = sp >= 0 ? a.srcBuf + (size_t) sp * 5 * NI : nullptr;
    const double *bb = a.bfBuf ? a.bfBuf + (size_t) e * 4 * NI : nullptr;
    for (int r = tid; r < 5 * M * M; r += NT) {       // rows along i
      T xx[M];
#pragma unroll
      for (int q = 0; q < M; ++q) {
        double x = sb ? sb[r * M + q] : 0.0;
        if (bb && r >= M * M) x += bb[r * M + q - NI];
        xx[q] = T(x);
      }
#pragma unroll
      for (int n = 0; n < K; ++n) {
        T s = 0;
#pragma unroll
        for (int q = 0; q < M; ++q) s += A[q * K + n] * xx[q];
        sBig[r * K + n] = s;
      }
    }
    __syncthreads();
    T *Ys = sBig + 5 * M * M * K;
    for (int pc = tid; pc < 5 * M * K; pc += NT) {    // pencils along j
      const int vk = pc / K, i = pc - vk * K;
      T xx[M];
#pragma unroll
      for (int q = 0; q < M; ++q) xx[q] = sBig[(vk * M + q) * K + i];
#pragma unroll
      for (int n = 0; n < K; ++n) {
        T s = 0;
#pragma unroll
        for (int q = 0; q < M; ++q) s += A[q * K + n] * xx[q];
        Ys[(vk * K + n) * K + i] = s;
      }
    }
    __syncthreads();
    for (int pc = tid; pc < 5 * K * K; pc += NT) {    // pencils along k, accumulated
      const int v = pc / (K * K), ji = pc - v * K * K;
      T xx[M];
#pragma unroll
      for (int q = 0; q < M; ++q) xx[q] = Ys[(v * M + q) * K * K + ji];
#pragma unroll
      for (int n = 0; n < K; ++n) {
        T s = 0;
#pragma unroll
        for (int q = 0; q < M; ++q) s += A[q * K + n] * xx[q];
        sU[v * SUV + n * K * K + ji] += s;
      }
    }
    __syncthreads();
  }

  // ---------------- gather the six face contributions
  // (a non-finite right-hand side is flagged: the solve's max-norms would
  // pass over it)
  bool bad = false;
  T r[5];
  if constexpr (kMixed) {
#pragma unroll
    for (int l = 0; l < 5; ++l) {
      if (tid < ND) racc[l] += double(sU[l * SUV + tid]);
      bad = bad || !isfinite(racc[l]);
      r[l] = T(racc[l]);
    }
  } else {
    if (tid < ND)
#pragma unroll
      for (int l = 0; l < 5; ++l) {
        racc[l] += sU[l * SUV + tid];
        bad = bad || !isfinite(racc[l]);
      }
#pragma unroll
    for (int l = 0; l < 5; ++l) r[l] = racc[l];
  }

  // ---------------- entropy-variable mass matrix: flexible PCG
  const double JacInv = 8.0 / elemJac;
  const bool own = tid < ND;
  T x[5], z[5], pv[5];
  int half = 0;
  double r0 = 0.0;
#pragma unroll
  for (int l = 0; l < 5; ++l) { x[l] = 0; r0 = fmax(r0, fabs(double(r[l]))); }
  {
    // with the element's maximum Mach^2 and eddy viscosity for the
    // monitoring data
    double red[3] = {r0, mach2, evMax};
    block_reduce1<NT, 3, 0>(red, sRed, half);
    r0 = red[0];
    if (args.ctl.monitor && tid == 0) a.mach2Elem[e] = red[1];
    if (a.eddyPart && tid == 0) a.eddyPart[e] = red[2];
  }
  int iters = 0;
  if (r0 * JacInv > 1e-10) {
    T *cz = sBig, *cy = cz + SZ, *pI = cy + 5 * M * M * K, *by = pI + 5 * NI;
    // z = dV/dU(centre) r, local to the thread owning the DOF
#define VCP_PRECOND()                                                                             \
    do {                                                                                          \
      z[0] = sDv[0] * r[0] + sDv[1] * r[1] + sDv[2] * r[2] + sDv[3] * r[3] + sDv[4] * r[4];       \
      z[1] = sDv[1] * r[0] + sDv[5] * r[1] + sDv[6] * r[2] + sDv[7] * r[3] + sDv[8] * r[4];       \
      z[2] = sDv[2] * r[0] + sDv[6] * r[1] + sDv[9] * r[2] + sDv[10] * r[3] + sDv[11] * r[4];     \
      z[3] = sDv[3] * r[0] + sDv[7] * r[1] + sDv[10] * r[2] + sDv[12] * r[3] + sDv[13] * r[4];    \
      z[4] = sDv[4] * r[0] + sDv[8] * r[1] + sDv[11] * r[2] + sDv[13] * r[3] + sDv[14] * r[4];    \
    } while (0)
    VCP_PRECOND();
    double rz = 0.0;
#pragma unroll
    for (int l = 0; l < 5; ++l) { pv[l] = z[l]; rz += double(r[l]) * double(z[l]); }
    { double red[1] = {rz}; block_reduce1<NT, 1, 1, (ND + 63) / 64>(red, sRed, half); rz = red[0]; }
    // Stages with fewer items than threads start at different waves, so that
    // the waves of the workgroup (one per SIMD) carry similar shares of the
    // iteration: the DOF owners and the second point pass sit in the first
    // waves, the two k stages in the last ones. rot(F) numbers the threads
    // from wave F on.
    constexpr int NWV = NT / 64, NWK = (5 * K * K + 63) / 64;
    constexpr int FK = NWV - NWK < 2 ? NWV - NWK : 2;
    auto rot = [tid](int F) { return (tid + NT - 64 * F) & (NT - 1); };
    for (int it = 0;; ++it) {
      if (it == 100) { atomicOr(a.flags, kFlagCGNotConverged); break; }
      if (own)
#pragma unroll
        for (int l = 0; l < 5; ++l) sU[l * SUV + tid] = pv[l];
      __syncthreads();
      for (int pc = rot(FK); pc < 5 * K * K; pc += NT) {
        const int v = pc / (K * K), ji = pc - v * K * K;
        T xx[K];
#pragma unroll
        for (int q = 0; q < K; ++q) xx[q] = sU[v * SUV + q * K * K + ji];
#pragma unroll
        for (int n = 0; n < M; ++n) {
          T s = 0;
#pragma unroll
          for (int q = 0; q < K; ++q) s += A[n * K + q] * xx[q];
          cz[(v * M + n) * K * K + ji] = s;
        }
      }
      __syncthreads();
      for (int pc = rot(1); pc < 5 * M * K; pc += NT) {
        const int i = pc / (5 * M), vk = pc - i * (5 * M);
        T xx[K];
#pragma unroll
        for (int q = 0; q < K; ++q) xx[q] = cz[(vk * K + q) * K + i];
#pragma unroll
        for (int n = 0; n < M; ++n) {
          T s = 0;
#pragma unroll
          for (int q = 0; q < K; ++q) s += A[n * K + q] * xx[q];
          cy[(vk * M + n) * K + i] = s;
        }
      }
      __syncthreads();
      // along i, one pencil (variable, row jk) per item with the operator from
      // the kernel arguments: K LDS reads per M outputs, where a per-point
      // contraction would read 5 K values and an operator row per point
      for (int pc = tid; pc < 5 * M * M; pc += NT) {
        const int l = pc / (M * M), jk = pc - l * M * M;
        T xx[K];
#pragma unroll
        for (int q = 0; q < K; ++q) xx[q] = cy[pc * K + q];
#pragma unroll
        for (int n = 0; n < M; ++n) {
          T s = 0;
#pragma unroll
          for (int q = 0; q < K; ++q) s += A[n * K + q] * xx[q];
          pI[l * NI + jk * M + n] = s;
        }
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < (P1 > 0 ? 2 : 1); ++q) {
        const int m = q == 0 ? tid : P0 + tid - T2;
        if (!(q == 0 ? tid < P0 : (tid >= T2 && tid - T2 < P1))) continue;
        T pp[5];
#pragma unroll
        for (int l = 0; l < 5; ++l) pp[l] = pI[l * NI + m];
        // w J dU/dV at the point (ElementClass.cpp:4228-4253): every entry is
        // homogeneous of degree one in (rho, p), so the scaled pair held in
        // prim gives the weighted matrix directly
        const T rho = prim[q][0], u = prim[q][1], v = prim[q][2], w = prim[q][3], p = prim[q][4];
        const T d44 = prim[q][5];
        const T eKin = T(0.5) * (u * u + v * v + w * w);
        const T rE = p * T(kInvGm1) + rho * eKin, rH = rE + p;
        const T ru = rho * u, rv = rho * v, rw = rho * w;
        pI[0 * NI + m] = rho * pp[0] + ru * pp[1] + rv * pp[2] + rw * pp[3] + rE * pp[4];
        pI[1 * NI + m] = ru * pp[0] + (ru * u + p) * pp[1] + ru * v * pp[2] + ru * w * pp[3] + rH * u * pp[4];
        pI[2 * NI + m] = rv * pp[0] + ru * v * pp[1] + (rv * v + p) * pp[2] + rv * w * pp[3] + rH * v * pp[4];
        pI[3 * NI + m] = rw * pp[0] + ru * w * pp[1] + rv * w * pp[2] + (rw * w + p) * pp[3] + rH * w * pp[4];
        pI[4 * NI + m] = rE * pp[0] + rH * u * pp[1] + rH * v * pp[2] + rH * w * pp[3] + d44 * pp[4];
      }
      __syncthreads();
      for (int rr = tid; rr < 5 * M * M; rr += NT) {
        T xx[M];
#pragma unroll
        for (int q = 0; q < M; ++q) xx[q] = pI[rr * M + q];
#pragma unroll
        for (int n = 0; n < K; ++n) {
          T s = 0;
#pragma unroll
          for (int q = 0; q < M; ++q) s += A[q * K + n] * xx[q];
          pI[rr * M + n] = s;
        }
      }
      __syncthreads();
      for (int pc = rot(2); pc < 5 * M * K; pc += NT) {
        const int i = pc / (5 * M), vk = pc - i * (5 * M);
        T xx[M];
#pragma unroll
        for (int q = 0; q < M; ++q) xx[q] = pI[(vk * M + q) * M + i];
#pragma unroll
        for (int n = 0; n < K; ++n) {
          T s = 0;
#pragma unroll
          for (int q = 0; q < M; ++q) s += A[q * K + n] * xx[q];
          by[(vk * K + n) * K + i] = s;
        }
      }
      __syncthreads();
      // Ap along k, with the partial p.Ap of the entries each thread computes
      double pAp = 0.0;
      for (int pc = rot(FK); pc < 5 * K * K; pc += NT) {
        const int v = pc / (K * K), ji = pc - v * K * K;
        T xx[M];
#pragma unroll
        for (int q = 0; q < M; ++q) xx[q] = by[(v * M + q) * K * K + ji];
#pragma unroll
        for (int n = 0; n < K; ++n) {
          T s = 0;
#pragma unroll
          for (int q = 0; q < M; ++q) s += A[q * K + n] * xx[q];
          const int idx = v * SUV + n * K * K + ji;
          cz[idx] = s;
          pAp += double(sU[idx]) * double(s);
        }
      }
      {
        double red[1] = {pAp};
        block_reduce1<NT, 1, 1, (NWK < NWV ? NWK : NWV), (NWK < NWV ? FK : 0)>(red, sRed, half);
        pAp = red[0];
      }
      // vector updates only in the waves that own DOFs
      double zAp = 0.0, rzn = 0.0, rmax = 0.0, alpha = 0.0;
      if (own) {
        T ap[5];
#pragma unroll
        for (int l = 0; l < 5; ++l) ap[l] = cz[l * SUV + tid];
        alpha = rz / pAp;
        const T alphaT = T(alpha);
#pragma unroll
        for (int l = 0; l < 5; ++l) {
          x[l] += alphaT * pv[l];
          r[l] -= alphaT * ap[l];
          rmax = fmax(rmax, fabs(double(r[l])));
        }
        VCP_PRECOND();
#pragma unroll
        for (int l = 0; l < 5; ++l) { zAp += double(z[l]) * double(ap[l]); rzn += double(r[l]) * double(z[l]); }
      }
      {
        double red[3] = {zAp, rzn, rmax};
        block_reduce1<NT, 3, 2, (ND + 63) / 64>(red, sRed, half);
        zAp = red[0]; rzn = red[1]; rmax = red[2];
      }
      iters = it + 1;
      // the reference's stop rule (CG_MassMatrix.cpp:465); the float form
      // stops at 1e-5, a few units of its rounding level
      if (rmax < (kMixed ? VCP_MIXED_CG_TOL : 1e-10) * r0) break;
      if (own) {
        const T beta = T(-alpha * zAp / rz);
#pragma unroll
        for (int l = 0; l < 5; ++l) pv[l] = beta * pv[l] + z[l];
      }
      rz = rzn;
    }
#undef VCP_PRECOND
  }
  if (tid == 0) a.cgIter[e] = iters;
  // ---------------- outputs: R and/or the in-place RK stage update
  double *Re = a.R + (size_t) e * 5 * ND;
  double *Uw = a.U + (size_t) e * 5 * ND;
  const double *U0e = a.U0 + (size_t) e * 5 * ND;
  const double bdt = args.ctl.update ? args.ctl.b * a.scal[kScalDt] : 0.0;
  if (own)
#pragma unroll
    for (int l = 0; l < 5; ++l) {
      const int i = l * ND + tid;
      const double xl = double(x[l]);
      if (!isfinite(xl)) bad = true;
      if (args.ctl.store_res) Re[i] = xl;
      if (args.ctl.update) Uw[i] = (1.0 - args.ctl.a) * Uw[i] + args.ctl.a * U0e[i] - bdt * xl;
    }
  if (bad) atomicOr(a.flags, kFlagNonFinite);
}

template <int K, int M, typename T>
void fill_vol_shape(const DeviceCase &dc, const StageCtl &ctl, VolArgs<K, M, T> &a)
{
  a.ctl = ctl; a.to = dc.to; a.bug = dc.bug_compat;
  for (int i = 0; i < M * K; ++i) { a.op.A[i] = T(dc.opA[i]); a.op.D[i] = T(dc.opD[i]); }
  for (int q = 0; q < K; ++q) {
    a.c0[q] = dc.opC0[q];
    for (int t = 0; t < 4; ++t) a.fvec[t][q] = dc.opF[t][q];
  }
}

template <int K, int M, int NT, typename T>
hipError_t volume_nt_t(const DeviceCase &dc, const StageCtl &ctl, hipStream_t s)
{
  VolArgs<K, M, T> a{};
  a.c = case_dev(dc);
  fill_vol_shape(dc, ctl, a);
  hipLaunchKernelGGL((volume_kernel<K, M, NT, false, T>), dim3(dc.nElem), dim3(NT), 0, s, a);
  return hipGetLastError();
}

template <int K, int M, int NT>
hipError_t volume_nt(const DeviceCase &dc, const StageCtl &ctl, hipStream_t s)
{
  return dc.mixed ? volume_nt_t<K, M, NT, float>(dc, ctl, s) : volume_nt_t<K, M, NT, double>(dc, ctl, s);
}

template <int K, int M, int NT, typename T>
hipError_t batch_volume_nt_t(const BatchGroup &g, const StageCtl &ctl, int w0, int nw, hipStream_t s)
{
  VolArgs<K, M, T> a{};
  a.cases = g.cases; a.work = g.work; a.w0 = w0;
  fill_vol_shape(*g.proto, ctl, a);
  hipLaunchKernelGGL((volume_kernel<K, M, NT, true, T>), dim3(nw), dim3(NT), 0, s, a);
  return hipGetLastError();
}

template <int K, int M, int NT>
hipError_t batch_volume_nt(const BatchGroup &g, const StageCtl &ctl, int w0, int nw, hipStream_t s)
{
  return g.proto->mixed ? batch_volume_nt_t<K, M, NT, float>(g, ctl, w0, nw, s)
                        : batch_volume_nt_t<K, M, NT, double>(g, ctl, w0, nw, s);
}

}  // namespace

template <int K, int M>
hipError_t volume_workgroup(const DeviceCase &dc, int nt, const StageCtl &ctl, hipStream_t s)
{
#define X(k, m, t) if constexpr (K == k && M == m) if (nt == t) return volume_nt<k, m, t>(dc, ctl, s);
  VCP_TILES(X)
#undef X
  return hipErrorInvalidValue;
}

template <int K, int M>
hipError_t batch_volume_workgroup(const BatchGroup &g, int nt, const StageCtl &ctl, int w0, int nw, hipStream_t s)
{
#define X(k, m, t) if constexpr (K == k && M == m) if (nt == t) return batch_volume_nt<k, m, t>(g, ctl, w0, nw, s);
  VCP_TILES(X)
#undef X
  return hipErrorInvalidValue;
}

template hipError_t volume_workgroup<VCP_SHAPE_K, VCP_SHAPE_M>(const DeviceCase &, int, const StageCtl &, hipStream_t);
template hipError_t batch_volume_workgroup<VCP_SHAPE_K, VCP_SHAPE_M>(const BatchGroup &, int, const StageCtl &, int,
                                                                     int, hipStream_t);

}  // namespace vcp
