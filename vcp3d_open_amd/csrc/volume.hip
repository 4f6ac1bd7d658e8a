// Volume residual, face-slot gather, entropy mass-matrix solve and RK stage
// update with one thread per column of integration points (gfx950). Compiled
// once per shape (VCP_SHAPE_K, VCP_SHAPE_M).
//
// Reference behaviour followed (VCP3D_CurviLinear/src/):
//   ElementClass::VolumeResidual          ElementClass.cpp:3809-4533
//   sponge layer / CML sources            ElementClass.cpp:3887-4117, :4450-4489
//   CG_EntropyVarMassMatrix               CG_MassMatrix.cpp:250-504
//   SolverClass::ExecuteTimeSynchronizationStep  SolverClass.cpp:2385-2393
#include "device.hpp"
#include "kernels.hpp"
#include "transforms.hpp"

#include <cstdint>
#include <type_traits>

namespace vcp {
namespace {

// Derivative of the Lagrange polynomials of the Gauss points, C[a][b] =
// l_b'(r_a), centro-antisymmetric: P and Q hold (C[a][b] +- C[a][M-1-b]) / 2
// for a, b < M/2, cm its middle column and mr its middle row (odd M).
template <int M>
struct LineDeriv {
  static constexpr int H = M / 2;
  double P[H * H], Q[H * H], cm[H], mr[H];
};

// The 1D operators as kernel arguments.
template <int K, int M, typename T>
struct ColOps {
  EvenOdd<K, M, T> a;
  EvenOdd<K, M, double> ad;
  LineDeriv<M> l;
  T A[M * K], D[M * K];        // full rows, for the planes
  double Ad[M * K], Dd[M * K];
  double w[M];                 // 1D Gauss weights
  double fvec[4 * K];          // phi(-1), phi(+1), phi'(-1), phi'(+1)
  double c03;                  // phi_0^3, the value of the constant mode
};

template <int K, int M, typename T>
struct ColArgs {
  CaseDev c;                   // single case
  const CaseDev *cases;        // batch: case table and work items
  const WorkItem *work;
  int w0, n;                   // first work item (batch), number of elements
  StageCtl ctl;
  int bug;
  int oW2, oCentre, oFace;     // offsets in the table block: w2, basis at the element centre, face vectors
  ColOps<K, M, T> op;
};

// derivative along a line of M point values, in place; TRANS: its transpose.
// In double in both forms: the nodal derivative cancels the constant part of
// the fluxes, which single precision would round first.
template <int M, bool TRANS>
__device__ __forceinline__ void line_deriv(cptr<LineDeriv<M>> op, double (&x)[M])
{
  constexpr int H = M / 2;
  double s[H], d[H];
#pragma unroll
  for (int b = 0; b < H; ++b) { s[b] = x[b] + x[M - 1 - b]; d[b] = x[b] - x[M - 1 - b]; }
  const double xm = x[H];
  double ym = 0.0;
  if constexpr (M % 2) {
    ym = (TRANS ? op->cm[0] : op->mr[0]) * d[0];
#pragma unroll
    for (int b = 1; b < H; ++b) ym += (TRANS ? op->cm[b] : op->mr[b]) * d[b];
  }
#pragma unroll
  for (int a = 0; a < H; ++a) {
    // forward: u from s with P, v from d with Q; the transpose swaps the roles
    double u = (TRANS ? op->Q[a] : op->P[a * H]) * s[0];
    double v = (TRANS ? op->P[a] : op->Q[a * H]) * d[0];
#pragma unroll
    for (int b = 1; b < H; ++b) {
      u += (TRANS ? op->Q[b * H + a] : op->P[a * H + b]) * s[b];
      v += (TRANS ? op->P[b * H + a] : op->Q[a * H + b]) * d[b];
    }
    if constexpr (M % 2) u += (TRANS ? op->mr[a] : op->cm[a]) * xm;
    x[a] = v + u;
    x[M - 1 - a] = v - u;
  }
  if constexpr (M % 2) x[H] = ym;
}

// ------------------------------------------------------ group reductions
// A group is the G threads of one element: 16 or 32 lanes of a wave, a wave,
// or two waves. Sum (the first NS values) or max of non-negative values; the
// result is returned to every thread. Two-wave groups exchange their partial
// results through alternating halves of red, with one barrier.
template <int G, int NV, int NS>
__device__ __forceinline__ void group_reduce(double (&v)[NV], double *red, int &half)
{
#pragma unroll
  for (int q = 0; q < NV; ++q) v[q] = q < NS ? lanes_reduce<G, false>(v[q]) : lanes_reduce<G, true>(v[q]);
  if constexpr (G > 64) {
    constexpr int NW = G / 64;
    static_assert(NV <= 5, "a half of red holds five values per wave");
    double *buf = red + half * 5 * NW;
    const int wid = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
#pragma unroll
      for (int q = 0; q < NV; ++q) buf[wid * NV + q] = v[q];
    group_sync<G>();
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      double s = buf[q];
#pragma unroll
      for (int w = 1; w < NW; ++w) s = q < NS ? s + buf[w * NV + q] : fmax(s, buf[w * NV + q]);
      v[q] = s;
    }
    half ^= 1;
  }
}

// -------------------------------------------------------------- layout
// Halves of a column in FP64 and float without regard to the number of
// elements. A column's points are handled by one thread, or by one thread of
// each half of the group: planes 0 .. (M-1)/2 by the first half, the others,
// from the last one down, by the second. The whole column in one thread needs a
// third fewer instructions (the even-odd transforms), but 10 M values and the
// solve's vectors must fit 256 registers: beyond K = 5 in FP64 they spill ((6, 8)
// at 16^3 halved: 0.81 of the whole column's time; (5, 7) at 32^3: 1.32 of it). At K = 3 cases of few elements take halves too (volume_kind): they
// fill twice as many waves, each with half of the column's serial work.
template <int K, typename T>
constexpr int kColHalves = K >= 6 && sizeof(T) == 8 ? 2 : 1;

template <int K, int M, typename T, int HALVES>
struct ColShape {
  static constexpr int ND = K * K * K, NI = M * M * M, N2 = M * M;
  static constexpr int H = HALVES;
  static constexpr int LH = N2 <= 16 ? 16 : N2 <= 32 ? 32 : N2 <= 64 ? 64 : 128;   // threads per half
  static constexpr int G = H * LH;                       // threads per element
  static constexpr int NE = G < 64 ? 64 / G : 1;         // elements per workgroup
  static constexpr int NT = G < 64 ? 64 : G;
  // waves per SIMD to compile for: at three (168 registers) every shape whose
  // LDS lets three run spills, between 4 registers ((4, 6), float) and 240
  // ((7, 9)); measured at (4, 5), where 135 spill: 16^3 0.164 against 0.081 ms
  static constexpr int WAVES = 2;
  static constexpr int HP = H == 1 ? M : (M + 1) / 2;    // planes of a thread (the second half of an odd M: one less)
  static constexpr bool kInWave = H == 2 && LH < 64;     // the halves share a wave
  // pitches, odd so that lanes a pitch apart fall into different banks
  static constexpr int KP = K | 1, MP = M | 1, NP = N2 | 1;
  // the planes' lines of one variable, PL apart: at M = 8 a value more than
  // their length, without which they collide in the banks (1.4 % of the launch
  // at (6, 8); at M = 4 and 6 the gaps cost more, 3 and 1 %)
  static constexpr int PL = M % 8 ? M : M + 1, LP = (M * PL) | 1;
  // half-transformed lines of one (variable, k): K lines without a gap at
  // K >= 6 (lines a pitch apart throughout: with a gap of one the 64 lanes of
  // (6, 8) collide four deep), otherwise an odd number for the reads across them
  static constexpr int YB = K >= 6 ? K * MP : (K * MP) | 1;
  static constexpr int UV = K * K * KP;                  // one variable of the modal state
  // LDS of one element, in T: B holds the modal state or the lines of the
  // planes of points, X the column coefficients
  // [variable][mode k][point j][point i], Y the lines between the two 1D passes along i and j
  // (in X itself where a region of their own would cost a workgroup per CU)
  // X holds doubles between the planes and the right-hand side in both forms:
  // a residual is a difference of large fluxes
  static constexpr int W = (int) (sizeof(double) / sizeof(T));
  static constexpr int X = 5 * K * NP * W;
  static constexpr int NL = 10 * H * LP;                 // the planes' lines, in double
  static constexpr int B = (cmax(5 * UV, NL * W) + 1) / 2 * 2;
  static constexpr int NY = 5 * K * YB * W;
  static constexpr int kOther = 8 * (NE * 12 + (G > 64 ? 10 * (G / 64) : 1) + 4 * K + (NE == 1 ? 1 : NE * 45));   // the other LDS arrays
  static constexpr int WGMAX = WAVES * 4 / (NT / 64);    // workgroups per CU by registers
  static constexpr bool SEPY = (NE * (X + B + NY) * (int) sizeof(T) + kOther) * WGMAX <= 160 * 1024;
  static constexpr int S = (X + B + (SEPY ? NY : 0) + 1) / 2 * 2;   // whole doubles
  static_assert(NY <= X && 5 * UV <= 5 * K * NP, "the half-transformed lines and A p fit X");
  static constexpr int NDL = (ND + G - 1) / G;           // modes per thread
  static constexpr int RA = (5 * K * K + G - 1) / G;     // lines along i per thread
  static constexpr int RB = (5 * K * M + G - 1) / G;     // lines along j per thread
};

// modal state (pitch KP) -> column coefficients: along i, then along j
template <int K, int M, class S, typename T>
__device__ __forceinline__ void modes_to_columns(const EvenOdd<K, M, T> &A, const T *u, T *X, T *Y, int t)
{
#pragma unroll
  for (int r = 0; r < S::RA; ++r) {
    const int l = t + r * S::G;                          // line (variable k j)
    if (l < 5 * K * K) {
      T c[K], o[M];
#pragma unroll
      for (int q = 0; q < K; ++q) c[q] = u[l * S::KP + q];
      to_points(A, c, o);
      T *y = Y + (l / K) * S::YB + (l % K) * S::MP;
#pragma unroll
      for (int p = 0; p < M; ++p) y[p] = o[p];
    }
  }
  group_sync<S::G>();
  T in[S::RB][K];
#pragma unroll
  for (int r = 0; r < S::RB; ++r) {
    const int l = t + r * S::G, i = l / (5 * K), vk = l - i * (5 * K);
    if (l < 5 * K * M)
#pragma unroll
      for (int q = 0; q < K; ++q) in[r][q] = Y[vk * S::YB + q * S::MP + i];
  }
  if constexpr (!S::SEPY) group_sync<S::G>();
#pragma unroll
  for (int r = 0; r < S::RB; ++r) {
    const int l = t + r * S::G, i = l / (5 * K), vk = l - i * (5 * K);
    if (l < 5 * K * M) {
      T o[M];
      to_points(A, in[r], o);
#pragma unroll
      for (int p = 0; p < M; ++p) X[vk * S::NP + p * M + i] = o[p];
    }
  }
  group_sync<S::G>();
}

// column coefficients -> modes (pitch KP) in dst (X itself, or the B region):
// along j, then along i; add(l, m) is applied to the modes m of line l
template <int K, int M, class S, bool TO_X, typename T, typename TD, class ADD>
__device__ __forceinline__ void columns_to_modes(const EvenOdd<K, M, T> &A, T *X, T *Y, TD *dst, int t, ADD add)
{
  T o[S::RB][K];
#pragma unroll
  for (int r = 0; r < S::RB; ++r) {
    const int l = t + r * S::G, i = l / (5 * K), vk = l - i * (5 * K);
    if (l < 5 * K * M) {
      T x[M];
#pragma unroll
      for (int p = 0; p < M; ++p) x[p] = X[vk * S::NP + p * M + i];
      to_modes(A, x, o[r]);
    }
  }
  if constexpr (!S::SEPY) group_sync<S::G>();
#pragma unroll
  for (int r = 0; r < S::RB; ++r) {
    const int l = t + r * S::G, i = l / (5 * K), vk = l - i * (5 * K);
    if (l < 5 * K * M)
#pragma unroll
      for (int q = 0; q < K; ++q) Y[vk * S::YB + q * S::MP + i] = o[r][q];
  }
  group_sync<S::G>();
  T m[S::RA][K];
#pragma unroll
  for (int r = 0; r < S::RA; ++r) {
    const int l = t + r * S::G;
    if (l < 5 * K * K) {
      const T *y = Y + (l / K) * S::YB + (l % K) * S::MP;
      T x[M];
#pragma unroll
      for (int p = 0; p < M; ++p) x[p] = y[p];
      to_modes(A, x, m[r]);
      add(l, m[r]);
    }
  }
  if constexpr (TO_X && !S::SEPY) group_sync<S::G>();
#pragma unroll
  for (int r = 0; r < S::RA; ++r) {
    const int l = t + r * S::G;
    if (l < 5 * K * K)
#pragma unroll
      for (int q = 0; q < K; ++q) dst[l * S::KP + q] = TD(m[r][q]);
  }
  group_sync<S::G>();
}

// One thread group of G threads per element. In each half of the group,
// thread tl < M^2 owns the column of points (j, i) = (tl / M, tl % M) over the
// half's planes; in the whole group, thread t owns the modes t, t + G, ... of
// all five variables.
//
// The workgroup form (volume_kernel) is held by its ~20 workgroup barriers and
// by LDS traffic: every 1D contraction of the solve goes through LDS. Here a
// thread contracts its whole column along k, applies dU/dV (or the fluxes) and
// contracts back in registers, so an iteration of the solve moves 39 KB of LDS
// data per element instead of 132 KB at (5, 7), and up to K = 5 the element's
// wave needs no barrier at all. What bounds it: the vector unit's issue and
// latency at two waves per SIMD (it issues 45-60 % of the time), which the
// registers set: scratch costs most of all (20 spilled registers cost 30 % at
// (5, 7)), so the scheduling barriers below keep the phases apart.
// Measured on one box, workgroup / column form, volume launch of a residual of a
// curvilinear Taylor-Green case:
//   FP64   (3, 4) 18^3 87 / 47 us    (4, 5) 16^3 109 / 66    (4, 6) 14^3 129 / 81
//          (5, 7) 32^3 1405 / 937   (6, 8) 16^3 540 / 272   (7, 9) 14^3 641 / 408
//   float  (3, 4) 56 / 33   (4, 5) 63 / 43   (4, 6) 87 / 60   (5, 7) 1021 / 676
//          (6, 8) 229 / 182   (7, 9) 365 / 207
template <int K, int M, bool BATCH, bool FULL, typename T, int HALVES>
__global__ __launch_bounds__((ColShape<K, M, T, HALVES>::NT), (ColShape<K, M, T, HALVES>::WAVES))
void volume_cols_kernel(ColArgs<K, M, T> args_)
{
  using S = ColShape<K, M, T, HALVES>;
  constexpr bool kMixed = sizeof(T) == 4;
  constexpr int G = S::G, NE = S::NE, ND = S::ND, NI = S::NI, N2 = S::N2, NP = S::NP, H = S::H, HP = S::HP;
  constexpr int LH = S::LH;
  constexpr bool kInWave = S::kInWave;
  constexpr bool kUniform = NE == 1;            // one element per workgroup
  // a whole column in FP64 fills the registers: the products of the point
  // state stay inside the solve's loop, and its solution is kept in LDS
  constexpr bool kTight = H == 1 && !kMixed && K >= 5;
  constexpr int SX = kTight ? S::NDL * 5 * G : 0;
  __shared__ __align__(8) T lds[NE * S::S + SX];
  __shared__ double sPre[NE][7];                // preconditioner of the solve
  __shared__ double sMean[NE][5];               // float form: mode 0 of each variable
  __shared__ double sRed[G > 64 ? 2 * 5 * (G / 64) : 1];
  __shared__ double sFv[4 * K];                 // phi(-1), phi(+1), phi'(-1), phi'(+1)
  __shared__ double sCm[kUniform ? 1 : NE][kUniform ? 1 : 45];   // metric of points 0..4 (bug)
  typedef const __attribute__((address_space(4))) ColArgs<K, M, T> *ArgP;
  const ArgP args = (ArgP) __builtin_amdgcn_kernarg_segment_ptr();
  // operators: laundering the pointer keeps one phase's scalar loads out of the next
  auto ops = [&]() { auto p = &args->op; asm volatile("" : "+s"(p)); return p; };

  const int tid = threadIdx.x, sub = G < 64 ? tid / G : 0, t = G < 64 ? tid % G : tid;
  const int h = H == 1 ? 0 : kInWave ? t / LH : __builtin_amdgcn_readfirstlane(tid / LH), tl = H == 1 ? t : t - h * LH;
  const int item = blockIdx.x * NE + sub;
  const bool inRange = kUniform || item < args->n;
  // the case part of the arguments: its fields are read where they are used
  // (scalar loads; from the case table, which does not change while a step's
  // launches run, in a batch), so that they take no registers in between
  constexpr bool kLaneCase = BATCH && !kUniform;
  using CaseP = typename std::conditional<kLaneCase, const CaseDev *, cptr<CaseDev>>::type;
  CaseP a;
  int e;
  bool live = inRange;
  if constexpr (BATCH) {
    const WorkItem w = args->work[args->w0 + (inRange ? item : 0)];
    e = w.e;
    if constexpr (kUniform) e = __builtin_amdgcn_readfirstlane(e);
    const CaseDev *cp = args->cases + (kUniform ? __builtin_amdgcn_readfirstlane(w.c) : w.c);
    a = (CaseP) (uintptr_t) cp;
    live = live && glob(cp->flags)[kWordActive] != 0;
    if (!__any(live)) return;
  } else {
    a = &args->c;
    e = inRange ? item : 0;
  }
  auto fresh = [&]() { if constexpr (!kLaneCase) asm volatile("" : "+s"(a)); };
  T *const B = lds + sub * S::S, *const X = B + S::B, *const Y = S::SEPY ? X + S::X : X;
  double *const XD = (double *) X;
  T *const XS = lds + S::S + t;                 // kTight: x of mode slot s, variable l at (s * 5 + l) * G
  const auto Ue = glob((const double *) a->U) + (size_t) e * 5 * ND;
  const auto vg = glob(a->vgeo) + (size_t) e * kVolGeo * NI;
  int sp = FULL && a->spIdx ? glob(a->spIdx)[e] : -1;
  if constexpr (kUniform) sp = __builtin_amdgcn_readfirstlane(sp);
  const bool act = tl < N2;
  const int col = act ? tl : 0, ci = col % M, cj = col / M;
  constexpr int PL = S::PL, LP = S::LP;
  const int line = cj * PL + ci, lineT = ci * PL + cj;   // its place in the planes' lines along i and j
  const T sgn = T(h ? -1 : 1);
  const double sgnD = sgn;
  int half = 0;
  // this thread's points of a column from its coefficients, and back (partial
  // sums over the thread's points): row p of A serves plane p, and with the
  // odd modes' sign changed plane M - 1 - p
  using E = EvenOdd<K, M, T>;
  auto col_points = [&](const E &A, const T (&c)[K], T (&o)[HP]) {
    if constexpr (H == 1) {
      to_points(A, c, o);
    } else {
      T co[E::KO];
#pragma unroll
      for (int q = 0; q < E::KO; ++q) co[q] = sgn * c[2 * q + 1];
#pragma unroll
      for (int p = 0; p < HP; ++p) {
        T v = A.e[p * E::KE] * c[0];
#pragma unroll
        for (int q = 1; q < E::KE; ++q) v += A.e[p * E::KE + q] * c[2 * q];
        if (p < E::HO)
#pragma unroll
          for (int q = 0; q < E::KO; ++q) v += A.o[p * E::KO + q] * co[q];
        o[p] = v;
      }
    }
  };
  auto col_modes = [&](const E &A, const T (&x)[HP], T (&c)[K]) {
    if constexpr (H == 1) {
      to_modes(A, x, c);
    } else {
#pragma unroll
      for (int q = 0; q < E::KE; ++q) {
        T v = A.e[q] * x[0];
#pragma unroll
        for (int p = 1; p < HP; ++p) v += A.e[p * E::KE + q] * x[p];
        c[2 * q] = v;
      }
#pragma unroll
      for (int q = 0; q < E::KO; ++q) {
        T v = A.o[q] * x[0];
#pragma unroll
        for (int p = 1; p < E::HO; ++p) v += A.o[p * E::KO + q] * x[p];
        c[2 * q + 1] = sgn * v;
      }
    }
  };
  // column coefficients into X, summed over the halves: each half stores the
  // variables that the other one adds to
  auto store_columns = [&](const auto (&c)[5][K], auto *X) {
    if constexpr (H == 1) {
      if (act)
#pragma unroll
        for (int v = 0; v < 5; ++v)
#pragma unroll
          for (int q = 0; q < K; ++q) X[(v * K + q) * NP + tl] = c[v][q];
    } else {
      if (act) {
        if (h == 0) {
#pragma unroll
          for (int v = 3; v < 5; ++v)
#pragma unroll
            for (int q = 0; q < K; ++q) X[(v * K + q) * NP + tl] = c[v][q];
          asm volatile("; first half");   // the two branches stay apart: merged, c would be indexed at run time
        } else {
#pragma unroll
          for (int v = 0; v < 3; ++v)
#pragma unroll
            for (int q = 0; q < K; ++q) X[(v * K + q) * NP + tl] = c[v][q];
        }
      }
      group_sync<G>();
      if (act) {
        if (h == 0) {
#pragma unroll
          for (int v = 0; v < 3; ++v)
#pragma unroll
            for (int q = 0; q < K; ++q) X[(v * K + q) * NP + tl] += c[v][q];
          asm volatile("; first half");
        } else {
#pragma unroll
          for (int v = 3; v < 5; ++v)
#pragma unroll
            for (int q = 0; q < K; ++q) X[(v * K + q) * NP + tl] += c[v][q];
        }
      }
    }
    group_sync<G>();
  };

  // ---------------- modal state, element-centre preconditioner
  {
    constexpr int NIT = (5 * ND + G - 1) / G;
    double uu[NIT];
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int i = t + it * G;
      uu[it] = Ue[i < 5 * ND ? i : 0];
    }
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int i = t + it * G;
      if (i < 5 * ND) {
        const int v = i / ND, d = i - v * ND;
        T x = T(uu[it]);
        if (kMixed && d == 0) { sMean[sub][v] = uu[it]; x = T(0); }
        B[v * S::UV + (d / K) * S::KP + d % K] = x;
      }
    }
  }
  for (int i = tid; i < 4 * K; i += S::NT) sFv[i] = glob(a->tables)[args->oFace + i];
  const double elemJac = glob(a->econst)[(size_t) e * kElemConst + 3];
  if constexpr (!kUniform)
    if (args->bug)
      for (int i = t; i < 45; i += G) sCm[sub][i] = vg[(1 + i % 9) * NI + i / 9];
  group_sync<G>();
  double meanPt[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  if constexpr (kMixed)
#pragma unroll
    for (int v = 0; v < 5; ++v) meanPt[v] = args->op.c03 * sMean[sub][v];
  {
    double Vc[5] = {0, 0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < S::NDL; ++s) {
      const int d = t + s * G;
      if (d < ND) {
        const double b = glob(a->tables)[args->oCentre + d];
#pragma unroll
        for (int v = 0; v < 5; ++v) Vc[v] += b * double(B[v * S::UV + (d / K) * S::KP + d % K]);
      }
    }
    group_reduce<G, 5, 5>(Vc, sRed, half);
#pragma unroll
    for (int v = 0; v < 5; ++v) Vc[v] += meanPt[v];
    double rho, u, v, w, p, eKin;
    ent2prim(Vc, rho, u, v, w, p, eKin);
    const double JacInv = 8.0 / elemJac, pInv = 1.0 / p;
    if (t == 0) {
      // dV/dU / Jbar = a1 b b^T + pInv (...), b = (eKin, -u, -v, -w, 1)
      double *pr = sPre[sub];
      pr[0] = eKin; pr[1] = u; pr[2] = v; pr[3] = w; pr[4] = JacInv * kGm1 * rho * pInv * pInv;
      pr[5] = JacInv * pInv; pr[6] = JacInv * (kGam / kGm1 / rho);
    }
  }
  modes_to_columns<K, M, S, T>(scalar_op<K, M, T>(&ops()->a), B, X, Y, t);

  // ---------------- the planes of points: state and gradients, fluxes, and
  // their contraction along k; the in-plane derivatives go through LDS lines
  // of the half
  double acc[5][K];
#pragma unroll
  for (int v = 0; v < 5; ++v)
#pragma unroll
    for (int q = 0; q < K; ++q) acc[v][q] = 0;
  double *const PB = (double *) B + h * 10 * LP;
  const double w2 = glob(a->tables)[args->oW2 + col];
  const double factHF = a->mu * kGam / kPrLam;
  const double lenLES = FULL && a->sgs ? glob(a->econst)[(size_t) e * kElemConst + kElemLenLES] : 0.0;
  const bool cml = FULL && sp >= 0 && a->cml;
  double mach2 = 0.0, evMax = 0.0;
  const int np = H == 1 ? M : h ? M / 2 : (M + 1) / 2;
  constexpr bool kEqual = LH > 64 || kInWave;      // the halves share barriers or a wave: equal trips
  // operator rows of plane k: of plane pl, with a change of sign in the odd
  // modes (of D in the even ones) for the second half, where the halves share
  // a wave
  auto row = [&](int pl, int k) { return kInWave ? pl : k; };
  // entropy variables and their derivatives along k at this thread's point of
  // plane k
  auto plane_values = [&](int rowK, T (&V)[5], T (&Gt)[5]) {
    const auto op = ops();
    cptr<T> Ak = op->A + rowK * K, Dk = op->D + rowK * K;
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      T c[K];
#pragma unroll
      for (int q = 0; q < K; ++q) c[q] = X[(v * K + q) * NP + col];
      T s = Ak[0] * c[0], d = Dk[1] * c[1];
#pragma unroll
      for (int q = 1; q < K; ++q) {
        const T cs = kInWave ? sgn * c[q] : c[q];
        s += Ak[q] * (q % 2 ? cs : c[q]);
        if (q > 1) d += Dk[q] * (q % 2 ? c[q] : cs);
      }
      V[v] = s; Gt[v] = d;
    }
  };
  // derivative (transposed: TRANS) of lines [0, NL) of the half, in place
  auto derive_lines = [&](auto nl, auto trans) {
    constexpr int NL = decltype(nl)::value;
    const auto ld = &ops()->l;
#pragma unroll
    for (int r = 0; r < (NL + LH - 1) / LH; ++r) {
      const int l = tl + r * LH;
      if (l < NL) {
        double *x = PB + (l / M) * LP + (l % M) * PL;
        double y[M];
#pragma unroll
        for (int p = 0; p < M; ++p) y[p] = x[p];
        line_deriv<M, decltype(trans)::value>(ld, y);
#pragma unroll
        for (int p = 0; p < M; ++p) x[p] = y[p];
      }
    }
  };
  // Cartesian gradient of variable v from its parametric derivatives
  auto cartesian = [&](int v, double gr, double gs, double gt, const double (&cur)[kVolGeo], double (&g)[3][5]) {
    cptr<double> vs = (cptr<double>) (uintptr_t) (vg + NI);
    if (args->bug) {
#pragma unroll
      for (int x = 0; x < 3; ++x) {
        if constexpr (kUniform)
          g[x][v] = gr * vs[x * NI + v] + gs * vs[(3 + x) * NI + v] + gt * vs[(6 + x) * NI + v];
        else
          g[x][v] = gr * sCm[sub][v * 9 + x] + gs * sCm[sub][v * 9 + 3 + x] + gt * sCm[sub][v * 9 + 6 + x];
      }
    } else {
#pragma unroll
      for (int x = 0; x < 3; ++x) g[x][v] = gr * cur[1 + x] + gs * cur[4 + x] + gt * cur[7 + x];
    }
  };
  // ---------------- sponge, matching-layer and body-force sources, in planes
  // of their own ahead of the fluxes': beside the fluxes they spilled 40
  // registers in every element, of those outside the sponge too; here (4, 5)
  // spills 2 (FP64) or 13 (24 in a batch), (7, 9) 4 or 10, the other shapes at
  // most 3. Volume launch of the 48 x 24 x 24 open box at (5, 7), 8 of 48 element
  // layers in the sponge: 888 us beside the fluxes, 718 us here; 18^3 (3, 4) with
  // WALE, which these sources spilled as well: 57 / 53 us.
  if constexpr (FULL)
    if (sp >= 0 || a->bfBuf) {
#pragma unroll 1
      for (int pl = 0; pl < (kEqual ? HP : np); ++pl) {
        const bool valid = !kEqual || pl < np;
        const int k = H == 2 && h ? M - 1 - pl : pl, m = k * N2 + col;
        double cur[kVolGeo];
#pragma unroll
        for (int q = 0; q < kVolGeo; ++q) cur[q] = vg[(unsigned) (q * NI + m)];
        T V[5], Gt[5];
        plane_values(row(pl, k), V, Gt);
        double g[3][5];
        if (cml) {
          if (act)
#pragma unroll
            for (int v = 0; v < 5; ++v) { PB[v * LP + line] = V[v]; PB[(5 + v) * LP + lineT] = V[v]; }
          group_sync<LH>();
          derive_lines(std::integral_constant<int, 10 * M>{}, std::false_type{});
          group_sync<LH>();
#pragma unroll
          for (int v = 0; v < 5; ++v) cartesian(v, PB[v * LP + line], PB[(5 + v) * LP + lineT], Gt[v], cur, g);
        }
        double Vp[5];
#pragma unroll
        for (int v = 0; v < 5; ++v) Vp[v] = double(V[v]) + meanPt[v];
        const EntState st = ent_state(Vp);
        const double wJ = w2 * args->op.w[row(pl, k)] * cur[0], weight = -wJ;
        double src[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        if (sp >= 0) {
          // sponge damping sigma J w (U - U_target) and CML sources
          // (ElementClass.cpp:4450-4489, :3887-4117)
          const auto fn = glob(a->dampFn) + (size_t) sp * 3 * NI, ds = glob(a->dampState) + (size_t) sp * 5 * NI;
          const double sigma = wJ * (fn[m] + fn[NI + m] + fn[2 * NI + m]);
          src[0] = sigma * (st.rho - ds[m]);
          src[1] = sigma * (st.rho * st.u - ds[NI + m]);
          src[2] = sigma * (st.rho * st.v - ds[2 * NI + m]);
          src[3] = sigma * (st.rho * st.w - ds[3 * NI + m]);
          src[4] = sigma * (st.p * kInvGm1 + st.rho * st.ek - ds[4 * NI + m]);
          if (cml) {
            const auto cf = glob(a->spCoef) + (size_t) sp * 8;
            const double wgt[3] = {weight * cf[0] * fn[m], weight * cf[1] * fn[NI + m], weight * cf[2] * fn[2 * NI + m]};
            const double nsg[3] = {cf[3], cf[4], cf[5]};
            cml_source(Vp, g[0], g[1], g[2], wgt, nsg, src);
          }
        }
        if (a->bfBuf) {
          // body force per unit volume (ElementClass.cpp:4492-4523): -w J f on
          // the momentum and -w J u.f on the energy equation
          const double bx = a->fbody[0], by = a->fbody[1], bz = a->fbody[2];
          src[1] += weight * bx; src[2] += weight * by; src[3] += weight * bz;
          src[4] += weight * (st.u * bx + st.v * by + st.w * bz);
        }
        if (valid) {
          cptr<double> Ak = ops()->Ad + row(pl, k) * K;
#pragma unroll
          for (int v = 0; v < 5; ++v)
#pragma unroll
            for (int q = 0; q < K; ++q) acc[v][q] += Ak[q] * (kInWave && q % 2 ? sgnD * src[v] : src[v]);
        }
        group_sync<LH>();
      }
    }
#pragma unroll 1
  for (int pl = 0; pl < (kEqual ? HP : np); ++pl) {
    const bool valid = !kEqual || pl < np;
    const int k = H == 2 && h ? M - 1 - pl : pl;
    double cur[kVolGeo];
#pragma unroll
    for (int q = 0; q < kVolGeo; ++q) cur[q] = vg[(unsigned) (q * NI + k * N2 + col)];
    T V[5], Gt[5];
    plane_values(row(pl, k), V, Gt);
    // lines along i (slots 0..3) and along j (4..7) of variables 1..4
    if (act)
#pragma unroll
      for (int v = 0; v < 4; ++v) { PB[v * LP + line] = V[1 + v]; PB[(4 + v) * LP + lineT] = V[1 + v]; }
    group_sync<LH>();
    derive_lines(std::integral_constant<int, 8 * M>{}, std::false_type{});
    group_sync<LH>();
    double g[3][5];                                   // Cartesian gradients
#pragma unroll
    for (int v = 1; v < 5; ++v) cartesian(v, PB[(v - 1) * LP + line], PB[(v + 3) * LP + lineT], Gt[v], cur, g);
    double Ft[5];
    {
      double Fr[5], Fs[5];
      double Vp[5];
#pragma unroll
      for (int v = 0; v < 5; ++v) Vp[v] = double(V[v]) + meanPt[v];
      const double *gx = g[0], *gy = g[1], *gz = g[2];
      const EntState st = ent_state(Vp);
      const double rho = st.rho, u = st.u, v = st.v, w = st.w, p = st.p, eKin = st.ek, V4Inv = -st.r;
      const double rE = p * kInvGm1 + rho * eKin;
      const double dudx = -V4Inv * (gx[1] + u * gx[4]), dudy = -V4Inv * (gy[1] + u * gy[4]), dudz = -V4Inv * (gz[1] + u * gz[4]);
      const double dvdx = -V4Inv * (gx[2] + v * gx[4]), dvdy = -V4Inv * (gy[2] + v * gy[4]), dvdz = -V4Inv * (gz[2] + v * gz[4]);
      const double dwdx = -V4Inv * (gx[3] + w * gx[4]), dwdy = -V4Inv * (gy[3] + w * gy[4]), dwdz = -V4Inv * (gz[3] + w * gz[4]);
      const double fe = V4Inv * V4Inv * kInvGm1;
      const double dedx = fe * gx[4], dedy = fe * gy[4], dedz = fe * gz[4];
      if (args->ctl.monitor && act && valid) mach2 = fmax(mach2, (u * u + v * v + w * w) * (-Vp[4] * (1.0 / kGam)));
      const double ru = rho * u, rv = rho * v, rw = rho * w;
      // eddy viscosity of the SGS model (ElementClass.cpp:4268-4287, :4305-4306)
      // in the total viscosity and heat-flux factor (:4339-4342)
      double mu = a->mu, fhT = factHF;
      if constexpr (FULL)
        if (a->sgs != kSgsNone) {
          const double Gv[3][3] = {{dudx, dudy, dudz}, {dvdx, dvdy, dvdz}, {dwdx, dwdy, dwdz}};
          const double ev = eddy_viscosity(a->sgs, lenLES, rho, Gv);
          if (act && valid) evMax = fmax(evMax, ev);
          mu = a->mu + ev;
          fhT = a->mu * (kGam / kPrLam) + ev * (kGam / kPrTurb);
        }
      const double divV = kLamOverMu * (dudx + dvdy + dwdz);
      const double txx = mu * (2.0 * dudx + divV), tyy = mu * (2.0 * dvdy + divV), tzz = mu * (2.0 * dwdz + divV);
      const double txy = mu * (dudy + dvdx), txz = mu * (dudz + dwdx), tyz = mu * (dvdz + dwdy);
      const double qx = -fhT * dedx, qy = -fhT * dedy, qz = -fhT * dedz;
      const double fx[5] = {ru, ru * u - txx + p, rv * u - txy, rw * u - txz, (rE + p) * u - (u * txx + v * txy + w * txz - qx)};
      const double fy[5] = {rv, ru * v - txy, rv * v - tyy + p, rw * v - tyz, (rE + p) * v - (u * txy + v * tyy + w * tyz - qy)};
      const double fz[5] = {rw, ru * w - txz, rv * w - tyz, rw * w - tzz + p, (rE + p) * w - (u * txz + v * tyz + w * tzz - qz)};
      const double wJ = w2 * args->op.w[row(pl, k)] * cur[0], weight = -wJ;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const double mx = weight * cur[1 + 3 * d], my = weight * cur[2 + 3 * d], mz = weight * cur[3 + 3 * d];
#pragma unroll
        for (int l = 0; l < 5; ++l) {
          const double F = fx[l] * mx + fy[l] * my + fz[l] * mz;
          if (d == 0) Fr[l] = F;
          else if (d == 1) Fs[l] = F;
          else Ft[l] = F;
        }
      }
      // in-plane fluxes: lines along i of the r fluxes (slots 0..4) and along j
      // of the s fluxes (5..9), contracted with the transposed derivative; they
      // overwrite the gradients once every thread has read its own
      group_sync<LH>();
      if (act)
#pragma unroll
        for (int l = 0; l < 5; ++l) { PB[l * LP + line] = Fr[l]; PB[(5 + l) * LP + lineT] = Fs[l]; }
    }
    group_sync<LH>();
    derive_lines(std::integral_constant<int, 10 * M>{}, std::true_type{});
    group_sync<LH>();
    if (valid) {
      const auto op = ops();
      cptr<double> Ak = op->Ad + row(pl, k) * K, Dk = op->Dd + row(pl, k) * K;
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        const double s = PB[v * LP + line] + PB[(5 + v) * LP + lineT];
#pragma unroll
        for (int q = 0; q < K; ++q) {
          acc[v][q] += Ak[q] * (kInWave && q % 2 ? sgnD * s : s);
          if (q > 0) acc[v][q] += Dk[q] * (kInWave && q % 2 == 0 ? sgnD * Ft[v] : Ft[v]);
        }
      }
    }
    group_sync<LH>();
  }

  // ---------------- w J rho, velocity and p / rho at the thread's points, for
  // the weighted dU/dV of the solve; in the float form w J p and the matrix's
  // last entry in place of p / rho, formed in double and rounded once
  constexpr int NPR = kMixed ? 6 : 5;
  T pr[HP][NPR];
  {
    double J[HP];
    T V[5][HP];
#pragma unroll
    for (int p = 0; p < HP; ++p) J[p] = vg[(unsigned) ((H == 2 && h ? M - 1 - p : p) * N2 + col)];
    const auto op = ops();
    const E A = scalar_op<K, M, T>(&op->a);
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      T c[K];
#pragma unroll
      for (int q = 0; q < K; ++q) c[q] = X[(v * K + q) * NP + col];
      col_points(A, c, V[v]);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int p = 0; p < HP; ++p) {
      double Vp[5];
#pragma unroll
      for (int l = 0; l < 5; ++l) Vp[l] = double(V[l][p]) + meanPt[l];
      const EntState st = ent_state(Vp);
      // the middle plane of an odd M belongs to the first half
      const bool mine = H == 1 || M % 2 == 0 || p < HP - 1 || h == 0;
      if constexpr (kMixed) {
        const double wr = mine ? w2 * op->w[p] * J[p] * st.rho : 0.0, P = wr * st.r, Et = st.r * kInvGm1 + st.ek;
        pr[p][0] = T(wr);
        pr[p][4] = T(P);
        pr[p][5] = T(wr * Et * Et + P * (Et + st.ek));
      } else {
        pr[p][0] = mine ? T(w2 * op->w[p] * J[p] * st.rho) : T(0);
        pr[p][4] = T(st.r);
      }
      pr[p][1] = T(st.u); pr[p][2] = T(st.v); pr[p][3] = T(st.w);
#pragma unroll
      for (int l = 0; l < NPR; ++l) asm volatile("" : "+v"(pr[p][l]));
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  group_sync<G>();
  // ---------------- the planes' contraction -> modes, with the six face
  // contributions: each face slot holds the value and normal-derivative
  // coefficient planes over its two tangential axes [0|1][variable][slow][fast],
  // times the face vectors phi(r_f), phi'(r_f) at the mode's normal index.
  // Thread (variable, k, j) adds them to its line of modes along i.
  fresh();
  store_columns(acc, XD);
  bool bad = false;
  {
    const auto fr = glob((const double *) a->faceRes) + (size_t) e * 6 * 10 * K * K;
    cptr<double> fv = args->op.fvec;
    auto add = [&](int l, double (&s)[K]) {
      const int v = l / (K * K), kj = l - v * K * K, kk = kj / K, jj = kj - kk * K;
#pragma unroll
      for (int side = 0; side < 2; ++side) {
        // i faces: (slow, fast) = (k, j); j faces: (k, i); k faces: (j, i)
        const auto b = fr + (unsigned) (side * 10 * K * K + v * K * K + kj);
        const double b0 = b[0], b1 = b[5 * K * K];
#pragma unroll
        for (int i = 0; i < K; ++i) s[i] += fv[side * K + i] * b0 + fv[(2 + side) * K + i] * b1;
#pragma unroll
        for (int dir = 1; dir < 3; ++dir) {
          const double cv = sFv[side * K + (dir == 1 ? jj : kk)], cd = sFv[(2 + side) * K + (dir == 1 ? jj : kk)];
          const auto f = fr + (unsigned) ((2 * dir + side) * 10 * K * K + v * K * K + (dir == 1 ? kk : jj) * K);
#pragma unroll
          for (int i = 0; i < K; ++i) s[i] += cv * f[i] + cd * f[5 * K * K + i];
        }
      }
      // a non-finite right-hand side is flagged: the solve's max-norms would
      // pass over it
#pragma unroll
      for (int i = 0; i < K; ++i) bad = bad || !isfinite(s[i]);
    };
    columns_to_modes<K, M, S, false>(scalar_op<K, M, double>(&ops()->ad), XD, (double *) Y, B, t, add);
  }
  T x[kTight ? 1 : S::NDL][5], r[S::NDL][5];
  int uo[S::NDL];
  double r0 = 0.0;
#pragma unroll
  for (int s = 0; s < S::NDL; ++s) {
    const int d = t + s * G;
    uo[s] = d < ND ? (d / K) * S::KP + d % K : 0;
#pragma unroll
    for (int l = 0; l < 5; ++l) {
      r[s][l] = d < ND ? B[l * S::UV + uo[s]] : T(0);
      if constexpr (kTight) XS[(s * 5 + l) * G] = 0;
      else x[s][l] = 0;
      r0 = fmax(r0, fabs(double(r[s][l])));
    }
  }
  {
    double red[3] = {r0, mach2, evMax};
    group_reduce<G, 3, 0>(red, sRed, half);
    r0 = red[0];
    if (live && t == 0) {
      if (args->ctl.monitor) glob(a->mach2Elem)[e] = red[1];
      if (FULL && a->eddyPart) glob(a->eddyPart)[e] = red[2];
    }
  }

  // ---------------- entropy-variable mass matrix: PCG with the element-centre
  // dV/dU; the preconditioner is symmetric and constant over the iterations,
  // so beta is the ratio of the successive r.z
  int iters = 0;
  bool on = r0 * (8.0 / elemJac) > 1e-10;
  if (__any(on)) {
    const double *pre = sPre[sub];
    auto uni = [](double v) {      // the same in every thread of a uniform workgroup
      if constexpr (kUniform)
        v = __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                             __builtin_amdgcn_readfirstlane(__double2loint(v)));
      return T(v);
    };
    const T ek = uni(pre[0]), pu = uni(pre[1]), pv = uni(pre[2]), pw = uni(pre[3]), a1 = uni(pre[4]), pi = uni(pre[5]),
            c0 = uni(pre[6]);
    // z = dV/dU(centre) r / Jbar
    auto precond = [&](const T (&rr)[5], T (&z)[5]) {
      const T d = a1 * (ek * rr[0] - pu * rr[1] - pv * rr[2] - pw * rr[3] + rr[4]);
      z[0] = ek * d + c0 * rr[0] - pi * rr[4];
      z[1] = pi * rr[1] - pu * d;
      z[2] = pi * rr[2] - pv * d;
      z[3] = pi * rr[3] - pw * d;
      z[4] = d - pi * rr[0];
    };
    const double tol = (kMixed ? 1e-5 : 1e-10) * r0;
    double rz = 0.0;
    group_sync<G>();
#pragma unroll
    for (int s = 0; s < S::NDL; ++s) {
      T z[5];
      precond(r[s], z);
#pragma unroll
      for (int l = 0; l < 5; ++l) {
        rz += double(r[s][l]) * double(z[l]);
        if (t + s * G < ND) B[l * S::UV + uo[s]] = z[l];
      }
    }
    { double red[1] = {rz}; group_reduce<G, 1, 1>(red, sRed, half); rz = red[0]; }
    const E A = scalar_op<K, M, T>(&ops()->a);
#pragma unroll 1
    for (int it = 0;; ++it) {
      if (it == 100) {
        if (live && on && t == 0) atomicOr(a->flags, kFlagCGNotConverged);
        break;
      }
      group_sync<G>();
      modes_to_columns<K, M, S, T>(A, B, X, Y, t);
      {
        T y[5][HP];
#pragma unroll
        for (int v = 0; v < 5; ++v) {
          T cc[K];
#pragma unroll
          for (int q = 0; q < K; ++q) cc[q] = X[(v * K + q) * NP + col];
          col_points(A, cc, y[v]);
          __builtin_amdgcn_sched_barrier(0);
        }
        // w J dU/dV at the points (ElementClass.cpp:4228-4253), with
        // E = e / (gamma - 1) + ek the total energy per mass:
        //   y0 = rho (p0 + u.p + E p4),  y_i = u_i y0 + P (p_i + u_i p4),
        //   y4 = E y0 + P (u.p + (E + ek) p4)
        // or with rho E and the last entry d: y4 = rho E p0 + (rho E + P) u.p + d p4
#pragma unroll
        for (int p = 0; p < HP; ++p) {
          if constexpr (kTight)
#pragma unroll
            for (int l = 0; l < NPR; ++l) asm volatile("" : "+v"(pr[p][l]));
          const T wr = pr[p][0], u = pr[p][1], v = pr[p][2], w = pr[p][3];
          const T kin = T(0.5) * (u * u + v * v + w * w);
          if constexpr (kMixed) {
            const T P = pr[p][4], d = pr[p][5], rE = P * T(kInvGm1) + wr * kin;
            const T p4 = y[4][p], up = u * y[1][p] + v * y[2][p] + w * y[3][p];
            const T y0 = wr * (y[0][p] + up) + rE * p4, yP = y0 + P * p4;
            y[4][p] = rE * y[0][p] + (rE + P) * up + d * p4;
            y[0][p] = y0;
            y[1][p] = u * yP + P * y[1][p];
            y[2][p] = v * yP + P * y[2][p];
            y[3][p] = w * yP + P * y[3][p];
          } else {
            const T eh = pr[p][4];
            const T Et = eh * T(kInvGm1) + kin, P = wr * eh;
            const T p4 = y[4][p];
            const T up = u * y[1][p] + v * y[2][p] + w * y[3][p];
            const T y0 = wr * (y[0][p] + up + Et * p4);
            y[0][p] = y0;
            y[1][p] = u * y0 + P * (y[1][p] + u * p4);
            y[2][p] = v * y0 + P * (y[2][p] + v * p4);
            y[3][p] = w * y0 + P * (y[3][p] + w * p4);
            y[4][p] = Et * y0 + P * (up + (Et + kin) * p4);
          }
          if (p % 2) __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (H == 1) {
#pragma unroll
          for (int v = 0; v < 5; ++v) {
            T cc[K];
            col_modes(A, y[v], cc);
            if (act)
#pragma unroll
              for (int q = 0; q < K; ++q) X[(v * K + q) * NP + tl] = cc[q];
            __builtin_amdgcn_sched_barrier(0);
          }
          group_sync<G>();
        } else {
          T cc[5][K];
#pragma unroll
          for (int v = 0; v < 5; ++v) col_modes(A, y[v], cc[v]);
          group_sync<G>();                       // both halves have read their columns
          store_columns(cc, X);
        }
      }
      columns_to_modes<K, M, S, true>(A, X, Y, X, t, [](int, T (&)[K]) {});
      double pAp = 0.0;
#pragma unroll
      for (int s = 0; s < S::NDL; ++s)
        if (t + s * G < ND)
#pragma unroll
          for (int l = 0; l < 5; ++l)
            pAp += double(B[l * S::UV + uo[s]]) * double(X[l * S::UV + uo[s]]);
      { double red[1] = {pAp}; group_reduce<G, 1, 1>(red, sRed, half); pAp = red[0]; }
      const double alpha = rz / pAp;
      const T al = T(alpha);
      double rzn = 0.0;
      bool more = false;
      T z[S::NDL][5];
      group_sync<64>();      // p and A p are read again instead of being kept over the reduction
#pragma unroll
      for (int s = 0; s < S::NDL; ++s) {
        if (on && t + s * G < ND)
#pragma unroll
          for (int l = 0; l < 5; ++l) {
            if constexpr (kTight) XS[(s * 5 + l) * G] += al * B[l * S::UV + uo[s]];
            else x[s][l] += al * B[l * S::UV + uo[s]];
            r[s][l] -= al * X[l * S::UV + uo[s]];
            // the reference's stop rule (CG_MassMatrix.cpp:465), max-norm; the
            // float form stops at 1e-5, a few units of its rounding level
            more = more || fabs(double(r[s][l])) >= tol;
          }
        precond(r[s], z[s]);
#pragma unroll
        for (int l = 0; l < 5; ++l) rzn += double(r[s][l]) * double(z[s][l]);
      }
      if constexpr (G > 64) {
        double red[2] = {rzn, more ? 1.0 : 0.0};
        group_reduce<G, 2, 1>(red, sRed, half);
        rzn = red[0]; more = red[1] > 0.0;
      } else {
        double red[1] = {rzn};
        group_reduce<G, 1, 1>(red, sRed, half);
        rzn = red[0];
        unsigned long long m = __ballot(more);
        if constexpr (G < 64) m = (m >> (sub * G)) & ((1ull << G) - 1);
        more = m != 0;
      }
      if (on) iters = it + 1;
      on = on && more;
      if (!__any(on)) break;
      if (on) {
        const T beta = T(rzn / rz);
#pragma unroll
        for (int s = 0; s < S::NDL; ++s)
          if (t + s * G < ND)
#pragma unroll
            for (int l = 0; l < 5; ++l) B[l * S::UV + uo[s]] = beta * B[l * S::UV + uo[s]] + z[s][l];
      }
      rz = rzn;
    }
  }
  if (!live) return;
  fresh();
  if (t == 0) glob(a->cgIter)[e] = iters;
  // ---------------- outputs: R and/or the in-place RK stage update
  const auto Re = glob(a->R) + (size_t) e * 5 * ND;
  const auto Uw = glob(a->U) + (size_t) e * 5 * ND;
  const auto U0e = glob((const double *) a->U0) + (size_t) e * 5 * ND;
  const double bdt = args->ctl.update ? args->ctl.b * glob(a->scal)[kScalDt] : 0.0;
#pragma unroll
  for (int s = 0; s < S::NDL; ++s) {
    const int d = t + s * G;
    if (d < ND)
#pragma unroll
      for (int l = 0; l < 5; ++l) {
        const int i = l * ND + d;
        const double xl = double(kTight ? XS[(s * 5 + l) * G] : x[kTight ? 0 : s][l]);
        if (!isfinite(xl)) bad = true;
        if (args->ctl.store_res) Re[i] = xl;
        if (args->ctl.update) Uw[i] = (1.0 - args->ctl.a) * Uw[i] + args->ctl.a * U0e[i] - bdt * xl;
      }
  }
  if (bad) atomicOr(a->flags, kFlagNonFinite);
}

template <int K, int M, typename T>
void fill_col_args(const DeviceCase &dc, const StageCtl &ctl, ColArgs<K, M, T> &a)
{
  constexpr int H = M / 2;
  a.ctl = ctl; a.bug = dc.bug_compat;
  a.oW2 = dc.to.w2; a.oCentre = dc.to.bc; a.oFace = dc.to.fmin;
  for (int i = 0; i < M * K; ++i) {
    a.op.A[i] = T(dc.opA[i]); a.op.D[i] = T(dc.opD[i]);
    a.op.Ad[i] = dc.opA[i]; a.op.Dd[i] = dc.opD[i];
  }
  fill_even_odd(dc.opA, a.op.a);
  fill_even_odd(dc.opA, a.op.ad);
  for (int p = 0; p < H; ++p) {
    for (int q = 0; q < H; ++q) {
      const double l = dc.opDL[p * M + q], m = dc.opDL[p * M + M - 1 - q];
      a.op.l.P[p * H + q] = 0.5 * (l + m);
      a.op.l.Q[p * H + q] = 0.5 * (l - m);
    }
    a.op.l.cm[p] = dc.opDL[p * M + H];
    a.op.l.mr[p] = dc.opDL[H * M + p];
  }
  for (int q = 0; q < M; ++q) a.op.w[q] = dc.opW[q];
  for (int f = 0; f < 4; ++f)
    for (int q = 0; q < K; ++q) a.op.fvec[f * K + q] = dc.opF[f][q];
  a.op.c03 = dc.opC0[0] * dc.opC0[0] * dc.opC0[0];
}

template <int K, int M, bool BATCH, int HALVES, typename T>
hipError_t launch_cols(bool full, ColArgs<K, M, T> &a, hipStream_t s)
{
  using S = ColShape<K, M, T, HALVES>;
  const dim3 grid((a.n + S::NE - 1) / S::NE), block(S::NT);
  if (full) hipLaunchKernelGGL((volume_cols_kernel<K, M, BATCH, true, T, HALVES>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((volume_cols_kernel<K, M, BATCH, false, T, HALVES>), grid, block, 0, s, a);
  return hipGetLastError();
}

template <int K, int M, bool BATCH, typename T>
hipError_t launch_kind(int kind, ColArgs<K, M, T> &a, hipStream_t s)
{
  const bool full = kind == kVolColsFull || kind == kVolHalvesFull;
  if constexpr (K == 3)
    if (kind == kVolHalves || kind == kVolHalvesFull) return launch_cols<K, M, BATCH, 2>(full, a, s);
  return launch_cols<K, M, BATCH, kColHalves<K, T>>(full, a, s);
}

}  // namespace

template <int K, int M>
hipError_t volume_cols(const DeviceCase &dc, int kind, const StageCtl &ctl, hipStream_t s)
{
  auto run = [&](auto zero) {
    ColArgs<K, M, decltype(zero)> a{};
    a.c = case_dev(dc); a.n = dc.nElem;
    fill_col_args(dc, ctl, a);
    return launch_kind<K, M, false>(kind, a, s);
  };
  return dc.mixed ? run(0.0f) : run(0.0);
}

template <int K, int M>
hipError_t batch_volume_cols(const BatchGroup &g, int kind, const StageCtl &ctl, int w0, int nw, hipStream_t s)
{
  auto run = [&](auto zero) {
    ColArgs<K, M, decltype(zero)> a{};
    a.cases = g.cases; a.work = g.work; a.w0 = w0; a.n = nw;
    fill_col_args(*g.proto, ctl, a);
    return launch_kind<K, M, true>(kind, a, s);
  };
  return g.proto->mixed ? run(0.0f) : run(0.0);
}

template hipError_t volume_cols<VCP_SHAPE_K, VCP_SHAPE_M>(const DeviceCase &, int, const StageCtl &, hipStream_t);
template hipError_t batch_volume_cols<VCP_SHAPE_K, VCP_SHAPE_M>(const BatchGroup &, int, const StageCtl &, int, int,
                                                                hipStream_t);

}  // namespace vcp
