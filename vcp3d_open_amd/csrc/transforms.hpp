// Even-odd 1D transforms between modes and Gauss points, with the operators in
// scalar registers, and the pointers they are read through.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace vcp {
namespace {

// Pointer into constant memory: wave-uniform reads through it are scalar loads.
template <class X>
using cptr = const X __attribute__((address_space(4))) *;
// Pointer into global memory (not flat: a flat access would be counted with
// the LDS operations in flight).
template <class X>
using gptr = X __attribute__((address_space(1))) *;
template <class X>
__device__ __forceinline__ gptr<X> glob(X *p) { return (gptr<X>) (uintptr_t) p; }

// The operator A[p][q] = phi_q(r_p) in even-odd form (the points are symmetric
// about 0 and phi_q has the parity of q): even modes at the points of the
// first half and the middle, odd modes at the points of the first half; 18
// coefficients and 24 operations per line at (5, 7) in place of 35.
template <int K, int M, typename T>
struct EvenOdd {
  static constexpr int HE = (M + 1) / 2, HO = M / 2, KE = (K + 1) / 2, KO = K / 2;
  T e[HE * KE], o[HO * KO];
};

// The operator D[p][q] = phi_q'(r_p), of the opposite parity: odd modes at the
// points of the first half and the middle, even modes from 2 on at the points
// of the first half.
template <int K, int M, typename T>
struct EvenOddD {
  static constexpr int HE = (M + 1) / 2, HO = M / 2, KO = K / 2, KE = (K - 1) / 2;
  T e[HE * KO], o[HO * KE];
};

template <int K, int M, typename T>
void fill_even_odd(const double *A, EvenOdd<K, M, T> &a)
{
  for (int p = 0; p < a.HE; ++p)
    for (int q = 0; q < K; ++q) {
      if (q % 2 == 0) a.e[p * a.KE + q / 2] = T(A[p * K + q]);
      else if (p < a.HO) a.o[p * a.KO + q / 2] = T(A[p * K + q]);
    }
}

template <int K, int M, typename T>
void fill_even_odd(const double *D, EvenOddD<K, M, T> &d)
{
  for (int p = 0; p < d.HE; ++p)
    for (int q = 1; q < K; ++q) {
      if (q % 2) d.e[p * d.KO + q / 2] = T(D[p * K + q]);
      else if (p < d.HO) d.o[p * d.KE + q / 2 - 1] = T(D[p * K + q]);
    }
}

// An operator into scalar registers, where it stays over the loops that use it.
template <int K, int M, typename T>
__device__ __forceinline__ EvenOdd<K, M, T> scalar_op(cptr<EvenOdd<K, M, T>> p)
{
  EvenOdd<K, M, T> a;
#pragma unroll
  for (int i = 0; i < a.HE * a.KE; ++i) { a.e[i] = p->e[i]; asm volatile("" : "+s"(a.e[i])); }
#pragma unroll
  for (int i = 0; i < a.HO * a.KO; ++i) { a.o[i] = p->o[i]; asm volatile("" : "+s"(a.o[i])); }
  return a;
}

template <int K, int M, typename T>
__device__ __forceinline__ EvenOddD<K, M, T> scalar_op(cptr<EvenOddD<K, M, T>> p)
{
  EvenOddD<K, M, T> a;
#pragma unroll
  for (int i = 0; i < a.HE * a.KO; ++i) { a.e[i] = p->e[i]; asm volatile("" : "+s"(a.e[i])); }
#pragma unroll
  for (int i = 0; i < a.HO * a.KE; ++i) { a.o[i] = p->o[i]; asm volatile("" : "+s"(a.o[i])); }
  return a;
}

// modes -> points: o[p] = sum_q A[p][q] c[q]
template <int K, int M, typename T>
__device__ __forceinline__ void to_points(const EvenOdd<K, M, T> &A, const T (&c)[K], T (&o)[M])
{
  using E = EvenOdd<K, M, T>;
#pragma unroll
  for (int p = 0; p < E::HE; ++p) {
    T e = A.e[p * E::KE] * c[0];
#pragma unroll
    for (int q = 1; q < E::KE; ++q) e += A.e[p * E::KE + q] * c[2 * q];
    if (p < E::HO) {
      T d = A.o[p * E::KO] * c[1];
#pragma unroll
      for (int q = 1; q < E::KO; ++q) d += A.o[p * E::KO + q] * c[2 * q + 1];
      o[p] = e + d;
      o[M - 1 - p] = e - d;
    } else {
      o[p] = e;
    }
  }
}

// points -> modes: o[q] = sum_p A[p][q] x[p]
template <int K, int M, typename T>
__device__ __forceinline__ void to_modes(const EvenOdd<K, M, T> &A, const T (&x)[M], T (&o)[K])
{
  using E = EvenOdd<K, M, T>;
  T s[E::HE], d[E::HO];
#pragma unroll
  for (int p = 0; p < E::HO; ++p) { s[p] = x[p] + x[M - 1 - p]; d[p] = x[p] - x[M - 1 - p]; }
  if constexpr (M % 2) s[E::HO] = x[E::HO];
#pragma unroll
  for (int q = 0; q < E::KE; ++q) {
    T v = A.e[q] * s[0];
#pragma unroll
    for (int p = 1; p < E::HE; ++p) v += A.e[p * E::KE + q] * s[p];
    o[2 * q] = v;
  }
#pragma unroll
  for (int q = 0; q < E::KO; ++q) {
    T v = A.o[q] * d[0];
#pragma unroll
    for (int p = 1; p < E::HO; ++p) v += A.o[p * E::KO + q] * d[p];
    o[2 * q + 1] = v;
  }
}

// derivatives at the points: o[p] = sum_q D[p][q] c[q]
template <int K, int M, typename T>
__device__ __forceinline__ void to_points(const EvenOddD<K, M, T> &D, const T (&c)[K], T (&o)[M])
{
  using E = EvenOddD<K, M, T>;
#pragma unroll
  for (int p = 0; p < E::HE; ++p) {
    T e = D.e[p * E::KO] * c[1];
#pragma unroll
    for (int q = 1; q < E::KO; ++q) e += D.e[p * E::KO + q] * c[2 * q + 1];
    if (p < E::HO) {
      T d = D.o[p * E::KE] * c[2];
#pragma unroll
      for (int q = 1; q < E::KE; ++q) d += D.o[p * E::KE + q] * c[2 * q + 2];
      o[p] = e + d;
      o[M - 1 - p] = e - d;
    } else {
      o[p] = e;
    }
  }
}

// its transpose, added: o[q] += sum_p D[p][q] x[p]
template <int K, int M, typename T>
__device__ __forceinline__ void add_modes(const EvenOddD<K, M, T> &D, const T (&x)[M], T (&o)[K])
{
  using E = EvenOddD<K, M, T>;
  T s[E::HE], d[E::HO];
#pragma unroll
  for (int p = 0; p < E::HO; ++p) { s[p] = x[p] + x[M - 1 - p]; d[p] = x[p] - x[M - 1 - p]; }
  if constexpr (M % 2) s[E::HO] = x[E::HO];
#pragma unroll
  for (int q = 0; q < E::KO; ++q)
#pragma unroll
    for (int p = 0; p < E::HE; ++p) o[2 * q + 1] += D.e[p * E::KO + q] * s[p];
#pragma unroll
  for (int q = 0; q < E::KE; ++q)
#pragma unroll
    for (int p = 0; p < E::HO; ++p) o[2 * q + 2] += D.o[p * E::KE + q] * d[p];
}

}  // namespace
}  // namespace vcp
