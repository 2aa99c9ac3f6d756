// tri_block.h -- what the triangular sweeps share: the substitution with a 64 x
// 64 triangle laid out in LDS in its own order, 16 lanes a right-hand side, the
// interchanges of right-hand sides in LDS, and the sentinel of values of x that
// are still to come.
#pragma once
#include "leaf.h"
#include "mfma.h"

namespace la {

// The coefficients below the diagonal by 16 x 16 sub-blocks: sub-block
// (mi >= mk) at mi (mi + 1) / 2 + mk holds -M(16 mi + i, 16 mk + k) at [k][i], zero
// for i <= k of the diagonal ones.
template <class T> struct TriBlock {
  T c[10][16][17];
};

// t / d from r = 1 / d: the product corrected by its remainder, which rounds
// like the division while d and t / d are normal numbers.
template <class T>
__device__ __forceinline__ T div_by(T t, T d, T r) {
  const T q = t * r;
  return fma(fma(-q, d, t), r, q);
}

enum Diag { DIAG_UNIT, DIAG_DIVIDE, DIAG_MULTIPLY };

template <class T, Diag D>
__device__ __forceinline__ T by_diag(T x, T d, T r) {
  if constexpr (D == DIAG_DIVIDE) return div_by(x, d, r);
  else if constexpr (D == DIAG_MULTIPLY) return x * r;
  else return x;
}

// Steps KS .. 15 of sub-block KM; lane sub of 16 holds rows 16 m + sub in x[m],
// with their diagonals d and reciprocals r.  Per step one DPP product a
// sub-block still to come, the first of them the chain (about 16 cycles).
template <class T, Diag D, int KM, int KS>
__device__ __forceinline__ void tri_step(T (&x)[4], const T (&d)[4], const T (&r)[4], const TriBlock<T>& tri, int sub) {
  if constexpr (KS < 16) {
    if constexpr (KS % 8 == 0) asm volatile("" ::: "memory");  // (coefficients of 8 steps in flight, not of all)
    const T q = by_diag<T, D>(x[KM], d[KM], r[KM]);
#pragma unroll
    for (int m = KM; m < 4; ++m) fmac_from<KS>(x[m], q, tri.c[m * (m + 1) / 2 + KM][KS][sub]);
    tri_step<T, D, KM, KS + 1>(x, d, r, tri, sub);
  } else {
    x[KM] = by_diag<T, D>(x[KM], d[KM], r[KM]);
  }
}

// Column j of the inverse of one 16 x 16 block by substitution, K the next step:
// lane sub of 16 holds row sub, the reciprocal r of its diagonal and, at c(k), the
// coefficients -M(sub, k), zero for k >= sub.  A lane keeps its value from its own step:
// the later products with zero would turn it into a NaN where a diagonal is zero
// and the steps are infinite, and so would a zero above the diagonal times r.
template <class T, Diag D, int K, class C>
__device__ __forceinline__ void diag_steps(T& own, T x, T r, int sub, C c) {
  if constexpr (K < 16) {
    const T q = by_diag<T, D>(x, r, r);
    own = sub == K ? q : own;
    if constexpr (K < 15) fmac_from<K>(x, q, c(K));
    diag_steps<T, D, K + 1>(own, x, r, sub, c);
  }
}
template <class T, Diag D, class C>
__device__ __forceinline__ T diag_inverse(T r, int sub, int j, C c) {
  T own = T(0);
  diag_steps<T, D, 0>(own, sub == j ? T(1) : T(0), sub >= j ? r : T(0), sub, c);
  return own;
}

// ---- the inverse V of a triangle M by 16 x 16 blocks, in the order of the substitution ----
// Which of V's two residuals is the small one, and so the error of x = V y, follows
// from the order of its products.  By columns, V(i, j) = V(i, i) sum -M(i, k) V(k, j),
// is the better one where M's rows are solved downwards (lower M), by rows, V(i, j) =
// (sum V(i, k) -M(k, j)) V(j, j), where they are solved upwards.  Every product of 16
// terms runs in two chains.  Error of V against doubling by 2 x 2 block triangles (64 rows, LU
// factors of N(0,1) matrices): 0.94 to 0.97; all four triangles by columns 0.95 to
// 1.24, -sum V(i, k) (M(k, j) V(j, j)) 1.07 to 1.45.

// Row j of the inverse of one 16 x 16 block: column 15 - j of the inverse of its
// mirror image P(a, b) = M(15 - b, 15 - a).  Lane sub of 16 gets V(j, 15 - sub); r
// is the reciprocal of M's diagonal 15 - sub, c(a, b) is -M(a, b), zero for a <= b.
template <class T, Diag D, class C>
__device__ __forceinline__ T diag_inverse_row(T r, int sub, int j, C c) {
  return diag_inverse<T, D>(r, sub, 15 - j, [&](int k) { return c(15 - k, 15 - sub); });
}

// The product of two 16 x 16 blocks on the matrix cores; lane (li, lk) gives
// A(li, s + lk) and B(s + lk, li) for s = 0, 4, 8, 12.
template <class T, class FA, class FB>
__device__ __forceinline__ typename Mfma<T>::acc_t product16(FA a, FB b) {
  typedef Mfma<T> MM;
  const typename MM::acc_t zero = {T(0), T(0), T(0), T(0)};
  typename MM::acc_t p = MM::op(a(0), b(0), zero), q = MM::op(a(4), b(4), zero);
  p = MM::op(a(8), b(8), p);
  q = MM::op(a(12), b(12), q);
  return p + q;
}

// Sub-blocks m_lo .. m_hi - 1 (the others hold rows past the matrix).
template <class T, Diag D>
__device__ __forceinline__ void tri_solve(T (&x)[4], const T (&d)[4], const T (&r)[4], const TriBlock<T>& tri, int sub,
                                          int m_lo, int m_hi) {
  if (m_lo <= 0 && m_hi > 0) tri_step<T, D, 0, 0>(x, d, r, tri, sub);
  if (m_lo <= 1 && m_hi > 1) tri_step<T, D, 1, 0>(x, d, r, tri, sub);
  if (m_lo <= 2 && m_hi > 2) tri_step<T, D, 2, 0>(x, d, r, tri, sub);
  if (m_lo <= 3 && m_hi > 3) tri_step<T, D, 3, 0>(x, d, r, tri, sub);
}

// Interchanges of X by one wave: in order (SRC/dgetrs.f:187), or in reverse
// order (:217).  Pivots outside the matrix move nothing.
template <class T, bool REVERSE>
__device__ __forceinline__ void interchange(const int* ipiv, int n, T* X, int ldx, int nr, int lane) {
  const int nblk = (n + 63) / 64;
  for (int ib = 0; ib < nblk; ++ib) {
    const int k0 = 64 * (REVERSE ? nblk - 1 - ib : ib);
    int p = k0 + lane;
    if (p < n) {
      const int v = ipiv[p] - 1;
      if (v >= 0 && v < n) p = v;
    }
    int from_k = k0 + lane, from_p = p;
    const int cnt = min(64, n - k0);
#pragma unroll 4
    for (int j = 0; j < cnt; ++j) {
      const int jj = REVERSE ? j : cnt - 1 - j;
      const int k = k0 + jj, pk = __builtin_amdgcn_readlane(p, jj);
      from_k = from_k == k ? pk : from_k == pk ? k : from_k;
      from_p = from_p == k ? pk : from_p == pk ? k : from_p;
    }
    if (k0 + lane < n) {
      for (int q = 0; q < nr; ++q) {
        T* x = X + q * ldx;
        const T a = x[from_k], b = x[from_p];
        wave_sync();
        x[k0 + lane] = a;
        x[p] = b;
      }
    }
    wave_sync();
  }
}

// The sentinel that marks a value of x not yet written: a quiet NaN with a
// fixed payload.  A computed value with exactly these bits (only a NaN
// carrying this payload from the input) is stored as the NaN `alt` instead.
template <class T> struct Sent;
template <> struct Sent<double> {
  using U = unsigned long long;
  static constexpr U bits = 0x7FFC00005E471E57ull, alt = 0x7FFC00005E471E56ull;
};
template <> struct Sent<float> {
  using U = unsigned;
  static constexpr U bits = 0x7FC5E471u, alt = 0x7FC5E470u;
};
template <class T>
__device__ __forceinline__ bool is_sent(T v) {
  return __builtin_bit_cast(typename Sent<T>::U, v) == Sent<T>::bits;
}
template <class T>
__device__ __forceinline__ T canon(T v) {
  return is_sent(v) ? __builtin_bit_cast(T, Sent<T>::alt) : v;
}

constexpr unsigned SPIN_LIMIT = 1u << 22;

}  // namespace la
