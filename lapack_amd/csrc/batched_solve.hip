// batched_solve.hip -- the batch's triangular solves: DGETRS('N') and DGETRS('T')
// (SRC/dgetrs.f:181-218) for many matrices in one persistent launch, and the
// adjoint built on the second.
//
// One workgroup per matrix at a time (the next one from a work counter, largest
// orders first; every loop is bounded by the matrix order), NR right-hand sides
// X in LDS.  Both directions of both operators are one routine, sweep(): blocks
// of 64 rows in the order of the substitution, and per block
//   1. X(block) -= op(A)(block, solved rows) X(solved rows) on the matrix cores,
//      16 rows of the block a wave (with 16 waves the solved rows are dealt over
//      4 groups of waves), A read once, straight into the operand registers;
//   2. the block's 64 x 64 triangle, loaded ahead of 1 and laid out in LDS in
//      the order of the substitution, is solved 16 lanes a right-hand side, the
//      solved value passed on by DPP; a division is a product with the
//      reciprocal and one correction by the remainder, which rounds like it.
// The interchanges are composed 64 at a time by one wave: each lane follows two
// rows back through the block's 64 exchanges.
//
// Step 1 does not test for zeros and the reciprocal does not take every
// divisor, so where a result is not finite the matrix is solved again in the
// reference's order with its zero tests (BLAS/SRC/dtrsm.f:277-300): solve_by_rows.
//
// Bound: A read once per NR right-hand sides.  Up to two matrices a CU get 16
// waves, whose loads in flight are a CU's share of the memory rate, and 8
// right-hand sides a pass (they have the LDS); more matrices get 4 waves and 4.
// Measured in 4 / 16 waves: 256 adjoints of order 1024 with 8 right-hand sides
// 2416 / 1174 us, 500 solves of order 65..512 259 / 179, 1000 309 / 344, 10000
// of order 16..512 1718 / 3033.  (One wave for orders up to 64 was no faster:
// 3000 of order 8..64 72 us against 70.)  Against one wave per block of rows,
// 64-step substitutions by shuffles and interchanges by one lane: 10000 solves
// of order 16..512 4700 -> 1720 us, the 256 adjoints 6420 -> 1152 (640 of them
// the solve: 3.3 TB/s of A; floor of both halves 930).
// Error against 80 bits on factors of N(0,1) matrices, relative to sums in 64
// lanes and a tree (T) and to rows taken off one by one (N): T 0.93 to 1.05, N 0.55
// to 0.91.  Two running sums over all solved rows instead of a new one for each 16:
// 1.0 to 1.7 and 0.8 to 1.2, 60 adjoints of order 1000 655 us instead of 690.
#include "tri_block.h"
#include "mfma.h"

#include <algorithm>

namespace la {
namespace {

// Groups of waves that share a block's product (4 waves: 16 rows each).
template <int NT> constexpr int groups() { return NT / 256; }

template <class T, int NT, int NR> struct SolveLds {
  TriBlock<T> tri;
  T dia[64], rec[64];
  T red[groups<NT>()][groups<NT>() > 1 ? NR : 1][64];
  int item;
};

// Rows are counted from X in LDS, ldx apart.  (One more than a multiple of 32
// keeps the rows that op(A) = A^T takes apart in the banks; 4 more, A's.)
inline int solve_ldx(int nmax, bool trans) { return (nmax + 63) / 64 * 64 + (trans ? 1 : 4); }

// One sweep: FWD rows 0, 1, ..; otherwise rows n-1, n-2, ..
template <class T, bool TRANS, bool FWD, bool UNIT, int NT, int NR>
__device__ __forceinline__ void sweep(const T* A, long lda, int n, T* X, int ldx, int nr, SolveLds<T, NT, NR>& S) {
  typedef Mfma<T> MM;
  typedef typename MM::acc_t acc_t;
  constexpr int G = groups<NT>();
  constexpr int SU = (10 + G - 1) / G;  // a thread's sub-blocks of the triangle, an element of each
  constexpr int U = 4;                  // chunks of 16 solved rows in flight
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nblk = (n + 63) / 64;
  for (int ib = 0; ib < nblk; ++ib) {
    const int kb = 64 * (FWD ? ib : nblk - 1 - ib), bs = min(64, n - kb);
    // rows of the block by their place in the substitution; past the matrix
    // they come last (FWD) or first and hold zeros
    auto row_of = [&](int i) { return FWD ? kb + i : kb + 63 - i; };
    const int m_lo = FWD ? 0 : (64 - bs) / 16, m_hi = FWD ? (bs + 15) / 16 : 4;
    // the triangle and its diagonal
    const int ta = tid & 15, tc = (tid & 255) >> 4;  // ta: the index that is contiguous in memory
    T t[SU];
#pragma unroll
    for (int u = 0; u < SU; ++u) {
      const int sb = tid / 256 + G * u;
      const int mi = sb >= 6 ? 3 : sb >= 3 ? 2 : sb >= 1 ? 1 : 0, mk = sb - mi * (mi + 1) / 2;
      const int i = 16 * mi + (TRANS ? tc : ta), k = 16 * mk + (TRANS ? ta : tc);
      const int gi = row_of(i), gk = row_of(k);
      t[u] = T(0);
      if (sb < 10 && i > k && gi < n && gk < n) t[u] = TRANS ? A[gk + (long)gi * lda] : A[gi + (long)gk * lda];
    }
    T dg = T(1);
    if (!UNIT && tid < 64 && row_of(tid) < n) dg = A[row_of(tid) + (long)row_of(tid) * lda];
    // 1. the solved rows r0 .. r0 + K - 1
    const int r0 = FWD ? 0 : kb + 64, K = FWD ? kb : n - r0;
    if (K > 0) {
      const int mt = wave & 3, ks = wave >> 2;
      const int m = min(kb + 16 * mt + li, n - 1);
      const T* const Am = TRANS ? A + (long)m * lda : A + m;
      const T* const Xq = X + (long)min(li, NR - 1) * ldx;
      // Every 16 products have a sum of their own, which is added to the running
      // one: none grows with the rows already solved.
      const acc_t zero = {T(0), T(0), T(0), T(0)};
      acc_t acc = zero;
      for (int k0 = 16 * ks; k0 < K; k0 += 16 * G * U) {
        T a[U][4];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int kk = r0 + min(k0 + 16 * G * u, K - 1);
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            if constexpr (TRANS) a[u][s] = Am[min(kk + 4 * lk + s, n - 1)];
            else a[u][s] = Am[(long)min(kk + 4 * s + lk, n - 1) * lda];
          }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (k0 + 16 * G * u >= K) break;
          const int kk = r0 + k0 + 16 * G * u;  // (X is zero from row n to the end of its block of 64)
          acc_t p = zero;
#pragma unroll
          for (int s = 0; s < 4; ++s) p = MM::op(a[u][s], Xq[TRANS ? kk + 4 * lk + s : kk + 4 * s + lk], p);
          acc = acc + p;
        }
      }
      if constexpr (G == 1) {
        if (li < nr) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int row = kb + 16 * mt + MM::row(lk, r);
            if (row < n) X[row + li * ldx] -= acc[r];
          }
        }
      } else if (li < NR) {
#pragma unroll
        for (int r = 0; r < 4; ++r) S.red[ks][li][16 * mt + MM::row(lk, r)] = acc[r];
      }
    }
    // the triangle into LDS
#pragma unroll
    for (int u = 0; u < SU; ++u) {
      const int sb = tid / 256 + G * u;
      if (sb < 10) S.tri.c[sb][TRANS ? ta : tc][TRANS ? tc : ta] = -t[u];
    }
    if (!UNIT && tid < 64) {
      S.dia[tid] = dg;
      S.rec[tid] = T(1) / dg;
    }
    __syncthreads();
    // 2.
    if (4 * wave < nr) {
      const int q = 4 * wave + lk, qx = min(q, NR - 1);
      T x[4], d[4], r[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int i = 16 * m + li;
        x[m] = X[row_of(i) + qx * ldx];
        if constexpr (G > 1) {
          if (K > 0) {
            const int ri = FWD ? i : 63 - i;
            T sum = S.red[0][qx][ri];
#pragma unroll
            for (int g = 1; g < G; ++g) sum += S.red[g][qx][ri];
            x[m] = kb + ri < n ? x[m] - sum : T(0);
          }
        }
        d[m] = UNIT ? T(1) : S.dia[i];
        r[m] = UNIT ? T(1) : S.rec[i];
      }
      tri_solve<T, UNIT ? DIAG_UNIT : DIAG_DIVIDE>(x, d, r, S.tri, li, m_lo, m_hi);
#pragma unroll
      for (int m = 0; m < 4; ++m)
        if (q < nr) X[row_of(16 * m + li) + q * ldx] = x[m];
    }
    __syncthreads();
  }
}

// The reference's order with its zero tests, for matrices whose result is not
// finite.  X holds B with its rows interchanged (N) or B (T).
template <class T, bool TRANS, int NT, int NR>
__device__ __attribute__((noinline)) void solve_by_rows(const T* A, long lda, int n, T* X, int ldx, int nr) {
  const int tid = threadIdx.x, lane = tid & 63;
  // first: L (N) or U^T (T), forward; second: U or L^T, backward
  for (int pass = 0; pass < 2; ++pass) {
    const bool fwd = pass == 0, unit = (pass == 0) != TRANS;
    const int nblk = (n + 63) / 64;
    for (int ib = 0; ib < nblk; ++ib) {
      const int kb = 64 * (fwd ? ib : nblk - 1 - ib), bs = min(64, n - kb);
      if (tid < 64) {
        T xi[NR];
#pragma unroll
        for (int q = 0; q < NR; ++q) xi[q] = (q < nr && lane < bs) ? X[kb + lane + q * ldx] : T(0);
        const T dii = (!unit && lane < bs) ? A[(kb + lane) + (long)(kb + lane) * lda] : T(1);
        for (int s = 0; s < bs; ++s) {
          const int k = fwd ? s : bs - 1 - s;
          const bool on = (fwd ? lane > k : lane < k) && lane < bs;
          T c = T(0);
          if (on) c = TRANS ? A[(kb + k) + (long)(kb + lane) * lda] : A[(kb + lane) + (long)(kb + k) * lda];
#pragma unroll
          for (int q = 0; q < NR; ++q) {
            if (!unit && lane == k && (TRANS || xi[q] != T(0))) xi[q] = xi[q] / dii;
            const T xk = __shfl(xi[q], k);
            if (on && (TRANS || xk != T(0))) xi[q] = xi[q] - xk * c;
          }
        }
#pragma unroll
        for (int q = 0; q < NR; ++q)
          if (q < nr && lane < bs) X[kb + lane + q * ldx] = xi[q];
      }
      __syncthreads();
      for (int i = (fwd ? kb + bs : 0) + tid; i < (fwd ? n : kb); i += NT) {
        T xi[NR];
#pragma unroll
        for (int q = 0; q < NR; ++q) xi[q] = (q < nr) ? X[i + q * ldx] : T(0);
        for (int s = 0; s < bs; ++s) {
          const int k = kb + (fwd ? s : bs - 1 - s);
          const T c = TRANS ? A[k + (long)i * lda] : A[i + (long)k * lda];
#pragma unroll
          for (int q = 0; q < NR; ++q) {
            const T xk = (q < nr) ? X[k + q * ldx] : T(0);
            if (TRANS || xk != T(0)) xi[q] = xi[q] - xk * c;
          }
        }
#pragma unroll
        for (int q = 0; q < NR; ++q)
          if (q < nr) X[i + q * ldx] = xi[q];
      }
      __syncthreads();
    }
  }
}

template <class T, bool TRANS, int NT, int NR>
__global__ __launch_bounds__(NT) void getrs_batched_kernel(int batch, const int* __restrict__ nv,
                                                           const int* __restrict__ nrhsv, T* const* __restrict__ av,
                                                           const int* __restrict__ ldav, int* const* __restrict__ ipv,
                                                           T* const* __restrict__ bv, const int* __restrict__ ldbv,
                                                           const int* __restrict__ order, unsigned* counter, int ldx) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  auto& S = *reinterpret_cast<SolveLds<T, NT, NR>*>(smem_raw);
  T* const X = reinterpret_cast<T*>(smem_raw + sizeof(SolveLds<T, NT, NR>));
  const int tid = threadIdx.x, lane = tid & 63;
  for (int guard = 0; guard <= batch; ++guard) {
    if (tid == 0) S.item = (int)atomicAdd(counter, 1u);
    __syncthreads();
    const int item = __builtin_amdgcn_readfirstlane(S.item);
    __syncthreads();
    if (item >= batch) break;
    const int b = order[item];
    const int n = nv[b], nrhs = nrhsv[b];
    const T* const A = av[b];
    const long lda = ldav[b];
    const int* const ipiv = ipv[b];
    T* const B = bv[b];
    const long ldb = ldbv[b];
    const int n64 = (n + 63) / 64 * 64;
    for (int q0 = 0; q0 < nrhs; q0 += NR) {
      const int nr = min(NR, nrhs - q0);
      auto load = [&] {
        for (int q = 0; q < nr; ++q)
          for (int r = tid; r < n64; r += NT) X[r + q * ldx] = r < n ? B[r + (long)(q0 + q) * ldb] : T(0);
        __syncthreads();
        if (!TRANS) {
          if (tid < 64) interchange<T, false>(ipiv, n, X, ldx, nr, lane);
          __syncthreads();
        }
      };
      load();
      sweep<T, TRANS, true, !TRANS, NT, NR>(A, lda, n, X, ldx, nr, S);
      sweep<T, TRANS, false, TRANS, NT, NR>(A, lda, n, X, ldx, nr, S);
      int bad = 0;
      for (int q = 0; q < nr; ++q)
        for (int r = tid; r < n; r += NT) bad |= !__builtin_isfinite(X[r + q * ldx]);
      if (__syncthreads_or(bad)) {
        load();
        solve_by_rows<T, TRANS, NT, NR>(A, lda, n, X, ldx, nr);
      }
      if (TRANS) {
        if (tid < 64) interchange<T, true>(ipiv, n, X, ldx, nr, lane);
        __syncthreads();
      }
      for (int q = 0; q < nr; ++q)
        for (int r = tid; r < n; r += NT) B[r + (long)(q0 + q) * ldb] = X[r + q * ldx];
      __syncthreads();
    }
  }
}

// Abar_b <- -Bbar_b X_b^T (+ Abar_b when accumulate), for every matrix b of
// the batch: the adjoint's rank-nrhs product, bound by the n^2 result
// written to HBM.  Grid (tiles of the largest order, batch): a 64 x 64 tile
// per 256-thread workgroup, 32 of the nrhs columns at a time staged in LDS,
// each lane writing 16 columns of one row; tiles past a matrix's order exit.
__global__ __launch_bounds__(256) void rankk_batched_kernel(const int* __restrict__ nv, const int* __restrict__ nrhsv,
                                                            double* const* __restrict__ bbv,
                                                            const int* __restrict__ ldbbv,
                                                            double* const* __restrict__ xv, const int* __restrict__ ldxv,
                                                            double* const* __restrict__ cv,
                                                            const int* __restrict__ ldcv, int tiles1, int accumulate) {
  constexpr int TL = 64, KC = 32;
  __shared__ double sa[KC][TL];
  __shared__ double sb[KC][TL + 1];
  const int b = blockIdx.y;
  const int n = nv[b];
  const int i0 = (blockIdx.x % tiles1) * TL, j0 = (blockIdx.x / tiles1) * TL;
  if (i0 >= n || j0 >= n) return;
  const int k = nrhsv[b];
  const double* A = bbv[b];
  const long lda = ldbbv[b];
  const double* Bm = xv[b];
  const long ldbm = ldxv[b];
  double* C = cv[b];
  const long ldc = ldcv[b];
  const int t = threadIdx.x;
  const int r = t % TL, cg = t / TL;
  double acc[16];
#pragma unroll
  for (int q = 0; q < 16; ++q) acc[q] = 0.0;
  for (int p0 = 0; p0 < k; p0 += KC) {
    const int kc = min(KC, k - p0);
    __syncthreads();
    for (int e = t; e < kc * TL; e += 256) {
      const int p = e / TL, rr = e % TL;
      sa[p][rr] = (i0 + rr < n) ? A[(i0 + rr) + (long)(p0 + p) * lda] : 0.0;
      sb[p][rr] = (j0 + rr < n) ? Bm[(j0 + rr) + (long)(p0 + p) * ldbm] : 0.0;
    }
    __syncthreads();
    for (int p = 0; p < kc; ++p) {
      const double a = sa[p][r];
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[q] = fma(a, sb[p][cg * 16 + q], acc[q]);
    }
  }
  const int i = i0 + r;
  if (i >= n) return;
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const int j = j0 + cg * 16 + q;
    if (j < n) {
      double* cp = C + i + (long)j * ldc;
      *cp = accumulate ? *cp - acc[q] : -acc[q];
    }
  }
}

template <class T, bool TRANS, int NT, int NR>
size_t solve_lds(int nmax) {
  return sizeof(SolveLds<T, NT, NR>) + sizeof(T) * (size_t)NR * solve_ldx(nmax, TRANS);
}

template <class T, bool TRANS, int NT, int NR>
int solve_grid(int count, int nmax, int ncu) {
  auto kern = getrs_batched_kernel<T, TRANS, NT, NR>;
  if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds_limit()) != hipSuccess)
    (void)hipGetLastError();
  int occ = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kern, NT, solve_lds<T, TRANS, NT, NR>(nmax)) != hipSuccess ||
      occ < 1) {
    (void)hipGetLastError();
    occ = 1;
  }
  return std::max(1, std::min(count, ncu * occ));
}

}  // namespace

// LA_ERR_LIMIT where the right-hand sides of the largest order do not fit in LDS.
template <class T, bool TRANS>
int batched_solve_plan(int batch, int nmax, BatchedSolvePlan* p) {
  // (what the solve needed of a matrix's order since its first form, so that
  // the orders it takes do not depend on this one's layout)
  if (sizeof(T) * 4 * (size_t)nmax + (TRANS ? sizeof(T) * 64 * 65 + 64 : 0) > (size_t)lds_limit()) return LA_ERR_LIMIT;
  int dev = 0, ncu = 256;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
  const size_t lim = (size_t)lds_limit();
  p->wide = batch <= 2 * ncu && solve_lds<T, TRANS, 1024, 8>(nmax) <= lim;
  if (!p->wide && solve_lds<T, TRANS, 256, 4>(nmax) > lim) return LA_ERR_LIMIT;
  p->grid = p->wide ? solve_grid<T, TRANS, 1024, 8>(batch, nmax, ncu) : solve_grid<T, TRANS, 256, 4>(batch, nmax, ncu);
  return 0;
}
template int batched_solve_plan<double, false>(int, int, BatchedSolvePlan*);
template int batched_solve_plan<float, false>(int, int, BatchedSolvePlan*);
template int batched_solve_plan<double, true>(int, int, BatchedSolvePlan*);

template <class T, bool TRANS>
static void launch_solve(const BatchedSolvePlan& p, int batch, int nmax, const int* nv, const int* nrhsv, T* const* av,
                         const int* ldav, int* const* ipv, T* const* bv, const int* ldbv, const int* order,
                         unsigned* counter, hipStream_t s) {
  launch_fill_u32(counter, 1, 0u, s);
  const int nm = std::max(nmax, 1), ldx = solve_ldx(nm, TRANS);
#define LA_SOLVE(NT, NR)                                                                              \
  getrs_batched_kernel<T, TRANS, NT, NR><<<p.grid, NT, solve_lds<T, TRANS, NT, NR>(nm), s>>>(           \
      batch, nv, nrhsv, av, ldav, ipv, bv, ldbv, order, counter, ldx)
  if (p.wide) LA_SOLVE(1024, 8);
  else LA_SOLVE(256, 4);
#undef LA_SOLVE
}

template <class T>
int launch_getrs_batched(const BatchedSolvePlan& p, int batch, int nmax, const int* nv, const int* nrhsv, T* const* av,
                         const int* ldav, int* const* ipv, T* const* bv, const int* ldbv, const int* order,
                         unsigned* counter, hipStream_t s) {
  launch_solve<T, false>(p, batch, nmax, nv, nrhsv, av, ldav, ipv, bv, ldbv, order, counter, s);
  return 0;
}
template int launch_getrs_batched<double>(const BatchedSolvePlan&, int, int, const int*, const int*, double* const*,
                                          const int*, int* const*, double* const*, const int*, const int*, unsigned*,
                                          hipStream_t);
template int launch_getrs_batched<float>(const BatchedSolvePlan&, int, int, const int*, const int*, float* const*,
                                         const int*, int* const*, float* const*, const int*, const int*, unsigned*,
                                         hipStream_t);

// The batched adjoint: Bbar = A^-T Xbar in place of Xbar ,
// then Abar = -Bbar X^T (+ Abar).
int launch_adjoint_batched(const BatchedSolvePlan& p, int batch, int nmax, const int* nv, const int* nrhsv,
                           double* const* luv, const int* ldluv, int* const* ipv, double* const* xv, const int* ldxv,
                           double* const* xbv, const int* ldxbv, double* const* abv, const int* ldabv, int accumulate,
                           const int* order, unsigned* counter, hipStream_t s) {
  launch_solve<double, true>(p, batch, nmax, nv, nrhsv, luv, ldluv, ipv, xbv, ldxbv, order, counter, s);
  const int tiles1 = (nmax + 63) / 64;
  for (int b0 = 0; b0 < batch; b0 += 65535) {
    const int nb = std::min(65535, batch - b0);
    rankk_batched_kernel<<<dim3(tiles1 * tiles1, nb), 256, 0, s>>>(nv + b0, nrhsv + b0, xbv + b0, ldxbv + b0, xv + b0,
                                                                 ldxv + b0, abv + b0, ldabv + b0, tiles1, accumulate);
  }
  return 0;
}


}  // namespace la
