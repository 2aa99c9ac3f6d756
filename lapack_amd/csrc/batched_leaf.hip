// batched_leaf.hip -- the batch's LU factorizations for matrices of up to 512
// rows: one workgroup per matrix, the panel in registers.
//
// The reference has no batched API; each matrix gets DGETRF
// (SRC/dgetrf.f:105-225).  batched.hip holds the form for larger matrices and
// the panel widths a caller selects.
//
// Scheduling: the matrices are sorted by decreasing n; each range of orders
// (<= 64, <= 128, <= 256, <= 512) is one persistent launch with that many
// threads a workgroup, and a workgroup takes the next matrix of its range from
// a work counter, so the grid drains when the counter passes the range's end.
//
// Per block of 32 columns, right-looking:
//   1. a row a thread, 32 values in registers: leaf_columns (leaf.h);
//   2. the factored columns go back, and each wave takes its 64 rows of L as
//      matrix-core operands (registers, for the whole pass over the columns to
//      the right);
//   3. the columns to the right, CB at a time, in one pass: their rows of the
//      block are gathered through the interchanges into LDS and solved with
//      the block's unit triangle (16 lanes a column, the solved value passed
//      on by DPP); every other row reads its element of C from the row its
//      content is in (the leaf's record), takes the product and writes it
//      back; the solved rows are written when every wave has read.
// The interchanges of the columns to the left wait until the last block: one
// pass per block of columns applies what all later blocks did.
// Bound: per column the leaf's latency chain (about 2000 cycles; two
// workgroups of 512 threads or more smaller ones on a CU overlap theirs), and
// the trailing matrix read and written once per 32 columns (n^3/6 bytes per
// matrix in FP64) where the batch exceeds the caches.  10000 matrices of
// order 16..512: 28.2 ms (best panel form 62.9); the substitution keeps 8 steps'
// coefficients at a time and its rounds are not unrolled (32.6 ms with all of
// them in flight, which spilled far more than the 25 registers that the FP64 forms
// of 256 and 512 threads still do, 104 and 108 bytes of scratch a lane).
#include "leaf.h"
#include "mfma.h"

#include <algorithm>

namespace la {
namespace {

constexpr int BW = 32;  // columns of a block

// Steps K .. BW-1 of the substitution: sl[k][i] = -L(i, k), a column's values
// 0..15 and 16..31 in x[0] and x[1] of its 16 lanes.
template <class T, int K>
__device__ __forceinline__ void unit_solve(T (&x)[2], T& t, const T (*sl)[BW + 1], int sub) {
  if constexpr (K < BW) {
    if constexpr (K % 8 == 0) asm volatile("" ::: "memory");  // (coefficients of 8 steps in flight, not of all)
    constexpr int KM = K / 16, KS = K % 16;
    T y = x[KM];
    fmac_from<KS>(y, x[KM], sl[K][16 * KM + sub]);
    if constexpr (KM == 0) {
      if (KS == 0) t = T(0);
      fmac_from<KS>(t, x[0], sl[K][16 + sub]);
      if (KS == 15) x[1] = x[1] + t;
    }
    x[KM] = sub > KS ? y : x[KM];
    unit_solve<T, K + 1>(x, t, sl, sub);
  }
}

// The same with DTRSM's test: a zero of the solution is not multiplied
// (BLAS/SRC/dtrsm.f:177-190), which matters where L is not finite.
template <class T>
__device__ __forceinline__ void unit_solve_tested(T (&x)[2], const T (*sl)[BW + 1], int lane, int sub) {
#pragma unroll 1
  for (int k = 0; k < BW; ++k) {
    const T xk = __shfl(k < 16 ? x[0] : x[1], (lane & 48) | (k & 15));
    if (xk != T(0)) {
      if (sub > k) x[0] = x[0] + xk * sl[k][sub];
      if (16 + sub > k) x[1] = x[1] + xk * sl[k][16 + sub];
    }
  }
}

template <class T, int NTH>
__global__ __launch_bounds__(NTH) __attribute__((amdgpu_waves_per_eu(4))) void getrf_batched_leaf_kernel(int first, int last, const int* __restrict__ nv,
                                                                    T* const* __restrict__ av,
                                                                    const int* __restrict__ ldav,
                                                                    int* const* __restrict__ ipv,
                                                                    int* __restrict__ infov,
                                                                    const int* __restrict__ order,
                                                                    unsigned* counter) {
  typedef Mfma<T> MM;
  typedef typename MM::acc_t acc_t;
  constexpr int NW = NTH / 64;
  constexpr int CB = NTH >= 256 ? 64 : NTH >= 128 ? 32 : 16;  // columns of a pass's piece
  constexpr int NBL = NTH / BW;                               // blocks of a matrix (at most)
  constexpr int GU = BW * CB / NTH;                           // gathered elements a thread
  __shared__ LeafLds<T, BW, NTH, false> S;
  __shared__ T s_x[BW][CB + 1];          // the piece's rows of U
  __shared__ T s_l[BW][BW + 1];          // -L of the block, [k][i]
  __shared__ short s_org[NBL][NTH];      // the blocks' records: row whose content came to row r
  __shared__ int s_item, s_info;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  for (int guard = first; guard <= last; ++guard) {
    if (tid == 0) {
      s_item = first + (int)atomicAdd(counter, 1u);
      s_info = 0;
    }
    __syncthreads();
    const int item = __builtin_amdgcn_readfirstlane(s_item);
    if (item >= last) break;
    const int bi = order[item];
    const int n = nv[bi];
    T* const A = av[bi];
    const long lda = ldav[bi];
    int* const ipiv = ipv[bi];
    const int nbl = (n + BW - 1) / BW;
    for (int jb = 0; jb < nbl; ++jb) {
      const int k0 = BW * jb, w = min(BW, n - k0), h = n - k0;
      // 1. the block's columns
      int tid = threadIdx.x;  // (new for every block: see below)
      asm volatile("" : "+v"(tid));
      // (uniform column addresses, one row offset a thread)
      const unsigned rt0 = (unsigned)min(k0 + tid, n - 1);
      T v[BW];
#pragma unroll
      for (int c = 0; c < BW; ++c) {
        const T x = (A + (long)min(k0 + c, n - 1) * lda)[rt0];
        v[c] = tid < h && c < w ? x : T(0);
      }
      wait_vm();
      int my_piv, corg, zero_at;
      leaf_columns<T, BW, NTH, false, false, false>(v, S, h, w, 0, 1, 0u, nullptr, nullptr, my_piv, corg, zero_at);
      // 2. its factors back
      if (wave == NW - 1) {
        if (lane < w) ipiv[k0 + lane] = k0 + my_piv + 1;
        if (lane == 0 && zero_at >= 0 && s_info == 0) s_info = k0 + zero_at + 1;
      }
      s_org[jb][tid] = (short)corg;
      if (tid < h) {
#pragma unroll
        for (int c = 0; c < BW; ++c)
          if (c < w) (A + (long)(k0 + c) * lda)[rt0] = v[c];
      }
      const int c1 = k0 + w;
      if (c1 < n) {  // w == BW
        // (made new for every block, so that what follows from them is not
        // kept in registers over the leaf's columns)
        int te = tid, le = lane;
        asm volatile("" : "+v"(te), "+v"(le));
        const int li = le & 15, lk = le >> 4;
        if (tid < BW) {
#pragma unroll
          for (int k = 0; k < BW; ++k) s_l[k][tid] = k < tid ? -v[k] : T(0);
        }
        const bool below = 64 * wave + 63 >= BW && 64 * wave < h;
        wait_vm();
        __syncthreads();
        for (int cb = c1; cb < n; cb += CB) {
          // 3a. the block's rows of these columns, interchanged
          T g[GU];
#pragma unroll
          for (int u = 0; u < GU; ++u) {
            const int e = te + NTH * u, i = e & (BW - 1), c = e / BW;
            g[u] = A[(k0 + s_org[jb][i]) + (long)min(cb + c, n - 1) * lda];
          }
#pragma unroll
          for (int u = 0; u < GU; ++u) {
            const int e = te + NTH * u;
            s_x[e & (BW - 1)][e / BW] = g[u];
          }
          __syncthreads();
#pragma unroll 1
          for (int q = 0; q < CB; q += NTH / 16) {
            const int c = q + te / 16;
            T x[2] = {s_x[li][c], s_x[16 + li][c]}, t;
            unit_solve<T, 0>(x, t, s_l, li);
            // (an L that is not finite shows in every column's result)
            if (__builtin_expect(__any(!__builtin_isfinite(x[0]) || !__builtin_isfinite(x[1])), 0)) {
              x[0] = s_x[li][c];
              x[1] = s_x[16 + li][c];
              unit_solve_tested(x, s_l, le, li);
            }
            s_x[li][c] = x[0];
            s_x[16 + li][c] = x[1];
          }
          __syncthreads();
          // 3b. the rows below, 32 rows by 16 columns at a time: C^T -= U^T
          // L^T, so that 16 lanes hold 16 consecutive rows of a column.  Lane
          // (li, lk) of row tile rt and step s holds L(16 rt + li, 4 s + lk)
          // (the wave's own stores, read back for every piece: kept in
          // registers for all of them they would not leave room for a second
          // workgroup on the CU).
          if (below) {
            const int nct = min(CB, n - cb + 15) / 16;
            const long lo = (long)MM::row(lk, 0) * lda;
#pragma unroll 1
            for (int rp = 64 * wave < BW ? BW / 32 : 0; rp < 2; ++rp) {
              T a[2][BW / 4];
              long src[2];
#pragma unroll
              for (int rt = 0; rt < 2; ++rt) {
                const int r = min(64 * wave + 32 * rp + 16 * rt + li, h - 1);
                src[rt] = lo + k0 + s_org[jb][r];
                const long o = (long)(k0 + r) + (long)lk * lda;
#pragma unroll
                for (int s = 0; s < BW / 4; ++s) a[rt][s] = (A + (long)(k0 + 4 * s) * lda)[o];
              }
#pragma unroll 1
              for (int ct = 0; ct < nct; ++ct) {
                // a lane's columns are MM::row(lk, r) past the tile's first;
                // past the matrix it reads and writes nothing
                const int cl = cb + 16 * ct + MM::row(lk, 0);
                acc_t acc[2];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                  const T* p = A + (long)(cb + 16 * ct + MM::row(0, r)) * lda;
                  const bool in = cl + MM::row(0, r) < n;
#pragma unroll
                  for (int rt = 0; rt < 2; ++rt) acc[rt][r] = in ? p[src[rt]] : T(0);
                }
#pragma unroll
                for (int s = 0; s < BW / 4; ++s) {
                  const T b = -s_x[4 * s + lk][16 * ct + li];
#pragma unroll
                  for (int rt = 0; rt < 2; ++rt) acc[rt] = MM::op(b, a[rt][s], acc[rt]);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                  T* p = A + (long)(cb + 16 * ct + MM::row(0, r)) * lda;
                  const bool in = cl + MM::row(0, r) < n;
#pragma unroll
                  for (int rt = 0; rt < 2; ++rt) {
                    const int r0 = 64 * wave + 32 * rp + 16 * rt + li;
                    if (in && r0 < h) p[lo + k0 + r0] = acc[rt][r];
                  }
                }
              }
            }
          }
          __syncthreads();  // every wave has read the block's old rows
#pragma unroll
          for (int u = 0; u < GU; ++u) {
            const int e = te + NTH * u, i = e & (BW - 1), c = e / BW;
            if (cb + c < n) A[(k0 + i) + (long)(cb + c) * lda] = s_x[i][c];
          }
        }
      }
      wait_vm();
      __syncthreads();  // the next block reads what this one wrote
    }
    // the interchanges of the columns left of each block: rows past block jb
    // take the composition of what blocks jb+1 .. nbl-1 did
    int r = tid;
    for (int jb = nbl - 2; jb >= 0; --jb) {
      const int k1 = BW * (jb + 1);
      if (tid >= k1 && tid < n) r = k1 + s_org[jb + 1][r - k1];
      const bool moves = tid >= k1 && tid < n && r != tid;
      const unsigned rs = (unsigned)min(r, n - 1);
#pragma unroll 1
      for (int c0 = 0; c0 < BW; c0 += 8) {
        T* const p = A + (long)(BW * jb + c0) * lda;
        T v[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) v[c] = (p + (long)c * lda)[rs];
        wait_vm();
        __syncthreads();
        if (moves) {
#pragma unroll
          for (int c = 0; c < 8; ++c) (p + (long)c * lda)[(unsigned)tid] = v[c];
        }
      }
    }
    if (tid == 0) infov[bi] = s_info;
    __syncthreads();
  }
}

constexpr int NCLASS = 4;
constexpr int class_threads(int k) { return 64 << k; }

template <class T, int NTH>
int class_grid(int count) {
  auto kern = getrf_batched_leaf_kernel<T, NTH>;
  int occ = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kern, NTH, 0) != hipSuccess || occ < 1) {
    (void)hipGetLastError();
    occ = 1;
  }
  int dev = 0, ncu = 256;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
  return std::max(1, std::min(count, ncu * occ));
}

}  // namespace

int batched_leaf_nmax() { return class_threads(NCLASS - 1); }

template <class T>
void batched_leaf_plan(int batch, const int* sorted, BatchedLeafPlan* p) {
  // sorted: the orders, decreasing; class k takes those in (threads(k-1), threads(k)]
  int at = 0;
  for (int k = NCLASS - 1; k >= 0; --k) {
    const int lo = k > 0 ? class_threads(k - 1) : -1;
    int end = at;
    while (end < batch && sorted[end] > lo) ++end;
    p->first[k] = at;
    p->last[k] = end;
    const int count = end - at;
    switch (k) {
      case 0: p->grid[k] = class_grid<T, 64>(count); break;
      case 1: p->grid[k] = class_grid<T, 128>(count); break;
      case 2: p->grid[k] = class_grid<T, 256>(count); break;
      default: p->grid[k] = class_grid<T, 512>(count); break;
    }
    at = end;
  }
}
template void batched_leaf_plan<double>(int, const int*, BatchedLeafPlan*);
template void batched_leaf_plan<float>(int, const int*, BatchedLeafPlan*);

template <class T>
int launch_getrf_batched_leaf(const BatchedLeafPlan& p, const int* nv, T* const* av, const int* ldav, int* const* ipv,
                              int* infov, const int* order, unsigned* counters, hipStream_t s) {
  launch_fill_u32(counters, NCLASS, 0u, s);
#define LA_CLASS(K, NTH)                                                                                         \
  if (p.last[K] > p.first[K])                                                                                    \
  getrf_batched_leaf_kernel<T, NTH><<<p.grid[K], NTH, 0, s>>>(p.first[K], p.last[K], nv, av, ldav, ipv, infov, order, \
                                                             counters + K)
  LA_CLASS(3, 512);
  LA_CLASS(2, 256);
  LA_CLASS(1, 128);
  LA_CLASS(0, 64);
#undef LA_CLASS
  return 0;
}
template int launch_getrf_batched_leaf<double>(const BatchedLeafPlan&, const int*, double* const*, const int*,
                                               int* const*, int*, const int*, unsigned*, hipStream_t);
template int launch_getrf_batched_leaf<float>(const BatchedLeafPlan&, const int*, float* const*, const int*,
                                              int* const*, int*, const int*, unsigned*, hipStream_t);

}  // namespace la
