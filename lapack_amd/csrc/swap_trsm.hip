// swap_trsm.hip -- what follows a factored block of w <= 256 columns on other
// columns of the matrix, in one pass over each: the block's row interchanges
// (DLASWP, SRC/dgetrf.f:193,199-200; SRC/dgetrf2.f:234-236) and, for the
// columns right of it, the unit lower triangular solve U12 = L11^-1 A12
// (DTRSM, SRC/dgetrf.f:204-207; SRC/dgetrf2.f:240-241).
//
// In the transposed workspace T = A^T a column of A is a row of T.  A
// workgroup owns 16 of them (16 consecutive values of every T column: whole
// 128-byte lines in FP64), reads the rows that the interchanges move into the
// block and out of it, and needs no other workgroup: the interchanged and
// solved values go back in place.
//
// The interchanges come as the leaves' record of where each row's content was
// (org, panel.hip): row k0 + i of the block takes row org[k0 + i], and a row r
// past the block that some step pivoted (r = ipiv[k0 + i] - 1) takes row
// org[r].  A row pivoted twice is moved twice from the same source to the same
// place, so nothing has to be composed or counted.
//
// The solve goes by 64-row blocks: four waves solve the 64 x 16 block by
// substitution, sixteen lanes a column with four rows each, the solved value
// passed on by DPP (row_newbcast); then every wave subtracts the products of
// the block's rows on the matrix cores from the 16-row tiles below.  The
// triangle's next pieces are read while a block is solved.
// Bound by latency for the few columns on the panel's path (a block: 64
// dependent steps), by the matrix cores and the triangle's re-reads from L2
// for all columns of a large matrix.
#include "leaf.h"
#include "mfma.h"

namespace la {
namespace {

constexpr int SB = 64;        // rows of a solve block
constexpr int SC = 16;        // columns of A a workgroup owns
constexpr int SWMAX = 256;    // widest block
constexpr int SNT = 512;

// Steps K .. SB-1 of the substitution: sl[k][i] = -L(i, k).  The products of
// sixteen steps are summed on their own (t) before they join the rows below.
template <class T, int K>
__device__ __forceinline__ void solve_steps(T (&x)[SB / 16], T (&t)[SB / 16], const T (*sl)[SB + 1], int sub) {
  if constexpr (K < SB) {
    constexpr int KM = K / 16, KS = K % 16;
    T y = x[KM];
    fmac_from<KS>(y, x[KM], sl[K][16 * KM + sub]);
#pragma unroll
    for (int m = KM + 1; m < SB / 16; ++m) {
      if (KS == 0) t[m] = T(0);
      fmac_from<KS>(t[m], x[KM], sl[K][16 * m + sub]);
      if (KS == 15) x[m] = x[m] + t[m];
    }
    x[KM] = sub > KS ? y : x[KM];
    solve_steps<T, K + 1>(x, t, sl, sub);
  }
}

// Columns of A [c0, c1) interchanged and solved (the first nsolve blocks),
// columns [s0, s1) interchanged only; nblk blocks in all.  nskip: blocks
// dispatched to XCDs 0 .. nskip-1 (blockIdx % 8) leave at once.
template <class T>
__global__ __launch_bounds__(SNT) void swap_trsm_kernel(T* __restrict__ Tm, long ldt, int k0, int w, int m, int c0,
                                                        int c1, int s0, int s1, const int* __restrict__ ipiv,
                                                        const int* __restrict__ org, int nsolve, int nblk,
                                                        int nskip) {
  typedef Mfma<T> MM;
  typedef typename MM::acc_t acc_t;
  constexpr int NW = SNT / 64;
  constexpr int RPP = SNT / SC;          // rows a pass moves
  constexpr int NU = SWMAX / RPP;        // passes (at most)
  __shared__ T sB[SWMAX][SC + 1];
  __shared__ T sL[SB][SB + 1];           // -L of the diagonal block, [k][i]
  __shared__ int s_top[SWMAX], s_dst[SWMAX], s_src[SWMAX];
  __shared__ int s_odd;
  int blk = blockIdx.x;
  if (nskip) {
    if (blk % 8 < nskip) return;
    blk = (blk / 8) * (8 - nskip) + (blk % 8 - nskip);
  }
  if (blk >= nblk) return;
  const bool solve = blk < nsolve;
  const int cb = solve ? c0 + blk * SC : s0 + (blk - nsolve) * SC;
  const int cend = solve ? c1 : s1;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c = tid & (SC - 1), q = tid / SC;
  const bool cok = cb + c < cend;
  T* const Tc = Tm + (cok ? cb + c : cb);
  const int nb = (w + SB - 1) / SB;
  const int kn = k0 + w;

  // the first diagonal block of L, in flight beside the interchanges
  const int lkk = tid & (SB - 1), li0 = tid / SB;
  T lv[SB * SB / SNT];
  auto load_l = [&](int b) {
#pragma unroll
    for (int u = 0; u < SB * SB / SNT; ++u) {
      const int i = SB * b + li0 + (SNT / SB) * u, k = SB * b + lkk;
      lv[u] = i < w && k < i ? Tm[(long)(k0 + k) + (long)(k0 + i) * ldt] : T(0);
    }
  };
  if (tid < w) {
    int s = org[k0 + tid];
    const int r = ipiv[k0 + tid] - 1;
    s_top[tid] = s >= k0 && s < m ? s : k0 + tid;  // (out of range only after a wait gave up)
    const bool out = r >= kn && r < m;
    int rs = out ? org[r] : -1;
    if (rs < k0 || rs >= m) rs = r;
    s_dst[tid] = out && rs != r ? r : -1;
    s_src[tid] = out ? rs : k0;
  }
  if (tid == 0) s_odd = 0;
  if (solve) load_l(0);
  __syncthreads();
  // every source in registers, all in flight together; one barrier; every
  // destination
  T v[NU], vo[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    if (RPP * u < w) {
      const int i = min(q + RPP * u, w - 1);
      v[u] = Tc[(long)s_top[i] * ldt];
      vo[u] = Tc[(long)s_src[i] * ldt];
    }
  }
  wait_vm();
  __syncthreads();
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int i = q + RPP * u;
    if (i < w && cok) {
      if (s_dst[i] >= 0) Tc[(long)s_dst[i] * ldt] = vo[u];
      if (!solve && s_top[i] != k0 + i) Tc[(long)(k0 + i) * ldt] = v[u];
    }
    if (solve && i < SB * nb) sB[i][c] = i < w && cok ? v[u] : T(0);
  }
  if (!solve) return;

  const int li = lane & 15, lk = lane >> 4;
  for (int b = 0; b < nb; ++b) {
    // -L of the block; the substitution skips a zero x(k) as the reference
    // does (BLAS/SRC/dtrsm.f:177-190), which differs from multiplying by it
    // only where L is not finite
    bool odd = false;
#pragma unroll
    for (int u = 0; u < SB * SB / SNT; ++u) {
      sL[lkk][li0 + (SNT / SB) * u] = -lv[u];
      odd |= !(fabs(lv[u]) <= (sizeof(T) == 8 ? (T)1.7976931348623157e308 : (T)3.4028234663852886e38));
    }
    if (odd) s_odd = 1;
    if (b + 1 < nb) load_l(b + 1);
    // the rows of L below the block that this wave multiplies: tile t covers
    // rows SB*(b+1) + 16t .. +15; lane (li, lk) takes row li, columns 16lk ..
    // +15 of the block (step s of the products uses column 16lk + s in both
    // operands)
    constexpr int TPW = ((SWMAX - SB) / 16 + NW - 1) / NW;  // tiles of a wave (at most)
    const int nt = (w - SB * (b + 1) + 15) / 16;
    T a[TPW][16];
#pragma unroll
    for (int z = 0; z < TPW; ++z) {
      const int t = wave + NW * z;
      if (t < nt) {
        const int i = SB * (b + 1) + 16 * t + li;
        const T* p = Tm + (long)(k0 + SB * b + 16 * lk) + (long)(k0 + min(i, w - 1)) * ldt;
#pragma unroll
        for (int s = 0; s < 16; ++s) a[z][s] = p[s];
      }
    }
    __syncthreads();
    if (wave < SC / 4) {
      const int cc = 4 * wave + lk, sub = li;
      T x[SB / 16];
#pragma unroll
      for (int z = 0; z < SB / 16; ++z) x[z] = sB[SB * b + 16 * z + sub][cc];
      if (s_odd == 0) {
        T t[SB / 16];
        solve_steps<T, 0>(x, t, sL, sub);
      } else {
        for (int k = 0; k < SB; ++k) {
          T xk = T(0);
#pragma unroll
          for (int z = 0; z < SB / 16; ++z)
            if (z == k / 16) xk = __shfl(x[z], (lane & 48) | (k & 15));
#pragma unroll
          for (int z = 0; z < SB / 16; ++z)
            if (xk != T(0) && 16 * z + sub > k) x[z] = x[z] + xk * sL[k][16 * z + sub];
        }
      }
#pragma unroll
      for (int z = 0; z < SB / 16; ++z) sB[SB * b + 16 * z + sub][cc] = x[z];
    }
    __syncthreads();
#pragma unroll
    for (int z = 0; z < TPW; ++z) {
      const int t = wave + NW * z;
      if (t < nt) {
        const int i0 = SB * (b + 1) + 16 * t;
        acc_t acc = acc_t{};
#pragma unroll
        for (int s = 0; s < 16; ++s) acc = MM::op(a[z][s], sB[SB * b + 16 * lk + s][li], acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) sB[i0 + MM::row(lk, r)][li] -= acc[r];
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int i = q + RPP * u;
    if (i < w && cok) Tc[(long)(k0 + i) * ldt] = sB[i][c];
  }
}

template <class T>
void launch_swap_trsm_t(T* Tm, long ldt, int k0, int w, int m, int c0, int c1, int s0, int s1, const int* ipiv,
                        const int* org, hipStream_t s, int nskip) {
  const int nsolve = c1 > c0 ? (c1 - c0 + SC - 1) / SC : 0;
  const int nblk = nsolve + (s1 > s0 ? (s1 - s0 + SC - 1) / SC : 0);
  if (nblk == 0 || w <= 0) return;
  const int grid = nskip ? (nblk + (8 - nskip) - 1) / (8 - nskip) * 8 : nblk;
  swap_trsm_kernel<T><<<grid, SNT, 0, s>>>(Tm, ldt, k0, w, m, c0, c1, s0, s1, ipiv, org, nsolve, nblk, nskip);
}

}  // namespace

void launch_swap_trsm_d(double* T, long ldt, int k0, int w, int m, int c0, int c1, int s0, int s1, const int* ipiv,
                        const int* org, hipStream_t s, int nskip) {
  launch_swap_trsm_t<double>(T, ldt, k0, w, m, c0, c1, s0, s1, ipiv, org, s, nskip);
}
void launch_swap_trsm_s(float* T, long ldt, int k0, int w, int m, int c0, int c1, int s0, int s1, const int* ipiv,
                        const int* org, hipStream_t s, int nskip) {
  launch_swap_trsm_t<float>(T, ldt, k0, w, m, c0, c1, s0, s1, ipiv, org, s, nskip);
}

}  // namespace la
