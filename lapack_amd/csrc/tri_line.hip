// tri_line.hip -- one right-hand side through a triangle: a sweep of DGETRS
// (SRC/dgetrs.f:181-218) as one launch.
//
// M x = y for triangular M = op(tri(A)).  A sweep reads the triangle once and is
// a chain through its diagonal blocks; every link of the chain between two
// workgroups costs a store to memory and a load from it (1 us and more across
// XCDs), so a block is as large as a workgroup can finish in about that time:
//   * one workgroup of 16 waves per 128 rows of x, ordered by a ticket taken at
//     the start: a workgroup waits only for blocks of lower tickets, which are
//     running, so every wait ends;
//   * each wave owns 1024 elements of every 128 x 128 tile of M that the block
//     depends on, reads them a tile ahead, polls the values of x it needs itself
//     (the sentinel says which are not there yet) and multiplies: no barrier
//     until the last tile is done;
//   * before the first tile both 64-row diagonal triangles are inverted, 16 x 16
//     blocks by substitution and the rest by products with them, and kept, with
//     the tile between them, in registers: 4 elements a thread, a row on 16
//     lanes.  After the last tile the two halves are a product each, and one
//     between them.
// Sums: 16 products of a tile, then one term per tile, then 8 parts.
// Bound: at n = 6001 a link takes 3.5 us (M = L, U) or 4.5 (transposed): reading a
// tile of 128 KB at what one CU gets from memory, 30 to 50 GB/s; 1.4 of it the
// way of x through memory.  64-row blocks of 4 waves with a round's x in LDS took
// 2.5 to 6.4 us for half the rows.  n = 6001, one right-hand side, FP64, with
// the permutation: 'N' 541 -> 379 us, 'T' 978 -> 468; n = 100 84 -> 43 (launches: one
// that clears, one that permutes up to 512 rows, the sweeps and one that ends).
// Every wait is bounded; one that gives up sets *err, and the others poll *err
// and give up as well, so every workgroup runs to its end.
#include "tri_block.h"
#include "mfma.h"

namespace la {
namespace {

constexpr int RB = 128;  // rows of a block

// Two (FP64) or four consecutive values with the alignment of one.
template <class T> struct LVec;
template <> struct LVec<double> {
  typedef double v __attribute__((ext_vector_type(2), aligned(8)));
  static constexpr int N = 2;
};
template <> struct LVec<float> {
  typedef float v __attribute__((ext_vector_type(4), aligned(4)));
  static constexpr int N = 4;
};

// A barrier that waits for LDS only: __syncthreads() also waits for the
// published values to be in memory.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Sum of m[e] times the x of lane e of the lane's 16.
template <class T>
__device__ __forceinline__ T dot16(const T (&m)[16], T x) {
  T p0 = T(0), p1 = T(0);
  fmac_from<0>(p0, x, m[0]);   fmac_from<1>(p1, x, m[1]);
  fmac_from<2>(p0, x, m[2]);   fmac_from<3>(p1, x, m[3]);
  fmac_from<4>(p0, x, m[4]);   fmac_from<5>(p1, x, m[5]);
  fmac_from<6>(p0, x, m[6]);   fmac_from<7>(p1, x, m[7]);
  fmac_from<8>(p0, x, m[8]);   fmac_from<9>(p1, x, m[9]);
  fmac_from<10>(p0, x, m[10]); fmac_from<11>(p1, x, m[11]);
  fmac_from<12>(p0, x, m[12]); fmac_from<13>(p1, x, m[13]);
  fmac_from<14>(p0, x, m[14]); fmac_from<15>(p1, x, m[15]);
  return p0 + p1;
}

// Sum over the 16 lanes of a row, in every lane.
template <int ROR>
__device__ __forceinline__ double ror16(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, 0x120 + ROR, 0xf, 0xf, true);
  const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), 0x120 + ROR, 0xf, 0xf, true);
  return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
}
template <int ROR>
__device__ __forceinline__ float ror16(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 + ROR, 0xf, 0xf, true));
}
template <class T>
__device__ __forceinline__ T sum16(T v) {
  v += ror16<8>(v);
  v += ror16<4>(v);
  v += ror16<2>(v);
  return v + ror16<1>(v);
}

template <class T>
struct LineLds {
  TriBlock<T> tri[2];
  T inv[2][64][66];
  T tmp[6][16][17];
  T rec[RB];
  T part[8][RB];  // the parts of a row's sum
  T y[RB];
  T x[64];        // the half solved first
  int t, failed;
};

// The inverses of both triangles into S.inv, which holds zeros (tri_block.h): the
// 16 x 16 blocks of the diagonal, then the blocks of equal i - j at once, a wave each.
template <class T, bool LOWERM, bool UNIT>
__device__ __forceinline__ void invert_triangles(LineLds<T>& S, int tid) {
  typedef Mfma<T> MM;
  constexpr Diag D = UNIT ? DIAG_UNIT : DIAG_MULTIPLY;
  const int lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  auto at = [](int i) { return LOWERM ? i : 63 - i; };
#pragma unroll 1
  for (int blk = 0; blk < 2; ++blk) {
    const int m = wave >> 2, j = tid / 16 & 15;  // block m, column (LOWERM) or row j
    const auto* const c = S.tri[blk].c[m * (m + 1) / 2 + m];
    if constexpr (LOWERM) {
      const T r = UNIT ? T(1) : S.rec[64 * blk + at(16 * m + li)];
      S.inv[blk][at(16 * m + li)][at(16 * m + j)] = diag_inverse<T, D>(r, li, j, [&](int k) { return c[k][li]; });
    } else {
      const T r = UNIT ? T(1) : S.rec[64 * blk + at(16 * m + 15 - li)];
      S.inv[blk][at(16 * m + j)][at(16 * m + 15 - li)] =
          diag_inverse_row<T, D>(r, li, j, [&](int a, int b) { return c[b][a]; });
    }
  }
#pragma unroll 1
  for (int d = 1; d < 4; ++d) {
    __syncthreads();
    const int cnt = 4 - d;
    if (wave < 2 * cnt) {
      const int blk = wave >= cnt, j = wave - blk * cnt, i = j + d;
      T(*const tmp)[17] = S.tmp[wave];
      auto V = [&](int r, int q, int a, int b) -> T& { return S.inv[blk][at(16 * r + a)][at(16 * q + b)]; };
      auto C = [&](int r, int q, int a, int b) { return S.tri[blk].c[r * (r + 1) / 2 + q][b][a]; };
      typename MM::acc_t acc = {T(0), T(0), T(0), T(0)};
#pragma unroll 1
      for (int z = 0; z < d; ++z) {
        const int k = LOWERM ? j + z : j + 1 + z;
        acc = acc + (LOWERM ? product16<T>([&](int s) { return C(i, k, li, s + lk); },
                                           [&](int s) { return V(k, j, s + lk, li); })
                            : product16<T>([&](int s) { return V(i, k, li, s + lk); },
                                           [&](int s) { return C(k, j, s + lk, li); }));
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) tmp[MM::row(lk, r)][li] = acc[r];
      wave_sync();
      acc = LOWERM ? product16<T>([&](int s) { return V(i, i, li, s + lk); }, [&](int s) { return tmp[s + lk][li]; })
                   : product16<T>([&](int s) { return tmp[li][s + lk]; }, [&](int s) { return V(j, j, s + lk, li); });
#pragma unroll
      for (int r = 0; r < 4; ++r) V(i, j, MM::row(lk, r), li) = acc[r];
    }
  }
  __syncthreads();
}

template <class T, bool LOWERM, bool UNIT, bool TRANS>
__global__ __launch_bounds__(1024) void tri_line_kernel(int n, const T* __restrict__ A, long lda, T* Xin, bool refill,
                                                        T* __restrict__ X, unsigned* ticket, int* err) {
  __shared__ LineLds<T> S;
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nblk = (n + RB - 1) / RB;
  if (tid == 0) S.failed = 0;
  if (tid == 0) S.t = (int)__hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const int t = __builtin_amdgcn_readfirstlane(S.t);
  if (t >= nblk) return;
  auto block_of = [&](int k) { return LOWERM ? k : nblk - 1 - k; };
  const int r0 = RB * block_of(t);
  auto M = [&](int i, int c) { return TRANS ? A[c + (long)i * lda] : A[i + (long)c * lda]; };

  T b, mt[4];
  // the diagonal triangles, in the order of the substitution, and the tile that
  // takes the half solved first to the other (every load unconditional, at a
  // clamped place, so that they are in flight together)
  constexpr int F = LOWERM ? 0 : 1, L = 1 - F;
  const int pr = tid >> 4, ps = tid & 15;  // row pr of a half, columns 4 ps .. + 3
  {
    const int a = tid & 15, c = (tid & 255) >> 4;  // a: the index that is contiguous in memory
    auto place = [&](int u, int& blk, int& sb, int& gi, int& gk) {
      const int s2 = tid / 256 + 4 * u;
      blk = s2 >= 10;
      sb = s2 - 10 * blk;
      const int mi = sb >= 6 ? 3 : sb >= 3 ? 2 : sb >= 1 ? 1 : 0, mk = sb - mi * (mi + 1) / 2;
      const int i = 16 * mi + (TRANS ? c : a), k = 16 * mk + (TRANS ? a : c);
      gi = r0 + 64 * blk + (LOWERM ? i : 63 - i);
      gk = r0 + 64 * blk + (LOWERM ? k : 63 - k);
    };
    auto at = [&](int i, int k) { return M(min(i, n - 1), min(k, n - 1)); };
    T v[5], mt0[4];
#pragma unroll
    for (int u = 0; u < 5; ++u) {
      int blk, sb, gi, gk;
      place(u, blk, sb, gi, gk);
      v[u] = at(gi, gk);
    }
    const int li2 = r0 + 64 * L + pr, lc2 = r0 + 64 * F + 4 * ps;
#pragma unroll
    for (int j = 0; j < 4; ++j) mt0[j] = at(li2, lc2 + j);
    const int g = min(r0 + (tid & (RB - 1)), n - 1);
    const T b0 = Xin[g], d0 = UNIT ? T(1) : A[g + (long)g * lda];
#pragma unroll
    for (int u = 0; u < 5; ++u) {
      int blk, sb, gi, gk;
      place(u, blk, sb, gi, gk);
      const bool in = (LOWERM ? gi > gk : gi < gk) && max(gi, gk) < n;
      S.tri[blk].c[sb][TRANS ? a : c][TRANS ? c : a] = in ? -v[u] : T(0);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      mt[j] = li2 < n && lc2 + j < n ? mt0[j] : T(0);
      asm volatile("" : "+v"(mt[j]));  // (here, not on the chain)
    }
    const bool in = r0 + (tid & (RB - 1)) < n;
    b = in ? b0 : T(0);
    if (tid < RB) S.rec[tid] = !UNIT && in ? T(1) / d0 : T(1);
#pragma unroll
    for (int u = 0; u < 8; ++u) S.inv[u / 4][(tid >> 6) + 16 * (u & 3)][lane] = T(0);
  }
  __syncthreads();
  // (a block's right side is read by its own workgroup only: its place can wait
  // for the values of the next sweep)
  if (refill && tid < RB && r0 + tid < n) Xin[r0 + tid] = __builtin_bit_cast(T, Sent<T>::bits);
  invert_triangles<T, LOWERM, UNIT>(S, tid);
  T inv[2][4];
#pragma unroll
  for (int blk = 0; blk < 2; ++blk)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      inv[blk][j] = S.inv[blk][pr][4 * ps + j];
      asm volatile("" : "+v"(inv[blk][j]));  // (kept: not read again on the chain)
    }

  // the tiles: wave w has, transposed, rows 16 (w / 2) .. and columns 64 (w % 2)
  // .. (lane (li, lk): row li, columns 16 c + 4 lk + 0..3); otherwise rows 64 (w %
  // 2) .. and columns 16 (w / 2) .. (a row a lane)
  const int wr = TRANS ? 16 * (wave >> 1) : 64 * (wave & 1), wc = TRANS ? 64 * (wave & 1) : 16 * (wave >> 1);
  const int row = min(r0 + wr + (TRANS ? li : lane), n - 1);
  auto load = [&](T(&m)[16], int k) {
    const int c0 = RB * block_of(k) + wc;
    if (TRANS) {
      typedef LVec<T> V;
      const T* p = A + (long)row * lda;
      if (c0 + 64 <= n) {
        p += c0 + 4 * lk;
#pragma unroll
        for (int e = 0; e < 16; e += V::N) {
          const typename V::v v = *reinterpret_cast<const typename V::v*>(p + 16 * (e / 4) + (e & 3));
#pragma unroll
          for (int q = 0; q < V::N; ++q) m[e + q] = v[q];
        }
      } else {
        T v[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = p[min(c0 + 4 * lk + 16 * (e / 4) + (e & 3), n - 1)];
#pragma unroll
        for (int e = 0; e < 16; ++e) m[e] = c0 + 4 * lk + 16 * (e / 4) + (e & 3) < n ? v[e] : T(0);
      }
    } else {
      T v[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) v[e] = (A + (long)min(c0 + e, n - 1) * lda)[(unsigned)row];
      if (c0 + 16 > n) {
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = c0 + e < n ? v[e] : T(0);
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) m[e] = v[e];
    }
  };
  bool failed = false;
  T acc = T(0);
  auto step = [&](const T(&m)[16], int k) {
    // (value e of a lane's 16 is multiplied by the x that lane e of its row of 16 lanes holds)
    const int c = RB * block_of(k) + wc + (TRANS ? 16 * (li >> 2) + 4 * lk + (li & 3) : li);
    const T* const px = X + min(c, n - 1);
    T x;
    for (unsigned spins = 0;;) {
      x = ld_dev(px);
      if (!__any(is_sent(x))) break;
      if (t - k > 2) __builtin_amdgcn_s_sleep(8);  // (its turn is not near: fewer loads)
      else __builtin_amdgcn_s_sleep(1);
      ++spins;
      if ((spins & 255u) == 0u && ld_dev(err) != 0) { failed = true; return; }
      if (spins > SPIN_LIMIT) { st_dev(err, 1); failed = true; return; }
    }
    x = c < n ? x : T(0);
    acc += dot16(m, x);
  };
  T m0[16], m1[16];
  if (t > 0) load(m0, 0);
  for (int k = 0; k < t && !failed; k += 2) {
    if (k + 1 < t) load(m1, k + 1);
    step(m0, k);
    if (k + 1 < t && !failed) {
      if (k + 2 < t) load(m0, k + 2);
      step(m1, k + 1);
    }
  }
  if (failed && lane == 0) S.failed = 1;
  S.part[TRANS ? 4 * (wave & 1) + lk : wave >> 1][wr + (TRANS ? li : lane)] = acc;
  lds_barrier();
  if (S.failed) return;
  if (tid < RB) {
    const T s0 = S.part[0][tid] + S.part[1][tid], s1 = S.part[2][tid] + S.part[3][tid];
    const T s2 = S.part[4][tid] + S.part[5][tid], s3 = S.part[6][tid] + S.part[7][tid];
    S.y[tid] = b - ((s0 + s1) + (s2 + s3));
  }
  lds_barrier();
  // row pr of a 64 x 64 matrix times v
  auto product = [&](const T(&a)[4], const T* v) {
    const T p0 = fma(a[2], v[4 * ps + 2], a[0] * v[4 * ps]), p1 = fma(a[3], v[4 * ps + 3], a[1] * v[4 * ps + 1]);
    return sum16(p0 + p1);
  };
  const T xf = product(inv[F], S.y + 64 * F);
  if (ps == 0) S.x[pr] = xf;
  lds_barrier();
  if (ps == 0 && r0 + 64 * F + pr < n) st_dev(X + r0 + 64 * F + pr, canon(xf));
  const T d = product(mt, S.x);
  if (ps == 0) S.y[64 * L + pr] -= d;
  lds_barrier();
  const T xl = product(inv[L], S.y + 64 * L);
  if (ps == 0 && r0 + 64 * L + pr < n) st_dev(X + r0 + 64 * L + pr, canon(xl));
}

// A wait gave up (not where the solve was called off by the factorization's INFO).
__device__ __forceinline__ void report_wait(int* waitflag, int* sticky, const int* gate) {
  if (gate && *gate != 0) return;
  if (waitflag) *waitflag = LA_ERR_SYNC;
  if (sticky) atomicOr(sticky, 1);
}

// Start of a solve: the wait-error word (set where the factorization has an INFO,
// and by the test hook), the sweeps' tickets, the first sweep's sentinels and, for a
// b that is not interchanged first, its right side.
template <class T>
__global__ __launch_bounds__(256) void line_init_kernel(int n, const T* __restrict__ b, T* X, T* Y, unsigned* tickets,
                                                        int* err, int fail, const int* __restrict__ gate) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) Y[i] = __builtin_bit_cast(T, Sent<T>::bits);
  if (b && i < n) X[i] = b[i];
  if (i < 2) tickets[i] = 0u;
  if (i == 0) *err = fail || (gate && *gate != 0);
}

// End of a solve: dst = src unless a wait gave up, which is reported instead.
template <class T>
__global__ __launch_bounds__(256) void line_end_kernel(int n, const T* __restrict__ src, T* __restrict__ dst,
                                                       const int* __restrict__ err, int* waitflag, int* sticky,
                                                       const int* __restrict__ gate) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  const bool failed = *err != 0;
  if (!failed && i < n) dst[i] = src[i];
  if (failed && i == 0) report_wait(waitflag, sticky, gate);
}

// dst = src with its rows interchanged, for columns that fit in LDS: one
// workgroup, the interchanges composed by its first wave (11 us at n = 512
// where composing them for any n, with the gather, takes three launches and 23).
// err: nothing is written where it is set, but it is reported.
constexpr int PERM_NMAX = 512;
template <class T, bool REVERSE>
__global__ __launch_bounds__(256) void permute_small_kernel(int n, const int* __restrict__ ipiv,
                                                            const T* __restrict__ src, T* __restrict__ dst,
                                                            const int* __restrict__ err, int* waitflag, int* sticky,
                                                            const int* __restrict__ gate) {
  __shared__ T x[PERM_NMAX];
  const int tid = threadIdx.x;
  if (err && *err != 0) {
    if (tid == 0) report_wait(waitflag, sticky, gate);
    return;
  }
  for (int i = tid; i < n; i += 256) x[i] = src[i];
  __syncthreads();
  if (tid < 64) interchange<T, REVERSE>(ipiv, n, x, 0, 1, tid);
  __syncthreads();
  for (int i = tid; i < n; i += 256) dst[i] = x[i];
}

void gather(int n, const int* perm, const double* src, double* dst, hipStream_t s) {
  launch_gather_rows_d(n, 1, perm, src, n, dst, n, s);
}
void gather(int n, const int* perm, const float* src, float* dst, hipStream_t s) {
  launch_gather_rows_s(n, 1, perm, src, n, dst, n, s);
}

template <class T>
void launch_line(int which, int n, const T* A, long lda, T* Xin, bool refill, T* X, unsigned* ticket, int* err,
                 hipStream_t s) {
  const int nblk = (n + RB - 1) / RB;
  switch (which) {
    case 0: tri_line_kernel<T, true, true, false><<<nblk, 1024, 0, s>>>(n, A, lda, Xin, refill, X, ticket, err); break;
    case 1: tri_line_kernel<T, false, false, false><<<nblk, 1024, 0, s>>>(n, A, lda, Xin, refill, X, ticket, err); break;
    case 2: tri_line_kernel<T, true, false, true><<<nblk, 1024, 0, s>>>(n, A, lda, Xin, refill, X, ticket, err); break;
    case 3: tri_line_kernel<T, false, true, true><<<nblk, 1024, 0, s>>>(n, A, lda, Xin, refill, X, ticket, err); break;
  }
}

}  // namespace

// which: 0 = L (unit lower), 1 = U (upper), 2 = U^T, 3 = L^T.  X is filled with
// the sentinel and *ticket is 0.
template <class T>
void launch_tri_line(int which, int n, const T* A, long lda, const T* Xin, T* X, unsigned* ticket, int* err,
                     hipStream_t s) {
  launch_line<T>(which, n, A, lda, const_cast<T*>(Xin), false, X, ticket, err, s);
}
template void launch_tri_line<double>(int, int, const double*, long, const double*, double*, unsigned*, int*,
                                      hipStream_t);
template void launch_tri_line<float>(int, int, const float*, long, const float*, float*, unsigned*, int*, hipStream_t);

// DGETRS of one right-hand side b (SRC/dgetrs.f:181-218): X and Y n values,
// tickets two words, perm and gpairs as launch_swaps_to_perm takes them.
template <class T>
void launch_getrs_line(bool notran, int n, const T* A, long lda, const int* ipiv, T* b, T* X, T* Y, unsigned* tickets,
                       int* err, int* perm, int* gpairs, bool fail, const int* gate, int* waitflag, int* sticky,
                       hipStream_t s) {
  const int nb = (n + 255) / 256;
  line_init_kernel<T><<<nb, 256, 0, s>>>(n, notran ? nullptr : b, X, Y, tickets, err, fail ? 1 : 0, gate);
  const bool small = n <= PERM_NMAX;
  if (notran) {
    if (small) {
      permute_small_kernel<T, false><<<1, 256, 0, s>>>(n, ipiv, b, X, nullptr, nullptr, nullptr, nullptr);
    } else {
      launch_swaps_to_perm(n, 0, n, ipiv, 1, perm, s, gpairs);
      gather(n, perm, b, X, s);
    }
    launch_line<T>(0, n, A, lda, X, true, Y, tickets, err, s);
    launch_line<T>(1, n, A, lda, Y, false, X, tickets + 1, err, s);
    line_end_kernel<T><<<nb, 256, 0, s>>>(n, X, b, err, waitflag, sticky, gate);
    return;
  }
  launch_line<T>(2, n, A, lda, X, true, Y, tickets, err, s);
  launch_line<T>(3, n, A, lda, Y, false, X, tickets + 1, err, s);
  if (small) {
    permute_small_kernel<T, true><<<1, 256, 0, s>>>(n, ipiv, X, b, err, waitflag, sticky, gate);
  } else {
    launch_swaps_to_perm(n, 0, n, ipiv, -1, perm, s, gpairs);
    gather(n, perm, X, Y, s);
    line_end_kernel<T><<<nb, 256, 0, s>>>(n, Y, b, err, waitflag, sticky, gate);
  }
}
template void launch_getrs_line<double>(bool, int, const double*, long, const int*, double*, double*, double*,
                                        unsigned*, int*, int*, int*, bool, const int*, int*, int*, hipStream_t);
template void launch_getrs_line<float>(bool, int, const float*, long, const int*, float*, float*, float*, unsigned*,
                                       int*, int*, int*, bool, const int*, int*, int*, hipStream_t);

}  // namespace la
