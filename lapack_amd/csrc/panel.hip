// panel.hip -- leaf factorization of a tall panel (the unblocked core of
// DGETRF2, SRC/dgetrf2.f:179-214 applied column by column).
//
// The panel is A(j0:m-1, j0:j0+w-1) of the matrix being factored, held in the
// transposed workspace T = A^T, so matrix row r of the panel is T column r and
// its w values are contiguous.  Three forms, chosen by the panel height h:
//   * h <= 512, and h <= 1024 in a matrix of no more rows: one workgroup keeps
//     the whole leaf in registers (getf2_leaf_kernel) and waits for nobody;
//   * other h <= 32768: G = h/512 workgroups keep it in registers and agree
//     on each column's pivot through a flag-in-data exchange in device memory
//     (the same kernel; needs its G workgroups resident together);
//   * taller panels, and every leaf of a factorization being redone after a
//     bounded wait gave up: one column per two launches over the leaf in HBM
//     (tall_*_kernel), no workgroup waits for another.
// Per column k every form does:
//   1. pivot search under the IDAMAX rule of BLAS/SRC/idamax.f:101-107 (first
//      index of max |x|, strict '>', a NaN at the head of the column wins, NaNs
//      elsewhere never do).  Each candidate gets a 64-bit key that orders
//      exactly like that rule: bits(|x|)+1 (IEEE bit patterns of non-negative
//      doubles sort like their values), row k's NaN -> bits(+inf)+1, other
//      NaNs -> 1, rows outside the active range -> 0; ties go to the lowest
//      row.  A wave takes the max key with DPP row shifts/broadcasts and the
//      lowest lane holding it with a ballot;
//   2. interchange (row k takes the pivot row, the pivot row takes the old row
//      k: SRC/dgetrf2.f:196-200), scaling by the reciprocal of the pivot, or
//      division when |pivot| < sfmin (SRC/dgetrf2.f:204-210), and the rank-1
//      update of the remaining columns (SRC/dgetrf2.f:245-246 one column at a
//      time), applied also for a zero pivot as the reference's DGEMM has no
//      zero test.  Every form does the same operations on each element in
//      FP64; in FP32 the register forms sum a group's products before they
//      join the element (leaf.h), so only their last bits depend on the form.
// IPIV receives absolute 1-based rows; INFO the first exact zero pivot
// (SRC/dgetrf2.f:192,212-214).  Every wait is bounded: a timeout sets *err,
// later waits give up at once, and the kernel always runs to its end.
#include "leaf.h"

#include <cstdlib>
#include <cstring>

namespace la {
namespace {

template <class T> struct Sfmin;
template <> struct Sfmin<double> { static constexpr double v = 0x1p-1022; };
template <> struct Sfmin<float> { static constexpr float v = 0x1p-126f; };

// XCDs a rank-mode panel of G workgroups occupies (32 CUs each).
__host__ __device__ __forceinline__ unsigned panel_xcds(int G) { return (unsigned)((G + 31) / 32); }

// The leaf A(j0:m-1, j0:j0+w-1) in registers (leaf.h).
template <class T, int W, int NTH, bool MULTI, bool XCD0, int DIRECT = 0>
__global__ __launch_bounds__(NTH) void getf2_leaf_kernel(T* __restrict__ Tm, long ldt, int j0, int w, int m,
                                                        int* __restrict__ ipiv, int* __restrict__ info,
                                                        unsigned tagbase, u64* __restrict__ xbuf,
                                                        int* __restrict__ err, int Gp, unsigned* __restrict__ ctr,
                                                        RowOrg org) {
  constexpr int NW = NTH / 64;
  constexpr int CP = NTH >= 1024 ? 8 : 16;  // columns of a piece (below)
  // (the leaf's first: 16 bits of offset reach the first 64 KB of LDS only)
  __shared__ struct {
    LeafLds<T, W, NTH, MULTI> leaf;
    int rank;
    T stage[NW][64][CP + 1];
  } s_all;
  auto& S = s_all.leaf;
  int& s_rank = s_all.rank;
  auto& s_stage = s_all.stage;
  const int tid = threadIdx.x;
  int G = gridDim.x;
  int b = blockIdx.x;
  if (XCD0) {
    // The blocks that run on XCD 0 (hardware register XCC_ID) take ranks in
    // arrival order (ctr[0]); the first Gp of them take part, rank r owning
    // rows [r*NTH, r*NTH + NTH), so the panel owns XCD 0's CUs while the
    // update leaves them alone; every other block leaves.  Each block then
    // counts its arrival (ctr[1]); the last to arrive -- every rank decision
    // is then made -- sets *err when fewer than Gp blocks ran on XCD 0, so
    // that every wait gives up and the call reports the failure instead of
    // leaving rows unfactored, and resets both counters for the next launch.
    if (tid == 0) {
      int r = -1;
      if ((__builtin_amdgcn_s_getreg(6164) & 15u) == 0u)  // HW_REG_XCC_ID
        r = (int)__hip_atomic_fetch_add(&ctr[0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const unsigned arrived = __hip_atomic_fetch_add(&ctr[1], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
      if (arrived == gridDim.x - 1) {
        const unsigned ranks = __hip_atomic_load(&ctr[0], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
        if (ranks < (unsigned)Gp) st_dev(err, 1);
        __hip_atomic_store(&ctr[0], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&ctr[1], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      s_rank = (r >= 0 && r < Gp) ? r : -1;
    }
    __syncthreads();
    if (s_rank < 0) return;
    G = Gp;
    b = __builtin_amdgcn_readfirstlane(s_rank);
  }
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = m - j0;
  const int kmax = min(h, w);
  const int wrow0 = b * NTH + wave * 64;       // the wave's first row
  const int lr = b * NTH + tid;
  if (MULTI && tid == 0) S.fail = 0;

  // The wave's 64 rows in and out through LDS, CP columns at a time: an access
  // of the matrix touches whole runs of CP values of 64 / CP rows (a row a lane
  // would touch 64 lines an instruction).  (16 waves' share of LDS is half.)
  constexpr int RP = 64 / CP;  // rows of one access
  T v[W];
  {
    const int c0 = lane & (CP - 1), q0 = lane / CP;
    const T* base = Tm + (long)(j0 + wrow0 + q0) * ldt + j0 + c0;
#pragma unroll
    for (int i = 0; i < W; ++i) {
      const int r = wrow0 + q0 + RP * (i % CP), c = c0 + CP * (i / CP);
      v[i] = r < h && c < w ? base[(long)(RP * (i % CP)) * ldt + CP * (i / CP)] : T(0);
    }
#pragma unroll
    for (int cp = 0; cp < W / CP; ++cp) {
#pragma unroll
      for (int i = 0; i < CP; ++i) s_stage[wave][q0 + RP * i][c0] = v[CP * cp + i];
      wave_sync();
#pragma unroll
      for (int i = 0; i < CP; ++i) v[CP * cp + i] = s_stage[wave][lane][i];
      wave_sync();
    }
  }
  // the row's loads complete here, before the column loop: left pending,
  // they would make the compiler wait for every outstanding memory operation
  // (the exchange's stores included) wherever the loop first reads v
  wait_vm();
  int my_piv, corg, zero_at;
  leaf_columns<T, W, NTH, MULTI, XCD0, (NTH < 1024), DIRECT>(v, S, h, w, b, G, tagbase, xbuf, err, my_piv, corg, zero_at);
  if (lr < h) {
    const int o = j0 + (corg >= 0 && corg < h ? corg : lr);  // (out of range only after a wait gave up)
    const int po = org.pin ? org.pin[o] : o;
    org.leaf[j0 + lr] = o;
    org.pout[j0 + lr] = po;
    if (org.last || lr < kmax) org.fin[j0 + lr] = po;
  }
  if (b == 0 && wave == NW - 1) {
    if (lane < kmax) ipiv[j0 + lane] = j0 + my_piv + 1;
    if (lane == 0 && zero_at >= 0) atomicCAS(info, 0, j0 + zero_at + 1);
  }
  {
    const int c0 = lane & (CP - 1), q0 = lane / CP;
    T* base = Tm + (long)(j0 + wrow0 + q0) * ldt + j0 + c0;
#pragma unroll
    for (int cp = 0; cp < W / CP; ++cp) {
#pragma unroll
      for (int i = 0; i < CP; ++i) s_stage[wave][lane][i] = v[CP * cp + i];
      wave_sync();
#pragma unroll
      for (int i = 0; i < CP; ++i) {
        const int r = wrow0 + q0 + RP * i, c = c0 + CP * cp;
        const T x = s_stage[wave][q0 + RP * i][c0];
        if (r < h && c < w) base[(long)(RP * i) * ldt + CP * cp] = x;
      }
      wave_sync();
    }
  }
}

// ---- tall leaf: one column per two launches -----------------------------------
// For panels taller than GMAX register-resident workgroups hold, and for the
// leaves of a factorization redone after a bounded wait gave up: the leaf
// stays in HBM and no workgroup ever waits for another.  Column k:
//   tall_final   one workgroup folds the per-workgroup maxima of column k
//                (IDAMAX keys as above), writes IPIV and INFO, and copies the
//                pivot row and row k of the leaf to the scratch;
//   tall_update  every row r > k of the leaf: the interchange, the scaling and
//                the rank-1 update, in the same operations as the register
//                forms; row k takes the pivot row.  Each workgroup also
//                leaves the maximum key of column k+1 over its rows for the
//                next tall_final.
// tall_keys gives column 0 its maxima.  Rows past the leaf's w columns are
// never touched.
constexpr int TALL_NB = 512;  // workgroups of tall_update / tall_keys (at most)

struct TallBuf {
  u64 key[TALL_NB];
  int row[TALL_NB];
  double prow[WMAX];
  double rowk[WMAX];
  int p;
};

__device__ __forceinline__ void key_fold(u64& k, int& r, u64 k2, int r2) {
  if (k2 > k || (k2 == k && r2 < r)) { k = k2; r = r2; }
}

// workgroup maximum of (key, row) -> tb->key/row[blockIdx.x]
__device__ __forceinline__ void tall_block_max(u64 k, int r, TallBuf* tb) {
  __shared__ u64 sk[4];
  __shared__ int sr[4];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const u64 k2 = ((u64)(unsigned)__shfl_xor((int)(unsigned)(k >> 32), off) << 32) |
                   (u64)(unsigned)__shfl_xor((int)(unsigned)(k & 0xffffffffull), off);
    const int r2 = __shfl_xor(r, off);
    key_fold(k, r, k2, r2);
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) { sk[wave] = k; sr[wave] = r; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int x = 1; x < (int)(blockDim.x >> 6); ++x) key_fold(k, r, sk[x], sr[x]);
    tb->key[blockIdx.x] = k;
    tb->row[blockIdx.x] = r;
  }
}

template <class T>
__global__ __launch_bounds__(256) void tall_keys_kernel(const T* __restrict__ Tm, long ldt, int j0, int k, int h,
                                                        TallBuf* __restrict__ tb) {
  u64 best = 0ull;
  int brow = 0x7fffffff;
  for (long r = k + (long)blockIdx.x * 256 + threadIdx.x; r < h; r += (long)gridDim.x * 256) {
    const u64 key = pivot_key(Tm[(long)(j0 + r) * ldt + j0 + k], r == k);
    key_fold(best, brow, key, (int)r);
  }
  tall_block_max(best, brow, tb);
}

template <class T>
__global__ __launch_bounds__(256) void tall_final_kernel(const T* __restrict__ Tm, long ldt, int j0, int k, int w,
                                                         int nparts, int* __restrict__ ipiv, int* __restrict__ info,
                                                         TallBuf* __restrict__ tb) {
  __shared__ u64 sk[4];
  __shared__ int sr[4];
  __shared__ int s_p;
  u64 best = 0ull;
  int brow = 0x7fffffff;
  for (int x = threadIdx.x; x < nparts; x += 256) key_fold(best, brow, tb->key[x], tb->row[x]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const u64 k2 = ((u64)(unsigned)__shfl_xor((int)(unsigned)(best >> 32), off) << 32) |
                   (u64)(unsigned)__shfl_xor((int)(unsigned)(best & 0xffffffffull), off);
    const int r2 = __shfl_xor(brow, off);
    key_fold(best, brow, k2, r2);
  }
  if ((threadIdx.x & 63) == 0) { sk[threadIdx.x >> 6] = best; sr[threadIdx.x >> 6] = brow; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int x = 1; x < 4; ++x) key_fold(best, brow, sk[x], sr[x]);
    // every active row has a key >= 1, so the fold always names a row of [k, h)
    const int p = (brow >= k && brow != 0x7fffffff) ? brow : k;
    s_p = p;
    tb->p = p;
    ipiv[j0 + k] = j0 + p + 1;
  }
  __syncthreads();
  const int p = s_p;
  if ((int)threadIdx.x < w) {
    const T pv = Tm[(long)(j0 + p) * ldt + j0 + threadIdx.x];
    tb->prow[threadIdx.x] = (double)pv;
    tb->rowk[threadIdx.x] = (double)Tm[(long)(j0 + k) * ldt + j0 + threadIdx.x];
    if ((int)threadIdx.x == k && pv == T(0)) atomicCAS(info, 0, j0 + k + 1);
  }
}

template <class T>
__global__ __launch_bounds__(256) void tall_update_kernel(T* __restrict__ Tm, long ldt, int j0, int k, int w, int h,
                                                          TallBuf* __restrict__ tb, int next_keys) {
  __shared__ T s_prow[WMAX], s_rowk[WMAX];
  const int p = tb->p;
  if ((int)threadIdx.x < WMAX) {
    s_prow[threadIdx.x] = (int)threadIdx.x < w ? (T)tb->prow[threadIdx.x] : T(0);
    s_rowk[threadIdx.x] = (int)threadIdx.x < w ? (T)tb->rowk[threadIdx.x] : T(0);
  }
  __syncthreads();
  const T piv = s_prow[k];
  const T sfmin = Sfmin<T>::v;
  u64 best = 0ull;
  int brow = 0x7fffffff;
  for (long r = k + (long)blockIdx.x * 256 + threadIdx.x; r < h; r += (long)gridDim.x * 256) {
    T* row = Tm + (long)(j0 + r) * ldt + j0;
    if (r == k) {
      for (int c = 0; c < w; ++c) row[c] = s_prow[c];
      continue;
    }
    const bool isp = r == p;
    T l = isp ? s_rowk[k] : row[k];
    if (piv != T(0)) l = (fabs(piv) >= sfmin) ? (T(1) / piv) * l : l / piv;
    if (isp)
      for (int c = 0; c < k; ++c) row[c] = s_rowk[c];
    row[k] = l;
    for (int c = k + 1; c < w; ++c) {
      const T x = isp ? s_rowk[c] : row[c];
      const T u = x - l * s_prow[c];
      row[c] = u;
      if (c == k + 1 && next_keys) key_fold(best, brow, pivot_key(u, r == k + 1), (int)r);
    }
  }
  if (next_keys) tall_block_max(best, brow, tb);
}

// The record of the tall form's interchanges (RowOrg), from IPIV: a row a thread,
// followed back through the at most 64 interchanges.
__global__ __launch_bounds__(256) void tall_org_kernel(int j0, int kmax, int m, const int* __restrict__ ipiv,
                                                       RowOrg org) {
  __shared__ int s_p[WMAX];
  if ((int)threadIdx.x < kmax) {
    const int k = j0 + (int)threadIdx.x, p = ipiv[k] - 1;
    s_p[threadIdx.x] = p > k && p < m ? p : k;
  }
  __syncthreads();
  const int r = j0 + (int)(blockIdx.x * 256 + threadIdx.x);
  if (r >= m) return;
  int o = r;
  for (int k = kmax - 1; k >= 0; --k) o = o == j0 + k ? s_p[k] : o == s_p[k] ? j0 + k : o;
  const int po = org.pin ? org.pin[o] : o;
  org.leaf[r] = o;
  org.pout[r] = po;
  if (org.last || r < j0 + kmax) org.fin[r] = po;
}

}  // namespace

// Launch configurations: one workgroup with a thread a row up to 512 rows
// (fewer threads for the shorter leaves: fewer waves to fold and to wait for).
// Beyond that G workgroups of 512 threads; past GMAX workgroups the tall form.
// A matrix of 513 to 1024 rows takes one workgroup of 1024 threads instead
// (128 registers each: 32 FP64 or 64 FP32 columns), and so has no wait that could
// give up where another kernel holds XCD 0.  Two of 512 take as long at n = 600 and
// 800 (1.22 and 1.73 ms) and 2 % less at 1024 (2.22 ms, 2.26).  Taller matrices
// have leaves of more than two workgroups, which wait in any case.
static size_t tall_offset() { return (sizeof(u64) * LL_WORDS + 255) / 256 * 256; }
// the XCD-0 panel's rank and arrival counters (zeroed with the exchange
// buffer at the start of a factorization; each launch resets its own)
static size_t rank_offset() { return tall_offset() + (sizeof(TallBuf) + 255) / 256 * 256; }
size_t panel_xchg_bytes(int) { return rank_offset() + 256; }

// Workgroups the panel kernel uses at height h of an m-row matrix (0 = a single
// workgroup), and the widest leaf it takes there.
int panel_groups(int h, int m) { return h <= 512 || m <= 1024 ? 0 : (h + 511) / 512; }
int panel_max_width(int h, int m, int elem) { return h > 512 && m <= 1024 && elem == 8 ? 32 : WMAX; }

// mode: PANEL_PLAIN (G workgroups), PANEL_XCD0 (8*G blocks, those of the
// first XCDs take part), PANEL_TALL (the form without waits).
template <class T>
static int launch_panel_t(T* Tm, long ldt, int j0, int w, int m, int* ipiv, int* info, unsigned tagbase,
                          double* xchg, int* err, int mode, const RowOrg& org, hipStream_t s) {
  const int h = m - j0;
  if (h <= 0 || w <= 0) return 0;
  if (w > panel_max_width(h, m, (int)sizeof(T))) return LA_ERR_LIMIT;
  u64* xb = reinterpret_cast<u64*>(xchg);
#define LA_LEAF(W, NTH, MULTI, XCD0, DIRECT, blocks, g, ctr) \
  getf2_leaf_kernel<T, W, NTH, MULTI, XCD0, DIRECT><<<blocks, NTH, 0, s>>>(Tm, ldt, j0, w, m, ipiv, info, tagbase, xb, \
                                                                      err, g, ctr, org)
  if (panel_groups(h, m) == 0) {
    if (h <= 128) LA_LEAF(64, 128, false, false, 0, 1, 1, nullptr);
    else if (h <= 256) LA_LEAF(64, 256, false, false, 0, 1, 1, nullptr);
    else if (h <= 512) LA_LEAF(64, 512, false, false, 0, 1, 1, nullptr);
    else LA_LEAF((sizeof(T) == 8 ? 32 : 64), 1024, false, false, 0, 1, 1, nullptr);
    return 0;
  }
  const int G = (h + 511) / 512;
  if (G > GMAX || mode == PANEL_TALL) {
    TallBuf* tb = reinterpret_cast<TallBuf*>(reinterpret_cast<char*>(xchg) + tall_offset());
    const int kmax = h < w ? h : w;
    auto parts = [&](int k) {
      const long rows = (long)h - k;
      const long g = (rows + 255) / 256;
      return (int)(g < TALL_NB ? (g < 1 ? 1 : g) : TALL_NB);
    };
    tall_keys_kernel<T><<<parts(0), 256, 0, s>>>(Tm, ldt, j0, 0, h, tb);
    for (int k = 0; k < kmax; ++k) {
      tall_final_kernel<T><<<1, 256, 0, s>>>(Tm, ldt, j0, k, w, parts(k), ipiv, info, tb);
      // the update's grid is also the next column's number of maxima
      tall_update_kernel<T><<<parts(k + 1 < kmax ? k + 1 : k), 256, 0, s>>>(Tm, ldt, j0, k, w, h, tb,
                                                                            k + 1 < kmax ? 1 : 0);
    }
    tall_org_kernel<<<(h + 255) / 256, 256, 0, s>>>(j0, kmax, m, ipiv, org);
    return 0;
  }
  unsigned* const ctr = reinterpret_cast<unsigned*>(reinterpret_cast<char*>(xchg) + rank_offset());
  const int direct = G <= 8 ? 1 : G <= 16 ? 2 : 0;
  if (mode == PANEL_XCD0) {
    const int blocks = (8 / (int)panel_xcds(G)) * G;
    if (direct == 1) LA_LEAF(64, 512, true, true, 1, blocks, G, ctr);
    else if (direct == 2) LA_LEAF(64, 512, true, true, 2, blocks, G, ctr);
    else LA_LEAF(64, 512, true, true, 0, blocks, G, ctr);
  } else {
    if (direct == 1) LA_LEAF(64, 512, true, false, 1, G, G, nullptr);
    else if (direct == 2) LA_LEAF(64, 512, true, false, 2, G, G, nullptr);
    else LA_LEAF(64, 512, true, false, 0, G, G, nullptr);
  }
#undef LA_LEAF
  return 0;
}

int launch_getf2_panel_d(double* T, long ldt, int j0, int w, int m, int* ipiv, int* info, unsigned tagbase,
                         double* xchg, int* err, int mode, const RowOrg& org, hipStream_t s) {
  return launch_panel_t<double>(T, ldt, j0, w, m, ipiv, info, tagbase, xchg, err, mode, org, s);
}
int launch_getf2_panel_s(float* T, long ldt, int j0, int w, int m, int* ipiv, int* info, unsigned tagbase,
                         double* xchg, int* err, int mode, const RowOrg& org, hipStream_t s) {
  return launch_panel_t<float>(T, ldt, j0, w, m, ipiv, info, tagbase, xchg, err, mode, org, s);
}

}  // namespace la
