// panel.hip -- leaf factorization of a tall panel (the unblocked core of
// DGETRF2, SRC/dgetrf2.f:179-214 applied column by column).
//
// The panel is A(j0:m-1, j0:j0+w-1) of the matrix being factored, held in the
// transposed workspace T = A^T, so matrix row r of the panel is T column r and
// its w values are contiguous.  Three forms, chosen by the panel height h:
//   * h <= 512: one workgroup keeps the whole leaf in registers
//     (getf2_leaf_kernel);
//   * 512 < h <= 32768: G = h/512 workgroups keep it in registers and agree
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
//      zero test.  Every form does the same operations on each element, so
//      the factors do not depend on the form.
// IPIV receives absolute 1-based rows; INFO the first exact zero pivot
// (SRC/dgetrf2.f:192,212-214).  Every wait is bounded: a timeout sets *err,
// later waits give up at once, and the kernel always runs to its end.
#include "la_common.h"

#include <cstdlib>
#include <cstring>

namespace la {
namespace {

constexpr int GMAX = 64;            // workgroups of a register-resident leaf
constexpr int WMAX = 64;            // widest leaf

template <class T> struct Sfmin;
template <> struct Sfmin<double> { static constexpr double v = 0x1p-1022; };
template <> struct Sfmin<float> { static constexpr float v = 0x1p-126f; };

typedef unsigned long long u64;

// XCDs a rank-mode panel of G workgroups occupies (32 CUs each).
__host__ __device__ __forceinline__ unsigned panel_xcds(int G) { return (unsigned)((G + 31) / 32); }

// Pivot key of the tall form: see the header comment.
template <class T>
__device__ __forceinline__ u64 pivot_key(T x, bool is_k) {
  const double a = fabs((double)x);
  if (a != a) return is_k ? 0x7FF0000000000001ull : 1ull;
  return (u64)__double_as_longlong(a) + 1ull;
}

// The register forms compare the upper word of |x| first (for FP32 all of
// it): it orders finite nonzero values, so a wave's or the workgroups' fold is
// one 32-bit DPP chain.  When the largest word is zero, an infinity or a NaN,
// or more than one lane holds it (FP64), the full keys decide.
template <class T> struct PBits;
template <> struct PBits<double> {
  static constexpr unsigned special = 0x7FF00000u;  // infinities and NaNs from here on
  static __device__ __forceinline__ unsigned hi(double x) {
    return (unsigned)((u64)__double_as_longlong(x) >> 32) & 0x7FFFFFFFu;
  }
};
template <> struct PBits<float> {
  static constexpr unsigned special = 0x7F800000u;
  static __device__ __forceinline__ unsigned hi(float x) { return __float_as_uint(x) & 0x7FFFFFFFu; }
};

// max(v, v of the lane CTRL names); 0 where there is none (0 is the identity,
// so the move folds into the maximum)
template <int CTRL, int ROWMASK>
__device__ __forceinline__ unsigned dpp_max(unsigned v) {
  const unsigned o = (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWMASK, 0xf, ROWMASK == 0xf);
  return o > v ? o : v;
}
// Max over the lanes l < N with l % STRIDE == STRIDE - 1 (uniform; powers of
// two, STRIDE <= 16): row_shr carries it to a 16-lane row's last lane (to lane
// N - 1 when N < 16), row_bcast 15 and 31 to lane 31 or 63.
template <int STRIDE, int N>
__device__ __forceinline__ unsigned lanes_max(unsigned v) {
  if (STRIDE <= 1 && N > 1) v = dpp_max<0x111, 0xf>(v);
  if (STRIDE <= 2 && N > 2) v = dpp_max<0x112, 0xf>(v);
  if (STRIDE <= 4 && N > 4) v = dpp_max<0x114, 0xf>(v);
  if (STRIDE <= 8 && N > 8) v = dpp_max<0x118, 0xf>(v);
  if (N > 16) v = dpp_max<0x142, 0xa>(v);
  if (N > 32) v = dpp_max<0x143, 0xc>(v);
  return (unsigned)__builtin_amdgcn_readlane((int)v, N - 1);
}
template <int STRIDE, int N>
constexpr u64 lanes_mask() {
  u64 lm = 0;
  for (int l = STRIDE - 1; l < N; l += STRIDE) lm |= 1ull << l;
  return lm;
}
// The lane whose candidate the pivot search takes (uniform): x among the
// lanes of <STRIDE, N> with cand set, the lowest lane where keys are equal;
// is_k marks row k.  No lane has cand set: *none.  hi: PBits<T>::hi(x) where
// cand, else 0; m: its maximum (lanes_max).
template <class T, int STRIDE, int N>
__device__ __forceinline__ int pick_lane(T x, bool cand, bool is_k, unsigned hi, unsigned m, bool* none) {
  constexpr u64 LM = lanes_mask<STRIDE, N>();
  u64 b = __ballot(hi == m) & LM;
  *none = false;
  // several lanes (zeros always are), an infinity or a NaN: the full keys
  if (__builtin_expect(__builtin_popcountll(m < PBits<T>::special ? b : 0ull) != 1, 0)) {
    const u64 key = cand ? pivot_key(x, is_k) : 0ull;
    const unsigned kh = (unsigned)(key >> 32);
    const unsigned mh = lanes_max<STRIDE, N>(kh);
    const unsigned kl = kh == mh ? (unsigned)key : 0u;
    const unsigned ml = lanes_max<STRIDE, N>(kl);
    b = __ballot(kh == mh && kl == ml) & LM;
    *none = (mh | ml) == 0u;
  }
  return (int)__builtin_ctzll(b);
}
template <class T, int STRIDE, int N>
__device__ __forceinline__ int pick_lane(T x, bool cand, bool is_k, bool* none) {
  const unsigned hi = cand ? PBits<T>::hi(x) : 0u;
  return pick_lane<T, STRIDE, N>(x, cand, is_k, hi, lanes_max<STRIDE, N>(hi), none);
}
// lanes_max<1, 64>(hi) and, between its steps (each waits for the one
// before), every lane's 1 / x.
__device__ __forceinline__ unsigned wave_max_recip(unsigned hi, float x, float* rp) {
  *rp = 1.0f / x;
  return lanes_max<1, 64>(hi);
}
__device__ __forceinline__ unsigned wave_max_recip(unsigned hi, double x, double* rp) {
  // the correctly rounded division's own sequence (scaled operands, reciprocal
  // refined twice, quotient, its residual, fix-up), in the DPP wait states
#define LA_STEP __builtin_amdgcn_sched_barrier(0)
  bool f0, f1;
  unsigned v = hi;
  const double d = __builtin_amdgcn_div_scale(1.0, x, false, &f0);
  LA_STEP;
  v = dpp_max<0x111, 0xf>(v);
  LA_STEP;
  const double r0 = __builtin_amdgcn_rcp(d);
  const double n = __builtin_amdgcn_div_scale(1.0, x, true, &f1);
  LA_STEP;
  v = dpp_max<0x112, 0xf>(v);
  LA_STEP;
  const double e0 = __builtin_fma(-d, r0, 1.0);
  LA_STEP;
  v = dpp_max<0x114, 0xf>(v);
  LA_STEP;
  const double r1 = __builtin_fma(r0, e0, r0);
  LA_STEP;
  v = dpp_max<0x118, 0xf>(v);
  LA_STEP;
  const double e1 = __builtin_fma(-d, r1, 1.0);
  LA_STEP;
  v = dpp_max<0x142, 0xa>(v);
  LA_STEP;
  const double r2 = __builtin_fma(r1, e1, r1);
  LA_STEP;
  v = dpp_max<0x143, 0xc>(v);
  LA_STEP;
  const double q = n * r2;
  LA_STEP;
  const unsigned m = (unsigned)__builtin_amdgcn_readlane((int)v, 63);
  LA_STEP;
  const double e2 = __builtin_fma(-d, q, n);
  double r = __builtin_amdgcn_div_fixup(__builtin_amdgcn_div_fmas(e2, r2, q, f1), x, 1.0);
  asm volatile("" : "+v"(r));  // here, not in the branch of the one lane that stores it
  *rp = r;
#undef LA_STEP
  return m;
}
__device__ __forceinline__ double lane_value(double x, int lane) {
  const u64 b = (u64)__double_as_longlong(x);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, lane);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
  return __longlong_as_double((long long)(((u64)hi << 32) | lo));
}
__device__ __forceinline__ float lane_value(float x, int lane) {
  return __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(x), lane));
}

// v[c] = fma(u of lane 16*(lane/16) + c, nl, v[c]) for c in [0, 8): the
// multiply-add takes its uniform operand straight from a lane (DPP
// row_newbcast), so a broadcast value costs no LDS read and no move of its
// own.  Every lane of the wave must be active.  The s_nop covers the two wait
// states a DPP source needs after a vector write of it.
__device__ __forceinline__ void fmac_lanes(double* v, double u, double nl) {
  asm("s_nop 1\n"
      "v_fmac_f64_dpp %0, %8, %9 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %8, %9 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %8, %9 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %3, %8, %9 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %4, %8, %9 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %5, %8, %9 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %6, %8, %9 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %7, %8, %9 row_newbcast:7 row_mask:0xf bank_mask:0xf"
      : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7])
      : "v"(u), "v"(nl));
}
__device__ __forceinline__ void fmac_lanes(float* v, float u, float nl) {
  asm("s_nop 1\n"
      "v_fmac_f32_dpp %0, %8, %9 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %8, %9 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %8, %9 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %3, %8, %9 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %4, %8, %9 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %5, %8, %9 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %6, %8, %9 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %7, %8, %9 row_newbcast:7 row_mask:0xf bank_mask:0xf"
      : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7])
      : "v"(u), "v"(nl));
}

// LDS written by this wave's lanes, read next by others of the same wave: LDS
// operations of one wave complete in order, so only the compiler is held.
__device__ __forceinline__ void wave_sync() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

// |piv| >= sfmin (or not a number) of a uniform pivot, on the scalar unit.
template <class T>
__device__ __forceinline__ bool recip_ok(T piv) {
  unsigned hb = PBits<T>::hi(piv);
  asm("" : "+s"(hb));
  return hb >= (sizeof(T) == 8 ? 0x00100000u : 0x00800000u);
}

// ---- the exchange words of the multi-workgroup leaf --------------------------
// Every 64-bit word carries 32 bits of payload and the 32-bit flag
// tagbase + k + 1 of the column it belongs to (a double travels as two
// words), so a reader validates each word it loads and needs no fence or tag
// from the writer -- 64-bit stores are single-copy atomic.  A workgroup
// cannot publish column k+1 before every workgroup has read column k, so two
// buffers (column parity) suffice for the candidates; it cannot publish the
// rows of a group before every workgroup has read those of the group before
// (each reads them before it publishes its next candidate), so one buffer
// suffices for the rows.  The exchange buffer must be zero before the first
// launch of a factorization (flags only grow after that: tagbase advances by
// 64 per launch).
constexpr int LG = 8;                        // columns of a group
constexpr int MSGS = 32;                     // words of a candidate's slot (padded)
constexpr size_t MSG_PAR = (size_t)(GMAX + 1) * MSGS;  // candidates of one column + row k
constexpr int ROWS_SLOTS = 2 * LG;           // rows an 8-column group's interchanges touch
constexpr int NOSLOT = 31;                   // a row no interchange of the group has touched
constexpr size_t LL_WORDS = 2 * MSG_PAR + (size_t)ROWS_SLOTS * 2 * WMAX;

__device__ __forceinline__ u64 ll_word(unsigned payload, unsigned flag) {
  return ((u64)flag << 32) | (u64)payload;
}

// ---- register-resident leaf ------------------------------------------------------
// Thread t of workgroup b holds row b*NTH + t of the leaf, W values.  The
// columns run in groups of 8: inside a group only the group's 8 columns are
// exchanged and updated (slots 0..7 of v); the other columns -- interchanged,
// solved against the group's 8x8 unit triangle and updated -- follow once per
// group, with the operations of the column-by-column form in the same order
// on each element.  Per column:
//   A   a wave's best candidate (its 8 group values, their pivot's reciprocal
//       and the row) -> LDS, and row k's 8 group values; the reciprocal is
//       taken by every lane of its own value beside the search's DPP chain,
//       which leaves the vector unit idle most of the time;
//   B   one barrier; with several workgroups the winning wave publishes the
//       workgroup's candidate and the wave holding row k that row, then every
//       thread polls its share of the G candidates' words into LDS, and a
//       second barrier;
//   C   every wave folds the candidates; the winner's values come out of the
//       fold's registers as scalars (readlane);
//   D   interchange, scaling, update of the group's remaining columns.
// Buffers alternate with the column parity, so no barrier ends a column.
// After each group:
//   E   the at most 16 rows that the group's interchanges touch go through
//       LDS (with several workgroups through the exchange buffer as well);
//       barrier; one wave solves the group's rows of U; barrier; every row
//       below takes the rank-8 update of the columns still to come.
// A touched row has a slot: 0..7 for the group's own rows, 8 + i for the row
// first touched as step i's pivot; each thread follows its row's slot and the
// slot its content came from, and a candidate carries the latter.
// It also follows the row that content was in at the leaf's start (corg),
// which tells the other columns' interchanges their sources (swap_trsm.hip).
// What bounds it: the chain A..D (1500-2100 cycles a column in one workgroup,
// 4200 with 32, 945 of them the exchange's round trip), then E (4000-7000 a
// group).  With several workgroups only the next group's columns are updated
// in E; each later step updates one further chunk while its exchange is in
// flight.  Measured, 64 columns of FP64 (before: the whole row exchanged and
// updated in every column, agent-scope stores): 512 rows 214 -> 95 us, 128
// rows 200 -> 69, 16384 rows on XCD 0 beside the update 276 -> 149; 32 columns
// of 1024 rows 120 -> 64.
template <class T, int W, int NTH, bool MULTI, bool XCD0>
__global__ __launch_bounds__(NTH) void getf2_leaf_kernel(T* __restrict__ Tm, long ldt, int j0, int w, int m,
                                                        int* __restrict__ ipiv, int* __restrict__ info,
                                                        unsigned tagbase, u64* __restrict__ xbuf,
                                                        int* __restrict__ err, int Gp, unsigned* __restrict__ ctr,
                                                        RowOrg org) {
  constexpr int NW = NTH / 64;
  constexpr int VW = (int)sizeof(T) / 4;      // words of a value
  constexpr int MW = (LG + 1) * VW + 2;       // words of a candidate
  constexpr int KW = LG * VW + 2;             // words of row k
  constexpr int NS = MULTI ? GMAX : NW;       // candidates a column folds (at most)
  constexpr int SR = W - LG + 2;              // row stride of s_sw / s_u
  // one workgroup's fold: LPS lanes a candidate, VPL values a lane, the
  // column searched in the candidate's last lane
  constexpr int LPS = NW >= 8 ? 8 : 16, VPL = LPS >= LG ? 1 : LG / LPS, LV = LG / VPL;
  static_assert(NW * LPS <= 64, "one lane set per wave");
  struct Msg {
    T v[LG];
    T rp;      // 1 / v[step]
    int meta;  // row | content's slot << 16 (NOSLOT: none), or -1: no candidate
    int org;   // the leaf's row its content was in at the start
  };
  struct RowK {
    T v[LG];
    int osl, org;
  };
  __shared__ __align__(16) Msg s_wmsg[2][NW];  // the waves' candidates
  __shared__ __align__(16) Msg s_msg[MULTI ? 2 : 1][MULTI ? NS : 1];
  __shared__ __align__(16) RowK s_rowk[2];
  __shared__ __align__(16) T s_l[LG][LG];      // the group's rows of L (and U) as they were pivoted
  __shared__ __align__(16) T s_sw[ROWS_SLOTS][SR];
  __shared__ __align__(16) T s_u[LG][SR];
  __shared__ int s_fail;
  __shared__ int s_rank;
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
  const int nch = (w + LG - 1) / LG;           // 8-column chunks of the leaf
  const int wrow0 = b * NTH + wave * 64;       // the wave's first row
  // the only wave with rows that leave the active range: its updates are
  // masked row by row, the other waves' are not (rows past h hold zeros that
  // are neither searched nor stored)
  const bool top_wave = wrow0 < W;
  const int lr = b * NTH + tid;
  if (MULTI && tid == 0) s_fail = 0;

  // The wave's 64 rows in and out through LDS, CP columns at a time: an access
  // of the matrix touches whole runs of CP values of 64 / CP rows (a row a lane
  // would touch 64 lines an instruction).
  constexpr int CP = 16;
  constexpr int RP = 64 / CP;  // rows of one access
  __shared__ T s_stage[NW][64][CP + 1];
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
  bool failed = false;

  int my_piv = 0;     // lane k: step k's pivot row
  int corg = lr;      // the leaf's row this row's content was in at the start
  int zero_at = -1;   // the first step with a zero pivot
  const bool valid = lr < h;
  // An exchange word to the other workgroups.  All of them on one XCD share
  // its L2: there a plain store (it reaches the L2; the readers' agent-scope
  // loads pass their own caches and hit it) does, and a round among 32
  // workgroups takes 945 cycles, beside HBM traffic of the other XCDs or not;
  // with agent-scope stores, which write through to memory, 2290 alone and
  // 3550 beside such traffic (gfx950, one word a workgroup).
  auto put = [&](u64* d, u64 x) {
    if (XCD0) __hip_atomic_store(d, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else st_dev(d, x);
  };
  // One more poll is due; false when the wait gives up.
  auto spin_check = [&](unsigned& spins) -> bool {
    __builtin_amdgcn_s_sleep(1);
    ++spins;
    if ((spins & 255u) == 1u && ld_dev(err) != 0) return false;
    if (spins > (1u << 20)) {
      st_dev(err, 1);
      return false;
    }
    return true;
  };

  // One chunk's rank-8 update with the rows of U in s_u: columns LG*cu.. of
  // s_u, values vq, multipliers -nl; rows from r0 on keep it (the waves below
  // the top one have no others)
  auto load_u = [&](T (&u)[LG], int cu) {
#pragma unroll
    for (int i = 0; i < LG; ++i) u[i] = s_u[i][LG * cu + (lane & (LG - 1))];
  };
  // In FP32 the eight products are summed on their own and added once: one
  // rounding at the element's size a group instead of eight.
  auto apply_u = [&](const T (&u)[LG], const T (&nl)[LG], T* vq, int r0) {
    constexpr bool SUM = sizeof(T) == 4;
    if (SUM || top_wave) {
      T t[LG];
#pragma unroll
      for (int c = 0; c < LG; ++c) t[c] = SUM ? T(0) : vq[c];
#pragma unroll
      for (int i = 0; i < LG; ++i) fmac_lanes(t, u[i], nl[i]);
#pragma unroll
      for (int c = 0; c < LG; ++c) {
        const T x = SUM ? vq[c] + t[c] : t[c];
        vq[c] = !top_wave || lr >= r0 ? x : vq[c];
      }
    } else {
#pragma unroll
      for (int i = 0; i < LG; ++i) fmac_lanes(vq, u[i], nl[i]);
    }
  };
  for (int g = 0; LG * g < kmax; ++g) {
    const int k0 = LG * g;
    const int rest = nch - 1 - g;        // chunks still to come
    int ts[LG];            // the slot whose content row k0 + i takes (uniform)
    unsigned touched = 0;  // slots in use (uniform)
    const bool in_group = lr >= k0 && lr < k0 + LG;
    int myslot = in_group ? lr - k0 : NOSLOT;  // this row's slot, and its content's
    int osl = myslot;
#pragma unroll
    for (int kk = 0; kk < LG; ++kk) {
      const int k = k0 + kk;
      ts[kk] = kk;
      if (k < kmax) {
        const int par = k & 1;
        const unsigned flag = tagbase + (unsigned)k + 1u;
        // ---- A
        {
          T rp;
          bool none;
          const bool cand = valid && (!top_wave || lr >= k);
          const unsigned hi = cand ? PBits<T>::hi(v[kk]) : 0u;
          if (top_wave && lr == k) {
#pragma unroll
            for (int c = 0; c < LG; ++c) s_rowk[par].v[c] = v[c];
            s_rowk[par].osl = osl;
            s_rowk[par].org = corg;
          }
          const unsigned wm = wave_max_recip(hi, v[kk], &rp);
          const int wl = pick_lane<T, 1, 64>(v[kk], cand, lr == k, hi, wm, &none);
          if (lane == wl) {
            Msg& ms = s_wmsg[par][wave];
#pragma unroll
            for (int c = 0; c < LG; ++c) ms.v[c] = v[c];
            ms.rp = rp;
            ms.meta = none ? -1 : lr | (osl << 16);
            ms.org = corg;
          }
        }
        // the wave's own candidate as words, should it be the workgroup's
        unsigned mine = 0;
        if (MULTI) {
          wave_sync();
          if (lane < MW) mine = reinterpret_cast<const unsigned*>(&s_wmsg[par][wave])[lane];
        }
        __syncthreads();
        // ---- B, C
        int meta, porg;
        T uc[LG], rp;  // the pivot row's group values and its pivot's reciprocal (uniform)
        if (MULTI) {
          {
            const Msg& ms = s_wmsg[par][lane & (NW - 1)];
            const int cm = ms.meta;
            bool none;
            const int bw = pick_lane<T, 1, NW>(ms.v[kk], cm >= 0, (cm & 0xffff) == k, &none);
            u64* buf = xbuf + (size_t)par * MSG_PAR;
            if (wave == bw && lane < MW) put(buf + (size_t)b * MSGS + lane, ll_word(mine, flag));
            // row k, which only the owner of the pivot row needs, after the candidate
            if (top_wave && lane < KW) {
              const unsigned x = reinterpret_cast<const unsigned*>(&s_rowk[par])[lane];
              put(buf + (size_t)GMAX * MSGS + lane, ll_word(x, flag));
            }
            // the previous group's update of one chunk, while the exchange is
            // in flight: chunk kk + 1, with that group's multipliers (the last
            // slots) and rows of U (s_u is written next after this group)
            if (kk + 1 < W / LG && g > 0 && kk + 1 <= rest) {
              T nl[LG], uu[LG];
              load_u(uu, kk + 1);
#pragma unroll
              for (int i = 0; i < LG; ++i) nl[i] = -v[W - LG + i];
              apply_u(uu, nl, v + LG * (kk + 1), k0);
            }
            // every thread polls its share: 32 lanes a slot, slot G = row k
            constexpr int SP = NTH / 32;                  // slots a pass
            constexpr int NP = (GMAX + 1 + SP - 1) / SP;  // passes (at most)
            const int wd = tid & 31;
            u64 x[NP];
            bool need[NP];
#pragma unroll
            for (int q = 0; q < NP; ++q) {
              const int sl = q * SP + (tid >> 5);
              need[q] = !failed && (sl < G ? wd < MW : (sl == G && wd < KW));
              x[q] = 0;
            }
            unsigned spins = 0;
            for (;;) {
              bool miss = false;
#pragma unroll
              for (int q = 0; q < NP; ++q) {
                if (q * SP <= G) {
                  const int sl = q * SP + (tid >> 5);
                  x[q] = ld_dev(buf + (size_t)(sl < G ? sl : GMAX) * MSGS + wd);
                }
              }
#pragma unroll
              for (int q = 0; q < NP; ++q) {
                if (q * SP <= G && need[q]) {
                  if ((unsigned)(x[q] >> 32) == flag) {
                    const int sl = q * SP + (tid >> 5);
                    unsigned* dst = sl < G ? reinterpret_cast<unsigned*>(&s_msg[par][sl])
                                           : reinterpret_cast<unsigned*>(&s_rowk[par]);
                    dst[wd] = (unsigned)x[q];
                    need[q] = false;
                  } else {
                    miss = true;
                  }
                }
              }
              if (!__any(miss)) break;
              if (!spin_check(spins)) {
                s_fail = 1;
                break;
              }
            }
          }
          __syncthreads();
          failed = s_fail != 0;
          const bool in = lane < G;
          const Msg& ms = s_msg[par][in ? lane : 0];
          const int cm = ms.meta, co = ms.org;
          const T crp = ms.rp;
          bool none;
          const int ws = pick_lane<T, 1, 64>(ms.v[kk], in && cm >= 0, (cm & 0xffff) == k, &none);
          const T x = s_msg[par][ws].v[lane & (LG - 1)];
          meta = __builtin_amdgcn_readlane(cm, ws);
          porg = __builtin_amdgcn_readlane(co, ws);
          rp = lane_value(crp, ws);
#pragma unroll
          for (int c = 0; c < LG; ++c) uc[c] = lane_value(x, c);
          if (wave == NW - 1 && lane < LG) s_l[kk][lane] = x;
        } else {
          const Msg& ms = s_wmsg[par][(lane / LPS) & (NW - 1)];
          // lane j of a candidate holds value (j + kk + 1) % LV of the LV
          // values around kk, and value j of the others
          const int H = kk / LV;
          T x[VPL];
#pragma unroll
          for (int z = 0; z < VPL; ++z) x[z] = ms.v[z * LV + ((lane + (z == H ? kk + 1 : 0)) & (LV - 1))];
          const int cm = ms.meta, co = ms.org;
          const T crp = ms.rp;
          bool none;
          const int wl = pick_lane<T, LPS, NW * LPS>(x[H], cm >= 0, (cm & 0xffff) == k, &none);
          meta = __builtin_amdgcn_readlane(cm, wl);
          porg = __builtin_amdgcn_readlane(co, wl);
          rp = lane_value(crp, wl);
          const int w0 = wl & ~(LPS - 1);
#pragma unroll
          for (int c = 0; c < LG; ++c)
            uc[c] = lane_value(x[c / LV], w0 + ((c - (c / LV == H ? kk + 1 : 0)) & (LV - 1)));
          if (wave == NW - 1 && (lane & ~(LPS - 1)) == w0) {
#pragma unroll
            for (int z = 0; z < VPL; ++z) s_l[kk][z * LV + ((lane + (z == H ? kk + 1 : 0)) & (LV - 1))] = x[z];
          }
        }
        // ---- D
        int p = meta & 0xffff;
        if (MULTI && (p < k || p >= h)) p = k;  // only after a wait gave up
        const T piv = uc[kk];
        const int csl = (meta >> 16) & NOSLOT;  // the slot the pivot row's content came from
        ts[kk] = csl == NOSLOT ? LG + kk : csl;
        if (MULTI) touched |= csl == NOSLOT ? 1u << (LG + kk) : 0u;
        my_piv = lane == k ? p : my_piv;
        if (p != k) {
          if (top_wave && lr == k) {
#pragma unroll
            for (int c = 0; c < LG; ++c) v[c] = uc[c];
            osl = ts[kk];
            corg = porg;
          }
          if (p >= wrow0 && p < wrow0 + 64) {
            if (lr == p) {
#pragma unroll
              for (int c = 0; c < LG; ++c) v[c] = s_rowk[par].v[c];
              osl = s_rowk[par].osl;
              corg = s_rowk[par].org;
              if (myslot == NOSLOT) myslot = LG + kk;
            }
          }
        }
        T l = v[kk];
        if (__builtin_expect(recip_ok(piv), 1)) {
          l = rp * l;
        } else if (piv != T(0)) {
          l = l / piv;
        } else if (zero_at < 0) {
          zero_at = k;
        }
        if (!top_wave || lr > k) {
          v[kk] = l;
#pragma unroll
          for (int c = kk + 1; c < LG; ++c) v[c] = v[c] - l * uc[c];
        }
      }
    }
    // ---- E: the group's interchanges on the other columns, its rows of U,
    // and the update of the columns still to come
    const int kg = min(LG, kmax - k0);   // columns of this group
    if (W > LG && nch > 1) {
      if (myslot != NOSLOT) {
        T* d = s_sw[myslot];
#pragma unroll
        for (int c = LG; c < W; ++c) d[c - LG] = v[c];
      }
      if (MULTI) {
        const unsigned flag = tagbase + (unsigned)(k0 + kg);
        u64* rows = xbuf + 2 * MSG_PAR;
        constexpr int RW = (W - LG) * VW;  // words of a row
        constexpr int RS = W * VW;         // words of a row's slot (the ones past RW hold nothing)
        // the touched rows this wave holds: the group's own at once, then the
        // others (at most one per step over all workgroups).  The indexes are
        // made new in every group, so that what follows from them is computed
        // here and not kept in registers over the column steps.
        int te = tid, le = lane;
        asm volatile("" : "+v"(te), "+v"(le));
        wave_sync();
        if (top_wave) {
          constexpr int NR = LG * RS / 64;
          unsigned x[NR];
#pragma unroll
          for (int q = 0; q < NR; ++q) {
            // (a word past RW reads on into the next slot: in bounds, unused)
            const int e = le + 64 * q;
            x[q] = reinterpret_cast<const unsigned*>(s_sw[e / RS])[e % RS];
          }
#pragma unroll
          for (int q = 0; q < NR; ++q) put(rows + le + 64 * q, ll_word(x[q], flag));
        }
        for (u64 mb = __ballot(myslot != NOSLOT && myslot >= LG); mb != 0ull; mb &= mb - 1) {
          const int sl = __builtin_amdgcn_readlane(myslot, (int)__builtin_ctzll(mb));
          const unsigned* sw = reinterpret_cast<const unsigned*>(s_sw[sl]);
          for (int x = le; x < RW; x += 64) put(rows + sl * RS + x, ll_word(sw[x], flag));
        }
        // every touched row's words, into this workgroup's LDS
        touched |= (1u << LG) - 1u;
        constexpr int PR = ROWS_SLOTS * RS / NTH;
        static_assert(PR * NTH == ROWS_SLOTS * RS && RW <= RS, "the threads' shares");
        u64 x[PR];
        bool need[PR];
#pragma unroll
        for (int q = 0; q < PR; ++q) {
          const int e = te + q * NTH;
          need[q] = e % RS < RW && (touched >> (e / RS) & 1u) != 0u && !failed;
          x[q] = 0;
        }
        unsigned spins = 0;
        for (;;) {
          bool miss = false;
#pragma unroll
          for (int q = 0; q < PR; ++q) x[q] = ld_dev(rows + te + q * NTH);
#pragma unroll
          for (int q = 0; q < PR; ++q) {
            const int e = te + q * NTH;
            if (need[q]) {
              if ((unsigned)(x[q] >> 32) == flag) {
                reinterpret_cast<unsigned*>(s_sw[e / RS])[e % RS] = (unsigned)x[q];
                need[q] = false;
              } else {
                miss = true;
              }
            }
          }
          if (!__any(miss)) break;
          if (!spin_check(spins)) {
            s_fail = 1;
            break;
          }
        }
      }
      __syncthreads();
      if (MULTI) failed = s_fail != 0;
      auto take = [&]() {
        if (osl != myslot) {
          const T* d = s_sw[osl];
#pragma unroll
          for (int c = LG; c < W; ++c) v[c] = d[c - LG];
        }
      };
      // (the solving wave takes its rows behind the barrier)
      if (wave != NW - 1 || rest == 0) take();
      if (rest > 0) {
        // U12: one column a lane, forward substitution with the group's
        // triangle (a zero multiplies like any other value, as in the update)
        if (wave == NW - 1 && lane < LG * rest) {
          T x[LG];
#pragma unroll
          for (int i = 0; i < LG; ++i) x[i] = s_sw[ts[i]][lane];
#pragma unroll
          for (int z = 0; z < LG - 1; ++z) {
#pragma unroll
            for (int i = z + 1; i < LG; ++i) x[i] = x[i] - s_l[i][z] * x[z];
          }
#pragma unroll
          for (int i = 0; i < LG; ++i) s_u[i][lane] = x[i];
        }
        __syncthreads();
        if (wave == NW - 1) take();
        T nl[LG], ua[LG], ub[LG];  // a chunk's values of U are read while the one before is applied
#pragma unroll
        for (int i = 0; i < LG; ++i) nl[i] = -v[i];
        load_u(ua, 0);
        if (MULTI) {
          // the next group's columns now; the others beside its exchanges
          apply_u(ua, nl, v + LG, k0 + LG);
        } else {
#pragma unroll
          for (int q = 1; q < W / LG; q += 2) {
            if (q <= rest) {
              if (q + 1 <= rest) load_u(ub, q);
              apply_u(ua, nl, v + LG * q, k0 + LG);
            }
            if (q + 1 < W / LG && q + 1 <= rest) {
              if (q + 2 <= rest) load_u(ua, q + 1);
              apply_u(ub, nl, v + LG * (q + 1), k0 + LG);
            }
          }
        }
        if (top_wave && in_group) {
          const T* d = s_u[lr - k0];
#pragma unroll
          for (int q = 1; q < W / LG; ++q)
            if (q <= rest) {
#pragma unroll
              for (int c = 0; c < LG; ++c) v[LG * q + c] = d[LG * (q - 1) + c];
            }
        }
      }
    }
    // the next group's columns to slots 0..7
    if (W > LG) {
      T t[LG];
#pragma unroll
      for (int c = 0; c < LG; ++c) t[c] = v[c];
#pragma unroll
      for (int c = 0; c < W - LG; ++c) v[c] = v[c + LG];
#pragma unroll
      for (int c = 0; c < LG; ++c) v[W - LG + c] = t[c];
    }
  }
  if (W > LG) {
    for (int g = (kmax + LG - 1) / LG; g < W / LG; ++g) {
      T t[LG];
#pragma unroll
      for (int c = 0; c < LG; ++c) t[c] = v[c];
#pragma unroll
      for (int c = 0; c < W - LG; ++c) v[c] = v[c + LG];
#pragma unroll
      for (int c = 0; c < LG; ++c) v[W - LG + c] = t[c];
    }
  }
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

// The record of the tall form's interchanges (RowOrg), from IPIV: one
// workgroup, thread 0 walking the at most 64 interchanges.
__global__ __launch_bounds__(256) void tall_org_kernel(int j0, int kmax, int m, const int* __restrict__ ipiv,
                                                       RowOrg org) {
  for (int r = j0 + (int)threadIdx.x; r < m; r += 256) org.leaf[r] = r;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = j0; k < j0 + kmax; ++k) {
      const int p = ipiv[k] - 1;
      if (p > k && p < m) {
        const int t = org.leaf[k];
        org.leaf[k] = org.leaf[p];
        org.leaf[p] = t;
      }
    }
  }
  __syncthreads();
  for (int r = j0 + (int)threadIdx.x; r < m; r += 256) {
    const int o = org.leaf[r];
    const int po = org.pin ? org.pin[o] : o;
    org.pout[r] = po;
    if (org.last || r < j0 + kmax) org.fin[r] = po;
  }
}

}  // namespace

// Launch configurations: one workgroup with a thread a row up to 512 rows
// (fewer threads for the shorter leaves: fewer waves to fold and to wait for).
// Beyond that G workgroups of 512 threads; past GMAX workgroups the tall form.
static size_t tall_offset() { return (sizeof(u64) * LL_WORDS + 255) / 256 * 256; }
// the XCD-0 panel's rank and arrival counters (zeroed with the exchange
// buffer at the start of a factorization; each launch resets its own)
static size_t rank_offset() { return tall_offset() + (sizeof(TallBuf) + 255) / 256 * 256; }
size_t panel_xchg_bytes(int) { return rank_offset() + 256; }

// Workgroups the panel kernel uses at height h (0 = a single workgroup).
int panel_groups(int h) { return h <= 512 ? 0 : (h + 511) / 512; }

// mode: PANEL_PLAIN (G workgroups), PANEL_XCD0 (8*G blocks, those of the
// first XCDs take part), PANEL_TALL (the form without waits).
template <class T>
static int launch_panel_t(T* Tm, long ldt, int j0, int w, int m, int* ipiv, int* info, unsigned tagbase,
                          double* xchg, int* err, int mode, const RowOrg& org, hipStream_t s) {
  const int h = m - j0;
  if (h <= 0 || w <= 0) return 0;
  if (w > WMAX) return LA_ERR_LIMIT;
  u64* xb = reinterpret_cast<u64*>(xchg);
#define LA_LEAF(W, NTH, MULTI, XCD0, blocks, g, ctr) \
  getf2_leaf_kernel<T, W, NTH, MULTI, XCD0><<<blocks, NTH, 0, s>>>(Tm, ldt, j0, w, m, ipiv, info, tagbase, xb, err, g, ctr, \
                                                              org)
  if (h <= 512) {
    if (h <= 128) LA_LEAF(64, 128, false, false, 1, 1, nullptr);
    else if (h <= 256) LA_LEAF(64, 256, false, false, 1, 1, nullptr);
    else LA_LEAF(64, 512, false, false, 1, 1, nullptr);
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
    tall_org_kernel<<<1, 256, 0, s>>>(j0, kmax, m, ipiv, org);
    return 0;
  }
  if (mode == PANEL_XCD0)
    LA_LEAF(64, 512, true, true, (8 / (int)panel_xcds(G)) * G, G,
            reinterpret_cast<unsigned*>(reinterpret_cast<char*>(xchg) + rank_offset()));
  else
    LA_LEAF(64, 512, true, false, G, G, nullptr);
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
