// leaf.h -- the column loop of a register-resident LU leaf: one thread a row,
// one workgroup (panel.hip's short leaves, batched_leaf.hip's matrices) or
// several that agree through device memory (panel.hip's tall leaves).
#pragma once
#include "la_common.h"

namespace la {
namespace {

typedef unsigned long long u64;

constexpr int GMAX = 64;            // workgroups of a register-resident leaf
constexpr int WMAX = 64;            // widest leaf

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
  // 1 / x as the CDNA instruction set documents its division instructions:
  // operands scaled (v_div_scale), the estimate v_rcp refined by two Newton steps,
  // the quotient corrected by its residual (Markstein, IBM J. R&D 34, 1990), the
  // scaling undone and special operands fixed up (v_div_fmas, v_div_fixup); laid
  // out in the DPP wait states
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

// acc += (x of lane 16*(lane/16) + KS) * l; every lane active.  The s_nop
// covers the wait states a DPP source needs after a vector write of it.
template <int KS>
__device__ __forceinline__ void fmac_from(double& acc, double x, double l) {
  asm("s_nop 1\n\tv_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
      : "+v"(acc)
      : "v"(x), "v"(l), "n"(KS));
}
template <int KS>
__device__ __forceinline__ void fmac_from(float& acc, float x, float l) {
  asm("s_nop 1\n\tv_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
      : "+v"(acc)
      : "v"(x), "v"(l), "n"(KS));
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
// launch of a factorization; after that flags only grow (tagbase advances by 64
// per launch), so a word of an earlier leaf never passes for a current one.
constexpr int LG = 8;                        // columns of a group
constexpr int MSGS = 32;                     // words of a candidate's slot (padded)
constexpr size_t MSG_PAR = 2880;             // candidates of one column + row k
constexpr int ROWS_SLOTS = 2 * LG;           // rows an 8-column group's interchanges touch
constexpr int NOSLOT = 31;                   // a row no interchange of the group has touched
constexpr size_t LL_WORDS = 2 * MSG_PAR + (size_t)ROWS_SLOTS * 2 * WMAX;

__device__ __forceinline__ u64 ll_word(unsigned payload, unsigned flag) {
  return ((u64)flag << 32) | (u64)payload;
}

// Up to 128 waves (16 workgroups of 8) exchange without a workgroup's own fold in
// between: each publishes its candidate's key -- the value, with the row's lane
// and slot beside a 20-bit flag in the upper word -- and then its values; every
// wave polls all the keys, one (DIRECT = 1) or two candidates a lane, folds them
// and reads the winner's values.  That leaves out the fold between two barriers
// (about 1000 of 5450 cycles a column) and takes the reciprocal out of the chain;
// a round of loads is what the polls take more as the waves grow (DGETRF at n =
// 1024 / 4096 / 8192: 2.30 / 10.86 / 24.04 -> 2.18 / 10.04 / 23.04 ms, SGETRF 2.03 /
// 9.58 / 20.52 -> 1.88 / 8.46 / 18.56).  A flag's top bit tells these upper words from
// the other ones (whose flags stay below 2^31); the 19 bits of the flag beside it
// repeat after 8192 leaves, which no factorization has that uses them (up to 8192
// rows; even leaves of one column are no more), and between factorizations the
// buffer is zeroed.
constexpr int DIRECT_CANDS = 128;
constexpr int DIRECT_ROWK = 2 * DIRECT_CANDS;     // row k's words
constexpr int DIRECT_VALUES = DIRECT_ROWK + 32;   // the candidates' values
constexpr unsigned DIRECT_NONE = 1u << 11;
static_assert(DIRECT_VALUES + DIRECT_CANDS * (2 * (LG + 1) + 2) <= MSG_PAR && (GMAX + 1) * MSGS <= MSG_PAR,
              "the candidates' buffer");
__device__ __forceinline__ unsigned direct_flag(unsigned flag, unsigned meta) {
  return (0x80000u | (flag & 0x7ffffu)) << 12 | meta;
}
// word w of a value (0: the lower half), a value of its words, and of the words
// that lanes l (and l + 1) hold (uniform)
__device__ __forceinline__ unsigned value_word(double x, int w) {
  return (unsigned)((u64)__double_as_longlong(x) >> (32 * w));
}
__device__ __forceinline__ unsigned value_word(float x, int) { return __float_as_uint(x); }
template <class T> __device__ __forceinline__ T value_of(unsigned top, unsigned low);
template <> __device__ __forceinline__ double value_of<double>(unsigned top, unsigned low) {
  return __longlong_as_double((long long)((u64)top << 32 | low));
}
template <> __device__ __forceinline__ float value_of<float>(unsigned top, unsigned) { return __uint_as_float(top); }
template <class T> __device__ __forceinline__ T word_value(int words, int l);
template <> __device__ __forceinline__ double word_value<double>(int words, int l) {
  return value_of<double>((unsigned)__builtin_amdgcn_readlane(words, l + 1),
                          (unsigned)__builtin_amdgcn_readlane(words, l));
}
template <> __device__ __forceinline__ float word_value<float>(int words, int l) {
  return __uint_as_float((unsigned)__builtin_amdgcn_readlane(words, l));
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
// (With up to 16 workgroups every wave publishes its candidate instead, and
// folds all of them: no barrier inside a group.)
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
// 3700 with up to 16, 4700 with 32, 945 of them the exchange's round trip), then
// E (4000-7000 a group).  With several workgroups only the next group's columns are updated
// in E; each later step updates one further chunk while its exchange is in
// flight.  Measured, 64 columns of FP64 (before: the whole row exchanged and
// updated in every column, agent-scope stores): 512 rows 214 -> 95 us, 128
// rows 200 -> 69, 16384 rows on XCD 0 beside the update 276 -> 149; 32 columns
// of 1024 rows 120 -> 59.
template <class T, int W, int NTH, bool MULTI>
struct LeafLds {
  static constexpr int NW = NTH / 64;
  static constexpr int VW = (int)sizeof(T) / 4;      // words of a value
  static constexpr int SR = W - LG + 2;              // row stride of s_sw / s_u
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
  alignas(16) Msg wmsg[2][NW];  // the waves' candidates
  alignas(16) Msg msg[MULTI ? 2 : 1][MULTI ? GMAX : 1];
  alignas(16) RowK rowk[2];
  alignas(16) T l[LG][LG];      // the group's rows of L (and U) as they were pivoted
  alignas(16) T sw[ROWS_SLOTS][SR];
  alignas(16) T u[LG][SR];
  int fail;                     // a wait gave up (zeroed before leaf_columns)
};

// Factors the leaf's w <= W columns held in v (thread t of workgroup b: row
// b*NTH + t of h; zeros past h and past w).  Returns the threads' shares of
// the record: my_piv (lane k: step k's pivot row), corg (the leaf's row whose
// content is in this thread's row now), zero_at (the first step with a zero
// pivot, or -1).  PREF: a chunk's values of U are read while the one before
// is applied.
template <class T, int W, int NTH, bool MULTI, bool XCD0, bool PREF = true, int DIRECT = 0>
__device__ __forceinline__ void leaf_columns(T (&v)[W], LeafLds<T, W, NTH, MULTI>& S, int h, int w, int b, int G,
                                             unsigned tagbase, u64* xbuf, int* err, int& my_piv, int& corg,
                                             int& zero_at) {
  typedef LeafLds<T, W, NTH, MULTI> L;
  constexpr int NW = NTH / 64;
  constexpr int VW = L::VW;
  constexpr int MW = (LG + 1) * VW + 2;       // words of a candidate
  constexpr int KW = LG * VW + 2;             // words of row k
  // one workgroup's fold: LPS lanes a candidate, VPL values a lane, the
  // column searched in the candidate's last lane
  constexpr int LPS = NW >= 16 ? 4 : NW >= 8 ? 8 : 16, VPL = LPS >= LG ? 1 : LG / LPS, LV = LG / VPL;
  static_assert(NW * LPS <= 64, "one lane set per wave");
  constexpr bool LEAN = NTH >= 1024 && sizeof(T) == 8;  // (128 registers, 64 of them values)
  int tid = threadIdx.x;
  if (!PREF) asm volatile("" : "+v"(tid));  // (nothing derived from it is kept outside the leaf)
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int kmax = min(h, w);
  const int nch = (w + LG - 1) / LG;           // 8-column chunks of the leaf
  const int wrow0 = b * NTH + wave * 64;       // the wave's first row
  // the only wave with rows that leave the active range: its updates are
  // masked row by row, the other waves' are not (rows past h hold zeros that
  // are neither searched nor stored)
  const bool top_wave = wrow0 < W;
  const int lr = b * NTH + tid;
  my_piv = 0;
  corg = lr;
  zero_at = -1;
  bool failed = false;

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
    if ((spins & 63u) == 0u && ld_dev(err) != 0) return false;  // (not in the first: a load more in every column)
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
    for (int i = 0; i < LG; ++i) u[i] = S.u[i][LG * cu + (lane & (LG - 1))];
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
            for (int c = 0; c < LG; ++c) S.rowk[par].v[c] = v[c];
            S.rowk[par].osl = osl;
            S.rowk[par].org = corg;
          }
          // (DIRECT: the reciprocal after the key, while that is on its way)
          const unsigned wm = DIRECT ? lanes_max<1, 64>(hi) : wave_max_recip(hi, v[kk], &rp);
          const int wl = pick_lane<T, 1, 64>(v[kk], cand, lr == k, hi, wm, &none);
          if (DIRECT && lane == wl) {  // its key at once
            u64* const kw = xbuf + (size_t)par * MSG_PAR + (b * NW + wave);
            put(kw, (u64)direct_flag(flag, (none ? DIRECT_NONE : 0u) | (unsigned)osl << 6 | (unsigned)lane) << 32 |
                        value_word(v[kk], VW - 1));
            if (VW > 1) put(kw + DIRECT_CANDS, ll_word(value_word(v[kk], 0), flag));
          }
          if (DIRECT) {
            rp = T(1) / v[kk];
            asm volatile("" : "+v"(rp));  // (on all lanes, not in the one lane's branch)
          }
          if (lane == wl) {
            typename L::Msg& ms = S.wmsg[par][wave];
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
          if (lane < MW) mine = reinterpret_cast<const unsigned*>(&S.wmsg[par][wave])[lane];
        }
        if (!DIRECT) __syncthreads();
        // ---- B, C
        int meta, porg;
        T uc[LG], rp;  // the pivot row's group values and its pivot's reciprocal (uniform)
        unsigned rk = 0;  // DIRECT: word `lane` of row k
        if (DIRECT) {
          const u64* const buf = xbuf + (size_t)par * MSG_PAR;
          u64* const out = xbuf + (size_t)par * MSG_PAR + DIRECT_VALUES;
          if (lane < MW) put(out + (b * NW + wave) * MW + lane, ll_word(mine, flag));
          if (top_wave && lane < KW) {
            const unsigned x = reinterpret_cast<const unsigned*>(&S.rowk[par])[lane];
            put(xbuf + (size_t)par * MSG_PAR + DIRECT_ROWK + lane, ll_word(x, flag));
          }
          if (kk + 1 < W / LG && g > 0 && kk + 1 <= rest) {  // (as below)
            T nl[LG], uu[LG];
            load_u(uu, kk + 1);
#pragma unroll
            for (int i = 0; i < LG; ++i) nl[i] = -v[W - LG + i];
            apply_u(uu, nl, v + LG * (kk + 1), k0);
          }
          // DIRECT candidates a lane: every wave folds them all
          constexpr int CL = DIRECT > 0 ? DIRECT : 1;
          const bool in = CL * lane < G * NW;  // (G * NW is a multiple of CL)
          const u64* const pk = buf + (in ? CL * lane : 0);
          const u64* const pr = buf + DIRECT_ROWK + (lane < KW ? lane : 0);
          u64 x0[CL], x1[CL], x2;
          unsigned spins = 0;
          for (;;) {
            bool miss = false;
#pragma unroll
            for (int q = 0; q < CL; ++q) {
              x0[q] = ld_dev(pk + q);
              x1[q] = VW > 1 ? ld_dev(pk + DIRECT_CANDS + q) : 0;
            }
            x2 = ld_dev(pr);
#pragma unroll
            for (int q = 0; q < CL; ++q)
              miss |= (unsigned)(x0[q] >> 44) != direct_flag(flag, 0) >> 12 || (VW > 1 && (unsigned)(x1[q] >> 32) != flag);
            miss |= (unsigned)(x2 >> 32) != flag;
            if (failed || !__any(miss)) break;
            if (!spin_check(spins)) {
              failed = true;
              S.fail = 1;
              break;
            }
          }
          rk = (unsigned)x2;
          T cv = value_of<T>((unsigned)x0[0], (unsigned)x1[0]);
          int cand = CL * lane;
          unsigned km = (unsigned)(x0[0] >> 32) & 0xfffu;
#pragma unroll
          for (int q = 1; q < CL; ++q) {
            const T ov = value_of<T>((unsigned)x0[q], (unsigned)x1[q]);
            const unsigned om = (unsigned)(x0[q] >> 32) & 0xfffu;
            const u64 ck = km & DIRECT_NONE ? 0ull : pivot_key(cv, cand * 64 + (int)(km & 63u) == k);
            const u64 ok = om & DIRECT_NONE ? 0ull : pivot_key(ov, (CL * lane + q) * 64 + (int)(om & 63u) == k);
            if (ok > ck) {
              cv = ov;
              km = om;
              cand = CL * lane + q;
            }
          }
          bool none;
          const int wl = pick_lane<T, 1, 64>(cv, in && !(km & DIRECT_NONE), cand * 64 + (int)(km & 63u) == k, &none);
          const int ws = __builtin_amdgcn_readlane(cand, wl);
          // the winner's values and row
          const u64* const pv = out + ws * MW + (lane < MW ? lane : 0);
          u64 y;
          for (;;) {
            y = ld_dev(pv);
            if (failed || !__any((unsigned)(y >> 32) != flag)) break;
            if (!spin_check(spins)) {
              failed = true;
              S.fail = 1;
              break;
            }
          }
          const unsigned wm = (unsigned)__builtin_amdgcn_readlane((int)km, wl);
          meta = (ws * 64 + (int)(wm & 63u)) | (int)(wm >> 6 & 31u) << 16;
          porg = __builtin_amdgcn_readlane((int)(unsigned)y, (LG + 1) * VW + 1);
#pragma unroll
          for (int c = 0; c < LG; ++c) uc[c] = word_value<T>((int)(unsigned)y, VW * c);
          rp = word_value<T>((int)(unsigned)y, VW * LG);
          if (wave == NW - 1 && lane < LG * VW) reinterpret_cast<unsigned*>(S.l[kk])[lane] = (unsigned)y;
        } else if (MULTI) {
          {
            const typename L::Msg& ms = S.wmsg[par][lane & (NW - 1)];
            const int cm = ms.meta;
            bool none;
            const int bw = pick_lane<T, 1, NW>(ms.v[kk], cm >= 0, (cm & 0xffff) == k, &none);
            u64* buf = xbuf + (size_t)par * MSG_PAR;
            if (wave == bw && lane < MW) put(buf + (size_t)b * MSGS + lane, ll_word(mine, flag));
            // row k, which only the owner of the pivot row needs, after the candidate
            if (top_wave && lane < KW) {
              const unsigned x = reinterpret_cast<const unsigned*>(&S.rowk[par])[lane];
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
                    unsigned* dst = sl < G ? reinterpret_cast<unsigned*>(&S.msg[par][sl])
                                           : reinterpret_cast<unsigned*>(&S.rowk[par]);
                    dst[wd] = (unsigned)x[q];
                    need[q] = false;
                  } else {
                    miss = true;
                  }
                }
              }
              if (!__any(miss)) break;
              if (!spin_check(spins)) {
                S.fail = 1;
                break;
              }
            }
          }
          __syncthreads();
          failed = S.fail != 0;
          const bool in = lane < G;
          const typename L::Msg& ms = S.msg[par][in ? lane : 0];
          const int cm = ms.meta, co = ms.org;
          const T crp = ms.rp;
          bool none;
          const int ws = pick_lane<T, 1, 64>(ms.v[kk], in && cm >= 0, (cm & 0xffff) == k, &none);
          const T x = S.msg[par][ws].v[lane & (LG - 1)];
          meta = __builtin_amdgcn_readlane(cm, ws);
          porg = __builtin_amdgcn_readlane(co, ws);
          rp = lane_value(crp, ws);
#pragma unroll
          for (int c = 0; c < LG; ++c) uc[c] = lane_value(x, c);
          if (wave == NW - 1 && lane < LG) S.l[kk][lane] = x;
        } else {
          int ln = lane;
          if (LEAN) asm volatile("" : "+v"(ln));  // (addresses made here, not kept over the steps)
          const typename L::Msg& ms = S.wmsg[par][(ln / LPS) & (NW - 1)];
          // lane j of a candidate holds value (j + kk + 1) % LV of the LV
          // values around kk, and value j of the others
          const int H = kk / LV;
          T x[VPL];
#pragma unroll
          for (int z = 0; z < VPL; ++z) x[z] = ms.v[z * LV + ((ln + (z == H ? kk + 1 : 0)) & (LV - 1))];
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
          if (wave == NW - 1 && (ln & ~(LPS - 1)) == w0) {
#pragma unroll
            for (int z = 0; z < VPL; ++z) S.l[kk][z * LV + ((ln + (z == H ? kk + 1 : 0)) & (LV - 1))] = x[z];
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
            T rv[LG];
            int ro = 0, rg = 0;
            if (DIRECT) {
#pragma unroll
              for (int c = 0; c < LG; ++c) rv[c] = word_value<T>((int)rk, VW * c);
              ro = __builtin_amdgcn_readlane((int)rk, VW * LG);
              rg = __builtin_amdgcn_readlane((int)rk, VW * LG + 1);
            }
            if (lr == p) {
#pragma unroll
              for (int c = 0; c < LG; ++c) v[c] = DIRECT ? rv[c] : S.rowk[par].v[c];
              osl = DIRECT ? ro : S.rowk[par].osl;
              corg = DIRECT ? rg : S.rowk[par].org;
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
        T* d = S.sw[myslot];
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
            x[q] = reinterpret_cast<const unsigned*>(S.sw[e / RS])[e % RS];
          }
#pragma unroll
          for (int q = 0; q < NR; ++q) put(rows + le + 64 * q, ll_word(x[q], flag));
        }
        for (u64 mb = __ballot(myslot != NOSLOT && myslot >= LG); mb != 0ull; mb &= mb - 1) {
          const int sl = __builtin_amdgcn_readlane(myslot, (int)__builtin_ctzll(mb));
          const unsigned* sw = reinterpret_cast<const unsigned*>(S.sw[sl]);
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
                reinterpret_cast<unsigned*>(S.sw[e / RS])[e % RS] = (unsigned)x[q];
                need[q] = false;
              } else {
                miss = true;
              }
            }
          }
          if (!__any(miss)) break;
          if (!spin_check(spins)) {
            S.fail = 1;
            break;
          }
        }
      }
      __syncthreads();
      if (MULTI) failed = S.fail != 0;
      auto take = [&]() {
        if (osl != myslot) {
          const T* d = S.sw[osl];
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
          for (int i = 0; i < LG; ++i) x[i] = S.sw[ts[i]][lane];
#pragma unroll
          for (int z = 0; z < LG - 1; ++z) {
#pragma unroll
            for (int i = z + 1; i < LG; ++i) x[i] = x[i] - S.l[i][z] * x[z];
          }
#pragma unroll
          for (int i = 0; i < LG; ++i) S.u[i][lane] = x[i];
        }
        __syncthreads();
        if (wave == NW - 1) take();
        T nl[LG], ua[LG];
#pragma unroll
        for (int i = 0; i < LG; ++i) nl[i] = -v[i];
        if (!LEAN) load_u(ua, 0);
        if (MULTI) {
          // the next group's columns now; the others beside its exchanges
          apply_u(ua, nl, v + LG, k0 + LG);
        } else if (LEAN) {
          // (four rows of U at a time: in FP64 the products join an element one by one)
#pragma unroll
          for (int q = 1; q < W / LG; ++q) {
            if (q <= rest) {
#pragma unroll
              for (int i0 = 0; i0 < LG; i0 += 4) {
                T u[4], t[LG];
#pragma unroll
                for (int i = 0; i < 4; ++i) u[i] = S.u[i0 + i][LG * (q - 1) + (lane & (LG - 1))];
                T* const vq = v + LG * q;
                if (top_wave) {
#pragma unroll
                  for (int c = 0; c < LG; ++c) t[c] = vq[c];
#pragma unroll
                  for (int i = 0; i < 4; ++i) fmac_lanes(t, u[i], nl[i0 + i]);
#pragma unroll
                  for (int c = 0; c < LG; ++c) vq[c] = lr >= k0 + LG ? t[c] : vq[c];
                } else {
#pragma unroll
                  for (int i = 0; i < 4; ++i) fmac_lanes(vq, u[i], nl[i0 + i]);
                }
              }
            }
          }
        } else if (!PREF) {
#pragma unroll
          for (int q = 1; q < W / LG; ++q) {
            if (q <= rest) {
              if (q > 1) load_u(ua, q - 1);
              apply_u(ua, nl, v + LG * q, k0 + LG);
            }
          }
        } else {
          T ub[LG];
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
          const T* d = S.u[lr - k0];
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
}

}  // namespace
}  // namespace la
