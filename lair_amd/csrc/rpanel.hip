// Panel leaf of the blocked LU with exact partial pivoting: the column loop of
// getrf_row_major (src/lapack/getrf.rs:55-117) with iamax's choice rule
// (src/blas/iamax.rs:6-21), for a tall leaf whose rows are spread over P
// cooperating workgroups of R = 256 RPT rows, RPT rows per thread.
//
// What bounds a leaf is the chain from one pivot to the next, so the leaf is
// cut into sub-panels of W columns, and one column's step is as short as the
// hardware lets it be:
//
//  * A row's W sub-panel entries live in registers and shift down by one each
//    column (entry c - 1 <- entry c - l u_c, the rank-1 update of
//    getrf.rs:76-88 with separate multiply and subtract), so every column is
//    the same short loop body and entry 0 is always the pivot column.
//  * Per column each wave finds its best row with 32-bit DPP maxima (the low
//    words and positions only on ties) and its lane puts the row into LDS.
//    With P = 1 one barrier later every thread picks the winner and updates.
//  * With P > 1 the workgroup's best row goes out as one record of tagged
//    64-bit words (position and the W entries, all updated), every wave polls
//    the records of P / 4 workgroups and puts them into LDS, and one barrier
//    later every thread picks the winner: one round trip through memory per
//    column.  A word is valid when its tag equals the column's tag, so no
//    fences are needed.
//  * After a sub-panel its L is written back, the pivot rows' other columns
//    are exchanged (one round trip per W columns), every workgroup solves
//    U = L11^-1 A for them and updates its own rows with rank W, in place in
//    global memory (its XCD's L2), with the same operations in the same order
//    as the unblocked loop: a leaf's factors do not depend on W or P.  (A
//    column without a candidate eliminates nothing; the sub-panel keeps a mask
//    of them.)  With P > 1 only the next sub-panel's columns are updated at once; the rest
//    fills the waits of the next column loop.
//
// Measured per leaf, against a leaf that kept 256 rows per workgroup in LDS
// and made two round trips per column (alone on the chip unless noted):
// FP64, 64 columns: 70 against 165 us at 100 rows, 104 / 172 at 512, 152 /
// 185 at 1024, 182 / 190 at 2048 inside a factorization; FP32, 128 columns:
// 211 / 370 us at 512 rows, 346 / 385 at 1024, 369 / 397 at 4096, 411 / 435
// at 16384; complex<f64>, 64 columns of 3000 rows, call included: 303 / 402.  A
// column costs about 0.9 us of instructions and LDS latencies (complex: 1.6)
// and, with P > 1, 0.8 us of round trip and 0.6 us for the slowest of the
// others.
//
// Rows do not move while the leaf is factored: every row carries its current
// position (its row index after the interchanges so far, as the reference
// would see it), which is also iamax's tie-break key (lowest index wins).  At
// the end the rows that changed place go through a tagged buffer and are
// stored by the workgroup that owns the destination: each address of the
// matrix is written by one workgroup only (two XCDs' L2 never hold dirty
// bytes of the same row).
#include <climits>
#include <type_traits>

#include "device_util.h"
#include "lair_internal.h"

namespace lair {

// Sub-panel width: its record (W entries, the position and the row) is one
// 64-bit word per lane.  Complex rows cost four times the arithmetic, and half
// of a sub-panel's entries are retired on average, so they take 8: complex<f32>
// 64 columns of 3000 rows 318 us against 327 with 16.
template <typename T>
struct RpW {
  static constexpr int W = cplx_traits<T>::is ? 8 : 16;
};

template <typename T>
struct RpArgs {
  T *a;
  int64_t lda;
  int row0, m, col0, wcols, npiv, P;
  int64_t *ipiv;
  int64_t *sing;
  unsigned long long *rec;  // [2][kMaxPanelWG][kRpRecWords] column records, by column parity
  unsigned long long *blk;  // [2][kRpMaxW][kRpRowWords] pivot rows of a sub-panel, by sub-panel parity
  unsigned long long *mv;   // [2 * kRpMaxCols][kRpRowWords] rows that change place
  int *map_rows, *map_src, *map_count;  // row map of the leaf's interchanges (optional)
  uint32_t seq;  // column j's tag is seq + j + 1, sub-panel s's seq + kRpTagBlk + s, the moves' seq + kRpTagMv
  int32_t *err;
  int wait_limit;  // polls before a wait gives up (0: every wait gives up at once)
};

constexpr uint32_t kRpTagBlk = 160, kRpTagMv = 192, kRpTags = 256;
static_assert(kRpMaxCols < (int)kRpTagBlk && kRpTagBlk + kRpMaxCols / 8 < kRpTagMv, "tags of a launch are distinct");

// iamax's key (src/blas/iamax.rs:14: |re| + |im| in the real type) and the
// pivot reciprocal (getrf.rs:76) of a real or complex element.
template <typename T>
__device__ __forceinline__ typename cplx_traits<T>::real rp_key(T x) {
  if constexpr (cplx_traits<T>::is)
    return fabs(x.re) + fabs(x.im);
  else
    return fabs(x);
}
template <typename T>
__device__ __forceinline__ T rp_recip(T v) {
  if constexpr (cplx_traits<T>::is)
    return cplx_recip(v);
  else
    return T(1) / v;
}

// Maximum of unsigned words over the wave (ROWS = 4) or over each row of 16
// lanes (ROWS = 1), in every lane.
template <int ROWS>
__device__ __forceinline__ uint32_t lanes_max_u32(uint32_t x) {
  auto step = [](uint32_t v, uint32_t o) { return v > o ? v : o; };
  x = step(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0xB1, 0xF, 0xF, true));
  x = step(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x4E, 0xF, 0xF, true));
  x = step(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x141, 0xF, 0xF, true));
  x = step(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x140, 0xF, 0xF, true));
  if constexpr (ROWS == 4) {
    const auto p = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    x = step(p[0], p[1]);
    const auto q = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    x = step(q[0], q[1]);
  }
  return x;
}

// iamax over one wave: the lane whose key is largest and, among equal keys,
// whose position is lowest; -1 without a candidate (key > 0, so zero and NaN
// are never chosen).  Keys are non-negative, so their bit patterns order as
// unsigned words.
template <typename R>
__device__ __forceinline__ int wave_best(R key, int pos) {
  const bool cand = key > R(0);
  if (!__builtin_amdgcn_ballot_w64(cand)) return -1;
  uint32_t kh, kl = 0;
  if constexpr (sizeof(R) == 8) {
    kh = (uint32_t)__double2hiint(key);
    kl = (uint32_t)__double2loint(key);
  } else {
    kh = __float_as_uint(key);
  }
  const uint32_t mh = lanes_max_u32<4>(cand ? kh : 0u);
  bool in = cand && kh == mh;
  if constexpr (sizeof(R) == 8) {
    const uint32_t ml = lanes_max_u32<4>(in ? kl : 0u);
    in = in && kl == ml;
  }
  const uint32_t mp = lanes_max_u32<4>(in ? ~(uint32_t)pos : 0u);
  const unsigned long long b = __builtin_amdgcn_ballot_w64(in && ~(uint32_t)pos == mp);
  return __ffsll((long long)b) - 1;
}

// The high word of an element's key, which alone decides a comparison unless
// two are equal or one is zero, subnormal, infinite or NaN: a maximum in
// [1, kKeyTop) with one holder is iamax's choice, anything else goes through
// wave_best.
template <typename T>
__device__ __forceinline__ uint32_t key_hi(T x) {
  typedef typename cplx_traits<T>::real R;
  R k;
  if constexpr (cplx_traits<T>::is)
    k = fabs(x.re) + fabs(x.im);
  else
    k = x;
  if constexpr (sizeof(R) == 8)
    return (uint32_t)__double2hiint(k);
  else
    return __float_as_uint(k);
}
template <typename R>
constexpr uint32_t kKeyTop = sizeof(R) == 8 ? 0x7FF00000u : 0x7F800000u;
// Whether a maximum needs wave_best (uniform).
template <typename R>
__device__ __forceinline__ bool key_rare(uint32_t mh, int holders) {
  const uint32_t m = (uint32_t)__builtin_amdgcn_readfirstlane((int)mh);
  return holders != 1 || m - 1u >= kKeyTop<R> - 1u;
}

// Values computed here, not later under a branch.
template <typename T>
__device__ __forceinline__ void pin(T &x) {
  if constexpr (cplx_traits<T>::is) {
    __asm__ volatile("" : "+v"(x.re), "+v"(x.im));
  } else {
    __asm__ volatile("" : "+v"(x));
  }
}

// N elements from 16-byte aligned LDS, by 16-byte reads.
template <typename T, int N>
__device__ __forceinline__ void lds_get(T (&x)[N], const T *src) {
  __builtin_memcpy(x, __builtin_assume_aligned(src, 16), sizeof(T) * N);
}

// Sizes of the kernel's LDS regions.
template <typename T, int RPT, int MR>
struct RpLds {
  typedef typename cplx_traits<T>::real R;
  static constexpr int W = RpW<T>::W;
  static constexpr int WPE = sizeof(T) / 4;
  // A record in 32-bit words: W entries, the position, the row it was loaded
  // from; RW is its pitch in LDS, with a spare word NW that the lanes past it
  // write.
  static constexpr int EW = W * WPE, PW = EW, OW = PW + 1, NW = OW + 1;
  static constexpr int RW = (NW + 4) & ~3;
  static constexpr int NR = kRpThreads * RPT;
  // Column pitch of the L tile: 16-byte aligned quads of rows, and the
  // coalesced loads (W lanes to a row) spread over all banks.
  static constexpr int LP = NR + (sizeof(T) == 4 ? 4 : 2);
  static constexpr int NBM = sizeof(T) == 4 ? kRpMaxCols : 64;  // widest leaf
  static constexpr int RESTM = NBM - W;
  static constexpr int MOVED = 2 * NBM < NR ? 2 * NBM : NR;  // rows of a workgroup that change place, at most
  // The update of the columns beyond the next sub-panel is put off into the
  // next column loop's waits (needs two L tiles).
  static constexpr bool kDefer = MR > 0 && RPT <= 2;
  static constexpr size_t kTile = sizeof(T) * W * LP;
  static constexpr size_t kL = (kDefer ? 2 : 1) * kTile;
  static constexpr size_t kC = sizeof(uint32_t) * 2 * kRpWaves * RW;
  static constexpr size_t kU11 = sizeof(T) * W * W;
  static constexpr size_t kRec = sizeof(uint32_t) * 2 * (MR * kRpWaves) * RW;
  static constexpr size_t kLL = sizeof(T) * W * W;
  static constexpr size_t kU = sizeof(T) * (size_t)W * RESTM;
  static constexpr size_t kRecLL = kRec > kLL ? kRec : kLL;
  static constexpr size_t total = kL + kC + kU11 + kRecLL + kU;
  static_assert(3 * sizeof(int) * MOVED <= kTile, "the lists of moved rows take the tile's place");
};

// RPT: rows per thread.  MR: workgroup records each wave polls (P <= MR *
// kRpWaves); 0: P = 1.
//
// A column costs its instructions (every wave's, four cycles each) plus a few
// LDS and memory latencies, so a workgroup is one wave per SIMD whatever its
// rows, and the column loop is written without branches where the hardware
// allows it (a taken branch costs as much as eight vector instructions):
// loads are clamped rather than masked, every row computes, and what a
// retired row computes is not used.
template <typename T, int RPT, int MR>
__global__ void __launch_bounds__(kRpThreads) rpanel_kernel(RpArgs<T> pa) {
#pragma clang fp contract(off)
  constexpr bool MULTI = MR > 0;
  typedef RpLds<T, RPT, MR> S;
  typedef typename S::R R;
  constexpr int W = S::W, WPE = S::WPE, EW = S::EW, PW = S::PW, OW = S::OW, NW = S::NW, RW = S::RW, LP = S::LP,
                NR = S::NR, NWV = kRpWaves, NT = kRpThreads;
  constexpr int WR = 64 * RPT;  // rows of a wave
  constexpr int RS = 64 / W;    // rows a wave copies at a time (W lanes to a row)
  typedef uint32_t raw_t __attribute__((ext_vector_type(WPE)));  // an element, for copies
  constexpr int JW = W / NWV;   // pivot rows of a sub-panel per wave
  static_assert(NW < 64 && kRpRecWords >= 64, "a record is one word per lane");
  static_assert(W <= kRpMaxW && S::NBM * WPE <= kRpRowWords, "exchanged rows fit their slots");
  static_assert(W * W <= NT && S::RESTM <= 2 * 64 && W % NWV == 0, "one pass over L11, two over a pivot row");
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *s_l = reinterpret_cast<T *>(smem_raw);                                // [W][LP] sub-panel, by column
  T *s_lold = reinterpret_cast<T *>(smem_raw + S::kL - S::kTile);          // the one before (kDefer)
  uint32_t *s_c = reinterpret_cast<uint32_t *>(smem_raw + S::kL);          // [2][NWV][RW] waves' best rows
  T *s_u11 = reinterpret_cast<T *>(smem_raw + S::kL + S::kC);              // [W][W] pivot rows, from their pivots on
  unsigned char *un_raw = smem_raw + S::kL + S::kC + S::kU11;
  uint32_t *s_r = reinterpret_cast<uint32_t *>(un_raw);                    // [2][MR * NWV][RW] workgroups' records
  T *s_lt = reinterpret_cast<T *>(un_raw);                                 // [W][W] L11 (between the column loops)
  T *s_u = reinterpret_cast<T *>(un_raw + S::kRecLL);                      // [W][un] pivot rows, then U
  __shared__ int s_po[kRpMaxCols];  // rows that the pivot rows were loaded from
  __shared__ __align__(16) int s_pw[kRpMaxCols];  // pivot positions of the leaf
  __shared__ int s_cnt, s_bail;
  __shared__ unsigned s_skip;  // columns of the sub-panel without a candidate

  const int g = blockIdx.x, t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int base = pa.row0 + g * NR;
  const int nvalid = min(NR, pa.m - base);  // rows of this workgroup
  const int ncols = pa.wcols;
  T *const rows = pa.a + (int64_t)base * pa.lda + pa.col0;  // this workgroup's rows of the leaf
  T *const wrows = rows + (int64_t)(wave * WR) * pa.lda;    // this wave's rows
  const int r0 = wave * WR + lane;                          // this thread's first row (the others 64 apart)

  int cpos[RPT];
  uint32_t amask[RPT];  // sign-clearing mask while the row is a candidate, else zero
#pragma unroll
  for (int s = 0; s < RPT; ++s) {
    cpos[s] = base + r0 + 64 * s;
    amask[s] = r0 + 64 * s < nvalid ? 0x7FFFFFFFu : 0u;
  }
  // Record keys of the waves and, in lanes, of the workgroups.
  const uint32_t wmask = lane < NWV ? 0x7FFFFFFFu : 0u, pmask = lane < pa.P ? 0x7FFFFFFFu : 0u;
  for (int e = t; e < kRpMaxCols; e += NT) s_po[e] = -1;
  if (t == 0) {
    s_bail = pa.wait_limit <= 0 ? 1 : 0;
    s_cnt = 0;
    s_skip = 0;
  }
  __syncthreads();
  bool bail = s_bail != 0;
  if (bail && t == 0) atomic_or_agent(pa.err, kErrWait);
  int done = 0;         // pivots decided
  int last_none = -1;  // last column without a candidate

  // The first sub-panel (each wave its own rows, W lanes to a row); the later
  // ones come from the update before them.
  {
    const int wc = lane % W, wr = lane / W, cw = min(W, ncols);
    const T *src = wrows + (int64_t)wr * pa.lda + wc;
#pragma unroll
    for (int s = 0; s < RPT; ++s) {
      T x[W];
#pragma unroll
      for (int i = 0; i < W; ++i)
        x[i] = wave * WR + 64 * s + wr + i * RS < nvalid && wc < cw ? src[(int64_t)(64 * s + i * RS) * pa.lda] : T(0);
#pragma unroll
      for (int i = 0; i < W; ++i) s_l[wc * LP + wave * WR + 64 * s + wr + i * RS] = x[i];
    }
  }

  // One block of the update A22 -= L21 U after a sub-panel that ended at
  // column c1: 64 of this wave's rows by W columns, separate multiply and
  // subtract, the columns of L in order: the same operations, in the same
  // order, as the unblocked column loop.  Each lane keeps 4 rows by TC
  // columns, so 16 bytes read from LDS feed four products.
  constexpr int TC = W / 4;
  struct Upd {
    int c1 = 0, rest = 0, un = 0, next = -1;  // next block (its rows vary fastest), counting down
    const T *l = nullptr;
    unsigned long long live[RPT] = {};
  } upd;
  const int rg = (lane >> 2) * 4, cg = (lane & 3) * TC;
  auto upd_live = [&](int rb) {
    unsigned long long m = upd.live[0];
#pragma unroll
    for (int s = 1; s < RPT; ++s) m = rb == s ? upd.live[s] : m;
    return (unsigned)(m >> rg) & 15u;
  };
  // C of block idx (whole: all its columns lie in the leaf).  Rows that do
  // not live load from a valid place and are not stored.
  auto upd_fetch = [&](int idx, T (&x)[4][TC]) {
    const int rb = idx % RPT, n0 = idx / RPT * W;
    const unsigned live = upd_live(rb);
    const T *cb = wrows + (int64_t)(64 * rb + rg) * pa.lda + upd.c1 + n0 + cg, *safe = rows + upd.c1;
#pragma unroll
    for (int i = 0; i < 4; ++i) __builtin_memcpy(x[i], live >> i & 1u ? cb + i * pa.lda : safe, sizeof(T) * TC);
  };
  auto upd_fetch_edge = [&](int idx, T (&x)[4][TC]) {
    const int rb = idx % RPT, n0 = idx / RPT * W;
    const unsigned live = upd_live(rb);
    const T *cb = wrows + (int64_t)(64 * rb + rg) * pa.lda + upd.c1, *safe = rows + upd.c1;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int q = 0; q < TC; ++q)
        x[i][q] = (live >> i & 1u ? cb + i * pa.lda : safe)[min(n0 + cg + q, upd.rest - 1)];
  };
  auto upd_mul_part = [&](int idx, T (&x)[4][TC], auto k0_, auto k1_) {
    constexpr int k0 = decltype(k0_)::value, k1 = decltype(k1_)::value;
    const int rb = idx % RPT, n0 = idx / RPT * W;
    const T *ucol = s_u + min(n0 + cg, upd.un - TC) + k0 * upd.un, *lcol = upd.l + wave * WR + 64 * rb + rg;
    T u[2][TC], l[2][4];
    lds_get<T, TC>(u[0], ucol);
    lds_get<T, 4>(l[0], lcol + k0 * LP);
#pragma unroll
    for (int k = k0; k < k1; ++k) {
      const int b = (k - k0) & 1;
      if (k + 1 < k1) {
        ucol += upd.un;
        lds_get<T, TC>(u[b ^ 1], ucol);
        lds_get<T, 4>(l[b ^ 1], lcol + (k + 1) * LP);
      }
      __builtin_amdgcn_sched_barrier(0);  // the next operands are on their way
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int q = 0; q < TC; ++q) {
          const T e = l[b][i] * u[b][q];
          x[i][q] = x[i][q] - e;
        }
    }
  };
  typedef std::integral_constant<int, 0> I0;
  typedef std::integral_constant<int, W / 2> IH;
  typedef std::integral_constant<int, W> IW;
  auto upd_mul = [&](int idx, T (&x)[4][TC]) { upd_mul_part(idx, x, I0(), IW()); };
  auto upd_store = [&](int idx, T (&x)[4][TC]) {
    const int rb = idx % RPT, n0 = idx / RPT * W;
    const unsigned live = upd_live(rb);
    T *cb = wrows + (int64_t)(64 * rb + rg) * pa.lda + upd.c1 + n0 + cg;
    if (n0 + W <= upd.rest) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (live >> i & 1u) __builtin_memcpy(cb + i * pa.lda, x[i], sizeof(T) * TC);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int q = 0; q < TC; ++q)
          if ((live >> i & 1u) && n0 + cg + q < upd.rest) cb[i * pa.lda + q] = x[i][q];
    }
  };

  for (int c0 = 0; c0 < pa.npiv && !bail; c0 += W) {
    const int sub = c0 / W;
    T *const s_lc = s_l;
    const int cw = min(W, ncols - c0);    // columns of the sub-panel
    const int np = min(W, pa.npiv - c0);  // pivots of the sub-panel
    uint32_t now[RPT];                    // rows that became pivot rows in this sub-panel
    T v[RPT][W];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int s = 0; s < RPT; ++s) {
      now[s] = 0u;
#pragma unroll
      for (int c = 0; c < W; ++c) v[s][c] = s_l[c * LP + r0 + 64 * s];
    }
    // Blocks of the previous sub-panel's update put off into this loop.
    const int nput = S::kDefer ? upd.next + 1 : 0;
    T cput[4][TC];
    if (S::kDefer && nput > 0) upd_fetch(upd.next + RPT, cput);

#pragma unroll 1
    for (int j = 0; j < np; ++j) {
      const int par = j & 1, jj = c0 + j, d = pa.row0 + jj;
      // The wave's candidate: largest |a| > 0, lowest position on ties.
      {
        uint32_t kh[RPT], km;
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
          kh[s] = key_hi(v[s][0]) & amask[s];
          km = s == 0 ? kh[0] : (km > kh[s] ? km : kh[s]);
        }
        const uint32_t mh = lanes_max_u32<4>(km);
        unsigned long long b[RPT];
        int holders = 0;
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
          b[s] = __builtin_amdgcn_ballot_w64(kh[s] == mh);
          holders += __popcll(b[s]);
        }
        int sw = 0, wl;
#pragma unroll
        for (int s = 1; s < RPT; ++s) sw = b[s] ? s : sw;
        {
          unsigned long long bb = b[0];
#pragma unroll
          for (int s = 1; s < RPT; ++s) bb |= b[s];
          wl = __ffsll((long long)bb) - 1;
        }
        uint32_t *dst = s_c + (par * NWV + wave) * RW;
        if (__builtin_expect(key_rare<R>(mh, holders), 0)) {
          R key = R(0);
          int pos = INT_MAX, sb = 0;
#pragma unroll
          for (int s = 0; s < RPT; ++s) {
            const R k = amask[s] ? rp_key(v[s][0]) : R(0);
            const bool better = k > key || (k == key && k > R(0) && cpos[s] < pos);
            key = better ? k : key;
            pos = better ? cpos[s] : pos;
            sb = better ? s : sb;
          }
          wl = wave_best<R>(key, pos);
          if (wl < 0) {
            // No candidate: an entry of zero, which no pick takes.
            if (lane == 0) {
              *reinterpret_cast<T *>(dst) = T(0);
              dst[PW] = (uint32_t)INT_MAX;
            }
          } else {
            sw = __builtin_amdgcn_readlane(sb, wl);
          }
        }
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
          if (sw == s && lane == wl) {
#pragma unroll
            for (int c = 0; c < W; ++c) reinterpret_cast<T *>(dst)[c] = v[s][c];
            dst[PW] = (uint32_t)cpos[s];
            dst[OW] = (uint32_t)(base + r0 + 64 * s);
          }
        }
      }
      __syncthreads();  // B1
      // The workgroup's candidate (the same choice among the waves' records).
      const uint32_t *rec = s_c + par * NWV * RW;
      int pw;
      bool none = false;
      {
        const uint32_t *rq = rec + min(lane, NWV - 1) * RW;
        int p = (int)rq[PW];
        T e0 = *reinterpret_cast<const T *>(rq);
        pin(p);
        pin(e0);
        const uint32_t kh = key_hi(e0) & wmask;
        const uint32_t mh = lanes_max_u32<1>(kh);
        const unsigned long long b = __builtin_amdgcn_ballot_w64(kh == mh) & 0xFFFFull;
        int q = __ffsll((long long)b) - 1;
        if (__builtin_expect(key_rare<R>(mh, __popcll(b)), 0)) {
          q = wave_best<R>(wmask && p != INT_MAX ? rp_key(e0) : R(0), p);
          none = q < 0;
          q = none ? 0 : q;
        }
        pw = __builtin_amdgcn_readlane(p, q);
        rec += q * RW;
      }
      bool due = false;
      if constexpr (MULTI) {
        const uint32_t tg = pa.seq + (uint32_t)jj + 1u;
        unsigned long long *rb = pa.rec + (size_t)par * kMaxPanelWG * kRpRecWords + lane;
        // Without a candidate every wave's record says so.
        if (wave == 0) st_agent(rb + g * kRpRecWords, tagged(tg, rec[min(lane, NW)]));
        // While the records travel: a block of the update put off, if one is
        // due; the loads go out in its middle, when the other records are
        // most likely there.
        due = S::kDefer && upd.next >= 0 && (nput - upd.next) * np <= nput * (j + 1);
        if constexpr (S::kDefer)
          if (due) upd_mul_part(upd.next + RPT, cput, I0(), IH());
        // Every wave takes the records wave, wave + NWV, ...
        unsigned long long w[MULTI ? MR : 1];
        auto poll = [&] {
#pragma unroll
          for (int i = 0; i < MR; ++i) w[i] = ld_agent(rb + min(wave + i * NWV, pa.P - 1) * kRpRecWords);
        };
        poll();
        if constexpr (S::kDefer)
          if (due) upd_mul_part(upd.next + RPT, cput, IH(), IW());
        for (int spins = 0;;) {
          bool ok = true;
#pragma unroll
          for (int i = 0; i < MR; ++i) ok = ok && (uint32_t)(w[i] >> 32) == tg;
          if (__builtin_expect(__all(ok), 1)) break;
          ++spins;
          if (__builtin_expect(spins >= pa.wait_limit || ((spins & 63) == 0 && ld_agent(pa.err) != 0), 0)) {
            if (lane == 0) {
              s_bail = 1;
              atomic_or_agent(pa.err, kErrWait);
            }
            break;
          }
          poll();
        }
        uint32_t *rr = s_r + par * (MR * NWV) * RW;
#pragma unroll
        for (int i = 0; i < MR; ++i) rr[(wave + i * NWV) * RW + min(lane, NW)] = (uint32_t)w[i];
        __syncthreads();  // B2
        const uint32_t *rq = rr + min(lane, pa.P - 1) * RW;
        int p = (int)rq[PW], bl = s_bail;
        T e0 = *reinterpret_cast<const T *>(rq);
        pin(p);
        pin(bl);
        pin(e0);
        bail = bl != 0;
        none = false;
        constexpr int LR = MR * NWV <= 16 ? 1 : 4;
        const uint32_t kh = key_hi(e0) & pmask;
        const uint32_t mh = lanes_max_u32<LR>(kh);
        const unsigned long long b = __builtin_amdgcn_ballot_w64(kh == mh) & (LR == 1 ? 0xFFFFull : ~0ull);
        int q = __ffsll((long long)b) - 1;
        if (__builtin_expect(key_rare<R>(mh, __popcll(b)), 0)) {
          q = wave_best<R>(pmask && p != INT_MAX ? rp_key(e0) : R(0), p);
          none = q < 0;
          q = none ? 0 : q;
        }
        pw = __builtin_amdgcn_readlane(p, q);
        rec = rr + q * RW;
        if (__builtin_expect(bail, 0)) break;
      }
      if (__builtin_expect(!none, 1)) {
        // The multipliers of column j and the update of the columns right of
        // it (getrf.rs:76-88).  One address register, the whole record in
        // flight at once.
        unsigned off = (unsigned)(reinterpret_cast<const unsigned char *>(rec) - smem_raw);
        __asm__ volatile("" : "+v"(off));
        const unsigned char *rv = smem_raw + off;
        T u[W];
        lds_get<T, W>(u, reinterpret_cast<const T *>(rv));
        const T ul = reinterpret_cast<const T *>(rv)[min(lane, W - 1)];
        const int po = (int)reinterpret_cast<const uint32_t *>(rv)[OW];
        __builtin_amdgcn_sched_barrier(0);
        const T ur = rp_recip(u[0]);  // (fills the wait for the rest of the record)
        // U's row j, kept for the sub-panel's store, and the pivot's place.
        s_u11[j * W + min(lane, W - 1)] = ul;
        s_po[jj] = po;
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
          const T l = v[s][0] * ur;
          s_l[j * LP + r0 + 64 * s] = l;
#pragma unroll
          for (int c = 1; c < W; ++c) {
            const T e = l * u[c];
            v[s][c - 1] = v[s][c] - e;
          }
        }
      } else {
        // A column without a nonzero candidate is left unscaled and nothing
        // is eliminated with it (getrf.rs:72-73); the row at position d is the
        // pivot row.
        pw = d;
        last_none = d;
        if (t == 0) s_skip |= 1u << j;
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
          s_l[j * LP + r0 + 64 * s] = v[s][0];
          if (cpos[s] == d) {
            s_po[jj] = base + r0 + 64 * s;
#pragma unroll
            for (int c = 0; c < W; ++c) s_u11[j * W + c] = v[s][c];
          }
#pragma unroll
          for (int c = 1; c < W; ++c) v[s][c - 1] = v[s][c];
        }
      }
      if constexpr (S::kDefer) {
        if (due) {
          upd_store(upd.next + RPT, cput);
          --upd.next;
          upd_fetch(max(upd.next, 0) + RPT, cput);
        }
      }
      s_pw[jj] = pw;
      // Interchange bookkeeping: the pivot row takes position d, the row at d
      // takes the pivot's old position (rows retired earlier lie above d).
#pragma unroll
      for (int s = 0; s < RPT; ++s) {
        const bool hit = cpos[s] == pw;
        now[s] = hit ? 1u : now[s];
        amask[s] = hit ? 0u : amask[s];
        cpos[s] = cpos[s] == d ? pw : cpos[s];
        cpos[s] = hit ? d : cpos[s];
      }
      done = jj + 1;
    }
    if (bail) break;

    // Opaque copies of the lane and the row pitch keep the addresses and masks
    // of the phases between the column loops from being computed ahead of the
    // loops and held in registers through them.
    if constexpr (S::kDefer) {
      for (; upd.next >= 0; --upd.next) {
        upd_mul(upd.next + RPT, cput);
        upd_store(upd.next + RPT, cput);
        upd_fetch(max(upd.next - 1, 0) + RPT, cput);
      }
    }
    int lane_o = lane;
    int64_t lda_o = pa.lda;
    __asm__ volatile("" : "+v"(lane_o));
    __asm__ volatile("" : "+s"(lda_o));
    unsigned long long m_live[RPT], m_store[RPT];
#pragma unroll
    for (int s = 0; s < RPT; ++s) {
      m_live[s] = __builtin_amdgcn_ballot_w64(amask[s] != 0u);
      m_store[s] = m_live[s] | __builtin_amdgcn_ballot_w64(now[s] != 0u);
    }
    const int c1 = c0 + W, rest = ncols - c1;
    const int un = (rest + 3) & ~3;  // pitch of U in LDS
    __syncthreads();
    // U11's rows into the tile, at the rows that own them.
    if (t < np * W) {
      const int j = t / W, c = t % W, pt = s_po[c0 + j] - base;
      if ((unsigned)pt < (unsigned)NR) {
        if (c >= j) s_l[c * LP + pt] = s_u11[j * W + c - j];
        // L11, when all of it is this workgroup's.
        if (!MULTI && rest > 0 && c < j) s_lt[j * W + c] = s_l[c * LP + pt];
      }
    }
    if (rest > 0) {
      // The pivot rows' multipliers and their entries right of the sub-panel.
      if constexpr (!MULTI) {
        raw_t x[JW][2];
#pragma unroll
        for (int i = 0; i < JW; ++i) {
          const int j = min(wave + i * NWV, np - 1);
          const T *src = rows + (int64_t)(s_po[c0 + j] - base) * lda_o + c1;
#pragma unroll
          for (int e = 0; e < 2; ++e) x[i][e] = *reinterpret_cast<const raw_t *>(src + min(lane_o + 64 * e, rest - 1));
        }
#pragma unroll
        for (int i = 0; i < JW; ++i) {
          const int j = min(wave + i * NWV, np - 1);
#pragma unroll
          for (int e = 0; e < 2; ++e)
            *reinterpret_cast<raw_t *>(s_u + j * un + min(lane_o + 64 * e, rest - 1)) = x[i][e];
        }
      } else {
        const uint32_t tb = pa.seq + kRpTagBlk + (uint32_t)sub;
        unsigned long long *bb = pa.blk + (size_t)(sub & 1) * kRpMaxW * kRpRowWords;
        const int rw = EW + rest * WPE;  // words per pivot row
        for (int j = wave; j < np; j += NWV) {
          const int pt = s_po[c0 + j] - base;
          if ((unsigned)pt >= (unsigned)NR) continue;
          const uint32_t *src = reinterpret_cast<const uint32_t *>(rows + (int64_t)pt * lda_o + c1) - EW;
          uint32_t x[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int k = min(lane_o + 64 * e, rw - 1);
            x[e] = src[max(k, EW)];
            const uint32_t y = reinterpret_cast<const uint32_t *>(s_l + (min(k, EW - 1) / WPE) * LP + pt)[k % WPE];
            x[e] = k < EW ? y : x[e];
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int k = min(lane_o + 64 * e, rw - 1);
            st_agent(bb + (size_t)j * kRpRowWords + k, tagged(tb, x[e]));
          }
        }
        unsigned long long w[JW][4];
        int spins = 0;
        for (;;) {
          bool ok = true;
#pragma unroll
          for (int i = 0; i < JW; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              w[i][e] = ld_agent(bb + (size_t)min(wave + i * NWV, np - 1) * kRpRowWords + min(lane_o + 64 * e, rw - 1));
#pragma unroll
          for (int i = 0; i < JW; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) ok = ok && (uint32_t)(w[i][e] >> 32) == tb;
          if (__all(ok)) break;
          ++spins;
          if (spins >= pa.wait_limit || ((spins & 63) == 0 && ld_agent(pa.err) != 0)) {
            if (lane_o == 0) {
              s_bail = 1;
              atomic_or_agent(pa.err, kErrWait);
            }
            break;
          }
        }
#pragma unroll
        for (int i = 0; i < JW; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int j = min(wave + i * NWV, np - 1), k = min(lane_o + 64 * e, rw - 1);
            *(k < EW ? reinterpret_cast<uint32_t *>(s_lt + j * W) + k
                     : reinterpret_cast<uint32_t *>(s_u + j * un) + (k - EW)) = (uint32_t)w[i][e];
          }
      }
    }
    __syncthreads();
    bail = s_bail != 0;
    if (bail) break;
    // The sub-panel back to the matrix (rows retired earlier already hold
    // their final entries there).
    {
      const int wc = lane_o % W, wr = lane_o / W;
#pragma unroll
      for (int s = 0; s < RPT; ++s) {
        const unsigned long long ms = wc < cw ? m_store[s] >> wr : 0ull;
        T *dst = wrows + (int64_t)(64 * s + wr) * lda_o + c0 + wc;
        T x[W];
#pragma unroll
        for (int i = 0; i < W; ++i) x[i] = s_l[wc * LP + wave * WR + 64 * s + wr + i * RS];
#pragma unroll
        for (int i = 0; i < W; ++i)
          if (ms >> (i * RS) & 1ull) dst[i * RS * lda_o] = x[i];
      }
    }
    if (rest <= 0) break;
    // U = L11^-1 A, one thread per column.
    const unsigned skip = (unsigned)__builtin_amdgcn_readfirstlane((int)s_skip);
    if (__builtin_expect(skip != 0, 0)) {
      if (t < rest)
#pragma unroll 1
        for (int i = 1; i < np; ++i) {
          T x = s_u[i * un + t];
#pragma unroll 1
          for (int q = 0; q < i; ++q)
            if (!(skip >> q & 1u)) {
              const T e = s_lt[i * W + q] * s_u[q * un + t];
              x = x - e;
            }
          s_u[i * un + t] = x;
        }
    } else if (t < rest) {
      T x[W];
#pragma unroll
      for (int i = 0; i < W; ++i) x[i] = s_u[i * un + t];
#pragma unroll
      for (int i = 1; i < W; ++i) {
        T l[W];
#pragma unroll
        for (int q = 0; q < i; ++q) l[q] = s_lt[i * W + q];
#pragma unroll
        for (int q = 0; q < i; ++q) {
          const T e = l[q] * x[q];
          x[i] = x[i] - e;
        }
        // Two rows of L11 at a time in registers.
        if (i % 2 == 0) __asm__ volatile("" : "+v"(reinterpret_cast<uint32_t &>(x[i])) : : "memory");
      }
#pragma unroll
      for (int i = 1; i < W; ++i)
        if (i < np) s_u[i * un + t] = x[i];
    }
    __syncthreads();
    if (t == 0) s_skip = 0;
    // The pivot rows' entries right of the sub-panel, by their owners.
#pragma unroll
    for (int i = 0; i < JW; ++i) {
      const int j = wave + i * NWV, pt = j < np ? s_po[c0 + j] - base : -1;
      if ((unsigned)pt < (unsigned)NR) {
        T *dst = rows + (int64_t)pt * lda_o + c1;
#pragma unroll
        for (int e = 0; e < 2; ++e)
          if (lane_o + 64 * e < rest) dst[lane_o + 64 * e] = s_u[j * un + lane_o + 64 * e];
      }
    }
    if (__builtin_expect(skip != 0, 0)) {
      // The update passes over columns without a candidate: with zeros for the
      // column of L and the row of U, both stored by now, it subtracts 0 from
      // every entry (their own values may be NaN, or meet an infinity).
      __syncthreads();
#pragma unroll 1
      for (int j = 0; j < np; ++j)
        if (skip >> j & 1u) {
#pragma unroll
          for (int s = 0; s < RPT; ++s) s_lc[j * LP + r0 + 64 * s] = T(0);
          if (t < un) s_u[j * un + t] = T(0);
        }
      __syncthreads();
    }
    // A22 -= L21 U on this wave's rows.  The next sub-panel's columns come
    // last and stay in LDS; with kDefer the whole blocks beyond them wait.
    upd.c1 = c1;
    upd.rest = rest;
    upd.un = un;
    upd.l = s_lc;
#pragma unroll
    for (int s = 0; s < RPT; ++s) upd.live[s] = m_live[s];
    if constexpr (S::kDefer) {
      // This tile's L is still needed: the next sub-panel goes to the other.
      s_l = s_lold;
      s_lold = s_lc;
    }
    {
      const int whole = rest / W;  // whole blocks of columns
      T c[4][TC], cnext[4][TC];
      if (whole * W < rest) {
        // A ragged last block.
        for (int rb = RPT - 1; rb >= 0; --rb) {
          const int idx = whole * RPT + rb;
          upd_fetch_edge(idx, c);
          upd_mul(idx, c);
          if (whole > 0) {
            upd_store(idx, c);
          } else {
            T *dst = s_l + wave * WR + 64 * rb + rg;
#pragma unroll
            for (int q = 0; q < TC; ++q)
#pragma unroll
              for (int i = 0; i < 4; ++i) dst[(cg + q) * LP + i] = c[i][q];
          }
        }
      }
      if (whole > 0) {
        const int last = S::kDefer ? RPT - 1 : whole * RPT - 1;
        upd_fetch(last, c);
#pragma unroll 1
        for (int idx = last; idx >= 0; --idx) {
          upd_fetch(max(idx - 1, 0), cnext);
          upd_mul(idx, c);
          if (idx >= RPT) {
            upd_store(idx, c);
          } else {
            T *dst = s_l + wave * WR + 64 * idx + rg;
#pragma unroll
            for (int q = 0; q < TC; ++q)
#pragma unroll
              for (int i = 0; i < 4; ++i) dst[(cg + q) * LP + i] = c[i][q];
          }
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int q = 0; q < TC; ++q) c[i][q] = cnext[i][q];
        }
      }
      // The blocks put off: RPT + next, ..., RPT.
      upd.next = S::kDefer ? max(whole - 1, 0) * RPT - 1 : -1;
    }
  }
  __syncthreads();
  if (g == 0) {
    // The pivots.  Given up: identity pivots for the columns not decided keep
    // the interchanges queued after this launch in bounds.
    for (int e = t; e < pa.npiv; e += NT) pa.ipiv[pa.row0 + e] = e < done ? s_pw[e] : pa.row0 + e;
    if (t == 0) {
      if (last_none >= 0) *pa.sing = last_none;
      if (pa.map_count) *pa.map_count = bail ? 0 : 2 * pa.npiv;
    }
  }
  if (bail) return;

  // Row map of the leaf's interchanges in gather form (rows[e] receives the
  // old contents of src[e]; rows[e] == src[e] is a no-op).  Slot e < npiv:
  // the final occupant of position row0 + e.  Slot npiv + e: where the row
  // that started at row0 + e went, when it left [row0, row0 + npiv).  Each
  // slot is written once, by the owner of the row it describes.
  const int top1 = pa.row0 + pa.npiv;
  int *s_mvt = reinterpret_cast<int *>(smem_raw), *s_out = s_mvt + S::MOVED, *s_in = s_out + S::MOVED;
#pragma unroll
  for (int s = 0; s < RPT; ++s) {
    if (r0 + 64 * s >= nvalid) continue;
    const int orig = base + r0 + 64 * s, fin = cpos[s];
    if (pa.map_rows) {
      if (fin < top1) {
        pa.map_rows[fin - pa.row0] = fin;
        pa.map_src[fin - pa.row0] = orig;
      }
      if (orig < top1) {
        pa.map_rows[pa.npiv + orig - pa.row0] = fin < top1 ? orig : fin;
        pa.map_src[pa.npiv + orig - pa.row0] = orig;
      }
    }
    if (fin != orig) {
      const int k = atomicAdd(&s_cnt, 1);
      s_mvt[k] = r0 + 64 * s;
      if constexpr (MULTI) {
        // This row leaves and another takes its place: the source of a
        // position is found by walking it back through the interchanges.  A
        // row's slot: its origin if that is one of the first npiv rows, else
        // its destination (which then is).
        int x = orig;
        for (int e = (pa.npiv - 1) & ~7; e >= 0; e -= 8) {
          int pe[8];
          lds_get<int, 8>(pe, s_pw + e);
#pragma unroll
          for (int q = 7; q >= 0; --q) {
            const int de = pa.row0 + e + q, pq = e + q < pa.npiv ? pe[q] : de;
            x = x == de ? pq : (x == pq ? de : x);
          }
        }
        s_out[k] = orig < top1 ? kRpMaxCols + orig - pa.row0 : fin - pa.row0;
        s_in[k] = x < top1 ? kRpMaxCols + x - pa.row0 : orig - pa.row0;
      } else {
        s_out[k] = fin - base;
      }
    }
  }
  __syncthreads();
  const int cnt = s_cnt;
  if (cnt == 0) return;
  if constexpr (!MULTI) {
    // Rows within the workgroup: 64 columns at a time through registers, all
    // loaded before any is stored.  Lanes and rows past the end repeat the
    // last one.
    constexpr int BR = 16, NB = (S::MOVED / NWV + BR - 1) / BR;
    for (int cb = 0; cb < ncols; cb += 64) {
      const T *src = rows + min(cb + lane, ncols - 1);
      T *dst = rows + min(cb + lane, ncols - 1);
      raw_t x[NB][BR];
#pragma unroll
      for (int b = 0; b < NB; ++b)
        if (b * BR * NWV < cnt) {
#pragma unroll
          for (int i = 0; i < BR; ++i)
            x[b][i] = *reinterpret_cast<const raw_t *>(
                src + (int64_t)s_mvt[min(wave + (b * BR + i) * NWV, cnt - 1)] * pa.lda);
        }
      // Every load has arrived before the first store.
      __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
#pragma unroll
      for (int b = 0; b < NB; ++b)
        if (b * BR * NWV < cnt) {
#pragma unroll
          for (int i = 0; i < BR; ++i)
            *reinterpret_cast<raw_t *>(dst + (int64_t)s_out[min(wave + (b * BR + i) * NWV, cnt - 1)] * pa.lda) =
                x[b][i];
        }
    }
  } else {
    // Through the tagged slots, 64 words of 16 rows at a time.
    constexpr int BR = 16;
    const int wpr = ncols * WPE;
    const uint32_t tm = pa.seq + kRpTagMv;
    for (int e0 = wave; e0 < cnt; e0 += BR * NWV)
      for (int k0 = 0; k0 < wpr; k0 += 64) {
        const int k = min(k0 + lane, wpr - 1);
        uint32_t x[BR];
#pragma unroll
        for (int i = 0; i < BR; ++i)
          x[i] = reinterpret_cast<const uint32_t *>(rows + (int64_t)s_mvt[min(e0 + i * NWV, cnt - 1)] * pa.lda)[k];
#pragma unroll
        for (int i = 0; i < BR; ++i)
          st_agent(pa.mv + (size_t)s_out[min(e0 + i * NWV, cnt - 1)] * kRpRowWords + k, tagged(tm, x[i]));
      }
    __syncthreads();
    for (int e0 = wave; e0 < cnt; e0 += BR * NWV)
      for (int k0 = 0; k0 < wpr; k0 += 64) {
        const int k = min(k0 + lane, wpr - 1);
        unsigned long long w[BR];
        int spins = 0;
        for (;;) {
          bool ok = true;
#pragma unroll
          for (int i = 0; i < BR; ++i)
            w[i] = ld_agent(pa.mv + (size_t)s_in[min(e0 + i * NWV, cnt - 1)] * kRpRowWords + k);
#pragma unroll
          for (int i = 0; i < BR; ++i) ok = ok && (uint32_t)(w[i] >> 32) == tm;
          if (__all(ok)) break;
          ++spins;
          if (spins >= pa.wait_limit || ((spins & 63) == 0 && ld_agent(pa.err) != 0)) {
            if (lane == 0) atomic_or_agent(pa.err, kErrWait);
            break;
          }
        }
#pragma unroll
        for (int i = 0; i < BR; ++i)
          reinterpret_cast<uint32_t *>(rows + (int64_t)s_mvt[min(e0 + i * NWV, cnt - 1)] * pa.lda)[k] = (uint32_t)w[i];
      }
  }
}

template <typename T, int RPT, int MR>
static hipError_t rp_launch(lair_context *ctx, const RpArgs<T> &pa) {
  auto *k = &rpanel_kernel<T, RPT, MR>;
  constexpr size_t shm = RpLds<T, RPT, MR>::total;
  static bool once = ((void)hipFuncSetAttribute(reinterpret_cast<const void *>(k),
                                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                                (int)shm),
                      (void)hipGetLastError(), true);
  (void)once;
  k<<<pa.P, kRpThreads, shm, ctx->stream>>>(pa);
  return hipGetLastError();
}

// Several workgroups, one or two rows per thread: the fewest records a wave
// has to poll.  (Complex leaves of two rows per thread have more than 32
// workgroups, unless the workgroups are capped.)
template <typename T>
static hipError_t rp_launch_multi(lair_context *ctx, const RpArgs<T> &pa, int rpt) {
  if constexpr (cplx_traits<T>::is) {
    if (rpt == 2) return rp_launch<T, 2, 16>(ctx, pa);
  }
  constexpr int RPT = cplx_traits<T>::is ? 1 : 2;
  const int mr = (pa.P + kRpWaves - 1) / kRpWaves;
  if (mr <= 1) return rp_launch<T, RPT, 1>(ctx, pa);
  if (mr <= 2) return rp_launch<T, RPT, 2>(ctx, pa);
  if (mr <= 4) return rp_launch<T, RPT, 4>(ctx, pa);
  if (mr <= 8) return rp_launch<T, RPT, 8>(ctx, pa);
  return rp_launch<T, RPT, 16>(ctx, pa);
}

// Rows per thread of a leaf over `rows` rows, or 0 when the leaf does not fit
// the cooperating workgroups.  `beside`: columns of the trailing update that
// runs at the same time.
//
// More rows per thread save exchanges (one workgroup needs none), fewer save
// arithmetic per column.  A factorization of m x 64, call included, us:
//   rows        f64: 4 a thread, one workgroup / 2, two workgroups  226 / 262
//   513 - 1024  f32                                                 206 / 243
//               complex: 4, one / 2, two / 1, four  f32: 336 / 302 / 262
//                                                   f64: 418 / 338 / 294
//   3000        complex: 2, six / 1, twelve         f32: 325 / 264, f64: 354 / 300
//   20000       4, twenty / 2, forty   f64: 374 / 299, f32: 349 / 288,
//                                      complex f32: 491 / 347, f64: 588 / 405
// Beyond 32 workgroups the trailing update loses as many CUs, so there the
// leaf has 4 rows a thread while that update sets the pace.  The two cross at
// about 24000 bytes of a row beside the panel: 24000 rows of n columns gain
// most at n = 6000 in f32 (34.3 against 25.9 ms), 3000 in f64 (17.9 / 15.3) and
// complex<f32> (23.4 / 19.2), 1500 - 2000 in complex<f64> (19.9 / 16.2), and
// lose beyond n = 14000 in f32 (78.8 / 81).
constexpr int64_t kRpBesideBytes = 24000;
template <typename T>
static int rp_rpt(lair_context *ctx, int rows, int beside) {
  const int maxp = std::min(ctx->rp_max_wg, kMaxPanelWG);
  // Complex<f64> keeps to 32768 rows, the limit its entry points state.
  if (sizeof(T) == 16 && rows > 32768) return 0;
  if (rows <= kRpThreads) return 1;
  if (rows <= 2 * kRpThreads) return 2;
  if (cplx_traits<T>::is && rows <= kRpThreads * maxp) return 1;
  if (rows <= 4 * kRpThreads) return 4;
  if (rows <= 2 * kRpThreads * std::min(maxp, 32)) return 2;
  if (rows <= 2 * kRpThreads * maxp && beside * (int64_t)sizeof(T) <= kRpBesideBytes) return 2;
  return rows <= 4 * kRpThreads * maxp ? 4 : 0;
}

template <typename T>
int rpanel_grid(lair_context *ctx, int rows, int beside) {
  const int nr = rp_rpt<T>(ctx, rows, beside) * kRpThreads;
  return nr > 0 ? (rows + nr - 1) / nr : 0;
}

// Widest leaf (<= want) for `rows` rows.
template <typename T>
int rpanel_leaf_width(lair_context *ctx, int want, int rows) {
  return rpanel_grid<T>(ctx, rows, 0) > 0 ? std::min(want, RpLds<T, 1, 0>::NBM) : 0;
}

template <typename T>
hipError_t launch_rpanel(lair_context *ctx, T *a, int64_t lda, int row0, int m, int col0, int wcols, int beside,
                         int64_t *ipiv, int *map_rows, int *map_src, int *map_count) {
  const int rows = m - row0;
  if (rows <= 0 || wcols <= 0) return hipSuccess;
  const int rpt = rp_rpt<T>(ctx, rows, beside);
  if (rpt == 0 || wcols > RpLds<T, 1, 0>::NBM) return hipErrorInvalidValue;
  // A reused tag could match a stale word: clear the buffers and restart the
  // tags before they wrap.
  if (ctx->rp_seq > 0xF0000000u) {
    hipError_t e = launch_fill_u32(ctx, reinterpret_cast<uint32_t *>(ctx->rp_buf), 2 * kRpBufWords, 0u);
    if (e != hipSuccess) return e;
    ctx->rp_seq = 1u;
  }
  RpArgs<T> pa;
  pa.a = a;
  pa.lda = lda;
  pa.row0 = row0;
  pa.m = m;
  pa.col0 = col0;
  pa.wcols = wcols;
  pa.npiv = wcols < rows ? wcols : rows;
  pa.P = rpanel_grid<T>(ctx, rows, beside);
  pa.ipiv = ipiv;
  pa.sing = ctx->sing;
  pa.map_rows = map_rows;
  pa.map_src = map_src;
  pa.map_count = map_count;
  pa.rec = ctx->rp_buf;
  pa.blk = ctx->rp_buf + kRpBlkOff;
  pa.mv = ctx->rp_buf + kRpMvOff;
  pa.seq = ctx->rp_seq;
  pa.err = ctx->err;
  pa.wait_limit = ctx->wait_limit;
  const int slot = prof_begin(ctx, LAIR_KCLASS_PANEL);
  hipError_t e;
  if (pa.P == 1)
    e = rpt == 1 ? rp_launch<T, 1, 0>(ctx, pa) : (rpt == 2 ? rp_launch<T, 2, 0>(ctx, pa) : rp_launch<T, 4, 0>(ctx, pa));
  else if (rpt == 4)
    e = rp_launch<T, 4, 16>(ctx, pa);
  else
    e = rp_launch_multi<T>(ctx, pa, rpt);
  prof_end(ctx, slot, LAIR_KCLASS_PANEL, (double)pa.npiv * rows * wcols,
           2.0 * sizeof(T) * (double)rows * wcols);
  ctx->rp_seq += kRpTags;
  return e;
}

#define LAIR_RP_INST(T)                                                                                \
  template int rpanel_grid<T>(lair_context *, int, int);                                               \
  template int rpanel_leaf_width<T>(lair_context *, int, int);                                         \
  template hipError_t launch_rpanel<T>(lair_context *, T *, int64_t, int, int, int, int, int, int64_t *, int *,        \
                                       int *, int *);
LAIR_RP_INST(float)
LAIR_RP_INST(double)
LAIR_RP_INST(zcplx)
LAIR_RP_INST(ccplx)

}  // namespace lair
