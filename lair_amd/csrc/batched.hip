// Batched solve of many independent small systems A_i X_i = B_i (n_i <= 256,
// nrhs_i <= 16): one workgroup per system, of one, two or four waves for
// n <= 64, 128, 256 (a thread per row), started in order of decreasing n.
//
// The augmented matrix [A | B] is factored in place by a blocked right-looking
// LU with partial pivoting (src/lapack/getrf.rs:46-120, blocked; the
// interchanges are applied to B as getrs.rs:23 does), so the forward
// substitution comes with the factorization; a blocked back substitution with
// U gives X (getrs.rs:30-36).  Blocks are 32 columns wide (two register panels
// of 16), which reads and writes the trailing matrix n / 32 times:
//  * thread t keeps row kb + t of a panel in registers.  Rows never move
//    during a panel: every thread tracks the position of its row, a pivot only
//    exchanges two positions, and the rows are put in place in LDS at the
//    panel's end.  Per column: an argmax per wave over the rows at positions
//    from the diagonal on (ties -> lowest position; NaN and zero never chosen,
//    src/blas/iamax.rs:6-21), each wave's winner publishes its row, one
//    barrier, the reciprocal scaling and rank-1 update (getrf.rs:76-88,
//    separate multiply and subtract);
//  * the left panel's elimination reaches the right one, and trailing columns
//    in chunks of 16 (a wave each, no barrier), on the matrix cores: the 32
//    interchanged rows are read through the row map, U12 = L11^-1 A12 takes
//    the two inverted 16 x 16 diagonal blocks, then A22 -= L21 U12.  An MFMA
//    result is laid out as the next one's second operand, so U12 never leaves
//    the registers; L comes from LDS;
//  * the interchanges of later blocks reach the columns of L once, at the end.
//
// Bound by the chain of columns (850 cycles with one wave, 1400 with four) at
// 2 to 7 workgroups per CU and, for large n, by the latency of the passes over
// the trailing matrix; the code (40 - 51 KB) has to stay within the 64 KB
// instruction cache (at 61 - 71 KB a column took twice as long).  Whole
// solves, input copies included, against one persistent kernel with panels of
// 8 or 16 columns and register-tile updates chosen by timing: 4096 systems in
// FP64 of n = 256: 4.80 ms against 10.66; 128: 1.16 against 2.38; 64: 0.27
// against 0.71; 32: 0.13 against 0.34; 5000 of n = 8 .. 256: 2.49 against 4.78;
// 3000 in FP32 of n = 8 .. 128: 0.23 against 0.48.
#include <algorithm>
#include <climits>

#include "lair_internal.h"

namespace lair {

constexpr int kBatchW = 32;        // block width: two register panels of 16
constexpr int kBatchMaxRhs = 16;

template <typename T>
struct BatchArgs {
  const int *n;          // [count]
  const int *nrhs;       // [count]
  const int64_t *a_off;  // element offsets of A_i (row-major, ld = n_i)
  const int64_t *b_off;  // element offsets of B_i (row-major, ld = nrhs_i)
  const int64_t *p_off;  // offsets of ipiv_i (n_i entries)
  const int *order;      // processing order
  T *a;
  T *b;
  int64_t *ipiv;
  int *info;             // -1, or the last zero-pivot column (getrf.rs:72-73)
};

template <int CTRL, int ROWM = 0xF>
__device__ __forceinline__ uint32_t bdpp(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROWM, 0xF, false);
}
__device__ __forceinline__ uint32_t bwave_max(uint32_t v) {
  v = max(v, bdpp<0xB1>(v));        // quad_perm [1,0,3,2]
  v = max(v, bdpp<0x4E>(v));        // quad_perm [2,3,0,1]
  v = max(v, bdpp<0x141>(v));       // row_half_mirror
  v = max(v, bdpp<0x140>(v));       // row_mirror
  v = max(v, bdpp<0x142, 0xA>(v));  // row_bcast:15
  v = max(v, bdpp<0x143, 0xC>(v));  // row_bcast:31
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// |x| as an ordered pattern; zero for zero and NaN (which are never chosen).
__device__ __forceinline__ unsigned long long pivot_key(double x) {
  const unsigned long long k = (unsigned long long)__double_as_longlong(x) & 0x7fffffffffffffffull;
  return k <= 0x7ff0000000000000ull ? k : 0;
}
__device__ __forceinline__ uint32_t pivot_key(float x) {
  const uint32_t k = __float_as_uint(x) & 0x7fffffffu;
  return k <= 0x7f800000u ? k : 0;
}
__device__ __forceinline__ uint32_t key_hi(unsigned long long k) { return (uint32_t)(k >> 32); }
__device__ __forceinline__ uint32_t key_hi(uint32_t k) { return k; }

// The value of lane I of each row of 16 lanes.
template <int I>
__device__ __forceinline__ double row_lane(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x150 + I, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x150 + I, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}
template <int I>
__device__ __forceinline__ float row_lane(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x150 + I, 0xF, 0xF, false));
}

// MFMA 16 x 16 x 4: lane (g = lane / 16, lc = lane % 16) gives A[lc][k] and
// B[k][lc] and holds rows row(g, r), column lc of the result.  Step s of a
// product over 16 k takes k = row(g, s), so that result register s is the
// second operand of step s.
template <typename T>
struct BatchMfma;
template <>
struct BatchMfma<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 op(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int g, int r) { return g + 4 * r; }
  static constexpr int kStep = 4;  // row step of a result register
};
template <>
struct BatchMfma<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 op(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int g, int r) { return 4 * g + r; }
  static constexpr int kStep = 1;
};

// A row-major matrix behind a buffer descriptor: an element past its end reads
// as zero and is not written, so ragged rows need no masks (and no code; the
// kernel has to fit the instruction cache).  Offsets are in elements.
template <typename T>
struct BatchBuf {
  __amdgpu_buffer_rsrc_t rsrc;
  static constexpr uint32_t kNone = 0x7fffffffu / sizeof(T);  // past any end
  __device__ __forceinline__ BatchBuf(T *p, int count)
      : rsrc(__builtin_amdgcn_make_buffer_rsrc(p, 0, count * (int)sizeof(T), 0x00020000)) {}
  __device__ __forceinline__ T load(uint32_t e) const {
    T v;
    if constexpr (sizeof(T) == 8) {
      const auto w = __builtin_amdgcn_raw_buffer_load_b64(rsrc, e * 8u, 0, 0);
      __builtin_memcpy(&v, &w, 8);
    } else {
      const auto w = __builtin_amdgcn_raw_buffer_load_b32(rsrc, e * 4u, 0, 0);
      __builtin_memcpy(&v, &w, 4);
    }
    return v;
  }
  __device__ __forceinline__ void store(uint32_t e, T v) const {
    if constexpr (sizeof(T) == 8) {
      typedef unsigned int u2 __attribute__((ext_vector_type(2)));
      u2 w;
      __builtin_memcpy(&w, &v, 8);
      __builtin_amdgcn_raw_buffer_store_b64(w, rsrc, e * 8u, 0, 0);
    } else {
      unsigned int w;
      __builtin_memcpy(&w, &v, 4);
      __builtin_amdgcn_raw_buffer_store_b32(w, rsrc, e * 4u, 0, 0);
    }
  }
};

template <typename T, int NW>
struct BatchSolver {
  typedef BatchMfma<T> M;
  typedef typename M::v4 v4;
  static constexpr int NT = 64 * NW;               // threads, and most rows
  static constexpr int W = kBatchW, H = 16;
  static constexpr int NBLK = NT / W;              // most blocks
  static constexpr int PL = W + 16 / sizeof(T);    // LDS row of a block: MFMA operand reads on distinct banks
  static constexpr int PI = H + (sizeof(T) == 8 ? 2 : 4);
  static constexpr int YP = NT + 4;                // LDS pitch of a right-hand side
  typedef decltype(pivot_key(T(0))) key_t;
  struct Lds {
    T p[NT][PL];                   // the block, rows by position; later Y
    T inv[2][H][PI];               // inverses of the block's two unit lower 16 x 16 triangles
    T cand[2][NW][H + 16 / sizeof(T)];  // each wave's candidate row, by column parity; [H]: its reciprocal pivot
    key_t key[2][NW];              // the candidate's pivot magnitude
    int pos[2][NW];                // and its position
    unsigned char src[NT];         // row (offset in the block) that each position receives
    unsigned char rows[W], from[W];  // positions >= W that receive another row, and that row
    unsigned char orig[NT];        // matrix row at each position
    unsigned char hist[NBLK][NT];  // position of each matrix row after each block
    unsigned char piv[NT];         // pivot positions
    int cnt, moved;
  };
  static_assert(kBatchMaxRhs * YP <= NT * PL, "Y fits the block's rows");

  Lds &S;
  const int t, lane, wave, g, lc;
  const int n, r;
  const BatchBuf<T> A, B;
  int sing;
  unsigned none;  // columns of the block without a candidate

  __device__ __forceinline__ BatchSolver(Lds &s, int n_, int r_, T *a, T *b)
      : S(s), t(threadIdx.x), lane(threadIdx.x & 63), wave(threadIdx.x >> 6), g(lane >> 4), lc(lane & 15), n(n_),
        r(r_), A(a, n_ * n_), B(b, n_ * r_), sing(-1), none(0) {}

  // Barrier for data in LDS only: unlike __syncthreads it does not wait for
  // global loads and stores in flight.
  __device__ __forceinline__ static void lds_sync() {
    __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (NW > 1) __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
  }
  // Sixteen values of an LDS row, at a 16-byte boundary.
  __device__ __forceinline__ static void get(T (&v)[H], const T *row) {
    __builtin_memcpy(v, __builtin_assume_aligned(row, 16), sizeof v);
  }
  __device__ __forceinline__ static void put(T *row, const T (&v)[H]) {
    __builtin_memcpy(__builtin_assume_aligned(row, 16), v, sizeof v);
  }

  // Sixteen columns (from offset d0 of the block) of the rows in registers.
  // Every lane takes the reciprocal of its own entry while the argmax (over
  // the high words, ties by the rest) goes on: the winner publishes it.
  __device__ __forceinline__ void panel(T (&v)[H], int &pos, int kb, int d0, int w) {
#pragma clang fp contract(off)
#pragma unroll
    for (int j = 0; j < H; ++j) {
      const int d = d0 + j, par = j & 1;
      if (__builtin_expect(d < w, 1)) {
        const key_t key = pos >= d ? pivot_key(v[j]) : key_t(0);
        T rec = T(1) / v[j];
        __asm__ volatile("" : "+v"(rec));  // now, not in the winner's branch
        const uint32_t hi = key_hi(key), hmax = bwave_max(hi);
        unsigned long long mm = __builtin_amdgcn_ballot_w64(hi == hmax && key != 0);
        int wl = mm ? __ffsll((long long)mm) - 1 : 0;
        if (__builtin_expect((mm & (mm - 1)) != 0 && mm != 0, 0)) {
          key_t bk = 0;
          int bp = INT_MAX;
          while (mm) {
            const int l = __ffsll((long long)mm) - 1;
            mm &= mm - 1;
            const int pl = __builtin_amdgcn_readlane(pos, l);
            key_t kl = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)key, l);
            if (sizeof(T) == 8) kl |= (key_t)(((unsigned long long)hmax << 16) << 16);
            if (kl > bk || (kl == bk && pl < bp)) {
              bk = kl;
              bp = pl;
              wl = l;
            }
          }
        }
        if (lane == wl) {
#pragma unroll
          for (int c = j & ~1; c < H; ++c) S.cand[par][wave][c] = v[c];
          S.cand[par][wave][H] = rec;
          S.key[par][wave] = key;
          S.pos[par][wave] = pos;
        }
        lds_sync();
        // The workgroup's winner, by the high words; equal ones in full.
        key_t ck[NW];
        int cp[NW];
#pragma unroll
        for (int q = 0; q < NW; ++q) {
          ck[q] = S.key[par][q];
          cp[q] = S.pos[par][q];
        }
        uint32_t ch = key_hi(ck[0]);
        int pw = 0;
        bool tie = false;
#pragma unroll
        for (int q = 1; q < NW; ++q) {
          const uint32_t oh = key_hi(ck[q]);
          tie = oh == ch || (tie && oh < ch);
          pw = oh > ch ? q : pw;
          ch = max(oh, ch);
        }
        if (NW > 1 && __builtin_expect(__builtin_amdgcn_ballot_w64(tie) != 0, 0)) {
          key_t bk = ck[0];
          int bp = cp[0];
          pw = 0;
#pragma unroll
          for (int q = 1; q < NW; ++q) {
            const bool take = ck[q] > bk || (ck[q] == bk && bk != 0 && cp[q] < bp);
            bk = take ? ck[q] : bk;
            bp = take ? cp[q] : bp;
            pw = take ? q : pw;
          }
        }
        const T *prow = S.cand[par][pw];
        T pv[H], prec = prow[H];
#pragma unroll
        for (int c = j + 1; c < H; ++c) pv[c] = prow[c];
        key_t bk = ck[0];
        int pr = cp[0];
#pragma unroll
        for (int q = 1; q < NW; ++q) {
          bk = pw == q ? ck[q] : bk;
          pr = pw == q ? cp[q] : pr;
        }
        const bool singular = bk == 0;
        pr = singular ? d : pr;
        none = singular ? none | 1u << d : none;
        pos = pos == d ? pr : (pos == pr ? d : pos);
        S.piv[kb + d] = (unsigned char)(kb + pr);
        if (__builtin_expect(!singular && pos > d, 1)) {
          const T l = v[j] * prec;
          v[j] = l;
#pragma unroll
          for (int c = j + 1; c < H; ++c) {
            const T e = l * pv[c];
            v[c] = v[c] - e;
          }
        }
      }
    }
  }

  // The rows to their positions in LDS: this half from registers, the other
  // half from where the row was.  org: the row's position before the block.
  __device__ __forceinline__ void place(const T (&v)[H], int pos, int half, int &org) {
    T other[H];
    const bool mv = pos != t;
    if (mv) get(other, &S.p[t][(1 - half) * H]);
    lds_sync();
    put(&S.p[pos][half * H], v);
    if (mv) put(&S.p[pos][(1 - half) * H], other);
    S.src[pos] = (unsigned char)org;
    lds_sync();
    org = S.src[t];
  }

  // One 16-deep product: the sum of a(row lc of `rowp`) * b.
  __device__ __forceinline__ v4 prod(const T *rowp, v4 b) const {
    v4 c = v4{T(0), T(0), T(0), T(0)};
#pragma unroll
    for (int s = 0; s < 4; ++s) c = M::op(rowp[M::row(g, s)], b[s], c);
    return c;
  }

  // 0, or NaN if an entry is not finite.
  __device__ __forceinline__ static T zero_if_finite(v4 x) {
    T s = T(0);
#pragma unroll
    for (int e = 0; e < 4; ++e) s = __builtin_elementwise_fma(x[e], T(0), s);
    return s;
  }

  // Inverse of unit lower triangle h of the block's diagonal: lane j column
  // j, by substitution.  Rows past the matrix are zero.
  __device__ __forceinline__ void invert(int h) {
    if (lane < H) {
      T x[H];
#pragma unroll
      for (int i = 0; i < H; ++i) x[i] = i == lane ? T(1) : T(0);
#pragma unroll
      for (int q = 0; q < H; ++q) {
        S.inv[h][q][lane] = x[q];
#pragma unroll
        for (int i = q + 1; i < H; ++i) x[i] -= S.p[h * H + i][h * H + q] * x[q];
        // Orders the reads: scheduled freely, all 120 would be held in registers.
        if (q % 2) __asm__ volatile("" ::: "memory");
      }
    }
  }

  // Products with an inverted triangle and with whole rows of L multiply every
  // row of a column with every other: they make NaN of rows that an infinity, a
  // NaN or a column without a candidate (which eliminates nothing,
  // getrf.rs:72-73) does not reach.  Where there is one, the elimination goes by
  // substitution, a column of L after the other.  Looking for them costs 1 - 2 %
  // (5000 systems of n = 8 .. 256: FP64 2.06 against 2.08 ms, FP32 1.25 against
  // 1.27).  The right panel, in LDS, a row per thread:
  __device__ __forceinline__ void right_panel_any(int rows) {
#pragma clang fp contract(off)
#pragma unroll 1
    for (int j = 0; j < H; ++j) {
      if (!(none >> j & 1u) && t > j && t < rows) {
        const T l = S.p[t][j];
#pragma unroll 1
        for (int c = H; c < W; ++c) {
          const T e = l * S.p[j][c];
          S.p[t][c] = S.p[t][c] - e;
        }
      }
      lds_sync();
    }
  }
  // A chunk (see chunk), in memory, four rows at a time, without the columns of
  // L in `skip` (right-hand sides take L as it is stored, getrs.rs:25-29).
  // (Rolled: it shares the registers of the loop that it stands in.)
  __device__ __forceinline__ void chunk_any(const BatchBuf<T> &q, uint32_t ld, uint32_t col, int kb, int w,
                                            unsigned skip) {
#pragma clang fp contract(off)
    const int rows = n - kb, cnt = S.cnt;
    const uint32_t base = kb * ld + col;
    T u[W / 4], val[W / 4];
#pragma unroll
    for (int e = 0; e < W / 4; ++e) {
      u[e] = q.load(base + S.src[4 * e + g] * ld);
      val[e] = q.load(base + S.from[max(min(4 * e + g, cnt - 1), 0)] * ld);
    }
#pragma unroll
    for (int e = 0; e < W / 4; ++e) {
      q.store(base + (4 * e + g) * ld, u[e]);
      if (4 * e + g < cnt) q.store(base + S.rows[4 * e + g] * ld, val[e]);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    // Rows of the block: column k of L11 after the others.
#pragma unroll 1
    for (int k = 0; k + 1 < w; ++k) {
      if (!(skip >> k & 1u)) {
        const T uk = q.load(base + k * ld);
#pragma unroll 1
        for (int i = k + 1 + g; i < w; i += 4) {
          const T e = S.p[i][k] * uk;
          q.store(base + i * ld, q.load(base + i * ld) - e);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
      }
    }
    // Rows below.
#pragma unroll 1
    for (int i = W + g; i < rows; i += 4) {
      T x = q.load(base + i * ld);
#pragma unroll 1
      for (int k0 = 0; k0 < W; k0 += 8) {
        T uk[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) uk[k] = q.load(base + (k0 + k) * ld);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const T e = S.p[i][k0 + k] * uk[k];
          x = skip >> (k0 + k) & 1u ? x : x - e;
        }
      }
      q.store(base + i * ld, x);
    }
  }

  // The left panel's elimination applied to the right panel, in LDS.
  __device__ __forceinline__ void right_panel(int rows) {
    v4 u;
#pragma unroll
    for (int e = 0; e < 4; ++e) u[e] = S.p[M::row(g, e)][H + lc];
    u = prod(&S.inv[0][lc][0], u);
    // (The same in every wave.)
    const bool odd = none != 0 || !__all(zero_if_finite(u) == T(0));
    lds_sync();
    if (__builtin_expect(odd, 0)) {
      right_panel_any(rows);
      return;
    }
    if (wave == 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) S.p[M::row(g, e)][H + lc] = u[e];
    }
    for (int i0 = H + 16 * wave; i0 < rows; i0 += 16 * NW) {
      const v4 c = prod(&S.p[i0 + lc][0], u);
#pragma unroll
      for (int e = 0; e < 4; ++e) S.p[i0 + M::row(g, e)][H + lc] -= c[e];
    }
    lds_sync();
  }

  // The columns right of the block and those of B, 16 per wave at a time.
  __device__ __forceinline__ void update(int kb, int w) {
    const int c0 = kb + w, na = (n - c0 + 15) / 16;  // chunks of A, then one of B
    for (int ch = wave; ch <= na; ch += NW) {
      const int c = ch < na ? c0 + 16 * ch + lc : lc, ld = ch < na ? n : r;
      const uint32_t col = c < ld ? c : A.kNone / 2;
      if (!chunk(ch < na ? A : B, ld, col, kb, w)) chunk_any(ch < na ? A : B, ld, col, kb, w, ch < na ? none : 0);
    }
  }

  // One chunk: lane column `col` of the row-major q with rows of ld.  False,
  // and nothing done, where it is for chunk_any.
  __device__ __forceinline__ bool chunk(const BatchBuf<T> &q, uint32_t ld, uint32_t col, int kb, int w) {
    const int rows = n - kb, cnt = S.cnt;
    const uint32_t base = kb * ld + col, lrow0 = base + M::row(g, 0) * ld;
    constexpr int RS = M::kStep;
    v4 u0, u1, cur[4];
    // Groups of four 16-row tiles below the block, the next group's loads in
    // flight during this one's products.
    auto load = [&](int i0, v4 (&x)[4]) {
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) x[b][e] = q.load(lrow0 + (i0 + 16 * b + RS * e) * ld);
    };
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      u0[e] = q.load(base + S.src[M::row(g, e)] * ld);
      u1[e] = q.load(base + S.src[M::row(g, e) + H] * ld);
    }
    // Rows below the block that receive another row.
    T val[W / 4];
    if (cnt) {
#pragma unroll
      for (int e = 0; e < W / 4; ++e) val[e] = q.load(base + S.from[min(4 * e + g, cnt - 1)] * ld);
    } else if (rows > W) {
      load(W, cur);
    }
    // Where it is for chunk_any every store goes past the end (a branch here
    // cost the registers of the loop below).
    const bool odd = none != 0 || !__all(zero_if_finite(u0) + zero_if_finite(u1) == T(0));
    const uint32_t off = odd ? q.kNone / 2 : 0;
    const uint32_t srow0 = lrow0 + off;
    if (cnt) {
#pragma unroll
      for (int e = 0; e < W / 4; ++e)
        if (4 * e + g < cnt) q.store(base + off + S.rows[4 * e + g] * ld, val[e]);
      // The tiles below are read with another lane layout.
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
      if (rows > W) load(W, cur);
    }
    u0 = prod(&S.inv[0][lc][0], u0);
    if (w > H) {
      u1 -= prod(&S.p[H + lc][0], u0);
      u1 = prod(&S.inv[1][lc][0], u1);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      q.store(srow0 + RS * e * ld, u0[e]);
      if (w > H) q.store(srow0 + (H + RS * e) * ld, u1[e]);
    }
    for (int i0 = W; i0 < rows; i0 += 64) {
      v4 nxt[4];
      if (i0 + 64 < rows) load(i0 + 64, nxt);
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        if (i0 + 16 * b < rows) {
          const T *lrow = &S.p[i0 + 16 * b + lc][0];
          cur[b] -= prod(lrow, u0) + prod(lrow + H, u1);
#pragma unroll
          for (int e = 0; e < 4; ++e) q.store(srow0 + (i0 + 16 * b + RS * e) * ld, cur[b][e]);
        }
      }
#pragma unroll
      for (int b = 0; b < 4; ++b) cur[b] = nxt[b];
    }
    return !odd;
  }

  __device__ __forceinline__ void factor() {
    constexpr int RP = NT / W;  // rows per pass over a block
    const int tr = t / W, tc = t % W;
    for (int kb = 0, blk = 0; kb < n; kb += W, ++blk) {
      const int w = min(W, n - kb), rows = n - kb;
      const uint32_t at = tc < w ? (kb + tr) * n + kb + tc : A.kNone / 2;
      // The block to LDS with coalesced reads, then half a row per thread.
      {
        T x[W];
#pragma unroll
        for (int e = 0; e < W; ++e) x[e] = A.load(at + RP * e * n);
#pragma unroll
        for (int e = 0; e < W; ++e) S.p[tr + RP * e][tc] = x[e];
      }
      if (t == 0) S.cnt = 0;
      none = 0;
      lds_sync();
      int org = t;
      for (int half = 0;; ++half) {
        T v[H];
        int pos = t;
        get(v, &S.p[t][half * H]);
        panel(v, pos, kb, half * H, w);
        none = (unsigned)__builtin_amdgcn_readfirstlane((int)none);
        place(v, pos, half, org);
        if (wave == 0) invert(half);
        if (half == 1 || w <= H) break;
        lds_sync();
        right_panel(rows);
      }
      const bool has = t < rows;
      const int o = has ? S.orig[kb + org] : 0;
#pragma unroll
      for (int e = 0; e < W; ++e) A.store(at + RP * e * n, S.p[tr + RP * e][tc]);
      lds_sync();
      if (none != 0) sing = kb + 31 - __builtin_clz(none);
      if (has) {
        S.orig[kb + t] = (unsigned char)o;
        S.hist[blk][o] = (unsigned char)(kb + t);
        if (org != t) {
          S.moved = 1;
          if (t >= W) {
            const int e = atomicAdd(&S.cnt, 1);
            S.rows[e] = (unsigned char)t;
            S.from[e] = (unsigned char)org;
          }
        }
      }
      lds_sync();
      update(kb, w);
      __syncthreads();
    }
  }

  // The interchanges of later blocks on the columns of L: after all of them
  // position i holds matrix row orig[i], which block blk left at
  // hist[blk][orig[i]].
  __device__ __forceinline__ void permute_left() {
    if (!S.moved) return;
    constexpr int RP = NT / W;
    const int tr = t / W, tc = t % W;
    for (int kb = 0, blk = 0; kb + W < n; kb += W, ++blk) {
      const int i0 = kb + W + tr;
      T x[W];
#pragma unroll
      for (int e = 0; e < W; ++e) x[e] = A.load(S.hist[blk][S.orig[min(i0 + RP * e, n - 1)]] * n + kb + tc);
      __syncthreads();  // every row is read
#pragma unroll
      for (int e = 0; e < W; ++e) A.store((i0 + RP * e) * n + kb + tc, x[e]);
    }
  }

  // One diagonal block of the back substitution: lane lc of each row of 16
  // lanes holds row lc of the block (u, its diagonal d) and of one right-hand
  // side (x); returns that row of the solution.  The quotient comes from the
  // reciprocal rd and one correction by its remainder, which gives the rounded
  // quotient itself while d, x and the quotient are clear of the subnormal range,
  // and about one unit in the last place (of the subnormals, there) otherwise.
  // The caller looks at the range of d and at the results.
  template <int I = H - 1>
  __device__ __forceinline__ void tri(const T (&u)[H], T d, T rd, int w, T x, T &out) const {
    if (__builtin_expect(I < w, 1)) {
      T q = x * rd;
      q = __builtin_elementwise_fma(__builtin_elementwise_fma(-q, d, x), rd, q);
      out = lc == I ? q : out;
      x -= u[I] * row_lane<I>(q);
    }
    if constexpr (I > 0) tri<I - 1>(u, d, rd, w, x, out);
  }
  // The same with the division itself, for any d and x (rolled: rarely taken).
  __device__ __noinline__ static T tri_any(BatchBuf<T> a, int n, int kb, int w, T d, T x) {
    const int l = threadIdx.x & 15;
    T out = T(0);
    for (int i = w - 1; i >= 0; --i) {
      const T q = x / d;
      out = l == i ? q : out;
      x -= a.load((kb + l) * n + kb + i) * __shfl(q, i, 16);
    }
    return out;
  }

  // Back substitution U X = Y (getrs.rs:30-36, true division), Y in LDS from
  // start to end, blocks of 16 rows from the bottom: 16 lanes per right-hand
  // side solve the diagonal block, then one thread per row above subtracts
  // the block's contribution.  The next block's rows of U are loaded while
  // the current block is solved.
  __device__ __forceinline__ void back() {
    T *sY = &S.p[0][0];  // [r][YP]: Y, then X
    for (int e = t; e < n * r; e += NT) sY[e % r * YP + e / r] = B.load(e);
    const bool solver = 4 * wave < r;
    const T lo = sizeof(T) == 8 ? T(0x1p-1000) : T(0x1p-100f), hi = sizeof(T) == 8 ? T(0x1p1000) : T(0x1p100f);
    auto load = [&](int kb, T &d, T (&ud)[H], T (&u)[H]) {
      const uint32_t row = (kb + lc) * n + kb, up = t < kb ? t * n + kb : A.kNone / 2;
      d = A.load(row + lc);
#pragma unroll
      for (int q = 0; q < H; ++q) ud[q] = A.load(row + q);
#pragma unroll
      for (int q = 0; q < H; ++q) u[q] = A.load(up + q);
    };
    T d, ud[H], u[H];
    int kb = (n - 1) / H * H;
    load(kb, d, ud, u);
    lds_sync();
    for (; kb >= 0; kb -= H) {
      const int w = min(H, n - kb);
      if (solver) {
        d = lc < w ? d : T(1);
        const T rd = T(1) / d;
        const T m = d < T(0) ? -d : d;
        const bool fast = __all(m >= lo && m <= hi);
        for (int c0 = 4 * wave; c0 < r; c0 += 4 * NW) {
          const int c = min(c0 + g, r - 1);
          const T x = sY[c * YP + kb + min(lc, w - 1)];
          T out = T(0);
          if (__builtin_expect(fast, 1)) tri(ud, d, rd, w, x, out);
          // (x infinite, or a quotient out of range: the remainder is NaN.)
          if (__builtin_expect(!fast || !__all(out - out == T(0)), 0)) out = tri_any(A, n, kb, w, d, x);
          if (c0 + g < r && lc < w) sY[c * YP + kb + lc] = out;
        }
      }
      T uc[H];
#pragma unroll
      for (int q = 0; q < H; ++q) uc[q] = u[q];
      if (kb > 0) load(kb - H, d, ud, u);
      lds_sync();
      if (t < kb) {
        for (int c = 0; c < r; ++c) {
          T x[H], acc[4] = {};
          get(x, sY + c * YP + kb);
#pragma unroll
          for (int q = 0; q < H; ++q)
            if (__builtin_expect(q < w, 1)) acc[q % 4] += uc[q] * x[q];
          sY[c * YP + t] -= (acc[0] + acc[1]) + (acc[2] + acc[3]);
        }
      }
      lds_sync();
    }
    for (int e = t; e < n * r; e += NT) B.store(e, sY[e % r * YP + e / r]);
  }
};

template <typename T, int NW>
__global__ void __launch_bounds__(64 * NW, sizeof(T) == 8 ? 2 : 3) batched_gesv_kernel(BatchArgs<T> p) {
  typedef BatchSolver<T, NW> Solver;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int sys = p.order[blockIdx.x];
  Solver s(*reinterpret_cast<typename Solver::Lds *>(smem_raw), p.n[sys], p.nrhs[sys], p.a + p.a_off[sys],
           p.b + p.b_off[sys]);
  if (s.t == 0) s.S.moved = 0;
  s.S.orig[s.t] = (unsigned char)s.t;
  s.factor();
  int64_t *ipiv = p.ipiv + p.p_off[sys];
  if (s.t < s.n) ipiv[s.t] = s.S.piv[s.t];
  s.permute_left();
  s.back();
  if (s.t == 0) p.info[sys] = s.sing;
}

template <typename T, int NW>
static hipError_t batched_go(const BatchArgs<T> &p, unsigned grid, hipStream_t stream) {
  typedef typename BatchSolver<T, NW>::Lds Lds;
  static const hipError_t once = hipFuncSetAttribute(reinterpret_cast<const void *>(batched_gesv_kernel<T, NW>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, sizeof(Lds));
  if (once != hipSuccess) return once;
  batched_gesv_kernel<T, NW><<<grid, 64 * NW, sizeof(Lds), stream>>>(p);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_batched_gesv(const BatchLaunch &bl, T *a, T *b, int64_t *ipiv, int *info, hipStream_t stream) {
  BatchArgs<T> p;
  p.n = bl.n;
  p.nrhs = bl.nrhs;
  p.a_off = bl.a_off;
  p.b_off = bl.b_off;
  p.p_off = bl.p_off;
  p.order = bl.order;
  p.a = a;
  p.b = b;
  p.ipiv = ipiv;
  p.info = info;
  // The fewest waves that hold the rows: 4096 systems of n = 64 take 247 us
  // with one wave and 409 with two, of n = 112 926 us with two and 1304 with
  // four (more columns' chains run side by side).
  const unsigned grid = (unsigned)bl.count;
  if (bl.nmax <= 64) return batched_go<T, 1>(p, grid, stream);
  if (bl.nmax <= 128) return batched_go<T, 2>(p, grid, stream);
  return batched_go<T, 4>(p, grid, stream);
}

template hipError_t launch_batched_gesv<double>(const BatchLaunch &, double *, double *, int64_t *, int *,
                                                hipStream_t);
template hipError_t launch_batched_gesv<float>(const BatchLaunch &, float *, float *, int64_t *, int *, hipStream_t);

}  // namespace lair
