// Row interchanges as gathers, blocked triangular solves and the dataflow
// triangular solve used by getrs.
//
//  * rowmap + rowgather: the interchanges ipiv[k0..k1) applied in forward
//    order (src/lapack/laswp.rs:21-39) compose to a permutation of at most
//    2*(k1-k0) rows; one wave composes it, then every column stripe moves the
//    affected rows in one read-all/write-all pass.  The same map updates the
//    running row permutation perm (perm[i] = original row now at row i,
//    src/decomposition/lu.rs:28-39).
//  * trsm_llu: B := L^-1 B for a unit lower L (src/blas/trsm.rs:6-22) with the
//    B stripe in LDS, 16-row diagonal sub-blocks solved per column and the rows
//    below updated in parallel.
//  * trtri_diag: inverses of the diagonal blocks of L (unit) and U.
//  * trsv_dataflow: block-row workgroups that wait for the solved values of
//    the blocks they depend on; those values are published as tagged 64-bit
//    words (tag = the solve's epoch), so a reader that sees its epoch in a
//    word also has the value, with no flags and no fences.  Tiles are fetched
//    before waiting, so the sequential chain only carries one round trip, one
//    tile product and one diagonal-inverse product per block (the
//    substitutions of src/lapack/getrs.rs:24-36, blocked).
#include <algorithm>
#include <climits>

#include "device_util.h"
#include "lair_internal.h"

namespace lair {

template <typename T>
__device__ __forceinline__ void st_sc1(T *p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ T ld_sc1(const T *p) {
  return __hip_atomic_load(const_cast<T *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}


// Allows a kernel to use up to the full 160 KB of LDS per workgroup.
// The attribute call's status is consumed here so that it cannot surface as
// the error of a later launch.
template <typename F>
static void allow_large_lds(F *kernel) {
  (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  (void)hipGetLastError();
}

// ------------------------------------------------------------- rowmap ---

// rows[e] <- contents of src[e] (before the interchanges), e < *count, for
// the interchanges ipiv[k0 .. k1) applied in order (k swaps with ipiv[k]).
// The rows involved are the block's rows k0 .. k1 - 1 and the distinct pivot
// rows outside it.  Each thread takes one such row r and finds its source by
// tracing r back through the interchanges, last to first (a swap of k and p
// maps k to p and p to k), so the rows are resolved independently of each
// other.
__global__ void __launch_bounds__(256)
    rowmap_kernel(const int64_t *ipiv, int k0, int k1, int *rows, int *src, int *count) {
  __shared__ int s_piv[kMaxSwapRows / 2], s_out[kMaxSwapRows / 2];
  __shared__ int s_wcnt[4];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int kb = k1 - k0;
  for (int e = t; e < kb; e += 256) s_piv[e] = (int)ipiv[k0 + e];
  __syncthreads();
  // Pivot rows outside the block, each listed once (first occurrence).
  int p = 0;
  bool first = false;
  if (t < kb) {
    p = s_piv[t];
    first = p < k0 || p >= k1;
    for (int e = 0; e < t && first; ++e) first = s_piv[e] != p;
  }
  const unsigned long long m = __ballot(first);
  if (lane == 0) s_wcnt[wv] = __popcll(m);
  __syncthreads();
  int base = 0;
  for (int w = 0; w < wv; ++w) base += s_wcnt[w];
  if (first) s_out[base + __popcll(m & ((1ull << lane) - 1))] = p;
  const int nout = s_wcnt[0] + s_wcnt[1] + s_wcnt[2] + s_wcnt[3];
  __syncthreads();
  const int total = kb + nout;
  for (int idx = t; idx < total; idx += 256) {
    const int r = idx < kb ? k0 + idx : s_out[idx - kb];
    int x = r;
#pragma unroll 8
    for (int e = kb - 1; e >= 0; --e) {
      const int pe = s_piv[e], ke = k0 + e;
      x = x == ke ? pe : (x == pe ? ke : x);
    }
    rows[idx] = r;
    src[idx] = x;
  }
  if (t == 0) *count = total;
}

// Columns [c0, c0+n1) and [s1, s1 + total-n1): 32 per workgroup.
template <typename T>
__global__ void __launch_bounds__(256)
    rowgather_kernel(T *a, int64_t lda, const int *rows, const int *src, const int *count, int c0,
                     int n1, int s1, int total) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *buf = reinterpret_cast<T *>(smem_raw);  // [nr][32]
  const int t = threadIdx.x, cl = t & 31, rg = t >> 5;
  const int i = blockIdx.x * 32 + cl;
  const bool act = i < total;
  const int c = act ? ((i < n1) ? c0 + i : s1 + (i - n1)) : 0;
  const int nr = *count;
  // Batches of 8 independent loads per thread.
  for (int e0 = rg; e0 < nr; e0 += 64) {
    T v[8];
    int sr[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int e = e0 + 8 * q;
      sr[q] = e < nr ? src[e] : -1;
      const bool mv = sr[q] >= 0 && sr[q] != rows[e];
      v[q] = (act && mv) ? a[(int64_t)sr[q] * lda + c] : T(0);
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int e = e0 + 8 * q;
      if (e < nr) buf[e * 32 + cl] = v[q];
    }
  }
  __syncthreads();
  for (int e = rg; e < nr; e += 8) {
    const int s = src[e];
    if (act && s != rows[e]) a[(int64_t)rows[e] * lda + c] = buf[e * 32 + cl];
  }
}

__global__ void __launch_bounds__(256)
    permgather_kernel(int *perm, const int *rows, const int *src, const int *count) {
  __shared__ int tmp[kMaxSwapRows];
  const int nr = *count;
  // Entries with rows[e] == src[e] do nothing (and may share their row with
  // an entry that moves one).
  for (int e = threadIdx.x; e < nr; e += 256)
    if (src[e] != rows[e]) tmp[e] = perm[src[e]];
  __syncthreads();
  for (int e = threadIdx.x; e < nr; e += 256)
    if (src[e] != rows[e]) perm[rows[e]] = tmp[e];
}

// The gather of a prepared row map over columns [c0, c1) minus [s0, s1).
template <typename T>
static hipError_t rowgather(lair_context *ctx, T *a, int64_t lda, int c0, int c1, int s0, int s1,
                            const int *rows, const int *src, const int *count, int nmax, int *perm) {
  if (s0 < c0) s0 = c0;
  if (s1 > c1) s1 = c1;
  if (s1 < s0) s1 = s0;
  const int n1 = s0 - c0;
  const int total = n1 + (c1 - s1);
  if (total > 0) {
    const size_t shm = (size_t)nmax * 32 * sizeof(T);
    if (shm > 160 * 1024) return hipErrorInvalidValue;
    static bool once = (allow_large_lds(rowgather_kernel<T>), true);
    (void)once;
    rowgather_kernel<T><<<(total + 31) / 32, 256, shm, ctx->stream>>>(a, lda, rows, src, count, c0, n1, s1,
                                                                       total);
  }
  if (perm) permgather_kernel<<<1, 256, 0, ctx->stream>>>(perm, rows, src, count);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_rowswap(lair_context *ctx, T *a, int64_t lda, int c0, int c1, int s0, int s1,
                          const int64_t *ipiv, int k0, int k1, int *perm) {
  if (k1 <= k0) return hipSuccess;
  if (k1 - k0 > kMaxSwapRows / 2) return hipErrorInvalidValue;
  const int slot = prof_begin(ctx, LAIR_KCLASS_LASWP);
  rowmap_kernel<<<1, 256, 0, ctx->stream>>>(ipiv, k0, k1, ctx->swap_rows, ctx->swap_src,
                                           ctx->swap_count);
  hipError_t e = rowgather<T>(ctx, a, lda, c0, c1, s0, s1, ctx->swap_rows, ctx->swap_src, ctx->swap_count,
                              2 * (k1 - k0), perm);
  prof_end(ctx, slot, LAIR_KCLASS_LASWP, 0.0, 4.0 * sizeof(T) * (double)(k1 - k0) * (c1 - c0));
  return e;
}

template <typename T>
hipError_t launch_rowswap_map(lair_context *ctx, T *a, int64_t lda, int c0, int c1, int s0, int s1,
                              const int *rows, const int *src, const int *count, int nmax, int *perm) {
  if (nmax <= 0) return hipSuccess;
  if (nmax > kMaxSwapRows) return hipErrorInvalidValue;
  const int slot = prof_begin(ctx, LAIR_KCLASS_LASWP);
  hipError_t e = rowgather<T>(ctx, a, lda, c0, c1, s0, s1, rows, src, count, nmax, perm);
  prof_end(ctx, slot, LAIR_KCLASS_LASWP, 0.0, 2.0 * sizeof(T) * (double)nmax * (c1 - c0));
  return e;
}

template hipError_t launch_rowswap_map<double>(lair_context *, double *, int64_t, int, int, int, int,
                                               const int *, const int *, const int *, int, int *);
template hipError_t launch_rowswap_map<float>(lair_context *, float *, int64_t, int, int, int, int,
                                              const int *, const int *, const int *, int, int *);
template hipError_t launch_rowswap_map<zcplx>(lair_context *, zcplx *, int64_t, int, int, int, int,
                                              const int *, const int *, const int *, int, int *);
template hipError_t launch_rowswap_map<ccplx>(lair_context *, ccplx *, int64_t, int, int, int, int,
                                              const int *, const int *, const int *, int, int *);

template hipError_t launch_rowswap<double>(lair_context *, double *, int64_t, int, int, int, int,
                                           const int64_t *, int, int, int *);
template hipError_t launch_rowswap<float>(lair_context *, float *, int64_t, int, int, int, int,
                                          const int64_t *, int, int, int *);
template hipError_t launch_rowswap<zcplx>(lair_context *, zcplx *, int64_t, int, int, int, int,
                                          const int64_t *, int, int, int *);
template hipError_t launch_rowswap<ccplx>(lair_context *, ccplx *, int64_t, int, int, int, int,
                                          const int64_t *, int, int, int *);

// perm from the full pivot vector (for factors supplied by the caller).
// Every thread traces kPermRows positions back through the interchanges, last
// to first (a swap of k and p maps k to p and p to k), so the positions are
// resolved independently; the pivots pass through LDS kPermChunk at a time.
// Bound by the trace, 32 ns per pivot whatever the number of positions (one
// wave per SIMD up to n = 131072 on 256 CUs): 64 us at n=1999, 18 us at n=512,
// against 203 and 53 us for one thread applying the interchanges in order.  A pivot
// outside [0, n) (compared as the full int64) is skipped rather than followed
// out of bounds and reported through the status word (kErrPivot).
constexpr int kPermRows = 2;
constexpr int kPermChunk = 4096;
__global__ void __launch_bounds__(256) perm_from_ipiv_kernel(const int64_t *ipiv, int n, int *perm,
                                                             int32_t *status) {
  __shared__ __align__(16) int s_piv[kPermChunk];
  const int t = threadIdx.x, i0 = blockIdx.x * 256 * kPermRows + t;
  int x[kPermRows];
#pragma unroll
  for (int r = 0; r < kPermRows; ++r) x[r] = i0 + 256 * r;
  for (int c0 = (n - 1) / kPermChunk * kPermChunk; c0 >= 0; c0 -= kPermChunk) {
    __syncthreads();
    const int cn = min(kPermChunk, (n - c0 + 7) & ~7);
    for (int e = t; e < cn; e += 256) {
      const int k = c0 + e;
      const int64_t p = k < n ? ipiv[k] : k;
      const bool ok = k >= n || (p >= 0 && p < n);
      if (!ok && blockIdx.x == 0) atomic_or_agent(status, kErrPivot);
      s_piv[e] = ok ? (int)p : k;  // k: no interchange
    }
    __syncthreads();
    for (int e = cn - 8; e >= 0; e -= 8) {
      int p[8];
      __builtin_memcpy(p, __builtin_assume_aligned(s_piv + e, 16), sizeof p);
#pragma unroll
      for (int q = 7; q >= 0; --q) {
        const int k = c0 + e + q;
#pragma unroll
        for (int r = 0; r < kPermRows; ++r) {
          const int y = x[r] == p[q] ? k : x[r];
          x[r] = x[r] == k ? p[q] : y;
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < kPermRows; ++r)
    if (i0 + 256 * r < n) perm[i0 + 256 * r] = x[r];
}

hipError_t launch_perm_from_ipiv(lair_context *ctx, const int64_t *ipiv, int n, int *perm) {
  if (n <= 0) return hipSuccess;
  perm_from_ipiv_kernel<<<(n + 256 * kPermRows - 1) / (256 * kPermRows), 256, 0, ctx->stream>>>(ipiv, n, perm,
                                                                                              ctx->err);
  return hipGetLastError();
}

__global__ void iota_kernel(int *p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = i;
}

hipError_t launch_iota(lair_context *ctx, int *p, int n) {
  if (n <= 0) return hipSuccess;
  iota_kernel<<<(n + 255) / 256, 256, 0, ctx->stream>>>(p, n);
  return hipGetLastError();
}

// y[i][q] = (D) x[perm[i]][q]  (gather) or y[perm[i]][q] = (D) x[i][q] (scatter);
// a null perm copies.
template <typename S, typename D>
__global__ void permute_rows_kernel(int rows, int cols, const int *perm, const S *x, int64_t ldx,
                                    D *y, int64_t ldy, int scatter, unsigned long long *zero, int nz) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (zero && idx < nz) zero[idx] = 0ull;
  if (idx >= (int64_t)rows * cols) return;
  const int i = (int)(idx / cols), q = (int)(idx % cols);
  const int pi = perm ? perm[i] : i;
  if (!scatter)
    y[(int64_t)i * ldy + q] = (D)x[(int64_t)pi * ldx + q];
  else
    y[(int64_t)pi * ldy + q] = (D)x[(int64_t)i * ldx + q];
}

template <typename S, typename D>
hipError_t launch_permute_rows(lair_context *ctx, int rows, int cols, const int *perm, const S *x,
                               int64_t ldx, D *y, int64_t ldy, bool scatter, unsigned long long *zero,
                               int nz) {
  const int64_t total = std::max<int64_t>((int64_t)rows * cols, zero ? nz : 0);
  if (total <= 0) return hipSuccess;
  permute_rows_kernel<S, D><<<(unsigned)((total + 255) / 256), 256, 0, ctx->stream>>>(
      rows, cols, perm, x, ldx, y, ldy, scatter ? 1 : 0, zero, nz);
  return hipGetLastError();
}

template hipError_t launch_permute_rows<double, double>(lair_context *, int, int, const int *,
                                                        const double *, int64_t, double *, int64_t,
                                                        bool, unsigned long long *, int);
template hipError_t launch_permute_rows<double, float>(lair_context *, int, int, const int *,
                                                       const double *, int64_t, float *, int64_t,
                                                       bool, unsigned long long *, int);
template hipError_t launch_permute_rows<float, float>(lair_context *, int, int, const int *,
                                                      const float *, int64_t, float *, int64_t,
                                                      bool, unsigned long long *, int);

// ------------------------------------------------------------ trsm_llu ---

template <typename T>
__global__ void __launch_bounds__(256)
    trsm_llu_kernel(int kb, int ncols, const T *__restrict__ L, int64_t ldl, T *__restrict__ B,
                    int64_t ldb) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *xs = reinterpret_cast<T *>(smem_raw);  // [kb][64]
  const int t = threadIdx.x, col = t & 63, rg = t >> 6;
  const int c = blockIdx.x * 64 + col;
  const bool act = c < ncols;
  for (int i = rg; i < kb; i += 4) xs[i * 64 + col] = act ? B[(int64_t)i * ldb + c] : T(0);
  __syncthreads();
  for (int s0 = 0; s0 < kb; s0 += 16) {
    const int sb = kb - s0 < 16 ? kb - s0 : 16;
    if (rg == 0) {
      for (int i = 1; i < sb; ++i) {
        T acc = xs[(s0 + i) * 64 + col];
        const T *lr = L + (int64_t)(s0 + i) * ldl + s0;
        for (int p = 0; p < i; ++p) acc -= lr[p] * xs[(s0 + p) * 64 + col];
        xs[(s0 + i) * 64 + col] = acc;
      }
    }
    __syncthreads();
    for (int r = s0 + sb + rg; r < kb; r += 4) {
      T acc = xs[r * 64 + col];
      const T *lr = L + (int64_t)r * ldl + s0;
#pragma unroll 4
      for (int p = 0; p < sb; ++p) acc -= lr[p] * xs[(s0 + p) * 64 + col];
      xs[r * 64 + col] = acc;
    }
    __syncthreads();
  }
  if (act)
    for (int i = rg; i < kb; i += 4) B[(int64_t)i * ldb + c] = xs[i * 64 + col];
}

// B := L^-1 B for kb <= 128 with 16 columns of B per workgroup, so that a
// 128-column strip (the next panel's columns) spreads over 8 workgroups and a
// wide strip over many.  L (strictly lower part) and the workgroup's columns
// are staged in LDS.  Diagonal 16-row blocks are solved with one thread per
// column; the rows below each block are then updated by all threads.  Every
// element receives its subtractions b -= b[k] * L[i][k] one at a time in
// increasing k (src/blas/trsm.rs:13-21 applies them in the same order).

template <typename T>
__global__ void __launch_bounds__(256)
    trsm_llu16_kernel(int kb, int ncols, const T *__restrict__ L, int64_t ldl, T *__restrict__ B,
                      int64_t ldb) {
#pragma clang fp contract(off)
  constexpr int CW = kTrsmCW, LX = CW + 1;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int LL = kb + 1;
  T *sL = reinterpret_cast<T *>(smem_raw);  // [kb][kb + 1]
  T *sX = sL + (size_t)kb * LL;             // [kb][CW + 1]
  const int t = threadIdx.x;
  const int c0 = blockIdx.x * CW;
  const int nc = ncols - c0 < CW ? ncols - c0 : CW;
  for (int e = t; e < kb * kb; e += 256) {
    const int r = e / kb, c = e % kb;
    if (c < r) sL[r * LL + c] = L[(int64_t)r * ldl + c];
  }
  for (int e = t; e < kb * CW; e += 256) {
    const int r = e / CW, c = e % CW;
    sX[r * LX + c] = c < nc ? B[(int64_t)r * ldb + c0 + c] : T(0);
  }
  __syncthreads();
  for (int b0 = 0; b0 < kb; b0 += 16) {
    const int bs = kb - b0 < 16 ? kb - b0 : 16;
    if (t < CW) {
      for (int i = 1; i < bs; ++i) {
        T acc = sX[(b0 + i) * LX + t];
        for (int p = 0; p < i; ++p) {
          const T e = sX[(b0 + p) * LX + t] * sL[(b0 + i) * LL + b0 + p];
          acc = acc - e;
        }
        sX[(b0 + i) * LX + t] = acc;
      }
    }
    __syncthreads();
    const int rows = kb - b0 - bs;
    for (int e = t; e < rows * CW; e += 256) {
      const int r = b0 + bs + e / CW, c = e % CW;
      T acc = sX[r * LX + c];
      for (int p = 0; p < bs; ++p) {
        const T pr = sX[(b0 + p) * LX + c] * sL[r * LL + b0 + p];
        acc = acc - pr;
      }
      sX[r * LX + c] = acc;
    }
    __syncthreads();
  }
  for (int e = t; e < kb * CW; e += 256) {
    const int r = e / CW, c = e % CW;
    if (c < nc) B[(int64_t)r * ldb + c0 + c] = sX[r * LX + c];
  }
}

// Barrier for data in LDS only: unlike __syncthreads it does not wait for
// global loads in flight.
__device__ __forceinline__ void lds_barrier() {
  __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  __asm__ volatile("" ::: "memory");
}

// Steps I .. 14 of a 16-row unit lower solve, a row per lane of a row of 16.
template <int I, typename T>
__device__ __forceinline__ void diag_steps(T &x, const T (&lrow)[15], int rr) {
#pragma clang fp contract(off)
  const T e = row_bcast<I>(x) * lrow[I];
  if (I < rr) x = x - e;
  if constexpr (I < 14) diag_steps<I + 1>(x, lrow, rr);
}

// Interchanges then U12 = L11^-1 A12 for columns [c0, c1) of a panel
// [k, k + kb) (kb <= 128): the laswp + trsm steps of recursive_inner
// (src/lapack/getrf.rs:270-278) fused per 16-column strip.  The strip's rows
// named by the row map (rows[e] receives the old contents of src[e]; the
// first kb entries are rows k .. k + kb - 1 in order) are read once into LDS;
// the rows moved below the panel are written back at once, and the top kb
// rows are solved in LDS and written as U12.  Diagonal 16-row blocks are
// solved in registers, 16 lanes per column; the rows below each block are
// then updated by all threads.  Every element receives its subtractions
// b -= b[p] * L[i][p] one at a time in increasing p (src/blas/trsm.rs:13-21
// applies them in the same order).
// Bound by latencies, not bytes: two round trips of loads, then per 16 rows
// the diagonal solve's 15 broadcasts (DPP, 4 cycles; an LDS permute took 130)
// and the update.  Loads are clamped instead of masked (a mask costs a branch
// per load).  FP64, 64 rows: 10.9 us a call, before 14.4; FP32, 128 rows: 18.3,
// before 42.
template <typename T>
__global__ void __launch_bounds__(256)
    swap_trsm_kernel(T *__restrict__ a, int64_t lda, int k, int kb, int c0, int ncols,
                     const int *__restrict__ rows, const int *__restrict__ src,
                     const int *__restrict__ count, int nmax) {
#pragma clang fp contract(off)
  constexpr int CW = kTrsmCW, LX = CW + 1, RG = 256 / CW, LB = sizeof(T) > 8 ? 16 : 32;
  static_assert(CW == 16, "the diagonal solve maps 4 waves x 4 columns x 16 rows onto 256 threads");
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *sL = reinterpret_cast<T *>(smem_raw);             // strictly lower L11, row r at r(r-1)/2
  T *sX = sL + ((size_t)kb * (kb - 1) / 2 + 1);         // [nmax][CW + 1] map rows' old values
  int *s_rows = reinterpret_cast<int *>(sX + (size_t)nmax * LX);  // [nmax]
  int *s_src = s_rows + nmax;                            // [nmax]
  const int t = threadIdx.x;
  const int cs = c0 + blockIdx.x * CW;
  const int nc = c0 + ncols - cs < CW ? c0 + ncols - cs : CW;
  // The row map and the first rows of L11 are requested together; the strip's
  // rows follow as soon as the map is in LDS, while L11 still arrives.  L11
  // goes by 256 / lw rows of lw columns per load, LB loads at a time (its
  // strictly lower part is kept).
  const int nr = *count;
  const T *L = a + (int64_t)k * lda + k;
  const int lw = kb <= 64 ? 64 : 128, lp = t & (lw - 1), lr0 = t / lw, ls = 256 / lw;
  // (A vector stands for a 16-byte struct, whose arrays would go to scratch.)
  typedef double d2 __attribute__((ext_vector_type(2)));
  typedef std::conditional_t<sizeof(T) == 16, d2, T> raw_t;
  auto ld = [](const T *p) { return *reinterpret_cast<const raw_t *>(p); };
  auto st = [](T *p, raw_t v) { *reinterpret_cast<raw_t *>(p) = v; };
  auto lload = [&](int r0, raw_t (&v)[LB]) {
#pragma unroll
    for (int q = 0; q < LB; ++q) {
      // Clamped, not masked (a mask per load costs a branch).
      v[q] = ld(&L[(int64_t)min(r0 + lr0 + q * ls, kb - 1) * lda + min(lp, kb - 1)]);
    }
  };
  auto lstore = [&](int r0, const raw_t (&v)[LB]) {
#pragma unroll
    for (int q = 0; q < LB; ++q) {
      const int r = r0 + lr0 + q * ls;  // the spare element takes what is not kept
      st(&sL[(r < kb && lp < r) ? r * (r - 1) / 2 + lp : kb * (kb - 1) / 2], v[q]);
    }
  };
  for (int e = t; e < nr; e += 256) {
    s_rows[e] = rows[e];
    s_src[e] = src[e];
  }
  raw_t lv[LB];
  lload(0, lv);
  lds_barrier();
  const int c = t % CW, rg = t / CW;
  for (int eb = 0; eb < nr; eb += RG * 16) {
    const int e0 = eb + rg;
    raw_t v[16];
#pragma unroll
    for (int q = 0; q < 16; ++q)
      v[q] = ld(&a[(int64_t)s_src[min(e0 + q * RG, nr - 1)] * lda + cs + min(c, nc - 1)]);
    if (eb == 0) lstore(0, lv);
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int e = e0 + q * RG;
      if (e < nr) st(&sX[e * LX + c], v[q]);
    }
  }
  for (int r0 = LB * ls; r0 < kb; r0 += LB * ls) {
    lload(r0, lv);
    lstore(r0, lv);
  }
  __syncthreads();
  // Rows moved below the panel (entries kb.. that move something).
  for (int e = kb + rg; e < nr; e += RG)
    if (c < nc && s_rows[e] != s_src[e]) a[(int64_t)s_rows[e] * lda + cs + c] = sX[e * LX + c];
  for (int b0 = 0; b0 < kb; b0 += 16) {
    const int bs = kb - b0 < 16 ? kb - b0 : 16;
    {
      // Diagonal block: 16 lanes per column, lane rr holding row b0 + rr of
      // column cc.  At step i row i is final; it is broadcast to the column's
      // lanes and the rows below it subtract their term.
      const int l = t & 63;
      const int cc = (t >> 6) * 4 + (l >> 4), rr = l & 15;
      const int rc = min(b0 + rr, kb - 1);
      T x = sX[rc * LX + cc];
      T lrow[15];
#pragma unroll
      for (int i = 0; i < 15; ++i) lrow[i] = sL[rc * (rc - 1) / 2 + b0 + min(i, max(rr - 1, 0))];
      diag_steps<0>(x, lrow, rr);
      if (rr < bs) sX[(b0 + rr) * LX + cc] = x;
    }
    __syncthreads();
    T xb[16];
#pragma unroll
    for (int p = 0; p < 16; ++p) xb[p] = sX[(b0 + min(p, bs - 1)) * LX + c];
    // (Rows below a block exist only if it has 16.)
    for (int r = b0 + bs + rg; r < kb; r += RG) {
      const T *lr = sL + r * (r - 1) / 2 + b0;
      T acc = sX[r * LX + c];
#pragma unroll
      for (int p = 0; p < 16; ++p) {
        const T pr = xb[p] * lr[p];
        acc = acc - pr;
      }
      sX[r * LX + c] = acc;
    }
    __syncthreads();
  }
  for (int r = rg; r < kb; r += RG)
    if (c < nc) a[(int64_t)(k + r) * lda + cs + c] = sX[r * LX + c];
}

template <typename T>
hipError_t launch_swap_trsm(lair_context *ctx, T *a, int64_t lda, int k, int kb, int c0, int c1,
                            const int *rows, const int *src, const int *count, int nmax) {
  if (c1 <= c0 || kb <= 0) return hipSuccess;
  if (kb > kTrsmMaxKb || nmax > kMaxSwapRows || nmax < kb) return hipErrorInvalidValue;
  const size_t shm = sizeof(T) * ((size_t)kb * (kb - 1) / 2 + 1 + (size_t)nmax * (kTrsmCW + 1)) +
                     2 * sizeof(int) * (size_t)nmax + 16;
  if (shm > 160 * 1024) return hipErrorInvalidValue;
  static bool once = (allow_large_lds(swap_trsm_kernel<T>), true);
  (void)once;
  const int slot = prof_begin(ctx, LAIR_KCLASS_TRSM);
  swap_trsm_kernel<T><<<(c1 - c0 + kTrsmCW - 1) / kTrsmCW, 256, shm, ctx->stream>>>(a, lda, k, kb, c0, c1 - c0,
                                                                                      rows, src, count, nmax);
  prof_end(ctx, slot, LAIR_KCLASS_TRSM, (double)kb * kb * (c1 - c0),
           sizeof(T) * (2.0 * (kb + nmax) * (c1 - c0) + 0.5 * kb * kb));
  return hipGetLastError();
}

template hipError_t launch_swap_trsm<double>(lair_context *, double *, int64_t, int, int, int, int,
                                             const int *, const int *, const int *, int);
template hipError_t launch_swap_trsm<float>(lair_context *, float *, int64_t, int, int, int, int,
                                            const int *, const int *, const int *, int);
template hipError_t launch_swap_trsm<zcplx>(lair_context *, zcplx *, int64_t, int, int, int, int,
                                            const int *, const int *, const int *, int);
template hipError_t launch_swap_trsm<ccplx>(lair_context *, ccplx *, int64_t, int, int, int, int,
                                            const int *, const int *, const int *, int);

hipError_t launch_rowmap(lair_context *ctx, const int64_t *ipiv, int k0, int k1) {
  if (k1 <= k0) return hipSuccess;
  if (k1 - k0 > kMaxSwapRows / 2) return hipErrorInvalidValue;
  rowmap_kernel<<<1, 256, 0, ctx->stream>>>(ipiv, k0, k1, ctx->swap_rows, ctx->swap_src, ctx->swap_count);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_trsm_llu(lair_context *ctx, int kb, int ncols, const T *L, int64_t ldl, T *B,
                           int64_t ldb) {
  if (kb <= 0 || ncols <= 0) return hipSuccess;
  if (kb <= kTrsmMaxKb) {
    const size_t shm = sizeof(T) * ((size_t)kb * (kb + 1) + (size_t)kb * (kTrsmCW + 1));
    if (shm > 160 * 1024) return hipErrorInvalidValue;
    static bool once16 = (allow_large_lds(trsm_llu16_kernel<T>), true);
    (void)once16;
    const int slot = prof_begin(ctx, LAIR_KCLASS_TRSM);
    trsm_llu16_kernel<T><<<(ncols + kTrsmCW - 1) / kTrsmCW, 256, shm, ctx->stream>>>(kb, ncols, L, ldl, B,
                                                                                      ldb);
    prof_end(ctx, slot, LAIR_KCLASS_TRSM, (double)kb * kb * ncols,
             sizeof(T) * (2.0 * kb * ncols + 0.5 * kb * kb));
    return hipGetLastError();
  }
  const size_t shm = (size_t)kb * 64 * sizeof(T);
  if (shm > 160 * 1024) return hipErrorInvalidValue;
  static bool once = (allow_large_lds(trsm_llu_kernel<T>), true);
  (void)once;
  const int slot = prof_begin(ctx, LAIR_KCLASS_TRSM);
  trsm_llu_kernel<T><<<(ncols + 63) / 64, 256, shm, ctx->stream>>>(kb, ncols, L, ldl, B, ldb);
  prof_end(ctx, slot, LAIR_KCLASS_TRSM, (double)kb * kb * ncols,
           sizeof(T) * (2.0 * kb * ncols + 0.5 * kb * kb));
  return hipGetLastError();
}

template hipError_t launch_trsm_llu<double>(lair_context *, int, int, const double *, int64_t,
                                            double *, int64_t);
template hipError_t launch_trsm_llu<float>(lair_context *, int, int, const float *, int64_t, float *,
                                           int64_t);
template hipError_t launch_trsm_llu<zcplx>(lair_context *, int, int, const zcplx *, int64_t, zcplx *,
                                           int64_t);
template hipError_t launch_trsm_llu<ccplx>(lair_context *, int, int, const ccplx *, int64_t, ccplx *,
                                           int64_t);

// ---------------------------------------------------------- trtri_diag ---

// DPP quad permutation.
template <int CTRL, typename T>
__device__ __forceinline__ T quad_xor(T x) {
  if constexpr (sizeof(T) == 8)
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xF, 0xF, false),
                            __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xF, 0xF, false));
  else
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, false));
}

// blockIdx.x = diagonal block; blockIdx.y = 0: unit lower L -> linv,
// 1: upper U -> uinv.  Each inverse is stored dense BS x BS (row-major).
// Four lanes per column: each sums every fourth term of an entry's dot product
// (four at a time, their LDS loads issued together) and the quad adds its sums
// pairwise.  Bound by the chain of rows, a few LDS round trips each: 31 us in
// FP64 whatever n (one lane per column, 16 loads of the block in turn: 70 us).
template <typename T, int BS>
__global__ void __launch_bounds__(4 * BS)
    trtri_diag_kernel(const T *__restrict__ lu, int64_t lda, int n, T *__restrict__ linv,
                      T *__restrict__ uinv) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *M = reinterpret_cast<T *>(smem_raw);  // [BS][BS+1]
  T *X = M + BS * (BS + 1);                // [BS][BS+1]
  constexpr int LD = BS + 1, NT = 4 * BS, NL = BS * BS / NT;
  const int b = blockIdx.x, t = threadIdx.x, j = t >> 2, h = t & 3;
  const bool upper = blockIdx.y == 1;
  const int r0 = b * BS;
  const int nb = n - r0 < BS ? n - r0 : BS;
  {
    T v[NL];
#pragma unroll
    for (int q = 0; q < NL; ++q) {
      const int e = t + q * NT, r = e / BS, c = e % BS;
      v[q] = (r < nb && c < nb) ? lu[(int64_t)(r0 + r) * lda + r0 + c] : T(0);
    }
#pragma unroll
    for (int q = 0; q < NL; ++q) {
      const int e = t + q * NT, r = e / BS, c = e % BS;
      M[r * LD + c] = v[q];
      X[r * LD + c] = T(0);
    }
  }
  __syncthreads();
  // Sum over p in [p0, p1) of M[i][p] X[p][j].
  auto dot = [&](int i, int p0, int p1) -> T {
    T a = T(0);
    for (int p = p0 + h; p < p1; p += 16) {
      T m[4], x[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = p + 4 * q, kc = k < p1 ? k : p;
        m[q] = M[i * LD + kc];
        x[q] = X[kc * LD + j];
      }
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (p + 4 * q < p1) a += m[q] * x[q];
    }
    a += quad_xor<0xB1>(a);  // lanes 1, 0, 3, 2
    a += quad_xor<0x4E>(a);  // lanes 2, 3, 0, 1
    return a;
  };
  // Column j of the inverse by substitution (its four lanes are in one wave).
  if (j < nb) {
    if (!upper) {
      if (h == 0) X[j * LD + j] = T(1);
      for (int i = j + 1; i < nb; ++i) {
        __asm__ volatile("" ::: "memory");  // the quad's store comes before its loads
        const T d = dot(i, j, i);
        if (h == 0) X[i * LD + j] = -d;
      }
    } else {
      if (h == 0) X[j * LD + j] = T(1) / M[j * LD + j];
      for (int i = j - 1; i >= 0; --i) {
        __asm__ volatile("" ::: "memory");  // the quad's store comes before its loads
        const T d = -dot(i, i + 1, j + 1) / M[i * LD + i];
        if (h == 0) X[i * LD + j] = d;
      }
    }
  }
  __syncthreads();
  T *out = (upper ? uinv : linv) + (size_t)b * BS * BS;
  for (int e = t; e < BS * BS; e += NT) out[e] = X[(e / BS) * LD + e % BS];
}

template <typename T>
hipError_t launch_trtri_diag(lair_context *ctx, const T *lu, int64_t lda, int n, T *linv, T *uinv) {
  if (n <= 0) return hipSuccess;
  constexpr int BS = TrsvBlock<T>::BS;
  const int nblk = (n + BS - 1) / BS;
  const size_t shm = 2 * (size_t)BS * (BS + 1) * sizeof(T);
  static bool once = (allow_large_lds(trtri_diag_kernel<T, BS>), true);
  (void)once;
  const int slot = prof_begin(ctx, LAIR_KCLASS_GETRS);
  trtri_diag_kernel<T, BS><<<dim3(nblk, 2), 4 * BS, shm, ctx->stream>>>(lu, lda, n, linv, uinv);
  prof_end(ctx, slot, LAIR_KCLASS_GETRS, (double)nblk * BS * BS * BS / 3.0);
  return hipGetLastError();
}

template hipError_t launch_trtri_diag<double>(lair_context *, const double *, int64_t, int, double *,
                                              double *);
template hipError_t launch_trtri_diag<float>(lair_context *, const float *, int64_t, int, float *,
                                             float *);

// ------------------------------------------------------ trsv_dataflow ---

template <typename T>
struct TrsvArgs {
  const T *lu;
  int64_t lda;
  const T *dinv;  // inverses of the diagonal blocks used by this solve
  const T *xin;   // right-hand sides (may alias x)
  T *x;           // n x nrhs solution
  int64_t ldx;
  int n, nrhs, nblk, nchunks;
  unsigned long long *xt;  // [n][nrhs][words per element] tagged solved values
  uint32_t epoch;
  int forward, trans, dinv_trans;
  int32_t *err;
  int wait_limit;  // polls before a wait gives up (0: every wait gives up at once)
};

// The refinement step fused with the backward solve of the correction
// d = U^-1 y (FP32): the workgroup that solves block i of d also forms
// x_i + d_i in FP64, stores it and publishes it as tagged words (two per
// value, tag = the solve's epoch); residual workgroups stream the FP64 A by
// row blocks (48 rows for one right-hand side, else 24) and consume those
// values column block by column block in the order the solve finishes them,
// so the residual's pass over A overlaps the solve's chain.  The column maxima of |x + d| and |r| fold into
// xbits and rbits (ordered bit patterns, zero at launch).
struct IrFuse {
  double *x;
  int64_t ldx;
  int x_zero;                // 1: x starts at zero (x is not read)
  const double *a;
  int64_t lda;
  const double *b;
  int64_t ldb;
  double *r;
  int64_t ldr;
  unsigned long long *xw;    // [n][nrhs][2] tagged words of x + d
  unsigned long long *xbits, *rbits;
};

// Effective matrix E: forward & !trans -> L (strictly lower part of lu);
// !forward & !trans -> U; forward & trans -> U^T; !forward & trans -> L^T.
// Workgroup (block row i, column chunk ch) computes
//   x_i = D_i^-1 (x_i - sum_j E_ij x_j)
// over the blocks j already solved (j < i forward, j > i backward).  Tiles
// move global -> registers (16-byte lane-contiguous loads, issued before the
// wait for the previous block) -> LDS -> row segments per thread.
template <typename T, int BS, int RC, bool FUSE>
__device__ __forceinline__ void trsv_block(const TrsvArgs<T> &p, int wid, const IrFuse &f) {
  constexpr int WPE = sizeof(T) / 4;  // 32-bit words per element
  constexpr int TPR = 256 / BS;   // threads per row in the product
  constexpr int SEG = BS / TPR;   // columns per thread
  constexpr int VEC = 16 / sizeof(T);           // elements per 16-byte load
  constexpr int NV = BS * BS / VEC / 256;       // 16-byte loads per thread per tile
  constexpr int LDT = BS + VEC;                 // padded LDS row
  typedef T vec_t __attribute__((ext_vector_type(VEC)));
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *tile = reinterpret_cast<T *>(smem_raw);    // [BS][LDT]
  __shared__ T xs[BS][RC];
  __shared__ T ys[BS][RC];
  __shared__ int s_bail;
  const int t = threadIdx.x;
  const int r = t / TPR, h = t % TPR;
  const int ib = wid / p.nchunks, ch = wid % p.nchunks;
  const int i = p.forward ? ib : p.nblk - 1 - ib;
  const int r0 = i * BS;
  const int c0 = ch * RC;
  const int ncols = p.nrhs - c0 < RC ? p.nrhs - c0 : RC;
  const int gr = r0 + r;
  const bool rowok = gr < p.n;

  // Register staging of one BS x BS block of a row-major matrix (base, ld) at
  // block coordinates (rb, cb), optionally transposed; out-of-range is zero.
  // Element e of load k covers row (t*VEC + k*256*VEC) / BS.
  auto fetch = [&](const T *base, int64_t ld, int rb, int cb, vec_t (&v)[NV]) {
    const bool aligned = ((ld * sizeof(T)) % 16 == 0) && (reinterpret_cast<uintptr_t>(base) % 16 == 0);
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int lin = (k * 256 + t) * VEC;
      const int rr = lin / BS, cc = lin % BS;
      const int grow = rb + rr, gcol = cb + cc;
      if (aligned && grow < p.n && gcol + VEC <= p.n) {
        v[k] = *reinterpret_cast<const vec_t *>(base + (int64_t)grow * ld + gcol);
      } else {
#pragma unroll
        for (int q = 0; q < VEC; ++q)
          v[k][q] = (grow < p.n && gcol + q < p.n) ? base[(int64_t)grow * ld + gcol + q] : T(0);
      }
    }
  };
  // Stores the staged block into LDS as E (row r, column c), transposing when
  // the staged block is stored M[c][r].
  auto stash = [&](const vec_t (&v)[NV], bool transposed) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int lin = (k * 256 + t) * VEC;
      const int rr = lin / BS, cc = lin % BS;
      if (!transposed) {
        *reinterpret_cast<vec_t *>(tile + rr * LDT + cc) = v[k];
      } else {
#pragma unroll
        for (int q = 0; q < VEC; ++q) tile[(cc + q) * LDT + rr] = v[k][q];
      }
    }
  };

  // Diagonal inverse D_i (dense BS x BS, row-major): row segment per thread.
  T dreg[SEG];
  {
    vec_t v[NV];
    const T *D = p.dinv + (size_t)i * BS * BS;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int lin = (k * 256 + t) * VEC;
      v[k] = *reinterpret_cast<const vec_t *>(D + lin);
    }
    stash(v, p.dinv_trans != 0);
    __syncthreads();
#pragma unroll
    for (int s = 0; s < SEG; ++s) dreg[s] = tile[r * LDT + h * SEG + s];
    __syncthreads();
  }
  T acc[RC];
#pragma unroll
  for (int q = 0; q < RC; ++q) acc[q] = T(0);
  if (t == 0) s_bail = 0;
  // Fused refinement: this block's rows of x, read while the chain runs.
  double xold[RC];
#pragma unroll
  for (int q = 0; q < RC; ++q)
    xold[q] = (FUSE && !f.x_zero && h == 0 && rowok && q < ncols) ? f.x[(int64_t)gr * f.ldx + c0 + q] : 0.0;

  const int nb = p.forward ? i : p.nblk - 1 - i;  // number of dependency blocks
  auto issue = [&](int d, vec_t (&v)[NV]) {
    const int j = p.forward ? d : p.nblk - 1 - d;
    if (!p.trans)
      fetch(p.lu, p.lda, r0, j * BS, v);   // E_ij = M[r0.., jBS..]
    else
      fetch(p.lu, p.lda, j * BS, r0, v);   // E_ij = (M[jBS.., r0..])^T
  };
  vec_t stage[NV];
  if (nb > 0) issue(0, stage);
  for (int d = 0; d < nb; ++d) {
    const int j = p.forward ? d : p.nblk - 1 - d;
    const int cb = j * BS;
    stash(stage, p.trans != 0);
    if (d + 1 < nb) issue(d + 1, stage);
    // The solved values of block j: every thread polls its own tagged words
    // (bounded waits), so the values arrive with the first load that sees
    // them.
    {
      bool bail = false;
      for (int e = t; e < BS * RC; e += 256) {
        const int rr = e / RC, q = e % RC;
        const int gi = cb + rr;
        T v = T(0);
        if (gi < p.n && q < ncols) {
          const unsigned long long *w = p.xt + ((int64_t)gi * p.nrhs + c0 + q) * WPE;
          int spins = 0;
          for (;;) {
            if (spins >= p.wait_limit) {
              bail = true;
              break;
            }
            uint32_t part[WPE];
            bool ok = true;
#pragma unroll
            for (int k = 0; k < WPE; ++k) {
              const unsigned long long x = ld_sc1(w + k);
              ok = ok && (uint32_t)(x >> 32) == p.epoch;
              part[k] = (uint32_t)x;
            }
            if (ok) {
              v = from_words<T>(part);
              break;
            }
            if ((++spins & 63) == 0 && ld_sc1(p.err) != 0) {
              bail = true;
              break;
            }
            __builtin_amdgcn_s_sleep(1);
          }
        }
        xs[rr][q] = v;
      }
      if (bail) {
        atomic_or_agent(p.err, kErrWait);
        s_bail = 1;
      }
    }
    __syncthreads();
    if (s_bail) return;
#pragma unroll
    for (int s = 0; s < SEG; ++s) {
      const int c = h * SEG + s;
      const T e = tile[r * LDT + c];
#pragma unroll
      for (int q = 0; q < RC; ++q) acc[q] += e * xs[c][q];
    }
    __syncthreads();
  }
  // Combine the TPR partial sums of each row (consecutive lanes).
#pragma unroll
  for (int q = 0; q < RC; ++q) {
#pragma unroll
    for (int off = TPR / 2; off >= 1; off >>= 1) acc[q] += __shfl_xor(acc[q], off);
  }
  if (h == 0) {
#pragma unroll
    for (int q = 0; q < RC; ++q) {
      T bval = (rowok && q < ncols) ? p.xin[(int64_t)gr * p.ldx + c0 + q] : T(0);
      ys[r][q] = bval - acc[q];
    }
  }
  __syncthreads();
  T out[RC];
#pragma unroll
  for (int q = 0; q < RC; ++q) out[q] = T(0);
#pragma unroll
  for (int s = 0; s < SEG; ++s) {
    const int c = h * SEG + s;
#pragma unroll
    for (int q = 0; q < RC; ++q) out[q] += dreg[s] * ys[c][q];
  }
#pragma unroll
  for (int q = 0; q < RC; ++q) {
#pragma unroll
    for (int off = TPR / 2; off >= 1; off >>= 1) out[q] += __shfl_xor(out[q], off);
  }
  if (h == 0 && rowok) {
#pragma unroll
    for (int q = 0; q < RC; ++q) {
      if (q < ncols) {
        p.x[(int64_t)gr * p.ldx + c0 + q] = out[q];
        unsigned long long *w = p.xt + ((int64_t)gr * p.nrhs + c0 + q) * WPE;
#pragma unroll
        for (int k = 0; k < WPE; ++k) st_sc1(w + k, tagged(p.epoch, word_of<T>(out[q], k)));
      }
    }
  }
  if constexpr (FUSE) {
    // x + d in FP64 (the chain's words above go first), published for the
    // residual workgroups; the block's maxima of |x + d| by one atomic per
    // column.
    __shared__ unsigned long long s_xm[4][RC];
    unsigned long long xm[RC];
#pragma unroll
    for (int q = 0; q < RC; ++q) {
      xm[q] = 0ull;
      if (h == 0 && rowok && q < ncols) {
        const double xn = xold[q] + (double)out[q];
        f.x[(int64_t)gr * f.ldx + c0 + q] = xn;
        unsigned long long *w = f.xw + ((int64_t)gr * p.nrhs + c0 + q) * 2;
        st_sc1(w, tagged(p.epoch, word_of<double>(xn, 0)));
        st_sc1(w + 1, tagged(p.epoch, word_of<double>(xn, 1)));
        xm[q] = (unsigned long long)__double_as_longlong(fabs(xn));
      }
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) {
        const unsigned long long o = __shfl_xor(xm[q], off);
        xm[q] = o > xm[q] ? o : xm[q];
      }
    }
    if ((t & 63) == 0) {
#pragma unroll
      for (int q = 0; q < RC; ++q) s_xm[t >> 6][q] = xm[q];
    }
    __syncthreads();
    if (t < RC && t < ncols) {
      unsigned long long m = s_xm[0][t];
#pragma unroll
      for (int w = 1; w < 4; ++w) m = s_xm[w][t] > m ? s_xm[w][t] : m;
      atomicMax(f.xbits + c0 + t, m);
    }
  }
}

template <typename T, int BS>
__global__ void __launch_bounds__(256) trsv_dataflow_kernel(TrsvArgs<T> p) {
  trsv_block<T, BS, 1, false>(p, blockIdx.x, IrFuse{});
}

// Residual workgroup rw of the fused refinement step: rows
// 3 RPW rw .. 3 RPW (rw + 1) - 1 of r = b - A (x + d).  Wave 0 only waits for
// the values: per column block (in the backward solve's order, last block
// first) every lane reads the words of its two columns, lane 0 alone polls
// while some are missing, and the values go to LDS (by block parity).
// Waves 1..3 hold RPW rows each, two columns per lane, and keep the next
// block's A loads in flight across the workgroup barrier
// (which waits for LDS only), so HBM latency overlaps the chain.  The
// per-lane partial sums of a wave's rows are reduced by a butterfly that
// halves the rows at each step (the top lane bits select the row).
template <int RC>
__device__ __forceinline__ void ir_residual_block(const TrsvArgs<float> &p, const IrFuse &f, int rw) {
  constexpr int BS = TrsvBlock<float>::BS;  // 2 columns per lane
  constexpr int RPW = RC == 1 ? 16 : 8;      // rows per worker wave
  constexpr int LOGR = RPW == 16 ? 4 : 3;
  static_assert(BS == 128, "two columns per lane");
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double *sx = reinterpret_cast<double *>(smem_raw);  // [2][BS][RC]
  __shared__ unsigned long long s_rm[4][RC];
  __shared__ int s_bail[2];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n = p.n, nq = p.nrhs, nblk = p.nblk;
  const int row0 = rw * 3 * RPW + (wave - 1) * RPW;

  // Worker waves: A's values of block d, columns cb + lane and cb + 64 + lane
  // of the wave's rows (each load instruction reads 512 contiguous bytes).
  // Rows and columns past the end are clamped to the last one, so the loads
  // carry no branch (the compiler can then wait for one block's loads while
  // the next block's are in flight); the products mask those columns.
  auto load_a = [&](int d, double (&a0)[RPW], double (&a1)[RPW]) {
    const int cb = (nblk - 1 - d) * BS;
    const int c0 = min(cb + lane, n - 1), c1 = min(cb + 64 + lane, n - 1);
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      const double *ap = f.a + (int64_t)min(row0 + i, n - 1) * f.lda;
      a0[i] = ap[c0];
      a1[i] = ap[c1];
    }
  };
  // Wave 0: block d's values of x + d into LDS; returns false if a wait gave up.
  auto wait_x = [&](int d) -> bool {
    const int cb = (nblk - 1 - d) * BS;
    double *dst = sx + (d & 1) * BS * RC;
    bool bail = false;
    int spins = 0;
    auto ready = [&](const unsigned long long *w, double *v) -> bool {
      const unsigned long long w0 = ld_sc1(w), w1 = ld_sc1(w + 1);
      if ((uint32_t)(w0 >> 32) != p.epoch || (uint32_t)(w1 >> 32) != p.epoch) return false;
      const uint32_t part[2] = {(uint32_t)w0, (uint32_t)w1};
      *v = from_words<double>(part);
      return true;
    };
    auto spin = [&]() -> bool {  // false once the wait gives up
      if (spins >= p.wait_limit) return false;
      if ((++spins & 63) == 0 && ld_sc1(p.err) != 0) return false;
      __builtin_amdgcn_s_sleep(2);
      return true;
    };
    // Every lane reads the words of its two columns (one round trip when the
    // block is already solved); while some are missing, lane 0 polls the
    // first missing one and then the lanes read theirs again.
    double v[2][RC];
    bool have[2][RC];
#pragma unroll
    for (int k2 = 0; k2 < 2; ++k2)
#pragma unroll
      for (int q = 0; q < RC; ++q) {
        v[k2][q] = 0.0;
        have[k2][q] = !(cb + 64 * k2 + lane < n && q < nq);
      }
    for (;;) {
      bool all = true;
#pragma unroll
      for (int k2 = 0; k2 < 2; ++k2)
#pragma unroll
        for (int q = 0; q < RC; ++q)
          if (!have[k2][q]) {
            have[k2][q] = ready(f.xw + ((int64_t)(cb + 64 * k2 + lane) * nq + q) * 2, &v[k2][q]);
            all = all && have[k2][q];
          }
      const unsigned long long missing = __ballot(!all);
      if (!missing) break;
      // The first missing word of the first lane that lacks one.
      const int ml = __ffsll((long long)missing) - 1;
      int mw = 0;
#pragma unroll
      for (int k2 = 1; k2 >= 0; --k2)
#pragma unroll
        for (int q = RC - 1; q >= 0; --q)
          if (!have[k2][q]) mw = (cb + 64 * k2 + lane) * nq + q;
      mw = __shfl(mw, ml);
      if (lane == 0) {
        double tmp;
        while (!ready(f.xw + (int64_t)mw * 2, &tmp))
          if (!spin()) {
            bail = true;
            break;
          }
      }
      if (__shfl((int)bail, 0)) {
        bail = true;
        break;
      }
    }
#pragma unroll
    for (int k2 = 0; k2 < 2; ++k2)
#pragma unroll
      for (int q = 0; q < RC; ++q) dst[(64 * k2 + lane) * RC + q] = bail ? 0.0 : v[k2][q];
    return !__any(bail);
  };

  if (threadIdx.x == 0) s_bail[0] = s_bail[1] = 0;
  double acc[RPW][RC];
#pragma unroll
  for (int i = 0; i < RPW; ++i)
#pragma unroll
    for (int q = 0; q < RC; ++q) acc[i][q] = 0.0;
  double ba0[RPW], ba1[RPW], bb0[RPW], bb1[RPW];
  if (wave > 0) load_a(0, ba0, ba1);
  // One block: wave 0 waits for its values while the workers issue the next
  // block's loads; after the barrier the workers multiply.  The bail word
  // alternates with the LDS buffer, so every wave leaves at the same block.
  auto step = [&](int d, double (&c0)[RPW], double (&c1)[RPW], double (&n0)[RPW], double (&n1)[RPW]) -> bool {
    if (wave == 0) {
      const bool ok = wait_x(d);
      if (lane == 0) s_bail[d & 1] = ok ? 0 : 1;
    } else if (d + 1 < nblk) {
      load_a(d + 1, n0, n1);
    }
    __syncthreads();
    if (s_bail[d & 1]) return false;
    if (wave > 0) {
      const double *xs = sx + (d & 1) * BS * RC + lane * RC;
      const int cb = (nblk - 1 - d) * BS;
      const bool ok0 = cb + lane < n, ok1 = cb + 64 + lane < n;
#pragma unroll
      for (int q = 0; q < RC; ++q) {
        const double x0 = xs[q], x1 = xs[64 * RC + q];
#pragma unroll
        for (int i = 0; i < RPW; ++i)
          acc[i][q] += (ok0 ? c0[i] : 0.0) * x0 + (ok1 ? c1[i] : 0.0) * x1;
      }
    }
    return true;
  };
  bool ok = true;
  for (int d = 0; d < nblk && ok; d += 2) {
    ok = step(d, ba0, ba1, bb0, bb1);
    if (ok && d + 1 < nblk) ok = step(d + 1, bb0, bb1, ba0, ba1);
  }
  if (!ok && threadIdx.x == 0) atomic_or_agent(p.err, kErrWait);
  unsigned long long rm[RC];
#pragma unroll
  for (int q = 0; q < RC; ++q) rm[q] = 0ull;
  if (wave > 0) {
#pragma unroll
    for (int q = 0; q < RC; ++q) {
      // Butterfly over lane bits 5, 4, ...: a lane keeps half of its rows,
      // summed with its partner's; then the lanes that share a row sum.
#pragma unroll
      for (int h = RPW / 2, o = 32; h >= 1; h >>= 1, o >>= 1) {
        const bool up = (lane & o) != 0;
#pragma unroll
        for (int m = 0; m < h; ++m) {
          const double send = up ? acc[m][q] : acc[m + h][q];
          const double keep = up ? acc[m + h][q] : acc[m][q];
          acc[m][q] = keep + __shfl_xor(send, o);
        }
      }
#pragma unroll
      for (int o = 32 >> LOGR; o >= 1; o >>= 1) acc[0][q] += __shfl_xor(acc[0][q], o);
    }
    int ri = 0;
#pragma unroll
    for (int s = 0; s < LOGR; ++s) ri += ((lane >> (5 - s)) & 1) * ((RPW / 2) >> s);
    const int row = row0 + ri;
    const bool owner = (lane & ((64 / RPW) - 1)) == 0;
#pragma unroll
    for (int q = 0; q < RC; ++q) {
      if (ok && owner && row < n && q < nq) {
        const double rv = f.b[(int64_t)row * f.ldb + q] - acc[0][q];
        f.r[(int64_t)row * f.ldr + q] = rv;
        rm[q] = (unsigned long long)__double_as_longlong(fabs(rv));
      }
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) {
        const unsigned long long o = __shfl_xor(rm[q], off);
        rm[q] = o > rm[q] ? o : rm[q];
      }
    }
  }
  if (lane == 0) {
#pragma unroll
    for (int q = 0; q < RC; ++q) s_rm[wave][q] = rm[q];
  }
  __syncthreads();
  if ((int)threadIdx.x < RC && (int)threadIdx.x < nq) {
    const int q = threadIdx.x;
    unsigned long long m = s_rm[0][q];
#pragma unroll
    for (int w = 1; w < 4; ++w) m = s_rm[w][q] > m ? s_rm[w][q] : m;
    atomicMax(f.rbits + q, m);
  }
}

// The fused refinement step: workgroups 0 .. nblk - 1 run the backward
// solve (and x += d), the rest the residual.  The solve's workgroups come
// first in dispatch order and wait only on each other, the residual's wait
// only on the solve, so every wait ends whichever workgroups are resident.
template <int RC>
__global__ void __launch_bounds__(256) trsv_ir_kernel(TrsvArgs<float> p, IrFuse f) {
  constexpr int BS = TrsvBlock<float>::BS;
  const int ntri = p.nblk * p.nchunks;
  if ((int)blockIdx.x < ntri)
    trsv_block<float, BS, RC, true>(p, blockIdx.x, f);
  else
    ir_residual_block<RC>(p, f, blockIdx.x - ntri);
}

// Matrix-core dataflow solve for several right-hand sides: workgroup (block
// row i, chunk of 16 columns) keeps its BS x 16 right-hand sides in MFMA
// accumulators (a wave BS / 4 rows by 16 columns), subtracts E_ij X_j for the
// blocks j solved before it and applies the inverted diagonal block.
//  * E_ij tiles are staged through registers into LDS as they lie in memory
//    (pitch BS + 16 bytes: the 16 rows, or with TRANS columns, that an MFMA
//    operand reads together are on distinct banks).  MFMA step (s, ks) takes
//    k = 16 s + 4 g + ks from lane group g.
//  * -X_j is staged transposed ([column][k]), so acc = b - sum E_ij X_j.  Its
//    tagged words are all requested at once, eight per thread (bounded
//    polls): one round trip per block, not one per word.
//  * Every block's product is four (FP32: two) partial sums added pairwise
//    before they meet the right-hand side, so rounding grows with the number of
//    blocks and not with n (one running accumulator: 1.35 times the error).
//  * D_i^-1 stays in registers in the MFMA operand layout; y goes through LDS
//    as the second operand of x = D y.
// Bound by the chain of blocks: one round trip of the words (0.8 us), the
// products with the last block and with D (0.4 us each in FP64) and their
// barriers: 3.7 us per block in FP64 (236 us a solve of n = 4096), 7.2 us per
// block of 128 rows in FP32.  Both solves of n = 4096 with 64 right-hand sides,
// call included: 0.50 ms, where the vector kernel took 1.88 ms (14.7 us per
// block); with 16: 0.42 ms against 1.03.
template <typename T>
struct TrsmMfma;
template <>
struct TrsmMfma<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 op(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int g, int r) { return g + 4 * r; }
};
template <>
struct TrsmMfma<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 op(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int g, int r) { return 4 * g + r; }
};

template <typename T, int BS, bool TRANS>
__global__ void __launch_bounds__(256, 2) trsm_mfma_kernel(TrsvArgs<T> p) {
  typedef TrsmMfma<T> M;
  typedef typename M::v4 v4;
  constexpr int RC = 16, WPE = sizeof(T) / 4, VEC = 16 / sizeof(T), P = BS + VEC;
  constexpr int RB = BS / 64, KS = BS / 16;        // row blocks of a wave, k groups of 16
  constexpr int NC = 256 / BS;                     // partial sums of a product
  constexpr int NV = BS * BS / VEC / 256;          // 16-byte loads per thread per tile
  constexpr int NWD = BS * RC * WPE / 256;         // tagged words per thread per block
  typedef T vec_t __attribute__((ext_vector_type(VEC)));
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *tile = reinterpret_cast<T *>(smem_raw);       // [BS][P], as in memory
  __shared__ __align__(16) T xs[RC][P];            // second operand, transposed
  __shared__ int s_bail;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int g = lane >> 4, lc = lane & 15;
  const int ib = blockIdx.x / p.nchunks, ch = blockIdx.x % p.nchunks;
  const int i = p.forward ? ib : p.nblk - 1 - ib;
  const int r0 = i * BS, c0 = ch * RC;
  const int ncols = p.nrhs - c0 < RC ? p.nrhs - c0 : RC;
  const int wrow = wave * (BS / 4);                // this wave's first row
  auto arow = [&](int rb, int r) { return wrow + 16 * rb + M::row(g, r); };

  vec_t stage[NV];
  const bool aligned = ((p.lda * (int64_t)sizeof(T)) % 16 == 0) && (reinterpret_cast<uintptr_t>(p.lu) % 16 == 0);
  auto fetch = [&](int cb) {
    const int rb0 = TRANS ? cb : r0, cb0 = TRANS ? r0 : cb;
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      const int lin = (q * 256 + t) * VEC, grow = rb0 + lin / BS, gcol = cb0 + lin % BS;
      if (aligned && grow < p.n && gcol + VEC <= p.n) {
        stage[q] = *reinterpret_cast<const vec_t *>(p.lu + (int64_t)grow * p.lda + gcol);
      } else {
#pragma unroll
        for (int e = 0; e < VEC; ++e)
          stage[q][e] = (grow < p.n && gcol + e < p.n) ? p.lu[(int64_t)grow * p.lda + gcol + e] : T(0);
      }
    }
  };
  auto stash = [&]() {
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      const int lin = (q * 256 + t) * VEC;
      *reinterpret_cast<vec_t *>(tile + lin / BS * P + lin % BS) = stage[q];
    }
  };
  // Four consecutive k of row `row` of E, of column lc of the second operand.
  auto a_of = [&](int row, int k) -> v4 {
    v4 v;
    if (TRANS) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = tile[(k + e) * P + row];
    } else {
      __builtin_memcpy(&v, __builtin_assume_aligned(tile + row * P + k, 16), sizeof v);
    }
    return v;
  };
  auto b_of = [&](int k) -> v4 {
    v4 v;
    __builtin_memcpy(&v, __builtin_assume_aligned(&xs[lc][k], 16), sizeof v);
    return v;
  };

  // D_i^-1 in the first operand's layout.
  v4 dreg[RB][KS];
  {
    const T *D = p.dinv + (size_t)i * BS * BS;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = wrow + 16 * rb + lc, k = 16 * s + 4 * g + e;
          dreg[rb][s][e] = TRANS ? D[k * BS + row] : D[row * BS + k];
        }
  }
  v4 acc[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int gi = r0 + arow(rb, r);
      acc[rb][r] = (gi < p.n && lc < ncols) ? p.xin[(int64_t)gi * p.ldx + c0 + lc] : T(0);
    }
  if (t == 0) s_bail = 0;

  const int nb = p.forward ? i : p.nblk - 1 - i;  // dependency blocks
  auto dep = [&](int d) { return p.forward ? d : p.nblk - 1 - d; };
  if (nb > 0) fetch(dep(0) * BS);
  for (int d = 0; d < nb; ++d) {
    const int cb = dep(d) * BS;
    __syncthreads();  // the previous product is done with tile and xs
    stash();
    if (d + 1 < nb) fetch(dep(d + 1) * BS);
    // The solved values of block j: word `part` (the high one first) of
    // element (kr, q).  Past the matrix the last row's words stand in.
    {
      unsigned long long w[NWD];
      bool bail = false;
      for (int spins = 0;;) {
        bool ok = spins < p.wait_limit;
        if (!ok) {
          bail = true;
          break;
        }
#pragma unroll
        for (int m = 0; m < NWD; ++m) {
          const int e = m * 256 + t, kr = e / (RC * WPE), q = e % (RC * WPE) / WPE, part = e % WPE;
          const int gi = min(cb + kr, p.n - 1), gq = c0 + min(q, ncols - 1);
          w[m] = ld_sc1(p.xt + ((int64_t)gi * p.nrhs + gq) * WPE + part);
        }
#pragma unroll
        for (int m = 0; m < NWD; ++m) ok = ok && (uint32_t)(w[m] >> 32) == p.epoch;
        if (ok) break;
        if ((++spins & 63) == 0 && ld_sc1(p.err) != 0) {
          bail = true;
          break;
        }
      }
#pragma unroll
      for (int m = 0; m < NWD; ++m) {
        const int e = m * 256 + t, kr = e / (RC * WPE), q = e % (RC * WPE) / WPE, part = e % WPE;
        uint32_t x = cb + kr < p.n ? (uint32_t)w[m] : 0u;
        x ^= part == 0 ? 0x80000000u : 0u;  // -X_j
        reinterpret_cast<uint32_t *>(&xs[q][kr])[WPE - 1 - part] = x;
      }
      if (bail) {
        atomic_or_agent(p.err, kErrWait);
        s_bail = 1;
      }
    }
    __syncthreads();
    if (s_bail) return;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      v4 sum[NC];
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const v4 bq = b_of(16 * s + 4 * g);
        const v4 aq = a_of(wrow + 16 * rb + lc, 16 * s + 4 * g);
        if (s < NC) sum[s] = v4{T(0), T(0), T(0), T(0)};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) sum[s % NC] = M::op(aq[ks], bq[ks], sum[s % NC]);
      }
#pragma unroll
      for (int w = NC / 2; w >= 1; w /= 2)
#pragma unroll
        for (int q = 0; q < w; ++q) sum[q] += sum[q + w];
      acc[rb] += sum[0];
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __syncthreads();  // the last product is done with xs
  // y (this block's right-hand sides minus the dependencies) as the second operand.
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int r = 0; r < 4; ++r) xs[lc][arow(rb, r)] = acc[rb][r];
  __syncthreads();
  v4 out[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    v4 sum[NC];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const v4 bq = b_of(16 * s + 4 * g);
      if (s < NC) sum[s] = v4{T(0), T(0), T(0), T(0)};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) sum[s % NC] = M::op(dreg[rb][s][ks], bq[ks], sum[s % NC]);
    }
#pragma unroll
    for (int w = NC / 2; w >= 1; w /= 2)
#pragma unroll
      for (int q = 0; q < w; ++q) sum[q] += sum[q + w];
    out[rb] = sum[0];
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int gi = r0 + arow(rb, r);
      if (gi < p.n && lc < ncols) {
        unsigned long long *w = p.xt + ((int64_t)gi * p.nrhs + c0 + lc) * WPE;
#pragma unroll
        for (int k = 0; k < WPE; ++k) st_sc1(w + k, tagged(p.epoch, word_of<T>(out[rb][r], k)));
        p.x[(int64_t)gi * p.ldx + c0 + lc] = out[rb][r];
      }
    }
}

// Tagged words of solved values; zeroed whenever they are (re)allocated or the
// epoch would wrap, so that no stale word carries a live tag.
hipError_t tri_words(lair_context *ctx, size_t words, unsigned long long **xt) {
  const size_t bytes = sizeof(unsigned long long) * words;
  const bool grow = ctx->ws_flags.bytes < bytes;
  hipError_t e = ensure(ctx->ws_flags, bytes);
  if (e != hipSuccess) return e;
  if (grow) ctx->ws_flags_zeroed = 0;
  if (ctx->ws_flags_zeroed < ctx->ws_flags.bytes || ctx->tri_epoch > 0x70000000u) {
    e = launch_fill_u32(ctx, static_cast<uint32_t *>(ctx->ws_flags.ptr),
                        (int64_t)(ctx->ws_flags.bytes / sizeof(uint32_t)), 0u);
    if (e != hipSuccess) return e;
    ctx->ws_flags_zeroed = ctx->ws_flags.bytes;
    ctx->tri_epoch = 0;
  }
  *xt = static_cast<unsigned long long *>(ctx->ws_flags.ptr);
  return hipSuccess;
}

template <typename T>
static hipError_t trsv_launch(lair_context *ctx, const T *lu, int64_t lda, const T *dinv,
                              bool dinv_trans, const T *xin, T *x, int64_t ldx, int n, int nrhs,
                              bool forward, bool trans, IrFuse *fz) {
  if (n <= 0 || nrhs <= 0) return hipSuccess;
  constexpr int BS = TrsvBlock<T>::BS;
  // From two right-hand sides on the matrix cores win over the vector kernel
  // (64-row blocks, chunks of 4), both solves of n = 4096 in FP64: 378 against
  // 569 us at 2, 373 against 667 at 4, 422 against 1027 at 16, 471 against
  // 1550 at 40; n = 300: 67 against 77 us at 2.  One right-hand side stays
  // with the vector kernel (285 us: no operand staging in its chain links).
  // The fused refinement step has its own kernel, in chunks of 4.
  const bool mfma = !fz && nrhs > 1;
  if (mfma && trans != dinv_trans) return hipErrorInvalidValue;
  const int rc = mfma ? 16 : (nrhs == 1 ? 1 : 4);
  const int nblk = (n + BS - 1) / BS;
  const int nchunks = (nrhs + rc - 1) / rc;
  // A caller-provided buffer (xt_override) was zeroed by the caller.
  unsigned long long *xt = ctx->xt_override;
  if (!xt) {
    // The fused refinement step also needs two words per value of x + d.
    const hipError_t e = tri_words(ctx, (size_t)n * nrhs * (sizeof(T) / 4 + (fz ? 2 : 0)), &xt);
    if (e != hipSuccess) return e;
  } else if (ctx->tri_epoch > 0x70000000u) {
    ctx->tri_epoch = 0;
  }
  TrsvArgs<T> a;
  a.lu = lu;
  a.lda = lda;
  a.dinv = dinv;
  a.xin = xin;
  a.x = x;
  a.ldx = ldx;
  a.n = n;
  a.nrhs = nrhs;
  a.nblk = nblk;
  a.nchunks = nchunks;
  a.xt = xt;
  a.epoch = ++ctx->tri_epoch;
  a.forward = forward ? 1 : 0;
  a.trans = trans ? 1 : 0;
  a.dinv_trans = dinv_trans ? 1 : 0;
  a.err = ctx->err;
  a.wait_limit = ctx->wait_limit;
  const unsigned grid = (unsigned)(nblk * nchunks);
  const size_t shm = (size_t)BS * (BS + 16 / sizeof(T)) * sizeof(T);
  static bool once = (allow_large_lds(trsv_dataflow_kernel<T, BS>), true);
  (void)once;
  if constexpr (std::is_same<T, float>::value) {
    if (fz) {
      static bool once_f = (allow_large_lds(trsv_ir_kernel<1>), allow_large_lds(trsv_ir_kernel<4>), true);
      (void)once_f;
      fz->xw = xt + (size_t)n * nrhs;
      // Residual workgroups: 48 rows each for one right-hand side, else 24.
      const int rrows = rc == 1 ? 48 : 24;
      const unsigned gridf = grid + (unsigned)((n + rrows - 1) / rrows);
      const int slot = prof_begin(ctx, LAIR_KCLASS_GETRS);
      if (rc == 1)
        trsv_ir_kernel<1><<<gridf, 256, shm, ctx->stream>>>(a, *fz);
      else
        trsv_ir_kernel<4><<<gridf, 256, shm, ctx->stream>>>(a, *fz);
      // The solve's bytes plus one pass over the FP64 A.
      prof_end(ctx, slot, LAIR_KCLASS_GETRS, (double)n * n * nrhs * 3,
               sizeof(T) * 0.5 * (double)n * n + 8.0 * n * n + 32.0 * n * nrhs);
      return hipGetLastError();
    }
  }
  const int slot = prof_begin(ctx, LAIR_KCLASS_GETRS);
  if (mfma) {
    static bool once_m = (allow_large_lds(trsm_mfma_kernel<T, BS, false>),
                          allow_large_lds(trsm_mfma_kernel<T, BS, true>), true);
    (void)once_m;
    if (trans)
      trsm_mfma_kernel<T, BS, true><<<grid, 256, shm, ctx->stream>>>(a);
    else
      trsm_mfma_kernel<T, BS, false><<<grid, 256, shm, ctx->stream>>>(a);
    prof_end(ctx, slot, LAIR_KCLASS_GETRS, (double)n * n * nrhs,
             sizeof(T) * (0.5 * (double)n * n + 2.0 * n * nrhs));
    return hipGetLastError();
  }
  trsv_dataflow_kernel<T, BS><<<grid, 256, shm, ctx->stream>>>(a);
  prof_end(ctx, slot, LAIR_KCLASS_GETRS, (double)n * n * nrhs,
           sizeof(T) * (0.5 * (double)n * n + 2.0 * n * nrhs));
  return hipGetLastError();
}

template <typename T>
hipError_t launch_trsv_dataflow(lair_context *ctx, const T *lu, int64_t lda, const T *dinv,
                                bool dinv_trans, const T *xin, T *x, int64_t ldx, int n, int nrhs,
                                bool forward, bool trans) {
  return trsv_launch<T>(ctx, lu, lda, dinv, dinv_trans, xin, x, ldx, n, nrhs, forward, trans, nullptr);
}

hipError_t launch_trsv_ir(lair_context *ctx, const float *lu, int64_t lda, const float *uinv,
                          const float *y, float *d, int n, int nrhs, double *x, int64_t ldx,
                          bool x_zero, const double *a, int64_t lda64, const double *b, int64_t ldb,
                          double *r, int64_t ldr, unsigned long long *xbits,
                          unsigned long long *rbits) {
  if (nrhs > 4) return hipErrorInvalidValue;
  IrFuse fz{};
  fz.x = x;
  fz.ldx = ldx;
  fz.x_zero = x_zero ? 1 : 0;
  fz.a = a;
  fz.lda = lda64;
  fz.b = b;
  fz.ldb = ldb;
  fz.r = r;
  fz.ldr = ldr;
  fz.xbits = xbits;
  fz.rbits = rbits;
  return trsv_launch<float>(ctx, lu, lda, uinv, false, y, d, nrhs, n, nrhs, false, false, &fz);
}

template hipError_t launch_trsv_dataflow<double>(lair_context *, const double *, int64_t,
                                                 const double *, bool, const double *, double *,
                                                 int64_t, int, int, bool, bool);
template hipError_t launch_trsv_dataflow<float>(lair_context *, const float *, int64_t,
                                                const float *, bool, const float *, float *, int64_t,
                                                int, int, bool, bool);

}  // namespace lair
