// Complex LU pieces that the real path does not share: the trailing update
// on the real MFMA GEMM through an embedding of U12, and the complex getrs.
//
// Trailing update A22 -= L21 U12 (src/lapack/getrf.rs:289-296, gemm.rs:6-32)
// in complex arithmetic, as one real GEMM: with interleaved storage, row i of
// L21 (K complex) is a real row of 2K values (re, im, re, im, ...) and row i
// of A22 one of 2N values, so
//   A22_int (M x 2N) -= L21_int (M x 2K) * E (2K x 2N)
// with E[2p] = (u.re, u.im) per column (row p of U12 as stored) and
// E[2p + 1] = (-u.im, u.re).  Same flop count as the complex product; L21 and
// A22 are read in place, only U12 (K rows) is copied.  E is indexed by the
// absolute column of the matrix, so the two streams of the look-ahead, which
// update disjoint column ranges of the same panel, never share a slot.
//
// getrs (src/lapack/getrs.rs:12-39): x = P b; unit-lower forward
// substitution x[i] -= a[i][k] x[k] for k < i; back substitution
// x[i] -= a[i][k] x[k] for k > i, then x[i] /= a[i][i].  For n <=
// kExactOrderMax one workgroup per right-hand side runs the reference's
// operations in its order (bit-identical, num-complex DivAssign included);
// beyond, both substitutions are dataflow solves over 64-row blocks.
#include <algorithm>

#include "device_util.h"
#include "lair_internal.h"

namespace lair {

template <typename R>
__global__ void __launch_bounds__(256)
    cembed_kernel(int K, int N, const cplx<R> *__restrict__ B, int64_t ldb, R *__restrict__ E, int64_t lde) {
  const int j = blockIdx.x * 256 + threadIdx.x, p = blockIdx.y;
  if (j >= N) return;
  const cplx<R> u = B[(int64_t)p * ldb + j];
  R *e0 = E + (int64_t)(2 * p) * lde + 2 * j;
  R *e1 = e0 + lde;
  e0[0] = u.re;
  e0[1] = u.im;
  e1[0] = -u.im;
  e1[1] = u.re;
}

template <typename T>
hipError_t launch_cgemm_minus(lair_context *ctx, int mode, int M, int N, int K, const T *A, int64_t lda,
                              const T *B, int64_t ldb, T *C, int64_t ldc, int col, int kclass) {
  typedef typename cplx_traits<T>::real R;
  if (M <= 0 || N <= 0 || K <= 0) return hipSuccess;
  R *E = static_cast<R *>(ctx->ws_cexp.ptr);
  const int64_t lde = ctx->cexp_ld;
  if (!E || K > kComplexMaxNb || col < 0 || 2 * ((int64_t)col + N) > lde ||
      ctx->ws_cexp.bytes < sizeof(R) * (size_t)(2 * kComplexMaxNb) * (size_t)lde)
    return hipErrorInvalidValue;
  R *Ec = E + 2 * (int64_t)col;
  cembed_kernel<R><<<dim3((N + 255) / 256, K), 256, 0, ctx->stream>>>(K, N, B, ldb, Ec, lde);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return launch_gemm_minus<R>(ctx, mode, M, 2 * N, 2 * K, reinterpret_cast<const R *>(A), 2 * lda, false, Ec, lde,
                              reinterpret_cast<R *>(C), 2 * ldc, kclass);
}

// n <= kExactOrderMax, thread t keeps row t.  The forward pass goes by 64-row
// blocks: the wave owning the block solves it (each row's subtractions in
// increasing k), the block's values go through LDS and the rows below subtract
// its 64 terms in increasing k.  The back substitution takes its terms in
// increasing k, which needs every later unknown first: one wave runs it row by
// row.
template <typename T>
__global__ void __launch_bounds__(kExactOrderMax)
    cgetrs_exact_kernel(int n, const T *__restrict__ lu, int64_t lda, const int *__restrict__ perm, T *__restrict__ b,
                        int64_t ldb) {
#pragma clang fp contract(off)
  constexpr int LB = 8;  // loads in flight per batch
  __shared__ T xs[64];
  __shared__ T xall[kExactOrderMax];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int r = blockIdx.x;
  T x = t < n ? b[(int64_t)perm[t] * ldb + r] : T(0);
  const int nblk = (n + 63) / 64;

  // Forward substitution with unit lower L.
  for (int bk = 0; bk < nblk; ++bk) {
    const int k0 = bk * 64, kn = min(64, n - k0);
    if (wave == bk) {
      const T *li = lu + (int64_t)(lane < kn ? k0 + lane : k0) * lda + k0;
      for (int kc = 0; kc < kn; kc += LB) {
        T lv[LB];
#pragma unroll
        for (int q = 0; q < LB; ++q) lv[q] = (kc + q < lane && lane < kn) ? li[kc + q] : T(0);
#pragma unroll
        for (int q = 0; q < LB; ++q) {
          const int kk = kc + q;
          if (kk < kn) {
            const T xk = readlane_t(x, kk);
            if (kk < lane && lane < kn) {
              const T e = lv[q] * xk;
              x = x - e;
            }
          }
        }
      }
      if (lane < kn) xs[lane] = x;
    }
    __syncthreads();
    if (t >= k0 + kn && t < n) {
      const T *li = lu + (int64_t)t * lda + k0;
      for (int kc = 0; kc < kn; kc += LB) {
        T lv[LB];
#pragma unroll
        for (int q = 0; q < LB; ++q) lv[q] = kc + q < kn ? li[kc + q] : T(0);
#pragma unroll
        for (int q = 0; q < LB; ++q) {
          if (kc + q < kn) {
            const T e = lv[q] * xs[kc + q];
            x = x - e;
          }
        }
      }
    }
    __syncthreads();
  }

  // Back substitution with U.
  if (t < n) xall[t] = x;
  __syncthreads();
  if (wave == 0) {
    for (int i = n - 1; i >= 0; --i) {
      const T *ui = lu + (int64_t)i * lda;
      const int c0 = i + 1 + lane, c1 = i + 65 + lane;
      const T u0 = c0 < n ? ui[c0] : T(0);
      const T u1 = c1 < n ? ui[c1] : T(0);
      T xi = xall[i];
      for (int k = i + 1; k < n; ++k) {
        const int q = k - i - 1;
        const T u = q < 64 ? readlane_t(u0, q) : readlane_t(u1, q - 64);
        const T e = u * xall[k];
        xi = xi - e;
      }
      const T xn = cplx_div(xi, ui[i]);
      if (lane == 0) xall[i] = xn;
    }
  }
  __syncthreads();
  if (t < n) b[(int64_t)t * ldb + r] = xall[t];
}

// acc - a b, by fused multiply-adds.
template <typename R>
__device__ __forceinline__ cplx<R> csub_mul(cplx<R> acc, cplx<R> a, cplx<R> b) {
  return cplx<R>(__builtin_elementwise_fma(a.im, b.im, __builtin_elementwise_fma(-a.re, b.re, acc.re)),
                 __builtin_elementwise_fma(-a.im, b.re, __builtin_elementwise_fma(-a.re, b.im, acc.im)));
}

// c ? a : b by components (a conditional on the struct goes through memory).
template <typename R>
__device__ __forceinline__ cplx<R> csel(bool c, cplx<R> a, cplx<R> b) {
  return cplx<R>(c ? a.re : b.re, c ? a.im : b.im);
}

// n > kExactOrderMax: one substitution (unit lower forward, or upper backward)
// as a dataflow.  Workgroup (block row i of 64 rows, right-hand side) has four
// threads per row subtract E_ij x_j, 16 columns each, for the blocks j solved
// before it (their E entries are requested before the wait for x_j), then one
// wave solves the diagonal block by substitution, a lane per row, from the
// block's transpose in LDS, and publishes its values as tagged words.  Blocks
// start in the order of the solve, so every wait ends; waits are bounded.
//
// The quotients of the back substitution are x conj(d) / |d|^2 by the
// precomputed inverse of d and one correction by the remainder, which is at
// least as close as the direct formula; blocks with a diagonal entry far from
// 1 in the exponent use the direct formula, and so does a block again whose
// result is not finite (an infinite right-hand side, or a quotient that
// overflows, makes NaN of the remainder).
//
// Bound by the chain: 64 substitution steps per block (1.4 us with f64
// components, 5.5 us with the quotients) and one round trip of the words.
// n = 1500 with three right-hand sides: 109 + 209 us, where one workgroup per
// right-hand side, a row per thread, took 1920 us.
constexpr int kCflowBS = 64;
template <typename T>
struct CflowArgs {
  const T *lu;
  int64_t lda;
  const int *perm;  // rows of x_in, or null
  const T *xin;
  int64_t ldi;
  T *x;
  int64_t ldx;
  int n, nrhs, nblk;
  unsigned long long *xt;  // [nrhs][n][words] tagged solved values
  uint32_t epoch;
  int32_t *err;
  int wait_limit;
};

template <typename T, bool UPPER>
__global__ void __launch_bounds__(256, 2) cgetrs_flow_kernel(CflowArgs<T> p) {
  typedef typename cplx_traits<T>::real R;
  constexpr int BS = kCflowBS, WPE = sizeof(T) / 4, H = WPE / 2, SEG = 16, LD = BS + 1;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *dt = reinterpret_cast<T *>(smem_raw);  // [k][row]: the diagonal block
  __shared__ T xs[2][BS];
  __shared__ T ys[BS];
  __shared__ int s_bail[2];  // by block parity
  const int t = threadIdx.x, lane = t & 63;
  const int ib = blockIdx.x / p.nrhs, c = blockIdx.x % p.nrhs;
  const int i = UPPER ? p.nblk - 1 - ib : ib;
  const int r0 = i * BS, w = min(BS, p.n - r0);
  const int r = t >> 2, h = t & 3;
  const int gr = min(r0 + r, p.n - 1);
  unsigned long long *xt = p.xt + (int64_t)c * p.n * WPE;
  if (t < 2) s_bail[t] = 0;
  __syncthreads();  // before a wave's first wait may set a flag

  for (int e = t; e < BS * BS; e += 256) {
    const int row = e / BS, k = e % BS;
    dt[k * LD + row] = p.lu[(int64_t)min(r0 + row, p.n - 1) * p.lda + min(r0 + k, p.n - 1)];
  }
  const T *row = p.lu + (int64_t)gr * p.lda;
  T seg[SEG], acc(0);
  auto dep = [&](int d) { return UPPER ? p.nblk - 1 - d : d; };
  auto fetch = [&](int cb) {
#pragma unroll
    for (int s = 0; s < SEG; ++s) seg[s] = row[min(cb + h * SEG + s, p.n - 1)];
  };
  T bval(0);
  if (h == 0) bval = p.xin[(int64_t)(p.perm ? p.perm[gr] : gr) * p.ldi + c];
  if (ib > 0) fetch(dep(0) * BS);
  for (int d = 0; d < ib; ++d) {
    const int cb = dep(d) * BS;
    T *xd = xs[d & 1];
    // Element kr's words; past the matrix (ragged last block) zeros.
    if (t < BS * H) {
      const int kr = t / H, gi = min(cb + kr, p.n - 1), part = t % H;
      const unsigned long long *wp = xt + (int64_t)gi * WPE + part;
      unsigned long long w0, w1;
      for (int spins = 0;;) {
        if (spins >= p.wait_limit) {
          atomic_or_agent(p.err, kErrWait);
          s_bail[d & 1] = 1;
          w0 = w1 = 0;
          break;
        }
        w0 = ld_agent(wp);
        w1 = ld_agent(wp + H);
        if ((uint32_t)(w0 >> 32) == p.epoch && (uint32_t)(w1 >> 32) == p.epoch) break;
        if ((++spins & 63) == 0 && ld_agent(p.err) != 0) {
          s_bail[d & 1] = 1;
          break;
        }
      }
      // word_of: the real part's words, then the imaginary part's, high first.
      uint32_t *dst = reinterpret_cast<uint32_t *>(&xd[kr]);
      const bool in = cb + kr < p.n;
      dst[H - 1 - part] = in ? (uint32_t)w0 : 0u;
      dst[WPE - 1 - part] = in ? (uint32_t)w1 : 0u;
    }
    __syncthreads();
    if (s_bail[d & 1]) return;
#pragma unroll
    for (int s = 0; s < SEG; ++s) acc = csub_mul(acc, seg[s], xd[h * SEG + s]);
    if (d + 1 < ib) fetch(dep(d + 1) * BS);
  }
#pragma unroll
  for (int off = 2; off >= 1; off >>= 1)
    acc = T(acc.re + __shfl_xor(acc.re, off), acc.im + __shfl_xor(acc.im, off));
  if (h == 0) ys[r] = r < w ? T(bval.re + acc.re, bval.im + acc.im) : T(0);
  __syncthreads();
  if (t >= 64) return;
  T x = ys[lane];
  if (!UPPER) {
    for (int k0 = 0; k0 < w; k0 += 8) {
      T l[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) l[q] = dt[(k0 + q) * LD + lane];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const T nx = csub_mul(x, l[q], readlane_t(x, k0 + q));
        x = csel(lane > k0 + q && lane < w, nx, x);
      }
    }
  } else {
    const T dg = dt[lane * LD + lane];
    const R ns = dg.re * dg.re + dg.im * dg.im;
    const R lo = sizeof(R) == 8 ? R(0x1p-500) : R(0x1p-60f), hi = sizeof(R) == 8 ? R(0x1p500) : R(0x1p60f);
    bool fast = __all(lane >= w || (ns >= lo && ns <= hi));
    const T inv(dg.re / ns, -dg.im / ns);
    for (;;) {
      for (int k0 = (w - 1) / 8 * 8; k0 >= 0; k0 -= 8) {
        T u[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) u[q] = dt[(k0 + q) * LD + lane];
#pragma unroll
        for (int q = 7; q >= 0; --q) {
          if (k0 + q < w) {
            T v;
            if (fast) {
              v = csub_mul(T(0), T(-x.re, -x.im), inv);
              v = csub_mul(v, T(0) - csub_mul(x, v, dg), inv);
            } else {
              v = cplx_div(x, dg);
            }
            x = csel(lane == k0 + q, v, x);
            const T nx = csub_mul(x, u[q], readlane_t(x, k0 + q));
            x = csel(lane < k0 + q, nx, x);
          }
        }
      }
      if (!fast || __all(lane >= w || (x.re - x.re == R(0) && x.im - x.im == R(0)))) break;
      fast = false;
      x = ys[lane];
    }
  }
  if (lane < w) {
    unsigned long long *wp = xt + (int64_t)(r0 + lane) * WPE;
#pragma unroll
    for (int k = 0; k < WPE; ++k) st_agent(wp + k, tagged(p.epoch, word_of<T>(x, k)));
    p.x[(int64_t)(r0 + lane) * p.ldx + c] = x;
  }
}

template <typename T>
hipError_t launch_cgetrs(lair_context *ctx, int n, int nrhs, const T *lu, int64_t lda, const int *perm, T *b,
                         int64_t ldb) {
  if (n <= 0 || nrhs <= 0) return hipSuccess;
  if (n > kComplexGetrsMax) return hipErrorInvalidValue;
  hipStream_t st = ctx->stream;
  if (n <= kExactOrderMax) {
    const int slot = prof_begin(ctx, LAIR_KCLASS_GETRS);
    cgetrs_exact_kernel<T><<<nrhs, kExactOrderMax, 0, st>>>(n, lu, lda, perm, b, ldb);
    prof_end(ctx, slot, LAIR_KCLASS_GETRS, 8.0 * (double)n * n * nrhs,
             (double)sizeof(T) * ((double)n * n * nrhs + 2.0 * n * nrhs));
    return hipGetLastError();
  }
  // Passes of as many right-hand sides as the workspaces hold: 64 of the
  // largest order (50 MB with f64 components), more of smaller ones, so that a
  // small system with many of them still fills the chip (n=150 with 300, f64
  // components: 171 us in one workgroup per right-hand side, 265 in passes of 64).
  const int chunk = std::min(nrhs, 64 * kComplexGetrsMax / n);
  hipError_t e = ensure(ctx->ws_tmp2, sizeof(T) * (size_t)n * chunk);
  if (e != hipSuccess) return e;
  CflowArgs<T> a;
  e = tri_words(ctx, (size_t)n * chunk * (sizeof(T) / 4), &a.xt);
  if (e != hipSuccess) return e;
  const size_t shm = sizeof(T) * kCflowBS * (kCflowBS + 1);
  static const hipError_t once[2] = {
      hipFuncSetAttribute(reinterpret_cast<const void *>(cgetrs_flow_kernel<T, false>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm),
      hipFuncSetAttribute(reinterpret_cast<const void *>(cgetrs_flow_kernel<T, true>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm)};
  for (hipError_t o : once)
    if (o != hipSuccess) return o;
  a.lu = lu;
  a.lda = lda;
  a.n = n;
  a.nblk = (n + kCflowBS - 1) / kCflowBS;
  a.err = ctx->err;
  a.wait_limit = ctx->wait_limit;
  T *tmp = static_cast<T *>(ctx->ws_tmp2.ptr);
  for (int c0 = 0; c0 < nrhs; c0 += chunk) {
    a.nrhs = std::min(chunk, nrhs - c0);
    const int slot = prof_begin(ctx, LAIR_KCLASS_GETRS);
    a.perm = perm;
    a.xin = b + c0;
    a.ldi = ldb;
    a.x = tmp;
    a.ldx = a.nrhs;
    a.epoch = ++ctx->tri_epoch;
    cgetrs_flow_kernel<T, false><<<a.nblk * a.nrhs, 256, shm, st>>>(a);
    a.perm = nullptr;
    a.xin = tmp;
    a.ldi = a.nrhs;
    a.x = b + c0;
    a.ldx = ldb;
    a.epoch = ++ctx->tri_epoch;
    cgetrs_flow_kernel<T, true><<<a.nblk * a.nrhs, 256, shm, st>>>(a);
    prof_end(ctx, slot, LAIR_KCLASS_GETRS, 8.0 * (double)n * n * a.nrhs,
             (double)sizeof(T) * ((double)n * n * a.nrhs + 2.0 * n * a.nrhs));
  }
  return hipGetLastError();
}

template hipError_t launch_cgemm_minus<zcplx>(lair_context *, int, int, int, int, const zcplx *, int64_t,
                                              const zcplx *, int64_t, zcplx *, int64_t, int, int);
template hipError_t launch_cgemm_minus<ccplx>(lair_context *, int, int, int, int, const ccplx *, int64_t,
                                              const ccplx *, int64_t, ccplx *, int64_t, int, int);
template hipError_t launch_cgetrs<zcplx>(lair_context *, int, int, const zcplx *, int64_t, const int *, zcplx *,
                                         int64_t);
template hipError_t launch_cgetrs<ccplx>(lair_context *, int, int, const ccplx *, int64_t, const int *, ccplx *,
                                         int64_t);

}  // namespace lair
