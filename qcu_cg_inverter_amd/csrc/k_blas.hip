// k_blas.hip -- level-1 kernels and the CGLS scalar steps.
//
// The reference does each BLAS-1 op as its own kernel plus a host round trip per
// reduction (src/qcu_complex_computation.cu:10-134, src/cg_inverter.cu:181-256).
// Here reductions are per-64-site partials (fixed butterfly order within a wave)
// summed by a one-block kernel in a fixed order, so every result is bitwise reproducible and
// independent of how right-hand sides are batched, and all scalars stay on the
// device: a CG iteration needs no host synchronisation.
#include "qcu_fields.h"
#include "qcu_kernels.h"

namespace qcu {

static inline unsigned nblk(long n, int b) { return (unsigned)((n + b - 1) / b); }

// a wave's partial, the sum over its 64-site chunk (first lane i), at slot i / 64
__device__ __forceinline__ void put_partial(double* part, long vh, int r, long i, double v) {
  v = group64_sum(v);
  if ((threadIdx.x & 63) == 0 && i < vh) part[(long)r * n_partials(vh) + i / 64] = v;
}

template <int P>
__global__ void zero_kernel(Vec v, long vh) {
  using T = typename Real<P>::T;
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= vh) return;
  cx<T> z[12];
#pragma unroll
  for (int c = 0; c < 12; ++c) z[c] = {T(0), T(0)};
  SpinorIO<P>::store(static_cast<char*>(v.p) + blockIdx.y * v.stride, vh, i, z);
}

template <int P>
__global__ void norm2_kernel(Vec v, long vh, double* part) {
  using T = typename Real<P>::T;
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  int r = blockIdx.y;
  double s = 0.0;
  if (i < vh) {
    cx<T> a[12];
    SpinorIO<P>::load(static_cast<const char*>(v.p) + r * v.stride, vh, i, a);
    T t = T(0);
#pragma unroll
    for (int c = 0; c < 12; ++c) t += norm2(a[c]);
    s = (double)t;
  }
  put_partial(part, vh, r, i, s);
}

// One block of kSumThreads threads per right-hand side.  Every thread adds its strided
// partials in 16 independent chains (16 loads in flight; the tail as predicated loads
// rather than a dependent loop), the chains are combined in a fixed tree, each wave
// folds its 64 values with lane shuffles, and one thread adds the 16 wave sums.  The
// order depends on nw only, so the sum of a right-hand side never depends on the batch.
constexpr int kSumThreads = 1024;
constexpr int kSumChains = 16;
__device__ __forceinline__ double block_sum_partials(const double* part, long nw) {
  __shared__ double red[kSumThreads / 64];
  double c[kSumChains];
#pragma unroll
  for (int k = 0; k < kSumChains; ++k) c[k] = 0.0;
  long w = threadIdx.x;
  for (; w + (kSumChains - 1) * kSumThreads < nw; w += kSumChains * kSumThreads) {
#pragma unroll
    for (int k = 0; k < kSumChains; ++k) c[k] += part[w + k * kSumThreads];
  }
#pragma unroll
  for (int k = 0; k < kSumChains - 1; ++k) {
    const long j = w + (long)k * kSumThreads;
    if (j < nw) c[k] += part[j];
  }
#pragma unroll
  for (int h = kSumChains / 2; h >= 1; h >>= 1)
#pragma unroll
    for (int k = 0; k < h; ++k) c[k] += c[k + h];
  double v = c[0];
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < kSumThreads / 64; ++k) s += red[k];
  }
  return s;  // valid in thread 0
}

__global__ void __launch_bounds__(kSumThreads) sum_partials_kernel(const double* part, long nw, double* out) {
  double s = block_sum_partials(part + (long)blockIdx.x * nw, nw);
  if (threadIdx.x == 0) out[blockIdx.x] = s;
}

template <int P>
__global__ void axpby_kernel(double a, Vec x, double b, Vec y, long vh, int nts) {
  using T = typename Real<P>::T;
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  int r = blockIdx.y;
  if (i >= vh) return;
  cx<T> xv[12], yv[12];
  SpinorIO<P>::load(static_cast<const char*>(x.p) + r * x.stride, vh, i, xv);
  char* yp = static_cast<char*>(y.p) + r * y.stride;
  SpinorIO<P>::load(yp, vh, i, yv);
#pragma unroll
  for (int c = 0; c < 12; ++c) yv[c] = T(a) * xv[c] + T(b) * yv[c];
  if (nts) SpinorIO<P>::template store<1>(yp, vh, i, yv);
  else SpinorIO<P>::template store<0>(yp, vh, i, yv);
}

template <int P>
__global__ void clover_apply_kernel(const void* clov, Vec in, Vec out, long vh) {
  using T = typename Real<P>::T;
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  int r = blockIdx.y;
  if (i >= vh) return;
  T cl[72];
  CloverIO<P>::load(clov, vh, i, cl);
  cx<T> v[12], o[12];
  SpinorIO<P>::load(static_cast<const char*>(in.p) + r * in.stride, vh, i, v);
  clover_mul(cl, v, o);
  SpinorIO<P>::store(static_cast<char*>(out.p) + r * out.stride, vh, i, o);
}

// ---------------------------------------------------------------- CGLS ------
__global__ void __launch_bounds__(kSumThreads) cg_beta_kernel(const double* part, long nw, CgScal* sc) {
  CgScal& s = sc[blockIdx.x];
  if (!s.active) return;
  double g = block_sum_partials(part + (long)blockIdx.x * nw, nw);
  if (threadIdx.x == 0) {
    if (s.first || s.converged || !(s.gamma > 0.0)) {
      s.beta = 0.0;
    } else {
      s.beta = g / s.gamma;
    }
    s.first = 0;
    s.gamma = g;
  }
}

__global__ void __launch_bounds__(kSumThreads) cg_alpha_kernel(const double* part, long nw, CgScal* sc) {
  CgScal& s = sc[blockIdx.x];
  if (!s.active) return;
  double tt = block_sum_partials(part + (long)blockIdx.x * nw, nw);
  if (threadIdx.x == 0) {
    s.tt = tt;
    if (s.converged) {
      s.alpha = 0.0;
    } else if (!(tt > 0.0) || !(s.gamma == s.gamma) || tt != tt || tt > 1.0e300) {
      s.alpha = 0.0;  // breakdown (p^dag Mhat^dag Mhat p <= 0 or not finite): freeze
      s.breakdown = 1;
    } else {
      s.alpha = s.gamma / tt;
    }
    s.gamma_old = s.gamma;  // for a later chunk whose vector kernels take the steps
  }
}

// host: the scalars as they leave the chunk, to the batch's pinned copy (a copy command
// and its hand-over from kernel to kernel take about 20 us)
__global__ void __launch_bounds__(kSumThreads) cg_ss_kernel(const double* part, long nw, CgScal* sc, CgScal* host) {
  CgScal& s = sc[blockIdx.x];
  if (s.active) {
    double ss = block_sum_partials(part + (long)blockIdx.x * nw, nw);
    if (threadIdx.x == 0) {
      if (!s.converged) {
        s.ss = ss;
        s.iter += 1;
        if (ss <= s.target2) s.converged = 1;
      }
    }
  }
  if (host && threadIdx.x == 0) host[blockIdx.x] = s;
}

// the way back, of n slots the host has changed
__global__ void cg_put_kernel(const CgScal* host, CgScal* sc, int n) {
  if ((int)threadIdx.x < n) sc[threadIdx.x] = host[threadIdx.x];
}

// The sum of a right-hand side's nw partials, by every block that needs it (256 threads, nw
// <= 1024 K), with the bits of block_sum_partials: thread u stands for its threads u + 256
// q, whose chains beyond K are empty, and the sixteen wave sums are added in its order.
constexpr int kStepThreads = 256;
template <int K>
__device__ __forceinline__ double step_sum(const double* part, long nw, double* red) {
  double v[kSumThreads / kStepThreads];
#pragma unroll
  for (int q = 0; q < kSumThreads / kStepThreads; ++q) {
    double c[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const long j = (long)threadIdx.x + q * kStepThreads + (long)k * kSumThreads;
      c[k] = j < nw ? part[j] : 0.0;
    }
#pragma unroll
    for (int h = K / 2; h >= 1; h >>= 1)
#pragma unroll
      for (int k = 0; k < h; ++k) c[k] += c[k + h];
    v[q] = c[0];
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1)
#pragma unroll
    for (int q = 0; q < kSumThreads / kStepThreads; ++q) v[q] += __shfl_xor(v[q], off, 64);
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int q = 0; q < kSumThreads / kStepThreads; ++q) red[(threadIdx.x >> 6) + q * (kStepThreads / 64)] = v[q];
  }
  __syncthreads();
  double sum = 0.0;
#pragma unroll
  for (int k = 0; k < kSumThreads / 64; ++k) sum += red[k];
  return sum;
}

// The beta step by every block of the p update: the sums of |r|^2 and, when the previous
// iteration's |s|^2 is still to be looked at (part_ss), of that; block 0 writes what the
// later steps read.  Nothing another block reads here is written here.
template <int K>
__device__ __forceinline__ double beta_step(CgScal& s, const double* part_rr, const double* part_ss, long nw,
                                            double (*red)[kSumThreads / 64]) {
  const double rr = step_sum<K>(part_rr, nw, red[0]);
  int conv = s.converged;
  double ss = 0.0;
  if (part_ss) {
    ss = step_sum<K>(part_ss, nw, red[1]);
    conv = conv || ss <= s.target2;
  }
  const double beta = s.first || conv || !(s.gamma_old > 0.0) ? 0.0 : rr / s.gamma_old;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (part_ss && !s.converged) {
      s.ss = ss;
      s.iter += 1;
    }
    s.conv_now = conv;
    s.beta = beta;
    s.gamma = rr;
  }
  return beta;
}

// the alpha step by every block of the s update, likewise
template <int K>
__device__ __forceinline__ double alpha_step(CgScal& s, const double* part_tt, long nw, double* red) {
  const double tt = step_sum<K>(part_tt, nw, red);
  const double g = s.gamma;
  const bool conv = s.conv_now, bad = !conv && (!(tt > 0.0) || g != g || tt != tt || tt > 1.0e300);
  const double alpha = conv || bad ? 0.0 : g / tt;  // breakdown freezes, as in cg_alpha_kernel
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    s.tt = tt;
    s.alpha = alpha;
    if (bad) s.breakdown = 1;
    s.converged = conv;
    s.gamma_old = g;
    s.first = 0;
  }
  return alpha;
}

// The share of a site that one thread of the two kernels below takes: half of it in FP64
// and FP32 (a wave takes one half of a 64-site chunk, so a launch has twice the waves and
// each keeps half the registers: 16^3x32 is otherwise one wave per SIMD), all of it in FP16.
// x and p update, s update, of 16^3x32 FP64 14.9 -> 12.7 and 9.6 -> 8.7 us, 8^4 FP32 5.5 ->
// 4.4 and 4.8 -> 3.8; 32^3x64 solves 3.3 % (FP32) and 4 % (FP16) faster.
template <int P>
struct Share {
  static constexpr int H = P == F16 ? 1 : 2, N = 12 / H;
  int h;
  long first, site;  // the chunk's first site, this thread's
  bool live;
  __device__ __forceinline__ explicit Share(long vh) {
    const long w = (long)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    h = (int)(w % H);
    first = w / H * 64;
    const long i = first + (threadIdx.x & 63);
    live = i < vh;
    site = live ? i : vh - 1;
  }
  static unsigned blocks(long vh) { return nblk((vh + 63) / 64 * H, 4); }
  template <int PX, typename T>
  __device__ __forceinline__ void load(const void* p, long vh, cx<T> v[N]) const {
    if constexpr (H == 2) SpinorIO<PX>::template load_half<1>(p, vh, site, h, v);
    else SpinorIO<PX>::load(p, vh, site, v);
  }
  template <int PX, typename T>
  __device__ __forceinline__ void store(void* p, long vh, const cx<T> v[N], int nts) const {
    if (!live) return;
    if constexpr (H == 2) {
      if (nts) SpinorIO<PX>::template store_half<1>(p, vh, site, h, v);
      else SpinorIO<PX>::template store_half<0>(p, vh, site, h, v);
    } else {
      if (nts) SpinorIO<PX>::template store<1>(p, vh, site, v);
      else SpinorIO<PX>::template store<0>(p, vh, site, v);
    }
  }
};

// x += alpha_k p_k of the previous iteration (still pending: alpha is that iteration's,
// p not yet overwritten), then p = r + beta p.  Folding the iterate update in here
// saves one read of p per iteration against doing it in the s update; the host
// applies a pending update itself (cg_xflush) before it reads x.  K > 0: the blocks take
// the beta step themselves (beta_step), while their fields load.
template <int P, int PX, int K>
__global__ void __launch_bounds__(256) cg_xpay_kernel(Vec r, Vec p, Vec x, CgScal* sc, const double* part_rr,
                                                      const double* part_ss, long nw, long vh, int nts) {
  using T = typename Real<P>::T;
  using TX = typename Real<PX>::T;
  constexpr int N = Share<P>::N;
  __shared__ double red[K ? 2 : 1][kSumThreads / 64];
  const Share<P> sh(vh);
  const int k = blockIdx.y;
  if (!sc[k].active) return;
  if (K == 0 && !sh.live) return;
  const double alpha = sc[k].alpha;
  char* pp = static_cast<char*>(p.p) + k * p.stride;
  char* xp = static_cast<char*>(x.p) + k * x.stride;
  const char* rp = static_cast<const char*>(r.p) + k * r.stride;
  cx<T> pv[N], rv[N];
  cx<TX> xv[N];
  T beta = K ? T(1) : T(sc[k].beta);
  if (alpha != 0.0 || beta != T(0)) sh.template load<P>(pp, vh, pv);
  if (alpha != 0.0) sh.template load<PX>(xp, vh, xv);
  sh.template load<P>(rp, vh, rv);
  if constexpr (K > 0)
    beta = T(beta_step<K>(sc[k], part_rr + k * nw, part_ss ? part_ss + k * nw : nullptr, nw, red));
  if (alpha != 0.0) {
    const TX ax = TX(alpha);
#pragma unroll
    for (int c = 0; c < N; ++c) xv[c] = {xv[c].re + ax * TX(pv[c].re), xv[c].im + ax * TX(pv[c].im)};
    sh.template store<PX>(xp, vh, xv, nts);
  }
  if (beta != T(0)) {  // else a restart (first iteration, after a restart, or converged): p = r
#pragma unroll
    for (int c = 0; c < N; ++c) rv[c] = rv[c] + beta * pv[c];
  }
  sh.template store<P>(pp, vh, rv, nts);
}

// s -= alpha t, with the 64-site partials of |s|^2, a chunk's two halves added by the wave
// of its first.  K > 0: the blocks take the alpha step themselves (alpha_step), while their
// fields load.
template <int P, int K>
__global__ void __launch_bounds__(256) cg_update_kernel(Vec t, Vec s, CgScal* sc, const double* part_tt, long nw,
                                                        double* part, long vh, int nts) {
  using T = typename Real<P>::T;
  constexpr int N = Share<P>::N;
  __shared__ double red[kSumThreads / 64], half[4];
  const Share<P> sh(vh);
  const int k = blockIdx.y;
  if (!sc[k].active) return;
  char* sp = static_cast<char*>(s.p) + k * s.stride;
  const char* tp = static_cast<const char*>(t.p) + k * t.stride;
  cx<T> tv[N], sv[N];
  sh.template load<P>(tp, vh, tv);
  sh.template load<P>(sp, vh, sv);
  T a;
  if constexpr (K > 0) a = T(alpha_step<K>(sc[k], part_tt + k * nw, nw, red));
  else a = T(sc[k].alpha);
  T n = T(0);
#pragma unroll
  for (int c = 0; c < N; ++c) {
    sv[c] = sv[c] - a * tv[c];
    n += norm2(sv[c]);
  }
  sh.template store<P>(sp, vh, sv, nts);
  double v = group64_sum(sh.live ? (double)n : 0.0);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if constexpr (Share<P>::H == 2) {
    if (lane == 0) half[w] = v;
    __syncthreads();
    if (sh.h == 0) v = half[w] + half[w | 1];
  }
  if (lane == 0 && sh.h == 0 && sh.first < vh) part[(long)k * nw + sh.first / 64] = v;
}

// x += alpha p for one slot of an FP64 loop: a pending iterate update applied by the host
__global__ void cg_xflush_kernel(Vec x, Vec p, double alpha, long vh) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= vh) return;
  cx<double> pv[12], xv[12];
  SpinorIO<F64>::load(p.p, vh, i, pv);
  SpinorIO<F64>::load(x.p, vh, i, xv);
#pragma unroll
  for (int c = 0; c < 12; ++c) xv[c] = {xv[c].re + alpha * pv[c].re, xv[c].im + alpha * pv[c].im};
  SpinorIO<F64>::store(x.p, vh, i, xv);
}

// The slots of a low-precision loop in `mask`: the pending update x += alpha p, xe += x in
// FP64, and x = 0, in one pass (24^3x48 FP16: 35 us, 50 in three passes).
template <int P>
__global__ void cg_fold_kernel(Vec x, Vec p, Vec xe, const SlotScal a, long vh, int nts) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int r = blockIdx.y;
  if (i >= vh || !((a.mask >> r) & 1u)) return;
  char* xp = static_cast<char*>(x.p) + r * x.stride;
  char* ep = static_cast<char*>(xe.p) + r * xe.stride;
  cx<float> xv[12], z[12];
  SpinorIO<F32>::load(xp, vh, i, xv);
  if (a.v[r] != 0.0) {
    cx<float> pv[12];
    SpinorIO<P>::load(static_cast<const char*>(p.p) + r * p.stride, vh, i, pv);
    const float ax = (float)a.v[r];
#pragma unroll
    for (int c = 0; c < 12; ++c) xv[c] = {xv[c].re + ax * pv[c].re, xv[c].im + ax * pv[c].im};
  }
#pragma unroll
  for (int c = 0; c < 12; ++c) z[c] = {0.f, 0.f};
  SpinorIO<F32>::store(xp, vh, i, z);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    cx<double> e[6];
    SpinorIO<F64>::load_half<1>(ep, vh, i, h, e);
#pragma unroll
    for (int c = 0; c < 6; ++c) e[c] = {e[c].re + (double)xv[6 * h + c].re, e[c].im + (double)xv[6 * h + c].im};
    if (nts) SpinorIO<F64>::store_half<1>(ep, vh, i, h, e);
    else SpinorIO<F64>::store_half<0>(ep, vh, i, h, e);
  }
}

// The FP64 residual b - t of the slots, its |.|^2 partials, and for those in `mask` its
// store to s in the loop's precision (t itself in an FP64 loop); nothing else is kept.
template <int P>
__global__ void residual_kernel(Vec b, Vec t, Vec s, unsigned mask, double* part, long vh) {
  using T = typename Real<P>::T;
  const long i0 = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int r = blockIdx.y;
  const bool live = i0 < vh;
  const long i = live ? i0 : vh - 1;
  cx<double> bv[12], tv[12];
  SpinorIO<F64>::load(static_cast<const char*>(b.p) + r * b.stride, vh, i, bv);
  SpinorIO<F64>::load(static_cast<const char*>(t.p) + r * t.stride, vh, i, tv);
  double n = 0.0;
#pragma unroll
  for (int c = 0; c < 12; ++c) {
    tv[c] = bv[c] - tv[c];
    n += norm2(tv[c]);
  }
  if (live && ((mask >> r) & 1u)) {
    cx<T> o[12];
#pragma unroll
    for (int c = 0; c < 12; ++c) o[c] = {T(tv[c].re), T(tv[c].im)};
    SpinorIO<P>::store(static_cast<char*>(s.p) + r * s.stride, vh, i, o);
  }
  put_partial(part, vh, r, i0, live ? n : 0.0);
}

// plain streaming copy, the bandwidth and PMC-counter reference kernel: one 16-byte
// element per lane over a full grid (on MI355X this moves about 6.2 TB/s at 1 GiB,
// where a grid-stride loop capped at 32 blocks per CU moves 4.5 TB/s)
__global__ void copy_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst, long n) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

void launch_copy(void* dst, const void* src, size_t bytes, hipStream_t st) {
  long n = (long)(bytes / 16);
  hipLaunchKernelGGL(copy_kernel, dim3(nblk(n, 256)), dim3(256), 0, st, static_cast<const uint4*>(src),
                     static_cast<uint4*>(dst), n);
}

// ------------------------------------------------------------- launchers ----
#define QCU_PSW(PV, K, ...)                                                      \
  do {                                                                           \
    if ((PV) == F64) hipLaunchKernelGGL(K<F64>, __VA_ARGS__);                    \
    else if ((PV) == F32) hipLaunchKernelGGL(K<F32>, __VA_ARGS__);               \
    else hipLaunchKernelGGL(K<F16>, __VA_ARGS__);                                \
  } while (0)

void launch_zero(int prec, Vec v, long vh, int nrhs, hipStream_t st) {
  QCU_PSW(prec, zero_kernel, dim3(nblk(vh, 256), nrhs), dim3(256), 0, st, v, vh);
}
void launch_norm2(int prec, Vec v, long vh, int nrhs, double* part, hipStream_t st) {
  QCU_PSW(prec, norm2_kernel, dim3(nblk(vh, 256), nrhs), dim3(256), 0, st, v, vh, part);
}
void launch_sum_partials(const double* part, long nw, int nrhs, double* out, hipStream_t st) {
  hipLaunchKernelGGL(sum_partials_kernel, dim3(nrhs), dim3(kSumThreads), 0, st, part, nw, out);
}
void launch_axpby(int prec, double a, Vec x, double b, Vec y, long vh, int nrhs, hipStream_t st) {
  QCU_PSW(prec, axpby_kernel, dim3(nblk(vh, 256), nrhs), dim3(256), 0, st, a, x, b, y, vh, nt_store(prec, vh, nrhs));
}
void launch_clover_apply(int prec, const void* clov, Vec in, Vec out, long vh, int nrhs, hipStream_t st) {
  QCU_PSW(prec, clover_apply_kernel, dim3(nblk(vh, 256), nrhs), dim3(256), 0, st, clov, in, out, vh);
}
void launch_cg_beta(const double* part, long nw, CgScal* sc, int nrhs, hipStream_t st) {
  hipLaunchKernelGGL(cg_beta_kernel, dim3(nrhs), dim3(kSumThreads), 0, st, part, nw, sc);
}
void launch_cg_alpha(const double* part, long nw, CgScal* sc, int nrhs, hipStream_t st) {
  hipLaunchKernelGGL(cg_alpha_kernel, dim3(nrhs), dim3(kSumThreads), 0, st, part, nw, sc);
}
void launch_cg_ss(const double* part, long nw, CgScal* sc, CgScal* host, int nrhs, hipStream_t st) {
  hipLaunchKernelGGL(cg_ss_kernel, dim3(nrhs), dim3(kSumThreads), 0, st, part, nw, sc, host);
}
void launch_cg_put(const CgScal* host, CgScal* sc, int n, hipStream_t st) {
  hipLaunchKernelGGL(cg_put_kernel, dim3(1), dim3(64), 0, st, host, sc, n);
}
void launch_cg_fold(int prec, Vec x, Vec p, Vec xe, const SlotScal& a, long vh, int nrhs, hipStream_t st) {
  const dim3 g(nblk(vh, 256), nrhs), b(256);
  const int nts = nt_store(F64, vh, nrhs);
  if (prec == F32) hipLaunchKernelGGL(cg_fold_kernel<F32>, g, b, 0, st, x, p, xe, a, vh, nts);
  else hipLaunchKernelGGL(cg_fold_kernel<F16>, g, b, 0, st, x, p, xe, a, vh, nts);
}
void launch_residual(int prec, Vec b, Vec t, Vec s, unsigned mask, long vh, int nrhs, double* part, hipStream_t st) {
  QCU_PSW(prec, residual_kernel, dim3(nblk(vh, 256), nrhs), dim3(256), 0, st, b, t, s, mask, part, vh);
}
// Every block sums all the partials, which costs nrhs nw^2 reads and saves two one-block
// launches and most of a third.  Solves with the steps apart and in the vector kernels
// (ms): 8^4 FP32 2.67 / 2.29, 16^3x32 FP64 16.61 / 15.58, FP32 7.97 / 7.32, 12 RHS 45.8 /
// 45.3, 16^3x64 6 RHS (nrhs nw^2 = 2.5e7) 53.3 / 52.6; but 24^3x48 (nw 5184) FP16 25.8 /
// 26.3, FP64 64.1 / 64.0, 4 RHS 102 / 106.
int cg_step_chains(long nw, int nrhs) {
  if (nw > 4 * kSumThreads || nrhs * nw * nw > 26000000) return 0;
  return nw <= kSumThreads ? 1 : 4;
}

template <int P, int PX>
static void xpay(Vec r, Vec p, Vec x, CgScal* sc, const double* part_rr, const double* part_ss, long nw, long vh,
                 int nrhs, hipStream_t st) {
  const dim3 g(Share<P>::blocks(vh), nrhs), b(256);
  const int n = nt_store(P, vh, nrhs);  // p decides for x as well
  const int k = part_rr ? cg_step_chains(nw, nrhs) : 0;
  if (k == 1) hipLaunchKernelGGL((cg_xpay_kernel<P, PX, 1>), g, b, 0, st, r, p, x, sc, part_rr, part_ss, nw, vh, n);
  else if (k) hipLaunchKernelGGL((cg_xpay_kernel<P, PX, 4>), g, b, 0, st, r, p, x, sc, part_rr, part_ss, nw, vh, n);
  else hipLaunchKernelGGL((cg_xpay_kernel<P, PX, 0>), g, b, 0, st, r, p, x, sc, part_rr, part_ss, nw, vh, n);
}
void launch_cg_xpay(int prec, int xprec, Vec r, Vec p, Vec x, CgScal* sc, const double* part_rr,
                    const double* part_ss, long nw, long vh, int nrhs, hipStream_t st) {
  if (prec == F64) xpay<F64, F64>(r, p, x, sc, part_rr, part_ss, nw, vh, nrhs, st);
  else if (prec == F32) xpay<F32, F32>(r, p, x, sc, part_rr, part_ss, nw, vh, nrhs, st);
  else xpay<F16, F32>(r, p, x, sc, part_rr, part_ss, nw, vh, nrhs, st);
}
void launch_cg_xflush(Vec x, Vec p, double alpha, long vh, hipStream_t st) {
  hipLaunchKernelGGL(cg_xflush_kernel, dim3(nblk(vh, 256)), dim3(256), 0, st, x, p, alpha, vh);
}
template <int P>
static void update(Vec t, Vec s, CgScal* sc, const double* part_tt, long nw, double* part, long vh, int nrhs,
                   hipStream_t st) {
  const dim3 g(Share<P>::blocks(vh), nrhs), b(256);
  const int n = nt_store(P, vh, nrhs);
  const int k = part_tt ? cg_step_chains(nw, nrhs) : 0;
  if (k == 1) hipLaunchKernelGGL((cg_update_kernel<P, 1>), g, b, 0, st, t, s, sc, part_tt, nw, part, vh, n);
  else if (k) hipLaunchKernelGGL((cg_update_kernel<P, 4>), g, b, 0, st, t, s, sc, part_tt, nw, part, vh, n);
  else hipLaunchKernelGGL((cg_update_kernel<P, 0>), g, b, 0, st, t, s, sc, part_tt, nw, part, vh, n);
}
void launch_cg_update(int prec, Vec t, Vec s, CgScal* sc, const double* part_tt, long nw, double* part_ss, long vh,
                      int nrhs, hipStream_t st) {
  if (prec == F64) update<F64>(t, s, sc, part_tt, nw, part_ss, vh, nrhs, st);
  else if (prec == F32) update<F32>(t, s, sc, part_tt, nw, part_ss, vh, nrhs, st);
  else update<F16>(t, s, sc, part_tt, nw, part_ss, vh, nrhs, st);
}

}  // namespace qcu
