// k_layout.hip -- conversions between the interface layouts (complex128 AoS, as the
// reference's entry points take them: include/qcu_point.cuh:65-72) and the internal
// SoA layouts of each precision, plus precision conversions between internal fields.
// Role of src/qcu_shift_storage.cu:74-194 (AoS <-> SoA, gauge packing); written for
// wave64 with one thread per site.
#include "qcu_fields.h"
#include "qcu_kernels.h"

namespace qcu {

static inline unsigned nblk(long n, int b) { return (unsigned)((n + b - 1) / b); }

template <int P>
__global__ void spinor_from_aos_kernel(const double2* aos, long aos_stride, Vec out, long vh) {
  using T = typename Real<P>::T;
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  int r = blockIdx.y;
  if (i >= vh) return;
  const double2* s = reinterpret_cast<const double2*>(reinterpret_cast<const char*>(aos) + r * aos_stride) + i * 12;
  cx<T> v[12];
#pragma unroll
  for (int c = 0; c < 12; ++c) {
    double2 q = s[c];
    v[c] = {T(q.x), T(q.y)};
  }
  SpinorIO<P>::store(static_cast<char*>(out.p) + r * out.stride, vh, i, v);
}

template <int P>
__global__ void spinor_to_aos_kernel(Vec in, double2* aos, long aos_stride, long vh) {
  using T = typename Real<P>::T;
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  int r = blockIdx.y;
  if (i >= vh) return;
  cx<T> v[12];
  SpinorIO<P>::load_cached(static_cast<const char*>(in.p) + r * in.stride, vh, i, v);
  double2* d = reinterpret_cast<double2*>(reinterpret_cast<char*>(aos) + r * aos_stride) + i * 12;
#pragma unroll
  for (int c = 0; c < 12; ++c) d[c] = double2{(double)v[c].re, (double)v[c].im};
}

void launch_spinor_from_aos(int prec, const void* aos, long aos_stride, Vec out, long vh, int nrhs, hipStream_t st) {
  dim3 grid(nblk(vh, 256), nrhs);
  const double2* a = static_cast<const double2*>(aos);
  if (prec == F64) hipLaunchKernelGGL(spinor_from_aos_kernel<F64>, grid, dim3(256), 0, st, a, aos_stride, out, vh);
  else if (prec == F32) hipLaunchKernelGGL(spinor_from_aos_kernel<F32>, grid, dim3(256), 0, st, a, aos_stride, out, vh);
  else hipLaunchKernelGGL(spinor_from_aos_kernel<F16>, grid, dim3(256), 0, st, a, aos_stride, out, vh);
}

void launch_spinor_to_aos(int prec, Vec in, void* aos, long aos_stride, long vh, int nrhs, hipStream_t st) {
  dim3 grid(nblk(vh, 256), nrhs);
  double2* a = static_cast<double2*>(aos);
  if (prec == F64) hipLaunchKernelGGL(spinor_to_aos_kernel<F64>, grid, dim3(256), 0, st, in, a, aos_stride, vh);
  else if (prec == F32) hipLaunchKernelGGL(spinor_to_aos_kernel<F32>, grid, dim3(256), 0, st, in, a, aos_stride, vh);
  else hipLaunchKernelGGL(spinor_to_aos_kernel<F16>, grid, dim3(256), 0, st, in, a, aos_stride, vh);
}

// one link, 9 complex row-major in u, to its packed words (the layout LinkIO reads)
template <int P, int R>
__device__ __forceinline__ void store_link(void* out, long vh, int mp, long i, const double2 u[9]) {
  constexpr int NE = R == 12 ? 6 : 9;
  static_assert(LinkLayout<F32, 12>::blocked && LinkLayout<F32, 18>::blocked && LinkLayout<F16, 12>::blocked &&
                    LinkLayout<F16, 18>::blocked,
                "the FP32 and FP16 stores below step by kSiteBlock");
  auto half2 = [](double2 z) { return (unsigned)f2h((float)z.x) | ((unsigned)f2h((float)z.y) << 16); };
  if constexpr (P == F64) {
    double2* d = link_word<F64, R>(static_cast<double2*>(out), vh, mp, i);
    const long ws = link_stride<F64, R>(vh);
#pragma unroll
    for (int e = 0; e < NE; ++e) d[e * ws] = u[e];
  } else if constexpr (P == F32 && R == 12) {
    float4* d = link_word<F32, 12>(static_cast<float4*>(out), vh, mp, i);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      d[k * kSiteBlock] = float4{(float)u[2 * k].x, (float)u[2 * k].y, (float)u[2 * k + 1].x, (float)u[2 * k + 1].y};
  } else if constexpr (P == F32) {
    float2* d = link_word<F32, 18>(static_cast<float2*>(out), vh, mp, i);
#pragma unroll
    for (int e = 0; e < 9; ++e) d[e * kSiteBlock] = float2{(float)u[e].x, (float)u[e].y};
  } else if constexpr (R == 12) {
    uint2* d = link_word<F16, 12>(static_cast<uint2*>(out), vh, mp, i);
#pragma unroll
    for (int k = 0; k < 3; ++k) d[k * kSiteBlock] = uint2{half2(u[2 * k]), half2(u[2 * k + 1])};
  } else {
    unsigned* d = link_word<F16, 18>(static_cast<unsigned*>(out), vh, mp, i);
#pragma unroll
    for (int e = 0; e < 9; ++e) d[e * kSiteBlock] = half2(u[e]);
  }
}

// ------------------------------------------------------------ fingerprint ---
// A 64-bit fingerprint of rows 0-1 of a gauge's links: the sum (mod 2^64) over their
// 64-bit words w_i, i the word's place in the gauge, of mix(w_i ^ (i * 0x9E3779B97F4A7C15)),
// mix being the splitmix64 finaliser (Steele, Lea and Flood, OOPSLA 2014).  A sum of
// integers does not depend on the order it is taken in, so the result is the same for any
// launch shape, and a change of any one word changes it except with probability about
// 2^-64.  Used by the drop-in entry points, which rebuild row 2 and so never read it, to
// notice a gauge the caller changed in place (16^3x32: 14.8 us, 21.3 + 3.8 over all nine
// words and with a kernel for the sum).
__device__ __forceinline__ uint64_t fp_mix(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
// of the complex number q at 16-byte word j of the gauge
__device__ __forceinline__ uint64_t fp_word(double2 q, long j) {
  constexpr uint64_t K = 0x9E3779B97F4A7C15ull;
  const uint64_t k = (uint64_t)(2 * j) * K;
  return fp_mix(__builtin_bit_cast(uint64_t, q.x) ^ k) + fp_mix(__builtin_bit_cast(uint64_t, q.y) ^ (k + K));
}

__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    unsigned lo = (unsigned)v, hi = (unsigned)(v >> 32);
    lo = __shfl_xor(lo, off, 64);
    hi = __shfl_xor(hi, off, 64);
    v += ((uint64_t)hi << 32) | lo;
  }
  return v;
}
// the block's sum to its word of `parts`, host memory: the host adds the words after the
// synchronisation it needs anyway, which saves a kernel and a copy
__device__ __forceinline__ void put_fingerprint(uint64_t h, uint64_t* parts, uint64_t* red) {
  h = wave_sum_u64(h);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = h;
  __syncthreads();
  if (threadIdx.x == 0) parts[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// gauge: a wave takes 64 links of one (mu, parity) field at a time as one run of 576
// 16-byte words through its LDS tile (a lane then reads its own 9-word record: odd stride,
// no bank conflicts), because a lane reading its own record from memory asks for 64 lines
// per load: 16^3x32 FP64 recon-18 54 us that way, 29 this way (5.2 TB/s), 24^3x48 273 and
// 150.  FP: with the fingerprint of rows 0-1 as they pass.
template <int P, int R, int FP>
__global__ void __launch_bounds__(256) gauge_pack_kernel(const double2* aos, void* out, long vh, uint64_t* parts) {
  __shared__ double2 tile[4][576];
  __shared__ uint64_t red[4];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const long nch = (vh + 63) / 64, units = 8 * nch;
  double2* T = tile[wv];
  uint64_t h = 0;
  for (long u = (long)blockIdx.x * 4 + wv; u < units; u += (long)gridDim.x * 4) {
    const int mp = (int)(u / nch);  // mu * 2 + parity
    const long l0 = (u - mp * nch) * 64;
    const int n = (int)(vh - l0 < 64 ? vh - l0 : 64);
    const long w0 = ((long)mp * vh + l0) * 9;
    double2 q[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      const int f = k * 64 + lane;
      q[k] = f < 9 * n ? aos[w0 + f] : double2{0.0, 0.0};
    }
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      const int f = k * 64 + lane;
      if (FP && f < 9 * n && f % 9 < 6) h += fp_word(q[k], w0 + f);
      T[f] = q[k];
    }
    wave_sync();
    if (lane < n) {
      double2 v[9];
#pragma unroll
      for (int e = 0; e < (R == 12 ? 6 : 9); ++e) v[e] = T[lane * 9 + e];
      store_link<P, R>(out, vh, mp, l0 + lane, v);
    }
    wave_sync();  // the tile is free again
  }
  if (FP) put_fingerprint(h, parts, red);
}

void launch_gauge_pack(int prec, int recon, const void* aos, void* out, long vh, hipStream_t st) {
  const dim3 grid(nblk(8 * ((vh + 63) / 64), 4));
  const double2* a = static_cast<const double2*>(aos);
#define QCU_GP(P, R)                                                                                  \
  if (prec == P && recon == R) {                                                                      \
    hipLaunchKernelGGL((gauge_pack_kernel<P, R, 0>), grid, dim3(256), 0, st, a, out, vh, (uint64_t*)nullptr); \
    return;                                                                                           \
  }
  QCU_GP(F64, 18) QCU_GP(F64, 12) QCU_GP(F32, 18) QCU_GP(F32, 12) QCU_GP(F16, 18) QCU_GP(F16, 12)
#undef QCU_GP
}

void launch_gauge_import(const void* aos, void* out, uint64_t* parts, long vh, hipStream_t st) {
  hipLaunchKernelGGL((gauge_pack_kernel<F64, 12, 1>), dim3(kFingerprintBlocks), dim3(256), 0, st,
                     static_cast<const double2*>(aos), out, vh, parts);
}

__global__ void __launch_bounds__(256) fingerprint_kernel(const double2* __restrict__ aos, long nlinks,
                                                          uint64_t* parts) {
  __shared__ uint64_t red[4];
  uint64_t h = 0;
  const long stride = (long)gridDim.x * blockDim.x;
#pragma unroll 4
  for (long j = (long)blockIdx.x * blockDim.x + threadIdx.x; j < nlinks * 6; j += stride) {
    const long l = j / 6, w = l * 9 + (j - l * 6);
    h += fp_word(aos[w], w);
  }
  put_fingerprint(h, parts, red);
}

void launch_fingerprint(const void* aos, uint64_t* parts, long vh, hipStream_t st) {
  hipLaunchKernelGGL(fingerprint_kernel, dim3(kFingerprintBlocks), dim3(256), 0, st,
                     static_cast<const double2*>(aos), 8 * vh, parts);
}

// packed FP64 rows 0-1 (recon-12) -> FP32 or FP16
template <int P>
__global__ void gauge_repack_kernel(const double2* rows, void* out, long vh) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int mp = blockIdx.y;
  if (i >= vh) return;
  const double2* b = link_word<F64, 12>(rows, vh, mp, i);
  double2 v[9];
#pragma unroll
  for (int e = 0; e < 6; ++e) v[e] = ld_nt(b + e * kSiteBlock);
  store_link<P, 12>(out, vh, mp, i, v);
}

void launch_gauge_repack(int prec, const void* rows, void* out, long vh, hipStream_t st) {
  const dim3 grid(nblk(vh, 256), 8);
  const double2* r = static_cast<const double2*>(rows);
  if (prec == F32) hipLaunchKernelGGL(gauge_repack_kernel<F32>, grid, dim3(256), 0, st, r, out, vh);
  else hipLaunchKernelGGL(gauge_repack_kernel<F16>, grid, dim3(256), 0, st, r, out, vh);
}

// ----------------------------------------------- reference storage shifts ---
// AoS <-> the reference's coalesced SoA (src/qcu_shift_storage.cu:74-161): an AoS
// record of `wa` doubles per site becomes `w` planes of n doubles (plane e holds
// element e of every site).  A block moves 64 sites through an LDS tile, so both the
// record reads and the plane writes are contiguous runs; blockIdx.y picks the field
// (the 8 (mu, parity) link fields of a gauge, or 1 for a half spinor).
constexpr int kTile = 64, kTilePad = kTile + 1, kTileMaxW = 24;

__global__ void __launch_bounds__(256) aos_to_soa_kernel(const double* src, double* dst, long n, int wa, int w,
                                                         long src_field, long dst_field) {
  __shared__ double tile[kTileMaxW * kTilePad];
  long s0 = (long)blockIdx.x * kTile;
  int ns = (int)min((long)kTile, n - s0);
  src += blockIdx.y * src_field + s0 * wa;
  dst += blockIdx.y * dst_field + s0;
  for (int j = threadIdx.x; j < ns * wa; j += blockDim.x) {
    int e = j % wa, s = j / wa;
    if (e < w) tile[e * kTilePad + s] = src[j];
  }
  __syncthreads();
  for (int j = threadIdx.x; j < kTile * w; j += blockDim.x) {
    int e = j / kTile, s = j % kTile;
    if (s < ns) dst[e * n + s] = tile[e * kTilePad + s];
  }
}

// the way back; RECON rebuilds link row 2 = conj(row0 x row1) from the 12 stored reals
template <bool RECON>
__global__ void __launch_bounds__(256) soa_to_aos_kernel(const double* src, double* dst, long n, int w, int wa,
                                                         long src_field, long dst_field) {
  __shared__ double tile[kTileMaxW * kTilePad];
  long s0 = (long)blockIdx.x * kTile;
  int ns = (int)min((long)kTile, n - s0);
  src += blockIdx.y * src_field + s0;
  dst += blockIdx.y * dst_field + s0 * wa;
  for (int j = threadIdx.x; j < kTile * w; j += blockDim.x) {
    int e = j / kTile, s = j % kTile;
    if (s < ns) tile[e * kTilePad + s] = src[e * n + s];
  }
  __syncthreads();
  if (RECON) {
    if ((int)threadIdx.x < ns) {
      int s = threadIdx.x;
      cx<double> u[9];
#pragma unroll
      for (int e = 0; e < 6; ++e) u[e] = {tile[(2 * e) * kTilePad + s], tile[(2 * e + 1) * kTilePad + s]};
      recon_row2(u);
#pragma unroll
      for (int e = 6; e < 9; ++e) {
        tile[(2 * e) * kTilePad + s] = u[e].re;
        tile[(2 * e + 1) * kTilePad + s] = u[e].im;
      }
    }
    __syncthreads();
  }
  for (int j = threadIdx.x; j < ns * wa; j += blockDim.x) dst[j] = tile[(j % wa) * kTilePad + j / wa];
}

void launch_shift_storage(int kind, int to_soa, const void* src, void* dst, long vh, hipStream_t st) {
  // kind 0: half spinor [Vh][24] <-> [24][Vh]; kind 1: gauge [8][Vh][18] <-> [8][12][Vh]
  int wa = kind == 0 ? 24 : 18, w = kind == 0 ? 24 : 12, nf = kind == 0 ? 1 : 8;
  dim3 grid(nblk(vh, kTile), nf);
  const double* s = static_cast<const double*>(src);
  double* d = static_cast<double*>(dst);
  if (to_soa)
    hipLaunchKernelGGL(aos_to_soa_kernel, grid, dim3(256), 0, st, s, d, vh, wa, w, vh * wa, vh * w);
  else if (kind == 0)
    hipLaunchKernelGGL(soa_to_aos_kernel<false>, grid, dim3(256), 0, st, s, d, vh, w, wa, vh * w, vh * wa);
  else
    hipLaunchKernelGGL(soa_to_aos_kernel<true>, grid, dim3(256), 0, st, s, d, vh, w, wa, vh * w, vh * wa);
}

// ------------------------------------------- lexicographic <-> even-odd ---
// lexicographic site l = ((t*Lz + z)*Ly + y)*Lx + x  <->  even-odd (parity, l/2) with
// parity = (x+y+z+t) mod 2, the half-site order of include/qcu_point.cuh:20-93.  One
// thread per 16-byte complex of a site record (NC complex per site), so consecutive
// lanes move consecutive bytes of the lexicographic field; blockIdx.y picks the field.
// The launcher guarantees vol < 2^31, the range of FastDiv.  NTL, NTS: streamed past the
// caches, loads and stores.
template <bool TO_EO, int NC, int NTL, int NTS>
__global__ void lex_eo_kernel(const double2* src, double2* dst, long vol, FastDiv dlx, FastDiv dly, FastDiv dlz,
                              long field) {
  long j = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= vol * NC) return;
  uint32_t l = (uint32_t)(j / NC);
  int k = (int)(j - (long)l * NC);
  uint32_t r = dlx.div(l), x = l - r * dlx.d;
  uint32_t r2 = dly.div(r), y = r - r2 * dly.d;
  uint32_t t = dlz.div(r2), z = r2 - t * dlz.d;
  uint32_t parity = (x + y + z + t) & 1u;
  long e = (long)parity * (vol / 2) + (l >> 1);
  src += blockIdx.y * field;
  dst += blockIdx.y * field;
  if (TO_EO) stp<NTS>(dst + e * NC + k, ldp<NTL>(src + (long)l * NC + k));
  else stp<NTS>(dst + (long)l * NC + k, ldp<NTL>(src + e * NC + k));
}

// A spinor of more than 128 MiB, which overflows the Infinity Cache together with its copy,
// is streamed past it (24^3x64 there and back 139 -> 132 us).  Up to there an even-odd one
// stays in it for what reads it next, and of those above 64 MiB the lexicographic output,
// which the library does not read again, is streamed: there and back with a hop between
// them, through the caches / both sides streamed / this: 24^3x32 (85 MB) 123 / 133 / 126,
// 24^3x48 (127 MB) 163 / 179 / 169, without the hop 73 / 79 / 74 and 100 / 105 / 97.  A gauge is
// streamed above 64 MiB: three states in turn of a gauge and two spinors, through the caches /
// this: 16^3x32 83 / 78, 16^3x48 105 / 97, 24^3x48 254 / 246.
void launch_lex_eo(int to_eo, const void* src, void* dst, const int L[4], int nc, int nfields, hipStream_t st) {
  long vol = (long)L[0] * L[1] * L[2] * L[3];
  long n = vol * nc;
  dim3 grid(nblk(n, 256), nfields);
  const double2* s = static_cast<const double2*>(src);
  double2* d = static_cast<double2*>(dst);
  FastDiv dlx((uint32_t)L[0]), dly((uint32_t)L[1]), dlz((uint32_t)L[2]);
  const size_t bytes = (size_t)n * nfields * 16;
  const bool half = bytes > kNtStoreBytes / 2;
  const int ntl = nc == 12 ? bytes > kNtStoreBytes : half, nts = ntl || (!to_eo && half);
#define QCU_LEX(E, N, NTL, NTS)                                                                                       \
  if (to_eo == E && nc == N && ntl == NTL && nts == NTS) {                                                            \
    hipLaunchKernelGGL((lex_eo_kernel<E, N, NTL, NTS>), grid, dim3(256), 0, st, s, d, vol, dlx, dly, dlz, n);         \
    return;                                                                                                           \
  }
  QCU_LEX(1, 12, 0, 0) QCU_LEX(1, 12, 1, 1) QCU_LEX(0, 12, 0, 0) QCU_LEX(0, 12, 0, 1) QCU_LEX(0, 12, 1, 1)
  QCU_LEX(1, 9, 0, 0) QCU_LEX(1, 9, 1, 1) QCU_LEX(0, 9, 0, 0) QCU_LEX(0, 9, 1, 1)
#undef QCU_LEX
}

// FP64 field -> internal layout of another precision (or a copy)
template <int P>
__global__ void spinor_convert_kernel(Vec in, Vec out, long vh) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  int r = blockIdx.y;
  if (i >= vh) return;
  using T = typename Real<P>::T;
  cx<double> a[12];
  SpinorIO<F64>::load(static_cast<const char*>(in.p) + r * in.stride, vh, i, a);
  cx<T> b[12];
#pragma unroll
  for (int c = 0; c < 12; ++c) b[c] = {T(a[c].re), T(a[c].im)};
  SpinorIO<P>::store(static_cast<char*>(out.p) + r * out.stride, vh, i, b);
}

void launch_spinor_convert(Vec in, int prec, Vec out, long vh, int nrhs, hipStream_t st) {
  const dim3 grid(nblk(vh, 256), nrhs);
  if (prec == F64) hipLaunchKernelGGL(spinor_convert_kernel<F64>, grid, dim3(256), 0, st, in, out, vh);
  else if (prec == F32) hipLaunchKernelGGL(spinor_convert_kernel<F32>, grid, dim3(256), 0, st, in, out, vh);
  else hipLaunchKernelGGL(spinor_convert_kernel<F16>, grid, dim3(256), 0, st, in, out, vh);
}

}  // namespace qcu
