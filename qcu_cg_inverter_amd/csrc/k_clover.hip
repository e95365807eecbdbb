// k_clover.hip -- clover term A = 1 + ck T and its inverse, per chiral 6x6 block.
//
// T(x) = -(1/8) sum_{mu<nu} (g_mu g_nu) (x) (Q_munu - Q_munu^dag) with Q the sum of the
// four plaquette leaves at x (reference: src/qcu_clover_dslash.cu:329-458 leaves and
// sum, :210-267 the g_mu g_nu table with factor -1/16 * 2, :537-540 A = 1 + T).
// The reference reads the off-origin links from 32 shifted copies of the gauge
// (src/qcu_communicator.cu:1270-1297); here every link is read from the one packed
// gauge at its neighbour coordinate.  The reference inverts with unpivoted
// Gauss-Jordan (src/qcu_clover_dslash.cu:42-100); here Cholesky in FP64, with a
// partially pivoted Gauss-Jordan fallback for blocks that are not positive definite
// (they occur at the reference normalisation ck = 1 on rough gauges).
#include "qcu_fields.h"
#include "qcu_kernels.h"

namespace qcu {

typedef cx<double> zd;

static inline unsigned nblk(long n, int b) { return (unsigned)((n + b - 1) / b); }

// U_dir at site c + dm e_mu + dn e_nu (dm, dn in -1, 0, 1)
template <int R>
__device__ __forceinline__ void load_link_at(const void* g, const Geom& geo, const int c[4], int mu, int nu, int dm,
                                             int dn, int dir, zd u[9]) {
  int x[4];
  int par = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    int v = c[k] + (k == mu ? dm : 0) + (k == nu ? dn : 0);
    v = v < 0 ? v + geo.L[k] : (v >= geo.L[k] ? v - geo.L[k] : v);
    x[k] = v;
    par ^= v & 1;
  }
  const long idx = x[3] * geo.st + x[2] * geo.sz + x[1] * geo.sy + (x[0] >> 1);
  LinkIO<F64, R>::template load<0>(g, geo.vh, dir, par, idx, u);
}

// r = a b and a b^dag; r must not alias a or b
__device__ __forceinline__ void mul_nn(zd r[9], const zd a[9], const zd b[9]) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      r[i * 3 + j] = cmad(a[i * 3 + 2], b[6 + j], cmad(a[i * 3 + 1], b[3 + j], a[i * 3] * b[j]));
}
__device__ __forceinline__ void mul_nd(zd r[9], const zd a[9], const zd b[9]) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      r[i * 3 + j] = cmadc(b[j * 3 + 2], a[i * 3 + 2], cmadc(b[j * 3 + 1], a[i * 3 + 1], mulc(a[i * 3], b[j * 3])));
}
// r -= a^dag b and r += a b
__device__ __forceinline__ void sub_dn(zd r[9], const zd a[9], const zd b[9]) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      r[i * 3 + j] =
          r[i * 3 + j] - cmadc(a[6 + i], b[6 + j], cmadc(a[3 + i], b[3 + j], mulc(b[j], a[i])));
}
__device__ __forceinline__ void add_nn(zd r[9], const zd a[9], const zd b[9]) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      r[i * 3 + j] =
          r[i * 3 + j] + cmad(a[i * 3 + 2], b[6 + j], cmad(a[i * 3 + 1], b[3 + j], a[i * 3] * b[j]));
}

// G = Q - Q^dag of plane (mu, nu) at site c, Q the sum of the four leaves
//   U_mu(x) S1, S1 = U_nu(x+mu) U_mu(x+nu)^dag U_nu(x)^dag
//   S2 U_mu(x-mu), S2 = U_nu(x) U_mu(x-mu+nu)^dag U_nu(x-mu)^dag
//   U_mu(x-mu)^dag S3, S3 = U_nu(x-mu-nu)^dag U_mu(x-mu-nu) U_nu(x-nu)
//   S4 U_mu(x)^dag, S4 = U_nu(x-nu)^dag U_mu(x-nu) U_nu(x-nu+mu)
// as D - D^dag with D = U_mu(x) (S1 - S4^dag) + (S2 - S3^dag) U_mu(x-mu): ten matrix
// products and twelve links.  G is anti-Hermitian: out holds the imaginary diagonal, then
// the entries (1,0) (2,0) (2,1) below it.
template <int R>
__device__ __forceinline__ void plane_field(const void* gauge, const Geom& geo, const int c[4], int mu, int nu,
                                            double out[9]) {
  auto at = [&](int dm, int dn, int dir, zd u[9]) { load_link_at<R>(gauge, geo, c, mu, nu, dm, dn, dir, u); };
  zd a[9], b[9], t[9], d[9], r[9];  // at most four of them live
  at(0, 0, nu, a); at(0, 1, mu, b); mul_nn(t, a, b);     // U_nu(x) U_mu(x+nu)
  at(1, 0, nu, b); mul_nd(d, b, t);                      // S1
  at(0, -1, mu, a); at(1, -1, nu, b); mul_nn(t, a, b);   // U_mu(x-nu) U_nu(x-nu+mu)
  at(0, -1, nu, a); sub_dn(d, t, a);                     // S1 - S4^dag
  at(0, 0, mu, a); mul_nn(r, a, d);
  at(-1, 0, nu, a); at(-1, 1, mu, b); mul_nn(t, a, b);   // U_nu(x-mu) U_mu(x-mu+nu)
  at(0, 0, nu, a); mul_nd(d, a, t);                      // S2
  at(-1, -1, mu, a); at(0, -1, nu, b); mul_nn(t, a, b);  // U_mu(x-mu-nu) U_nu(x-nu)
  at(-1, -1, nu, a); sub_dn(d, t, a);                    // S2 - S3^dag
  at(-1, 0, mu, a); add_nn(r, d, a);
#pragma unroll
  for (int k = 0; k < 3; ++k) out[k] = r[4 * k].im + r[4 * k].im;
  const zd g10 = r[3] - conj(r[1]), g20 = r[6] - conj(r[2]), g21 = r[7] - conj(r[5]);
  out[3] = g10.re; out[4] = g10.im; out[5] = g20.re; out[6] = g20.im; out[7] = g21.re; out[8] = g21.im;
}

// g_mu g_nu entries per plane: phase i^k by row spin; planes 0 and 5 couple a spin to
// itself, the others the two spins of a chiral block (the reference's table)
__device__ constexpr int CL_PH[6][4] = {{3, 1, 3, 1}, {2, 0, 2, 0}, {1, 1, 3, 3}, {3, 3, 3, 3}, {2, 0, 0, 2}, {1, 3, 3, 1}};

// a packed Hermitian 6x6 block: real diagonal d, entry (i, j) below it at
// l[i (i - 1) / 2 + j]
struct Block6 {
  double d[6];
  zd l[15];
  __device__ __forceinline__ zd& at(int i, int j) { return l[i * (i - 1) / 2 + j]; }
};

// plane fields of one site in LDS, [plane][9 reals][64 lanes]
typedef double PlaneLds[6][9][64];
__device__ __forceinline__ zd plane_entry(const PlaneLds& G, int pl, int lane, int i, int j) {
  if (i == j) return {0.0, G[pl][i][lane]};
  const int k = 3 + 2 * (i + j - 1);
  const double re = G[pl][k][lane], im = G[pl][k + 1][lane];
  return i > j ? zd{re, im} : zd{-re, im};
}

// chiral block B of 1 + ck T
template <int B>
__device__ __forceinline__ void assemble_block(const PlaneLds& G, int lane, double ck, Block6& m) {
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    constexpr int planes[2] = {0, 5};
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j <= i; ++j) {
        zd v = {0.0, 0.0};
#pragma unroll
        for (int p = 0; p < 2; ++p)
          v = v + -0.125 * iph(plane_entry(G, planes[p], lane, i, j), CL_PH[planes[p]][2 * B + s]);
        if (i == j) m.d[3 * s + i] = 1.0 + ck * v.re;
        else m.at(3 * s + i, 3 * s + j) = ck * v;
      }
  }
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      zd v = {0.0, 0.0};
#pragma unroll
      for (int pl = 1; pl < 5; ++pl) v = v + -0.125 * iph(plane_entry(G, pl, lane, i, j), CL_PH[pl][2 * B + 1]);
      m.at(3 + i, j) = ck * v;
    }
}

// Inverse of a Hermitian 6x6 in place by Cholesky, W = L^-1, W^dag W; every step
// overwrites only entries no later step reads, so the block never leaves 72 registers.
// false, with the block spoilt, if it is not positive definite.
__device__ __forceinline__ bool chol_inv6(Block6& m) {
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    double d = m.d[j];
#pragma unroll
    for (int k = 0; k < j; ++k) d -= norm2(m.at(j, k));
    if (!(d > 0.0)) return false;
    m.d[j] = 1.0 / sqrt(d);  // 1 / l_jj from here on
#pragma unroll
    for (int i = j + 1; i < 6; ++i) {
      zd s = m.at(i, j);
#pragma unroll
      for (int k = 0; k < j; ++k) s = s - mulc(m.at(i, k), m.at(j, k));
      m.at(i, j) = m.d[j] * s;
    }
  }
#pragma unroll
  for (int j = 0; j < 6; ++j)
#pragma unroll
    for (int i = j + 1; i < 6; ++i) {
      zd s = m.d[j] * m.at(i, j);
#pragma unroll
      for (int k = j + 1; k < i; ++k) s = s + m.at(i, k) * m.at(k, j);
      m.at(i, j) = (-m.d[i]) * s;
    }
#pragma unroll
  for (int i = 0; i < 6; ++i) {
#pragma unroll
    for (int j = 0; j < i; ++j) {
      zd s = m.d[i] * m.at(i, j);
#pragma unroll
      for (int k = i + 1; k < 6; ++k) s = s + mulc(m.at(k, j), m.at(k, i));
      m.at(i, j) = s;
    }
    double s = m.d[i] * m.d[i];
#pragma unroll
    for (int k = i + 1; k < 6; ++k) s += norm2(m.at(k, i));
    m.d[i] = s;
  }
  return true;
}

// Gauss-Jordan with partial pivoting (any nonsingular 6x6)
// of the packed block, for the rare blocks that are not positive definite; out of line, so
// its arrays stay out of the common path's registers
__device__ __attribute__((noinline)) void gj_inv6(Block6& m) {
  zd inv[36];
  zd a[36];
  for (int i = 0; i < 6; ++i) {
    a[i * 7] = {m.d[i], 0.0};
    for (int j = 0; j < i; ++j) {
      a[i * 6 + j] = m.at(i, j);
      a[j * 6 + i] = conj(m.at(i, j));
    }
  }
  for (int k = 0; k < 36; ++k) inv[k] = {(k % 7 == 0) ? 1.0 : 0.0, 0.0};
  for (int c = 0; c < 6; ++c) {
    int piv = c;
    double best = norm2(a[c * 6 + c]);
    for (int r = c + 1; r < 6; ++r) {
      double v = norm2(a[r * 6 + c]);
      if (v > best) { best = v; piv = r; }
    }
    if (piv != c) {
      for (int k = 0; k < 6; ++k) {
        zd t = a[c * 6 + k]; a[c * 6 + k] = a[piv * 6 + k]; a[piv * 6 + k] = t;
        t = inv[c * 6 + k]; inv[c * 6 + k] = inv[piv * 6 + k]; inv[piv * 6 + k] = t;
      }
    }
    zd p = a[c * 6 + c];
    double d = 1.0 / norm2(p);
    zd pi = {p.re * d, -p.im * d};
    for (int k = 0; k < 6; ++k) {
      a[c * 6 + k] = a[c * 6 + k] * pi;
      inv[c * 6 + k] = inv[c * 6 + k] * pi;
    }
    for (int r = 0; r < 6; ++r) {
      if (r == c) continue;
      zd f = a[r * 6 + c];
      for (int k = 0; k < 6; ++k) {
        a[r * 6 + k] = a[r * 6 + k] - f * a[c * 6 + k];
        inv[r * 6 + k] = inv[r * 6 + k] - f * inv[c * 6 + k];
      }
    }
  }
  for (int i = 0; i < 6; ++i) {
    m.d[i] = inv[i * 7].re;
    for (int j = 0; j < i; ++j) m.at(i, j) = inv[i * 6 + j];
  }
}

__device__ __forceinline__ void pack_block(const Block6& m, void* out, long site, int b) {
  double2* o = site_block<36>(static_cast<double2*>(out), site) + b * 18 * kSiteBlock;
#pragma unroll
  for (int q = 0; q < 3; ++q) o[q * kSiteBlock] = double2{m.d[2 * q], m.d[2 * q + 1]};
#pragma unroll
  for (int q = 0; q < 15; ++q) o[(3 + q) * kSiteBlock] = double2{m.l[q].re, m.l[q].im};
}

template <int B>
__device__ __forceinline__ void build_block(const PlaneLds& G, int lane, bool live, const CloverBuild& a, int parity,
                                            long site) {
  Block6 m;
  assemble_block<B>(G, lane, a.ck, m);
  if (a.A[parity] && live) pack_block(m, a.A[parity], site, B);
  if (!a.Ainv[parity]) return;
  if (!chol_inv6(m)) {
    Block6 f;  // of its own: its address leaves the function, m's registers must not
    assemble_block<B>(G, lane, a.ck, f);
    gj_inv6(f);
    m = f;
    if (live) atomicAdd(a.nbad, 1);
  }
  if (live) pack_block(m, a.Ainv[parity], site, B);
}

// A block of six waves per (64-site chunk, parity), the two parities of a chunk side by
// side: wave pl multiplies out the leaves of plane pl for the 64 sites and leaves G in
// LDS; then waves 0 and 1 assemble chiral blocks 0 and 1, write A and invert them in
// place.  G never goes to memory and a block lives in 72 registers: the two kernels this
// replaces wrote and read 864 B of G a site and kept four full 6x6 complex arrays, mostly
// in scratch.  The leaves bound it (12 links of 144 B and 1,080 FP64 instructions a site
// and plane, one block of 256-register waves per CU).  16^3x32: A of both parities 92 us,
// with the odd inverse 117 (1,030 before); 24^3x48: 520 and 660 us (3,100 before).  Three
// waves a SIMD (168 registers) spill: 125 and 720 us for A.
template <int R>
__global__ void __launch_bounds__(384, 2) clover_build_kernel(const CloverBuild a) {
  __shared__ PlaneLds G;
  const Geom& geo = a.geo;
  const int lane = threadIdx.x & 63;
  const int pl = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned u = remap_block(blockIdx.x, gridDim.x, 1);
  const int parity = a.only < 0 ? (int)(u & 1u) : a.only;
  const long l = (long)(a.only < 0 ? u >> 1 : u) * 64 + lane;
  const bool live = l < geo.vh;
  const long site = live ? l : geo.vh - 1;
  const uint32_t q1 = geo.dx.div((uint32_t)site), q2 = geo.dy.div(q1), q3 = geo.dz.div(q2);
  const int y = (int)(q1 - q2 * geo.dy.d), z = (int)(q2 - q3 * geo.dz.d), t = (int)q3;
  const int c[4] = {2 * (int)((uint32_t)site - q1 * geo.dx.d) + ((parity + y + z + t) & 1), y, z, t};
  double g[9];
  switch (pl) {
    case 0: plane_field<R>(a.gauge, geo, c, 0, 1, g); break;
    case 1: plane_field<R>(a.gauge, geo, c, 0, 2, g); break;
    case 2: plane_field<R>(a.gauge, geo, c, 0, 3, g); break;
    case 3: plane_field<R>(a.gauge, geo, c, 1, 2, g); break;
    case 4: plane_field<R>(a.gauge, geo, c, 1, 3, g); break;
    default: plane_field<R>(a.gauge, geo, c, 2, 3, g); break;
  }
#pragma unroll
  for (int k = 0; k < 9; ++k) G[pl][k][lane] = g[k];
  __syncthreads();
  if (pl == 0) build_block<0>(G, lane, live, a, parity, site);
  else if (pl == 1) build_block<1>(G, lane, live, a, parity, site);
}

// packed F64 -> F32 (18 float4 words per site) / F16 (9 uint4 words); one parity
template <int P>
__global__ void clover_convert_kernel(const double2* src, void* dst, long vh) {
  long site = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (site >= vh) return;
  float r[72];
  const double2* sp = site_block<36>(src, site);
#pragma unroll
  for (int k = 0; k < 36; ++k) {
    double2 q = sp[k * kSiteBlock];
    r[2 * k] = (float)q.x;
    r[2 * k + 1] = (float)q.y;
  }
  if (P == F32) {
    float4* o = site_block<18>(static_cast<float4*>(dst), site);
#pragma unroll
    for (int k = 0; k < 18; ++k)
      o[k * kSiteBlock] = float4{r[4 * k], r[4 * k + 1], r[4 * k + 2], r[4 * k + 3]};
  } else {
    uint4* o = site_block<9>(static_cast<uint4*>(dst), site);
#pragma unroll
    for (int k = 0; k < 9; ++k) o[k * kSiteBlock] = pack8(r + 8 * k);
  }
}

// packed F64 -> complex128 [vh][2][6][6] (reference layout, include/qcu_point.cuh:91-93)
__global__ void clover_unpack_kernel(const double2* src, double2* out, long vh) {
  long site = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (site >= vh) return;
  double a[72];
  const double2* sp = site_block<36>(src, site);
#pragma unroll
  for (int k = 0; k < 36; ++k) {
    double2 q = sp[k * kSiteBlock];
    a[2 * k] = q.x;
    a[2 * k + 1] = q.y;
  }
  double2* o = out + site * 72;
  for (int b = 0; b < 2; ++b) {
    const double* m = a + 36 * b;
    for (int i = 0; i < 6; ++i) o[b * 36 + i * 7] = double2{m[i], 0.0};
    int k = 6;
    for (int i = 1; i < 6; ++i)
      for (int j = 0; j < i; ++j) {
        o[b * 36 + i * 6 + j] = double2{m[k], m[k + 1]};
        o[b * 36 + j * 6 + i] = double2{m[k], -m[k + 1]};
        k += 2;
      }
  }
}

void launch_clover_build(int recon, const CloverBuild& a, hipStream_t st) {
  const dim3 grid((a.only < 0 ? 2 : 1) * nblk(a.geo.vh, 64)), block(384);
  if (recon == 12) hipLaunchKernelGGL(clover_build_kernel<12>, grid, block, 0, st, a);
  else hipLaunchKernelGGL(clover_build_kernel<18>, grid, block, 0, st, a);
}
void launch_clover_convert(int prec, const void* src, void* dst, long vh, hipStream_t st) {
  if (prec == F32)
    hipLaunchKernelGGL(clover_convert_kernel<F32>, dim3(nblk(vh, 256)), dim3(256), 0, st,
                       static_cast<const double2*>(src), dst, vh);
  else
    hipLaunchKernelGGL(clover_convert_kernel<F16>, dim3(nblk(vh, 256)), dim3(256), 0, st,
                       static_cast<const double2*>(src), dst, vh);
}
void launch_clover_unpack(const void* packed, void* out, long vh, hipStream_t st) {
  hipLaunchKernelGGL(clover_unpack_kernel, dim3(nblk(vh, 256)), dim3(256), 0, st,
                     static_cast<const double2*>(packed), static_cast<double2*>(out), vh);
}

}  // namespace qcu
