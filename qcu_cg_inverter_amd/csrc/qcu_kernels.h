// qcu_kernels.h -- host-side launchers of the HIP kernels (all asynchronous on the
// given stream).  Fields are one half lattice in the internal layout unless noted;
// a batch of right-hand sides is strided by `stride` bytes.
#pragma once

#include "qcu_common.h"

namespace qcu {

struct Vec {
  void* p;
  long stride;  // bytes between right-hand sides
};
inline Vec vec(void* p, long stride = 0) { return Vec{p, stride}; }

// number of 64-site reduction partials of one half lattice
__host__ __device__ inline long n_partials(long vh) { return (vh + 63) / 64; }

// ------------------------------------------------------------------ hop -----
// block threads = sg * rb; the rb groups share sites (and link loads); a.rpw
// right-hand sides per wave (1, 2 or 4), rpt per thread (1..4)
void launch_hop(int prec, int recon, int epi, const HopArgs& a, int block, int rb, int rpt, hipStream_t st);

// the hop on internal fields with each chunk's legs split over four waves
void launch_hop_split(int prec, int recon, int epi, const HopSplit& a, hipStream_t st);

// the hop straight from and to the caller's interface fields (complex128 [Vh][4][3], or
// full spinors), computed in `prec` (k_hop_split.inc); FP32 and FP16 take the plain
// epilogue.  No out buffer may overlap an in buffer or another out buffer.
void launch_hop_iface(int prec, int recon, int epi, int dagger, const IfaceArgs& a, hipStream_t st);
// out(parity) = D in, FP64, periodic, with links from the caller's own gauge
// [4][2][Vh][3][3], of which rows 0-1 are read; no overlap
void launch_dslash(const void* in, void* out, const void* gauge, const Geom& g, int parity, hipStream_t st);

// --------------------------------------------------------------- layout -----
// interface spinor (complex128 [Vh][4][3]) <-> internal layout of `prec`
void launch_spinor_from_aos(int prec, const void* aos, long aos_stride, Vec out, long vh, int nrhs, hipStream_t st);
void launch_spinor_to_aos(int prec, Vec in, void* aos, long aos_stride, long vh, int nrhs, hipStream_t st);
// interface gauge (complex128 [4][2][Vh][3][3]) -> packed planes
void launch_gauge_pack(int prec, int recon, const void* aos, void* out, long vh, hipStream_t st);
// packed FP64 recon-12 links -> FP32 or FP16 recon-12
void launch_gauge_repack(int prec, const void* rows, void* out, long vh, hipStream_t st);
// 64-bit fingerprint of rows 0-1 of an interface gauge: the sum of the kFingerprintBlocks
// words that the kernel writes to `parts` (pinned host memory); launch_gauge_import packs
// those rows in the same pass (FP64 recon-12)
constexpr int kFingerprintBlocks = 1024;
void launch_fingerprint(const void* aos, uint64_t* parts, long vh, hipStream_t st);
void launch_gauge_import(const void* aos, void* out, uint64_t* parts, long vh, hipStream_t st);
// reference storage shifts: kind 0 half spinor [Vh][24] <-> [24][Vh] doubles; kind 1
// gauge [8][Vh][18] -> [8][12][Vh] (back with row 2 rebuilt)
void launch_shift_storage(int kind, int to_soa, const void* src, void* dst, long vh, hipStream_t st);
// lexicographic <-> even-odd, nc (12 or 9) complex per site, nfields fields of V sites
void launch_lex_eo(int to_eo, const void* src, void* dst, const int L[4], int nc, int nfields, hipStream_t st);
// out, in `prec`, = in, in FP64
void launch_spinor_convert(Vec in, int prec, Vec out, long vh, int nrhs, hipStream_t st);

// ----------------------------------------------------------------- blas -----
// per-right-hand-side CG scalars kept in device memory
struct CgScal {
  double alpha, beta, gamma, tt, ss, target2, ss_ref;
  double gamma_old;  // |r|^2 of the iteration before, where the vector kernels take the steps
  int first, converged, active, breakdown, iter;
  int conv_now;      // converged, as the beta step of the iteration saw it
};

void launch_zero(int prec, Vec v, long vh, int nrhs, hipStream_t st);
// dst = src, bytes a multiple of 16 (reference kernel for bandwidth and counters)
void launch_copy(void* dst, const void* src, size_t bytes, hipStream_t st);
// partials[r][w] = sum over wave w of |v_r|^2
void launch_norm2(int prec, Vec v, long vh, int nrhs, double* partials, hipStream_t st);
// out[r] = sum_w partials[r][w] in a fixed order (one block per right-hand side); out may
// be pinned host memory
void launch_sum_partials(const double* partials, long nw, int nrhs, double* out, hipStream_t st);
// y = a x + b y (F64 or same-precision fields)
void launch_axpby(int prec, double a, Vec x, double b, Vec y, long vh, int nrhs, hipStream_t st);
// out = C in with C packed clover of one parity (same precision as the fields)
void launch_clover_apply(int prec, const void* clov, Vec in, Vec out, long vh, int nrhs, hipStream_t st);

// CGLS steps (see solver.cpp).  All skip right-hand sides with active == 0.
void launch_cg_beta(const double* part_rr, long nw, CgScal* sc, int nrhs, hipStream_t st);
void launch_cg_alpha(const double* part_tt, long nw, CgScal* sc, int nrhs, hipStream_t st);
// host: null, or pinned memory that receives a copy of the scalars
void launch_cg_ss(const double* part_ss, long nw, CgScal* sc, CgScal* host, int nrhs, hipStream_t st);
// sc[0 .. n) = host[0 .. n), pinned memory that stays as it is until the kernel has run
void launch_cg_put(const CgScal* host, CgScal* sc, int n, hipStream_t st);
// nonzero: nrhs right-hand sides of nw partials take their scalar steps inside the vector
// kernels below (pass the partials); 0: by the one-block kernels above, before them
int cg_step_chains(long nw, int nrhs);
// x += alpha p with the alpha and p of the previous iteration (pending until here), then
// p = r + beta p.  With part_rr (|r|^2) the blocks take the beta step themselves, and with
// part_ss they also look at the |s|^2 that the previous iteration left.
void launch_cg_xpay(int prec, int xprec, Vec r, Vec p, Vec x, CgScal* sc, const double* part_rr,
                    const double* part_ss, long nw, long vh, int nrhs, hipStream_t st);
// s -= alpha t ; partials of |s|^2.  With part_tt (|t|^2) the blocks take the alpha step.
void launch_cg_update(int prec, Vec t, Vec s, CgScal* sc, const double* part_tt, long nw, double* part_ss, long vh,
                      int nrhs, hipStream_t st);
// x += alpha p for one right-hand side of an FP64 loop (a pending iterate update, applied
// by the host)
void launch_cg_xflush(Vec x, Vec p, double alpha, long vh, hipStream_t st);
// a scalar per right-hand side, and those a launch is about (bit r of mask)
struct SlotScal {
  double v[kMaxRhs];
  unsigned mask;
};
// x += v p ; xe += x ; x = 0, with x in FP32 and p in `prec` (FP32 or FP16)
void launch_cg_fold(int prec, Vec x, Vec p, Vec xe, const SlotScal& a, long vh, int nrhs, hipStream_t st);
// partials of |b - t|^2 in FP64; the residual of those in mask stored to s in `prec`
void launch_residual(int prec, Vec b, Vec t, Vec s, unsigned mask, long vh, int nrhs, double* part, hipStream_t st);

// --------------------------------------------------------------- clover -----
// A = 1 + ck T and A^-1, packed F64, of both parities (only = -1) or one; any null output
// is left out.  gauge: packed F64 links of `recon`; nbad counts blocks that needed the
// pivoted fallback instead of Cholesky.
struct CloverBuild {
  const void* gauge;
  void* A[2];
  void* Ainv[2];
  int* nbad;
  double ck;
  int only;
  Geom geo;
};
void launch_clover_build(int recon, const CloverBuild& a, hipStream_t st);
// packed F64 -> packed F32 / F16 (one parity)
void launch_clover_convert(int prec, const void* src, void* dst, long vh, hipStream_t st);
// packed F64 -> reference layout complex128 [Vh][2][6][6] (one parity)
void launch_clover_unpack(const void* packed, void* out, long vh, hipStream_t st);

// ------------------------------------------------------------ measurement --
// S site-legs (a multiple of 262144) of the 12-right-hand-side link product Y = U H
// (6x6 by 6x24, FP64) on VALU (mfma = 0) or v_mfma_f64_16x16x4f64 (mfma = 1), operands
// in registers; out receives 262144 partial sums of Y (k_linkprod.hip)
void launch_linkprod(int mfma, long site_legs, double* out, hipStream_t st);

// ------------------------------------------------------------ generators ---
// U_mu(x) = SU3-project(exp(i eps H)) into the interface gauge layout
void launch_gauge_random(void* aos, long vh, uint64_t seed, double eps, hipStream_t st);
// N(0,1) per real of n complex128 values, counter = element index
void launch_source_gauss(void* aos, long n_complex, uint64_t seed, hipStream_t st);

}  // namespace qcu
