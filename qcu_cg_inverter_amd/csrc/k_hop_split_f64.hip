// k_hop_split_f64.hip -- FP64 leg-split hops, on interface and internal fields, and dslashQcu
// (k_hop_split.inc).
#include "k_hop_split.inc"

namespace qcu {

template <int R>
static void iface(int epi, int dagger, const IfaceArgs& a, hipStream_t st) {
  if (epi == EPI_PLAIN) launch_iface<F64, R, EPI_PLAIN>(a, dagger, st);
  else if (epi == EPI_XPAY) launch_iface<F64, R, EPI_XPAY>(a, dagger, st);
  else if (epi == EPI_CLOV) launch_iface<F64, R, EPI_CLOV>(a, dagger, st);
  else launch_iface<F64, R, EPI_CLOV_XPAY>(a, dagger, st);
}

void launch_iface_f64(int recon, int epi, int dagger, const IfaceArgs& a, hipStream_t st) {
  if (recon == 12) iface<12>(epi, dagger, a, st);
  else iface<18>(epi, dagger, a, st);
}

// the kernel behind dslashQcu: one half spinor, s = +1, the caller's own gauge records.
// FAR: the call's data (records of 144 B a link, read whole) is well past the Infinity Cache.
// Then the chunks go round-robin over the XCDs, so that all of them read one region of HBM
// at a time; before, each XCD takes a contiguous range and finds more of it in its L2.
template <int FAR>
__global__ void __launch_bounds__(256, 3) dslash_kernel(const double2* in, double2* out, const double2* gauge,
                                                        const Geom g, int parity) {
  __shared__ __attribute__((aligned(16))) char S[SplitLds<F64>::bytes(1)];
  split_chunk<F64, 0, EPI_PLAIN, 0, 1, FAR>(in, out, nullptr, gauge, nullptr, g, parity, 1.0, 1.0, nullptr,
                                            (long)remap_block(blockIdx.x, gridDim.x, !FAR) * 64, S);
}

// Calls, ranges / round-robin (us), on three states in turn and back and forth on one gauge,
// as a caller's own solver makes them: 16^3x32 (100 MB) 29.4 / 31.3 and 28.6 / 30.9, 20^3x40
// (246 MB) 65.0 / 67.3 and 54.1 / 66.0, 16^2x32x48 (302 MB) 80.7 / 74.5 and 66.6 / 66.6,
// 20x24x28x32 (330 MB) 82.5 / 84.2 and 74.9 / 82.8, 24^3x32 (340 MB) 83.6 / 83.9 and 78.0 / 81.1,
// 24^3x34 (361 MB) 92.9 / 88.1 and 85.8 / 85.7, 32^2x16x32 (403 MB) 98.2 / 92.1 and 96.2 / 90.8,
// 24^3x48 (510 MB) 121.6 / 118.0 and 120.5 / 117.9, 32^3x64 (1.6 GB) 366 / 329 and 365 / 328.
void launch_dslash(const void* in, void* out, const void* gauge, const Geom& g, int parity, hipStream_t st) {
  const dim3 grid((unsigned)((g.vh + 63) / 64)), block(256);
  const double2* i = static_cast<const double2*>(in);
  double2* o = static_cast<double2*>(out);
  const double2* u = static_cast<const double2*>(gauge);
  if ((size_t)g.vh * (8 * 144 + 2 * 192) > (size_t)340 << 20)
    hipLaunchKernelGGL(dslash_kernel<1>, grid, block, 0, st, i, o, u, g, parity);
  else
    hipLaunchKernelGGL(dslash_kernel<0>, grid, block, 0, st, i, o, u, g, parity);
}

void launch_split_f64(int recon, int epi, const HopSplit& a, hipStream_t st) {
  if (recon == 12) launch_split_epi<F64, 12>(epi, a, st);
  else launch_split_epi<F64, 18>(epi, a, st);
}

}  // namespace qcu
