// k_hop_split_f64.hip -- FP64 hops on interface fields (k_hop_split.inc).
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
// FAR: the call's data (records of 144 B a link, read whole) is past the Infinity Cache.
// Then the chunks go round-robin over the XCDs, so that all of them read one region of HBM
// at a time; before, each XCD takes a contiguous range and finds more of it in its L2.
template <int FAR>
__global__ void __launch_bounds__(256, 3) dslash_kernel(const double2* in, double2* out, const double2* gauge,
                                                        const Geom g, int parity) {
  __shared__ __attribute__((aligned(16))) char S[SplitLds<F64>::bytes(1)];
  split_chunk<F64, 0, EPI_PLAIN, 0, 1, FAR>(in, out, nullptr, gauge, nullptr, g, parity, 1.0, 1.0, nullptr,
                                            (long)remap_block(blockIdx.x, gridDim.x, !FAR) * 64, S);
}

// Calls on three states in turn, ranges / round-robin (us): 16^3x32 (100 MB) 29.4 / 31.3,
// 20^3x40 (246 MB) 64.0 / 67.3; 16^2x32x64 (403 MB) 96.4 / 93.5, 24^3x48 (510 MB) 118.3 /
// 117.5, 28^3x64 251 / 242, 32^3x48 281 / 251, 32^3x64 (1.6 GB) 360 / 330.
void launch_dslash(const void* in, void* out, const void* gauge, const Geom& g, int parity, hipStream_t st) {
  const dim3 grid((unsigned)((g.vh + 63) / 64)), block(256);
  const double2* i = static_cast<const double2*>(in);
  double2* o = static_cast<double2*>(out);
  const double2* u = static_cast<const double2*>(gauge);
  if ((size_t)g.vh * (8 * 144 + 2 * 192) > (size_t)256 << 20)
    hipLaunchKernelGGL(dslash_kernel<1>, grid, block, 0, st, i, o, u, g, parity);
  else
    hipLaunchKernelGGL(dslash_kernel<0>, grid, block, 0, st, i, o, u, g, parity);
}

void launch_split_f64(int recon, int epi, const HopSplit& a, hipStream_t st) {
  if (recon == 12) launch_split_epi<F64, 12>(epi, a, st);
  else launch_split_epi<F64, 18>(epi, a, st);
}

}  // namespace qcu
