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

// the kernel behind dslashQcu: one half spinor, s = +1, the caller's own gauge records
__global__ void __launch_bounds__(256, 3) dslash_kernel(const double2* in, double2* out, const double2* gauge,
                                                        const Geom g, int parity) {
  __shared__ __attribute__((aligned(16))) char S[SplitLds<F64>::bytes(1)];
  split_chunk<F64, 0, EPI_PLAIN, 0, 1>(in, out, nullptr, gauge, nullptr, g, parity, 1.0, 1.0, nullptr,
                                       (long)remap_block(blockIdx.x, gridDim.x, 1) * 64, S);
}

void launch_dslash(const void* in, void* out, const void* gauge, const Geom& g, int parity, hipStream_t st) {
  hipLaunchKernelGGL(dslash_kernel, dim3((unsigned)((g.vh + 63) / 64)), dim3(256), 0, st,
                     static_cast<const double2*>(in), static_cast<double2*>(out),
                     static_cast<const double2*>(gauge), g, parity);
}

void launch_split_f64(int recon, int epi, const HopSplit& a, hipStream_t st) {
  if (recon == 12) launch_split_epi<F64, 12>(epi, a, st);
  else launch_split_epi<F64, 18>(epi, a, st);
}

}  // namespace qcu
