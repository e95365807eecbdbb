// k_hop_split_f16.hip -- FP16 leg-split hops, on interface and internal fields (k_hop_split.inc).
#include "k_hop_split.inc"

namespace qcu {

void launch_iface_f16(int recon, int dagger, const IfaceArgs& a, hipStream_t st) {
  if (recon == 12) launch_iface<F16, 12, EPI_PLAIN>(a, dagger, st);
  else launch_iface<F16, 18, EPI_PLAIN>(a, dagger, st);
}

void launch_split_f16(int recon, int epi, const HopSplit& a, hipStream_t st) {
  if (recon == 12) launch_split_epi<F16, 12>(epi, a, st);
  else launch_split_epi<F16, 18>(epi, a, st);
}

}  // namespace qcu
