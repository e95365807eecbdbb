// k_hop_split_f32.hip -- FP32 leg-split hops, on interface and internal fields (k_hop_split.inc).
#include "k_hop_split.inc"

namespace qcu {

void launch_iface_f32(int recon, int dagger, const IfaceArgs& a, hipStream_t st) {
  if (recon == 12) launch_iface<F32, 12, EPI_PLAIN>(a, dagger, st);
  else launch_iface<F32, 18, EPI_PLAIN>(a, dagger, st);
}

void launch_split_f32(int recon, int epi, const HopSplit& a, hipStream_t st) {
  if (recon == 12) launch_split_epi<F32, 12>(epi, a, st);
  else launch_split_epi<F32, 18>(epi, a, st);
}

}  // namespace qcu
