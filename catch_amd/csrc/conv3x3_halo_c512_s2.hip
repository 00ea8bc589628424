// Patch-resident 3x3 convolution: the stride-2 instances for 512 input channels.
#include "conv3x3_halo_kernel.inc"

namespace catchq {

int halo_launch_c512_s2(const void *x, const void *w, const HaloParams &hp, const EpiDev &e, int tn, int lds_bytes, int waves,
                        hipStream_t s) {
  return launch_halo<512, 2>(x, w, hp, e, tn, lds_bytes, waves, s);
}

}  // namespace catchq
