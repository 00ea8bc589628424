// Patch-resident 3x3 convolution: the instances for 128 input channels.
#include "conv3x3_halo_kernel.inc"

namespace catchq {

int halo_launch_c128(int stride, const void *x, const void *w, const HaloParams &hp, const EpiDev &e, int tn, int lds_bytes, int waves,
                    hipStream_t s) {
  return stride == 2 ? launch_halo<128, 2>(x, w, hp, e, tn, lds_bytes, waves, s) : launch_halo<128, 1>(x, w, hp, e, tn, lds_bytes, waves, s);
}

}  // namespace catchq
