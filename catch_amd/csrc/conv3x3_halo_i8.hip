// Entry points of the patch-resident 3x3 kernel (conv3x3_halo_kernel.inc); the instances of each channel count are
// compiled in files of their own (conv3x3_halo_c*.hip), the ones with a 1x1 head here.
#include "conv3x3_halo_kernel.inc"

namespace catchq {

int halo_launch_c64(int stride, const void *x, const void *w, const HaloParams &hp, const EpiDev &e, int tn, int lds_bytes, int waves,
                    hipStream_t s);
int halo_launch_c128(int stride, const void *x, const void *w, const HaloParams &hp, const EpiDev &e, int tn, int lds_bytes, int waves,
                    hipStream_t s);
int halo_launch_c256(int stride, const void *x, const void *w, const HaloParams &hp, const EpiDev &e, int tn, int lds_bytes, int waves,
                    hipStream_t s);
int halo_launch_c512(int stride, const void *x, const void *w, const HaloParams &hp, const EpiDev &e, int tn, int lds_bytes, int waves,
                    hipStream_t s);

// 3x3, stride 1 or 2 (both directions alike), padding 1, no dilation, Ci in {64, 128, 256, 512} (stride 2: not 64);
// input [N, Hi, Wi, Ci]; -1: not this kernel's shape
int conv2d_halo_i8(const void *x, const void *w, int N, int Hi, int Wi, int Ci, int Co, int stride, const EpiDev &e,
                   hipStream_t s) {
  HaloParams hp;
  int tn, lds_bytes, waves;
  if (!halo_plan(N, Hi, Wi, Ci, Co, stride, hp, tn, lds_bytes, waves, 0, 1, e.cus)) return -1;
  switch (Ci) {
    case 64: return halo_launch_c64(stride, x, w, hp, e, tn, lds_bytes, waves, s);
    case 128: return halo_launch_c128(stride, x, w, hp, e, tn, lds_bytes, waves, s);
    case 256: return halo_launch_c256(stride, x, w, hp, e, tn, lds_bytes, waves, s);
    default: return halo_launch_c512(stride, x, w, hp, e, tn, lds_bytes, waves, s);
  }
}

// Whether a stride-1 layer runs here as a single round of blocks
bool conv2d_halo_one_round(int N, int H, int W, int Ci, int Co, int cus) {
  HaloParams hp;
  int tn, lds_bytes, waves;
  return halo_plan(N, H, W, Ci, Co, 1, hp, tn, lds_bytes, waves, 0, 1, cus) && hp.nblocks <= cus;
}

// The head's shapes: 1x1 convolution K1 -> 64 channels (+ ReLU, int8 requantization with unit scale) feeding a 3x3
// layer 64 -> 64, stride 1, padding 1, whose tiles are bands of rows; K1 in {64, 256}.
bool conv2d_head_halo_i8_ok(int N, int H, int W, int K1, int Cm, int Co) {
  if (Cm != 64 || Co != 64 || (K1 != 64 && K1 != 256)) return false;
  if ((int64_t)N * H * W * K1 >= (1ll << 31)) return false;
  HaloParams hp;
  int tn, lds_bytes, waves;
  if (!halo_plan(N, H, W, Cm, Co, 1, hp, tn, lds_bytes, waves, Co / 32)) return false;
  return hp.image_mode == 0 && waves == 4 && hp.tiles_n == 1 && (hp.PR * hp.W + 31) / 32 <= 12;
}

// x [N, H, W, K1] int8, head filters [Cm, K1], w [Co, 3, 3, Cm]; -1: not this kernel's shape
int conv2d_head_halo_i8(const void *x, int K1, const void *w1, const float *div1, const float *rcp1, const float *bias1,
                        int exp2_1, int q_position1, const void *w, int N, int H, int W, int Cm, int Co, const EpiDev &e,
                        hipStream_t s) {
  if (!conv2d_head_halo_i8_ok(N, H, W, K1, Cm, Co)) return -1;
  if (!div1 || !rcp1 || !bias1 || exp2_1 < -64 || exp2_1 > 64 || !aligned16(x) || !aligned16(w1) || !aligned16(w)) return -1;
  HaloParams hp;
  int tn, lds_bytes, waves;
  halo_plan(N, H, W, Cm, Co, 1, hp, tn, lds_bytes, waves, Co / 32);
  hp.x_bytes = (unsigned)((int64_t)N * H * W * K1);
  lds_bytes += 1024;  // the head's per-channel constants behind the ring
  if (lds_bytes > 160 * 1024) return -1;
  HeadDev hd = {(const int8_t *)w1, div1, rcp1, bias1, exp2_1, -q_position1, (unsigned)(Cm * K1)};
  const int epi = pick_epilogue(Co, e);
  if (epi == EPI_SCALAR) return -1;
#define CATCHQ_HEAD(K1_, TMW_)                                                                                                  \
  return epi == EPI_Q8_RELU ? launch_halo_epi<64, 2, TMW_, 1, EPI_Q8_RELU, 4, K1_, 3>(x, w, hp, e, lds_bytes, s, hd)             \
                            : launch_halo_epi<64, 2, TMW_, 1, EPI_VECTOR, 4, K1_, 3>(x, w, hp, e, lds_bytes, s, hd)
#define CATCHQ_HEAD8(K1_)                                                                                                       \
  return epi == EPI_Q8_RELU ? launch_halo_epi<64, 2, 1, 1, EPI_Q8_RELU, 8, K1_, 2>(x, w, hp, e, lds_bytes, s, hd)                \
                            : launch_halo_epi<64, 2, 1, 1, EPI_VECTOR, 8, K1_, 2>(x, w, hp, e, lds_bytes, s, hd)
  // Five to eight sub-tiles behind a head of 256 channels run on eight waves: the head's eleven or twelve sub-tiles of
  // matrix and epilogue work spread over twice the waves and need two thirds of the fragment registers (measured on
  // ResNet-50's first stage, 32 images: 20.7 -> 18.7 us per launch, +0.6 % end to end; the 64-channel head gains nothing)
  int head_waves = (K1 == 256 && hp.nsub > 4 && hp.nsub <= 8) ? 8 : 4;
  if (const char *t = tuning_env("CATCHQ_HEAD_WAVES")) head_waves = (atoi(t) == 8 && hp.nsub <= 8) ? 8 : 4;
  if (head_waves == 8) {
    if (K1 == 64) CATCHQ_HEAD8(64);
    CATCHQ_HEAD8(256);
  }
#undef CATCHQ_HEAD8
  if (K1 == 64) {
    if (hp.nsub <= 4) CATCHQ_HEAD(64, 1);
    CATCHQ_HEAD(64, 2);
  }
  if (hp.nsub <= 4) CATCHQ_HEAD(256, 1);
  CATCHQ_HEAD(256, 2);
#undef CATCHQ_HEAD
}

}  // namespace catchq
