// 3x3 convolution of int8 activations (stride 1, padding 1, channels a multiple of 32) with filters laid out by pack_filters
// (float_rows.hip).
//
// What bounds the tiled kernel (igemm_i8_dma_conv.hip) on such a layer is the chain of a block: set-up with a tap mask per pixel,
// nine taps' deliveries through a ring of slots with a barrier each, epilogue -- one round of blocks in which none of the three
// overlaps.  Here a block requests the whole run of input pixels that its outputs read (TM * 32 + 2 W + 2 of them: same size,
// stride 1) at once and meets one barrier; filters go from L2 to registers, nine fragments ahead.  Taps outside the image read a
// pixel of zeros, per lane and tap.  A wave has TM * 32 pixels x 32 channels, a block up to eight waves side by side.
// us with the quantizer in front, repeated in a graph on the same inputs, tiled / this: 5 x 57 x 75, 96 -> 160 on NCHW floats 18.7 /
// 16.0 (17.6 / 15.5 on changing inputs), on NHWC halfs 16.8 / 14.1; on NCHW floats 8 x 28 x 28, 192 14.3 / 11.4, 16 x 14 x 14, 384
// 19.9 / 14.6, 20 x 57 x 75, 96 -> 160 51.6 / 41.9.
#include "conv3x3_halo.h"

namespace catchq {

struct PackedI8Params {
  IgemmParams g;  // M, N, H, W, Ci, tiles_n, nblocks
  unsigned x_bytes, w_bytes;
  unsigned magic;   // quotients by Ci / 16
  int rows;         // of the patch
  int batches;      // of kPatchPieces pieces of 16 B a thread stages
};

constexpr int kPatchPieces = 6;

template <int TM, int EPI>
__global__ __launch_bounds__(512, 2) void conv3x3_i8_packed_kernel(const int8_t *__restrict__ X, const int8_t *__restrict__ B,
                                                                   PackedI8Params p, EpiDev e) {
  resolve_exp2(e);
  constexpr unsigned OOB = 0x80000000u;
  extern __shared__ __attribute__((aligned(16))) int8_t lds_dyn[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int frow = lane & 31, fhalf = lane >> 5, threads = (int)blockDim.x;
  const int logical = xcd_remap(blockIdx.x, p.g.nblocks);
  const int tile_m = logical / p.g.tiles_n, tile_n = logical - tile_m * p.g.tiles_n;
  const int m0 = tile_m * TM * 32;  // (fewer than 2^26 pixels)
  const int n0 = (tile_n * (threads >> 6) + wave) * 32;
  const int W = p.g.W, Ci = p.g.Ci, nc = Ci / 32, M = (int)p.g.M;
  const int pitch = Ci + 16;  // an odd number of 16 B pieces: neighbours cover a 256 B line of LDS
  const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc((void *)X, 0, (int)p.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc((void *)B, 0, (int)p.w_bytes, 0x00020000);

  // filters: one KiB for 32 columns x 32 channels of a tap, taps first; columns that do not exist read others'
  const int w_at = n0 < p.g.N ? (n0 >> 5) * 9 * nc * 1024 : 0;
  auto load_w = [&](int tap, int c) {  // (behind the last channels: the last ones again)
    return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_w, lane * 16, w_at + (tap * nc + (c < nc ? c : nc - 1)) * 1024, 0));
  };
  v4i fb[9];
#pragma unroll
  for (int t = 0; t < 9; ++t) fb[t] = load_w(t, 0);

  const int per_row = Ci / 16, px0 = m0 - W - 1;
  for (int b = 0; b < p.batches; ++b) {
    v4i v[kPatchPieces];
#pragma unroll
    for (int i = 0; i < kPatchPieces; ++i) {
      const int at = (b * kPatchPieces + i) * threads + (int)threadIdx.x;
      const int row = (int)__umulhi((unsigned)at, p.magic), q = at - row * per_row;
      const bool in = row < p.rows && (unsigned)(px0 + row) < (unsigned)M;
      const unsigned from = select_u32(in, (unsigned)(px0 + row) * (unsigned)Ci + (unsigned)q * 16u, OOB);
      v[i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_x, (int)from, 0, 0));
    }
#pragma unroll
    for (int i = 0; i < kPatchPieces; ++i) {
      const int at = (b * kPatchPieces + i) * threads + (int)threadIdx.x;
      const int row = (int)__umulhi((unsigned)at, p.magic), q = at - row * per_row;
      if (row < p.rows) *reinterpret_cast<v4i *>(lds_dyn + row * pitch + q * 16) = v[i];
    }
  }
  const int zero = p.rows * pitch;  // a pixel of zeros
  for (int i = threadIdx.x; i < per_row; i += threads) *reinterpret_cast<v4i *>(lds_dyn + zero + i * 16) = v4i{0, 0, 0, 0};

  int own[TM];
  unsigned mask[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + i * 32 + frow;
    const unsigned mm = (unsigned)(m < M ? m : 0), t = mm / (unsigned)W, h = t % (unsigned)p.g.H;
    const int wo = (int)(mm - t * (unsigned)W);
    const unsigned cols = (wo > 0 ? 1u : 0u) | 2u | (wo + 1 < W ? 4u : 0u);
    mask[i] = m < M ? ((h > 0 ? cols : 0u) | cols << 3 | (h + 1 < (unsigned)p.g.H ? cols << 6 : 0u)) : 0u;
    own[i] = (i * 32 + frow) * pitch + fhalf * 16;
  }
  __syncthreads();

  v16i acc[TM][1];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][0][r] = 0;
  for (int c = 0; c < nc; ++c) {
    static_for<0, 9>([&](auto tap_c) {
      constexpr int tap = decltype(tap_c)::value;
      const int shift = (tap / 3 * W + tap % 3) * pitch + c * 32, none = zero + c * 32 + fhalf * 16;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const v4i a = *reinterpret_cast<const v4i *>(lds_dyn + ((mask[i] >> tap) & 1 ? own[i] + shift : none));
        acc[i][0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, fb[tap], acc[i][0], 0, 0, 0);
      }
      fb[tap] = load_w(tap, c + 1);
    });
  }
  __syncthreads();
  int *const stage = reinterpret_cast<int *>(lds_dyn) + wave * 32 * (32 + 8);
  if constexpr (EPI == EPI_SCALAR) igemm_epilogue_any<TM, 1>(acc, stage, m0, n0, lane, p.g, e);
  else igemm_epilogue<TM, 1, EPI>(acc, stage, m0, n0, lane, p.g, e);
}

template <int TM>
static int launch_packed_i8(const void *x, const void *w, const PackedI8Params &p, int waves, const EpiDev &e, hipStream_t s) {
  const int a_bytes = p.rows * (p.g.Ci + 16) + p.g.Ci, stage = waves * 32 * 40 * 4, lds = a_bytes > stage ? a_bytes : stage;
#define CATCHQ_PACKED(EPI_)                                                                                              \
  case EPI_: {                                                                                                           \
    auto kern = conv3x3_i8_packed_kernel<TM, EPI_>;                                                                      \
    if (lds > 64 * 1024) {                                                                                               \
      static std::atomic<bool> raised[64];                                                                               \
      if (raise_lds_limit((const void *)kern, 160 * 1024, raised) != CATCHQ_OK) return CATCHQ_ERR_LAUNCH;                \
    }                                                                                                                    \
    kern<<<p.g.nblocks, 64 * waves, lds, s>>>((const int8_t *)x, (const int8_t *)w, p, e);                               \
    return launch_status();                                                                                              \
  }
  switch (pick_epilogue(p.g.N, e)) {
    CATCHQ_PACKED(EPI_Y32)
    CATCHQ_PACKED(EPI_Y16)
    CATCHQ_PACKED(EPI_Y16_STEPS)
    CATCHQ_PACKED(EPI_VECTOR)
    CATCHQ_PACKED(EPI_SCALAR)
    default: return -1;
  }
#undef CATCHQ_PACKED
}

// The rows of 32 pixels a wave takes, 0: not this kernel's shape
static int packed_i8_plan(int64_t N, int H, int W, int Ci, int Co, bool any_rows, const EpiDev &e) {
  if (Co % 4 != 0 && !any_rows) return 0;
  const int64_t M = N * H * W, groups = ((int64_t)Co + 31) / 32;
  // (the patch-resident kernels: 32 x 28 x 28, 128 channels, 16.4 / 16.8 us with this one, 32 x 14 x 14, 256 14.0 / 15.0)
  if (!conv3x3_i8_packed_channels(Ci, Co) || W > 512 || H >= (1 << 20) || M * Ci >= (1ll << 31) || groups * Ci * 288 >= (1ll << 31)) return 0;
  const int epi = pick_epilogue(Co, e);
  if (epi != EPI_Y32 && epi != EPI_Y16 && epi != EPI_Y16_STEPS && epi != EPI_VECTOR && !(any_rows && epi == EPI_SCALAR && ragged_epilogue(Co, e, true)))
    return 0;
  // Half a block of 32 pixels for a unit (us, tiled / this: 1 x 57 x 75, 96 -> 160, 134 blocks, 9.7 / 9.0, 10 x 14 x 14, 160 -> 512, 124,
  // 11.2 / 11.3, 3 x 30 x 33, 448 -> 224, 93, 14.9 / 16.0, 1 x 28 x 28, 192, 25, 7.9 / 9.8); blocks of 64, which read half the
  // filters, from as many of those on (8 x 25 x 25, 160 -> 320, 158, 13.3 / 12.6 with 64; 8 x 28 x 28, 192, 98, 11.5 / 13.4).
  // 96 and 128 pixels a block gain nothing more.
  const int64_t columns = (groups + 7) / 8;
  auto patch = [&](int tm) { return (int64_t)(tm * 32 + 2 * W + 2) * (Ci + 16) + Ci; };
  auto fits = [&](int tm) { return patch(tm) <= 80 * 1024; };  // two blocks a unit
  auto blocks = [&](int tm) { return (M + tm * 32 - 1) / (tm * 32) * columns; };
  // Up to 64 channels leave a block one wave or two: more than a round of blocks, and four (three) of them to a unit, have to hide
  // what it waits for (with the quantizer: 6 x 28 x 28, 384 -> 16, 74 blocks, 9.1 / 13.4, 64 x 14 x 14, 192 -> 32, 196, 9.4 / 12.2, 64
  // 11.2 / 12.3; 32 x 28 x 28, 96 -> 32, 392, 11.8 / 10.9, 64 12.5 / 11.8; but 60 x 60, 384 -> 16, 562 of 75 KB, a quarter slower).
  // Wide images ask for two rounds of them (5 x 57 x 75, 160 -> 16, 334 blocks, 14.3 / 15.4).
  if (groups <= 2) {
    if (blocks(2) * 8 >= 9 * (int64_t)e.cus && patch(2) <= (groups == 1 ? 40 : 52) * 1024 && (W <= 48 || blocks(2) >= 2 * (int64_t)e.cus)) return 2;
    // Channels that are no multiple of 64 make the tiled kernel's steps cross filter taps, and fewer blocks or larger patches will do
    // (40 x 28 x 28, 608 -> 64, 490 of 75 KB, a tenth ahead; of 32 pixels 10 x 28 x 28, 480 -> 64, 245 blocks, a seventh, 64 x 14 x 14,
    // 992 -> 64 a sixth, 6 x 28 x 28, 147, 800 -> 64 an eighth, 224 -> 64 equal; not up to 44 channels or on wide images: 227 of 160 -> 36
    // on rows of 55 8 % behind)
    if (Ci % 64 == 0 || Co < 48 || W > 48) return 0;
    if (blocks(2) * 2 >= 3 * (int64_t)e.cus && fits(2)) return 2;
    return fits(1) && (blocks(1) * 8 >= 7 * (int64_t)e.cus || (Ci >= 480 && blocks(1) * 2 >= e.cus)) ? 1 : 0;
  }
  if (blocks(1) * 2 < e.cus) return 0;
  if (blocks(2) * 2 < e.cus) return fits(1) ? 1 : 0;
  if (fits(2)) return 2;
  // Where only blocks of 32 fit, the wider tiles of many columns are ahead on many rows (with the quantizer: 5 x 57 x 75, 384 -> 192
  // 46.7 / 39.8, 320 60.0 / 55.3, 512, 1336 blocks, 65.4 / 80.0; 8 x 56 x 56, 480 -> 192 62.3 / 55.0, 512, 1568, 84.9 / 109.8; but
  // 10 x 28 x 28, 768 -> 320, 490, 50.6 / 36.8, 64 x 14 x 14, 992 -> 384, 784, 118 / 87).
  return fits(1) && (groups <= 10 || blocks(1) * 4 <= 13 * (int64_t)e.cus) ? 1 : 0;
}

bool conv3x3_i8_packed_takes(int64_t N, int H, int W, int Ci, int Co, bool any_rows, const EpiDev &e) {
  return packed_i8_plan(N, H, W, Ci, Co, any_rows, e) != 0;
}

// x [N, H, W, Ci] int8, packed: pack_filters of w [Co, 9 Ci]; any_rows: also rows of outputs of any length and alignment; -1: not this
// kernel's shape
int conv3x3_i8_packed(const void *x, const void *packed, int64_t N, int H, int W, int Ci, int Co, bool any_rows, const EpiDev &e,
                      hipStream_t s) {
  const int tm = packed_i8_plan(N, H, W, Ci, Co, any_rows, e);
  if (!tm) return -1;
  const int groups = (Co + 31) / 32;
  PackedI8Params p = {};
  p.g.M = N * H * W;
  p.g.ragged = pick_epilogue(Co, e) == EPI_SCALAR ? ragged_epilogue(Co, e, true) : EPI_SCALAR;
  p.g.N = Co; p.g.K = 9 * Ci; p.g.H = H; p.g.W = W; p.g.Ci = Ci;
  p.x_bytes = (unsigned)(p.g.M * Ci);
  p.w_bytes = (unsigned)((int64_t)groups * Ci * 288);
  p.g.tiles_n = (groups + 7) / 8;
  const int waves = (groups + p.g.tiles_n - 1) / p.g.tiles_n;
  const int64_t nb = (p.g.M + tm * 32 - 1) / (tm * 32) * p.g.tiles_n;
  if (nb > 0x7fffffff) return -1;
  p.g.nblocks = (int)nb;
  p.magic = (unsigned)(((1ull << 32) + Ci / 16 - 1) / (Ci / 16));
  p.rows = tm * 32 + 2 * W + 2;
  const int pieces = p.rows * (Ci / 16), a_pass = kPatchPieces * 64 * waves;
  p.batches = (pieces + a_pass - 1) / a_pass;
  return tm == 1 ? launch_packed_i8<1>(x, packed, p, waves, e, s) : launch_packed_i8<2>(x, packed, p, waves, e, s);
}

}  // namespace catchq
