// 3x3 convolution of 16 or 32 int8 channels (padding 1, stride 1 or 2, up to 256 output channels): blocks that walk over tiles of
// 8 x 4 output pixels with their filters in registers, as conv3x3_a16_walk.hip does for int16.
//
// What bounds such layers is their output: 9 x 16 products per channel are over before a tiled kernel's operands and epilogue have
// taken turns once.  A block has as many waves as groups of 32 output channels; the next tile's patch is on its way while this
// one's is multiplied.  us, tiled kernels / this: 16 x 112 x 112, 16 -> 16 to fp32 16.5 / 9.7, 32 -> 32 17.8 / 11.4, 32 -> 128 30.9 /
// 25.6.  With 64 channels and more the filters leave too few registers (32 x 56 x 56, 64 -> 64 12.9 / 22.8): not this kernel's.
#include "conv3x3_halo.h"

namespace catchq {

struct WalkI8Params {
  IgemmParams g;  // M, N, H, W, Ci, Ho, Wo
  int tiles_x, tiles_y, ntiles;
  unsigned x_bytes;
};

constexpr int kWalkPasses = 4;  // of a block's threads over a patch, 16 B each, at most
template <int S>
struct WalkI8 {
  static constexpr int CI = 32;                       // (of 16 channels, the upper half is zeros)
  static constexpr int TW = 8, TH = 4, PW = (TW - 1) * S + 3, PH = (TH - 1) * S + 3;
  static constexpr int ROW = S == 1 ? PW : 20;        // places of a patch row
  static constexpr int PIECES = CI / 16;              // of 16 B of a pixel
  static constexpr int PITCH = CI + 16;               // an odd number of pieces: neighbours cover a 256 B line of LDS
  static constexpr int PATCH = ROW * PH * PITCH;
};

template <int S, int EPI>
__global__ __launch_bounds__(512, 4) void conv3x3_i8_walk_kernel(const int8_t *__restrict__ X, const int8_t *__restrict__ B,
                                                                 WalkI8Params p, EpiDev e) {
  resolve_exp2(e);
  typedef typename EpiOf<EPI>::type Spec;
  typedef WalkI8<S> G;
  constexpr int TW = G::TW;
  constexpr int STRIDE = 32 + 8;  // ints of a staged row
  constexpr unsigned OOB = 0x80000000u;
  extern __shared__ __attribute__((aligned(16))) int8_t lds_dyn[];
  int8_t *const patch = lds_dyn;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int frow = lane & 31, fhalf = lane >> 5;
  const int Co = p.g.N, Ci = p.g.Ci, threads = (int)blockDim.x;
  const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc((void *)X, 0, (int)p.x_bytes, 0x00020000);

  v4i fb[9];
  const int n = wave * 32 + frow;
#pragma unroll
  for (int t = 0; t < 9; ++t) {
    fb[t] = v4i{0, 0, 0, 0};
    if (n < Co && fhalf * 16 < Ci) fb[t] = *reinterpret_cast<const v4i *>(B + (n * 9 + t) * Ci + fhalf * 16);
  }

  auto place = [](int r, int c) { return r * G::ROW + (S == 1 ? c : (c & 1) * (TW + 1) + (c >> 1)); };
  struct Tile { int img, y0, x0; };
  auto tile_at = [&](int t) {
    const int l = xcd_remap(t, p.ntiles), row = l / p.tiles_x;
    return Tile{row / p.tiles_y, row % p.tiles_y * G::TH, (l - row * p.tiles_x) * TW};
  };
  v4i piece[kWalkPasses];
  auto load_patch = [&](int t) {  // (behind the last tile: nothing is read)
    const Tile k = tile_at(t < p.ntiles ? t : 0);
#pragma unroll
    for (int it = 0; it < kWalkPasses; ++it) {
      const int i = it * threads + (int)threadIdx.x, px = i / G::PIECES, q = i - px * G::PIECES, r = px / G::PW, c = px - r * G::PW;
      const int hi = k.y0 * S - 1 + r, wi = k.x0 * S - 1 + c;
      const bool in = t < p.ntiles && r < G::PH && q * 16 < Ci && (unsigned)hi < (unsigned)p.g.H && (unsigned)wi < (unsigned)p.g.W;
      const unsigned from = ((unsigned)(k.img * p.g.H + hi) * (unsigned)p.g.W + (unsigned)wi) * (unsigned)Ci + q * 16u;
      piece[it] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_x, (int)select_u32(in, from, OOB), 0, 0));
    }
  };
  auto store_patch = [&]() {
#pragma unroll
    for (int it = 0; it < kWalkPasses; ++it) {
      const int i = it * threads + (int)threadIdx.x, px = i / G::PIECES, q = i - px * G::PIECES, r = px / G::PW, c = px - r * G::PW;
      if (r < G::PH) *reinterpret_cast<v4i *>(patch + place(r, c) * G::PITCH + q * 16) = piece[it];
    }
  };

  const int8_t *const own = patch + (place(frow / TW * S, 0) + frow % TW) * G::PITCH + fhalf * 16;  // of this lane's output pixel
  const int c0 = wave * 32 + (lane & 7) * 4;
  int *const stage = reinterpret_cast<int *>(lds_dyn + G::PATCH) + wave * 32 * STRIDE;
  const EpiLane L = epi_lane_setup<Spec>(c0, c0 < Co, e);

  load_patch(blockIdx.x);
  store_patch();
  for (int t = blockIdx.x; t < p.ntiles; t += gridDim.x) {
    __syncthreads();
    load_patch(t + gridDim.x);
    const Tile k = tile_at(t);
    const int64_t uni = (((int64_t)k.img * p.g.Ho + k.y0) * p.g.Wo + k.x0) * Co;
    auto exists = [&](int it) { return k.y0 + it < p.g.Ho && k.x0 + (lane >> 3) < p.g.Wo && c0 < Co; };
    auto offset = [&](int it) { return (unsigned)((it * p.g.Wo + (lane >> 3)) * Co + c0); };

    v16i acc;
    static_for<0, 9>([&](auto i_c) {
      constexpr int i = decltype(i_c)::value, r = i / 3, s = i % 3;
      constexpr int off = (r * G::ROW + (S == 1 ? s : (s & 1) * (TW + 1) + (s >> 1))) * G::PITCH;
      const v4i a = *reinterpret_cast<const v4i *>(own + off);
      if constexpr (i == 0) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, fb[i], v16i{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}, 0, 0, 0);
      else acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, fb[i], acc, 0, 0, 0);
    });
    __syncthreads();
    store_patch();  // the next tile's

    v4f res[4];
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      res[it] = v4f{0.f, 0.f, 0.f, 0.f};
      if (L.use_res && exists(it)) res[it] = load_stream(reinterpret_cast<const v4f *>((e.resid + uni) + offset(it)), e.resid_stream != 0);
    }
    // wave-private staging: stores then loads of the same wave, ordered by the LDS counter
#pragma unroll
    for (int r = 0; r < 16; ++r) stage[(8 * (r >> 2) + 4 * fhalf + (r & 3)) * STRIDE + frow] = acc[r];
    v4i av[4];
#pragma unroll
    for (int it = 0; it < 4; ++it) av[it] = *reinterpret_cast<const v4i *>(stage + (it * 8 + (lane >> 3)) * STRIDE + (lane & 7) * 4);
#pragma unroll
    for (int it = 0; it < 4; ++it)
      if (exists(it)) epi_vec4<Spec>(av[it], res[it], L, EpiAtSplit{uni, offset(it)}, e);
  }
}

template <int S>
static int launch_walk_i8(const void *x, const void *w, const WalkI8Params &p, const EpiDev &e, hipStream_t s) {
  typedef WalkI8<S> G;
  const int waves = (p.g.N + 31) / 32, threads = 64 * waves, lds = G::PATCH + waves * 32 * 40 * 4;
  const int most = 256 * (16 / waves), blocks = p.ntiles < most ? p.ntiles : most;
#define CATCHQ_WALK(EPI_)                                                                                              \
  case EPI_:                                                                                                           \
    conv3x3_i8_walk_kernel<S, EPI_><<<blocks, threads, lds, s>>>((const int8_t *)x, (const int8_t *)w, p, e);      \
    return launch_status()
  switch (pick_epilogue(p.g.N, e)) {
    CATCHQ_WALK(EPI_Y32);
    CATCHQ_WALK(EPI_Y16_STEPS);
    CATCHQ_WALK(EPI_Q8_RELU);
    CATCHQ_WALK(EPI_VECTOR);
    default: return -1;
  }
#undef CATCHQ_WALK
}

template <int S>
static bool walk_i8_patch_fits(int Co) { return WalkI8<S>::PW * WalkI8<S>::PH * WalkI8<S>::PIECES <= kWalkPasses * 64 * ((Co + 31) / 32); }

// 3 x 3, padding 1
bool conv3x3_i8_walk_takes(int N, int H, int W, int Ci, int Co, int stride, int Ho, int Wo, const EpiDev &e) {
  const int64_t tiles_x = (Wo + 7) / 8, tiles_y = (Ho + 3) / 4, tiles = N * tiles_x * tiles_y;
  if ((Ci != 16 && Ci != 32) || Co > 256 || (stride != 1 && stride != 2)) return false;
  if ((int64_t)N * H * W * Ci >= (1ll << 31) || tiles >= (1 << 30) || (int64_t)Wo * Co >= (1 << 28) || (int64_t)N * Ho * Wo >= (1ll << 31))
    return false;
  // Four tiles a unit pay for a block's filters (us, tiled kernels / this, 1568 tiles: 16 -> 256 channels 18.7 / 16.9, 32 -> 64 9.0 /
  // 8.9, 32 -> 32 7.8 / 5.8; 392 tiles: 32 -> 64 4.6 / 5.0, 16 -> 256 8.6 / 9.1); of 16 channels one and a half (392 tiles: 16 -> 16
  // 5.2 / 4.0, 16 -> 128 6.5 / 5.8; 112 tiles: 16 -> 16 3.2 / 3.8).
  if (tiles < 4 * (int64_t)e.cus && !(Ci == 16 && Co <= 128 && tiles * 2 >= 3 * (int64_t)e.cus)) return false;
  if (!(stride == 1 ? walk_i8_patch_fits<1>(Co) : walk_i8_patch_fits<2>(Co))) return false;
  const int epi = pick_epilogue(Co, e);
  // The generic epilogue holds up what the walk overlaps (to int8 behind a leaky ReLU: 8 x 112 x 112, 16 -> 192 35.0 / 44.1, 4 x 112 x
  // 112, 1568 tiles, 32 -> 64 10.8 / 11.8, 128 equal; 8 x 112 x 112, 3136 tiles, 64 6 % ahead, 96 a fifth, 32 a quarter).
  if (epi == EPI_VECTOR && Co > 32) return Co <= 128 && tiles >= (Co <= 64 ? 8 : 4) * (int64_t)e.cus;
  return epi == EPI_Y32 || epi == EPI_Y16_STEPS || epi == EPI_Q8_RELU || epi == EPI_VECTOR;
}

// x [N, H, W, Ci] int8, w [Co, 3, 3, Ci], a call that conv3x3_i8_walk_takes
int conv3x3_i8_walk(const void *x, const void *w, int N, int H, int W, int Ci, int Co, int stride, int Ho, int Wo, const EpiDev &e,
                    hipStream_t s) {
  const int tiles_x = (Wo + 7) / 8, tiles_y = (Ho + 3) / 4;
  WalkI8Params p = {};
  p.g.M = (int64_t)N * Ho * Wo;
  p.g.N = Co; p.g.K = 9 * Ci; p.g.H = H; p.g.W = W; p.g.Ci = Ci; p.g.Ho = Ho; p.g.Wo = Wo;
  p.tiles_x = tiles_x; p.tiles_y = tiles_y; p.ntiles = N * tiles_x * tiles_y;
  p.x_bytes = (unsigned)((int64_t)N * H * W * Ci);
  return stride == 1 ? launch_walk_i8<1>(x, w, p, e, s) : launch_walk_i8<2>(x, w, p, e, s);
}

}  // namespace catchq
