// 3x3 convolution of 32 or 64 int16 channels with int8 filters (padding 1, stride 1 or 2, up to twice as many output channels):
// the layers in front of a detector, where images are large and channels few.
//
// What bounds them is HBM -- 32 channels of 16 images of 416 x 416 to 64 at stride 2, with fp32 and int16 outputs, are 443 MB for
// 51 GOP -- and the kernel of the other layers (igemm_a16_dma.hip) is far from it: five K steps of a 64 x 64 tile leave each
// block a chain of one start-up, five operand deliveries and one epilogue.  Here a wave keeps its filters in registers (9 taps x
// 32 columns: 36 of them, 72 with 64 channels) and a block walks over tiles of 64 (32) output pixels: the next tile's patch is on
// its way while this one's is multiplied.  What fills HBM is the number of tiles on their way at once, so everything is small: one
// set of accumulators (the high digits' sums are shifted up before the low digits are added), 128 registers and 27 KB for four
// blocks a unit of 32 channels at stride 1, three otherwise, two of 64 channels at stride 2 behind a generic epilogue (182 registers;
// as many blocks are started as fit: with three started for places of two 2 x 208 x 208, 64 -> 128 took 17.1, now 14.2, 15.0 before
// this kernel).  Stride 2 of 32 channels would fit four (128 registers, 40 KB; not tried).  The digits and the constant are those of
// igemm_a16_dma.hip; a patch is split into digits once, on its way into LDS, and pixels outside the image arrive as zeros.
// us, before / now / at 6 TB/s, 16 images: 32 channels, 416 x 416 at stride 2 126 / 83 / 74, 208 x 208 with a residual 123 / 58 / 52;
// 64 channels, 208 x 208 at stride 2 58 / 44 / 37, 104 x 104 with a residual and fp32 output 71 / 48 / 41, to int16 only 55 / 37 / 11.
// One image: 13.2 / 10.6, 11.7 / 9.1, 9.9 / 9.9, 10.1 / 9.7.  To halfs only, which the tiled kernel has an instance for as well:
// 2 x 208 x 208, 64 -> 128 35.4 / 22.3, at stride 2 12.3 / 12.7, 6 x 190 x 190 at stride 2 24.2 / 20.0; with the generic epilogue 28.6,
// 16.9 and 29.9.  With tiles of 16 x 8, 64 columns a wave and both digits' sums at once (two blocks a unit) the first two of 16
// images were 91 and 113.
#include "conv3x3_halo.h"

namespace catchq {

struct WalkParams {
  IgemmParams g;  // M, N, H, W, Ho, Wo
  int tiles_x, tiles_y, ntiles;
  unsigned x_bytes;
};

// Blocks of a unit: what an instance's registers are bounded for and what its launch starts
template <int CI, int S, int EPI>
constexpr int walk_blocks() { return CI == 32 && S == 1 ? 4 : (CI == 64 && S == 2 && EPI == EPI_VECTOR ? 2 : 3); }

template <int CI, int S, int EPI>
__global__ __launch_bounds__(256, (walk_blocks<CI, S, EPI>())) void conv3x3_a16_walk_kernel(const int16_t *__restrict__ X,
                                                                                          const int8_t *__restrict__ B,
                                                                                          WalkParams p, EpiDev e) {
  resolve_exp2(e);
  typedef typename EpiOf<EPI>::type Spec;
  constexpr int CG = CI == 32 ? 2 : 4;  // waves side by side on a tile, 32 columns each; 4 / CG runs of 32 pixels
  constexpr int TW = CI == 32 ? 16 : 8, TH = 32 * (4 / CG) / TW;
  constexpr int KK = CI / 32;
  constexpr int PW = (TW - 1) * S + 3, PH = (TH - 1) * S + 3, PX = PW * PH;
  constexpr int PLACES = S == 1 ? PX : (PW + 1) * PH;
  constexpr int TPP = CI / 16, PPP = 256 / TPP, NP = (PX + PPP - 1) / PPP;  // threads of 16 channels per pixel; pixels of a pass; passes
  constexpr int STRIDE = 32 + 8;        // ints of a staged row
  constexpr unsigned OOB = 0x80000000u;
  __shared__ __attribute__((aligned(256))) int8_t patch[PLACES * CI * 2];  // the high digits of a pixel's channels, then the low ones
  __shared__ __attribute__((aligned(16))) int staged[4 * 32 * STRIDE];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int frow = lane & 31, fhalf = lane >> 5;
  const int Co = p.g.N;
  const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc((void *)X, 0, (int)p.x_bytes, 0x00020000);

  // ---- filters and 128 times their sums ----------------------------------------------------------------------------
  const int cg = wave % CG, pg = wave / CG;
  const int n = cg * 32 + frow;
  v4i fb[9 * KK];
  int sum = 0;
#pragma unroll
  for (int t = 0; t < 9 * KK; ++t) {
    fb[t] = v4i{0, 0, 0, 0};
    if (n < Co) fb[t] = *reinterpret_cast<const v4i *>(B + (n * 9 * KK + t) * 32 + fhalf * 16);
#pragma unroll
    for (int d = 0; d < 4; ++d) sum = __builtin_amdgcn_sdot4(fb[t][d], 0x01010101, sum, false);
  }
  const unsigned ws = (unsigned)(sum + __shfl_xor(sum, 32, 64)) << 7;

  // A pixel's place in the patch: rows of PW, the columns of a row that one tap of neighbouring outputs reads side by side.
  // Its 16 B pieces are swizzled with the low bits of the output pixel whose first tap it is: sixteen neighbours cover a 256 B
  // line of LDS.
  auto place = [](int r, int c) { return S == 1 ? r * PW + c : r * (PW + 1) + (c & 1) * (TW + 1) + (c >> 1); };
  auto address = [](int at, int pixel, int piece) {
    return at * (CI * 2) + ((piece ^ (CI == 32 ? (pixel >> 2) & 3 : (pixel >> 1) & 7)) << 4);
  };

  struct Tile { int img, y0, x0; };
  auto tile_at = [&](int t) {
    const int l = xcd_remap(t, p.ntiles), row = l / p.tiles_x;
    return Tile{row / p.tiles_y, row % p.tiles_y * TH, (l - row * p.tiles_x) * TW};
  };
  struct Piece { v4i a, b; };
  Piece piece[NP];
  auto load_patch = [&](int t) {  // (behind the last tile: nothing is read)
    const Tile k = tile_at(t < p.ntiles ? t : 0);
#pragma unroll
    for (int it = 0; it < NP; ++it) {
      const int i = it * PPP + (int)(threadIdx.x / TPP), r = i / PW, c = i - r * PW;
      const int hi = k.y0 * S - 1 + r, wi = k.x0 * S - 1 + c;
      const bool in = t < p.ntiles && i < PX && (unsigned)hi < (unsigned)p.g.H && (unsigned)wi < (unsigned)p.g.W;
      const unsigned from = ((unsigned)(k.img * p.g.H + hi) * (unsigned)p.g.W + (unsigned)wi) * (CI * 2u) + (threadIdx.x % TPP) * 32u;
      const int off = (int)select_u32(in, from, OOB);
      piece[it].a = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_x, off, 0, 0));
      piece[it].b = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_x, off, 16, 0));
    }
  };
  auto store_patch = [&]() {
#pragma unroll
    for (int it = 0; it < NP; ++it) {
      const int i = it * PPP + (int)(threadIdx.x / TPP), r = i / PW, c = i - r * PW;
      if (i < PX) {
        v4i hi, lo;
        split_i16(piece[it].a, piece[it].b, hi, lo);
        const int to = address(place(r, c), r / S * TW + c / S, (int)(threadIdx.x % TPP));
        *reinterpret_cast<v4i *>(patch + to) = hi;
        *reinterpret_cast<v4i *>(patch + (to ^ CI)) = lo;
      }
    }
  };

  // this lane's output pixel within the tile, and its four channels of a staged row
  const int ty = pg * (32 / TW) + frow / TW, tx = frow % TW;
  const int c0 = cg * 32 + (lane & 7) * 4;
  int *const stage = staged + wave * 32 * STRIDE;
  const EpiLane L = epi_lane_setup<Spec>(c0, c0 < Co, e);
  constexpr bool kResid = EPI == EPI_LK_RESA_Q16 || EPI == EPI_LK_RESA_Y_Q16;

  load_patch(blockIdx.x);
  store_patch();
  for (int t = blockIdx.x; t < p.ntiles; t += gridDim.x) {
    __syncthreads();
    load_patch(t + gridDim.x);
    const Tile k = tile_at(t);
    const int ho = k.y0 + pg * (32 / TW);  // of the first of this wave's rows
    const int64_t uni = (((int64_t)k.img * p.g.Ho + ho) * p.g.Wo + k.x0) * Co;
    auto exists = [&](int it) { return ho + it * 8 / TW < p.g.Ho && k.x0 + it * 8 % TW + (lane >> 3) < p.g.Wo && c0 < Co; };
    auto offset = [&](int it) { return (unsigned)((it * 8 / TW * p.g.Wo + it * 8 % TW + (lane >> 3)) * Co + c0); };
    v4f res[4];
    auto load_resid = [&]() {
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        res[it] = v4f{0.f, 0.f, 0.f, 0.f};
        if (exists(it)) res[it] = load_stream(reinterpret_cast<const v4f *>((e.resid + uni) + offset(it)), e.resid_stream != 0);
      }
    };
    if constexpr (kResid) load_resid();

    // 256 * sum of the high digits' products + that of the low ones', modulo 2^32, in one set of accumulators
    v16i acc;
    // (opaque: the addresses of all taps, kept in registers across the loop, leave none for reads on their way)
    int at0 = place(ty * S, 0) + tx, px0 = ty * TW + tx;
    asm volatile("" : "+v"(at0), "+v"(px0));
    static_for<0, 18 * KK>([&](auto i_c) {
      constexpr int i = decltype(i_c)::value, t = i % (9 * KK), r = t / KK / 3, s = t / KK % 3;
      const v4i digits = *reinterpret_cast<const v4i *>(patch + address(at0 + place(r, s), px0 + r / S * TW + s / S, i / (9 * KK) * (CI / 16) + t % KK * 2 + fhalf));
      if constexpr (i == 0) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(digits, fb[t], v16i{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}, 0, 0, 0);
      else acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(digits, fb[t], acc, 0, 0, 0);
      if constexpr (i == 9 * KK - 1) {
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[q] = (int)(((unsigned)acc[q] << 8) + ws);
      }
    });
    __syncthreads();
    store_patch();  // the next tile's

    if (Spec::kGeneric && L.use_res) load_resid();
    // wave-private staging: stores then loads of the same wave, ordered by the LDS counter
#pragma unroll
    for (int r = 0; r < 16; ++r) stage[(8 * (r >> 2) + 4 * fhalf + (r & 3)) * STRIDE + frow] = acc[r];
    v4i av[4];
#pragma unroll
    for (int it = 0; it < 4; ++it) av[it] = *reinterpret_cast<const v4i *>(stage + (it * 8 + (lane >> 3)) * STRIDE + (lane & 7) * 4);
#pragma unroll
    for (int it = 0; it < 4; ++it)
      if (exists(it)) epi_vec4<Spec>(av[it], L.use_res ? res[it] : v4f{0.f, 0.f, 0.f, 0.f}, L, EpiAtSplit{uni, offset(it)}, e);
  }
}

template <int CI, int S>
static int launch_walk(const void *x, const void *w, const WalkParams &p, const EpiDev &e, hipStream_t s) {
#define CATCHQ_WALK(EPI_)                                                                                             \
  case EPI_: {                                                                                                        \
    const int most = 256 * walk_blocks<CI, S, EPI_>(), blocks = p.ntiles < most ? p.ntiles : most;                    \
    conv3x3_a16_walk_kernel<CI, S, EPI_><<<blocks, 256, 0, s>>>((const int16_t *)x, (const int8_t *)w, p, e);         \
    return launch_status();                                                                                           \
  }
  const int epi = pick_epilogue(p.g.N, e);
  if constexpr (S == 1) {  // (a residual branch has its block's size)
    switch (epi) {
      CATCHQ_WALK(EPI_LK_RESA_Q16)
      CATCHQ_WALK(EPI_LK_RESA_Y_Q16)
      default: break;
    }
  }
  switch (epi) {
    CATCHQ_WALK(EPI_LK_Q16)
    CATCHQ_WALK(EPI_LK_Y_Q16)
    CATCHQ_WALK(EPI_Y32)
    CATCHQ_WALK(EPI_Y16)
    default:
    CATCHQ_WALK(EPI_VECTOR)
  }
#undef CATCHQ_WALK
}

static int walk_tile_columns(int Ci) { return Ci == 32 ? 16 : 8; }

// 3 x 3, padding 1
bool conv3x3_a16_walk_takes(int N, int H, int W, int Ci, int Co, int stride, int Ho, int Wo, const EpiDev &e) {
  const int tw = walk_tile_columns(Ci);
  const int64_t tiles_x = (Wo + tw - 1) / tw, tiles_y = (Ho + 3) / 4, tiles = N * tiles_x * tiles_y;
  if ((Ci != 32 && Ci != 64) || Co <= Ci || Co > 2 * Ci || (stride != 1 && stride != 2)) return false;
  if ((int64_t)N * H * W * Ci * 2 >= (1ll << 31) || tiles >= (1 << 30) || (int64_t)Wo * Co >= (1 << 28) || (int64_t)N * Ho * Wo >= (1ll << 31))
    return false;
  // 64 channels on a few tiles: what reads the filters as it needs them is ahead (us, this / that: 26 x 26, 28 tiles, 6.1 / 5.0,
  // 64 x 64, 128 tiles, 6.0 / 5.9; 2 x 64 x 64, 256, 6.0 / 8.6); 32 channels are ahead from one tile on (4 x 7 x 7 4.6 / 7.6)
  // At stride 2 more columns ask for more of them (128 columns, two outputs: 208 x 208, 338 tiles, 9.7 / 10.0, 2 x 208 x 208, 676, 14.0 /
  // 13.5; 96 columns, 338 tiles, 9.6 / 9.3).
  if (Ci == 64 && (tiles * 4 < 3 * (int64_t)e.cus || (stride == 2 && Co > 96 && tiles < 2 * (int64_t)e.cus))) return false;
  return pick_epilogue(Co, e) != EPI_SCALAR;
}

// x [N, H, W, Ci] int16, w [Co, 3, 3, Ci], a call that conv3x3_a16_walk_takes
int conv3x3_a16_walk(const void *x, const void *w, int N, int H, int W, int Ci, int Co, int stride, int Ho, int Wo, const EpiDev &e,
                     hipStream_t s) {
  const int tw = walk_tile_columns(Ci), tiles_x = (Wo + tw - 1) / tw, tiles_y = (Ho + 3) / 4;
  WalkParams p = {};
  p.g.M = (int64_t)N * Ho * Wo;
  p.g.N = Co; p.g.K = 9 * Ci; p.g.H = H; p.g.W = W; p.g.Ci = Ci; p.g.Ho = Ho; p.g.Wo = Wo;
  p.tiles_x = tiles_x; p.tiles_y = tiles_y; p.ntiles = N * tiles_x * tiles_y;
  p.x_bytes = (unsigned)((int64_t)N * H * W * Ci * 2);
  if (Ci == 32) return stride == 1 ? launch_walk<32, 1>(x, w, p, e, s) : launch_walk<32, 2>(x, w, p, e, s);
  return stride == 1 ? launch_walk<64, 1>(x, w, p, e, s) : launch_walk<64, 2>(x, w, p, e, s);
}

}  // namespace catchq
