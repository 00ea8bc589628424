// 3x3 convolution of int16 activations with int8 filters at stride 2 (padding 1, images of even height and width), the filters laid out
// once: the layers that halve a detector's image, with the digits, the packed filters and the block of conv3x3_a16_packed.hip.
//
// The tiled kernel (igemm_a16_dma.hip) brings an input pixel once for each tap that reads it and splits it into digits each time.  At
// stride 2 a run of consecutive outputs reads no run of inputs, but it does in each of the four planes that the parities of row and
// column make of an image: with even extents plane pixel q of (row parity, column parity) lies where output q lies, and a tap reads
// the plane of its parities at q, q - 1, q - Wo or q - Wo - 1.  So a block stages four runs, BM, BM + 1, BM + Wo and BM + Wo + 1 pixels,
// already split, and the nine taps are constant shifts in LDS as they are at stride 1.  The patch is four times as large as there:
// 32 channels a step instead of 64, so that two buffers leave room for two blocks a unit.
// What bounds it now: no unit by itself.  Counters of the three layers below (676, 338 and 340 blocks): matrix pipes 28 % of all SIMD
// cycles, vector instructions 14 to 27 %, LDS 15 to 17 %; waves wait a fifth to a third of their lives, and the blocks are no whole
// number of rounds (two a unit, 237 registers with 64 pixels; three of 32 pixels, 145 to 158).  Where channels are few (128) every block
// reads whole cache lines of the input in two steps.
// us, tiled kernel / this, fp32 and int16 outputs, repeated in a graph: 16 images of 104 x 104, 128 -> 256 43.6 / 37.3, 52 x 52, 256 ->
// 512 37.1 / 33.8, 26 x 26, 512 -> 1024 44.4 / 34.3; 12 images 33.7 / 26.7, 34.3 / 25.4, 33.1 / 26.3; 4 x 80 x 80, 128 -> 256 13.5 /
// 10.1; one of 110 x 104, 192 -> 1024 20.2 / 15.7; 8 x 102 x 96, 384 -> 512 118 / 81.
#include "conv3x3_halo.h"
#include "packed_rules.h"

namespace catchq {

struct PackedConvS2Params {
  IgemmParams g;  // M, N, W (of the input), Wo, Ci, tiles_n, tiles_m, nblocks
  int Ho;
  int m_fastest;  // order of the blocks: the longer operand is shared by neighbours
  unsigned x_bytes, w_bytes;
  const int *sums;  // 128 * sum of a column's weights, modulo 2^32
};

int64_t packed3x3_filter_bytes(int64_t Co, int64_t Ci);
int64_t packed3x3_bytes(int64_t Co, int64_t Ci);

constexpr int kS2Pass = 128;  // pixels a pass of a block's 256 threads stages, 32 channels of each

// A block: TM * 32 output pixels x 256 channels.  NIT: passes over the four runs.
template <int TM, int NIT, int EPI>
__global__ __launch_bounds__(256, 2) void conv3x3_a16_packed_s2_kernel(const int16_t *__restrict__ X, const int8_t *__restrict__ B,
                                                                       PackedConvS2Params p, EpiDev e) {
  resolve_exp2(e);
  constexpr int BM = TM * 32, BN = 256;
  constexpr int RING = 3;                  // taps of filters in registers (a divisor of 9: its slots are constants)
  constexpr int PATCH = NIT * kS2Pass * 64;  // bytes: 32 high digits, 32 low ones of a pixel
  constexpr unsigned OOB = 0x80000000u;
  extern __shared__ __attribute__((aligned(256))) int8_t lds_dyn[];
  int8_t *const zero = lds_dyn + 2 * PATCH;  // digits of a pixel of zeros

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int frow = lane & 31, fhalf = lane >> 5;
  const int logical = xcd_remap(blockIdx.x, p.g.nblocks);
  const int tile_m = p.m_fastest ? logical % p.g.tiles_m : logical / p.g.tiles_n;
  const int tile_n = p.m_fastest ? logical / p.g.tiles_m : logical % p.g.tiles_n;
  const int64_t m0 = (int64_t)tile_m * BM;
  const int n0 = tile_n * BN + wave * 64;
  const int W = p.g.W, Wo = p.g.Wo, nc = p.g.Ci / 32;

  const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc((void *)X, 0, (int)p.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc((void *)B, 0, (int)p.w_bytes, 0x00020000);

  // ---- staging: thread = place tid / 2 of a pass, 16 of its 32 channels -------------------------------------------
  // places: the runs of (even row, even column), (even, odd), (odd, even), (odd, odd)
  const int start01 = BM, start10 = 2 * BM + 1, start11 = 3 * BM + 1 + Wo, places = 4 * BM + 2 + 2 * Wo;
  unsigned st_from[NIT];
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    const int place = it * kS2Pass + (int)(threadIdx.x >> 1);
    const int pr = place >= start10, pc = pr ? place >= start11 : place >= start01;
    const int start = pr ? (pc ? start11 : start10) : (pc ? start01 : 0);
    const int q = (int)m0 + place - start - (pr ? Wo : 0) - pc;  // (fewer than 2^24 outputs)
    const bool exists = place < places && (unsigned)q < (unsigned)p.g.M;
    const unsigned qq = exists ? (unsigned)q : 0u, row = qq / (unsigned)Wo;
    const unsigned px = 2u * (row * (unsigned)Wo + qq) + (unsigned)(pr * W + pc);  // (2 row + pr) W + 2 (q - row Wo) + pc, W = 2 Wo
    st_from[it] = select_u32(exists, px * (unsigned)(p.g.Ci * 2) + (threadIdx.x & 1) * 32u, OOB);
  }
  const int st_row = (int)(threadIdx.x >> 1);
  const int st_to = st_row * 64 + (int)(((threadIdx.x & 1) ^ ((st_row >> 2) & 3)) << 4);
  struct Piece { v4i a, b; };
  auto load_piece = [&](int it, int c) {  // (c = nc: nothing is read, zeros come back)
    const unsigned from = select_u32(c < nc, st_from[it], OOB);
    Piece r;
    r.a = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_x, (int)from, c * 64, 0));
    r.b = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_x, (int)from, c * 64 + 16, 0));
    return r;
  };
  auto store_piece = [&](int it, const Piece &r, int buffer) {
    v4i hi, lo;
    split_i16(r.a, r.b, hi, lo);
    int8_t *const at = lds_dyn + buffer * PATCH + it * kS2Pass * 64;
    *reinterpret_cast<v4i *>(at + st_to) = hi;
    *reinterpret_cast<v4i *>(at + (st_to ^ 32)) = lo;
  };

  // ---- filters: 32 columns x (channels / 64) x 9 taps x 2 halves, 1 KiB each -------------------------------------
  const int w_tile = p.g.Ci * 288;  // bytes of 32 columns
  const int w_lane = lane * 16;
  int w_at[2];  // wave-uniform; columns that do not exist read others' filters and are not stored
#pragma unroll
  for (int j = 0; j < 2; ++j) w_at[j] = n0 + j * 32 < p.g.N ? ((n0 >> 5) + j) * w_tile : 0;
  auto load_w = [&](v4i (&fb)[2], int c, int tap) {  // (c = nc, taps 0 and 1: not used, inside the packed operand)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      fb[j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(
                                          rsrc_w, w_lane, w_at[j] + ((c >> 1) * 18 + tap * 2 + (c & 1)) * 1024, 0));
  };

  // ---- this lane's pixels -----------------------------------------------------------------------------------------
  unsigned inside[TM];  // bit 0: the output exists, 1: and has a column to its left, 2: a row above it, 3: both
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int64_t m = m0 + i * 32 + frow;
    const unsigned mm = (unsigned)(m < p.g.M ? m : 0);
    const unsigned t = mm / (unsigned)Wo, h = t % (unsigned)p.Ho;
    const bool left = mm != t * (unsigned)Wo, above = h > 0;
    inside[i] = m < p.g.M ? (1u | (left ? 2u : 0u) | (above ? 4u : 0u) | (left && above ? 8u : 0u)) : 0u;
  }
  const int fh16 = fhalf << 4;

  if (threadIdx.x < 4) reinterpret_cast<v4i *>(zero)[threadIdx.x] = threadIdx.x < 2 ? v4i{0, 0, 0, 0} : v4i{(int)0x80808080, (int)0x80808080, (int)0x80808080, (int)0x80808080};

  v16i acc_hi[TM][2], acc_lo[TM][2];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) { acc_hi[i][j][r] = 0; acc_lo[i][j][r] = 0; }

  v4i fb[RING][2], fa[2][TM][2];
#pragma unroll
  for (int h = 0; h < RING - 1; ++h) load_w(fb[h], 0, h);
  {
    Piece r[NIT];
#pragma unroll
    for (int it = 0; it < NIT; ++it) r[it] = load_piece(it, 0);
#pragma unroll
    for (int it = 0; it < NIT; ++it) store_piece(it, r[it], 0);
  }
  __syncthreads();

  auto read_tap = [&](v4i (&f)[TM][2], auto tap_c, int buffer) {
    constexpr int dy = decltype(tap_c)::value / 3, dx = decltype(tap_c)::value % 3;
    const int start = dy == 1 ? (dx == 1 ? 0 : start01) : (dx == 1 ? start10 : start11);
    const int shift = start + (dy == 2 ? Wo : 0) + (dx == 2 ? 1 : 0);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int row = i * 32 + frow + shift;
      const int a = buffer * PATCH + (row << 6) + (((row << 2) & 0x30) ^ fh16);
      const int at = (inside[i] >> ((dy == 0 ? 2 : 0) + (dx == 0 ? 1 : 0))) & 1 ? a : 2 * PATCH + fh16;
#pragma unroll
      for (int d = 0; d < 2; ++d) f[i][d] = *reinterpret_cast<const v4i *>(lds_dyn + (at ^ (d * 32)));
    }
  };

  for (int c = 0; c < nc; ++c) {
    const int buffer = c & 1;
    read_tap(fa[0], std::integral_constant<int, 0>{}, buffer);
    constexpr bool BURST = TM == 1;  // one burst where its registers are at hand: a load of filters behind it waits for it
    Piece piece[BURST ? NIT : 2];
    static_for<0, 9>([&](auto h_c) {
      constexpr int h = decltype(h_c)::value;
      __builtin_amdgcn_sched_barrier(0);
      load_w(fb[(h + RING - 1) % RING], h + RING - 1 < 9 ? c : c + 1, (h + RING - 1) % 9);
      if constexpr (BURST && h == 0) {
#pragma unroll
        for (int it = 0; it < NIT; ++it) piece[it] = load_piece(it, c + 1);
      }
      if constexpr (!BURST && h % 2 == 0 && h / 2 < NIT) piece[(h / 2) % 2] = load_piece(h / 2, c + 1);
      if constexpr (h + 1 < 9) read_tap(fa[(h + 1) & 1], std::integral_constant<int, h + 1>{}, buffer);
      if constexpr (BURST && h >= 5 && h - 5 < NIT) store_piece(h - 5, piece[h - 5], buffer ^ 1);
      if constexpr (!BURST && h % 2 == 1 && h >= 3 && (h - 3) / 2 < NIT) store_piece((h - 3) / 2, piece[((h - 3) / 2) % 2], buffer ^ 1);
      if constexpr (!BURST && h == 8 && NIT == 4) store_piece(3, piece[1], buffer ^ 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          acc_hi[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[h & 1][i][0], fb[h % RING][j], acc_hi[i][j], 0, 0, 0);
          acc_lo[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[h & 1][i][1], fb[h % RING][j], acc_lo[i][j], 0, 0, 0);
        }
    });
    __syncthreads();
  }

#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int n = n0 + j * 32 + frow;
    const unsigned ws = n < p.g.N ? (unsigned)p.sums[n] : 0u;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc_lo[i][j][r] = (int)(((unsigned)acc_hi[i][j][r] << 8) + (unsigned)acc_lo[i][j][r] + ws);
  }
  int *stage = reinterpret_cast<int *>(lds_dyn) + wave * 32 * (64 + 8);
  igemm_epilogue<TM, 2, EPI>(acc_lo, stage, m0, n0, lane, p.g, e);
}

template <int TM, int NIT, int EPI>
static int launch_s2_epi(const void *x, const void *w, const PackedConvS2Params &p, const EpiDev &e, hipStream_t s) {
  static_assert(NIT <= 4);
  constexpr int LDS = 2 * NIT * kS2Pass * 64 + 64, STAGE = 4 * 32 * (64 + 8) * 4;
  constexpr int LDS_BYTES = LDS > STAGE ? LDS : STAGE;
  auto kern = conv3x3_a16_packed_s2_kernel<TM, NIT, EPI>;
  if (LDS_BYTES > 64 * 1024) {
    static std::atomic<bool> raised[64];
    if (raise_lds_limit((const void *)kern, LDS_BYTES, raised) != CATCHQ_OK) return CATCHQ_ERR_LAUNCH;
  }
  kern<<<p.g.nblocks, 256, LDS_BYTES, s>>>((const int16_t *)x, (const int8_t *)w, p, e);
  return launch_status();
}

template <int TM, int NIT>
static int launch_s2(const void *x, const void *w, const PackedConvS2Params &p, const EpiDev &e, hipStream_t s) {
  switch (pick_epilogue(p.g.N, e)) {
    case EPI_LK_Q16: return launch_s2_epi<TM, NIT, EPI_LK_Q16>(x, w, p, e, s);
    case EPI_LK_Y_Q16: return launch_s2_epi<TM, NIT, EPI_LK_Y_Q16>(x, w, p, e, s);
    case EPI_Y16: return launch_s2_epi<TM, NIT, EPI_Y16>(x, w, p, e, s);
    case EPI_SCALAR: return -1;
    default: return launch_s2_epi<TM, NIT, EPI_VECTOR>(x, w, p, e, s);
  }
}

// As at stride 1, blocks of 32 pixels for five eighths of the units: 2 x 104 x 104, 128 -> 256 (169 blocks) 11.1 / 9.6 us, 8 x 26 x 26,
// 512 -> 1024 (172) 25.6 / 25.3; below, the waves that split K (ksplit.hip) are ahead.  They are up to more blocks on long K: 768 ->
// 448, 98 blocks for 128 units 29.7 / 34.1, 768 -> 512, 226 for 256 43.6 / 36.7.  A quarter of the columns missing costs what is won
// if they are a quarter of all: 16 x 52 x 52, 128 -> 192 (two launches at a time) 11.9 / 12.7, 8 x 82 x 76, 384 -> 192 35.3 / 35.2, but
// 2 x 60 x 54, 128 -> 384 9.7 / 8.4, 16 x 72 x 70, 256 -> 384 85 / 61.  Odd extents have no such planes.
bool conv3x3_a16_packed_s2_takes(int N, int H, int W, int Ci, int Co, const EpiDev &e) {
  if (H % 2 != 0 || W % 2 != 0 || W > 254 || H >= (1 << 20)) return false;
  const int64_t in = (int64_t)N * H * W, M = in / 4, columns = ((int64_t)Co + 255) / 256 * 256;
  if (!conv3x3_a16_packed_s2_filters(Co, Ci) || in * Ci * 2 >= (1ll << 31) || columns / 32 * Ci * 288 >= (1ll << 31) - (1 << 20)) return false;
  const int epi = pick_epilogue(Co, e);
  if (epi == EPI_SCALAR) return false;
  const int64_t blocks = (M + 31) / 32 * (columns / 256);
  return blocks * 8 >= (Ci > 512 ? 7 : 5) * (int64_t)e.cus;
}

// x [N, H, W, Ci] int16, packed: pack3x3's, outputs [N, H / 2, W / 2, Co]; -1: not this kernel's shape
int conv3x3_a16_packed_s2(const void *x, const void *packed, int N, int H, int W, int Ci, int Co, const EpiDev &e, hipStream_t s) {
  if (!conv3x3_a16_packed_s2_takes(N, H, W, Ci, Co, e)) return -1;
  PackedConvS2Params p = {};
  p.Ho = H / 2;
  p.g.M = (int64_t)N * p.Ho * (W / 2);
  p.g.N = Co; p.g.K = 9 * Ci; p.g.H = H; p.g.W = W; p.g.Ci = Ci; p.g.Ho = p.Ho; p.g.Wo = W / 2;
  p.x_bytes = (unsigned)(4 * p.g.M * Ci * 2);
  p.w_bytes = (unsigned)packed3x3_bytes(Co, Ci);
  p.sums = reinterpret_cast<const int *>(static_cast<const int8_t *>(packed) + packed3x3_filter_bytes(Co, Ci));
  p.g.tiles_n = (Co + 255) / 256;
  const bool wide = (p.g.M + 63) / 64 * p.g.tiles_n >= e.cus;  // (as at stride 1)
  const int bm = wide ? 64 : 32;
  p.g.tiles_m = (int)((p.g.M + bm - 1) / bm);
  if ((int64_t)p.g.tiles_m * p.g.tiles_n > 0x7fffffff) return -1;
  p.g.nblocks = p.g.tiles_m * p.g.tiles_n;
  p.m_fastest = p.w_bytes > p.x_bytes;
  const bool one_more = p.g.Wo > 63;  // 4 bm + 2 + 2 Wo places in passes of 128
  if (wide) return one_more ? launch_s2<2, 4>(x, packed, p, e, s) : launch_s2<2, 3>(x, packed, p, e, s);
  return one_more ? launch_s2<1, 3>(x, packed, p, e, s) : launch_s2<1, 2>(x, packed, p, e, s);
}

}  // namespace catchq
