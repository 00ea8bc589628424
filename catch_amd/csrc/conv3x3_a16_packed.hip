// 3x3 convolution of int16 activations with int8 filters (stride 1, padding 1), the filters laid out once in the order of the
// matrix instruction.
//
// The digits and the constant are those of igemm_a16_dma.hip: x = 256 * hi + lo + 128, sums modulo 2^32.  What bounds that kernel
// on a detector's layers is the delivery of operands: a step of its 64 x 128 tile brings 16 KB through L2 and back out of LDS for
// 256 clocks of matrix work, 64 B a clock each way, and every tap splits its int16 values anew.  Here
// - a block's activations come once per 64 channels, not once per tap: nine taps of 64 consecutive output pixels (stride 1, same
//   size) read one run of 64 + 2 W + 2 consecutive input pixels.  They are split into digits on their way into LDS; taps outside
//   the image read a pixel of zeros instead (per lane and tap);
// - filters go from L2 to registers (each wave has 64 columns of its own), two half steps ahead (five with 32 rows a wave), and
//   never through LDS;
// - a wave has 64 (or 32) x 64 outputs: 16 matrix instructions of 32 clocks a step for 8 KB out of LDS and 4 KB out of L2.
// Barriers: one per 64 channels.  Two waves a SIMD (246 to 253 registers with 64 rows a wave, 169 to 187 with 32, where 168 would be
// three; a shorter ring of filters there is not tried): one's address arithmetic and loads run under the other's matrix
// instructions.  What bounds it now: the matrix pipes while a block has its unit to itself (46 clocks an instruction at 2.4 GHz,
// whatever the depth of the filter ring), the last round of blocks, and an epilogue that all blocks reach together.
// us, before / now (16 images unless said): 13 x 13, 512 -> 1024 46 / 33, 26 x 26, 256 -> 512 37 / 30, 52 x 52, 128 -> 256 42 / 31,
// with the residual and fp32 output 51 / 42; 8 images 26 / 18, 25 / 18, 22 / 19 (launches in their sequence; repeated in a graph, 16
// images, 47 / 33, 38 / 32, 43 / 33, 52 / 45).
// Tried: 96 and 128 rows a wave on one wave a SIMD (30 and 36 us on 16 x 26 x 26, 37 and 45 on 52 x 52), filters five or
// eight half steps ahead (equal), 128 x 128 blocks for 64 -> 128 channels on 104 x 104 (51 / 52: its outputs bound it).
#include "conv3x3_halo.h"

namespace catchq {

struct PackedConvParams {
  IgemmParams g;        // M, N, H, W, Ci, tiles_n, tiles_m, nblocks
  int m_fastest;        // order of the blocks: the longer operand is shared by neighbours
  unsigned x_bytes, w_bytes;
  const int *sums;      // 128 * sum of a column's weights, modulo 2^32
};

constexpr int kPatchPx = 64;  // pixels a pass of a block's 256 threads stages
constexpr int kMaxAhead = 5;  // half steps of filters, 1 KiB each for 32 columns, that a wave requests behind its last one

// A block: TM * 32 pixels x 256 channels.  NIT: passes over the patch.
template <int TM, int NIT, int EPI>
__global__ __launch_bounds__(256, 2) void conv3x3_a16_packed_kernel(const int16_t *__restrict__ X, const int8_t *__restrict__ B,
                                                                    PackedConvParams p, EpiDev e) {
  resolve_exp2(e);
  constexpr int BM = TM * 32, BN = 256;
  constexpr int RING = TM == 1 ? 6 : 3;  // half steps of filters in registers (a divisor of 18: its slots are constants)
  static_assert(18 % RING == 0 && RING - 1 <= kMaxAhead);
  constexpr int PATCH = NIT * kPatchPx * 128;  // bytes: 64 high digits, 64 low ones of a pixel
  constexpr unsigned OOB = 0x80000000u;
  extern __shared__ __attribute__((aligned(128))) int8_t lds_dyn[];
  int8_t *const zero = lds_dyn + 2 * PATCH;  // digits of a pixel of zeros

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int frow = lane & 31, fhalf = lane >> 5;
  const int logical = xcd_remap(blockIdx.x, p.g.nblocks);
  const int tile_m = p.m_fastest ? logical % p.g.tiles_m : logical / p.g.tiles_n;
  const int tile_n = p.m_fastest ? logical / p.g.tiles_m : logical % p.g.tiles_n;
  const int64_t m0 = (int64_t)tile_m * BM;
  const int n0 = tile_n * BN + wave * 64;
  const int W = p.g.W, nc = p.g.Ci / 64;

  const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc((void *)X, 0, (int)p.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc((void *)B, 0, (int)p.w_bytes, 0x00020000);

  // ---- staging: thread = pixel tid / 4, 16 of its 64 channels ----------------------------------------------------
  const int st_px = (int)m0 - W - 1 + (int)(threadIdx.x >> 2);  // (fewer than 2^24 pixels)
  const unsigned st_from = (unsigned)st_px * (unsigned)(p.g.Ci * 2) + (threadIdx.x & 3) * 32u;
  const int st_to = (int)(threadIdx.x >> 2) * 128 + (int)(((threadIdx.x & 3) ^ ((threadIdx.x >> 3) & 7)) << 4);
  struct Piece { v4i a, b; };
  auto load_piece = [&](int it, int c) {  // (c = nc: nothing is read, zeros come back)
    const int px = st_px + it * kPatchPx;
    const unsigned from = select_u32((unsigned)px < (unsigned)p.g.M && c < nc, st_from + (unsigned)(it * kPatchPx * 2) * (unsigned)p.g.Ci, OOB);
    Piece r;
    r.a = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_x, (int)from, c * 128, 0));
    r.b = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_x, (int)from, c * 128 + 16, 0));
    return r;
  };
  auto store_piece = [&](int it, const Piece &r, int buffer) {
    v4i hi, lo;
    split_i16(r.a, r.b, hi, lo);
    int8_t *const at = lds_dyn + buffer * PATCH + it * kPatchPx * 128;
    *reinterpret_cast<v4i *>(at + st_to) = hi;
    *reinterpret_cast<v4i *>(at + (st_to ^ 64)) = lo;
  };

  // ---- filters: 32 columns x (channels / 64) x 9 taps x 2 halves, 1 KiB each -------------------------------------
  const int w_tile = p.g.Ci * 288;  // bytes of 32 columns
  const int w_lane = lane * 16;
  int w_at[2];  // wave-uniform; columns that do not exist read others' filters and are not stored
#pragma unroll
  for (int j = 0; j < 2; ++j) w_at[j] = n0 + j * 32 < p.g.N ? ((n0 >> 5) + j) * w_tile : 0;
  auto load_w = [&](v4i (&fb)[2], int half) {  // (up to kMaxAhead halves behind the end: not used, inside the packed operand)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      fb[j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_w, w_lane, w_at[j] + half * 1024, 0));
  };

  // ---- this lane's two pixels -----------------------------------------------------------------------------------
  int prow[TM];
  unsigned mask[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int r = i * 32 + frow;
    const int64_t m = m0 + r;
    const unsigned mm = (unsigned)(m < p.g.M ? m : 0);
    const unsigned t = mm / (unsigned)W, h = t % (unsigned)p.g.H;
    const int wo = (int)(mm - t * (unsigned)W);
    const unsigned cols = (wo > 0 ? 1u : 0u) | 2u | (wo + 1 < W ? 4u : 0u);
    mask[i] = m < p.g.M ? ((h > 0 ? cols : 0u) | cols << 3 | (h + 1 < (unsigned)p.g.H ? cols << 6 : 0u)) : 0u;
    prow[i] = r;
  }
  const int fh16 = fhalf << 4;

  if (threadIdx.x < 8) reinterpret_cast<v4i *>(zero)[threadIdx.x] = threadIdx.x < 4 ? v4i{0, 0, 0, 0} : v4i{(int)0x80808080, (int)0x80808080, (int)0x80808080, (int)0x80808080};

  v16i acc_hi[TM][2], acc_lo[TM][2];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) { acc_hi[i][j][r] = 0; acc_lo[i][j][r] = 0; }

  v4i fb[RING][2], fa[2][TM][2];
#pragma unroll
  for (int h = 0; h < RING - 1; ++h) load_w(fb[h], h);
  {
    Piece r[NIT];
#pragma unroll
    for (int it = 0; it < NIT; ++it) r[it] = load_piece(it, 0);
#pragma unroll
    for (int it = 0; it < NIT; ++it) store_piece(it, r[it], 0);
  }
  __syncthreads();

  int at[TM];  // LDS offsets of the pixels of the tap in hand
  auto enter_tap = [&](int tap, int buffer) {
    const int shift = (tap / 3) * W + tap % 3;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int row = prow[i] + shift;
      const int a = buffer * PATCH + (row << 7) + (((row << 3) & 0x70) ^ fh16);
      at[i] = (mask[i] >> tap) & 1 ? a : 2 * PATCH + fh16;
    }
  };
  auto read_half = [&](v4i (&f)[TM][2], int half) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int d = 0; d < 2; ++d) f[i][d] = *reinterpret_cast<const v4i *>(lds_dyn + (at[i] ^ (half * 32 + d * 64)));
  };

  for (int c = 0; c < nc; ++c) {
    const int buffer = c & 1;
    enter_tap(0, buffer);
    read_half(fa[0], 0);
    // one burst where its registers are at hand: a load of filters behind it waits for it
    constexpr bool BURST = TM == 1 || NIT <= 2;
    Piece piece[BURST ? NIT : 2];
    static_for<0, 18>([&](auto h_c) {
      constexpr int h = decltype(h_c)::value;
      __builtin_amdgcn_sched_barrier(0);
      load_w(fb[(h + RING - 1) % RING], c * 18 + h + RING - 1);
      if constexpr (BURST && h == 0) {
#pragma unroll
        for (int it = 0; it < NIT; ++it) piece[it] = load_piece(it, c + 1);
      }
      if constexpr (!BURST && h % 2 == 0 && h / 2 < NIT) piece[(h / 2) % 2] = load_piece(h / 2, c + 1);
      if constexpr (h + 1 < 18) {
        if constexpr (h % 2 == 1) enter_tap((h + 1) / 2, buffer);
        read_half(fa[(h + 1) & 1], (h + 1) & 1);
      }
      if constexpr (BURST && h >= 4 && h - 4 < NIT) store_piece(h - 4, piece[h - 4], buffer ^ 1);
      if constexpr (!BURST && h % 2 == 1 && h >= 3 && (h - 3) / 2 < NIT) store_piece((h - 3) / 2, piece[((h - 3) / 2) % 2], buffer ^ 1);
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
static int launch_packed_epi(const void *x, const void *w, const PackedConvParams &p, const EpiDev &e, hipStream_t s) {
  constexpr int LDS = 2 * NIT * kPatchPx * 128 + 128, STAGE = 4 * 32 * (64 + 8) * 4;
  constexpr int LDS_BYTES = LDS > STAGE ? LDS : STAGE;
  auto kern = conv3x3_a16_packed_kernel<TM, NIT, EPI>;
  if (LDS_BYTES > 64 * 1024) {
    static std::atomic<bool> raised[64];
    if (raise_lds_limit((const void *)kern, LDS_BYTES, raised) != CATCHQ_OK) return CATCHQ_ERR_LAUNCH;
  }
  kern<<<p.g.nblocks, 256, LDS_BYTES, s>>>((const int16_t *)x, (const int8_t *)w, p, e);
  return launch_status();
}

template <int TM, int NIT>
static int launch_packed(const void *x, const void *w, const PackedConvParams &p, const EpiDev &e, hipStream_t s) {
  switch (pick_epilogue(p.g.N, e)) {
    case EPI_LK_Q16: return launch_packed_epi<TM, NIT, EPI_LK_Q16>(x, w, p, e, s);
    case EPI_LK_Y_Q16: return launch_packed_epi<TM, NIT, EPI_LK_Y_Q16>(x, w, p, e, s);
    case EPI_LK_RESA_Q16: return launch_packed_epi<TM, NIT, EPI_LK_RESA_Q16>(x, w, p, e, s);
    case EPI_LK_RESA_Y_Q16: return launch_packed_epi<TM, NIT, EPI_LK_RESA_Y_Q16>(x, w, p, e, s);
    case EPI_Y16: return launch_packed_epi<TM, NIT, EPI_Y16>(x, w, p, e, s);
    case EPI_SCALAR: return -1;
    default: return launch_packed_epi<TM, NIT, EPI_VECTOR>(x, w, p, e, s);
  }
}

// Where the blocks of 32 pixels leave most units without one, the waves that split K (ksplit.hip) are ahead: 5 x 13 x 13, 512 ->
// 1024 (108 blocks for 256 units; the whole network 1000 / 1045 us), 2 x 13 x 13 (44) 9.8 / 16.9, 2 x 26 x 26 (86) 10.8 / 10.6;
// 4 x 26 x 26 (170) 15.5 / 11.3.
// Columns that do not exist cost as much as others.  Beyond an eighth of them, epilogues without an instance of their own are behind
// (us, that kernel / this, to int16 behind a ReLU: 8 x 52 x 52, 128 -> 192 24.7 / 28.3, 16 x 26 x 26, 256 -> 384 37.9 / 39.7; of 224
// columns 2 x 52 x 52, 64 10.7 / 11.5), and so are the others' single rounds of blocks with long K (2 x 52 x 52, 512 -> 192, 169
// blocks of 32, 18.0 / 19.7; 4 x 52 x 52, 338, 34.1 / 32.8) and wide images (4 x 80 x 80, 192 -> 384 50.2 / 52.0).
bool conv3x3_a16_packed_takes(int N, int H, int W, int Ci, int Co, const EpiDev &e) {
  const int64_t M = (int64_t)N * H * W, columns = ((int64_t)Co + 255) / 256 * 256;
  if (!conv3x3_a16_packed_filters(Co, Ci) || M * Ci * 2 >= (1ll << 31) || columns / 32 * Ci * 288 >= (1ll << 31) - (1 << 20)) return false;
  const int epi = pick_epilogue(Co, e);
  if (W > 95 || H >= (1 << 20) || epi == EPI_SCALAR) return false;
  const int64_t blocks = (M + 31) / 32 * (columns / 256);
  if (blocks * 8 < 5 * (int64_t)e.cus) return false;
  const bool own = epi == EPI_LK_Q16 || epi == EPI_LK_Y_Q16 || epi == EPI_LK_RESA_Q16 || epi == EPI_LK_RESA_Y_Q16 || epi == EPI_Y16;
  if (!own) return Co * 16ll >= columns * 15;
  return Co * 8ll >= columns * 7 || ((Ci < 256 || blocks * 4 >= 5 * (int64_t)e.cus) && (W <= 63 || Co < 256));
}

int64_t packed3x3_filter_bytes(int64_t Co, int64_t Ci) { return (Co + 31) / 32 * Ci * 288; }
// (with the sums, and what the last waves request beyond their filters)
int64_t packed3x3_bytes(int64_t Co, int64_t Ci) { return packed3x3_filter_bytes(Co, Ci) + (Co + 31) / 32 * 128 + kMaxAhead * 1024; }

// x [N, H, W, Ci] int16, packed: pack3x3's; -1: not this kernel's shape
int conv3x3_a16_packed(const void *x, const void *packed, int N, int H, int W, int Ci, int Co, const EpiDev &e, hipStream_t s) {
  if (!conv3x3_a16_packed_takes(N, H, W, Ci, Co, e)) return -1;
  PackedConvParams p = {};
  p.g.M = (int64_t)N * H * W;
  p.g.N = Co; p.g.K = 9 * Ci; p.g.H = H; p.g.W = W; p.g.Ci = Ci;
  p.x_bytes = (unsigned)(p.g.M * Ci * 2);
  p.w_bytes = (unsigned)packed3x3_bytes(Co, Ci);
  p.sums = reinterpret_cast<const int *>(static_cast<const int8_t *>(packed) + packed3x3_filter_bytes(Co, Ci));
  p.g.tiles_n = (Co + 255) / 256;
  // Blocks of 64 pixels read half the filters; with fewer than one for a unit, blocks of 32 (8 x 13 x 13, 512 -> 1024 28 / 18 us,
  // 4 x 26 x 26, 256 -> 512 18 / 11; but 16 x 52 x 52 31 / 35).
  const bool wide = (p.g.M + 63) / 64 * p.g.tiles_n >= e.cus;
  const int bm = wide ? 64 : 32;
  p.g.tiles_m = (int)((p.g.M + bm - 1) / bm);
  if ((int64_t)p.g.tiles_m * p.g.tiles_n > 0x7fffffff) return -1;
  p.g.nblocks = p.g.tiles_m * p.g.tiles_n;
  p.m_fastest = p.w_bytes > p.x_bytes;
  const int passes = (bm + 2 * W + 2 + kPatchPx - 1) / kPatchPx;
  if (wide) {
    switch (passes) {
      case 1: case 2: return launch_packed<2, 2>(x, packed, p, e, s);
      case 3: return launch_packed<2, 3>(x, packed, p, e, s);
      case 4: return launch_packed<2, 4>(x, packed, p, e, s);
      default: return -1;
    }
  }
  switch (passes) {
    case 1: case 2: return launch_packed<1, 2>(x, packed, p, e, s);
    case 3: return launch_packed<1, 3>(x, packed, p, e, s);
    case 4: return launch_packed<1, 4>(x, packed, p, e, s);
    default: return -1;
  }
}

// w [Co, 3, 3, Ci] -> [32 columns][64 channels][tap][half] in fragment order, then 128 times the columns' sums (zeros beyond Co).
// One block per 32 columns, its waves every sixteenth KiB; runs once per plan.
constexpr int kPackWaves3 = 16;
__global__ __launch_bounds__(64 * kPackWaves3) void pack3x3_kernel(const int8_t *__restrict__ w, int8_t *__restrict__ out,
                                                                   int *__restrict__ sums, int Co, int Ci) {
  __shared__ int parts[kPackWaves3][32];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int frow = lane & 31, fhalf = lane >> 5;
  const int n = blockIdx.x * 32 + frow;
  const int pieces = Ci / 64 * 18;
  int sum = 0;
  for (int i = wave; i < pieces; i += kPackWaves3) {
    const int half = i & 1, tap = (i >> 1) % 9, c = (i >> 1) / 9;
    v4i v = {0, 0, 0, 0};
    if (n < Co) v = *reinterpret_cast<const v4i *>(w + ((int64_t)n * 9 + tap) * Ci + c * 64 + half * 32 + fhalf * 16);
#pragma unroll
    for (int d = 0; d < 4; ++d) sum = __builtin_amdgcn_sdot4(v[d], 0x01010101, sum, false);
    *reinterpret_cast<v4i *>(out + (int64_t)blockIdx.x * Ci * 288 + (int64_t)i * 1024 + lane * 16) = v;
  }
  sum += __shfl_xor(sum, 32, 64);
  if (fhalf == 0) parts[wave][frow] = sum;
  __syncthreads();
  if (threadIdx.x < 32) {
    unsigned total = 0;
    for (int i = 0; i < kPackWaves3; ++i) total += (unsigned)parts[i][threadIdx.x];
    sums[blockIdx.x * 32 + threadIdx.x] = (int)(total << 7);
  }
}

int pack3x3(const void *w, void *packed, int64_t Co, int64_t Ci, hipStream_t s) {
  int *sums = reinterpret_cast<int *>(static_cast<int8_t *>(packed) + packed3x3_filter_bytes(Co, Ci));
  pack3x3_kernel<<<(unsigned)((Co + 31) / 32), 64 * kPackWaves3, 0, s>>>((const int8_t *)w, (int8_t *)packed, sums, (int)Co, (int)Ci);
  return launch_status();
}

}  // namespace catchq
