// int16 linears and convolutions on operands split into digits beforehand: exact in 64 bits.
//
// With  x = 256 xh + xl + 128  and  w = 256 wh + wl + 128  (high byte signed, low byte biased into int8)
//   sum x w = 65536 S_hh + 256 (S_hl + S_lh) + S_ll + 128 (X + sum w),   X = sum (256 xh + xl)
// over the K positions walked; positions beyond K and rows beyond M and N hold the value 0.  The four sums are int8 products
// (|S| <= K 2^14, K < 2^14), the combination is done in fp64, which holds every value of it, and its one
// conversion to fp32 is the int64 sum's.
//
// The kernel for int16 operands as they lie splits every fragment in every wave that reads it: 20 vector operations a fragment
// beside the matrix instructions, and sums of both operands' digits.  Here the quantizer writes the activations' digits and the
// preparation of a weight writes its, both in the order of the matrix instruction's lanes -- [row / 32][k / 32][high, low
// digits], a kilobyte each --, so that every transfer is a run of memory and every LDS read is conflict-free as it lies.  A
// block of NW waves owns 64 rows x 32 NW columns: the rows go to LDS, 256 values of K at a time and the next ones under way; a
// wave's weights come straight into its registers, eight K sub-steps of 32 ahead.  64 x 32 outputs a wave are eight matrix
// instructions for two kilobytes of weights and four LDS reads.  What bounds it: the transfers from the Infinity Cache through
// L2 (25 B a clock and unit, a slab of 96 KB in 3700 clocks where its multiplications take 2800), the first slab (4100 clocks)
// and the epilogue (4000).  Tried without gain: floats converted by the blocks themselves (every run of columns converts them
// again: 67 us), K shared between two groups of waves.
//
// A convolution's activations lie by pixels instead, [pixel][channel / 32][high, low digits of 32 channels] with a pixel of zeros behind
// the last one, and a transfer of 32 pixels' digits is 64 lanes' addresses: tap and channels are the wave's, whether the tap is in the
// image a bit of the lane's.  It lands as the linear's do.
//
// Measured: see gemm_digits_bytes and conv_digits_bytes below.
#include <type_traits>

#include "nchw_quantize.h"

namespace catchq {

typedef __attribute__((address_space(3))) void *lds_ptr_t;

struct DigitParams {
  int64_t M;
  int N, nk;  // sub-steps of 32 values of K, a multiple of four
  int tiles_m, tiles_n;
  int die_cols, rect_m, rect_n;  // the dies as a grid, tiles of a die's rectangle
  unsigned a_bytes, b_bytes;
};

__device__ __forceinline__ v4i digit_read(unsigned addr) {
  v4i v;
  asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(addr));
  return v;
}
template <int N>
__device__ __forceinline__ void digit_wait(v4i (&f)[2][2]) {  // at most N LDS reads under way: f is valid
#pragma unroll
  for (int i = 0; i < 2; ++i) asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(f[i][0]), "+v"(f[i][1]) : "n"(N) : "memory");
}

struct DigitConv {
  int H, W, Ho, Wo, ph, pw, sh, sw, dh, dw, kh, kw;
  int c32;              // channels / 32, rounded up
  unsigned pitch;       // bytes of a pixel
  unsigned zero;        // the pixel of zeros
  unsigned magic_c32, mask_c32, magic_kw, mask_kw;  // ceil(2^32 / d), mask 0; for d = 1 magic 0, mask ~0
};
struct NoConv {};
__device__ __forceinline__ unsigned digit_div(unsigned n, unsigned magic, unsigned mask) { return __umulhi(n, magic) + (n & mask); }

// WN of the four waves side by side, 32 columns each; SUB: sub-steps of a slab
template <int EPI, bool RAGGED, int WN, int SUB, class Conv>
__global__ __launch_bounds__(256, 2) void gemm_digits_kernel(const int8_t *__restrict__ A, const int8_t *__restrict__ B,
                                                                      const int *__restrict__ col_sums, DigitParams p, EpiDev e, Conv c) {
  constexpr bool CONV = !std::is_same<Conv, NoConv>::value;
  resolve_exp2(e);
  constexpr int NW = 4, BM = 64 * (NW / WN), TM = 2, RING = SUB, STAGE = 36;
  constexpr int ROW_TILES = BM / 32, PIECES = ROW_TILES * SUB * 2, SLAB_BYTES = PIECES * 1024;  // [row / 32][sub-step][digit]
  extern __shared__ __attribute__((aligned(16))) int8_t lds_dyn[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wn = wave % WN, wm = wave / WN;
  // a die's blocks (every eighth) cover a rectangle of tiles: what its L2 takes in is a part of the rows and a part of the weights
  const int die = blockIdx.x & 7, place = blockIdx.x >> 3;
  const int tile_m = die / p.die_cols * p.rect_m + place / p.rect_n, chunk = die % p.die_cols * p.rect_n + place % p.rect_n;
  if (tile_m >= p.tiles_m || chunk >= p.tiles_n) return;
  const int64_t m0 = (int64_t)tile_m * BM + wm * 64;  // this wave's rows
  const int n32 = (p.N + 31) / 32, m32 = (int)((p.M + 31) / 32), t = chunk * WN + wn;
  const bool columns = t < n32;  // (without: the wave helps with the rows)
  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void *)A, 0, (int)p.a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void *)B, 0, (int)p.b_bytes, 0x00020000);
  const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) int8_t *)lds_dyn;
  const int my16 = lane * 16;

  // rows: piece j of a slab = (row tile j / (2 SUB), sub-step j / 2 % SUB, digit j % 2).  Pieces past the last sub-step or row
  // tile repeat the last one (a convolution's are zeros): their products are not taken, or met by zeros, their rows not stored.
  constexpr int MINE = PIECES / NW;  // pieces a wave moves, all of one row tile
  static_assert(ROW_TILES <= NW);
  const int row_tile = wave * MINE / (2 * SUB);
  unsigned px_off = 0, px_zero = 0, px_taps = 0;  // of this lane's pixel: its first tap, a pixel of zeros, bit per tap in the image
  if constexpr (CONV) {
    const int64_t m = (int64_t)tile_m * BM + row_tile * 32 + (lane & 31);
    const unsigned mm = (unsigned)(m < p.M ? m : 0), t = mm / (unsigned)c.Wo, img = t / (unsigned)c.Ho;
    const int hi = (int)(t - img * (unsigned)c.Ho) * c.sh - c.ph, wi = (int)(mm - t * (unsigned)c.Wo) * c.sw - c.pw;
    px_off = ((img * (unsigned)c.H + (unsigned)hi) * (unsigned)c.W + (unsigned)wi) * c.pitch + (unsigned)(lane >> 5) * 16u;  // mod 2^32
    px_zero = c.zero + (unsigned)(lane >> 5) * 16u;
    unsigned cols = 0;
    for (int q = 0; q < c.kw; ++q) cols |= ((unsigned)(wi + q * c.dw) < (unsigned)c.W ? 1u : 0u) << q;
    for (int r = 0; r < c.kh; ++r) px_taps |= (m < p.M && (unsigned)(hi + r * c.dh) < (unsigned)c.H ? cols : 0u) << (r * c.kw);
  }
  auto issue_a = [&](int slab) {
#pragma unroll
    for (int i = 0; i < MINE; i += 2) {
      const int j = wave * MINE + i, ks = slab * SUB + j / 2 % SUB;
      lds_ptr_t dst = (lds_ptr_t)(lds_dyn + (slab & 1) * SLAB_BYTES + j * 1024);
      if constexpr (CONV) {
        const unsigned tap = digit_div((unsigned)ks, c.magic_c32, c.mask_c32), ch = (unsigned)ks - tap * (unsigned)c.c32;
        const unsigned r = digit_div(tap, c.magic_kw, c.mask_kw), q = tap - r * (unsigned)c.kw;
        const unsigned at = (r * (unsigned)(c.dh * c.W) + q * (unsigned)c.dw) * c.pitch;
        unsigned from = (px_taps >> tap) & 1u ? px_off + at : px_zero;
        asm volatile("" : "+v"(from));  // one select and one load, not two loads under complementary masks
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, dst, 16, (int)from, (int)(ch * 64u), 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_ptr_t)(lds_dyn + (slab & 1) * SLAB_BYTES + j * 1024 + 1024), 16, (int)from,
                                                 (int)(ch * 64u + 32u), 0, 0);
      } else {
        const int from = (min(tile_m * ROW_TILES + row_tile, m32 - 1) * p.nk + min(ks, p.nk - 1)) * 2048;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, dst, 16, my16, from, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_ptr_t)(lds_dyn + (slab & 1) * SLAB_BYTES + j * 1024 + 1024), 16, my16,
                                                 from + 1024, 0, 0);
      }
    }
  };
  v4i fb[RING][2];  // this wave's weights of a slab; a slot is refilled for the next slab
  const int b_run = min(t, n32 - 1) * p.nk;
  auto fetch_b = [&](v4i (&f)[2], int ks) {  // (past the last step: a spare load of it)
    const int off = (b_run + min(ks, p.nk - 1)) * 2048;
    f[0] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_b, my16, off, 0));
    f[1] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_b, my16, off + 1024, 0));
  };

  v16i hh[TM], mid[TM], ll[TM];  // (|S_hl + S_lh| <= K 2^15)
  int xh_sum[TM] = {}, xl_sum[TM] = {};
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) hh[i][r] = mid[i][r] = ll[i][r] = 0;
  auto multiply = [&](v4i (&x)[TM][2], v4i (&w)[2]) {  // (the two that share an accumulator stay four instructions apart)
#pragma unroll
    for (int i = 0; i < TM; ++i) mid[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x[i][0], w[1], mid[i], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < TM; ++i) hh[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x[i][0], w[0], hh[i], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < TM; ++i) mid[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x[i][1], w[0], mid[i], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < TM; ++i) ll[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x[i][1], w[1], ll[i], 0, 0, 0);
  };
  auto add_digits = [&](v4i (&x)[TM][2]) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        xh_sum[i] = __builtin_amdgcn_sdot4(x[i][0][d], 0x01010101, xh_sum[i], false);
        xl_sum[i] = __builtin_amdgcn_sdot4(x[i][1][d], 0x01010101, xl_sum[i], false);
      }
  };
  const int slabs = (p.nk + SUB - 1) / SUB;
  issue_a(0);
#pragma unroll
  for (int r = 0; r < RING; ++r) fetch_b(fb[r], r);
  // the outputs' constants, needed at the very end
  typedef typename EpiOf<EPI>::type S;
  const int n0 = min(t, n32 - 1) * 32, cg = lane & 7, n = n0 + cg * 4;
  EpiLane L;
  if constexpr (RAGGED) L = epi_lane_setup_ragged<S>(n, p.N, e);
  else L = epi_lane_setup<S>(n, n < p.N, e);
  const v4i col_sum = *reinterpret_cast<const v4i *>(col_sums + n0 + cg * 4);
  for (int slab = 0; slab < slabs; ++slab) {
    // this wave's pieces of the slab have landed: what was sent for behind them are weights of this wave.  (Of a wave without columns
    // nothing uses those: whether they were sent for at all is the compiler's choice, so it waits for everything.)
    if (slab == 0 || (CONV && !columns)) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * 4) : "memory");
    __syncthreads();  // everyone's; and nobody reads the other half of the buffer any more
    if (slab + 1 < slabs) issue_a(slab + 1);
    const int first = slab * SUB, sub = min(SUB, p.nk - first);  // (four or eight)
    const unsigned at = lds_base + (unsigned)((slab & 1) * SLAB_BYTES + wm * TM * SUB * 2048 + my16);
    v4i fa[2][TM][2];
    auto fetch_a = [&](v4i (&f)[TM][2], int s) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int d = 0; d < 2; ++d) f[i][d] = digit_read(at + (unsigned)(((i * SUB + s) * 2 + d) * 1024));
    };
    fetch_a(fa[0], 0);
    auto four = [&](auto from) {
      constexpr int FROM = decltype(from)::value;
#pragma unroll
      for (int r = FROM; r < FROM + 4; ++r) {
        fetch_a(fa[(r + 1) & 1], r + 1 < RING ? r + 1 : r);  // under way before this step's multiplications
        digit_wait<2 * TM>(fa[r & 1]);
        if (!CONV || columns) multiply(fa[r & 1], fb[r]);  // (the question costs a linear 4 %)
        fetch_b(fb[r], first + RING + r);
        if (wn == r % WN) add_digits(fa[r & 1]);  // a wave takes the sums of every WN-th step
      }
    };
    four(std::integral_constant<int, 0>{});
    if constexpr (SUB > 4) {
      if (sub > 4) four(std::integral_constant<int, 4>{});
    }
    digit_wait<0>(fa[0]);  // (the spare read)
  }

  // ---- outputs -----------------------------------------------------------------------------------------------------------------
  // value = 65536 hh + 128 (2 mid + row's digit sum + sum w) + ll, in fp64.  The sums go through LDS as they are, and the
  // arithmetic is a rolled loop: in the registers' order, with its carries in 32-bit integers and its eight turns unrolled it
  // took 0.5 us of 19 more at 1379 x 1000 -> 1001 and 2 us of 52 at 4096 x 768 -> 3072.
  __syncthreads();  // the slabs are dead: the waves' shares of the rows' digit sums, then [row tile's sums][32][STAGE] of a wave
  int *rows = reinterpret_cast<int *>(lds_dyn);  // [NW][64]
  const int frow = lane & 31, fhalf = lane >> 5;
#pragma unroll
  for (int i = 0; i < TM; ++i) {  // a lane holds the sums of row (lane & 31) over its half of a sub-step
    const int part = 256 * xh_sum[i] + xl_sum[i], both = part + __shfl_xor(part, 32, 64);
    if (fhalf == 0) rows[wave * 64 + i * 32 + frow] = both;
  }
  int *const stage = rows + NW * 64 + wave * 3 * 32 * STAGE;
  __syncthreads();
  if (!columns) return;
  int my_row = 0;  // the digit sum of row `lane`
#pragma unroll
  for (int w = 0; w < WN; ++w) my_row += rows[(wm * WN + w) * 64 + lane];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      int *at = stage + (8 * (r >> 2) + 4 * fhalf + (r & 3)) * STAGE + frow;
      at[0] = hh[i][r];
      at[32 * STAGE] = mid[i][r];
      at[2 * 32 * STAGE] = ll[i][r];
    }
#pragma unroll 1
    for (int it = 0; it < 4; ++it) {
      const int row = it * 8 + (lane >> 3);
      const int *at = stage + row * STAGE + cg * 4;
      const v4i h16 = *reinterpret_cast<const v4i *>(at), m16 = *reinterpret_cast<const v4i *>(at + 32 * STAGE);
      const v4i l16 = *reinterpret_cast<const v4i *>(at + 2 * 32 * STAGE);
      const int row_sum = __shfl(my_row, i * 32 + row, 64);
      v4f sums;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int both = 2 * m16[k] + row_sum + col_sum[k];  // (fewer than 2^14 positions of K: each less than 2^17)
        sums[k] = (float)__builtin_fma((double)h16[k], 65536.0, __builtin_fma((double)both, 128.0, (double)l16[k]));
      }
      const int64_t m = m0 + i * 32 + row;
      if (m < p.M && n < p.N) {
        const v4f none = {0.f, 0.f, 0.f, 0.f};
        if constexpr (RAGGED) epi_vec4<S>(sums, none, L, EpiAtRagged{m * p.N + n, p.N - n}, e);
        else epi_vec4<S>(sums, none, L, m * p.N + n, e);
      }
    }
  }
}

// 16 values of lane's row and half of a sub-step -> their digits, at [run][ks]
__device__ __forceinline__ void store_digits(int8_t *out, int64_t run, int ks, int nk, int lane, const int (&q)[16]) {
  v4i c[2], hi, lo;
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int d = 0; d < 4; ++d) c[h][d] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_pk_i16(q[h * 8 + d * 2], q[h * 8 + d * 2 + 1]));
  split_i16(c[0], c[1], hi, lo);
  v4i *dst = reinterpret_cast<v4i *>(out) + (run * nk + ks) * 128;
  dst[lane] = hi;
  dst[64 + lane] = lo;
}

// x [M, K] floats -> digits of sat(rne(x 2^-position)) at 16 bits.  A wave takes 32 rows x a sub-step: a lane reads 16 values of
// its row, wherever they lie; two lanes share a cache line of halfs.  (4096 x 768 floats 5.0 us, 1379 x 1000 halfs 3.9.)
template <typename TIn>
__global__ __launch_bounds__(256) void quantize_digits_kernel(const TIn *__restrict__ x, int8_t *__restrict__ out, int64_t M, int K,
                                                              int nk, int64_t tasks, int neg_pos) {
  struct __attribute__((aligned(sizeof(TIn)))) run16 { TIn v[16]; };
  const int lane = threadIdx.x & 63;
  const int64_t task = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (task >= tasks) return;
  const int64_t run = task / nk, m = run * 32 + (lane & 31);
  const int ks = (int)(task - run * nk), k = ks * 32 + (lane >> 5) * 16;
  const TIn *row = x + (m < M ? m : M - 1) * K;
  float v[16];
  if (k + 16 <= K) {
    const run16 t = *reinterpret_cast<const run16 *>(row + k);
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = (float)t.v[i];
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = k + i < K ? (float)row[k + i] : 0.0f;
  }
  int q[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) q[i] = cvt_i32_sat(__builtin_rintf(__builtin_ldexpf(m < M ? v[i] : 0.0f, neg_pos)));
  store_digits(out, run, ks, nk, lane, q);
}

// w [N, ld] int16, K values of a row used -> digits, zeros beyond N and K, and the rows' sums (once per weight that is
// read packed).  Rows of `taps` runs of K values: every run starts on a sub-step.  A block takes 32 rows, its waves every sixteenth
// sub-step: bound by the latency of the steps that a wave takes one after the other.  1001 x 1000: 5.7 us; a pass that packs (1379 rows,
// half, on a new weight) 191 us with one wave for a block's rows, 137 with sixteen.
constexpr int kPackWaves = 16;
__global__ __launch_bounds__(64 * kPackWaves) void pack_digits_kernel(const int16_t *__restrict__ w, int8_t *__restrict__ out,
                                                                      int *__restrict__ sums, int N, int taps, int K, int64_t ld, int nk) {
  struct __attribute__((aligned(2))) run16 { int16_t v[16]; };
  __shared__ int parts[kPackWaves][32];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = blockIdx.x * 32 + (lane & 31);
  const int16_t *const row = w + (n < N ? n : N - 1) * ld;
  int sum = 0;
  for (int ks = wave; ks < nk; ks += kPackWaves) {
    const int tap = taps > 1 ? ks / ((K + 31) / 32) : 0, k = (ks - tap * ((K + 31) / 32)) * 32 + (lane >> 5) * 16;
    const int16_t *const run = row + (tap < taps ? tap : 0) * (int64_t)K;
    int q[16];
    if (k + 16 <= K) {
      const run16 t = *reinterpret_cast<const run16 *>(run + k);
#pragma unroll
      for (int i = 0; i < 16; ++i) q[i] = t.v[i];
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) q[i] = k + i < K ? run[k + i] : 0;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      q[i] = n < N && tap < taps ? q[i] : 0;
      sum += q[i];
    }
    store_digits(out, blockIdx.x, ks, nk, lane, q);
  }
  sum += __shfl_xor(sum, 32, 64);
  if (lane < 32) parts[wave][lane] = sum;
  __syncthreads();
  if (threadIdx.x < 32) {
    int total = 0;
#pragma unroll
    for (int i = 0; i < kPackWaves; ++i) total += parts[i][threadIdx.x];
    sums[n] = total;
  }
}

static int64_t digit_steps(int64_t K) { return (K + 127) / 128 * 4; }
static int64_t digit_bytes(int64_t rows, int64_t K) { return (rows + 31) / 32 * digit_steps(K) * 2048; }

static int64_t conv_digit_steps(int64_t taps, int64_t Ci) { return (taps * ((Ci + 31) / 32) + 3) / 4 * 4; }

// (with the sums)
int64_t packed_digits_bytes(int64_t N, int64_t taps, int64_t K) {
  return (N + 31) / 32 * ((taps > 1 ? conv_digit_steps(taps, K) : digit_steps(K)) * 2048 + 32 * 4);
}

// rows of `taps` runs of K values each, ld values apart
int pack_digits(const void *w, int64_t N, int64_t taps, int64_t K, int64_t ld, void *packed, hipStream_t s) {
  const int64_t nk = taps > 1 ? conv_digit_steps(taps, K) : digit_steps(K), runs = (N + 31) / 32;
  int *sums = reinterpret_cast<int *>(static_cast<int8_t *>(packed) + runs * nk * 2048);
  pack_digits_kernel<<<(unsigned)runs, 64 * kPackWaves, 0, s>>>((const int16_t *)w, (int8_t *)packed, sums, (int)N, (int)taps, (int)K, ld, (int)nk);
  return launch_status();
}

// EPI_Y32 or EPI_Y16, with or without aligned rows; 0: an epilogue this kernel does not have
static int digit_epilogue(int N, const EpiDev &e) {
  int epi = pick_epilogue(N, e);
  if (epi != EPI_Y32 && epi != EPI_Y16) epi = ragged_epilogue(N, e);
  return epi == EPI_Y32 || epi == EPI_Y16 ? epi : 0;
}

// The tiles of blocks of WN waves side by side, and the dies' share of them; the blocks of the launch.
static int64_t digit_tiles(DigitParams &p, int WN) {
  const int BM = 64 * (4 / WN);
  p.tiles_m = (int)((p.M + BM - 1) / BM);
  p.tiles_n = ((p.N + 31) / 32 + WN - 1) / WN;
  int64_t best = -1;
  for (int cols = 1; cols <= 8; cols *= 2) {
    const int64_t rm = (p.tiles_m + 8 / cols - 1) / (8 / cols), rn = (p.tiles_n + cols - 1) / cols;
    // the tiles of the fullest die, then the rows that its L2 takes in: 4096 x 768 -> 3072 54.6 us with the rows' tiles dealt
    // out alone, 50.4 in rectangles, 512 x 768 -> 3072 13.4 and 11.4
    const int64_t cost = rm * rn * 64 + rm * 64 + rn * 128;
    if (best < 0 || cost < best) best = cost, p.die_cols = cols, p.rect_m = (int)rm, p.rect_n = (int)rn;
  }
  return 8ll * p.rect_m * p.rect_n;
}
static int conv_digits_side(int Co) { return Co <= 64 ? 2 : 4; }  // waves side by side

template <int WN, int SUB, class Conv>
static int launch_digits(const int8_t *a, const int8_t *b, const int *sums, DigitParams p, const Conv &c, const EpiDev &e, hipStream_t s) {
  constexpr int LDS_BYTES = 64 * 1024;  // two slabs; behind the loop 4 x (64 + 3 x 32 x 36) sums
  static_assert(2 * 64 * (4 / WN) / 32 * SUB * 2048 <= LDS_BYTES);
  const unsigned blocks = (unsigned)digit_tiles(p, WN);
  const bool whole = pick_epilogue(p.N, e) == EPI_Y32 || pick_epilogue(p.N, e) == EPI_Y16;
  auto kern = digit_epilogue(p.N, e) == EPI_Y32
                  ? (whole ? gemm_digits_kernel<EPI_Y32, false, WN, SUB, Conv> : gemm_digits_kernel<EPI_Y32, true, WN, SUB, Conv>)
                  : (whole ? gemm_digits_kernel<EPI_Y16, false, WN, SUB, Conv> : gemm_digits_kernel<EPI_Y16, true, WN, SUB, Conv>);
  kern<<<blocks, 256, LDS_BYTES, s>>>(a, b, sums, p, e, c);
  return launch_status();
}

// Bytes of the activations' digits where this route serves the product; 0: another one does.
//
// With the quantizer, before (the quantizer of int16 and the kernel for operands as they lie) and now, us (half activations
// where marked): 4096 x 768 -> 3072 99 / 54, 8192 x 1024 -> 1024 half 79 / 46, 5000 x 2048 -> 1024 94 / 58,
// 3398 x 168 -> 3583 half 64 / 34, 16384 x 256 -> 256 28.5 / 19.5, 2048 x 256 -> 2048 24.4 / 15.8, 1379 x 1000 -> 1001 half
// 19.7 / 18.0, 860 x 88 -> 2531 20.7 / 13.3, 3290 x 360 -> 310 (156 blocks) 14.6 / 13.3.  A block walks all of K, so few of
// them leave units idle: 339 x 203 -> 2765 half (132 blocks) 10.3 / 11.8, 908 x 875 -> 737 half (90) 14.9 / 16.7,
// 1202 x 2480 -> 253 (38) 19.6 / 27.4, 116 x 1514 -> 627 half (10) 10.5 / 19.0.
int64_t gemm_digits_bytes(int64_t M, int64_t N, int64_t K, const EpiDev &e) {
  if (M >= (1ll << 31) - 64 || N >= (1 << 24) || !digits_sizes(M, N, K, e.cus)) return 0;
  const int64_t blocks = (M + 63) / 64 * ((N + 127) / 128), bytes = digit_bytes(M, K);
  if (blocks >= (1 << 27) || bytes >= (1ll << 31) || digit_bytes(N, K) >= (1ll << 31)) return 0;
  return digit_epilogue((int)N, e) ? bytes : 0;
}

// x [M, K] floats (halfs) -> its digits in `digits` -> the product with the packed weights of N rows
int gemm_digits(const void *x, bool half, int position, const void *packed, int64_t M, int64_t N, int64_t K, void *digits,
                const EpiDev &e, hipStream_t s) {
  DigitParams p = {};
  p.M = M;
  p.N = (int)N;
  p.nk = (int)digit_steps(K);
  p.a_bytes = (unsigned)digit_bytes(M, K);
  p.b_bytes = (unsigned)digit_bytes(N, K);
  const int8_t *const a = static_cast<const int8_t *>(digits), *const b = static_cast<const int8_t *>(packed);
  const int *const sums = reinterpret_cast<const int *>(b + p.b_bytes);
  // (a sub-step a wave: two or four of them measured 0.4 to 1 us slower)
  const int64_t tasks = (M + 31) / 32 * p.nk;
  const unsigned quantizers = (unsigned)((tasks + 3) / 4);
  if (half) quantize_digits_kernel<_Float16><<<quantizers, 256, 0, s>>>((const _Float16 *)x, (int8_t *)digits, M, (int)K, p.nk, tasks, -position);
  else quantize_digits_kernel<float><<<quantizers, 256, 0, s>>>((const float *)x, (int8_t *)digits, M, (int)K, p.nk, tasks, -position);
  const int st = launch_status();
  if (st != CATCHQ_OK) return st;
  return launch_digits<4, 8>(a, b, sums, p, NoConv{}, e, s);
}

// channels-last floats -> digits by pixels, [pixel][channel / 32][high, low digits of 32 channels], and a pixel of zeros behind them: two
// lanes have a pixel's 32 channels (planes: nchw_quantize.h).
template <typename TIn>
__global__ __launch_bounds__(256) void quantize_pixel_digits_kernel(const TIn *__restrict__ x, int8_t *__restrict__ out, int64_t pixels,
                                                                    int C, int c32, int64_t tasks, int neg_pos) {
  struct __attribute__((aligned(sizeof(TIn)))) run16 { TIn v[16]; };
  const int64_t task = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (task >= tasks) return;
  const int64_t px = task / (2 * c32);
  const int ch = (int)(task - px * (2 * c32)) * 16;
  float v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = 0.0f;
  if (px < pixels) {
    const TIn *const row = x + px * C + ch;
    if (ch + 16 <= C) {
      const run16 t = *reinterpret_cast<const run16 *>(row);
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = (float)t.v[i];
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (ch + i < C) v[i] = (float)row[i];
    }
  }
  v4i c[2], hi, lo;
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int a = cvt_i32_sat(__builtin_rintf(__builtin_ldexpf(v[g * 8 + d * 2], neg_pos)));
      const int b = cvt_i32_sat(__builtin_rintf(__builtin_ldexpf(v[g * 8 + d * 2 + 1], neg_pos)));
      c[g][d] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_pk_i16(a, b));  // (saturates)
    }
  split_i16(c[0], c[1], hi, lo);
  v4i *const dst = reinterpret_cast<v4i *>(out + (px * c32 + ch / 32) * 64 + (ch & 16));
  dst[0] = hi;
  dst[2] = lo;
}

// Bytes of the activations' digits where this route serves the convolution; 0: another one does.
int64_t conv_digits_bytes(int N, int H, int W, int Ci, int Co, int kh, int kw, int Ho, int Wo, const EpiDev &e) {
  const int64_t M = (int64_t)N * Ho * Wo, pixels = (int64_t)N * H * W, c32 = (Ci + 31) / 32, taps = (int64_t)kh * kw;
  const int64_t bytes = (pixels + 1) * c32 * 64;
  if (taps > 25 || conv_digit_steps(taps, Ci) * 32 >= (1 << 14) || M >= (1ll << 31) - 128 || bytes >= (1ll << 31)) return 0;
  if (packed_digits_bytes(Co, taps, Ci) >= (1ll << 31) || e.resid || e.q || e.acc_out || !digit_epilogue(Co, e)) return 0;
  DigitParams tiles = {};
  tiles.M = M;
  tiles.N = Co;
  if (digit_tiles(tiles, conv_digits_side(Co)) >= (1 << 24)) return 0;  // (a launch has less than 2^32 lanes)
  return conv_digits_sizes(M, Co, Ci, taps, e.cus) ? bytes : 0;
}

// x: x_ci channels of the filters' Ci, [N, H, W, x_ci] or (apart) [N, x_ci, H, W] floats or halfs; packed: pack_digits of Co rows of
// kh * kw runs of Ci
int conv_digits(const void *x, bool half, int position, int x_ci, bool apart, const void *packed, int N, int H, int W, int Ci, int Co,
                int kh, int kw, int ph, int pw, int sh, int sw, int dh, int dw, int Ho, int Wo, void *digits, const EpiDev &e,
                hipStream_t s) {
  const int64_t pixels = (int64_t)N * H * W;
  const int c32 = (Ci + 31) / 32;
  int8_t *const a = static_cast<int8_t *>(digits);
  if (apart) {
    auto planes = [&](auto *from) { return pixel_quantize<typename std::remove_cv<typename std::remove_reference<decltype(*from)>::type>::type, PX_DIGITS>(from, a, N, x_ci, (int64_t)H * W, c32 * 64, position, 1.0f, pixels * c32 * 64, s); };
    if (!(half ? planes(static_cast<const _Float16 *>(x)) : planes(static_cast<const float *>(x)))) return CATCHQ_ERR_UNSUPPORTED;
  } else {
    const int64_t tasks = (pixels + 1) * c32 * 2;
    const unsigned quantizers = (unsigned)((tasks + 255) / 256);
    if (half) quantize_pixel_digits_kernel<_Float16><<<quantizers, 256, 0, s>>>((const _Float16 *)x, a, pixels, x_ci, c32, tasks, -position);
    else quantize_pixel_digits_kernel<float><<<quantizers, 256, 0, s>>>((const float *)x, a, pixels, x_ci, c32, tasks, -position);
  }
  const int st = launch_status();
  if (st != CATCHQ_OK) return st;
  DigitParams p = {};
  p.M = (int64_t)N * Ho * Wo;
  p.N = Co;
  p.nk = (int)conv_digit_steps(kh * kw, Ci);
  p.a_bytes = (unsigned)((pixels + 1) * c32 * 64);
  p.b_bytes = (unsigned)((int64_t)(Co + 31) / 32 * p.nk * 2048);
  DigitConv c = {H, W, Ho, Wo, ph, pw, sh, sw, dh, dw, kh, kw, c32, (unsigned)c32 * 64u, (unsigned)(pixels * c32 * 64), 0, 0, 0, 0};
  auto magic = [](unsigned d, unsigned *m, unsigned *mask) {  // (dividends and divisors below 2^16)
    *m = d <= 1 ? 0u : (unsigned)(((1ull << 32) + d - 1) / d);
    *mask = d <= 1 ? ~0u : 0u;
  };
  magic(c32, &c.magic_c32, &c.mask_c32);
  magic(kw, &c.magic_kw, &c.mask_kw);
  const int8_t *const b = static_cast<const int8_t *>(packed);
  const int *const sums = reinterpret_cast<const int *>(b + p.b_bytes);
  return conv_digits_side(Co) == 2 ? launch_digits<2, 4>(a, b, sums, p, c, e, s) : launch_digits<4, 8>(a, b, sums, p, c, e, s);
}

}  // namespace catchq
