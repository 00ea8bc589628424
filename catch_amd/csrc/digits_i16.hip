// int16 linears on operands split into digits beforehand: exact in 64 bits.
//
// With  x = 256 xh + xl + 128  and  w = 256 wh + wl + 128  (high byte signed, low byte biased into int8)
//   sum x w = 65536 S_hh + 256 (S_hl + S_lh) + S_ll + 128 (X + sum w),   X = sum (256 xh + xl)
// over the K positions walked; positions beyond K and rows beyond M and N hold the value 0.  The four sums are int8 products
// (|S| <= K 2^14, K <= 2^13), the combination is done in fp64, which holds every value of it, and its one
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
// Measured: see gemm_digits_bytes below.
#include <type_traits>

#include "igemm_common.h"

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

template <int EPI, bool RAGGED>
__global__ __launch_bounds__(256, 2) void gemm_digits_kernel(const int8_t *__restrict__ A, const int8_t *__restrict__ B,
                                                                      const int *__restrict__ col_sums, DigitParams p, EpiDev e) {
  resolve_exp2(e);
  constexpr int NW = 4, BM = 64, TM = 2, SUB = 8, RING = 8, STAGE = 36;
  constexpr int PIECES = TM * SUB * 2, SLAB_BYTES = PIECES * 1024;  // of 256 values of K: [row / 32][sub-step][digit]
  extern __shared__ __attribute__((aligned(16))) int8_t lds_dyn[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // a die's blocks (every eighth) cover a rectangle of tiles: what its L2 takes in is a part of the rows and a part of the weights
  const int die = blockIdx.x & 7, place = blockIdx.x >> 3;
  const int tile_m = die / p.die_cols * p.rect_m + place / p.rect_n, chunk = die % p.die_cols * p.rect_n + place % p.rect_n;
  if (tile_m >= p.tiles_m || chunk >= p.tiles_n) return;
  const int64_t m0 = (int64_t)tile_m * BM;
  const int n32 = (p.N + 31) / 32, m32 = (int)((p.M + 31) / 32), t = chunk * NW + wave;
  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void *)A, 0, (int)p.a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void *)B, 0, (int)p.b_bytes, 0x00020000);
  const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) int8_t *)lds_dyn;
  const int my16 = lane * 16;

  // rows: piece j of a slab = (row tile j / (2 SUB), sub-step j / 2 % SUB, digit j % 2).  Pieces past the last sub-step or row
  // tile repeat the last one: their products are not taken, their rows not stored.
  auto issue_a = [&](int slab) {
#pragma unroll
    for (int i = 0; i < PIECES / NW; ++i) {
      const int j = wave * (PIECES / NW) + i;
      const int run = min(tile_m * TM + j / (2 * SUB), m32 - 1), ks = min(slab * SUB + j / 2 % SUB, p.nk - 1);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_ptr_t)(lds_dyn + (slab & 1) * SLAB_BYTES + j * 1024), 16, my16,
                                               ((run * p.nk + ks) * 2 + j % 2) * 1024, 0, 0);
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
    // this wave's pieces of the slab have landed: what was sent for behind them are weights of this wave
    if (slab == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * 4) : "memory");
    __syncthreads();  // everyone's; and nobody reads the other half of the buffer any more
    if (slab + 1 < slabs) issue_a(slab + 1);
    const int first = slab * SUB, sub = min(SUB, p.nk - first);  // (four or eight)
    const unsigned at = lds_base + (unsigned)((slab & 1) * SLAB_BYTES + my16);
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
        multiply(fa[r & 1], fb[r]);
        fetch_b(fb[r], first + RING + r);
        if (wave == r % NW) add_digits(fa[r & 1]);  // a wave takes the sums of every NW-th step
      }
    };
    four(std::integral_constant<int, 0>{});
    if (sub > 4) four(std::integral_constant<int, 4>{});
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
    if (fhalf == 0) rows[wave * BM + i * 32 + frow] = both;
  }
  int *const stage = rows + NW * BM + wave * 3 * 32 * STAGE;
  __syncthreads();
  if (t >= n32) return;
  int my_row = 0;  // the digit sum of row `lane`
#pragma unroll
  for (int w = 0; w < NW; ++w) my_row += rows[w * BM + lane];
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
        const int both = 2 * m16[k] + row_sum + col_sum[k];  // (K <= 8192)
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
// read packed).  A block takes 32 rows, its waves every sixteenth sub-step: bound by the latency of the steps that a wave
// takes one after the other.  1001 x 1000: 5.7 us; a pass that packs (1379 rows, half, on a new weight) 191 us with one wave for
// a block's rows, 137 with sixteen.
constexpr int kPackWaves = 16;
__global__ __launch_bounds__(64 * kPackWaves) void pack_digits_kernel(const int16_t *__restrict__ w, int8_t *__restrict__ out,
                                                                      int *__restrict__ sums, int N, int K, int64_t ld, int nk) {
  struct __attribute__((aligned(2))) run16 { int16_t v[16]; };
  __shared__ int parts[kPackWaves][32];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = blockIdx.x * 32 + (lane & 31);
  const int16_t *const row = w + (n < N ? n : N - 1) * ld;
  int sum = 0;
  for (int ks = wave; ks < nk; ks += kPackWaves) {
    const int k = ks * 32 + (lane >> 5) * 16;
    int q[16];
    if (k + 16 <= K) {
      const run16 t = *reinterpret_cast<const run16 *>(row + k);
#pragma unroll
      for (int i = 0; i < 16; ++i) q[i] = t.v[i];
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) q[i] = k + i < K ? row[k + i] : 0;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      q[i] = n < N ? q[i] : 0;
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

int64_t packed_digits_bytes(int64_t N, int64_t K) { return digit_bytes(N, K) + (N + 31) / 32 * 32 * 4; }  // (with the sums)

int pack_digits(const void *w, int64_t N, int64_t K, int64_t ld, void *packed, hipStream_t s) {
  int *sums = reinterpret_cast<int *>(static_cast<int8_t *>(packed) + digit_bytes(N, K));
  pack_digits_kernel<<<(unsigned)((N + 31) / 32), 64 * kPackWaves, 0, s>>>((const int16_t *)w, (int8_t *)packed, sums, (int)N, (int)K,
                                                                           ld, (int)digit_steps(K));
  return launch_status();
}

// EPI_Y32 or EPI_Y16, with or without aligned rows; 0: an epilogue this kernel does not have
static int digit_epilogue(int N, const EpiDev &e) {
  int epi = pick_epilogue(N, e);
  if (epi != EPI_Y32 && epi != EPI_Y16) epi = ragged_epilogue(N, e);
  return epi == EPI_Y32 || epi == EPI_Y16 ? epi : 0;
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
  constexpr int LDS_BYTES = 64 * 1024;  // two slabs; behind the loop 4 x (64 + 3 x 32 x 36) sums
  p.tiles_m = (int)((p.M + 63) / 64);
  p.tiles_n = ((p.N + 31) / 32 + 3) / 4;
  int64_t best = -1;
  for (int cols = 1; cols <= 8; cols *= 2) {
    const int64_t rm = (p.tiles_m + 8 / cols - 1) / (8 / cols), rn = (p.tiles_n + cols - 1) / cols;
    // the tiles of the fullest die, then the rows that its L2 takes in: 4096 x 768 -> 3072 54.6 us with the rows' tiles dealt
    // out alone, 50.4 in rectangles, 512 x 768 -> 3072 13.4 and 11.4
    const int64_t cost = rm * rn * 64 + rm * 64 + rn * 128;
    if (best < 0 || cost < best) best = cost, p.die_cols = cols, p.rect_m = (int)rm, p.rect_n = (int)rn;
  }
  const unsigned blocks = (unsigned)(8 * p.rect_m * p.rect_n);
  const bool whole = pick_epilogue((int)N, e) == EPI_Y32 || pick_epilogue((int)N, e) == EPI_Y16;
  auto kern = digit_epilogue((int)N, e) == EPI_Y32 ? (whole ? gemm_digits_kernel<EPI_Y32, false> : gemm_digits_kernel<EPI_Y32, true>)
                                                   : (whole ? gemm_digits_kernel<EPI_Y16, false> : gemm_digits_kernel<EPI_Y16, true>);
  kern<<<blocks, 256, LDS_BYTES, s>>>(a, b, sums, p, e);
  return launch_status();
}

}  // namespace catchq
