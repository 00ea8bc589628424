// Pointwise layers of 64 or 128 int16 channels with int8 filters, up to 128 of them.
//
// What bounds them is HBM, and the tiled kernel (igemm_a16_dma.hip) is a chain of set-up, one delivery, one or two K steps and an
// epilogue behind a ring of slots that it never fills.  Here a block requests all of its rows at once, splits them into digits on
// their way into LDS and meets one barrier; a wave's 32 filters (2 or 4 fragments) come straight into registers, and small blocks
// leave room for many.  us, tiled / this: 16 x 208 x 208, 64 -> 32 channels 39 / 22 (22 at 6 TB/s), 104 x 104, 64 -> 96 23.7 / 15.8,
// 128 -> 64 16.9 / 14.7, 52 x 52, 128 -> 128 9.2 / 9.0; one image 5.2 / 4.1, 4.3 / 3.7, 3.9 / 3.8, 3.8 / 3.6; to half outputs equal.
// With 256 channels and more (filters through a ring of registers) it was equal on many rows and slower on few (16 x 52 x 52,
// 256 -> 128 10.9 / 10.4, 8 x 13 x 13, 1024 -> 512 6.5 / 7.4): not this kernel's.
#include "conv3x3_halo.h"

namespace catchq {

struct PwA16Params {
  IgemmParams g;   // M, N, K, nblocks
  unsigned x_bytes;
  int col_groups;  // waves side by side, 32 columns each (a power of two); the others take further rows
};

template <int KK, int EPI>
__global__ __launch_bounds__(256, 4) void pw_a16_short_kernel(const int16_t *__restrict__ X, const int8_t *__restrict__ B, PwA16Params p,
                                                             EpiDev e) {
  resolve_exp2(e);
  constexpr int K = KK * 32, PER_ROW = K / 16, PITCH = 2 * K + 16;  // (an odd number of 16 B pieces: neighbours cover a 256 B line)
  constexpr int ROWS = KK == 2 ? 128 : 64, PIECES = ROWS * PER_ROW / 256;
  constexpr unsigned OOB = 0x80000000u;
  constexpr int A_BYTES = ROWS * PITCH, STAGE_BYTES = 4 * 32 * 40 * 4;
  __shared__ __attribute__((aligned(16))) int8_t lds[A_BYTES > STAGE_BYTES ? A_BYTES : STAGE_BYTES];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int frow = lane & 31, fhalf = lane >> 5;
  const int cg = wave & (p.col_groups - 1), pg = wave / p.col_groups;
  const int rows = 128 / p.col_groups;  // of the block
  const int64_t m0 = (int64_t)xcd_remap(blockIdx.x, p.g.nblocks) * rows;
  const int n0 = cg * 32;
  const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc((void *)X, 0, (int)p.x_bytes, 0x00020000);

  // rows -> digits in LDS: 16 values a piece
  v4i v[PIECES][2];
#pragma unroll
  for (int i = 0; i < PIECES; ++i) {
    const int at = i * 256 + (int)threadIdx.x, row = at / PER_ROW, q = at % PER_ROW;
    const unsigned from = select_u32(row < rows && m0 + row < p.g.M, (unsigned)(m0 + row) * (unsigned)(2 * K) + (unsigned)q * 32u, OOB);
    v[i][0] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_x, (int)from, 0, 0));
    v[i][1] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_x, (int)from, 16, 0));
  }
  v4i fb[KK];
  int sum = 0;
#pragma unroll
  for (int k = 0; k < KK; ++k) {
    fb[k] = v4i{0, 0, 0, 0};
    if (n0 + frow < p.g.N) fb[k] = *reinterpret_cast<const v4i *>(B + (int64_t)(n0 + frow) * K + k * 32 + fhalf * 16);
#pragma unroll
    for (int d = 0; d < 4; ++d) sum = __builtin_amdgcn_sdot4(fb[k][d], 0x01010101, sum, false);
  }
#pragma unroll
  for (int i = 0; i < PIECES; ++i) {
    const int at = i * 256 + (int)threadIdx.x, row = at / PER_ROW, q = at % PER_ROW;
    if (row < rows) {
      v4i hi, lo;
      split_i16(v[i][0], v[i][1], hi, lo);
      *reinterpret_cast<v4i *>(lds + row * PITCH + q * 16) = hi;
      *reinterpret_cast<v4i *>(lds + row * PITCH + q * 16 + K) = lo;
    }
  }
  __syncthreads();

  // 256 * sum of the high digits' products + that of the low ones' + 128 * sum of the weights, modulo 2^32
  const unsigned ws = (unsigned)(sum + __shfl_xor(sum, 32, 64)) << 7;
  const int8_t *const own = lds + (pg * 32 + frow) * PITCH + fhalf * 16;
  v16i acc[1][1];
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[0][0][r] = 0;
#pragma unroll
  for (int d = 0; d < 2; ++d) {
#pragma unroll
    for (int k = 0; k < KK; ++k)
      acc[0][0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(*reinterpret_cast<const v4i *>(own + d * K + k * 32), fb[k], acc[0][0], 0, 0, 0);
    if (d == 0)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[0][0][r] = (int)(((unsigned)acc[0][0][r] << 8) + ws);
  }
  __syncthreads();
  int *const stage = reinterpret_cast<int *>(lds) + wave * 32 * (32 + 8);
  igemm_epilogue<1, 1, EPI>(acc, stage, m0 + pg * 32, n0, lane, p.g, e);
}

template <int KK>
static int launch_pw_a16(const void *x, const void *w, const PwA16Params &p, const EpiDev &e, hipStream_t s) {
  if (pick_epilogue(p.g.N, e) == EPI_LK_Q16)
    pw_a16_short_kernel<KK, EPI_LK_Q16><<<p.g.nblocks, 256, 0, s>>>((const int16_t *)x, (const int8_t *)w, p, e);
  else
    pw_a16_short_kernel<KK, EPI_VECTOR><<<p.g.nblocks, 256, 0, s>>>((const int16_t *)x, (const int8_t *)w, p, e);
  return launch_status();
}

// A few columns of 64 channels on less than half a block for a unit stay with the tiled kernel (us to int16 behind a ReLU, tiled / this:
// 52 x 52, 64 -> 4 6.9 / 7.7, 8 7.0 / 7.5, 12 ahead by 8 %; 4 x 104 x 104, 338 blocks, 4 a fifth ahead).
bool pw_a16_short_takes(int64_t M, int64_t N, int64_t K, const EpiDev &e) {
  if ((K != 64 && K != 128) || N > 128 || M * K * 2 >= (1ll << 31)) return false;
  if (K == 64 && N <= 8 && (M + 127) / 128 * 2 < e.cus) return false;
  const int epi = pick_epilogue((int)N, e);
  return epi == EPI_LK_Q16 || epi == EPI_VECTOR;
}

// x [M, K] int16, w [N, K], a call that pw_a16_short_takes
int pw_a16_short(const void *x, const void *w, int64_t M, int64_t N, int64_t K, const EpiDev &e, hipStream_t s) {
  const int groups = (int)((N + 31) / 32);
  PwA16Params p = {};
  p.g.M = M; p.g.N = (int)N; p.g.K = (int)K;
  p.x_bytes = (unsigned)(M * K * 2);
  p.col_groups = groups > 2 ? 4 : groups;
  if (K == 128 && p.col_groups == 1) p.col_groups = 2;  // (128 rows of 128 channels: twice the room)
  const int rows = 128 / p.col_groups;
  p.g.nblocks = (int)((M + rows - 1) / rows);  // (fewer than 2^24 rows)
  return K == 64 ? launch_pw_a16<2>(x, w, p, e, s) : launch_pw_a16<4>(x, w, p, e, s);
}

}  // namespace catchq
