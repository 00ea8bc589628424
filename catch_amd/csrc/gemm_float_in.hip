// Pointwise convolutions and linears of few output channels on floating activations: quantized on the way into LDS.
//
// As two launches the quantizer reads the activations and writes a quarter (half: a half) of them, the contraction reads
// that back.  Where a block's tile covers the output channels every activation is read once and converted once.  What
// bounds the kernel is then the read of the activations: a block of four waves owns 64 rows x 64 or 128 channels; per K
// step of 64 a lane loads 16 activations of a row (four lanes a row: whole cache lines), two steps ahead of their use,
// converts them in registers (about seven vector instructions each, four blocks a compute unit cover them) and writes one
// 16-byte piece to LDS; the filters come by LDS-DMA through a ring of four.  One barrier a step.
//
// Measured: see gemm_float_ok at the bottom.
#include "igemm_i8_dma.inc"

namespace catchq {

template <int IN, int BN, int EPI>
__global__ __launch_bounds__(256) void gemm_float_kernel(const void *__restrict__ A, const int8_t *__restrict__ B, IgemmParams p,
                                                        EpiDev e, int x_neg_pos, unsigned a_bytes, unsigned b_bytes) {
  resolve_exp2(e);
  constexpr int BM = 64, BKB = 64, STAGES = 4;
  constexpr int ES = IN == IN_F32 ? 4 : 2, RAW = ES;  // bytes per activation, 16-byte loads per 16 activations
  constexpr int NB = BN / 64;                         // filter instructions (16 rows x 64 bytes) per wave and step
  constexpr int TN = BN / 64, WN = BN / 2;            // a wave's tile: 32 x WN
  constexpr int EPI_STRIDE = WN + 8;
  constexpr int A_SLOT = BM * BKB, B_STAGE = BN * BKB;
  constexpr unsigned OOB = 0x80000000u;  // the hardware answers an offset beyond the buffer with zeros
  extern __shared__ __attribute__((aligned(16))) int8_t lds_dyn[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave_m = wave >> 1, wave_n = wave & 1;
  const int logical = xcd_remap(blockIdx.x, p.nblocks);
  const int tile_n = logical % p.tiles_n, tile_m = logical / p.tiles_n;
  const int64_t m0 = (int64_t)tile_m * BM;
  const int n0 = tile_n * BN;
  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void *)A, 0, (int)a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void *)B, 0, (int)b_bytes, 0x00020000);

  // ---- loader: activations, 16 of row threadIdx / 4 per lane; filters, rows of 64 bytes as in the int8 kernel ---------
  const int arow = threadIdx.x >> 2, achunk = threadIdx.x & 3;
  const bool a_ok = m0 + arow < p.M;
  unsigned a_pix = a_ok ? (unsigned)(m0 + arow) : 0u;
  if (p.sh * p.sw != 1) {  // strided: output pixel -> input pixel (fewer than 2^31 pixels: 32-bit divisions)
    const unsigned t = a_pix / (unsigned)p.Wo, wo = a_pix - t * (unsigned)p.Wo;
    const unsigned img = t / (unsigned)p.Ho, ho = t - img * (unsigned)p.Ho;
    a_pix = (img * (unsigned)p.H + ho * (unsigned)p.sh) * (unsigned)p.W + wo * (unsigned)p.sw;
  }
  const unsigned a_row = a_pix * (unsigned)p.K;  // elements
  int ak = achunk * 16;
  unsigned b_off[NB];
  const int bchunk = (lane & 3) ^ ((lane >> 4) & 3);
  int bk = bchunk * 16;
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int n = n0 + (wave * NB + j) * 16 + (lane >> 2);
    b_off[j] = n < p.N ? (unsigned)n * (unsigned)p.K : OOB;
  }
  v4i raw[2][RAW];
  int wr_stage = 0;
  auto issue = [&](v4i (&r)[RAW]) {  // the next step: activations into r, filters into the ring; zeros past the end of K
    const unsigned voff = select_u32(a_ok && ak < p.K, (a_row + (unsigned)ak) * (unsigned)ES, OOB);
#pragma unroll
    for (int i = 0; i < RAW; ++i)
      r[i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_a, (int)voff + 16 * i, 0, 0));
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const unsigned boff = select_u32(bk < p.K, b_off[j] + (unsigned)bk, OOB);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsrc_b, (lds_ptr_t)(lds_dyn + 2 * A_SLOT + wr_stage * B_STAGE + (wave * NB + j) * 1024), 16, (int)boff, 0, 0, 0);
    }
    ak += BKB;
    bk += BKB;
    wr_stage = (wr_stage + 1) & (STAGES - 1);
  };

  v16i acc[1][TN];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][j][r] = 0;

  const int frow = lane & 31, fhalf = lane >> 5, sw = (frow >> 2) & 3;
  const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) int8_t *)lds_dyn;
  const unsigned k0 = (unsigned)((fhalf ^ sw) * 16), k1 = k0 ^ 32u;
  const unsigned fa_row = lds_base + (unsigned)((wave_m * 32 + frow) * BKB);
  const unsigned fb_row = lds_base + (unsigned)(2 * A_SLOT + (wave_n * WN + frow) * BKB);
  const unsigned wr_addr = lds_base + (unsigned)(arow * BKB + (achunk ^ ((arow >> 2) & 3)) * 16);

  int rd_stage = 0;
  auto step = [&](auto dc) {
    constexpr int d = decltype(dc)::value;
    const v4i q = quantize16<IN>(raw[d], x_neg_pos);
    asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(wr_addr), "v"(q), "n"(d * A_SLOT) : "memory");
    issue(raw[d]);
    // this wave's piece of the step is in LDS, its filters have landed; two steps may travel
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * (RAW + NB)) : "memory");
    __builtin_amdgcn_s_barrier();
    const unsigned b = fb_row + (unsigned)(rd_stage * B_STAGE);
    rd_stage = (rd_stage + 1) & (STAGES - 1);
    v4i fa[2], fb[2][TN];
    fa[0] = ds_read_b128<d * A_SLOT>(fa_row + k0);
    fa[1] = ds_read_b128<d * A_SLOT>(fa_row + k1);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      fb[0][j] = ds_read_b128<0>(b + k0 + (unsigned)(j * 32 * BKB));
      fb[1][j] = ds_read_b128<0>(b + k1 + (unsigned)(j * 32 * BKB));
    }
    lgkm_wait<0>(fa[0], fa[1]);
#pragma unroll
    for (int j = 0; j < TN; ++j) lgkm_wait<0>(fb[0][j], fb[1][j]);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[0][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[h], fb[h][j], acc[0][j], 0, 0, 0);
  };
  const int nsteps = (p.K + BKB - 1) / BKB;
  issue(raw[0]);
  issue(raw[1]);
  for (int s = 0; s < nsteps; s += 2) {
    step(std::integral_constant<int, 0>{});
    if (s + 1 >= nsteps) break;
    step(std::integral_constant<int, 1>{});
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();  // the slots are dead: staging area
  int *stage = reinterpret_cast<int *>(lds_dyn) + wave * 32 * EPI_STRIDE;
  if constexpr (EPI == EPI_SCALAR) igemm_epilogue_any<1, TN>(acc, stage, m0 + wave_m * 32, n0 + wave_n * WN, lane, p, e);
  else igemm_epilogue<1, TN, EPI>(acc, stage, m0 + wave_m * 32, n0 + wave_n * WN, lane, p, e);
}

template <int IN, int BN>
static int launch_gemm_float(const void *a, const void *b, IgemmParams p, const EpiDev &e, int x_neg_pos, int64_t a_bytes,
                             int64_t b_bytes, hipStream_t s) {
  constexpr int PIPE = 2 * 64 * 64 + 4 * BN * 64, STAGING = 4 * 32 * (BN / 2 + 8) * 4;
  constexpr int LDS_BYTES = PIPE > STAGING ? PIPE : STAGING;
  p.tiles_n = (p.N + BN - 1) / BN;
  const int64_t nb = (p.M + 63) / 64 * p.tiles_n;
  if (nb > 0x7fffffff) return -1;
  p.nblocks = (int)nb;
  p.ragged = pick_epilogue(p.N, e) == EPI_SCALAR ? ragged_epilogue(p.N, e, true) : EPI_SCALAR;
#define CATCHQ_FLOAT_CASE(E)                                                                                          \
  case E:                                                                                                             \
    gemm_float_kernel<IN, BN, E><<<p.nblocks, 256, LDS_BYTES, s>>>(a, (const int8_t *)b, p, e, x_neg_pos, (unsigned)a_bytes, \
                                                                   (unsigned)b_bytes);                                \
    break
  switch (pick_epilogue(p.N, e)) {
    CATCHQ_FLOAT_CASE(EPI_SCALAR);
    CATCHQ_FLOAT_CASE(EPI_Y32);
    CATCHQ_FLOAT_CASE(EPI_Y16);
    CATCHQ_FLOAT_CASE(EPI_Y16_STEPS);
    default: gemm_float_kernel<IN, BN, EPI_VECTOR><<<p.nblocks, 256, LDS_BYTES, s>>>(
        a, (const int8_t *)b, p, e, x_neg_pos, (unsigned)a_bytes, (unsigned)b_bytes);
  }
#undef CATCHQ_FLOAT_CASE
  return launch_status();
}

// Whether quantization and product [M, K] x [N, K]^T run as one launch of this kernel.
//
// Measured (one launch / two, us, half activations; float ones in brackets), M x K -> N:
//   100352 x 256 -> 64 14.4 / 25.3 (21.9 / 33.6), 100352 x 64 -> 256 17.4 / 22.6 (21.3 / 27.5), 25088 x 512 -> 128
//   9.7 / 19.7 (14.0 / 20.2), 6272 x 1024 -> 256 10.1 / 12.4 (12.7 / 14.5), 6272 x 1024 -> 512 14.2 / 15.4 (16.5 / 17.8),
//   12544 x 256 -> 64 4.3 / 7.5, 50176 x 96 -> 24 5.7 / 10.2
// More columns convert every activation more often: 6272 x 256 -> 1024 ties.  Few blocks are a serial chain of steps that
// nothing covers: 1568 x 2048 -> 512 16.0 / 14.4, 2048 x 1024 -> 512 9.9 / 9.6 (11.7 / 9.8), 3136 x 512 -> 128 6.5 / 7.0
// (7.4 / 7.1), 4096 x 3072 -> 128 22.3 / 21.1 (33.1 / 22.7).
// A strided layer leaves most of the pixels unread that a quantizer converts, so it takes more columns: stride 2 on
// 32 images, 56x56 256 -> 512 17.7 / 31.3 (21.4 / 39.1), 28x28 512 -> 1024 15.3 / 20.9 (19.2 / 26.4), 14x14 1024 -> 2048
// 15.3 / 16.6 (17.0 / 19.1), 56x56 64 -> 128 5.1 / 10.1 (6.1 / 13.1).
// in_pixels: pixels of the input, M of the output.
bool gemm_float_ok(int64_t in_pixels, int64_t M, int64_t N, int64_t K, int elem_bytes, int cus) {
  if (K % 16 != 0 || M >= (1ll << 31) - 64 || in_pixels * K * elem_bytes >= (1ll << 31) || N * K >= (1ll << 31)) return false;
  if (N > (in_pixels > M ? 2048 : 512) || M < 1024 || K > 1024) return false;
  const int64_t blocks = (M + 63) / 64 * (N <= 64 ? 1 : (N + 127) / 128);
  return blocks * 4 >= 3 * cus || K <= (elem_bytes == 2 ? 512 : 256);
}

int gemm_float(const void *x, bool half, int position, const void *w, int N_img, int H, int W, int Ci, int Co, int sh, int sw, int Ho,
               int Wo, const EpiDev &e, hipStream_t s) {
  IgemmParams p = {};
  p.M = (int64_t)N_img * Ho * Wo;
  p.N = Co;
  p.K = Ci;
  p.H = H; p.W = W; p.Ho = Ho; p.Wo = Wo; p.sh = sh; p.sw = sw;
  const int64_t N = Co, a_bytes = (int64_t)N_img * H * W * Ci * (half ? 2 : 4), b_bytes = N * Ci;
  if (N <= 64) {
    return half ? launch_gemm_float<IN_F16, 64>(x, w, p, e, -position, a_bytes, b_bytes, s)
                : launch_gemm_float<IN_F32, 64>(x, w, p, e, -position, a_bytes, b_bytes, s);
  }
  return half ? launch_gemm_float<IN_F16, 128>(x, w, p, e, -position, a_bytes, b_bytes, s)
              : launch_gemm_float<IN_F32, 128>(x, w, p, e, -position, a_bytes, b_bytes, s);
}

}  // namespace catchq
