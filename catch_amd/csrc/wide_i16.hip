// int16 x int16 contractions on the int8 matrix cores, exact in 64 bits.
//
// Both operands split into digits:  x = 256*xh + xl + 128,  w = 256*wh + wl + 128  (high byte signed, low byte biased
// into int8), so
//   sum x*w = 65536*S_hh + 256*(S_hl + S_lh) + S_ll + 32768*(sum xh + sum wh) + 128*(sum xl + sum wl) + 16384*Kp
// with four int8 x int8 MFMA sums S_.. , the digit sums of the row (activations) and of the column (weights), which a wave
// collects from the fragments it loads anyway, and Kp the number of K positions walked (whole steps: a position beyond K,
// a row beyond M or N and an out-of-image tap all read as zeros, which decode to the value 0 on either side, so the
// identity covers them).  Every partial sum fits an int32 (|S| <= Kp * 2^14, K < 2^16); the combination is done in fp64,
// whose 53 bits hold every value of it (|sum| < 2^47), and its one conversion to fp32 is the int64 sum's.
//
// What bounds it: instruction issue.  A wave issues about one instruction every four clocks, and per 32 K positions and
// fragment of 32 rows there are 20 vector operations of splitting and summing besides the reads and transfers, for
// TM * TN products of four matrix instructions (32 clocks each).  Large wave tiles serve that; large blocks would leave the
// sizes of a linear or a convolution without enough of them.  So the waves of a block share one tile and split K: a wave
// owns a contiguous slice of K, moves the slice's 128-byte row pieces (64 values) to LDS slots of its own with LDS-DMA,
// two K steps in flight, and waits for nothing but its own transfers -- no barrier in the loop; the partial sums meet in
// LDS behind it.  64 x 64 tiles keep 192 accumulator registers per wave, one wave per SIMD; the smaller ones run two or
// more waves per SIMD, whose matrix and vector instructions overlap.
//
// Measured (us, against a 128 x 128 tile walked by all waves of a block): 1 x 768 -> 3072 12.4 -> 4.9, 64 x 3072 -> 768
// 40.4 -> 9.8, 1379 x 1000 -> 1001 24.3 -> 18.6, 4096 x 768 -> 3072 112 -> 92, 8192 x 1024 -> 1024 88 -> 68; 3 x 3
// convolutions: 8 x 14 x 14, 256 channels 34.7 -> 13.0, 8 x 28 x 28, 128 channels 23.0 -> 13.3, 5 x 57 x 75, 96 -> 160
// channels 47.5 -> 36.4, 16 x 56 x 56, 64 channels 38.2 -> 29.8.
#include <type_traits>

#include "igemm_common.h"

namespace catchq {

typedef __attribute__((address_space(3))) void *lds_ptr_t;
typedef double v2d __attribute__((ext_vector_type(2)));

struct WideParams {
  const void *x;  // int16, or floats that the loader quantizes
  const int16_t *w;
  int M, N, K;  // K < 2^16
  int H, W, Ci, Ho, Wo, kw, ph, pw, sh, sw, dh, dw;
  unsigned img_stride, row_stride, pix_stride;  // elements
  int x_neg_pos;      // floating activations: quantized at 2^-x_neg_pos
  unsigned magic_ci, magic_kw, mask_ci, mask_kw;  // ceil(2^32 / d), mask 0; for d = 1 magic 0, mask ~0
  int tiles_m, tiles_n, nblocks;
  int m_fastest;  // consecutive blocks walk the row tiles of one column tile first
  int epi;
  int ragged;         // epi serves rows whose length or alignment is not its own (EpiAtRagged)
  unsigned a_bytes, b_bytes;
};

#define CATCHQ_WIDE_VMCNT(n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(n) : "memory")

__device__ __forceinline__ unsigned wide_div(unsigned n, unsigned magic, unsigned mask) { return __umulhi(n, magic) + (n & mask); }

__device__ __forceinline__ v4i wide_ds_read(unsigned addr) {
  v4i v;
  asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(addr));
  return v;
}

template <int TM, int TN, int NW, bool DENSE, int IN>
__global__ __launch_bounds__(64 * NW) void wide_i16_kernel(WideParams p, EpiDev e) {
  resolve_exp2(e);
  constexpr int BM = TM * 32, BN = TN * 32;
  constexpr int KS = 64;                                   // values of K per step: 128 bytes of a row
  constexpr int SLOT_BYTES = (BM + BN) * KS * 2, WAVE_BYTES = 2 * SLOT_BYTES;
  constexpr int NA = BM / 8, NB = BN / 8, NI = NA + NB;    // DMA instructions (8 rows each) per step
  static_assert(BM * BN * 8 <= WAVE_BYTES, "a partial tile (fp64) fits the wave's slots");
  extern __shared__ __attribute__((aligned(16))) int8_t lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int logical = xcd_remap(blockIdx.x, p.nblocks);
  const int tile_m = p.m_fastest ? logical % p.tiles_m : logical / p.tiles_n;
  const int tile_n = p.m_fastest ? logical / p.tiles_m : logical % p.tiles_n;
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void *)p.x, 0, (int)p.a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void *)p.w, 0, (int)p.b_bytes, 0x00020000);
  constexpr unsigned OOB = 0x80000000u;  // the hardware answers an offset beyond the buffer with zeros

  // ---- loader: a DMA instruction fills 8 rows of 128 bytes; lane l writes piece l & 7 of row l >> 3 and fetches piece
  // (l & 7) ^ ((row >> 1) & 7) of that row, so that the fragment reads of 16 rows fall into 16 different 16-byte slots
  const int lrow = lane >> 3;
  const int chunk0 = (lane & 7) ^ (lane >> 4);
  unsigned a_base[NA], b_base[NB];  // elements
  int a_hi[NA], a_wi[NA];
#pragma unroll
  for (int j = 0; j < NA; ++j) {
    const int m = m0 + j * 8 + lrow;
    if constexpr (DENSE) {
      a_hi[j] = m < p.M ? 0 : -1;
      a_wi[j] = 0;
      a_base[j] = (unsigned)m * p.pix_stride;
    } else {
      const unsigned t = (unsigned)m / (unsigned)p.Wo, wo = (unsigned)m - t * (unsigned)p.Wo;
      const unsigned img = t / (unsigned)p.Ho, ho = t - img * (unsigned)p.Ho;
      a_hi[j] = m < p.M ? (int)ho * p.sh - p.ph : -(1 << 30);  // a row that does not exist is outside the image
      a_wi[j] = (int)wo * p.sw - p.pw;
      a_base[j] = img * p.img_stride + (unsigned)a_hi[j] * p.row_stride + (unsigned)a_wi[j] * p.pix_stride;  // mod 2^32
    }
  }
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int n = n0 + j * 8 + lrow;
    b_base[j] = n < p.N ? (unsigned)n * (unsigned)p.K : OOB;
  }
  const int steps = (p.K + KS - 1) / KS;
  const int per = steps / NW, rem = steps - per * NW;
  const int first = wave * per + (wave < rem ? wave : rem);
  const int mine = per + (wave < rem ? 1 : 0);
  int8_t *const my = lds + wave * WAVE_BYTES;

  // Full steps of a dense operand: one vector offset per row, fixed for the whole walk, and the step as the scalar offset.
  // (A row that does not exist has an offset beyond the buffer; all others stay inside their row.)
  unsigned a_off[NA], b_off[NB];
#pragma unroll
  for (int j = 0; j < NA; ++j)
    a_off[j] = DENSE && a_hi[j] == 0 ? 2u * (a_base[j] + (unsigned)((chunk0 ^ (4 * (j & 1))) * 8)) : OOB;
#pragma unroll
  for (int j = 0; j < NB; ++j) b_off[j] = b_base[j] != OOB ? 2u * (b_base[j] + (unsigned)((chunk0 ^ (4 * (j & 1))) * 8)) : OOB;

  constexpr int ES = IN == IN_I8 ? 2 : in_bytes(IN);  // bytes per activation (IN_I8: integers as they are, of 16 bits)
  FloatPiece<IN, 8> raw[NA];
  (void)raw;
  const unsigned chan_stride = in_apart(IN) ? (unsigned)(p.H * p.W) : 1u;

  auto issue = [&](int s) {
    const int slot = (s & 1) * SLOT_BYTES;
    const bool full = (first + s + 1) * KS <= p.K;
    if (DENSE && IN == IN_I8 && full) {
      const int step = (first + s) * (KS * 2);
#pragma unroll
      for (int j = 0; j < NA; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_ptr_t)(my + slot + j * 1024), 16, (int)a_off[j], step, 0, 0);
#pragma unroll
      for (int j = 0; j < NB; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, (lds_ptr_t)(my + slot + (NA + j) * 1024), 16, (int)b_off[j], step, 0, 0);
      return;
    }
    unsigned koff[2];
    int dy[2], dx[2];
    bool ok[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const unsigned k = (unsigned)((first + s) * KS + (chunk0 ^ (4 * h)) * 8);
      ok[h] = k < (unsigned)p.K;
      koff[h] = k;
      dy[h] = dx[h] = 0;
      if constexpr (!DENSE) {
        const unsigned tap = wide_div(k, p.magic_ci, p.mask_ci), ci = k - tap * (unsigned)p.Ci;
        const unsigned r = wide_div(tap, p.magic_kw, p.mask_kw), q = tap - r * (unsigned)p.kw;
        dy[h] = (int)r * p.dh;
        dx[h] = (int)q * p.dw;
        koff[h] = (unsigned)dy[h] * p.row_stride + (unsigned)dx[h] * p.pix_stride + ci * chan_stride;
      }
    }
    const int step = (first + s) * (KS * 2);
    auto filters = [&] {
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        unsigned voff = ok[j & 1] ? b_off[j] + (unsigned)step : OOB;
        voff = b_off[j] == OOB ? OOB : voff;
        asm volatile("" : "+v"(voff));
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, (lds_ptr_t)(my + slot + (NA + j) * 1024), 16, (int)voff, 0, 0, 0);
      }
    };
    // (in front of floating activations: loads complete in order, so a wave that has those has its filters)
    if constexpr (IN != IN_I8) filters();
#pragma unroll
    for (int j = 0; j < NA; ++j) {
      const int h = j & 1;
      bool in = ok[h];
      if constexpr (DENSE) in = in & (a_hi[j] == 0);
      else in = in & ((unsigned)(a_hi[j] + dy[h]) < (unsigned)p.H) & ((unsigned)(a_wi[j] + dx[h]) < (unsigned)p.W);
      unsigned voff = in ? (unsigned)ES * (a_base[j] + koff[h]) : OOB;
      asm volatile("" : "+v"(voff));  // one select and one load, not two loads under complementary masks
      if constexpr (IN == IN_I8)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_ptr_t)(my + slot + j * 1024), 16, (int)voff, 0, 0, 0);
      else raw[j].load(rsrc_a, voff, chan_stride * (unsigned)ES);
    }
    if constexpr (IN == IN_I8) filters();
  };

  // ---- K loop --------------------------------------------------------------------------------------------------------
  v16i s_hh[TM][TN], s_mid[TM][TN], s_ll[TM][TN];  // (the two middle sums share one accumulator: |S_hl + S_lh| <= Kp * 2^15, and a wave walks at most half of K, NW >= 2)
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) { s_hh[i][j][r] = 0; s_mid[i][j][r] = 0; s_ll[i][j][r] = 0; }
  int xh_sum[TM] = {}, xl_sum[TM] = {}, wh_sum[TN] = {}, wl_sum[TN] = {};
  const int frow = lane & 31, fhalf = lane >> 5;
  const unsigned row_addr = (unsigned)(uintptr_t)(__attribute__((address_space(3))) int8_t *)my + (unsigned)(frow * (KS * 2));
  const unsigned sw = (unsigned)((frow >> 1) & 7);

  // 32 K positions (half u of a step): this lane's 16 values of a row are pieces 4u + 2 fhalf and the next
  struct Frags { v4i a[TM][2], b[TN][2]; };
  auto fetch = [&](Frags &f, unsigned base, int u) {
    const unsigned piece = (((unsigned)(u * 4 + fhalf * 2)) ^ sw) * 16;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      f.a[i][0] = wide_ds_read(base + i * 32 * KS * 2 + piece);
      f.a[i][1] = wide_ds_read(base + i * 32 * KS * 2 + (piece ^ 16u));
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      f.b[j][0] = wide_ds_read(base + (BM + j * 32) * KS * 2 + piece);
      f.b[j][1] = wide_ds_read(base + (BM + j * 32) * KS * 2 + (piece ^ 16u));
    }
  };
  auto arrived = [&](Frags &f) {
#pragma unroll
    for (int i = 0; i < TM; ++i) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f.a[i][0]), "+v"(f.a[i][1])::"memory");
#pragma unroll
    for (int j = 0; j < TN; ++j) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f.b[j][0]), "+v"(f.b[j][1])::"memory");
  };
  auto multiply = [&](const Frags &f) {
    v4i xh[TM], xl[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      split_i16(f.a[i][0], f.a[i][1], xh[i], xl[i]);
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        xh_sum[i] = __builtin_amdgcn_sdot4(xh[i][d], 0x01010101, xh_sum[i], false);
        xl_sum[i] = __builtin_amdgcn_sdot4(xl[i][d], 0x01010101, xl_sum[i], false);
      }
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      v4i wh, wl;
      split_i16(f.b[j][0], f.b[j][1], wh, wl);
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        wh_sum[j] = __builtin_amdgcn_sdot4(wh[d], 0x01010101, wh_sum[j], false);
        wl_sum[j] = __builtin_amdgcn_sdot4(wl[d], 0x01010101, wl_sum[j], false);
      }
      // one kind of product for all row tiles before the next: the two that share an accumulator stay apart
#pragma unroll
      for (int i = 0; i < TM; ++i) s_mid[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(xh[i], wl, s_mid[i][j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < TM; ++i) s_hh[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(xh[i], wh, s_hh[i][j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < TM; ++i) s_ll[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(xl[i], wl, s_ll[i][j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < TM; ++i) s_mid[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(xl[i], wh, s_mid[i][j], 0, 0, 0);
    }
  };

  double *const part = reinterpret_cast<double *>(my);                                 // [BM][BN]
  double *const row_part = reinterpret_cast<double *>(lds + NW * WAVE_BYTES) + wave * BM;  // [BM]
  if (mine > 0) {
    issue(0);
    if (IN == IN_I8 && mine > 1) issue(1);
    for (int s = 0; s < mine; ++s) {
      if constexpr (IN == IN_I8) {
        if (s + 1 < mine) CATCHQ_WIDE_VMCNT(NI);
        else CATCHQ_WIDE_VMCNT(0);
      } else {
        // the step's activations, quantized into the slot as a transfer would have left them; its filters came before them
        v4i q[NA];
#pragma unroll
        for (int j = 0; j < NA; ++j) q[j] = quantize_piece<IN>(raw[j], p.x_neg_pos);
        CATCHQ_WIDE_VMCNT(0);
        const unsigned to = (unsigned)(uintptr_t)(__attribute__((address_space(3))) int8_t *)my + (unsigned)((s & 1) * SLOT_BYTES + lane * 16);
#pragma unroll
        for (int j = 0; j < NA; ++j) asm volatile("ds_write_b128 %0, %1" ::"v"(to + (unsigned)(j * 1024)), "v"(q[j]) : "memory");
        if (s + 1 < mine) issue(s + 1);
      }
      const unsigned base = row_addr + (unsigned)((s & 1) * SLOT_BYTES);
      Frags f0, f1;
      fetch(f0, base, 0);
      arrived(f0);
      fetch(f1, base, 1);  // under the first half's arithmetic
      multiply(f0);
      arrived(f1);
      if (IN == IN_I8 && s + 2 < mine) issue(s + 2);  // the slot has been read
      multiply(f1);
    }
    // a lane holds the digit sums of row (lane & 31) over its half of every K step: add the halves
    const double kp = 16384.0 * (double)(mine * KS);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int h = xh_sum[i] + __shfl_xor(xh_sum[i], 32, 64), l = xl_sum[i] + __shfl_xor(xl_sum[i], 32, 64);
      if (fhalf == 0) row_part[i * 32 + frow] = 32768.0 * (double)h + 128.0 * (double)l;
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int h = wh_sum[j] + __shfl_xor(wh_sum[j], 32, 64), l = wl_sum[j] + __shfl_xor(wl_sum[j], 32, 64);
      const double col = 32768.0 * (double)h + 128.0 * (double)l + kp;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = i * 32 + 8 * (r >> 2) + 4 * fhalf + (r & 3);
          part[row * BN + j * 32 + frow] = __builtin_fma((double)s_hh[i][j][r], 65536.0,
                                                         __builtin_fma((double)s_mid[i][j][r], 256.0, (double)s_ll[i][j][r] + col));
        }
    }
  }
  __syncthreads();

  // ---- partial sums -> outputs ---------------------------------------------------------------------------------------
  const int active = steps < NW ? steps : NW;
  const double *const parts = reinterpret_cast<const double *>(lds);
  const double *const rows = reinterpret_cast<const double *>(lds + NW * WAVE_BYTES);
  if (p.epi == EPI_SCALAR) {
    // rows of N elements start anywhere: a lane keeps one column, so that its channel's operands are loaded once and the
    // stores of a wave are runs of a row
    const int c = threadIdx.x % BN, n = n0 + c;
    if (n >= p.N) return;
    const EpiColumn k = epi_column(e, n);
    for (int px = threadIdx.x / BN; px < BM; px += 64 * NW / BN) {
      const int m = m0 + px;
      if (m >= p.M) break;
      double v = 0.0;
      for (int w = 0; w < active; ++w) v += parts[w * (WAVE_BYTES / 8) + px * BN + c] + rows[w * BM + px];
      const int64_t idx = (int64_t)m * p.N + n;
      epi_store(epi_value((float)v, idx, k, e), idx, e);
    }
    return;
  }
  constexpr int CPR = BN / 4;  // 64 * NW is a multiple of it: a lane keeps its four channels
  const int cg = threadIdx.x % CPR, n = n0 + cg * 4;
  if (n >= p.N) return;
  auto finish = [&](auto spec, auto ragged_c) {
    typedef decltype(spec) S;
    constexpr bool RAGGED = decltype(ragged_c)::value;
    EpiLane L;
    if constexpr (RAGGED) L = epi_lane_setup_ragged<S>(n, p.N, e);
    else L = epi_lane_setup<S>(n, true, e);
    for (int t = threadIdx.x; t < BM * CPR; t += 64 * NW) {
      const int px = t / CPR, m = m0 + px;
      if (m >= p.M) break;
      const int64_t idx = (int64_t)m * p.N + n;
      v4f res = {0.f, 0.f, 0.f, 0.f};
      if constexpr (!RAGGED) {
        if (L.use_res) res = *reinterpret_cast<const v4f *>(e.resid + idx);
      }
      double v[4] = {0.0, 0.0, 0.0, 0.0};
      for (int w = 0; w < active; ++w) {
        const v2d *src = reinterpret_cast<const v2d *>(parts + w * (WAVE_BYTES / 8) + t * 4);
        const v2d a = src[0], b = src[1];
        const double r = rows[w * BM + px];
        v[0] += a[0] + r; v[1] += a[1] + r; v[2] += b[0] + r; v[3] += b[1] + r;
      }
      const v4f sums = {(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
      if constexpr (RAGGED) epi_vec4<S>(sums, res, L, EpiAtRagged{idx, p.N - n}, e);
      else epi_vec4<S>(sums, res, L, idx, e);
    }
  };
  const std::true_type ragged;
  const std::false_type whole;
  switch (p.epi) {
    case EPI_Y32: p.ragged ? finish(EpiOf<EPI_Y32>::type{}, ragged) : finish(EpiOf<EPI_Y32>::type{}, whole); break;
    case EPI_Y16: p.ragged ? finish(EpiOf<EPI_Y16>::type{}, ragged) : finish(EpiOf<EPI_Y16>::type{}, whole); break;
    default: finish(EpiGeneric{}, whole); break;
  }
}

template <int TM, int TN, int NW, bool DENSE, int IN = IN_I8>
static int launch_wide(WideParams p, const EpiDev &e, hipStream_t s) {
  constexpr int LDS_BYTES = NW * (2 * (TM + TN) * 32 * 128 + TM * 32 * 8);
  auto kern = wide_i16_kernel<TM, TN, NW, DENSE, IN>;
  if (LDS_BYTES > 64 * 1024) {
    static std::atomic<bool> raised[64];
    if (raise_lds_limit((const void *)kern, LDS_BYTES, raised) != CATCHQ_OK) return CATCHQ_ERR_LAUNCH;
  }
  const int64_t tm = ((int64_t)p.M + TM * 32 - 1) / (TM * 32), tn = ((int64_t)p.N + TN * 32 - 1) / (TN * 32);
  if (tm * tn > 0x7fffffff) return -1;
  p.tiles_m = (int)tm;
  p.tiles_n = (int)tn;
  p.nblocks = (int)(tm * tn);
  kern<<<p.nblocks, 64 * NW, LDS_BYTES, s>>>(p, e);
  return launch_status();
}

template <bool DENSE>
static int pick_wide(const WideParams &p, const EpiDev &e, hipStream_t s) {
  // The largest wave tile that still fills the chip once: 64 x 64 blocks of two waves are at home two on a compute unit
  // (352 of them leave more idle than the larger tile saves, 500 do not), 32 x 64 ones three, 32 x 32 ones five; below
  // that four waves split K.
  auto tiles = [&](int bm, int bn) { return ((int64_t)p.M + bm - 1) / bm * (((int64_t)p.N + bn - 1) / bn); };
  int plan = tiles(64, 64) >= 7 * e.cus / 4 ? 642 : tiles(32, 64) >= 2 * e.cus ? 362 : tiles(32, 32) >= 2 * e.cus ? 322 : 324;
  if (const char *f = tuning_env("CATCHQ_WIDE")) plan = std::atoi(f);
  switch (plan) {
    case 642: return launch_wide<2, 2, 2, DENSE>(p, e, s);
    case 362: return launch_wide<1, 2, 2, DENSE>(p, e, s);
    case 322: return launch_wide<1, 1, 2, DENSE>(p, e, s);
    default: return launch_wide<1, 1, 4, DENSE>(p, e, s);
  }
}

// The kernel's constants; false where its arithmetic does not cover the shape.  x_ci channels of x_size bytes in the activations, Ci in
// the filters; apart: activations in the order [N, channel, H, W].
static bool wide_params(WideParams *q, const void *x, int x_size, const void *w, int N, int H, int W, int x_ci, bool apart, int Ci, int Co,
                        int kh, int kw, int ph, int pw, int sh, int sw, int dh, int dw, int Ho, int Wo, bool dense, const EpiDev &e) {
  const int64_t M = (int64_t)N * Ho * Wo, K = (int64_t)kh * kw * Ci;
  const int64_t a_bytes = ((int64_t)N * H * W * x_ci * x_size + 3) / 4 * 4, b_bytes = (int64_t)Co * K * 2;
  if (Ci % 8 != 0 || x_ci > Ci || a_bytes >= (1ll << 31) || b_bytes >= (1ll << 31) || a_bytes <= 0 || b_bytes <= 0 || e.acc_out) return false;
  if (apart && (int64_t)H * W * x_size * (Ci - x_ci + 16) >= (1ll << 30)) return false;  // (no offset wraps)
  if (M >= (1ll << 31) - 64 || K >= (1 << 16) || (int64_t)kh * kw * kw >= (1ll << 31)) return false;
  if (!dense && (H >= (1 << 20) || W >= (1 << 20) || (int64_t)dh * kh >= (1 << 20) || (int64_t)dw * kw >= (1 << 20))) return false;
  WideParams &p = *q;
  p = {};
  p.x = x; p.w = (const int16_t *)w;
  p.M = (int)M; p.N = Co; p.K = (int)K;
  p.H = H; p.W = W; p.Ci = Ci; p.Ho = Ho; p.Wo = Wo; p.kw = kw; p.ph = ph; p.pw = pw; p.sh = sh; p.sw = sw; p.dh = dh; p.dw = dw;
  p.img_stride = (unsigned)((int64_t)H * W * x_ci);
  p.row_stride = (unsigned)(apart ? W : (int64_t)W * x_ci);
  p.pix_stride = apart ? 1u : (unsigned)x_ci;
  auto magic = [](unsigned d, unsigned *m, unsigned *mask) {  // dividends below 2^16: exact for every divisor below 2^16
    *m = d <= 1 ? 0u : (unsigned)(((1ull << 32) + d - 1) / d);
    *mask = d <= 1 ? ~0u : 0u;
  };
  magic(Ci, &p.magic_ci, &p.mask_ci);
  magic(kw, &p.magic_kw, &p.mask_kw);
  p.m_fastest = b_bytes > a_bytes;
  p.epi = pick_epilogue(Co, e);
  if (p.epi == EPI_SCALAR) {
    // (33759 x 192 -> 146 62.8 us with one element at a time, 47.5 so, 148 channels 46.3)
    const int epi = ragged_epilogue(Co, e);
    if (epi != EPI_SCALAR) { p.epi = epi; p.ragged = 1; }
  }
  p.a_bytes = (unsigned)a_bytes; p.b_bytes = (unsigned)b_bytes;
  return true;
}

// int16 x int16; -1 when the shape is not eligible (or an int32 accumulator output is asked for: the exact sum has 64 bits)
int conv2d_mfma_a16w16(const void *x, const void *w, int N, int H, int W, int Ci, int Co, int kh, int kw, int ph, int pw,
                       int sh, int sw, int dh, int dw, int Ho, int Wo, const EpiDev &e, hipStream_t s) {
  const bool dense = kh == 1 && kw == 1 && sh == 1 && sw == 1 && ph == 0 && pw == 0;
  WideParams p;
  if (!wide_params(&p, x, 2, w, N, H, W, Ci, false, Ci, Co, kh, kw, ph, pw, sh, sw, dh, dw, Ho, Wo, dense, e)) return -1;
  return dense ? pick_wide<true>(p, e, s) : pick_wide<false>(p, e, s);
}

template <bool DENSE, int IN>
static int launch_wide_float(int waves, const WideParams &p, const EpiDev &e, hipStream_t s) {
  return waves == 4 ? launch_wide<1, 1, 4, DENSE, IN>(p, e, s) : launch_wide<1, 1, 2, DENSE, IN>(p, e, s);
}

// Floating activations with int16 filters in one launch; -1: another route.  Arguments as contract_small_float's (Ci a multiple of 8).
//
// Every block converts its rows again, so the one launch pays while a wave has few K steps of 64 and the device few tiles (a call's time,
// us, two launches / one): 32 x 32 tiles on four waves, up to one per unit, one step a wave 9.2 / 5.6 (linears), two 9.2 / 5.7, four 9.1 /
// 7.1, five 10.9 / 9.3 (3 x 3), six 9.7 / 8.4, seven 10.2 / 10.0, eight and more 12 / 14; up to two per unit three 9.5 / 8.0, four 10.6 / 9.7, seven
// 14.6 / 15.4; on two waves up to four per unit one 9.4 / 6.0, two 9.4 / 7.4, three 10.0 / 9.3, four 11.0 / 10.8; up to eight per unit two 12.4 / 15.7.
// Channels that lie apart: two steps 10.2 / 7.1, three 10.4 / 9.0, four 10.4 / 10.2, up to two tiles per unit two 10 / 8, three 11 / 15;
// on two waves one 13 / 9, two 14.4 / 15.
int contract_wide_float(const void *x, bool half, int position, const void *w, int N, int H, int W, int x_ci, bool apart, int Ci, int Co,
                        int kh, int kw, int ph, int pw, int sh, int sw, int dh, int dw, int Ho, int Wo, const EpiDev &e, hipStream_t s) {
  const bool dense = kh == 1 && kw == 1 && sh == 1 && sw == 1 && ph == 0 && pw == 0 && !apart;
  const int64_t M = (int64_t)N * Ho * Wo, tiles = (M + 31) / 32 * ((Co + 31) / 32);
  const int64_t steps = ((int64_t)kh * kw * Ci + 63) / 64;
  const int waves = tiles >= 2 * e.cus ? 2 : 4;
  const int most = apart ? (waves == 2 ? 1 : tiles <= e.cus ? 3 : 2) : (waves == 2 ? 3 : tiles <= e.cus ? 6 : 4);
  if (tiles > 4 * e.cus || (steps + waves - 1) / waves > most) return -1;
  WideParams p;
  if (!wide_params(&p, x, half ? 2 : 4, w, N, H, W, x_ci, apart, Ci, Co, kh, kw, ph, pw, sh, sw, dh, dw, Ho, Wo, dense, e)) return -1;
  p.x_neg_pos = -position;
  if (apart) return half ? launch_wide_float<false, IN_F16_APART>(waves, p, e, s) : launch_wide_float<false, IN_F32_APART>(waves, p, e, s);
  if (half && x_ci % 2 != 0)
    return dense ? launch_wide_float<true, IN_F16_ANY>(waves, p, e, s) : launch_wide_float<false, IN_F16_ANY>(waves, p, e, s);
  if (half) return dense ? launch_wide_float<true, IN_F16>(waves, p, e, s) : launch_wide_float<false, IN_F16>(waves, p, e, s);
  return dense ? launch_wide_float<true, IN_F32>(waves, p, e, s) : launch_wide_float<false, IN_F32>(waves, p, e, s);
}

int gemm_nt_mfma_a16w16(const void *a, const void *b, int64_t M, int64_t N, int64_t K, const EpiDev &e, hipStream_t s) {
  if (M >= (1ll << 31) - 64 || K >= (1 << 16)) return -1;
  return conv2d_mfma_a16w16(a, b, (int)M, 1, 1, (int)K, (int)N, 1, 1, 0, 0, 1, 1, 1, 1, 1, 1, e, s);
}

}  // namespace catchq
