// Linears and pointwise convolutions of unit stride on floating activations, filters in the order of the matrix instruction's
// lanes: a block converts its rows once, keeps them in LDS and streams the filters past them.
//
// As two launches -- quantizer, then GEMM -- every block of the GEMM walks K in steps that wait for their transfers, and its
// epilogue follows when the matrix cores are done: 4096 x 768 -> 3072 spent 5.5 us in the first and 17 in the second, 7.5 of
// them in six K steps and 4.5 in the epilogue.  Here a block owns 64 rows, all of K, and a run of columns.  Its activations are
// one run of memory, read sixteen bytes a lane with eight loads of a lane in flight, converted in registers and written to LDS.
// Then every wave walks column tiles of 64 of its own: the filters come straight into registers, a ring of RING sub-steps of
// K ahead and across the ends of tiles (packed, a load is a contiguous kilobyte; rows as they lie, sixteen bytes from each of
// 32, came at 36 KB/us a unit instead of 124).  The waves share nothing but the rows: there is no barrier after the first, and
// one wave's epilogue runs beside another's multiplications.
//
// What bounds it: the filters' way from the Infinity Cache through an XCD's L2 (33 B a clock and unit; without the
// multiplications the loop takes as long), then the conversions (19 vector instructions for 16 bytes) and the stores.  Tried
// without gain: a ring of eight, twelve waves, the filters touched into L2 beforehand, K started at a different step in each
// block, an L2-channel-sized shift between the filters' runs.
//
// Measured: see float_rows below.
#include "igemm_i8_dma.inc"

namespace catchq {

constexpr int kLdsBytes = 160 * 1024, kStageBytes = 32 * 72 * 4;  // a wave's staging area: 32 rows of 64 columns

template <int IN, int NW, int RING, int EPI>
__global__ __launch_bounds__(64 * NW, 2) void float_rows_kernel(const void *__restrict__ A, const int8_t *__restrict__ B,
                                                                  IgemmParams p, EpiDev e, int x_neg_pos, unsigned a_bytes,
                                                                  unsigned b_bytes, int col_tiles, unsigned units_magic) {
  resolve_exp2(e);
  constexpr int BM = 64, TM = 2, TN = 2, WN = 64, EPI_STRIDE = WN + 8;
  constexpr int ES = IN == IN_F32 ? 4 : 2, V = 16 / ES;  // activations per 16-byte load
  extern __shared__ __attribute__((aligned(16))) int8_t lds_dyn[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int logical = xcd_remap(blockIdx.x, p.nblocks);
  const int chunk = logical % p.tiles_n, tile_m = logical / p.tiles_n;
  const int64_t m0 = (int64_t)tile_m * BM;
  const int nk = (p.K + 31) / 32;                   // K sub-steps of 32
  const unsigned pitch = (unsigned)(nk * 2 + 1) * 16;  // an odd number of 16-byte pieces: fragment reads meet all banks
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void *)B, 0, (int)b_bytes, 0x00020000);

  // ---- this wave's filters, RING sub-steps ahead; the first go out behind the first activations ----------------------------
  const int tiles = (p.N + 63) / 64;
  int t = chunk * col_tiles + wave;
  const int t_end = min(tiles, (chunk + 1) * col_tiles);
  const int n32 = (p.N + 31) / 32;
  v4i fb[RING][TN];
  const int b_lane = lane * 16;
  auto fetch_b = [&](v4i (&f)[TN], int tile, int ks) {  // (a second half beyond N: the first one again, never stored)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int run = min(tile * TN + j, n32 - 1);
      f[j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_b, b_lane, (run * nk + ks) * 1024, 0));
    }
  };
  const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) int8_t *)lds_dyn;
  auto fetch_first = [&] {
#pragma unroll
    for (int r = 0; r < RING; ++r) fetch_b(fb[r], min(t, tiles - 1), min(r, nk - 1));
  };

  // ---- activations -> LDS ---------------------------------------------------------------------------------------------
  // The block's rows are one run of memory: unit u (16 bytes) is the u-th of it, its row u / units of a row (a 24-bit
  // multiplication).  What lies behind the run reads as zeros and is written behind the rows, where nothing is yet.
  {
    const unsigned tile_src = (unsigned)m0 * (unsigned)p.K * ES, tile_bytes = BM * (unsigned)p.K * ES;
    const unsigned src_end = a_bytes - tile_src < tile_bytes ? a_bytes : tile_src + tile_bytes;
    const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void *)A, 0, (int)src_end, 0x00020000);
    const unsigned units = tile_bytes / 16, pad = pitch - (unsigned)p.K;
    unsigned src = tile_src + threadIdx.x * 16, u9 = threadIdx.x << 9, dst = lds_base + threadIdx.x * V;
    auto load = [&](v4i &r) {
      r = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_a, (int)src, 0, 0));
      src += 64 * NW * 16;
    };
    auto convert = [&](const v4i &r) {
      int q[V / 4];
#pragma unroll
      for (int d = 0; d < V / 4; ++d) {
        int b[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          float v;
          if constexpr (IN == IN_F32) v = __int_as_float(r[k]);
          else {
            const int pair = r[d * 2 + (k >> 1)];
            v = (float)__builtin_bit_cast(_Float16, (short)((k & 1) ? pair >> 16 : pair & 0xffff));
          }
          b[k] = cvt_i32_sat(__builtin_rintf(__builtin_ldexpf(v, x_neg_pos)));
        }
        // two integers, saturated, to two bytes
        int lo, hi;
        asm("v_ashr_pk_i8_i32 %0, %1, %2, 0" : "=v"(lo) : "v"(b[0]), "v"(b[1]));
        asm("v_ashr_pk_i8_i32 %0, %1, %2, 0" : "=v"(hi) : "v"(b[2]), "v"(b[3]));
        q[d] = (int)__builtin_amdgcn_perm((unsigned)hi, (unsigned)lo, 0x05040100u);
      }
      unsigned row, at;
      asm("v_mul_hi_u32_u24 %0, %1, %2" : "=v"(row) : "v"(u9), "s"(units_magic));
      asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(at) : "v"(row), "s"(pad), "v"(dst));
      if constexpr (V == 4) asm volatile("ds_write_b32 %0, %1" ::"v"(at), "v"(q[0]) : "memory");
      else asm volatile("ds_write_b64 %0, %1" ::"v"(at), "v"(v2i{q[0], q[V / 4 - 1]}) : "memory");
      u9 += (64 * NW) << 9;
      dst += 64 * NW * V;
    };
    auto run = [&](auto wc) {
      constexpr int W = decltype(wc)::value;
      v4i raw[W];
#pragma unroll
      for (int i = 0; i < W; ++i) load(raw[i]);
      fetch_first();
      unsigned done = 0;
      do {
#pragma unroll
        for (int i = 0; i < W; ++i) {
          convert(raw[i]);
          load(raw[i]);
        }
        done += 64 * NW * W;
      } while (done < units);
    };
    if (units <= 64 * NW * 2) run(std::integral_constant<int, 2>{});
    else run(std::integral_constant<int, 8>{});
    if (p.K & 31) {  // K is a multiple of 16: the last sub-step's other half
      if (threadIdx.x < BM) *reinterpret_cast<v4i *>(lds_dyn + threadIdx.x * pitch + p.K) = v4i{0, 0, 0, 0};
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (writes the compiler does not know of)
  __syncthreads();

  const int8_t *fa_at = lds_dyn + (unsigned)(lane & 31) * pitch + (unsigned)(lane >> 5) * 16;
  int *stage = reinterpret_cast<int *>(lds_dyn + BM * pitch) + wave * 32 * EPI_STRIDE;
  typedef typename EpiOf<EPI>::type S;
  for (; t < t_end; t += NW) {
    const int n_w = t * WN;
    const int n = epi_lane_channel<TN>(n_w, lane);
    const EpiLane L = epi_lane_setup<S>(n, n < p.N, e);
    v16i acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;
    const int t_next = t + NW < t_end ? t + NW : t;
    v4i fa[2][TM];
    auto fetch_a = [&](v4i (&f)[TM], int ks) {
#pragma unroll
      for (int i = 0; i < TM; ++i) f[i] = *reinterpret_cast<const v4i *>(fa_at + (unsigned)(i * 32) * pitch + (unsigned)(ks * 32));
    };
    auto multiply = [&](v4i (&f)[TM], v4i (&g)[TN]) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f[i], g[j], acc[i][j], 0, 0, 0);
    };
    // a slot's next use: this tile's step RING further on, or the next tile's step r
    const int here = t * TN * nk * 1024, there = t_next * TN * nk * 1024;
    const int half_here = (min(t * TN + 1, n32 - 1) - t * TN) * nk * 1024, half_there = (min(t_next * TN + 1, n32 - 1) - t_next * TN) * nk * 1024;
    auto refill = [&](int r, int s) {
      const bool more = s + RING < nk;
      const int off = more ? here + (s + RING) * 1024 : there + min(r, nk - 1) * 1024;
      fb[r][0] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_b, b_lane, off, 0));
      fb[r][1] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_b, b_lane, off + (more ? half_here : half_there), 0));
    };
    fetch_a(fa[0], 0);
    int s = 0;
    for (; s + RING <= nk; s += RING) {
#pragma unroll
      for (int r = 0; r < RING; ++r) {
        fetch_a(fa[(r + 1) & 1], s + r + 1);  // (past the last step: a spare read, inside the block's LDS)
        __builtin_amdgcn_sched_barrier(0);    // the next step's rows are on their way before this one's multiplications
        multiply(fa[r & 1], fb[r]);
        refill(r, s + r);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (s < nk) {  // K ends inside a turn of the ring
#pragma unroll
      for (int r = 0; r < RING - 1; ++r) {
        if (s + r < nk) {
          fetch_a(fa[(r + 1) & 1], s + r + 1);
          multiply(fa[r & 1], fb[r]);
        }
        refill(r, s + r);
      }
    }
    igemm_epilogue_vec<TM, TN, EPI>(acc, stage, m0, n_w, lane, p, e, L);
  }
}

// w [N, K], K a multiple of 16 -> runs of 32 filters x 32 of K, a kilobyte each in the order of a wave's lanes; zeros beyond both.
__global__ __launch_bounds__(256) void pack_filters_kernel(const int8_t *__restrict__ w, int8_t *__restrict__ out, int N, int K, int nk) {
  const int64_t block = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);  // (32 filters, 32 of K): one kilobyte
  const int lane = threadIdx.x & 63;
  if (block >= (int64_t)((N + 31) / 32) * nk) return;
  const int64_t n = block / nk * 32 + (lane & 31);
  const int k = (int)(block % nk) * 32 + (lane >> 5) * 16;
  v4i v = {0, 0, 0, 0};
  if (n < N && k < K) v = *reinterpret_cast<const v4i *>(w + n * K + k);
  reinterpret_cast<v4i *>(out)[block * 64 + lane] = v;
}

template <int IN, int NW>
static int launch_float_rows(const void *a, const void *b, IgemmParams p, const EpiDev &e, int epi, int x_neg_pos, int col_tiles,
                             int lds, hipStream_t s) {
  constexpr int ES = IN == IN_F32 ? 4 : 2, RING = 4;
  const unsigned a_bytes = (unsigned)(p.M * p.K * ES), b_bytes = (unsigned)((p.N + 31) / 32 * ((p.K + 31) / 32) * 1024);
  // (u << 9) * magic >> 32 = u / upr for u < 64 upr, upr <= 362: the error, at most u / 2^23, stays below 1 / upr
  const unsigned upr = (unsigned)(p.K * ES / 16), magic = ((1u << 23) + upr - 1) / upr;
#define CATCHQ_ROWS_CASE(E)                                                                                                \
  case E: {                                                                                                                \
    auto kern = float_rows_kernel<IN, NW, RING, E>;                                                                        \
    static std::atomic<bool> raised[64];                                                                                   \
    if (raise_lds_limit((const void *)kern, kLdsBytes, raised) != CATCHQ_OK) return CATCHQ_ERR_LAUNCH;                     \
    kern<<<p.nblocks, 64 * NW, lds, s>>>(a, (const int8_t *)b, p, e, x_neg_pos, a_bytes, b_bytes, col_tiles, magic);       \
    break;                                                                                                                 \
  }
  switch (epi) {
    CATCHQ_ROWS_CASE(EPI_Y32)
    CATCHQ_ROWS_CASE(EPI_Y16)
    CATCHQ_ROWS_CASE(EPI_Y16_STEPS)
    default: return -1;
  }
#undef CATCHQ_ROWS_CASE
  return launch_status();
}

// x [M, K] floats (halfs), packed filters of N rows; -1: another route serves the call.
//
// Whether (one launch here / the routes without packed filters, us, fp32 output, half activations where marked):
//   4096 x 768 -> 3072 20 / 28, 12000 x 768 -> 2304 half 42 / 53, 5000 x 1024 -> 1024 half 16 / 21, 3901 x 720 -> 896 12 / 18,
//   14785 x 208 -> 800 18 / 22, 1462 x 848 -> 3392 17 / 21, 5168 x 128 -> 608 half 7.8 / 9.5, 1025 x 544 -> 2060 half
//   10.7 / 11.0, 18208 x 336 -> 268 17.2 / 18.4.  Small outputs and few rows do not pay for a block's conversions:
//   673 x 624 -> 776 half 9.0 / 7.7, 528 x 640 -> 2516 half 10.2 / 10.0, 2992 x 1088 -> 312 12.8 / 12.1; nor do few columns,
//   which the GEMM for them reads once as well: 9565 x 224 -> 128 half 6.6 / 6.0, 7132 x 256 -> 228 half 7.4 / 6.6.
//   Half outputs are half the stores of that GEMM, so they take more columns: 6272 x 256 -> 1024 10.2 / 12.8, 1568 x 512 -> 2048
//   8.8 / 10.0, 31360 x 96 -> 576 18.5 / 20.2; 25088 x 128 -> 512 13.7 / 14.0, 100352 x 64 -> 256 20.1 / 18.9.
// How (M x K -> N, waves and column tiles of a block): a short K leaves LDS for two blocks of four waves, one in its
// conversions while the other multiplies, with a tile a wave -- 13145 x 384 -> 3384 half 55.3 on 4 x 4, 68 on 8 x 8 and
// 8 x 16; 22255 x 240 -> 960 half 23.7 / 27.0 on 8 x 8 -- and so does a K that fits twice where the rows make more than a
// round of blocks (20853 x 560 -> 572 half 25.4 / 31.4).  Else eight waves, one block a unit, and the fewest blocks that give
// one round: every run of columns converts the rows again (14938 x 1200 -> 512 half 23.5 on all columns, 29.6 on half of
// them; 3689 x 912 -> 2160 half 19.9 on 12 tiles, 23.0 on nine, which leave waves without a second tile).
bool float_rows_takes(bool half, int64_t M, int64_t N, int64_t K, const EpiDev &e) {
  if (!float_rows_sizes(M, N, K, e.y_f16 != 0)) return false;
  if (M * K * (half ? 2 : 4) >= (1ll << 31) || (N + 31) / 32 * ((K + 31) / 32) * 1024 >= (1ll << 31) ||
      (M + 63) / 64 * ((N + 63) / 64) >= (1ll << 31))
    return false;
  const int epi = pick_epilogue((int)N, e);
  return epi == EPI_Y32 || epi == EPI_Y16 || epi == EPI_Y16_STEPS;
}

int float_rows(const void *x, bool half, int position, const void *packed, int64_t M, int64_t N, int64_t K, const EpiDev &e,
               hipStream_t s) {
  if (!float_rows_takes(half, M, N, K, e)) return -1;
  const int64_t row_tiles = (M + 63) / 64, tiles = (N + 63) / 64;
  const int epi = pick_epilogue((int)N, e);
  const int64_t rows_lds = 64 * ((K + 31) / 32 * 2 + 1) * 16;
  auto lds = [&](int nw) { return (int)(rows_lds + nw * kStageBytes); };
  const bool four = K <= 448 || (row_tiles > e.cus && 2 * lds(4) <= kLdsBytes);
  int64_t run = 4;  // column tiles of a block
  if (!four) {
    const int64_t runs = row_tiles < e.cus ? e.cus / row_tiles : 1;
    run = (tiles + runs - 1) / runs;
    if (runs > 1) run = (run + 3) / 4 * 4;
  }
  const int64_t runs = (tiles + run - 1) / run;
  run = (tiles + runs - 1) / runs;
  IgemmParams p = {};
  p.M = M; p.N = (int)N; p.K = (int)K;
  p.tiles_n = (int)((tiles + run - 1) / run);
  p.nblocks = (int)(row_tiles * p.tiles_n);
  if (four)
    return half ? launch_float_rows<IN_F16, 4>(x, packed, p, e, epi, -position, (int)run, lds(4), s)
                : launch_float_rows<IN_F32, 4>(x, packed, p, e, epi, -position, (int)run, lds(4), s);
  return half ? launch_float_rows<IN_F16, 8>(x, packed, p, e, epi, -position, (int)run, lds(8), s)
              : launch_float_rows<IN_F32, 8>(x, packed, p, e, epi, -position, (int)run, lds(8), s);
}

int pack_filters(const void *w, void *packed, int64_t N, int64_t K, hipStream_t s) {
  const int64_t nk = (K + 31) / 32, blocks = ((N + 31) / 32 * nk + 3) / 4;
  pack_filters_kernel<<<(unsigned)blocks, 256, 0, s>>>((const int8_t *)w, (int8_t *)packed, (int)N, (int)K, (int)nk);
  return launch_status();
}

}  // namespace catchq
