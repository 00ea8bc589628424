// Contractions of int8 or int16 activations with int8 weights, long in K, of which the chip holds only a few blocks per
// compute unit: the K loop split over the waves of a block, each with a tile of its own of 64 x 64 (or 32 x 64) outputs.
//
// What bounds such a launch in the tiled kernels: a block walks K in steps of 64 with a barrier and an LDS round trip each,
// 410 (int8) to 570 (int16) clocks a step for 64 to 128 clocks of matrix instructions, and with one or two blocks a unit
// nothing runs under that.  Here a wave owns a contiguous slice of K and walks it alone: its transfers (LDS-DMA) go to
// slots of its own, it waits for nothing but those, the first half of the next step is requested before the second half of
// this one is multiplied, and the loop is NW times shorter.  A wave's tile of 64 x 64 reads a quarter less from LDS per matrix
// instruction than four waves of 32 x 32 do (int16: a third), which is what many blocks a unit are bound by.  The partial
// sums meet in LDS once, behind the loop.
//
// int16 activations are split into digits in registers as in igemm_a16_dma.hip (x = 256 hi + lo + 128); the weights' sums that
// the constant 128 needs are collected from the fragments and added with the partial sums.
#include "igemm_i8_dma.inc"

namespace catchq {

struct KsplitParams {
  const void *x;
  const int8_t *w;
  int M, N, K;                                    // M * max(Wo, Ho) < 2^32
  int H, W, Ci, Wo, Ho, kh, kw, ph, pw, sh, sw, dh, dw;
  unsigned magic_wo, magic_ho, magic_t, mask_wo, mask_ho, mask_t;  // quotients through multiplication (ksplit_div)
  int tiles_m, tiles_n, nblocks;
  int m_fastest;                                  // consecutive blocks walk the row tiles of one column tile first
  int epi, ragged;                                // as in WideParams
  unsigned a_bytes, b_bytes;
};

// (No barrier orders the transfers against the waits and the reads: the compiler has to keep them where they are written.)
#define CATCHQ_KSPLIT_VMCNT(n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(n) : "memory")

// n / d for n * d < 2^32 through magic = ceil(2^32 / d) (d = 1: magic 0, mask ~0)
__device__ __forceinline__ unsigned ksplit_div(unsigned n, unsigned magic, unsigned mask) { return __umulhi(n, magic) + (n & mask); }

// how the loader walks K: a plain GEMM; a convolution whose steps of 64 lie within one filter tap (Ci a multiple of 64); one
// whose 16-byte pieces do (a multiple of 16, int8)
enum { KW_DENSE = 0, KW_TAP = 1, KW_PIECE = 2 };

// A16: int16 activations.  SLOTS: K steps a wave has in LDS or on the way there.
template <int TM, int TN, int NW, int SLOTS, int WALK, bool A16>
__global__ __launch_bounds__(64 * NW, TM * TN == 4 ? 2 : 0) void ksplit_kernel(KsplitParams p, EpiDev e) {
  fetch_arguments<sizeof(KsplitParams) + sizeof(EpiDev)>();  // plans, us: six 208 x 208 ResNet-18 133.1 / 128.0, four 320 x 320 Darknet-53 773 / 765
  resolve_exp2(e);
  constexpr int BM = TM * 32, BN = TN * 32, KS = 64;  // values of K per step
  constexpr int ES = A16 ? 2 : 1, AROW = KS * ES;     // bytes per activation, of a tile row of them per step
  constexpr int ARPI = 1024 / AROW;                   // activation rows per transfer (1 KiB)
  constexpr int NA = BM / ARPI, NB = BN / 16, NI = NA + NB;
  constexpr int A_BYTES = BM * AROW, SLOT_BYTES = A_BYTES + BN * KS, WAVE_BYTES = SLOTS * SLOT_BYTES;
  static_assert(BM * BN * 4 <= WAVE_BYTES, "a partial tile fits the wave's slots");
  static_assert(SLOTS >= 2 && !(A16 && WALK == KW_PIECE), "two steps in flight; int16 walks whole taps");
  constexpr unsigned OOB = 0x80000000u;  // the hardware answers an offset beyond the buffer with zeros
  extern __shared__ __attribute__((aligned(16))) int8_t lds_dyn[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int logical = xcd_remap(blockIdx.x, p.nblocks);
  const int outer = (int)ksplit_div((unsigned)logical, p.magic_t, p.mask_t);
  const int inner = logical - outer * (p.m_fastest ? p.tiles_m : p.tiles_n);
  const int m0 = (p.m_fastest ? inner : outer) * BM, n0 = (p.m_fastest ? outer : inner) * BN;
  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void *)p.x, 0, (int)p.a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void *)p.w, 0, (int)p.b_bytes, 0x00020000);

  // ---- what the epilogue needs, requested before anything else: a lane's four channels, and its residual where it has one
  // pixel ------------------------------------------------------------------------------------------------------------------
  constexpr int CPR = BN / 4, ITEMS = BM * CPR, THREADS = 64 * NW;
  static_assert(THREADS % CPR == 0, "a lane keeps its four channels");
  constexpr bool ONE_ROUND = ITEMS <= THREADS;
  const int cg = threadIdx.x % CPR, n = n0 + cg * 4;
  v4f c_div = {1.f, 1.f, 1.f, 1.f}, c_rcp = c_div, c_res = {0.f, 0.f, 0.f, 0.f};
  Bias4 c_bias;
  if (!p.ragged) {
    const int cc = min(n, p.N - 4);
    const float *rcps = e.chan_rcp ? e.chan_rcp : e.half_rcp;
    if (e.chan_div) c_div = *reinterpret_cast<const v4f *>(e.chan_div + cc);
    if (rcps) c_rcp = *reinterpret_cast<const v4f *>(rcps + cc);
    c_bias.load(e, cc);
    if (ONE_ROUND && e.resid)
      c_res = *reinterpret_cast<const v4f *>(e.resid + (int64_t)min(m0 + (int)threadIdx.x / CPR, p.M - 1) * p.N + cc);
  }

  // ---- this wave's slice of K ------------------------------------------------------------------------------------------
  const int steps = (p.K + KS - 1) / KS;
  const int per = steps / NW, rem = steps - per * NW;
  const int first = wave * per + (wave < rem ? wave : rem);
  const int mine = per + (wave < rem ? 1 : 0);

  // ---- loader: as in the tiled kernels, whole waves of rows; the 16-byte piece a lane fetches is swizzled by the row so that
  // the fragment reads of 16 rows fall into different 16-byte slots -------------------------------------------------------
  int a_piece[2];  // piece (of 16 bytes) of this lane in even and odd transfers
  if constexpr (A16) {
    a_piece[0] = (lane & 7) ^ (lane >> 4);
    a_piece[1] = a_piece[0] ^ 4;
  } else {
    a_piece[0] = a_piece[1] = (lane & 3) ^ ((lane >> 4) & 3);
  }
  const int b_piece = (lane & 3) ^ ((lane >> 4) & 3);
  unsigned a_base[NA], a_off[NA], b_off[NB];  // bytes; a_off: of the tap in hand, OOB where there is nothing
  int hi0[NA], wi0[NA];
#pragma unroll
  for (int j = 0; j < NA; ++j) {
    const unsigned m = (unsigned)(m0 + j * ARPI + (A16 ? lane >> 3 : lane >> 2));
    hi0[j] = wi0[j] = 0;
    if constexpr (WALK == KW_DENSE) {
      a_off[j] = m < (unsigned)p.M ? m * (unsigned)p.K * ES + a_piece[j & 1] * 16 : OOB;
    } else {
      const unsigned t = ksplit_div(m, p.magic_wo, p.mask_wo), wo = m - t * (unsigned)p.Wo;
      const unsigned img = ksplit_div(t, p.magic_ho, p.mask_ho), ho = t - img * (unsigned)p.Ho;
      hi0[j] = m < (unsigned)p.M ? (int)ho * p.sh - p.ph : -(1 << 30);  // a row that does not exist is outside the image
      wi0[j] = (int)wo * p.sw - p.pw;
      a_base[j] = ((img * (unsigned)p.H + (unsigned)((int)ho * p.sh - p.ph)) * (unsigned)p.W + (unsigned)wi0[j]) * (unsigned)(p.Ci * ES) +
                  (WALK == KW_TAP ? a_piece[j & 1] * 16 : 0);  // mod 2^32
    }
  }
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int n = n0 + j * 16 + (lane >> 2);
    b_off[j] = n < p.N ? (unsigned)n * (unsigned)p.K + b_piece * 16 : OOB;
  }
  // Where the next transfer reads: (tap row, tap column, channel), one for the wave (KW_TAP) or one per lane (KW_PIECE).  A
  // lane's offsets are rebuilt when its tap changes and walk along the channels in between.
  int k_next = first * KS, tr = 0, tq = 0, ci = 0;
  auto enter_tap = [&]() {
    const int dy = tr * p.dh, dx = tq * p.dw;
    const unsigned off = (unsigned)((dy * p.W + dx) * p.Ci + (WALK == KW_PIECE ? ci : 0)) * ES;
#pragma unroll
    for (int j = 0; j < NA; ++j) {
      // (past the last tap: nothing)
      const bool in = (tr < p.kh) & ((unsigned)(hi0[j] + dy) < (unsigned)p.H) & ((unsigned)(wi0[j] + dx) < (unsigned)p.W);
      a_off[j] = select_u32(in, a_base[j] + off, OOB);
    }
  };
  if constexpr (WALK != KW_DENSE) {
    const int k = k_next + (WALK == KW_PIECE ? a_piece[0] * 16 : 0);
    const int tap = k / p.Ci;
    ci = k - tap * p.Ci;
    tr = tap / p.kw;
    tq = tap - tr * p.kw;
    enter_tap();
  }
  int8_t *const my = lds_dyn + wave * WAVE_BYTES;
  auto issue = [&](int slot_off) {  // the next step of the slice into a slot
    int a_soff = 0;
    if constexpr (WALK == KW_DENSE) a_soff = k_next * ES;
    if constexpr (WALK == KW_TAP) a_soff = ci * ES;
    if (WALK == KW_DENSE && k_next + KS > p.K) {  // K ends inside this step
#pragma unroll
      for (int j = 0; j < NA; ++j)
        a_off[j] = select_u32(k_next + a_piece[j & 1] * (16 / ES) < p.K, a_off[j], OOB);
    }
#pragma unroll
    for (int j = 0; j < NA; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_ptr_t)(my + slot_off + j * 1024), 16, (int)a_off[j], a_soff, 0, 0);
    // (weights beyond K meet zeros; a row that does not exist stays out of range whatever is added)
#pragma unroll
    for (int j = 0; j < NB; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, (lds_ptr_t)(my + slot_off + A_BYTES + j * 1024), 16, (int)b_off[j], k_next, 0, 0);
    k_next += KS;
    if constexpr (WALK == KW_TAP) {
      ci += KS;
      if (ci == p.Ci) {
        ci = 0;
        if (++tq == p.kw) { tq = 0; ++tr; }
        enter_tap();
      }
    }
    if constexpr (WALK == KW_PIECE) {
      ci += KS;
      if (__builtin_amdgcn_ballot_w64(ci >= p.Ci) != 0) {
        while (ci >= p.Ci) {
          ci -= p.Ci;
          if (++tq == p.kw) { tq = 0; ++tr; }
        }
        enter_tap();
      } else {
#pragma unroll
        for (int j = 0; j < NA; ++j) a_off[j] += KS;  // (out of range stays out of range: fewer than 2^31 bytes of channels)
      }
    }
  };

  // ---- K loop ----------------------------------------------------------------------------------------------------------
  // Weights are the matrix instruction's first operand: a lane ends up with four consecutive channels of one pixel.
  v16i acc[TM][TN], acc_hi[A16 ? TM : 1][A16 ? TN : 1];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[i][j][r] = 0;
        if constexpr (A16) acc_hi[i][j][r] = 0;
      }
  int wsum[TN] = {};
  const int frow = lane & 31, fhalf = lane >> 5;
  const unsigned my_addr = (unsigned)(uintptr_t)(__attribute__((address_space(3))) int8_t *)my;
  const unsigned a_row = my_addr + (unsigned)(frow * AROW), b_row = my_addr + (unsigned)(A_BYTES + frow * KS);
  // half u of a step (32 values): int16 pieces 4u + 2 fhalf and the next, int8 piece 2u + fhalf
  const unsigned a_p0 = A16 ? (unsigned)(((fhalf * 2) ^ ((frow >> 1) & 7)) * 16) : (unsigned)((fhalf ^ ((frow >> 2) & 3)) * 16);
  const unsigned b_p0 = (unsigned)((fhalf ^ ((frow >> 2) & 3)) * 16);
  constexpr unsigned A_FLIP = A16 ? 64 : 32;
  struct Half { v4i a[TM][ES], b[TN]; };
  constexpr int NF = TM * ES + TN;  // LDS reads per half
  auto fetch = [&](Half &f, int slot_off, int u) {
    const unsigned a = a_row + (unsigned)slot_off + (u ? a_p0 ^ A_FLIP : a_p0);
    const unsigned b = b_row + (unsigned)slot_off + (u ? b_p0 ^ 32u : b_p0);
    f.a[0][0] = ds_read_b128<0>(a);
    if constexpr (A16) f.a[0][ES - 1] = ds_read_b128<0>(a ^ 16u);
    if constexpr (TM > 1) {
      f.a[TM - 1][0] = ds_read_b128<32 * AROW>(a);
      if constexpr (A16) f.a[TM - 1][ES - 1] = ds_read_b128<32 * AROW>(a ^ 16u);
    }
    f.b[0] = ds_read_b128<0>(b);
    if constexpr (TN > 1) f.b[TN - 1] = ds_read_b128<32 * KS>(b);
  };
  static_assert(TM <= 2 && TN <= 2, "a wave's tile is at most 64 x 64");
  auto arrived = [&](Half &f, auto behind_c) {  // but for the reads issued behind them
    constexpr int BEHIND = decltype(behind_c)::value;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int h = 0; h < ES; ++h) lgkm_wait<BEHIND>(f.a[i][h]);
#pragma unroll
    for (int j = 0; j < TN; ++j) lgkm_wait<BEHIND>(f.b[j]);
    asm volatile("" ::: "memory");
  };
  auto multiply = [&](const Half &f) {
    if constexpr (A16) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int d = 0; d < 4; ++d) wsum[j] = __builtin_amdgcn_sdot4(f.b[j][d], 0x01010101, wsum[j], false);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        v4i hi, lo;
        split_i16(f.a[i][0], f.a[i][ES - 1], hi, lo);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          acc_hi[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f.b[j], hi, acc_hi[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f.b[j], lo, acc[i][j], 0, 0, 0);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f.b[j], f.a[i][0], acc[i][j], 0, 0, 0);
    }
  };
  const int issued = mine < SLOTS ? mine : SLOTS;
  for (int s = 0; s < issued; ++s) issue(s * SLOT_BYTES);
  if (mine > 0) {
    Half f0, f1;
    // (a wait that leaves the newer steps on their way needs all of them to have been issued)
    if (issued == SLOTS) CATCHQ_KSPLIT_VMCNT(NI * (SLOTS - 1));
    else CATCHQ_KSPLIT_VMCNT(0);
    fetch(f0, 0, 0);
    int rd = 0;
    for (int s = 0; s < mine; ++s) {
      fetch(f1, rd, 1);
      arrived(f0, std::integral_constant<int, NF>{});
      multiply(f0);
      arrived(f1, std::integral_constant<int, 0>{});  // the slot has been read
      const int slot = rd;
      rd = rd + SLOT_BYTES == WAVE_BYTES ? 0 : rd + SLOT_BYTES;
      if (s + SLOTS <= mine) CATCHQ_KSPLIT_VMCNT(NI * (SLOTS - 2));
      else CATCHQ_KSPLIT_VMCNT(0);
      // Always, past the last step too (what the slot holds, not used): under a condition the compiler may copy fragments that
      // have not arrived.
      fetch(f0, rd, 0);
      if (s + SLOTS < mine) issue(slot);
      multiply(f1);
    }
    arrived(f0, std::integral_constant<int, 0>{});
  }
  {  // ---- this wave's partial sums (without steps: zeros): [pixel][channel], 16-byte pieces swizzled by the pixel ---------
    int *const part = reinterpret_cast<int *>(my);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          v4i v;
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            v[u] = acc[i][j][4 * g + u];
            if constexpr (A16) v[u] = (int)(((unsigned)acc_hi[i][j][4 * g + u] << 8) + (unsigned)v[u]);
          }
          const int piece = j * 8 + g * 2 + fhalf;
          *reinterpret_cast<v4i *>(part + (i * 32 + frow) * BN + (piece ^ (frow & (BN / 4 - 1))) * 4) = v;
        }
  }
  if constexpr (A16) {  // 128 x the sum of a channel's weights over this wave's slice (a wave without steps: 0)
    int *const sums = reinterpret_cast<int *>(lds_dyn + NW * WAVE_BYTES) + wave * BN;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int ws = wsum[j] + __shfl_xor(wsum[j], 32, 64);
      if (fhalf == 0) sums[j * 32 + frow] = (int)((unsigned)ws << 7);
    }
  }

  // ---- partial sums -> outputs -----------------------------------------------------------------------------------------
  auto finish = [&](auto spec, auto ragged_c) {
    typedef decltype(spec) S;
    constexpr bool RAGGED = decltype(ragged_c)::value;
    constexpr int BATCH = ONE_ROUND ? 1 : 4;  // rounds whose residuals travel together
    const bool n_ok = n < p.N;
    EpiLane L;
    if constexpr (RAGGED) L = epi_lane_setup_ragged<S>(n_ok ? n : 0, p.N, e);
    else L = epi_lane_finish<S>(c_div, c_rcp, c_bias.values(e), e);
    v4f res[BATCH];
    auto load_residuals = [&](int t0) {
#pragma unroll
      for (int b = 0; b < BATCH; ++b) {
        const int t = t0 + b * THREADS, m = m0 + t / CPR;
        res[b] = v4f{0.f, 0.f, 0.f, 0.f};
        if (!RAGGED && L.use_res && n_ok && t < ITEMS && m < p.M)
          res[b] = load_stream(reinterpret_cast<const v4f *>(e.resid + (int64_t)m * p.N + n), e.resid_stream != 0);
      }
    };
    if constexpr (ONE_ROUND) res[0] = c_res;
    else load_residuals(threadIdx.x);
    __syncthreads();
    if (!n_ok) return;
    v4i ws = {0, 0, 0, 0};
    if constexpr (A16) {
      const int *sums = reinterpret_cast<const int *>(lds_dyn + NW * WAVE_BYTES) + cg * 4;
#pragma unroll
      for (int w = 0; w < NW; ++w) ws += *reinterpret_cast<const v4i *>(sums + w * BN);
    }
    for (int t0 = threadIdx.x; t0 < ITEMS; t0 += BATCH * THREADS) {
      if (t0 != (int)threadIdx.x) load_residuals(t0);
#pragma unroll
      for (int b = 0; b < BATCH; ++b) {
        const int t = t0 + b * THREADS, px = t / CPR, m = m0 + px;
        if (t >= ITEMS || m >= p.M) break;
        const int *src = reinterpret_cast<const int *>(lds_dyn) + px * BN + (cg ^ (px & (CPR - 1))) * 4;
        v4i a = ws;
#pragma unroll
        for (int w = 0; w < NW; ++w) a += *reinterpret_cast<const v4i *>(src + w * (WAVE_BYTES / 4));
        const int64_t idx = (int64_t)m * p.N + n;
        if constexpr (RAGGED) epi_vec4<S>(a, res[b], L, EpiAtRagged{idx, p.N - n}, e);
        else epi_vec4<S>(a, res[b], L, idx, e);
      }
    }
  };
  const std::true_type ragged;
  const std::false_type whole;
  if constexpr (A16) {
    switch (p.epi) {
      case EPI_LK_Q16: finish(EpiOf<EPI_LK_Q16>::type{}, whole); break;
      case EPI_LK_Y_Q16: finish(EpiOf<EPI_LK_Y_Q16>::type{}, whole); break;
      case EPI_LK_RESA_Q16: finish(EpiOf<EPI_LK_RESA_Q16>::type{}, whole); break;
      case EPI_LK_RESA_Y_Q16: finish(EpiOf<EPI_LK_RESA_Y_Q16>::type{}, whole); break;
      case EPI_Y16: finish(EpiOf<EPI_Y16>::type{}, whole); break;
      default: finish(EpiGeneric{}, whole); break;
    }
  } else {
    switch (p.epi) {
      case EPI_Q8_RELU: finish(EpiOf<EPI_Q8_RELU>::type{}, whole); break;
      case EPI_RES_Y_Q8: finish(EpiOf<EPI_RES_Y_Q8>::type{}, whole); break;
      case EPI_RES_Q8: finish(EpiOf<EPI_RES_Q8>::type{}, whole); break;
      case EPI_Y32: p.ragged ? finish(EpiOf<EPI_Y32>::type{}, ragged) : finish(EpiOf<EPI_Y32>::type{}, whole); break;
      case EPI_Y16: p.ragged ? finish(EpiOf<EPI_Y16>::type{}, ragged) : finish(EpiOf<EPI_Y16>::type{}, whole); break;
      case EPI_Y16_RELU: finish(EpiOf<EPI_Y16_RELU>::type{}, whole); break;
      case EPI_Y16_STEPS: finish(EpiOf<EPI_Y16_STEPS>::type{}, whole); break;
      case EPI_Q8_RELU6: finish(EpiOf<EPI_Q8_RELU6>::type{}, whole); break;
      case EPI_LIN_Q8: finish(EpiOf<EPI_LIN_Q8>::type{}, whole); break;
      case EPI_LIN_RES_Q8: finish(EpiOf<EPI_LIN_RES_Q8>::type{}, whole); break;
      case EPI_LIN_Y_Q8: finish(EpiOf<EPI_LIN_Y_Q8>::type{}, whole); break;
      case EPI_LIN_RES_Y_Q8: finish(EpiOf<EPI_LIN_RES_Y_Q8>::type{}, whole); break;
      default: finish(EpiGeneric{}, whole); break;
    }
  }
}

template <int TM, int TN, int NW, int SLOTS, int WALK, bool A16>
static int launch_ksplit(KsplitParams p, const EpiDev &e, hipStream_t s) {
  constexpr int BM = TM * 32, BN = TN * 32;
  constexpr int LDS_BYTES = NW * SLOTS * (BM * (A16 ? 128 : 64) + BN * 64) + (A16 ? NW * BN * 4 : 0);
  auto kern = ksplit_kernel<TM, TN, NW, SLOTS, WALK, A16>;
  if (LDS_BYTES > 64 * 1024) {
    static std::atomic<bool> raised[64];
    if (raise_lds_limit((const void *)kern, LDS_BYTES, raised) != CATCHQ_OK) return CATCHQ_ERR_LAUNCH;
  }
  const int64_t tm = ((int64_t)p.M + BM - 1) / BM, tn = ((int64_t)p.N + BN - 1) / BN, inner = p.m_fastest ? tm : tn;
  if (tm * tn > 0x7fffffff || tm * tn * inner >= (1ll << 32)) return -1;
  p.tiles_m = (int)tm;
  p.tiles_n = (int)tn;
  p.nblocks = (int)(tm * tn);
  p.magic_t = inner <= 1 ? 0u : (unsigned)(((1ull << 32) + inner - 1) / inner);
  p.mask_t = inner <= 1 ? ~0u : 0u;
  kern<<<p.nblocks, 64 * NW, LDS_BYTES, s>>>(p, e);
  return launch_status();
}

// The plan (tile rows and columns / 32, waves, slots) for M x N outputs over `steps` steps of 64, 0: not this kernel's shape.
//
// Measured with the launch repeated in a graph (us, this kernel / what served the shape before; MI355X), in brackets with
// operands that the caches of the units' own dies do not hold, as inside a network.  t: 32 x 32 tiles, t2: 32 x 64 ones, t4:
// 64 x 64 ones, for 256 units.
// int8.  Where 16 x 16 tiles (small_i8.hip) leave no unit more than two they are ahead.  Beyond, 32 x 32 tiles while no unit
//   has more than 1.75: 784 x 1024 -> 512 (t 400) 4.2 / 5.1 (4.4 / 5.3), 196 x 256 -> 1024 (224) 3.1 / 3.3, 300 x 2048 -> 900 5.2 /
//   6.0, 3 x 3 on 4 x 28 x 28, 128 channels (392) 4.5 / 5.7 (5.0 / 5.8), on 4 x 14 x 14, 256 (200) 4.4 on eight waves / 5.6
//   (4.9 / 5.5).  A GEMM of more than 40 steps (512 x 3072 -> 768, t 384, 7.5 / 7.3) stays as it was, and
//   beyond 24 one whose rows do not start on cache lines (with the quantizer: 1794 x 1936 -> 84 10.4 / 9.8, 716 x 1904 -> 364
//   10.7 / 10.2, 1099 x 1712 -> 120 9.2 / 8.7, but 1993 x 2048 -> 136 11.4 / 12.0).
//   Convolutions: 32 x 64 tiles up to one per unit -- 5 x 28 x 28, 128 channels (t2 246) 5.0 / 6.3 (5.5 / 6.3) -- and up to two for
//   short K, 5 x 56 x 56, 64 channels (490, nine steps) 4.9 / 5.7 (5.3 / 5.7).  64 x 64 tiles up to one per unit -- 5 x 5, 256 ->
//   128 on 8 x 28 x 28 (t4 196) 15.1 / 24.0 (15.6 / 24.7), 40 x 7 x 7, 512 (248) 12.5 / 20.8, 12 x 28 x 28 / 2, 256 (148) 7.5 / 9.6
//   (8.5 / 9.6), 20 x 14 x 14, 256 (245) 7.8 / 8.6 (8.5 / 8.6); 7 x 25 x 25, 160 -> 320 (345) 9.8 / 10.0.  Three slots a wave: 2-5 %
//   with cold operands.  More than 64 steps: 8 x 7 x 7, 512 (t 208) 6.2 / 7.1 (6.8 / 7.1), 12 x 7 x 7 (304) 8.3 / 9.0 (8.6 /
//   9.1), 16 x 7 x 7 (t2 200) 8.7 / 9.2 (9.5 / 9.7); the few-tiles kernel is ahead for 20 x 7 x 7 (t 496, t2 248) 9.3 / 9.6, and the
//   patch-resident one, where it makes one round, for 6 x 17 x 17, 512 -> 448 (t4 196) 10.9 / 12.1, not for 24 x 7 x 7 (152)
//   11.3 / 10.2 (11.9 / 11.2).
//   GEMMs: 64 x 64 tiles up to 0.9 per unit from K = 4096 on, 900 x 4096 -> 900 (t4 225) 13.3 / 15.8; 700 x 3008 -> 1500 (264)
//   14.0 / 13.4, 1024 x 1024 -> 1024 (256) 6.0 / 5.6, with the quantizer 981 x 3200 -> 492 (128) 16.1 / 15.1, 2219 x 2128 -> 384
//   (210) 16.9 / 16.0.
// int16, 3 x 3: one 13 x 13 image, 512 -> 1024 (t 192) 7.7 on eight waves / 29.9 (8.3 / 30.4), two (t2 176) 10.7 / 30.4, six
//   (t4 256) 18.0 / 31.0, eight (t2 688, two waves) 26.7 / 34.0; 26 x 26, 256 -> 512: one image (t2 176) 7.1 / 18.0, two (t 688)
//   11.1 / 18.8, four (t2 680, two waves) 15.8 / 21.3; 52 x 52, 128 -> 256: one (t 680) 7.6 / 12.4, two (t2 676, two waves) 11.1 /
//   15.0, four (1352) 19.6 / 17.4; 1 x 1, 1024 -> 512 on eight 13 x 13 images (t 688) 6.9 / 8.1.
// patch: the patch-resident kernel would serve the shape in one round of blocks.
static int ksplit_plan(int64_t M, int64_t N, int64_t K, bool dense, bool a16, bool patch, int cus) {
  auto tiles = [&](int bm, int bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  const int64_t t = tiles(32, 32), t2 = tiles(32, 64), t4 = tiles(64, 64), steps = (K + 63) / 64;
  if (const char *f = tuning_env("CATCHQ_KSPLIT")) return std::atoi(f);
  if (K < 256) return 0;
  if (a16) {
    if (t <= cus) return steps >= 32 ? 1182 : 1142;
    if (t2 * 4 <= 3 * cus && steps >= 32) return 1282;
    if (t * 4 <= 11 * cus && steps <= 40) return 1142;
    if (t4 <= cus && steps >= 32) return 2242;
    if (t2 * 4 <= 11 * cus && !dense && steps >= 9) return 1222;
    return 0;
  }
  if (tiles(16, 16) <= 2 * cus) return 0;
  if (t * 4 <= 7 * cus && (dense ? steps <= 24 || (steps <= 40 && K % 128 == 0) : steps <= 40))
    return !dense && steps >= 32 && t <= cus ? 1182 : 1142;
  if (dense) return t * 4 > 7 * cus && t4 * 10 <= 9 * cus && K >= 4096 ? 2242 : 0;
  if (steps > 64) {
    if (t <= cus) return 1182;
    if (t * 4 <= 5 * cus) return 1142;
    if (t2 * 5 <= 4 * cus) return 1282;
    if (t <= 2 * cus || (patch && t4 * 5 > 3 * cus)) return 0;
  } else if (t2 <= cus || (t2 <= 2 * cus && steps <= 13)) {
    return 1242;
  }
  return t4 <= cus ? 2242 : 0;
}

template <int WALK, bool A16>
static int pick_ksplit(int plan, const KsplitParams &p, const EpiDev &e, hipStream_t s) {
  switch (plan) {
    case 1142: return launch_ksplit<1, 1, 4, 2, WALK, A16>(p, e, s);
    case 2242: return launch_ksplit<2, 2, 4, A16 ? 2 : 3, WALK, A16>(p, e, s);
    case 1182:
      if constexpr (A16 || WALK != KW_DENSE) return launch_ksplit<1, 1, 8, 2, WALK, A16>(p, e, s);
      return -1;
    case 1282:
      if constexpr (A16 || WALK != KW_DENSE) return launch_ksplit<1, 2, 8, 2, WALK, A16>(p, e, s);
      return -1;
    case 1242:
      if constexpr (!A16 && WALK != KW_DENSE) return launch_ksplit<1, 2, 4, 2, WALK, A16>(p, e, s);
      return -1;
    case 1222:
      if constexpr (A16 && WALK == KW_TAP) return launch_ksplit<1, 2, 2, 2, WALK, A16>(p, e, s);
      return -1;
    default: return -1;
  }
}

// kh = kw = 1, stride 1, no padding: a GEMM of M = N_img * H * W rows.  -1: not this kernel's shape.
int contract_ksplit(const void *x, bool a16, const void *w, int N_img, int H, int W, int Ci, int Co, int kh, int kw, int ph, int pw,
                    int sh, int sw, int dh, int dw, int Ho, int Wo, bool patch, const EpiDev &e, hipStream_t s) {
  const int64_t M = (int64_t)N_img * Ho * Wo, K = (int64_t)kh * kw * Ci;
  const bool dense = kh == 1 && kw == 1 && sh == 1 && sw == 1 && ph == 0 && pw == 0;
  const int plan = ksplit_plan(M, Co, K, dense, a16, patch, e.cus);
  if (!plan) return -1;
  const int64_t a_bytes = (int64_t)N_img * H * W * Ci * (a16 ? 2 : 1), b_bytes = (int64_t)Co * K;
  if (Ci % (a16 ? (dense ? 16 : 64) : 16) != 0 || a_bytes >= (1ll << 31) || b_bytes >= (1ll << 31) || a_bytes <= 0 || b_bytes <= 0) return -1;
  // (quotients through multiplication: dividend * divisor < 2^32, the rows of a last tile included)
  if (M >= (1 << 30) || (!dense && ((M + 64) * Wo >= (1ll << 32) || (M + 64) * Ho >= (1ll << 32)))) return -1;
  if (H >= (1 << 20) || W >= (1 << 20) || (int64_t)dh * kh >= (1 << 20) || (int64_t)dw * kw >= (1 << 20)) return -1;
  KsplitParams p = {};
  p.x = x; p.w = (const int8_t *)w;
  p.M = (int)M; p.N = Co; p.K = (int)K;
  p.H = H; p.W = W; p.Ci = Ci; p.Ho = Ho; p.Wo = Wo; p.kh = kh; p.kw = kw; p.ph = ph; p.pw = pw;
  p.sh = sh; p.sw = sw; p.dh = dh; p.dw = dw;
  auto magic = [](unsigned d, unsigned *m, unsigned *mask) {
    *m = d <= 1 ? 0u : (unsigned)(((1ull << 32) + d - 1) / d);
    *mask = d <= 1 ? ~0u : 0u;
  };
  magic(Wo, &p.magic_wo, &p.mask_wo);
  magic(Ho, &p.magic_ho, &p.mask_ho);
  p.m_fastest = b_bytes > a_bytes;
  p.epi = pick_epilogue(Co, e);
  if (p.epi == EPI_SCALAR) {
    p.epi = a16 ? EPI_SCALAR : ragged_epilogue(Co, e);
    if (p.epi == EPI_SCALAR) return -1;
    p.ragged = 1;
  }
  p.a_bytes = (unsigned)a_bytes; p.b_bytes = (unsigned)b_bytes;
  if (a16) return dense ? pick_ksplit<KW_DENSE, true>(plan, p, e, s) : pick_ksplit<KW_TAP, true>(plan, p, e, s);
  return dense ? pick_ksplit<KW_DENSE, false>(plan, p, e, s)
               : (Ci % 64 == 0 ? pick_ksplit<KW_TAP, false>(plan, p, e, s) : pick_ksplit<KW_PIECE, false>(plan, p, e, s));
}

}  // namespace catchq
