// The last 1x1 convolution of an image classifier and the global average pooling behind it in one launch.
//
// Run layer by layer the convolution writes its fp32 output (ResNet-50: 7 x 7 x 2048 floats per image, the largest
// tensor of the last stage) and the pooling reads it back to keep one value per channel -- two launches whose time
// is their start-up and the round trip of that tensor.  Here a block owns one image and 64 to 256 channels, a wave 32
// of them and all pixels of the image or one of its two groups of 32:
//
//   1  the block's filter rows and the image's pixels (at most 64, int8) travel from global memory straight into
//      LDS (buffer_load ... lds, 16 bytes per lane, whole cache lines per instruction), K in chunks of at most 512
//      bytes; a row's 16-byte pieces are stored XOR-swizzled so that the fragment reads of 16 rows fall into 16
//      different pieces of an LDS line.  (Filter fragments fetched by the lanes themselves, 16 bytes per lane at a
//      stride of K bytes, cost one cache-line request per lane and made this kernel twice as slow.)
//   2  every wave multiplies on the matrix cores with the operands swapped (filters as A, pixels as B), so that a
//      lane ends up with four consecutive channels of one pixel; the integer sums go to the wave's tile in LDS;
//   3  the lanes take the tile row-wise -- eight lanes a pixel, four channels each, so that the fp32 residual is read
//      in whole cache lines -- and apply the convolution's epilogue (reciprocal-form division, bias, residual,
//      activation): the arithmetic of the stand-alone launch, value for value;
//   4  one lane per channel adds the pixels up in storage order, one fp32 addition each, divides once by the pixel
//      count and stores the mean and / or its quantized form -- the arithmetic of the stand-alone pooling kernel.
//
// The convolution's output never reaches memory; mean and quantized mean are those of the two launches bit for bit.
#include "igemm_i8_dma.inc"

namespace catchq {

struct GapConvDev {
  const float *div, *rcp, *bias, *resid;
  int exp2, act;
  float *mean;  // [N, Co] or null
  void *q;      // [N, Co] int8 / int16 or null
  int q_bw, q_neg_pos;
  float q_scale;
};

struct GapConvParams {
  int N, HW, K, Co;
  int KC;      // bytes of K per pass through LDS: a divisor of K, a multiple of 32, at most 512
  int sw;      // swizzle mask: (largest power of two that divides KC / 16, at most 16) - 1
  int groups;  // 32-pixel groups: 1 or 2
  int off_x;   // LDS offset of the pixels (behind the filter rows)
  unsigned magic;  // ceil(2^32 / (KC / 16))
};

constexpr int GC_YP = 36;  // dwords per pixel row of a wave's output tile

// NW waves, PG of them (one for each 32 pixels) to 32 channels
template <int NW, int PG, bool RES>
__global__ __launch_bounds__(64 * NW) void conv1x1_gap_kernel(const int8_t *__restrict__ X, const int8_t *__restrict__ Wt,
                                                             GapConvDev e, GapConvParams p) {
  fetch_arguments<16 + sizeof(GapConvDev) + sizeof(GapConvParams)>();
  extern __shared__ __attribute__((aligned(1024))) int8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int frow = lane & 31, fhalf = lane >> 5;
  const int img = blockIdx.x;
  constexpr int TILES = NW / PG, G = 2 / PG;  // groups of 32 channels, groups of 32 pixels of a wave
  constexpr int EP = 8 / PG;             // rounds of the epilogue: eight pixels each
  const int cb = blockIdx.y * TILES * 32;  // the block's first channel
  const int tile = wave / PG, pg = PG > 1 ? wave % PG : 0;
  const int c_own = cb + tile * 32;      // this wave's
  const bool live = c_own < p.Co;        // wave-uniform; rows past the last channel are zero-filled by the loads
  const int chw = p.KC >> 4;             // 16-byte pieces per row of a pass
  const int w_rows = TILES * 32;

  // epilogue operands in the row-wise layout: lane -> (pixel 32 pg + lane / 8 + 8 j, channels c_own + 4 (lane % 8) .. + 3)
  const int cc = lane & 7, pp = pg * 32 + (lane >> 3);
  const int ch_e = (live ? c_own : 0) + 4 * cc;
  v4f dv = *reinterpret_cast<const v4f *>(e.div + ch_e), rc = *reinterpret_cast<const v4f *>(e.rcp + ch_e);
  const v4f bs = *reinterpret_cast<const v4f *>(e.bias + ch_e);
  v4f res[EP];
#pragma unroll
  for (int j = 0; j < EP; ++j) {
    res[j] = v4f{0.f, 0.f, 0.f, 0.f};
    const int px = pp + 8 * j < p.HW ? pp + 8 * j : p.HW - 1;  // rows past the image repeat its last pixel
    if constexpr (RES) res[j] = __builtin_nontemporal_load(reinterpret_cast<const v4f *>(e.resid + ((int64_t)img * p.HW + px) * p.Co + ch_e));
  }

  const __amdgpu_buffer_rsrc_t rsrc_w =
      __builtin_amdgcn_make_buffer_rsrc((void *)(Wt + (int64_t)cb * p.K), 0, (int)((int64_t)(p.Co - cb) * p.K < (1 << 30) ? (int64_t)(p.Co - cb) * p.K : (1 << 30)), 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_x =
      __builtin_amdgcn_make_buffer_rsrc((void *)(X + (int64_t)img * p.HW * p.K), 0, p.HW * p.K, 0x00020000);
  const int w_instr = w_rows * chw / 64;            // DMA instructions of a pass: filter rows ...
  const int x_instr = (p.HW * chw + 63) / 64;       // ... and pixels
  const int8_t *arow = lds + (tile * 32 + frow) * p.KC;
  const int a_key = frow & p.sw;
  const int8_t *xrow[G];
  int x_key[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int at = (pg + g) * 32 + frow, px = at < p.HW ? at : p.HW - 1;  // lanes past the image repeat its last pixel
    xrow[g] = lds + p.off_x + px * p.KC;
    x_key[g] = px & p.sw;
  }
  v16i acc[G];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[g][r] = 0;

  for (int k0 = 0; k0 < p.K; k0 += p.KC) {
    if (k0 > 0) __syncthreads();  // the previous pass has been read
    // ---- 1: this pass of the filter rows and the pixels, straight into LDS ---------------------------------------------
    for (int b = wave; b < w_instr + x_instr; b += NW) {  // wave-uniform
      const bool is_w = b < w_instr;
      const int g = (is_w ? b : b - w_instr) * 64 + lane;  // piece index within the slab = LDS position
      const int row = (int)__umulhi((unsigned)g, p.magic), slot = g - row * chw;
      const int piece = slot ^ (row & p.sw);               // the swizzle is applied on the source side
      const int rows = is_w ? w_rows : p.HW;
      const unsigned voff = row < rows ? (unsigned)(row * p.K + k0 + piece * 16) : 0x80000000u;  // out of range: zeros
      lds_ptr_t dst = (lds_ptr_t)(lds + (is_w ? 0 : p.off_x) + (is_w ? b : b - w_instr) * 1024);
      if (is_w) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_w, dst, 16, (int)voff, 0, 0, 0);
      else __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_x, dst, 16, (int)voff, 0, 0, 0);
    }
    CATCHQ_VMCNT(0);  // this wave's transfers have landed; the barrier makes that true of every wave's
    __syncthreads();
    // ---- 2: the convolution over this pass -----------------------------------------------------------------------------
    const int steps = p.KC >> 5;
    v4i fa = *reinterpret_cast<const v4i *>(arow + ((fhalf ^ a_key) << 4));
    v4i fb[G];
#pragma unroll
    for (int g = 0; g < G; ++g) fb[g] = *reinterpret_cast<const v4i *>(xrow[g] + ((fhalf ^ x_key[g]) << 4));
    for (int s = 0; s < steps; ++s) {
      const v4i a = fa;
      v4i b[G];
      const int cn = (s + 1 < steps ? s + 1 : s) * 2 + fhalf;  // fragments one step ahead of the matrix instructions
      fa = *reinterpret_cast<const v4i *>(arow + ((cn ^ a_key) << 4));
#pragma unroll
      for (int g = 0; g < G; ++g) {
        b[g] = fb[g];
        fb[g] = *reinterpret_cast<const v4i *>(xrow[g] + ((cn ^ x_key[g]) << 4));
      }
#pragma unroll
      for (int g = 0; g < G; ++g)
        if (g == 0 || p.groups > 1) acc[g] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b[g], acc[g], 0, 0, 0);
    }
  }
  __syncthreads();  // every wave is done with the operands: the output tiles overlay them

  // ---- 3: the sums into the wave's tile, the epilogue row-wise -----------------------------------------------------------
  int *yt = reinterpret_cast<int *>(lds) + tile * (p.HW * GC_YP);
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int px = (pg + g) * 32 + frow;
    if (px < p.HW) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<v4i *>(yt + px * GC_YP + 8 * i + 4 * fhalf) =
            v4i{acc[g][4 * i], acc[g][4 * i + 1], acc[g][4 * i + 2], acc[g][4 * i + 3]};
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 4; ++j) {  // the power of two folded into the reciprocal form
    dv[j] = __builtin_ldexpf(dv[j], -e.exp2);
    rc[j] = __builtin_ldexpf(rc[j], e.exp2);
  }
#pragma unroll
  for (int j = 0; j < EP; ++j) {
    const int px = pp + 8 * j;
    if (px < p.HW) {
      int *cell = yt + px * GC_YP + 4 * cc;
      const v4i a = *reinterpret_cast<const v4i *>(cell);
      v4f y;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        float v = div_by_rcp((float)a[t], dv[t], rc[t]) + bs[t];
        if constexpr (RES) v = v + res[j][t];
        if (e.act >= CATCHQ_ACT_RELU) v = (v > 0.0f) ? v : 0.0f;
        if (e.act == CATCHQ_ACT_RELU6) v = (v < 6.0f) ? v : 6.0f;
        y[t] = v;
      }
      *reinterpret_cast<v4f *>(cell) = y;
    }
  }
  __syncthreads();
  // ---- 4: the ordered sum over the pixels ----------------------------------------------------------------------------------
  if (live && pg == 0 && lane < 32) {
    const float *yf = reinterpret_cast<const float *>(yt);
    // in storage order, one addition per pixel: the order is part of the result; eight reads are requested at a time
    float s = 0.0f;
    int px = 0;
    for (; px + 8 <= p.HW; px += 8) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = yf[(px + u) * GC_YP + lane];
#pragma unroll
      for (int u = 0; u < 8; ++u) s = s + v[u];
    }
    for (; px < p.HW; ++px) s = s + yf[px * GC_YP + lane];
    const float mean = s / (float)p.HW;
    const int64_t idx = (int64_t)img * p.Co + c_own + lane;
    if (e.mean) e.mean[idx] = mean;
    if (e.q) {
      if (e.q_bw == 8) reinterpret_cast<int8_t *>(e.q)[idx] = (int8_t)quant1<8>(mean, e.q_scale, e.q_neg_pos);
      else reinterpret_cast<int16_t *>(e.q)[idx] = (int16_t)quant1<16>(mean, e.q_scale, e.q_neg_pos);
    }
  }
}

// waves per block, waves per 32 channels, bytes of K per pass and LDS bytes; false: not this kernel's shape (images of at most 64
// pixels, K a multiple of 32, Co a multiple of 32)
static bool gap_plan(int N, int HW, int K, int Co, bool resid, int &nw, int &pg, GapConvParams &p, int &lds_bytes) {
  if (!(N > 0 && HW >= 1 && HW <= 64 && K >= 32 && K % 32 == 0 && K <= 8192 && Co >= 32 && Co % 32 == 0 &&
        (int64_t)N * HW * K < (1ll << 31) && (int64_t)N * HW * Co < (1ll << 31) && (int64_t)Co * K < (1ll << 30)))
    return false;
  // Images of two groups of pixels: a wave for each, so that a wave's matrix instructions and epilogue are halved, 64 channels a block
  // while every block has a unit to itself and 128 while those do; beyond, 64 channels and, with a residual (and the longer K that
  // such layers have: fewer reads of the pixels), 256 with both groups in a wave.  us, 49 pixels, images of 320 -> 1280 / of 512 -> 2048
  // with a residual, four waves of 32 channels each (eight from 256 blocks on), as it was, / now: one image 9.0 / 5.0 and 11.8 / 5.9,
  // 16 8.9 / 5.5 and 12.6 / 6.3, 27 9.4 / 6.4 and 10.3 / 9.1, 64 10.8 / 8.2 and 15.8 / 15.1.  Images of one group: 256 channels, also where
  // that leaves units without a block (16 pixels, 128 channels there, as it was, / 256: one image 6.0 / 5.3 and 8.0 / 6.7, 16 6.3 / 5.5 and
  // 8.5 / 7.0, 31 7.0 / 5.6 and 9.6 / 7.2; 25 pixels, one 6.5 / 5.8 and 8.8 / 7.1; this kernel's other changes among them).
  p = GapConvParams{};
  p.N = N; p.HW = HW; p.K = K; p.Co = Co;
  p.groups = (HW + 31) / 32;
  auto blocks = [&](int channels) { return (int64_t)N * ((Co + channels - 1) / channels); };
  nw = 8; pg = 1;
  if (p.groups == 2) {
    if (blocks(64) <= 256 || (blocks(128) > 256 && !resid)) { nw = 4; pg = 2; }
    else if (blocks(128) <= 256) pg = 2;
  }
  const int channels = nw / pg * 32;
  // K in passes of at most 512 bytes; of at most 256 where the launch has more blocks than the device has compute
  // units, so that two blocks share a unit and one's transfers run under the other's arithmetic (64 images: 9.5 -> 8.2 and
  // 18.3 -> 15.1 us; with one block per unit the second pass costs 0.2 to 0.3 us instead)
  const int dmax = blocks(channels) > 256 ? 8 : 16;
  for (int d = dmax; d >= 1; --d)
    if ((K / 32) % d == 0) { p.KC = 32 * d; break; }
  p.magic = (unsigned)(((1ull << 32) + p.KC / 16 - 1) / (p.KC / 16));  // (pieces of a pass: below 2^16)
  int sw = 1;
  while (sw < 16 && (p.KC / 16) % (2 * sw) == 0) sw *= 2;
  p.sw = sw - 1;
  p.off_x = channels * p.KC;
  const int x_bytes = (HW * (p.KC / 16) + 63) / 64 * 1024;  // whole DMA instructions
  const int operands = p.off_x + x_bytes, tiles = nw / pg * HW * GC_YP * 4;
  lds_bytes = ((operands > tiles ? operands : tiles) + 255) / 256 * 256;
  return lds_bytes <= 160 * 1024;
}

bool conv1x1_gap_i8_ok(int N, int HW, int K, int Co) {
  int nw, pg, lds;
  GapConvParams p;
  return gap_plan(N, HW, K, Co, false, nw, pg, p, lds) && gap_plan(N, HW, K, Co, true, nw, pg, p, lds);
}

template <int NW, int PG, bool RES>
static int launch_gap(const void *x, const void *w, const GapConvDev &e, const GapConvParams &p, int lds_bytes, hipStream_t st) {
  auto kern = conv1x1_gap_kernel<NW, PG, RES>;
  if (lds_bytes > 64 * 1024) {
    static std::atomic<bool> raised[64];
    if (raise_lds_limit((const void *)kern, 160 * 1024, raised) != CATCHQ_OK) return CATCHQ_ERR_LAUNCH;
  }
  constexpr int channels = NW / PG * 32;
  kern<<<dim3(p.N, (p.Co + channels - 1) / channels), 64 * NW, lds_bytes, st>>>((const int8_t *)x, (const int8_t *)w, e, p);
  return launch_status();
}

// x [N, HW, K] int8, w [Co, K] int8; mean / q [N, Co].  -1: not this kernel's shape.
int conv1x1_gap_i8(const void *x, const void *w, int N, int HW, int K, int Co, const GapConvDev &e, hipStream_t st) {
  int nw, pg, lds_bytes;
  GapConvParams p;
  if (!gap_plan(N, HW, K, Co, e.resid != nullptr, nw, pg, p, lds_bytes)) return -1;
  if (pg == 1) return e.resid ? launch_gap<8, 1, true>(x, w, e, p, lds_bytes, st) : launch_gap<8, 1, false>(x, w, e, p, lds_bytes, st);
  if (nw == 8) return e.resid ? launch_gap<8, 2, true>(x, w, e, p, lds_bytes, st) : launch_gap<8, 2, false>(x, w, e, p, lds_bytes, st);
  return e.resid ? launch_gap<4, 2, true>(x, w, e, p, lds_bytes, st) : launch_gap<4, 2, false>(x, w, e, p, lds_bytes, st);
}

}  // namespace catchq
