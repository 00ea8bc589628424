// 3x3 depthwise convolution (groups == Ci == Co, dilation 1, stride 1 or 2) on floating activations, int8 or int16, in one launch: the
// quantizer runs where the stencil's input is staged.
//
// Bound by memory: an activation read once, an output written once.  As two launches the quantized activations go through memory in
// between, and channel counts that are no multiple of four, or 16 bits, had one thread for an output in the direct kernel.
//
// Device time, us, before (quantizer + stencil, the direct kernel where marked) / now: 16 x 56 x 56, 96 channels, fp32 8 bits 15.7 / 11.4,
// 16 bits (direct) 83 / 16.3; 91 channels 8 bits (direct) 71 / 12.9, halfs in planes 75 / 13.6; 64 x 56 x 56, 256 channels, 410 MB of
// activations, 87.7 (4.7 TB/s).  Whole calls: every one of 150 drawn layers is faster, 1.06 to 5.2 times (they are one launch).
//
// A block owns 32 channels of a tile of TH x TW output pixels of one image:
//   1  stage    the input pixels of the tile are read (channels-last: eight lanes a pixel, four channels each; planes: 64 lanes along a
//               row, two pixels of four planes each), quantized and stored as [pixel][channel] in LDS, the padding as zeros.  The pixel's stride
//               is odd in units of four channels, so that a wave's stores and reads go over all banks.
//   2  stencil  a lane owns four channels of PH x PW outputs.  8 bits: dw3x3.h.  16 bits: nine products of up to 2^30 do not fit 32 bits,
//               and 64-bit integer products are a quarter of the rate of doubles, which hold the sum exactly.  It starts at +0.0: a sum
//               of zeros under negative filters is the integer's +0.0.
// Channels beyond the last group of four: the group is read from where it lies whole and shifted, outputs are stored one by one.
#include "dw3x3.h"
#include "igemm_common.h"

namespace catchq {

struct DwFloatParams {
  int N, H, W, C, ph, pw, Ho, Wo;
  int TH, TW;                 // output tile
  int PR, PC;                 // input tile
  unsigned magic;             // ceil(2^20 / PC)
  int strips, bands, slabs;   // tiles of a row, of an image, groups of 32 channels
  unsigned blocks;
  int nchw, neg_pos;
};

constexpr int DWF_CH = 32;  // channels of a block
constexpr int dwf_pixel(int bits) { return (DWF_CH + 4) * bits / 8; }  // bytes of a pixel in LDS

template <bool HALF>
struct DwfFour {  // four activations as they lie in memory
  v4f v;
  __device__ __forceinline__ void load(const void *x, int64_t at) {
    if constexpr (HALF) {
      typedef _Float16 f16x4 __attribute__((ext_vector_type(4), aligned(2)));
      v = __builtin_convertvector(*reinterpret_cast<const f16x4 *>(reinterpret_cast<const _Float16 *>(x) + at), v4f);
    } else {
      typedef float f32x4 __attribute__((ext_vector_type(4), aligned(4)));
      v = *reinterpret_cast<const f32x4 *>(reinterpret_cast<const float *>(x) + at);
    }
  }
};

// four quantized channels into LDS, the first `skip` of them left out (they belong to the group before)
template <int BITS>
__device__ __forceinline__ void dwf_store(char *dst, const v4f v, int neg_pos, int skip) {
  int q[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) q[t] = quant1_unit<BITS>(v[t], neg_pos);
  if constexpr (BITS == 8) {
    const unsigned lo = __builtin_amdgcn_perm((unsigned)q[1], (unsigned)q[0], 0x0c0c0400u);
    const unsigned hi = __builtin_amdgcn_perm((unsigned)q[3], (unsigned)q[2], 0x04000c0cu);
    *reinterpret_cast<unsigned *>(dst) = (lo | hi) >> (8 * skip);
  } else {
    const unsigned lo = __builtin_amdgcn_perm((unsigned)q[1], (unsigned)q[0], 0x05040100u);
    const unsigned hi = __builtin_amdgcn_perm((unsigned)q[3], (unsigned)q[2], 0x05040100u);
    *reinterpret_cast<uint64_t *>(dst) = (((uint64_t)hi << 32) | lo) >> (16 * skip);
  }
}

template <bool HALF, int BITS, int S, int EPI>
__global__ __launch_bounds__(256) void dw_float_kernel(const void *__restrict__ x, const void *__restrict__ w, DwFloatParams p, EpiDev e) {
  resolve_exp2(e);
  extern __shared__ __attribute__((aligned(16))) char dwf_lds[];
  typedef typename EpiOf<EPI>::type Sp;
  constexpr int PIXEL = dwf_pixel(BITS), QUAD = BITS / 2;
  constexpr int PH = DW3_PH, PW = BITS == 8 ? DW3_PW : 2;

  // blocks of one XCD (id % 8) take consecutive tiles: neighbours read the same rows
  unsigned b = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (b >= p.blocks) return;
  const int slab = (int)(b % (unsigned)p.slabs);
  b /= (unsigned)p.slabs;
  const int strip = (int)(b % (unsigned)p.strips);
  b /= (unsigned)p.strips;
  const int band = (int)(b % (unsigned)p.bands), img = (int)(b / (unsigned)p.bands);
  const int c0 = slab * DWF_CH, ho_b = band * p.TH, wo_b = strip * p.TW;
  const int hi0 = ho_b * S - p.ph, wi0 = wo_b * S - p.pw;
  const int npix = p.PR * p.PC;

  // ---- the lane's filters and constants: requested first ---------------------------------------------------------------------
  const int quad = threadIdx.x & 7, c = c0 + quad * 4;
  const bool have = c < p.C;
  int wraw[BITS == 8 ? 9 : 18];
#pragma unroll
  for (int i = 0; i < (BITS == 8 ? 9 : 18); ++i) wraw[i] = 0;
  if (c + 4 <= p.C) {
    const char *at = (const char *)w + (int64_t)c * (9 * BITS / 8);
    typedef int dword __attribute__((aligned(1)));
#pragma unroll
    for (int i = 0; i < (BITS == 8 ? 9 : 18); ++i) wraw[i] = *reinterpret_cast<const dword *>(at + 4 * i);
  } else if (have) {
#pragma unroll
    for (int i = 0; i < 27; ++i) {  // (at most three channels)
      if (i >= (p.C - c) * 9) break;
      if constexpr (BITS == 8) wraw[i >> 2] |= (int)((unsigned)reinterpret_cast<const uint8_t *>(w)[(int64_t)c * 9 + i] << (8 * (i & 3)));
      else wraw[i >> 1] |= (int)((unsigned)reinterpret_cast<const uint16_t *>(w)[(int64_t)c * 9 + i] << (16 * (i & 1)));
    }
  }
  const EpiLane L = epi_lane_setup_ragged<Sp>(have ? c : 0, p.C, e);

  // ---- 1: stage ---------------------------------------------------------------------------------------------------------------
  constexpr int U = 6;  // loads on their way at once
  if (!p.nchw) {
    const int cl = min(c, p.C - 4), skip = have ? c - cl : 0;
    const int64_t img_at = (int64_t)img * p.H * p.W * p.C + cl;
    for (int first = (int)threadIdx.x >> 3; first < npix; first += 32 * U) {
      DwfFour<HALF> v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const unsigned pix = (unsigned)(first + 32 * u), row = (pix * p.magic) >> 20;
        const int hi = hi0 + (int)row, wi = wi0 + (int)(pix - row * (unsigned)p.PC);
        v[u].v = v4f{0.f, 0.f, 0.f, 0.f};
        if (have && (int)row < p.PR && (unsigned)hi < (unsigned)p.H && (unsigned)wi < (unsigned)p.W)
          v[u].load(x, img_at + (int64_t)(hi * p.W + wi) * p.C);
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (have && first + 32 * u < npix) dwf_store<BITS>(dwf_lds + (first + 32 * u) * PIXEL + quad * QUAD, v[u].v, p.neg_pos, skip);
    }
  } else {
    // two pixels of a row at once (the input tile has an even number of columns), of which the padding may hold one: the load then
    // takes the pair beside it
    typedef typename std::conditional<HALF, _Float16, float>::type T;
    typedef T pair_t __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    constexpr int UP = 4;
    const T *const xt = reinterpret_cast<const T *>(x);
    const int lane = threadIdx.x & 63, plane = p.H * p.W;
    for (int qd = (int)threadIdx.x >> 6; qd < 8 && c0 + qd * 4 < p.C; qd += 4) {
      const int64_t img_at = ((int64_t)img * p.C + c0 + qd * 4) * plane;
      const int last = p.C - 1 - (c0 + qd * 4);  // planes beyond the last channel: its own again
      for (int first = lane; 2 * first < npix; first += 64 * UP) {
        v4f a[UP], b2[UP];
#pragma unroll
        for (int u = 0; u < UP; ++u) {
          const unsigned pix = 2u * (unsigned)(first + 64 * u), row = (pix * p.magic) >> 20;
          const int hi = hi0 + (int)row, wi = wi0 + (int)(pix - row * (unsigned)p.PC);
          a[u] = v4f{0.f, 0.f, 0.f, 0.f};
          b2[u] = a[u];
          if ((int)row < p.PR && (unsigned)hi < (unsigned)p.H && wi >= -1 && wi < p.W) {
            const int at = hi * p.W + min(max(wi, 0), p.W - 2);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              const pair_t v = *reinterpret_cast<const pair_t *>(xt + img_at + (int64_t)min(t, last) * plane + at);
              a[u][t] = wi < 0 ? 0.f : (float)(wi > p.W - 2 ? v[1] : v[0]);
              b2[u][t] = wi > p.W - 2 ? 0.f : (float)(wi < 0 ? v[0] : v[1]);
            }
          }
        }
#pragma unroll
        for (int u = 0; u < UP; ++u)
          if (2 * (first + 64 * u) < npix) {
            char *const at = dwf_lds + 2 * (first + 64 * u) * PIXEL + qd * QUAD;
            dwf_store<BITS>(at, a[u], p.neg_pos, 0);
            dwf_store<BITS>(at + PIXEL, b2[u], p.neg_pos, 0);
          }
      }
    }
  }
  __syncthreads();
  if (!have) return;

  // ---- 2: stencil -------------------------------------------------------------------------------------------------------------
  const int groups = p.TW / PW, items = p.TH / PH * groups;
  const int64_t img_out = (int64_t)img * p.Ho * p.Wo;
  auto finish = [&](int py, int px, int ho0, int wo0, const auto &sums) {
    const int ho = ho0 + py, wo = wo0 + px;
    if (ho >= p.Ho || wo >= p.Wo) return;
    epi_vec4<Sp>(sums, v4f{0.f, 0.f, 0.f, 0.f}, L, EpiAtRagged{(img_out + ho * p.Wo + wo) * p.C + c, p.C - c}, e);
  };
  if constexpr (BITS == 8) {
    int wa[4][3], wb[4][3];
    dw3_pack(wraw, wa);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 3; ++r) wb[j][r] = (int)((unsigned)wa[j][r] << 8);
    for (int item = (int)threadIdx.x >> 3; item < items; item += 32) {
      const int hg = item / groups, wg = item - hg * groups;
      if (ho_b + hg * PH >= p.Ho || wo_b + wg * PW >= p.Wo) continue;
      const char *at = dwf_lds + (hg * PH * S * p.PC + wg * PW * S) * PIXEL + quad * QUAD;
      int acc[PH][PW][4];
#pragma unroll
      for (int ri = 0; ri < Dw3Window<S>::NR; ++ri) {
        unsigned xr[Dw3Window<S>::NCL];
#pragma unroll
        for (int col = 0; col < Dw3Window<S>::NCL; ++col) xr[col] = *reinterpret_cast<const unsigned *>(at + (ri * p.PC + col) * PIXEL);
        dw3_row<S>(ri, xr, wa, wb, acc);
      }
#pragma unroll
      for (int py = 0; py < PH; ++py)
#pragma unroll
        for (int px = 0; px < PW; ++px)
          finish(py, px, ho_b + hg * PH, wo_b + wg * PW, v4i{acc[py][px][0], acc[py][px][1], acc[py][px][2], acc[py][px][3]});
    }
  } else {
    double wd[9][4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int t = 0; t < 9; ++t) wd[t][j] = (double)(int)(int16_t)(wraw[(j * 9 + t) >> 1] >> (16 * ((j * 9 + t) & 1)));
    constexpr int NR = (PH - 1) * S + 3, NC = (PW - 1) * S + 3;
    for (int item = (int)threadIdx.x >> 3; item < items; item += 32) {
      const int hg = item / groups, wg = item - hg * groups;
      if (ho_b + hg * PH >= p.Ho || wo_b + wg * PW >= p.Wo) continue;
      const char *at = dwf_lds + (hg * PH * S * p.PC + wg * PW * S) * PIXEL + quad * QUAD;
      double acc[PH][PW][4];
#pragma unroll
      for (int ri = 0; ri < NR; ++ri)
#pragma unroll
        for (int col = 0; col < NC; ++col) {
          const v2i raw = *reinterpret_cast<const v2i *>(at + (ri * p.PC + col) * PIXEL);
          const double xv[4] = {(double)(int)(int16_t)raw[0], (double)(raw[0] >> 16), (double)(int)(int16_t)raw[1], (double)(raw[1] >> 16)};
#pragma unroll
          for (int py = 0; py < PH; ++py)
#pragma unroll
            for (int px = 0; px < PW; ++px) {
              const int r = ri - py * S, q = col - px * S;
              if (r < 0 || r > 2 || q < 0 || q > 2) continue;
#pragma unroll
              for (int j = 0; j < 4; ++j)
                acc[py][px][j] = __builtin_fma(xv[j], wd[r * 3 + q][j], r == 0 && q == 0 ? 0.0 : acc[py][px][j]);  // (0 x -1 + 0: +0)
            }
        }
#pragma unroll
      for (int py = 0; py < PH; ++py)
#pragma unroll
        for (int px = 0; px < PW; ++px)  // (one rounding to fp32: the integer's)
          finish(py, px, ho_b + hg * PH, wo_b + wg * PW,
                 v4f{(float)acc[py][px][0], (float)acc[py][px][1], (float)acc[py][px][2], (float)acc[py][px][3]});
    }
  }
}

// The tile: a row of up to 64 outputs; rows of input that two tiles read are read twice, so as many rows as the outputs below (8 bits,
// 16 x 56 x 56, 96 channels: 128 outputs 14.2 us, 256 11.5; 64 x 56 x 56, 256: 128 outputs 106-122 us, 256 90, 512 88; 16 bits 128 outputs
// 19.0, 256 16.4; stride 2 stages four times the pixels, 128 and 256 tie), fewer while there are not two blocks for a unit.
static void dwf_tile(DwFloatParams &p, int bits, int s, int cus) {
  p.slabs = (p.C + DWF_CH - 1) / DWF_CH;
  p.strips = (p.Wo + 63) / 64;
  p.TW = ((p.Wo + p.strips - 1) / p.strips + 3) / 4 * 4;
  p.strips = (p.Wo + p.TW - 1) / p.TW;
  const int rows = (p.Ho + 1) / 2 * 2;
  int pixels = s == 2 ? 128 : bits == 8 ? 512 : 256;
  for (;; pixels /= 2) {
    p.TH = std::min(std::max(pixels / p.TW / 2 * 2, 2), rows);
    p.bands = (p.Ho + p.TH - 1) / p.TH;
    if (p.TH == 2 || (int64_t)p.N * p.bands * p.strips * p.slabs >= 2 * (int64_t)cus) break;
  }
  p.PR = s == 1 ? p.TH + 2 : 2 * p.TH + 1;
  p.PC = s == 1 ? p.TW + 2 : 2 * p.TW + 2;
  p.magic = ((1u << 20) + (unsigned)p.PC - 1) / (unsigned)p.PC;
}

template <bool HALF, int BITS, int S, int EPI>
static void dwf_launch(const void *x, const void *w, const DwFloatParams &p, const EpiDev &e, hipStream_t s) {
  const unsigned grid = (p.blocks + 7) / 8 * 8;
  dw_float_kernel<HALF, BITS, S, EPI><<<grid, 256, p.PR * p.PC * dwf_pixel(BITS), s>>>(x, w, p, e);
}

// CATCHQ_ERR_UNSUPPORTED: not this kernel's layer
int dw_float(const void *x, bool half, int position, bool nchw, const void *w, int bits, int N, int H, int W, int C, int ph, int pw,
             int stride, int Ho, int Wo, const EpiDev &e, hipStream_t s) {
  if (C < 4 || (nchw && W < 2) || (int64_t)H * W * C >= (1ll << 31) || (int64_t)Ho * Wo * C >= (1ll << 31)) return CATCHQ_ERR_UNSUPPORTED;
  const int epi = ragged_epilogue(C, e, true);
  if ((epi != EPI_Y32 || half) && ((epi != EPI_Y16 && epi != EPI_Y16_STEPS) || !half)) return CATCHQ_ERR_UNSUPPORTED;
  DwFloatParams p = {};
  p.N = N; p.H = H; p.W = W; p.C = C; p.ph = ph; p.pw = pw; p.Ho = Ho; p.Wo = Wo; p.nchw = nchw; p.neg_pos = -position;
  dwf_tile(p, bits, stride, e.cus);
  const int64_t blocks = (int64_t)N * p.bands * p.strips * p.slabs;
  if (blocks >= (1 << 24)) return CATCHQ_ERR_UNSUPPORTED;  // (a launch has less than 2^32 lanes)
  p.blocks = (unsigned)blocks;
#define CATCHQ_DWF(H_, E_)                                                                                            \
  if (bits == 8) stride == 1 ? dwf_launch<H_, 8, 1, E_>(x, w, p, e, s) : dwf_launch<H_, 8, 2, E_>(x, w, p, e, s);     \
  else stride == 1 ? dwf_launch<H_, 16, 1, E_>(x, w, p, e, s) : dwf_launch<H_, 16, 2, E_>(x, w, p, e, s);
  if (epi == EPI_Y32) {
    CATCHQ_DWF(false, EPI_Y32)
  } else if (epi == EPI_Y16) {
    CATCHQ_DWF(true, EPI_Y16)
  } else {
    CATCHQ_DWF(true, EPI_Y16_STEPS)
  }
#undef CATCHQ_DWF
  return launch_status();
}

}  // namespace catchq
