// The first two layers of an inverted-residual block (1x1 expansion -> 3x3 depthwise, both int8 behind ReLU / ReLU6) in one launch.
//
// Run as two launches, the expanded tensor (six times the block's input) goes to memory and comes back, and on the small images of a
// network's later layers each launch is bound by its start-up.  All three layers in one launch (irb_i8.hip) need every hidden channel
// of a pixel in one block: few blocks, and phases that wait for each other.  The depthwise layer needs no other channel than its own, so
// here the hidden channels are split over the blocks: a block has TR output rows of an image, whole, and 32 or 64 hidden channels.
//
//   1  expansion   a wave has 32 hidden channels, whose filters and constants it keeps in registers, and every second or fourth 32
//                  pixels of the band's input rows (with one row of halo on either side), fetched from memory ahead of the matrix
//                  instructions.  Filters are operand A and pixels operand B, so that a lane ends with four consecutive channels of
//                  one pixel: requantized, a dword of the patch in LDS.  Pixels outside the image are zeros there.
//   2  depthwise   a lane has four channels, whose filters and constants were requested before phase 1, x 2 x 4 output pixels: the
//                  stencil of dwconv_i8.hip with the patch as its input.
//
// Every integer is the one that the two launches produce: the same sums, the same float operations in the same order.
//
// What bounds it: the vector arithmetic of the two requantizers and the stencil where the images are many (64 x 112x112, 16 -> 96, stride
// 2: 32 us, of which the instructions' issue is 26), a block's start where they are few.  MobileNetV2's graphs (one part, us, two
// launches / one): one 224 x 224 image 192 / 148, 8 234 / 186, 27 of 192 x 192 269 / 230, 64 of 224 x 224 501 / 387.
#include "dw3x3.h"
#include "igemm_common.h"

namespace catchq {

struct ExpandDwParams {
  int N, H, W, Cin, hid, Ho, Wo;
  int TR, bands;    // output rows of a block (the last band of an image may be shorter), bands of an image
  int chunks, nblocks;
  int PCA;          // columns of the patch as allocated (what the stencil's windows may touch)
  int WG;           // stencil groups in a row of outputs
  unsigned magic_w, mask_w, magic_wg, mask_wg;  // ceil(2^32 / d), mask 0; for d = 1 magic 0, mask ~0
  unsigned w_bytes;
};

constexpr int XDW_NW = 4;  // waves

__device__ __forceinline__ unsigned xdw_div(unsigned n, unsigned magic, unsigned mask) { return __umulhi(n, magic) + (n & mask); }

// KS: input channels / 32, rounded up.  KC: hidden channels of a block / 32.
template <int S, int KS, int KC>
__global__ __launch_bounds__(64 * XDW_NW) void expand_dw_kernel(const int8_t *__restrict__ X, IrbStageDev s1, IrbStageDev s2,
                                                                int8_t *__restrict__ Q, ExpandDwParams p) {
  constexpr int NT = 64 * XDW_NW, QC = KC * 8;
  constexpr int HS = KC * 32 + 4;  // bytes of a patch pixel: an odd number of dwords, 32 pixels of a store fall on 32 banks
  constexpr int NR = Dw3Window<S>::NR, NCL = Dw3Window<S>::NCL;
  constexpr unsigned OOB = 0x80000000u;
  extern __shared__ __attribute__((aligned(16))) int8_t lds[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int frow = lane & 31, fhalf = lane >> 5;
  const int logical = xcd_remap(blockIdx.x, p.nblocks);  // neighbours on a die share input rows and the lines they write
  const int chunk = logical % p.chunks, tile = logical / p.chunks;
  const int img = tile / p.bands, band = tile - img * p.bands;
  const int ho0 = band * p.TR, rows = p.Ho - ho0 < p.TR ? p.Ho - ho0 : p.TR;
  const int hi0 = ho0 * S - 1;  // input row of patch row 0
  const int r0 = hi0 < 0 ? 0 : hi0, end = hi0 + (rows - 1) * S + 3, r1 = end < p.H ? end : p.H;
  const int c0 = chunk * (KC * 32);

  // ---- requests: this wave's filters and first pixels, the constants, the stencil's filters -------------------------------------
  const int cj = wave % KC, cw = c0 + cj * 32;
  const int px_n = (r1 - r0) * p.W;  // (consecutive in memory)
  const int8_t *const x0 = X + ((int64_t)img * p.H + r0) * p.W * p.Cin;
  const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc((void *)x0, 0, px_n * p.Cin, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc((void *)s1.w, 0, (int)p.w_bytes, 0x00020000);
  v4i fw[KS], fx[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {  // (channels beyond Cin or hid: zeros)
    const int k = ks * 32 + fhalf * 16;
    const unsigned off = cw + frow < p.hid && k < p.Cin ? (unsigned)((cw + frow) * p.Cin + k) : OOB;
    fw[ks] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_w, (int)off, 0, 0));
  }
  auto load_x = [&](int sa) {  // (a pixel's channels beyond Cin are the next one's: they meet zeros; pixels beyond the band: zeros)
    const int off = (sa * 32 + frow) * p.Cin + fhalf * 16;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) fx[ks] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_x, off + ks * 32, 0, 0));
  };
  constexpr int STEP = XDW_NW / KC;
  const int first = wave / KC;
  load_x(first);
  v4f dv1[4], rc1[4], bs1[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) {  // (channels that do not exist take others' constants and are not stored)
    const int c = cw + 8 * g + 4 * fhalf, cc = c < p.hid ? c : 0;
    dv1[g] = *reinterpret_cast<const v4f *>(s1.div + cc);
    rc1[g] = *reinterpret_cast<const v4f *>(s1.rcp + cc);
    bs1[g] = *reinterpret_cast<const v4f *>(s1.bias + cc);
  }
  const int q = threadIdx.x % QC, c2 = c0 + q * 4, cc2 = c2 < p.hid ? c2 : 0;
  int wraw[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) wraw[i] = *reinterpret_cast<const int *>(s2.w + (int64_t)cc2 * 9 + 4 * i);
  v4f dv2 = *reinterpret_cast<const v4f *>(s2.div + cc2), rc2 = *reinterpret_cast<const v4f *>(s2.rcp + cc2);
  const v4f bs2 = *reinterpret_cast<const v4f *>(s2.bias + cc2);

  // ---- the depthwise layer's padding: columns -1 and W, and rows -1 and H where the band reaches them -----------------------------
  {
    const int patch_rows = (rows - 1) * S + 3;
    int8_t *const at = lds + q * 4;
    for (int i = (int)threadIdx.x / QC; i < 2 * patch_rows; i += NT / QC)
      *reinterpret_cast<int *>(at + ((i >> 1) * p.PCA + ((i & 1) ? p.W + 1 : 0)) * HS) = 0;
    if (hi0 < 0)
      for (int i = (int)threadIdx.x / QC; i < p.W; i += NT / QC) *reinterpret_cast<int *>(at + (i + 1) * HS) = 0;
    if (end > p.H)
      for (int i = (int)threadIdx.x / QC; i < p.W; i += NT / QC)
        *reinterpret_cast<int *>(at + ((p.H - hi0) * p.PCA + i + 1) * HS) = 0;
  }

  // ---- 1: expansion ---------------------------------------------------------------------------------------------------------------
  const ReluRequant rq1(s1), rq2(s2);
#pragma unroll
  for (int g = 0; g < 4; ++g)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      dv1[g][t] = __builtin_ldexpf(dv1[g][t], -s1.exp2);
      rc1[g][t] = __builtin_ldexpf(rc1[g][t], s1.exp2);
    }
  if (cw < p.hid) {
    const int nsa = (px_n + 31) / 32;
    for (int sa = first; sa < nsa; sa += STEP) {
      v16i acc;
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = 0;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fw[ks], fx[ks], acc, 0, 0, 0);
      load_x(sa + STEP);  // (beyond the band: nothing is read)
      const unsigned m = (unsigned)(sa * 32 + frow);
      const unsigned pr = xdw_div(m, p.magic_w, p.mask_w), wi = m - pr * (unsigned)p.W;
      int8_t *const cell = lds + (((int)pr + r0 - hi0) * p.PCA + (int)wi + 1) * HS + cj * 32 + 4 * fhalf;
      const bool in = (int)m < px_n;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int a[4] = {acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
        const unsigned packed = rq1.four(a, dv1[g], rc1[g], bs1[g]);
        if (in) *reinterpret_cast<unsigned *>(cell + 8 * g) = packed;
      }
    }
  }
  int wa[4][3], wb[4][3];
  dw3_pack(wraw, wa);
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int r = 0; r < 3; ++r) wb[j][r] = (int)((unsigned)wa[j][r] << 8);
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    dv2[t] = __builtin_ldexpf(dv2[t], -s2.exp2);
    rc2[t] = __builtin_ldexpf(rc2[t], s2.exp2);
  }
  __syncthreads();
  if (c2 >= p.hid) return;

  // ---- 2: depthwise ---------------------------------------------------------------------------------------------------------------
  int8_t *const out = Q + ((int64_t)img * p.Ho + ho0) * p.Wo * p.hid + c2;
  const int groups = ((rows + DW3_PH - 1) / DW3_PH) * p.WG;
  for (int t0 = (int)threadIdx.x / QC; t0 < groups; t0 += NT / QC) {
    const int hg = (int)xdw_div((unsigned)t0, p.magic_wg, p.mask_wg), wg = t0 - hg * p.WG;
    int acc[DW3_PH][DW3_PW][4];
    const int8_t *const win = lds + ((hg * DW3_PH * S) * p.PCA + wg * DW3_PW * S) * HS + q * 4;
#pragma unroll
    for (int ri = 0; ri < NR; ++ri) {
      unsigned xr[NCL];
#pragma unroll
      for (int col = 0; col < NCL; ++col) xr[col] = *reinterpret_cast<const unsigned *>(win + (ri * p.PCA + col) * HS);
      dw3_row<S>(ri, xr, wa, wb, acc);
    }
#pragma unroll
    for (int py = 0; py < DW3_PH; ++py) {
      const int ho = hg * DW3_PH + py;
#pragma unroll
      for (int px = 0; px < DW3_PW; ++px) {
        const int wo = wg * DW3_PW + px;
        const unsigned packed = rq2.four(acc[py][px], dv2, rc2, bs2);
        if (ho < rows && wo < p.Wo) *reinterpret_cast<unsigned *>(out + (unsigned)((ho * p.Wo + wo) * p.hid)) = packed;
      }
    }
  }
}

struct ExpandDwPlan {
  ExpandDwParams p;
  int ks, kc, lds;
  int64_t cost;
};

// The plan with `bands` bands of an image and 32 * kc hidden channels a block; false: these are no balanced bands, or too large ones.
static bool expand_dw_tile(int N, int H, int W, int Cin, int hid, int S, int cus, int kc, int bands, ExpandDwPlan *plan) {
  const int Ho = (H - 1) / S + 1, Wo = (W - 1) / S + 1;
  const int chunks = (hid + 32 * kc - 1) / (32 * kc);
  const int tr = (Ho + bands - 1) / bands;
  if ((Ho + tr - 1) / tr != bands) return false;
  const int hg = (tr + 1) / 2, wg = (Wo + 3) / 4, in_rows = (tr - 1) * S + 3;
  // what the stencil's windows touch
  const int rows = S == 1 ? 2 * hg + 2 : 4 * hg + 1, cols = S == 1 ? 4 * wg + 2 : 8 * wg + 2;
  const int pca = cols < W + 2 ? W + 2 : cols;
  const int64_t lds = (int64_t)(rows < in_rows ? in_rows : rows) * pca * (kc * 32 + 4);
  const int64_t blocks = (int64_t)N * bands * chunks;
  if (lds > 64 * 1024 || blocks >= (1 << 24)) return false;  // (a launch has less than 2^32 lanes)
  // Both phases are vector arithmetic: a 32 x 32 piece of the expansion counts as 250 instructions of a wave, 64 lanes' stencils as
  // 600, and a block as 400 more.  The cost is what the busiest unit's SIMDs have to do and, once for every generation of co-resident
  // blocks, a block's start (400) and its own chain.  On 56 shapes (MobileNetV2's at 192 x 192 and 224 x 224, 1 to 64 images) the tile it
  // picks takes 1 % more than the best one on average and 10 % at most.
  const int steps = XDW_NW / kc, pieces = ((in_rows < H ? in_rows : H) * W + 31) / 32, groups = hg * wg * kc * 8;
  const int rounds1 = (pieces + steps - 1) / steps, rounds2 = (groups + 64 * XDW_NW - 1) / (64 * XDW_NW);
  const int64_t fit = 160 * 1024 / lds, resident = fit < 4 ? fit : 4;
  const int64_t per_cu = (blocks + cus - 1) / cus, generations = (per_cu + resident - 1) / resident;
  ExpandDwParams p = {};
  p.N = N; p.H = H; p.W = W; p.Cin = Cin; p.hid = hid; p.Ho = Ho; p.Wo = Wo;
  p.TR = tr; p.bands = bands; p.chunks = chunks; p.nblocks = (int)blocks; p.PCA = pca; p.WG = wg;
  auto magic = [](unsigned d, unsigned *m, unsigned *mask) {  // (dividends and divisors below 2^16)
    *m = d <= 1 ? 0u : (unsigned)(((1ull << 32) + d - 1) / d);
    *mask = d <= 1 ? ~0u : 0u;
  };
  magic(W, &p.magic_w, &p.mask_w);
  magic(wg, &p.magic_wg, &p.mask_wg);
  p.w_bytes = (unsigned)(hid * Cin);
  *plan = {p, (Cin + 31) / 32, kc, (int)lds,
           generations * (400 + 250 * rounds1 + 600 * rounds2) + per_cu * (400 + (250 * pieces * kc + 600 * ((groups + 63) / 64)) / 4)};
  return true;
}

// Band height and hidden channels of a block; false: not this kernel's shape.
static bool expand_dw_plan(int N, int H, int W, int Cin, int hid, int S, int cus, ExpandDwPlan *plan) {
  if (N <= 0 || (S != 1 && S != 2) || Cin % 16 != 0 || Cin > 160 || hid % 16 != 0 || hid <= 0 || H < 2 || W < 2 || W > 256) return false;
  if ((int64_t)hid * Cin >= (1ll << 31) || (int64_t)H * W * Cin >= (1ll << 31) || (int64_t)H * W * hid >= (1ll << 31)) return false;
  bool any = false;
  ExpandDwPlan t;
  for (int kc = 1; kc <= 2; ++kc)
    for (int bands = (H - 1) / S + 1; bands >= 1; --bands)
      if (expand_dw_tile(N, H, W, Cin, hid, S, cus, kc, bands, &t) && (!any || t.cost < plan->cost)) {
        *plan = t;
        any = true;
      }
  return any;
}

bool expand_dw_i8_ok(int N, int H, int W, int Cin, int hid, int S, int cus) {
  ExpandDwPlan plan;
  return expand_dw_plan(N, H, W, Cin, hid, S, cus, &plan);
}

template <int S, int KS>
static int expand_dw_launch(const ExpandDwPlan &l, const void *x, const IrbStageDev &s1, const IrbStageDev &s2, void *q, hipStream_t s) {
  if (l.kc == 1) expand_dw_kernel<S, KS, 1><<<l.p.nblocks, 64 * XDW_NW, l.lds, s>>>((const int8_t *)x, s1, s2, (int8_t *)q, l.p);
  else expand_dw_kernel<S, KS, 2><<<l.p.nblocks, 64 * XDW_NW, l.lds, s>>>((const int8_t *)x, s1, s2, (int8_t *)q, l.p);
  return launch_status();
}

template <int S>
static int expand_dw_launch_s(const ExpandDwPlan &l, const void *x, const IrbStageDev &s1, const IrbStageDev &s2, void *q, hipStream_t s) {
  switch (l.ks) {
    case 1: return expand_dw_launch<S, 1>(l, x, s1, s2, q, s);
    case 2: return expand_dw_launch<S, 2>(l, x, s1, s2, q, s);
    case 3: return expand_dw_launch<S, 3>(l, x, s1, s2, q, s);
    default: return expand_dw_launch<S, 5>(l, x, s1, s2, q, s);
  }
}

// x [N, H, W, Cin] int8; s1.w [hid][Cin]; s2.w [hid][3][3]; q [N, Ho, Wo, hid] int8 (padding 1).  Both stages requantize to int8 behind
// ReLU (relu6 = 0) or ReLU6.  -1: not this kernel's shape.
int expand_dw_i8(const void *x, int N, int H, int W, int Cin, int hid, int S, const IrbStageDev &s1, const IrbStageDev &s2, void *q,
                 int cus, hipStream_t s) {
  ExpandDwPlan plan;
  if (!expand_dw_plan(N, H, W, Cin, hid, S, cus, &plan)) return -1;
  return S == 1 ? expand_dw_launch_s<1>(plan, x, s1, s2, q, s) : expand_dw_launch_s<2>(plan, x, s1, s2, q, s);
}

}  // namespace catchq
