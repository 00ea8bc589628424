// Contiguous floating activations [n, c, hw] -> integers by pixels, [n, hw][channel]: a transposition through LDS on the way.
//
// Bound by memory (us before, with a tile of 64 pixels x 64 channels in launch order / now: 5 x 256 x 83 x 94 fp32 -> int8 11.2 / 8.7,
// 5.8 TB/s, fp16 11.6 / 6.3; 24 x 160 x 54 x 59 fp16 14.0 / 7.6; 36 x 15 x 65 x 70 fp32 5.5 / 3.1; digits of 2 x 256 x 73 x 73 fp16,
// 32 scattered loads and four stores a lane, 10.1 / 4.6).  A lane takes PXL consecutive pixels of four channels (a 16-byte load each, where PXL fills one: a wave instruction
// covers 256 consecutive bytes of four planes), packs a pixel's four channels into DW dwords in LDS -- an odd pitch spreads a
// wave's stores over all banks -- and leaves with 16-byte stores that cover the block's channels of a pixel.  A block has CQ groups of four
// channels: 16, 32 or 64 of them, whichever leave fewer lanes beyond the last channel.  The blocks of one
// XCD take consecutive tiles, the channels of a run of pixels first: the lines that two tiles share, at the ends of the planes' runs and
// of the pixels' pieces, then meet in one L2.
// Halfs: eight pixels a lane from a block a unit on.  Images of fewer than four pixels: one.
#pragma once
#include "igemm_common.h"

namespace catchq {

// int8; int16; the digits of 32 channels' int16 values, high bytes and biased low bytes apart (digits_i16.hip)
enum { PX_I8 = 8, PX_I16 = 16, PX_DIGITS = 17 };

struct PixelQuantParams {
  int c, hw;          // channels and pixels of an image as they are
  unsigned ctiles, ptiles, blocks;
  int pitch;          // bytes of a pixel of the output
  int neg_pos;
  float scale;
  int64_t zeros;      // PX_DIGITS: byte offset of the pixel of zeros behind all others
};

template <typename TIn, int OUT, int PXL, int CQ>
__global__ __launch_bounds__(256) void pixel_quantize_kernel(const TIn *__restrict__ x, int8_t *__restrict__ q, PixelQuantParams p) {
  constexpr int DW = OUT == PX_I8 ? 1 : 2;  // dwords of a pixel's four channels
  constexpr int PITCH = CQ * DW + 1, GROUPS = 256 / CQ, PX = GROUPS * PXL;
  __shared__ int tile[PX * PITCH];
  unsigned b = (unsigned)xcd_remap(blockIdx.x, (int)p.blocks);
  const unsigned r = b / p.ctiles, img = r / p.ptiles;
  const int c0 = (int)(b - r * p.ctiles) * (4 * CQ), p0 = (int)(r - img * p.ptiles) * PX;
  const int pg = threadIdx.x % GROUPS, cq = threadIdx.x / GROUPS;
  // the last pixels of an image once more where a lane's run would end behind them, the last channel's plane beyond it: no branches
  const int px = min(p0 + pg * PXL, p.hw - PXL), ch = c0 + cq * 4;
  typedef TIn run __attribute__((ext_vector_type(PXL), aligned(sizeof(TIn))));
  const TIn *const src = x + (int64_t)img * p.c * p.hw + px;
  run v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = *reinterpret_cast<const run *>(src + (int64_t)min(ch + j, p.c - 1) * p.hw);
#pragma unroll
  for (int i = 0; i < PXL; ++i) {
    int b4[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (OUT == PX_DIGITS) b4[j] = quant1_unit<16>((float)v[j][i], p.neg_pos);
      else b4[j] = quant1<OUT>((float)v[j][i], p.scale, p.neg_pos);
      b4[j] = ch + j < p.c ? b4[j] : 0;
    }
    if (px + i < p0) continue;  // (another tile's)
    int *const dst = tile + (px - p0 + i) * PITCH;
    if constexpr (OUT == PX_I8) {
      dst[cq] = (int)(__builtin_amdgcn_perm((unsigned)b4[1], (unsigned)b4[0], 0x0c0c0400u) |
                      __builtin_amdgcn_perm((unsigned)b4[3], (unsigned)b4[2], 0x04000c0cu));
    } else if constexpr (OUT == PX_I16) {
      dst[2 * cq] = (b4[0] & 0xffff) | (b4[1] << 16);
      dst[2 * cq + 1] = (b4[2] & 0xffff) | (b4[3] << 16);
    } else {
      const unsigned hi01 = __builtin_amdgcn_perm((unsigned)b4[1], (unsigned)b4[0], 0x0c0c0501u), lo01 = __builtin_amdgcn_perm((unsigned)b4[1], (unsigned)b4[0], 0x0c0c0400u);
      const unsigned hi23 = __builtin_amdgcn_perm((unsigned)b4[3], (unsigned)b4[2], 0x05010c0cu), lo23 = __builtin_amdgcn_perm((unsigned)b4[3], (unsigned)b4[2], 0x04000c0cu);
      const int at = (cq >> 3) * 16 + (cq & 7);
      dst[at] = (int)(hi01 | hi23);
      dst[at + 8] = (int)((lo01 | lo23) ^ 0x80808080u);
    }
  }
  __syncthreads();
  constexpr int PIECES = CQ * DW / 4;  // 16-byte pieces of a pixel's channels
  const int piece = threadIdx.x % PIECES;
  if (c0 * DW + piece * 16 < p.pitch) {
    int8_t *const out = q + ((int64_t)img * p.hw + p0) * p.pitch + c0 * DW + piece * 16;
#pragma unroll
    for (int k = 0; k < (PX * PIECES + 255) / 256; ++k) {
      const int at = threadIdx.x / PIECES + k * (256 / PIECES);
      if (at >= PX || p0 + at >= p.hw) continue;
      const int *const s = tile + at * PITCH + piece * 4;
      *reinterpret_cast<v4i *>(out + (int64_t)at * p.pitch) = v4i{s[0], s[1], s[2], s[3]};
    }
  }
  if constexpr (OUT == PX_DIGITS) {
    if (b == 0)
      for (int i = threadIdx.x * 16; i < p.pitch; i += 256 * 16) {
        const int low = (i & 32) ? (int)0x80808080u : 0;
        *reinterpret_cast<v4i *>(q + p.zeros + i) = v4i{low, low, low, low};
      }
  }
}

// pitch a multiple of 16 bytes, q on 16 bytes; false: more tiles than a launch has blocks
template <typename TIn, int OUT>
static bool pixel_quantize(const TIn *x, int8_t *q, int64_t n, int c, int64_t hw, int pitch, int pos, float scale, int64_t zeros,
                           hipStream_t s) {
  constexpr int CH = OUT == PX_I8 ? 1 : 2;
  const int channels = pitch / CH, last = channels % 64;
  const int cq = hw < 4 ? 16 : channels <= 16 && OUT != PX_DIGITS ? 4 : last != 0 && last <= 32 ? 8 : 16;
  PixelQuantParams p = {c, (int)hw, (unsigned)((channels + 4 * cq - 1) / (4 * cq)), 0, 0, pitch, -pos, scale, zeros};
  const int groups = 256 / cq;
  auto tiles = [&](int px) { return n * ((hw + px - 1) / px) * p.ctiles; };
  if (hw >= (1ll << 31) - 1024 || tiles(groups) >= (1 << 24)) return false;  // (a launch has less than 2^32 lanes)
  const int pxl = hw < 4 ? 1 : sizeof(TIn) == 2 && hw >= 8 && tiles(groups * 8) >= planned_cus(1) ? 8 : 4;
  p.ptiles = (unsigned)((hw + groups * pxl - 1) / (groups * pxl));
  p.blocks = (unsigned)tiles(groups * pxl);
  if (pxl == 1) {
    pixel_quantize_kernel<TIn, OUT, 1, 16><<<p.blocks, 256, 0, s>>>(x, q, p);
    return true;
  }
  auto launch = [&](auto quads) {
    constexpr int CQ = decltype(quads)::value;
    if constexpr (sizeof(TIn) == 2) {
      if (pxl == 8) {
        pixel_quantize_kernel<TIn, OUT, 8, CQ><<<p.blocks, 256, 0, s>>>(x, q, p);
        return;
      }
    }
    pixel_quantize_kernel<TIn, OUT, 4, CQ><<<p.blocks, 256, 0, s>>>(x, q, p);
  };
  if (cq == 16) launch(std::integral_constant<int, 16>{});
  else if (cq == 8) launch(std::integral_constant<int, 8>{});
  else if constexpr (OUT != PX_DIGITS) launch(std::integral_constant<int, 4>{});
  return true;
}

}  // namespace catchq
