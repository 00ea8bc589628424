// Pieces of the 3x3 depthwise stencil that the stand-alone kernel (dwconv_i8.hip), the one-launch inverted-residual block
// (irb_i8.hip) and the expansion + stencil (expand_dw_i8.hip) share.  A lane owns four channels x 2 rows x 4 columns of outputs.
//
// The sums run on v_dot4_i32_i8, which adds four byte products: the four bytes of an operand must be four taps of ONE channel.  A
// pixel's dword holds four channels, so groups of four horizontally adjacent pixels are transposed (4x4 bytes, 8 byte permutes, the
// first stage shared between overlapping groups) into one dword per channel; a filter row is the byte vector (w0, w1, w2, 0) or, for
// the output one pixel to the right within the same group, (0, w0, w1, w2).
#pragma once
#include "catchq_common.h"

namespace catchq {

constexpr int DW3_PW = 4, DW3_PH = 2;  // columns and rows of a lane's outputs

// S: the stride
template <int S>
struct Dw3Window {
  static constexpr int NR = (DW3_PH - 1) * S + 3;   // input rows
  static constexpr int NG = S == 1 ? 2 : 4;         // transposed groups per input row: pixels 0-3, 2-5 [, 4-7, 6-9]
  static constexpr int NCL = 2 * NG + 2;            // input columns (stride 2: one more than the window, weight 0)
};

// 36 filter bytes of four channels, [channel][tap] -> [channel][filter row]: bytes (w0, w1, w2, 0)
__device__ __forceinline__ void dw3_pack(const int (&raw)[9], int (&wa)[4][3]) {
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      unsigned v = 0;
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const int b = j * 9 + r * 3 + q;
        v |= (((unsigned)raw[b >> 2] >> (8 * (b & 3))) & 0xffu) << (8 * q);
      }
      wa[j][r] = (int)v;
    }
}

// input row ri of the window (xr: four channels of NCL pixels) into the sums; wb: wa shifted by a byte.  Every sum starts with
// filter row 0 (accumulator operand 0), no zeroing pass.
template <int S>
__device__ __forceinline__ void dw3_row(int ri, const unsigned (&xr)[Dw3Window<S>::NCL], const int (&wa)[4][3], const int (&wb)[4][3],
                                        int (&acc)[DW3_PH][DW3_PW][4]) {
  constexpr int NG = Dw3Window<S>::NG;
  // first transposition stage on pixel pairs (2m, 2m+1): bytes (a0,b0,a1,b1) and (a2,b2,a3,b3)
  unsigned lo[NG + 1], hi[NG + 1];
#pragma unroll
  for (int m = 0; m <= NG; ++m) {
    lo[m] = __builtin_amdgcn_perm(xr[2 * m + 1], xr[2 * m], 0x05010400u);
    hi[m] = __builtin_amdgcn_perm(xr[2 * m + 1], xr[2 * m], 0x07030602u);
  }
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    // second stage: group g = pixels 2g .. 2g+3, one dword per channel
    int t[4];
    t[0] = (int)__builtin_amdgcn_perm(lo[g + 1], lo[g], 0x05040100u);
    t[1] = (int)__builtin_amdgcn_perm(lo[g + 1], lo[g], 0x07060302u);
    t[2] = (int)__builtin_amdgcn_perm(hi[g + 1], hi[g], 0x05040100u);
    t[3] = (int)__builtin_amdgcn_perm(hi[g + 1], hi[g], 0x07060302u);
#pragma unroll
    for (int py = 0; py < DW3_PH; ++py) {
      const int r = ri - py * S;
      if (r < 0 || r > 2) continue;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (S == 1) {  // group g serves outputs 2g (taps at bytes 0..2) and 2g+1 (bytes 1..3)
          acc[py][2 * g][j] = __builtin_amdgcn_sdot4(t[j], wa[j][r], r == 0 ? 0 : acc[py][2 * g][j], false);
          acc[py][2 * g + 1][j] = __builtin_amdgcn_sdot4(t[j], wb[j][r], r == 0 ? 0 : acc[py][2 * g + 1][j], false);
        } else {                 // stride 2: group g starts at input pixel 2g = the window of output g
          acc[py][g][j] = __builtin_amdgcn_sdot4(t[j], wa[j][r], r == 0 ? 0 : acc[py][g][j], false);
        }
      }
    }
  }
}

// ReLU or ReLU6 and the requantizer behind it: (acc / div + bias) clamped to [0, hi], scaled, rounded to even; four bytes.
struct ReluRequant {
  float hi, scale;
  __device__ __forceinline__ explicit ReluRequant(const IrbStageDev &s) {
    hi = __builtin_ldexpf(127.0f, -s.q_neg_pos);
    if (s.relu6) hi = hi < 6.0f ? hi : 6.0f;
    scale = __builtin_ldexpf(1.0f, s.q_neg_pos);
  }
  __device__ __forceinline__ unsigned four(const int *a, const v4f dv, const v4f rc, const v4f bs) const {
    unsigned b[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      float x = div_by_rcp((float)a[t], dv[t], rc[t]) + bs[t];
      x = __builtin_amdgcn_fmed3f(x, 0.0f, hi);  // ReLU and the upper clamp; NaN -> 0
      b[t] = __builtin_bit_cast(unsigned, __builtin_fmaf(x, scale, 12582912.0f));
    }
    const unsigned lo = __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400u);
    const unsigned up = __builtin_amdgcn_perm(b[3], b[2], 0x04000c0cu);
    return lo | up;
  }
};

}  // namespace catchq
