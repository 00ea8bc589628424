// Which products the routes on packed weights take, by their sizes: asked by their launchers (float_rows.hip, digits_i16.hip,
// where both sides of every bound are measured) and by the operators, which lay a weight out only for calls that will read it.
#pragma once
#include <cstdint>

namespace catchq {

// compute units one launch should plan its tile shapes for: the device's 256, divided by the number of
// launches the caller says share the device (catchq_epilogue_t::sharing)
inline int planned_cus(int sharing) {
  const int cus = 256 / (sharing < 1 ? 1 : sharing);
  return cus < 1 ? 1 : cus;
}

// int8, float_rows
inline bool float_rows_sizes(int64_t m, int64_t n, int64_t k, bool half_out) {
  return m >= 1024 && n > (half_out ? 512 : 256) && m * n >= 1250000 && k >= 64 && k <= 1312 && k % 16 == 0;
}

// int16, gemm_digits: five eighths of a tile of 64 x 128 outputs per unit; the digits' sums fit 32 bits up to kDigitsMaxK
constexpr int64_t kDigitsMaxK = 8192;
inline bool digits_sizes(int64_t m, int64_t n, int64_t k, int cus) {
  return k >= 32 && k <= kDigitsMaxK && (m + 63) / 64 * ((n + 127) / 128) * 8 >= 5 * (int64_t)cus;
}

// int16 convolutions, conv_digits: five eighths of a tile of 64 x 128 (up to 64 columns 128 x 64) outputs per unit, and 16 sub-steps of
// 32 values of K for each.  Whole calls, us, operands as they lie / digits: 5 x 59x59, 222 -> 40, 3 x 3 stride 2 55.4 / 21.5, 8 x 76x76,
// 269 -> 56 163 / 65, 93x93, 326 -> 322, 5 x 5 231 / 127, 2 x 97x97, 192 -> 108 61 / 40, 3 x 91x102, 16 -> 281 half 54 / 36, 3 x 66x77,
// 90 -> 110 24.1 / 21.4; below the lines 12 x 11x16 -> 8 x 6, 32 -> 476 13.0 / 15.9 (192 tiles of 12 sub-steps), 1 x 51x62, 48 -> 261, 5 x
// 5 18.4 / 26.5 (150 tiles), 3 x 37x42 -> 18x29, 448 -> 137, 5 x 5 36.5 / 96.8 (50: a lone block waits for its filters).
inline bool conv_digits_sizes(int64_t m, int64_t n, int64_t ci, int64_t taps, int cus) {
  const int64_t tiles = n <= 64 ? (m + 127) / 128 : (m + 63) / 64 * ((n + 127) / 128);
  return taps > 1 && tiles * 8 >= 5 * (int64_t)cus && tiles * ((ci + 31) / 32 * taps) >= 16 * (int64_t)cus;
}

// int8, conv3x3_i8_packed: the patch-resident kernels (conv3x3_halo_i8.hip) are ahead on the channels they have instances for, the one
// that walks over tiles (conv3x3_i8_walk.hip) on 32; neither takes rows of outputs that are no multiple of four
inline bool conv3x3_i8_packed_channels(int64_t ci, int64_t co) {
  return ci >= 64 && ci <= 1024 && ci % 32 == 0 && (co % 4 != 0 || (ci >= 96 && ci != 128 && ci != 256 && ci != 512));
}

// int16 x int8, conv3x3_a16_packed: what its rule asks of the filters alone.  Blocks have 256 columns; those that do not exist cost as
// much as others, up to a quarter of them pays.
inline bool conv3x3_a16_packed_filters(int64_t co, int64_t ci) {
  return ci % 64 == 0 && co % 4 == 0 && co * 4 >= (co + 255) / 256 * 256 * 3;
}

// ... at stride 2 (conv3x3_a16_packed_s2.hip, where both sides are measured): not a quarter of one column of blocks, nor 64 channels, whose
// four steps do not repay the longer way to the first (108 x 114, 64 -> 768 14.0 us on the tiled kernel / 17.5, 4 x 64 x 58, 64 -> 1024
// 17.1 / 18.4, two launches at a time)
inline bool conv3x3_a16_packed_s2_filters(int64_t co, int64_t ci) { return conv3x3_a16_packed_filters(co, ci) && ci >= 128 && co >= 224; }

}  // namespace catchq
