// Pieces shared by the int8 implicit-GEMM kernels: parameters, the LDS swizzle, and the epilogue.
#pragma once
#include <type_traits>

#include "catchq_common.h"

namespace catchq {

struct IgemmParams {
  int64_t M;
  int N, K;
  int H, W, Ci, Ho, Wo, kh, kw, ph, pw, sh, sw, dh, dw;
  int kwq;  // LOAD_C4: chunks (groups of 4 taps) per filter row
  // LDS-DMA im2col loader: element strides of the activation tensor (image, image row, output-column
  // step unit).  A plain NHWC tensor has H*W*Ci, W*Ci, Ci; the pixel-window form of a few-channel
  // input (a filter row = one contiguous run of kw*C elements) uses other values.
  unsigned img_stride, row_stride, pix_stride;
  int tiles_n;
  int nblocks;
  // Order in which consecutive block ids walk the tile grid: 0 = row by row (all column tiles of one row tile,
  // then the next row tile); g > 0 = in bands of g row tiles, column by column inside a band, so that the blocks
  // running at the same time cover a g x (concurrent / g) patch of tiles and share both operands' panels in L2
  // instead of streaming the whole B operand past every row tile.
  int group_m;
  int tiles_m;
  // Leading dimension of the output matrices (y, q, acc_out, resid); 0 = N.  A grouped convolution runs one GEMM per
  // group (grid dimension y) whose N is the group's share of the output channels while the rows stay Co apart.
  int ldc;
  // groups > 1: per-group offsets -- bytes into the activation tensor (a pixel's channel slice), bytes into the
  // weights (the group's filters) and output channels (columns of the outputs and entries of the per-channel vectors)
  int groups, a_group_bytes, n_group;
  int ragged;  // EPI_SCALAR: the epilogue that serves the rows all the same (ragged_epilogue), or EPI_SCALAR
  int64_t b_group_bytes;
};

__device__ __forceinline__ int out_ld(const IgemmParams &p) { return p.ldc ? p.ldc : p.N; }

constexpr int BK = 64;  // bytes of K per pipeline step (one LDS row)
enum { LOAD_GEMM = 0, LOAD_CONV = 1, LOAD_C4 = 2 };

// LDS rows are 64 bytes = four 16-byte chunks; the chunk index is XOR-ed with (row>>2)&3 so that
// 16 consecutive rows at one logical chunk fall into 16 different 16-byte bank groups
// (measured: 176 B/clk/CU with the swizzle, 62 B/clk/CU without).
__device__ __forceinline__ int swz(int row, int chunk) { return chunk ^ ((row >> 2) & 3); }

// block id -> tile index, XCD-aware: ids that land on one XCD (id % 8) take a contiguous run of
// tiles, so neighbouring tiles (same A rows, same weights) share that XCD's L2.
__device__ __forceinline__ int xcd_remap(int bid, int nb) {
  const int xcd = bid & 7, local = bid >> 3;
  const int q = nb >> 3, rem = nb & 7;
  return xcd * q + (xcd < rem ? xcd : rem) + local;
}

// bit r * kw + q: filter tap (r, q) of a pixel whose tap (0, 0) lies at (hi0, wi0) is inside the image (at most 32 taps).
// Rows and columns apart: tap by tap it was nine branches a pixel, half of the 6500 clocks in front of a block's first
// transfer (5 x 57 x 75, 96 -> 160 channels 14.7 -> 13.9 us, 8 x 28 x 28, 5 x 5, 256 -> 128 24.0 -> 21.9).
__device__ __forceinline__ unsigned tap_mask(int hi0, int wi0, const IgemmParams &p) {
  unsigned cols = 0, mask = 0;
  for (int q = 0; q < p.kw; ++q) cols |= ((unsigned)(wi0 + q * p.dw) < (unsigned)p.W ? 1u : 0u) << q;
  for (int r = 0; r < p.kh; ++r) mask |= ((unsigned)(hi0 + r * p.dh) < (unsigned)p.H ? cols : 0u) << (r * p.kw);
  return mask;
}

inline bool vec_epilogue_ok(int N, const EpiDev &e) {
  // (N < 2^24: the per-lane part of an element index, at most 32 rows, fits 32 bits with room to spare)
  return N % 4 == 0 && N < (1 << 24) && aligned16(e.chan_div) && aligned16(e.chan_rcp) && aligned16(e.bias) && aligned16(e.resid) && aligned16(e.y) &&
         aligned16(e.acc_out) && aligned16(e.q);
}

// What an epilogue instance knows at compile time.  A field of -1 is decided at run time from the
// EpiDev (the generic instance); fixed fields let the compiler drop every untaken branch, which
// matters because the epilogue is VALU-bound (about a dozen fp32 operations per output element).
//   DIV  0 none, 1 reciprocal form (the constants of a launch without divisors or bias are 1 and -0: nothing changes), 2 true
//   division, 3 reciprocal form with every step rounded to binary16 (half_steps)      BIAS 0/1     RESID 0 none, 1 before, 2 after the activation
//   ACT  CATCHQ_ACT_*       YM  0 none, 1 fp32, 2 fp16     QM  0 none, 8, 16     ACC 0/1
template <int DIV, int BIAS, int RESID, int ACT, int YM, int QM, int ACC>
struct EpiSpec {
  static constexpr bool kGeneric = DIV < 0;
  static constexpr bool kSteps = DIV == 3;
  static constexpr int kAct = ACT;
  static constexpr int kQ = QM;
  // the instances of layers with a floating output and nothing else read a bias of either precision
  static constexpr bool kAnyBias = DIV < 0 || (QM == 0 && RESID == 0);
  // ReLU / ReLU6 feeding nothing but an int8 requantization: the activation folds into the clamp of the
  // quantizer, 0 <= x <= min(6, 127 * 2^pos)
  static constexpr bool kFoldAct = DIV >= 0 && QM == 8 && YM == 0 && ACC == 0 && RESID != 2 &&
                                   (ACT == CATCHQ_ACT_RELU || ACT == CATCHQ_ACT_RELU6);
  // ... and with the reciprocal form and no residual the requantization's power of two folds into the per-channel
  // constants as well (scaling by 2^k is exact, so every intermediate is the scaled image of the unfolded one): the
  // value arrives in units of the output's step, and one instruction (v_cvt_pk_u8_f32: round to nearest even,
  // saturate to 0 .. 255, insert the byte) rounds and packs it
  static constexpr bool kFoldScale = kFoldAct && DIV == 1 && RESID == 0;
  static __device__ __forceinline__ bool rcp(const EpiDev &e) { return DIV < 0 ? e.chan_rcp != nullptr : DIV == 1; }
  static __device__ __forceinline__ bool truediv(const EpiDev &e) {
    return DIV < 0 ? (e.chan_div != nullptr && e.chan_rcp == nullptr) : DIV == 2;
  }
  static __device__ __forceinline__ bool bias(const EpiDev &e) { return BIAS < 0 ? e.bias != nullptr : BIAS == 1; }
  static __device__ __forceinline__ bool resid(const EpiDev &e) { return RESID < 0 ? e.resid != nullptr : RESID >= 1; }
  static __device__ __forceinline__ bool resid_after(const EpiDev &e) { return RESID < 0 ? e.resid_after != 0 : RESID == 2; }
  static __device__ __forceinline__ int act(const EpiDev &e) { return ACT < 0 ? e.act : ACT; }
  static __device__ __forceinline__ bool y32(const EpiDev &e) { return YM < 0 ? (e.y && !e.y_f16) : YM == 1; }
  static __device__ __forceinline__ bool y16(const EpiDev &e) { return YM < 0 ? (e.y && e.y_f16) : YM == 2; }
  static __device__ __forceinline__ bool q8(const EpiDev &e) { return QM < 0 ? (e.q && e.q_bw == 8) : QM == 8; }
  static __device__ __forceinline__ bool q16(const EpiDev &e) { return QM < 0 ? (e.q && e.q_bw == 16) : QM == 16; }
  static __device__ __forceinline__ bool acc(const EpiDev &e) { return ACC < 0 ? e.acc_out != nullptr : ACC == 1; }
};
typedef EpiSpec<-1, -1, -1, -1, -1, -1, -1> EpiGeneric;

// epilogue variants a kernel can be instantiated with
enum {
  EPI_SCALAR = 0,   // any N / alignment: one element at a time, straight from the accumulators
  EPI_VECTOR = 1,   // generic, vectorised through LDS (N % 4 == 0, 16-byte aligned pointers)
  EPI_Q8_RELU = 2,  // reciprocal-form dequant + bias + ReLU -> int8                 (conv feeding a conv)
  EPI_RES_Y_Q8 = 3, // ... + residual + ReLU -> fp32 and int8                         (end of a residual block)
  EPI_Y32 = 4,      // reciprocal-form dequant + bias -> fp32                         (projection shortcut)
  EPI_RES_Y = 5,    // ... + residual + ReLU -> fp32                                   (last block)
  EPI_Y16_RELU = 6, // reciprocal-form dequant + bias + ReLU -> fp16                  (standalone linear)
  EPI_Q8_RELU6 = 7, // reciprocal-form dequant + bias + ReLU6 -> int8
  EPI_RES_Q8 = 8,   // ... + residual + ReLU -> int8 only                             (last block of a stage)
  // linear bottlenecks (no activation), reciprocal-form dequant + bias:
  EPI_LIN_Q8 = 9,          // -> int8
  EPI_LIN_Y_Q8 = 10,       // -> fp32 and int8
  EPI_LIN_RES_Q8 = 11,     // + residual -> int8
  EPI_LIN_RES_Y_Q8 = 12,   // + residual -> fp32 and int8
  // per-tensor weights (no divisor), bias, leaky ReLU, int16 requantization:
  EPI_LK_Q16 = 13,         // -> int16
  EPI_LK_Y_Q16 = 14,       // -> fp32 and int16
  EPI_LK_RESA_Q16 = 15,    // residual added after the activation -> int16
  EPI_LK_RESA_Y_Q16 = 16,  // residual added after the activation -> fp32 and int16
  EPI_Y16 = 17,        // reciprocal-form dequant + bias -> fp16
  EPI_Y16_STEPS = 18,  // ... with every step rounded to binary16, as half tensor ops would leave it
  EPI_COUNT = 19
};
template <int EPI> struct EpiOf { typedef EpiGeneric type; };
template <> struct EpiOf<EPI_Q8_RELU> { typedef EpiSpec<1, 1, 0, CATCHQ_ACT_RELU, 0, 8, 0> type; };
template <> struct EpiOf<EPI_RES_Y_Q8> { typedef EpiSpec<1, 1, 1, CATCHQ_ACT_RELU, 1, 8, 0> type; };
template <> struct EpiOf<EPI_Y32> { typedef EpiSpec<1, 1, 0, CATCHQ_ACT_NONE, 1, 0, 0> type; };
template <> struct EpiOf<EPI_RES_Y> { typedef EpiSpec<1, 1, 1, CATCHQ_ACT_RELU, 1, 0, 0> type; };
template <> struct EpiOf<EPI_Y16_RELU> { typedef EpiSpec<1, 1, 0, CATCHQ_ACT_RELU, 2, 0, 0> type; };
template <> struct EpiOf<EPI_Y16> { typedef EpiSpec<1, 1, 0, CATCHQ_ACT_NONE, 2, 0, 0> type; };
template <> struct EpiOf<EPI_Y16_STEPS> { typedef EpiSpec<3, 1, 0, CATCHQ_ACT_NONE, 2, 0, 0> type; };
template <> struct EpiOf<EPI_Q8_RELU6> { typedef EpiSpec<1, 1, 0, CATCHQ_ACT_RELU6, 0, 8, 0> type; };
template <> struct EpiOf<EPI_RES_Q8> { typedef EpiSpec<1, 1, 1, CATCHQ_ACT_RELU, 0, 8, 0> type; };
template <> struct EpiOf<EPI_LIN_Q8> { typedef EpiSpec<1, 1, 0, CATCHQ_ACT_NONE, 0, 8, 0> type; };
template <> struct EpiOf<EPI_LIN_Y_Q8> { typedef EpiSpec<1, 1, 0, CATCHQ_ACT_NONE, 1, 8, 0> type; };
template <> struct EpiOf<EPI_LIN_RES_Q8> { typedef EpiSpec<1, 1, 1, CATCHQ_ACT_NONE, 0, 8, 0> type; };
template <> struct EpiOf<EPI_LIN_RES_Y_Q8> { typedef EpiSpec<1, 1, 1, CATCHQ_ACT_NONE, 1, 8, 0> type; };
template <> struct EpiOf<EPI_LK_Q16> { typedef EpiSpec<0, 1, 0, CATCHQ_ACT_LEAKY, 0, 16, 0> type; };
template <> struct EpiOf<EPI_LK_Y_Q16> { typedef EpiSpec<0, 1, 0, CATCHQ_ACT_LEAKY, 1, 16, 0> type; };
template <> struct EpiOf<EPI_LK_RESA_Q16> { typedef EpiSpec<0, 1, 2, CATCHQ_ACT_LEAKY, 0, 16, 0> type; };
template <> struct EpiOf<EPI_LK_RESA_Y_Q16> { typedef EpiSpec<0, 1, 2, CATCHQ_ACT_LEAKY, 1, 16, 0> type; };

// which variant serves this launch (the specialised ones also need a unit requantization scale: a
// fractional one costs them 2-4 % end to end even when it is not used, measured); a kernel family
// that has no instance of the variant returned uses the generic EPI_VECTOR
inline int pick_epilogue(int N, const EpiDev &e) {
  if (!vec_epilogue_ok(N, e)) return EPI_SCALAR;
  if (e.acc_out || (e.q && e.q_scale != 1.0f) || (e.chan_div && !e.chan_rcp && !e.half_rcp)) return EPI_VECTOR;
  if (e.bias_f16 && (e.q || e.resid)) return EPI_VECTOR;  // (kAnyBias)
  // (the instances that fold the requantization's power of two into the per-channel constants keep those in range)
  if (e.q && (e.q_neg_pos < -40 || e.q_neg_pos > 40)) return EPI_VECTOR;
  const int div = e.half_steps ? (e.half_rcp ? 3 : 2) : (e.chan_rcp ? 1 : 0), bias = e.bias ? 1 : 0;
  // without divisors the reciprocal form runs on ones (x * 2^e exactly, the correction is zero), without a bias on -0
  // (x + -0 = x for every x, -0 among them: a small negative sum rounded to binary16); the power of two has to stay in the
  // range that form is stated for
  const bool ones = div == 0 && !e.exp2_a && !e.exp2_b && e.exp2 >= -64 && e.exp2 <= 64;
  const int res = !e.resid ? 0 : (e.resid_after ? 2 : 1);
  const int ym = !e.y ? 0 : (e.y_f16 ? 2 : 1);
  const int qm = !e.q ? 0 : e.q_bw;
  static const struct { int epi, div, bias, res, act, ym, qm; } rows[] = {
      {EPI_Q8_RELU, 1, 1, 0, CATCHQ_ACT_RELU, 0, 8},        {EPI_RES_Y_Q8, 1, 1, 1, CATCHQ_ACT_RELU, 1, 8},
      {EPI_Y32, 1, 1, 0, CATCHQ_ACT_NONE, 1, 0},            {EPI_RES_Y, 1, 1, 1, CATCHQ_ACT_RELU, 1, 0},
      {EPI_Y16_RELU, 1, 1, 0, CATCHQ_ACT_RELU, 2, 0},       {EPI_Q8_RELU6, 1, 1, 0, CATCHQ_ACT_RELU6, 0, 8},
      {EPI_RES_Q8, 1, 1, 1, CATCHQ_ACT_RELU, 0, 8},         {EPI_LIN_Q8, 1, 1, 0, CATCHQ_ACT_NONE, 0, 8},
      {EPI_LIN_Y_Q8, 1, 1, 0, CATCHQ_ACT_NONE, 1, 8},       {EPI_LIN_RES_Q8, 1, 1, 1, CATCHQ_ACT_NONE, 0, 8},
      {EPI_LIN_RES_Y_Q8, 1, 1, 1, CATCHQ_ACT_NONE, 1, 8},   {EPI_LK_Q16, 0, 1, 0, CATCHQ_ACT_LEAKY, 0, 16},
      {EPI_LK_Y_Q16, 0, 1, 0, CATCHQ_ACT_LEAKY, 1, 16},     {EPI_LK_RESA_Q16, 0, 1, 2, CATCHQ_ACT_LEAKY, 0, 16},
      {EPI_LK_RESA_Y_Q16, 0, 1, 2, CATCHQ_ACT_LEAKY, 1, 16}, {EPI_Y16, 1, 1, 0, CATCHQ_ACT_NONE, 2, 0},
      {EPI_Y16_STEPS, 3, 1, 0, CATCHQ_ACT_NONE, 2, 0}};
  for (const auto &r : rows)
    if ((r.div == div || (r.div == 1 && ones)) && (r.bias == bias || bias == 0) && r.res == res && r.act == e.act && r.ym == ym && r.qm == qm) return r.epi;
  return EPI_VECTOR;
}

// For rows whose length or alignment the vectorised epilogues do not take, a floating output and nothing else: the epilogue
// (EPI_Y32, EPI_Y16 or, where the caller has it, EPI_Y16_STEPS) that serves them with stores that need no alignment (EpiAtRagged);
// EPI_SCALAR: none does.
inline int ragged_epilogue(int N, const EpiDev &e, bool steps = false) {
  if (N >= (1 << 24)) return EPI_SCALAR;
  EpiDev aligned = e;
  auto stand_in = [](const auto *q) { return reinterpret_cast<decltype(q)>(q ? (uintptr_t)16 : 0); };  // (presence only)
  aligned.chan_div = stand_in(e.chan_div); aligned.chan_rcp = stand_in(e.chan_rcp); aligned.bias = stand_in(e.bias);
  aligned.y = const_cast<void *>((const void *)stand_in((const char *)e.y));
  const int epi = pick_epilogue((N + 3) / 4 * 4, aligned);
  return epi == EPI_Y32 || epi == EPI_Y16 || (steps && epi == EPI_Y16_STEPS) ? epi : EPI_SCALAR;
}

// per-channel constants of one lane's four consecutive channels
struct EpiLane {
  v4f div, rcp, bias;
  bool use_rcp, use_div, use_bias, use_res, res_after, unit_q, half_steps;
  bool steps_rcp = false;  // half_steps with the division in reciprocal form
  int act;
};

__device__ __forceinline__ v4f half4_values(const v2i bits) {
  typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
  return __builtin_convertvector(__builtin_bit_cast(f16x4, bits), v4f);
}
// A bias of four consecutive channels (n a multiple of four), of either precision.  (One load and a conditional one: a branch
// to either load measured the same or slower.)
struct Bias4 {
  v2i lo = {kNoBias, kNoBias}, hi = {kNoBias, kNoBias};  // halfs: all four in lo
  static constexpr int kNoBias = (int)0x80000000u;       // -0: x + -0 = x
  __device__ __forceinline__ void load(const EpiDev &e, int n) {
    if (!e.bias) return;
    const char *at = (const char *)e.bias + ((int64_t)n << (e.bias_f16 ? 1 : 2));
    lo = *reinterpret_cast<const v2i *>(at);
    if (!e.bias_f16) hi = *reinterpret_cast<const v2i *>(at + 8);
  }
  __device__ __forceinline__ v4f values(const EpiDev &e) const {
    return e.bias_f16 ? half4_values(lo) : __builtin_bit_cast(v4f, v4i{lo[0], lo[1], hi[0], hi[1]});
  }
};

// The lane's constants from the raw values of its four channels (1 / 1 / -0 where a constant is absent).
template <class S>
__device__ __forceinline__ EpiLane epi_lane_finish(v4f div, v4f rcp, v4f bias, const EpiDev &e) {
  EpiLane L;
  L.use_rcp = S::rcp(e); L.use_div = S::truediv(e); L.use_bias = S::bias(e); L.use_res = S::resid(e);
  L.res_after = S::resid_after(e);
  L.act = S::act(e);
  L.unit_q = S::kGeneric ? (e.q_scale == 1.0f) : true;
  L.half_steps = S::kGeneric ? (e.half_steps != 0) : S::kSteps;
  L.steps_rcp = S::kSteps;
  // Reciprocal form with the power of two folded in:
  //   v = (f*2^e)/d  ==  q = f*(r*2^e); err = fma(-q, d*2^-e, f); fma(err, r*2^e, q)
  // (scaling by 2^e is exact, so every intermediate is the scaled image of the unfolded one)
  L.div = div; L.rcp = rcp; L.bias = bias;
  if (L.use_rcp) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      L.rcp[t] = __builtin_ldexpf(L.rcp[t], e.exp2 + (S::kFoldScale ? e.q_neg_pos : 0));
      L.div[t] = __builtin_ldexpf(L.div[t], -e.exp2 - (S::kFoldScale ? e.q_neg_pos : 0));
    }
  }
  if constexpr (S::kFoldScale) {
#pragma unroll
    for (int t = 0; t < 4; ++t) L.bias[t] = __builtin_ldexpf(L.bias[t], e.q_neg_pos);
  }
  return L;
}

// the same from vectors of any alignment and length N (channels beyond it: the last one's constants)
template <class S>
__device__ __forceinline__ EpiLane epi_lane_setup_ragged(int n, int N, const EpiDev &e) {
  v4f div, rcp, bias;
  const float *rcps = S::kSteps ? e.half_rcp : e.chan_rcp;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int c = min(n + t, N - 1);
    div[t] = e.chan_div ? e.chan_div[c] : 1.0f;
    rcp[t] = rcps ? rcps[c] : 1.0f;
    bias[t] = e.bias ? bias_value(e, c) : -0.0f;
  }
  return epi_lane_finish<S>(div, rcp, bias, e);
}

template <class S>
__device__ __forceinline__ EpiLane epi_lane_setup(int n, bool n_ok, const EpiDev &e) {
  v4f div = {1.f, 1.f, 1.f, 1.f}, rcp = {1.f, 1.f, 1.f, 1.f}, bias = {-0.f, -0.f, -0.f, -0.f};
  const float *rcps = S::kSteps ? e.half_rcp : e.chan_rcp;
  if (n_ok && (S::rcp(e) || S::truediv(e) || S::kSteps) && e.chan_div) div = *reinterpret_cast<const v4f *>(e.chan_div + n);
  if (n_ok && (S::rcp(e) || S::kSteps) && rcps) rcp = *reinterpret_cast<const v4f *>(rcps + n);
  if constexpr (S::kAnyBias) {
    Bias4 b;
    if (n_ok && S::bias(e)) b.load(e, n);
    bias = b.values(e);
  } else {
    if (n_ok && S::bias(e) && e.bias) bias = *reinterpret_cast<const v4f *>(e.bias + n);
  }
  return epi_lane_finish<S>(div, rcp, bias, e);
}

// dequantization and bias of one integer sum (converted to fp32 once): channel t of the lane's four
__device__ __forceinline__ float epi_dequant1(float x, int t, const EpiLane &L, int exp2) {
  if (L.steps_rcp) {
    // fp32 operations on binary16 values rounded to binary16 are the binary16 operations.  The reciprocal form gives the
    // correctly rounded fp32 quotient of the finite values; an infinite one (the scaled sum overflowed) stays infinite.  The
    // residual is taken as q d - x and subtracted: a zero quotient then keeps its sign (x - q d would be +0 and make -0 positive).
    x = round_f16(__builtin_ldexpf(x, exp2));
    const float q = x * L.rcp[t];
    float v = __builtin_fmaf(-__builtin_fmaf(q, L.div[t], -x), L.rcp[t], q);
    v = __builtin_isinf(q) ? q : v;
    asm volatile("" : "+v"(v));  // keeps the conversion below apart: fused into one operation it would round once
    return round_f16(v) + L.bias[t];  // (rounded to binary16 by the conversion of the output)
  }
  if (L.use_rcp) x = div_by_rcp(x, L.div[t], L.rcp[t]);
  else {
    x = __builtin_ldexpf(x, exp2);
    if (L.half_steps) x = round_f16(x);
    if (L.use_div) {
      x = x / L.div[t];
      if (L.half_steps) x = round_f16(x);
    }
  }
  if (L.use_bias) {
    x = x + L.bias[t];
    if (L.half_steps) x = round_f16(x);
  }
  return x;
}

// Where an output element lives: a 64-bit element index, or a wave-uniform 64-bit part plus a 32-bit
// per-lane part (then the uniform part stays in scalar registers and a store needs one vector add).
struct EpiAt64 {
  int64_t idx;
  template <class T> __device__ __forceinline__ T *at(T *base) const { return base + idx; }
};
struct EpiAtSplit {
  int64_t uni;   // same for every lane of the wave
  unsigned off;  // this lane's part
  template <class T> __device__ __forceinline__ T *at(T *base) const { return (base + uni) + off; }
};

// Rows of any length and alignment: four channels of which the first `left` exist (floating outputs only).
struct EpiAtRagged {
  int64_t idx;
  int left;
  template <class T> __device__ __forceinline__ T *at(T *base) const { return base + idx; }
};
// four elements at once (global memory takes any element's alignment), one by one at the end of a row
template <class T, class V>
__device__ __forceinline__ void store_ragged(T *dst, const V v, int left) {
  typedef T vec_t __attribute__((ext_vector_type(4), aligned(sizeof(T))));
  if (left >= 4) {
    *reinterpret_cast<vec_t *>(dst) = __builtin_bit_cast(vec_t, v);
  } else {
#pragma unroll
    for (int t = 0; t < 3; ++t)
      if (t < left) dst[t] = v[t];
  }
}

// A store / load with or without the non-temporal hint, chosen by a wave-uniform flag.  The empty volatile
// statements keep the two branches apart: merged into one access, they would lose the hint.
template <class T>
__device__ __forceinline__ void store_stream(T *dst, const T v, bool stream) {
  if (stream) {
    asm volatile("");
    __builtin_nontemporal_store(v, dst);
    asm volatile("");
  } else {
    *dst = v;
  }
}
template <class T>
__device__ __forceinline__ T load_stream(const T *src, bool stream) {
  T v;
  if (stream) {
    asm volatile("");
    v = __builtin_nontemporal_load(src);
    asm volatile("");
  } else {
    v = *src;
  }
  return v;
}

// four integer sums of one pixel (channels n..n+3 at `where`) -> all requested outputs; sums too wide for an int32 come
// converted to fp32 (v4f)
template <class S, class At, class Sums>
__device__ __forceinline__ void epi_vec4(const Sums a, const v4f res, const EpiLane &L, const At where, const EpiDev &e) {
  if constexpr (std::is_same<Sums, v4i>::value) {
    if (S::acc(e)) *reinterpret_cast<v4i *>(where.at(e.acc_out)) = a;
  }
  float v[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    float x = epi_dequant1((float)a[t], t, L, e.exp2);
    if (L.use_res && !L.res_after) x = x + res[t];
    if constexpr (!S::kFoldAct) {
      if (L.act == CATCHQ_ACT_LEAKY) x = (x > 0.0f) ? x : x * e.act_slope;
      else if (L.act >= CATCHQ_ACT_RELU) x = (x > 0.0f) ? x : 0.0f;
      if (L.act == CATCHQ_ACT_RELU6) x = (x < 6.0f) ? x : 6.0f;
      if (L.use_res && L.res_after) x = x + res[t];
    }
    v[t] = x;
  }
  if (S::y16(e)) {
    // two values per conversion instruction (v_cvt_pk_f16_f32: round to nearest even, like the single conversion)
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    const f16x2 h01 = __builtin_convertvector(f32x2{v[0], v[1]}, f16x2), h23 = __builtin_convertvector(f32x2{v[2], v[3]}, f16x2);
    const v2i packed = {__builtin_bit_cast(int, h01), __builtin_bit_cast(int, h23)};
    if constexpr (std::is_same<At, EpiAtRagged>::value) {
      typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
      store_ragged(where.at(reinterpret_cast<_Float16 *>(e.y)), __builtin_bit_cast(f16x4, packed), where.left);
    } else
      store_stream(reinterpret_cast<v2i *>(where.at(reinterpret_cast<__half *>(e.y))), packed, e.y_stream != 0);
  } else if (S::y32(e)) {
    v4f o = {v[0], v[1], v[2], v[3]};
    if constexpr (std::is_same<At, EpiAtRagged>::value) store_ragged(where.at(reinterpret_cast<float *>(e.y)), o, where.left);
    else
      store_stream(reinterpret_cast<v4f *>(where.at(reinterpret_cast<float *>(e.y))), o, e.y_stream != 0);
  }
  if constexpr (S::kFoldScale) {
    // v is already in units of the output's step: clamp to 0 .. min(127, 6 / step) (the median maps a NaN to 0, as
    // ReLU does), then round, saturate and insert byte by byte
    float hi = 127.0f;
    if constexpr (S::kAct == CATCHQ_ACT_RELU6) {
      const float six = __builtin_ldexpf(6.0f, e.q_neg_pos);
      hi = (six < hi) ? six : hi;
    }
    unsigned packed = 0;
#pragma unroll
    for (int t = 0; t < 4; ++t)
      packed = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_amdgcn_fmed3f(v[t], 0.0f, hi), (unsigned)t, packed);
    *reinterpret_cast<unsigned *>(where.at(reinterpret_cast<int8_t *>(e.q))) = packed;
  } else if constexpr (!S::kGeneric && S::kQ == 8 && (S::kAct == CATCHQ_ACT_RELU || S::kAct == CATCHQ_ACT_RELU6)) {
    // values are >= 0 and never NaN here (or, with the activation folded in, are made so by the median:
    // for a NaN operand it returns the smallest of the other two, 0, which is what ReLU makes of a NaN);
    // the requantization scale is 1:
    //   sat(rne(x * 2^-pos)) = low byte of the float  fma(min(x, 127 * 2^pos), 2^-pos, 1.5 * 2^23)
    // (the product is exact, so the fma rounds once, to an integer, ties to even; clamping before
    // the rounding equals clamping after it because the bound is an integer multiple of 2^pos; a ReLU6
    // bound of 6 below that one takes its place: min(min(x, 6), hi) = min(x, min(6, hi)))
    float hi = __builtin_ldexpf(127.0f, -e.q_neg_pos);
    const float sc = __builtin_ldexpf(1.0f, e.q_neg_pos);
    if constexpr (S::kFoldAct && S::kAct == CATCHQ_ACT_RELU6) hi = (hi < 6.0f) ? hi : 6.0f;
    unsigned b[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float x = __builtin_amdgcn_fmed3f(v[t], 0.0f, hi);  // one instruction for max(0, min(v, hi))
      b[t] = __builtin_bit_cast(unsigned, __builtin_fmaf(x, sc, 12582912.0f));
    }
    const unsigned lo = __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400u);
    const unsigned hi2 = __builtin_amdgcn_perm(b[3], b[2], 0x04000c0cu);
    *reinterpret_cast<unsigned *>(where.at(reinterpret_cast<int8_t *>(e.q))) = lo | hi2;
  } else if (S::q8(e)) {
    int b[4];
    if (L.unit_q) {
#pragma unroll
      for (int t = 0; t < 4; ++t) b[t] = quant1_unit<8>(v[t], e.q_neg_pos);
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t) b[t] = quant1<8>(v[t], e.q_scale, e.q_neg_pos);
    }
    // four clamped values -> four bytes: two byte permutes and a merge
    const unsigned lo = __builtin_amdgcn_perm((unsigned)b[1], (unsigned)b[0], 0x0c0c0400u);
    const unsigned hi = __builtin_amdgcn_perm((unsigned)b[3], (unsigned)b[2], 0x04000c0cu);
    *reinterpret_cast<unsigned *>(where.at(reinterpret_cast<int8_t *>(e.q))) = lo | hi;
  } else if (S::q16(e)) {
    // rounded to an integer and converted (NaN -> 0, out-of-range values saturate to the int32 range), then
    // v_cvt_pk_i16_i32 saturates two of them to int16 and packs them: no clamp, mask or shift of our own
    int i32[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float x = L.unit_q ? v[t] : v[t] * e.q_scale;
      i32[t] = cvt_i32_sat(__builtin_rintf(__builtin_ldexpf(x, e.q_neg_pos)));
    }
    v2i pk;
    pk[0] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_pk_i16(i32[0], i32[1]));
    pk[1] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_pk_i16(i32[2], i32[3]));
    *reinterpret_cast<v2i *>(where.at(reinterpret_cast<int16_t *>(e.q))) = pk;
  }
}
template <class S, class Sums>
__device__ __forceinline__ void epi_vec4(const Sums a, const v4f res, const EpiLane &L, int64_t idx, const EpiDev &e) {
  epi_vec4<S, EpiAt64, Sums>(a, res, L, EpiAt64{idx}, e);
}

// this lane's four channels within a wave tile of TN*32 columns starting at n_w
template <int TN>
__device__ __forceinline__ int epi_lane_channel(int n_w, int lane) { return n_w + (lane % (TN * 8)) * 4; }

// Vector epilogue of one wave with the lane's per-channel constants supplied by the caller (kernels
// that run many row groups against the same columns set them up once).  m_w and n_w are the same for
// every lane of the wave.  An element's index splits into the uniform (m_w + i*32) * N + n_w and a
// 32-bit per-lane rest, and a wave whose tile lies wholly inside the matrix (the usual case) runs
// without any per-lane bounds checks (FAST_PATH = false leaves that copy of the code out: kernels that
// unroll the epilogue several times over cannot afford the registers its free scheduling takes).
// BATCHES > 1 handles the 32 rows of a staged block in that many passes (residual loads, staged reads and
// arithmetic of one pass before the next): fewer values live at once, for instances that would otherwise lose a
// wave per SIMD to their register count.
template <int TM, int TN, int EPI, bool FAST_PATH = true, int BATCHES = 1>
__device__ __forceinline__ void igemm_epilogue_vec(v16i (&acc)[TM][TN], int *stage, int64_t m_w, int n_w, int lane,
                                                   const IgemmParams &p, const EpiDev &e, const EpiLane &L) {
  typedef typename EpiOf<EPI>::type S;
  constexpr int WN = TN * 32;
  constexpr int EPI_STRIDE = WN + 8;  // +8 ints: the two half-waves write different banks
  const int frow = lane & 31, fhalf = lane >> 5;
  constexpr int CPR = WN / 4;    // 4-channel groups per staged row
  constexpr int RPI = 64 / CPR;  // rows the wave moves per iteration
  constexpr int NIT = 32 / RPI;
  const int cg = lane % CPR, rsub = lane / CPR;
  const bool use_res = L.use_res;
  const unsigned lane_off0 = (unsigned)rsub * (unsigned)out_ld(p) + (unsigned)(cg * 4);
  const unsigned it_step = (unsigned)RPI * (unsigned)out_ld(p);
  auto tile = [&](auto full_c) {
    constexpr bool FULL = decltype(full_c)::value;
    const bool n_ok = FULL || (n_w + cg * 4 < p.N);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int64_t uni = (m_w + i * 32) * (int64_t)out_ld(p) + n_w;
      const int64_t left = p.M - (m_w + i * 32);
      const int rows = FULL ? 32 : (left < 0 ? 0 : (left > 32 ? 32 : (int)left));  // uniform
      // Opaque copy: a kernel that calls this in a loop would otherwise keep every iteration's byte
      // offsets (loop invariants) in registers across the whole loop; recomputing them costs one add each.
      unsigned lane_off = lane_off0;
      asm volatile("" : "+v"(lane_off));
      constexpr int NB = NIT / BATCHES;
      static_assert(NIT % BATCHES == 0, "the passes must divide the iterations");
      v4f resv[NB];
      auto load_resid = [&](int b) {
#pragma unroll
        for (int k = 0; k < NB; ++k) {
          const int it = b * NB + k;
          resv[k] = v4f{0.f, 0.f, 0.f, 0.f};
          if (FULL || (n_ok && it * RPI + rsub < rows))
            resv[k] = load_stream(reinterpret_cast<const v4f *>((e.resid + uni) + (lane_off + it * it_step)), e.resid_stream != 0);
        }
      };
      // residual rows of this 32-row block (of its first pass): all loads in flight before the staging below
      if (use_res) load_resid(0);
      // wave-private staging: stores then loads of the same wave, ordered by the LDS counter
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          stage[(8 * (r >> 2) + 4 * fhalf + (r & 3)) * EPI_STRIDE + j * 32 + frow] = acc[i][j][r];
#pragma unroll
      for (int b = 0; b < BATCHES; ++b) {
        if (b > 0 && use_res) load_resid(b);
        // all reads first: one LDS latency per pass instead of one per iteration
        v4i av[NB];
#pragma unroll
        for (int k = 0; k < NB; ++k)
          av[k] = *reinterpret_cast<const v4i *>(stage + ((b * NB + k) * RPI + rsub) * EPI_STRIDE + cg * 4);
#pragma unroll
        for (int k = 0; k < NB; ++k) {
          const int it = b * NB + k;
          if (!FULL && !(n_ok && it * RPI + rsub < rows)) continue;
          epi_vec4<S>(av[k], use_res ? resv[k] : v4f{0.f, 0.f, 0.f, 0.f}, L, EpiAtSplit{uni, lane_off + it * it_step}, e);
        }
      }
    }
  };
  // wave-uniform: the whole TM*32 x WN tile inside the matrix?
  if (FAST_PATH && m_w + TM * 32 <= p.M && n_w + WN <= p.N) tile(std::true_type{});
  else tile(std::false_type{});
}

// Vector epilogue of one wave whose residual comes from a second set of accumulators (same tile,
// same layout) instead of memory: both sets go through the wave's staging area, the shortcut's first.
template <int TM, int TN, int EPI>
__device__ __forceinline__ void igemm_epilogue_dual(v16i (&acc)[TM][TN], v16i (&acc_sc)[TM][TN], int *stage, int64_t m_w,
                                                    int n_w, int lane, const IgemmParams &p, const EpiDev &e,
                                                    const ShortcutDev &sc) {
  typedef typename EpiOf<EPI>::type S;
  static_assert(EPI != EPI_SCALAR, "the two-branch epilogue is the vector one");
  constexpr int WN = TN * 32;
  constexpr int EPI_STRIDE = WN + 8;
  const int frow = lane & 31, fhalf = lane >> 5;
  constexpr int CPR = WN / 4;
  constexpr int RPI = 64 / CPR;
  const int cg = lane % CPR, rsub = lane / CPR;
  const int n = n_w + cg * 4;
  const bool n_ok = n < p.N;
  EpiLane L = epi_lane_setup<S>(n, n_ok, e);
  L.use_res = true;
  L.res_after = e.resid_after != 0;
  EpiDev e_sc = {};
  e_sc.exp2 = sc.exp2; e_sc.chan_div = sc.chan_div; e_sc.chan_rcp = sc.chan_rcp; e_sc.bias = sc.bias;
  const EpiLane L_sc = epi_lane_setup<EpiGeneric>(n, n_ok, e_sc);
  const unsigned lane_off = (unsigned)rsub * (unsigned)out_ld(p) + (unsigned)(cg * 4);
  const unsigned it_step = (unsigned)RPI * (unsigned)out_ld(p);
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    // shortcut sums -> fp32 residual values in the row-major layout of the stores
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        stage[(8 * (r >> 2) + 4 * fhalf + (r & 3)) * EPI_STRIDE + j * 32 + frow] = acc_sc[i][j][r];
    v4f resv[32 / RPI];
#pragma unroll
    for (int it = 0; it < 32 / RPI; ++it) {
      const v4i a = *reinterpret_cast<const v4i *>(stage + (it * RPI + rsub) * EPI_STRIDE + cg * 4);
#pragma unroll
      for (int t = 0; t < 4; ++t) resv[it][t] = epi_dequant1((float)a[t], t, L_sc, sc.exp2);
    }
    // the wave's LDS operations complete in order: these stores cannot overtake the reads above
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        stage[(8 * (r >> 2) + 4 * fhalf + (r & 3)) * EPI_STRIDE + j * 32 + frow] = acc[i][j][r];
    const int64_t uni = (m_w + i * 32) * (int64_t)out_ld(p) + n_w;
    const int64_t left = p.M - (m_w + i * 32);
    const int rows = left < 0 ? 0 : (left > 32 ? 32 : (int)left);
    v4i av[32 / RPI];
#pragma unroll
    for (int it = 0; it < 32 / RPI; ++it)
      av[it] = *reinterpret_cast<const v4i *>(stage + (it * RPI + rsub) * EPI_STRIDE + cg * 4);
#pragma unroll
    for (int it = 0; it < 32 / RPI; ++it) {
      if (!n_ok || it * RPI + rsub >= rows) continue;
      epi_vec4<S>(av[it], resv[it], L, EpiAtSplit{uni, lane_off + it * it_step}, e);
    }
  }
}

// Epilogue of one wave.  acc[i][j] is the 32x32 accumulator of rows m_w + i*32 .., columns
// n_w + j*32 ..; stage is this wave's private LDS area of 32 * (TN*32 + 8) ints.
template <int TM, int TN, int EPI, int BATCHES = 1>
__device__ __forceinline__ void igemm_epilogue(v16i (&acc)[TM][TN], int *stage, int64_t m_w, int n_w, int lane,
                                               const IgemmParams &p, const EpiDev &e) {
  typedef typename EpiOf<EPI>::type S;
  const int frow = lane & 31, fhalf = lane >> 5;
  if constexpr (EPI == EPI_SCALAR) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = n_w + j * 32 + frow;
        if (n >= p.N) continue;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int64_t m = m_w + i * 32 + 8 * (r >> 2) + 4 * fhalf + (r & 3);
          if (m >= p.M) continue;
          const int64_t idx = m * out_ld(p) + n;
          const int a = acc[i][j][r];
          if (e.acc_out) e.acc_out[idx] = a;
          epi_store(epi_value((float)a, idx, n, e), idx, e);
        }
      }
    }
  } else {
    const int n = epi_lane_channel<TN>(n_w, lane);
    const EpiLane L = epi_lane_setup<S>(n, n < p.N, e);
    igemm_epilogue_vec<TM, TN, EPI, true, BATCHES>(acc, stage, m_w, n_w, lane, p, e, L);
  }
}

// Epilogue of one wave for rows of any length and alignment, through the wave's staging area (32 * (TN*32 + 8) ints): a lane
// keeps its columns, so their constants are read once and a store is a run of a row.  The loop is rolled: straight-line code
// for every accumulator, as EPI_SCALAR has it above, is 30 KB of divisions and branches that a short launch waits for
// (1089 x 16 -> 126 in one launch 16.0 us with it).
template <int TM, int TN>
__device__ __forceinline__ void igemm_epilogue_columns(v16i (&acc)[TM][TN], int *stage, int64_t m_w, int n_w, int lane,
                                                       const IgemmParams &p, const EpiDev &e) {
  constexpr int WN = TN * 32, EPI_STRIDE = WN + 8;
  constexpr int LC = WN < 64 ? WN : 64, RPI = 64 / LC;  // lanes along a row, rows a wave handles at once
  const int frow = lane & 31, fhalf = lane >> 5;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    // wave-private staging: stores then loads of the same wave, ordered by the LDS counter
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        stage[(8 * (r >> 2) + 4 * fhalf + (r & 3)) * EPI_STRIDE + j * 32 + frow] = acc[i][j][r];
    const int64_t left = p.M - (m_w + i * 32);
    const int rows = left < 0 ? 0 : (left > 32 ? 32 : (int)left);
#pragma unroll 1
    for (int c = lane % LC; c < WN; c += LC) {
      const int n = n_w + c;
      if (n >= p.N) break;
      const EpiColumn k = epi_column(e, n);
#pragma unroll 2
      for (int row = lane / LC; row < rows; row += RPI) {
        const int a = stage[row * EPI_STRIDE + c];
        const int64_t idx = (m_w + i * 32 + row) * out_ld(p) + n;
        if (e.acc_out) e.acc_out[idx] = a;
        epi_store(epi_value((float)a, idx, k, e), idx, e);
      }
    }
  }
}

// Epilogue of one wave for floating rows of any length and alignment (ragged_epilogue) through the wave's staging area, four columns a
// lane: the vector epilogue's arithmetic on constants read one by one, stores that take any element's alignment.
template <int TM, int TN, int EPI>
__device__ __forceinline__ void igemm_epilogue_ragged(v16i (&acc)[TM][TN], int *stage, int64_t m_w, int n_w, int lane,
                                                      const IgemmParams &p, const EpiDev &e) {
  typedef typename EpiOf<EPI>::type S;
  constexpr int WN = TN * 32, EPI_STRIDE = WN + 8, CPR = WN / 4, RPI = 64 / CPR, NIT = 32 / RPI, BATCH = NIT < 4 ? NIT : 4;
  const int frow = lane & 31, fhalf = lane >> 5, cg = lane % CPR, rsub = lane / CPR;
  const int n = n_w + cg * 4;
  const bool n_ok = n < p.N;
  const EpiLane L = epi_lane_setup_ragged<S>(n_ok ? n : 0, p.N, e);
  const v4f none = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    // wave-private staging: stores then loads of the same wave, ordered by the LDS counter
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        stage[(8 * (r >> 2) + 4 * fhalf + (r & 3)) * EPI_STRIDE + j * 32 + frow] = acc[i][j][r];
    const int64_t left = p.M - (m_w + i * 32);
    const int rows = !n_ok || left < 0 ? 0 : (left > 32 ? 32 : (int)left);
#pragma unroll 1
    for (int it = 0; it < NIT; it += BATCH) {
      v4i av[BATCH];
#pragma unroll
      for (int b = 0; b < BATCH; ++b) av[b] = *reinterpret_cast<const v4i *>(stage + ((it + b) * RPI + rsub) * EPI_STRIDE + cg * 4);
#pragma unroll
      for (int b = 0; b < BATCH; ++b) {
        const int row = (it + b) * RPI + rsub;
        if (row < rows) epi_vec4<S>(av[b], none, L, EpiAtRagged{(m_w + i * 32 + row) * out_ld(p) + n, p.N - n}, e);
      }
    }
  }
}

// EPI_SCALAR of the tiled kernels: any length and alignment, the rule's choice first.  (Straight from the accumulators, one element at
// a time, 8127 x 1742 -> 1747 took 110 us where 1748 columns took 34.)
template <int TM, int TN>
__device__ __forceinline__ void igemm_epilogue_any(v16i (&acc)[TM][TN], int *stage, int64_t m_w, int n_w, int lane, const IgemmParams &p,
                                                   const EpiDev &e) {
  switch (p.ragged) {
    case EPI_Y32: igemm_epilogue_ragged<TM, TN, EPI_Y32>(acc, stage, m_w, n_w, lane, p, e); break;
    case EPI_Y16: igemm_epilogue_ragged<TM, TN, EPI_Y16>(acc, stage, m_w, n_w, lane, p, e); break;
    case EPI_Y16_STEPS: igemm_epilogue_ragged<TM, TN, EPI_Y16_STEPS>(acc, stage, m_w, n_w, lane, p, e); break;
    default: igemm_epilogue_columns<TM, TN>(acc, stage, m_w, n_w, lane, p, e); break;
  }
}

// 16 consecutive int16 (two 16-byte chunks) -> their high bytes and their biased low bytes
__device__ __forceinline__ void split_i16(const v4i c0, const v4i c1, v4i &hi, v4i &lo) {
  hi[0] = (int)__builtin_amdgcn_perm((unsigned)c0[1], (unsigned)c0[0], 0x07050301u);
  hi[1] = (int)__builtin_amdgcn_perm((unsigned)c0[3], (unsigned)c0[2], 0x07050301u);
  hi[2] = (int)__builtin_amdgcn_perm((unsigned)c1[1], (unsigned)c1[0], 0x07050301u);
  hi[3] = (int)__builtin_amdgcn_perm((unsigned)c1[3], (unsigned)c1[2], 0x07050301u);
  lo[0] = (int)(__builtin_amdgcn_perm((unsigned)c0[1], (unsigned)c0[0], 0x06040200u) ^ 0x80808080u);
  lo[1] = (int)(__builtin_amdgcn_perm((unsigned)c0[3], (unsigned)c0[2], 0x06040200u) ^ 0x80808080u);
  lo[2] = (int)(__builtin_amdgcn_perm((unsigned)c1[1], (unsigned)c1[0], 0x06040200u) ^ 0x80808080u);
  lo[3] = (int)(__builtin_amdgcn_perm((unsigned)c1[3], (unsigned)c1[2], 0x06040200u) ^ 0x80808080u);
}

// type of the activations a contraction reads: int8, or floats that its loader quantizes
enum { IN_I8 = 0, IN_F32 = 1, IN_F16 = 2 };

// 16 floats (or halfs) -> 16 int8, the quantizer's own arithmetic with unit scale
template <int IN>
__device__ __forceinline__ v4i quantize16(const v4i *raw, int neg_pos) {
  v4i q;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    int b[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      float v;
      if constexpr (IN == IN_F32) v = __int_as_float(raw[d][t]);
      else {
        const int pair = raw[d >> 1][(d & 1) * 2 + (t >> 1)];
        v = (float)__builtin_bit_cast(_Float16, (short)((t & 1) ? pair >> 16 : pair & 0xffff));
      }
      b[t] = quant1_unit<8>(v, neg_pos);
    }
    const unsigned lo = __builtin_amdgcn_perm((unsigned)b[1], (unsigned)b[0], 0x0c0c0400u);
    const unsigned hi = __builtin_amdgcn_perm((unsigned)b[3], (unsigned)b[2], 0x04000c0cu);
    q[d] = (int)(lo | hi);
  }
  return q;
}

// What the kernels of few output tiles (small_i8.hip, wide_i16.hip) read beyond that: halfs whose rows start on any element, and
// floats or halfs whose channels lie `chan_bytes` apart (NCHW).
enum { IN_F16_ANY = 3, IN_F32_APART = 4, IN_F16_APART = 5 };
constexpr bool in_apart(int in) { return in == IN_F32_APART || in == IN_F16_APART; }
constexpr int in_bytes(int in) { return in == IN_I8 ? 1 : (in == IN_F32 || in == IN_F32_APART ? 4 : 2); }
// loads per V values, and the dwords that hold them
constexpr int in_loads(int in, int v) { return in_apart(in) ? v : in == IN_F16_ANY ? v / 8 + 1 : v * in_bytes(in) / 16; }
constexpr int in_dwords(int in, int v) { return in_apart(in) ? v : in == IN_F16_ANY ? v / 2 + 1 : v * in_bytes(in) / 4; }

// V values from byte `off` of a buffer on; an offset past its end gives zeros.
template <int IN, int V>
struct FloatPiece {
  int d[in_dwords(IN, V)];
  unsigned shift;  // IN_F16_ANY: bits in front of the first value
  __device__ __forceinline__ void load(const __amdgpu_buffer_rsrc_t rsrc, unsigned off, unsigned chan_bytes) {
    if constexpr (in_apart(IN)) {
#pragma unroll
      for (int i = 0; i < V; ++i) {
        const int at = (int)(off + (unsigned)i * chan_bytes);
        if constexpr (IN == IN_F32_APART) d[i] = (int)__builtin_amdgcn_raw_buffer_load_b32(rsrc, at, 0, 0);
        else d[i] = (int)__builtin_amdgcn_raw_buffer_load_b16(rsrc, at, 0, 0);
      }
    } else {
      constexpr int WIDE = in_dwords(IN, V) / 4;
      if constexpr (IN == IN_F16_ANY) {  // whole dwords around the values
        shift = (off & 2u) * 8u;
        off &= ~3u;
        d[4 * WIDE] = (int)__builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)off + 16 * WIDE, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < WIDE; ++r) {
        const v4i t = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)off + 16 * r, 0, 0));
#pragma unroll
        for (int u = 0; u < 4; ++u) d[4 * r + u] = t[u];
      }
    }
  }
  __device__ __forceinline__ float value(int i) const {
    if constexpr (IN == IN_F32 || IN == IN_F32_APART) return __int_as_float(d[i]);
    else if constexpr (IN == IN_F16_APART) return (float)__builtin_bit_cast(_Float16, (short)d[i]);
    else {
      int pair = d[i / 2];
      if constexpr (IN == IN_F16_ANY) pair = (int)__builtin_amdgcn_alignbit((unsigned)d[i / 2 + 1], (unsigned)d[i / 2], shift);
      return (float)__builtin_bit_cast(_Float16, (short)((i & 1) ? pair >> 16 : pair & 0xffff));
    }
  }
};

// 16 values -> 16 int8, 8 values -> 8 int16: the quantizer's own arithmetic with unit scale
template <int IN>
__device__ __forceinline__ v4i quantize_piece(const FloatPiece<IN, 16> &p, int neg_pos) {
  v4i q;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    int b[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) b[t] = quant1_unit<8>(p.value(4 * d + t), neg_pos);
    const unsigned lo = __builtin_amdgcn_perm((unsigned)b[1], (unsigned)b[0], 0x0c0c0400u);
    const unsigned hi = __builtin_amdgcn_perm((unsigned)b[3], (unsigned)b[2], 0x04000c0cu);
    q[d] = (int)(lo | hi);
  }
  return q;
}
template <int IN>
__device__ __forceinline__ v4i quantize_piece(const FloatPiece<IN, 8> &p, int neg_pos) {
  v4i q;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const int a = cvt_i32_sat(__builtin_rintf(__builtin_ldexpf(p.value(2 * d), neg_pos)));
    const int b = cvt_i32_sat(__builtin_rintf(__builtin_ldexpf(p.value(2 * d + 1), neg_pos)));
    q[d] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_pk_i16(a, b));  // (saturates)
  }
  return q;
}

// launchers of the LDS-DMA pipelined kernel (igemm_i8_dma.hip); return -1 when the shape is not
// eligible (operand of 2 GiB or more, four-channel stem) and the caller takes the register-staged kernel
int igemm_dma_launch(int load, const void *a, const void *b, IgemmParams p, const EpiDev &e, int64_t a_bytes,
                     int64_t b_bytes, hipStream_t s);


}  // namespace catchq
