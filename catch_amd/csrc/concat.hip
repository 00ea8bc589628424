// Channel concatenation of quantized NHWC tensors, with what usually stands in front of it folded in: a source may be
// upsampled (nearest neighbour, factor two) or still be in fp32 and quantized on the way.
//
// Pure traffic: what bounds it is HBM.  As separate operations a detector's route pays for every one of them -- two
// repetitions along the axes, a quantizer and the concatenation move each byte two to four times in launches that the small
// grids do not fill: for 16 images of 416 x 416 (Darknet-53 with YOLOv3 heads, int16) 42.5 us in front of the 26 x 26 head
// and 64.9 us in front of the 52 x 52 one, for 41 and 80 MB that cannot be avoided (the whole network in two parts: 2397 ->
// 2356 us with one launch for each).
#include "catchq_common.h"

namespace catchq {

struct ConcatSource {
  const void *x;
  int kind;    // CATCHQ_CONCAT_*
  int chunk0;  // first 16-byte piece of the output pixel that comes from it, and the piece behind its last one
  int chunk1;
};
struct ConcatArgs {
  ConcatSource src[CATCHQ_CONCAT_MAX];
  int n;
  int chunks;         // 16-byte pieces of an output pixel
  int H, W;
  unsigned pieces;    // of the whole output
  unsigned per_block; // pieces of a block
  int neg_pos;
  float scale;
};

// One 16-byte piece of the output per lane and turn: neighbouring lanes hold neighbouring pieces of a pixel.  ES: bytes per
// output element.
template <int ES>
__global__ __launch_bounds__(256) void concat_kernel(ConcatArgs a, v4i *__restrict__ out) {
  constexpr int EPP = 16 / ES;  // elements of a piece
  const unsigned end = min((blockIdx.x + 1u) * a.per_block, a.pieces);
  for (unsigned i = blockIdx.x * a.per_block + threadIdx.x; i < end; i += 256) {
    const unsigned px = i / (unsigned)a.chunks;
    const int c = (int)(i - px * (unsigned)a.chunks);
    ConcatSource s = a.src[0];
#pragma unroll
    for (int k = 1; k < CATCHQ_CONCAT_MAX; ++k)
      if (k < a.n && c >= a.src[k].chunk0) s = a.src[k];
    const int own = s.chunk1 - s.chunk0;
    v4i v;
    if (s.kind == CATCHQ_CONCAT_FLOAT) {
      const v4f *f = reinterpret_cast<const v4f *>(s.x) + ((int64_t)px * own + (c - s.chunk0)) * (EPP / 4);
      v4f x[EPP / 4];
#pragma unroll
      for (int k = 0; k < EPP / 4; ++k) x[k] = f[k];
      if constexpr (ES == 2) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int lo = quant1<16>(x[k >> 1][2 * (k & 1)], a.scale, a.neg_pos), hi = quant1<16>(x[k >> 1][2 * (k & 1) + 1], a.scale, a.neg_pos);
          v[k] = (lo & 0xffff) | (hi << 16);
        }
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          int b[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) b[j] = quant1<8>(x[k][j], a.scale, a.neg_pos);
          v[k] = (b[0] & 0xff) | ((b[1] & 0xff) << 8) | ((b[2] & 0xff) << 16) | (b[3] << 24);
        }
      }
    } else {
      unsigned from = px;
      if (s.kind == CATCHQ_CONCAT_UP2) {
        const unsigned row = px / (unsigned)a.W, w = px - row * (unsigned)a.W;  // row: image * H + h, and H is even
        from = (row >> 1) * ((unsigned)a.W >> 1) + (w >> 1);
      }
      v = reinterpret_cast<const v4i *>(s.x)[(int64_t)from * own + (c - s.chunk0)];
    }
    out[i] = v;
  }
}

}  // namespace catchq

using namespace catchq;

CATCHQ_API int catchq_concat_nhwc(const catchq_concat_source_t *sources, int nsources, int bitwidth, int position, float scale,
                                  int n, int h, int w, void *out, catchq_stream_t stream) {
  if (!sources || nsources <= 0 || n < 0 || h <= 0 || w <= 0) return CATCHQ_ERR_ARG;
  if (bitwidth != 8 && bitwidth != 16) return CATCHQ_ERR_BITWIDTH;
  if (position < -126 || position > 126) return CATCHQ_ERR_ARG;
  if (nsources > CATCHQ_CONCAT_MAX) return CATCHQ_ERR_UNSUPPORTED;
  const int per = 128 / bitwidth;
  ConcatArgs a = {};
  for (int i = 0; i < nsources; ++i) {
    const catchq_concat_source_t &s = sources[i];
    if (s.channels <= 0 || s.kind < CATCHQ_CONCAT_COPY || s.kind > CATCHQ_CONCAT_FLOAT) return CATCHQ_ERR_ARG;
    if (n > 0 && !s.x) return CATCHQ_ERR_ARG;
    if (s.channels % per != 0 || !aligned16(s.x)) return CATCHQ_ERR_UNSUPPORTED;
    if (s.kind == CATCHQ_CONCAT_UP2 && (h % 2 != 0 || w % 2 != 0)) return CATCHQ_ERR_SHAPE;
    if (s.channels > (1 << 24) || a.chunks > (1 << 24)) return CATCHQ_ERR_UNSUPPORTED;
    a.src[i] = {s.x, s.kind, a.chunks, a.chunks + s.channels / per};
    a.chunks += s.channels / per;
  }
  if (n == 0) return CATCHQ_OK;
  if (!out) return CATCHQ_ERR_ARG;
  const int64_t pixels = (int64_t)n * h * w;
  if (!aligned16(out) || pixels >= (1ll << 31) || pixels * a.chunks >= (1ll << 31)) return CATCHQ_ERR_UNSUPPORTED;
  a.n = nsources; a.H = h; a.W = w;
  a.pieces = (unsigned)(pixels * a.chunks);
  a.neg_pos = -position; a.scale = scale;
  // four turns of a block, fewer where that would leave compute units without one
  unsigned turns = a.pieces / (256u * 2048u);
  turns = turns < 1 ? 1 : (turns > 4 ? 4 : turns);
  a.per_block = 256 * turns;
  const unsigned blocks = (a.pieces + a.per_block - 1) / a.per_block;
  if (bitwidth == 8) concat_kernel<1><<<blocks, 256, 0, as_stream(stream)>>>(a, (v4i *)out);
  else concat_kernel<2><<<blocks, 256, 0, as_stream(stream)>>>(a, (v4i *)out);
  return launch_status();
}
