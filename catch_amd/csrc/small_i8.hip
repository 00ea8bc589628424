// int8 contractions of few output tiles: the K loop split over the waves of a block, no barrier inside it.
//
// What bounds such a launch (one image through a late layer, a few tokens through a linear): the tiled kernels give it
// a handful of blocks, each a serial chain of K steps with a barrier and a memory latency per step -- 256 channels of a
// 3x3 layer on one 14 x 14 image took 8.6 us on 8 blocks, 512 channels on 7 x 7 11.1 us on 16, where all of the
// operands fit one microsecond of L2 traffic.  Here a block owns one tile of T x T outputs (T = 32 or 16: the smallest
// that fills the device once) and its NW waves take a contiguous slice of K each: a wave's transfers (LDS-DMA, whole
// 128-byte lines, two 128-byte K steps in flight per wave) go to a slice of LDS of its own, so it waits for nothing but
// its own loads; the partial sums meet in LDS once, behind the loop, and every output is finished by the epilogue code
// of the other kernels.  Residual and per-channel constants are requested before the first K step.
#include <type_traits>

#include "igemm_common.h"

namespace catchq {

typedef __attribute__((address_space(3))) void *lds_ptr_t;

// One contraction: activations [.., H, W, Ci] (int8, or floats that the loader quantizes) against filters [N][K]
struct SmallSide {
  const void *x;
  const int8_t *w;
  int K;             // kh * kw * Ci < 2^20
  int H, W, Ci, kw, ph, pw, sh, sw, dh, dw;  // Ci: channels of the filters; where the activations have fewer, those beyond read
                                             // whatever lies there, against zeros
  unsigned img_stride, row_stride, pix_stride;  // elements
  unsigned magic_ci, magic_kw, mask_ci, mask_kw;  // ceil(2^32 / d), mask 0; for d = 1 magic 0, mask ~0
  unsigned a_bytes, b_bytes;
};

struct SmallParams {
  SmallSide side[2];  // [1]: the projection shortcut of a two-branch launch
  int M, N;           // M < 2^20
  int Ho, Wo;
  unsigned magic_wo, magic_ho, magic_t, mask_wo, mask_ho, mask_t;
  int tiles_m, tiles_n, nblocks;
  int m_fastest;      // consecutive blocks walk the row tiles of one column tile first
  int epi;            // epilogue variant (EPI_*), the same for every block
  int main_waves;     // two-branch launches: waves 0 .. main_waves - 1 run side 0, the others side 1
  int x_neg_pos;      // floating activations: quantized at 2^-x_neg_pos
  ShortcutDev sc;
};

#define CATCHQ_SMALL_VMCNT(n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(n) : "memory")

// n / d for n * d < 2^32 through magic = ceil(2^32 / d) (d = 1: magic 0, mask ~0)
__device__ __forceinline__ unsigned div_magic(unsigned n, unsigned magic, unsigned mask) { return __umulhi(n, magic) + (n & mask); }

__device__ __forceinline__ v4i small_ds_read(unsigned addr) {
  v4i v;
  asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(addr));
  return v;
}
__device__ __forceinline__ void small_ds_write(unsigned addr, v4i v) {
  asm volatile("ds_write_b128 %0, %1" ::"v"(addr), "v"(v) : "memory");
}

// DENSE: a plain GEMM -- row m starts at m * pix_stride (the channels of the activations, which may be fewer than K), no taps.  IN: type of the activations.  DUAL: a residual block's last
// convolution and its projection shortcut over the same output tile; the block's waves are shared out between the two
// in proportion to their K steps, and the shortcut's sums, dequantized with its own constants, are the residual.
// HALF_BIAS: there is a bias, in half precision (a choice at run time costs every launch 0.05 us).
template <int T, int NW, bool DENSE, int IN, bool DUAL, bool HALF_BIAS>
__global__ __launch_bounds__(64 * NW) void small_i8_kernel(SmallParams p, EpiDev e) {
  fetch_arguments<sizeof(SmallParams) + sizeof(EpiDev)>();
  resolve_exp2(e);
  constexpr int SLOTS = 2, BKB = 128;
  constexpr int SLOT_BYTES = 2 * T * BKB, WAVE_BYTES = SLOTS * SLOT_BYTES;
  constexpr int NA = T / 8, NI = 2 * NA;   // DMA instructions (8 rows of 128 bytes each) per K step
  constexpr int SUB = T == 32 ? 4 : 2;     // matrix instructions per K step: 32 x 32 x 32 or 16 x 16 x 64
  constexpr int PITCH = T + 4;             // ints per pixel of a partial tile
  static_assert(T * PITCH * 4 <= WAVE_BYTES, "a partial tile fits the wave's slots");
  extern __shared__ __attribute__((aligned(16))) int8_t lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int logical = xcd_remap(blockIdx.x, p.nblocks);
  const int outer = (int)div_magic((unsigned)logical, p.magic_t, p.mask_t);
  const int inner = logical - outer * (p.m_fastest ? p.tiles_m : p.tiles_n);
  const int tile_m = p.m_fastest ? inner : outer, tile_n = p.m_fastest ? outer : inner;
  const int m0 = tile_m * T, n0 = tile_n * T;
  const bool second = DUAL && wave >= p.main_waves;  // wave-uniform
  const SmallSide &o = p.side[second ? 1 : 0];
  const int group_wave = second ? wave - p.main_waves : wave;
  const int group = DUAL ? (second ? NW - p.main_waves : p.main_waves) : NW;
  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void *)o.x, 0, (int)o.a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void *)o.w, 0, (int)o.b_bytes, 0x00020000);
  constexpr unsigned OOB = 0x80000000u;  // the hardware answers an offset beyond the buffer with zeros

  // the epilogue's lanes: four channels of one pixel each, T * T / 4 of them (waves 0 ..)
  constexpr int EPI_LANES = T * T / 4, CPR = T / 4;
  const bool epi_wave = wave * 64 < EPI_LANES;
  const bool vec = p.epi != EPI_SCALAR;
  constexpr int ROUNDS = (EPI_LANES + 64 * NW - 1) / (64 * NW);
  v4f c_div = {1.f, 1.f, 1.f, 1.f}, c_rcp = c_div, c_res[ROUNDS];
  v4f c_bias = {-0.f, -0.f, -0.f, -0.f};
  v2i c_bias16 = {0, 0};  // (converted behind the K loop: here the conversion would wait for the load)
  v4f s_div = c_div, s_rcp = c_div, s_bias = {0.f, 0.f, 0.f, 0.f};  // the shortcut's constants
  // 64 * NW is a multiple of CPR: a lane has the same four channels in every round.  (Plain loads: the transfers below
  // and the statements that clobber memory keep them here, in front of the K loop.)
  const int ec = n0 + (threadIdx.x % CPR) * 4;
  if (epi_wave && vec) {
    const int cc = min(ec, p.N - 4);
    if (e.chan_div) c_div = *reinterpret_cast<const v4f *>(e.chan_div + cc);
    const float *rcps = e.chan_rcp ? e.chan_rcp : e.half_rcp;
    if (rcps) c_rcp = *reinterpret_cast<const v4f *>(rcps + cc);
    if constexpr (HALF_BIAS) c_bias16 = *reinterpret_cast<const v2i *>(reinterpret_cast<const __half *>(e.bias) + cc);
    else if (e.bias) c_bias = *reinterpret_cast<const v4f *>(e.bias + cc);
    if constexpr (DUAL) {
      if (p.sc.chan_div) s_div = *reinterpret_cast<const v4f *>(p.sc.chan_div + cc);
      if (p.sc.chan_rcp) s_rcp = *reinterpret_cast<const v4f *>(p.sc.chan_rcp + cc);
      if (p.sc.bias) s_bias = *reinterpret_cast<const v4f *>(p.sc.bias + cc);
    }
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
      c_res[r] = v4f{0.f, 0.f, 0.f, 0.f};
      const int em = min(m0 + (int)(threadIdx.x + r * 64 * NW) / CPR, p.M - 1);
      if (!DUAL && e.resid) c_res[r] = *reinterpret_cast<const v4f *>(e.resid + (int64_t)em * p.N + cc);
    }
  }

  // ---- loader ------------------------------------------------------------------------------------------------------
  // A DMA instruction fills 8 rows of 128 bytes: lane l writes 16-byte piece l & 7 of row l >> 3.  It fetches the piece
  // (l & 7) ^ ((row >> 1) & 7) of that row, so that the 16-byte fragment reads of 16 consecutive rows fall into 16
  // different pieces of a 256-byte LDS line; row = 8 j + (l >> 3), so even and odd j differ in bit 2 of the piece.
  const int lrow = lane >> 3;
  const int chunk0 = (lane & 7) ^ (lane >> 4);
  unsigned a_base[NA], b_base[NA];
  int a_hi[NA], a_wi[NA];
#pragma unroll
  for (int j = 0; j < NA; ++j) {
    const int m = m0 + j * 8 + lrow;
    if constexpr (DENSE) {
      a_hi[j] = a_wi[j] = 0;
      a_base[j] = m < p.M ? (unsigned)m * o.pix_stride : OOB;
    } else {
      const unsigned t = div_magic((unsigned)m, p.magic_wo, p.mask_wo), wo = (unsigned)m - t * (unsigned)p.Wo;
      const unsigned img = div_magic(t, p.magic_ho, p.mask_ho), ho = t - img * (unsigned)p.Ho;
      a_hi[j] = m < p.M ? (int)ho * o.sh - o.ph : -(1 << 30);  // a row that does not exist is outside the image
      a_wi[j] = (int)wo * o.sw - o.pw;
      a_base[j] = img * o.img_stride + (unsigned)a_hi[j] * o.row_stride + (unsigned)a_wi[j] * o.pix_stride;  // mod 2^32
    }
    const int n = n0 + j * 8 + lrow;
    b_base[j] = n < p.N ? (unsigned)n * (unsigned)o.K : OOB;
  }
  const int steps = (o.K + BKB - 1) / BKB;
  const int per = steps / group, rem = steps - per * group;
  const int first = group_wave * per + (group_wave < rem ? group_wave : rem);
  const int mine = per + (group_wave < rem ? 1 : 0);
  int8_t *const my = lds + wave * WAVE_BYTES;

  constexpr int ES = in_bytes(IN);          // bytes per activation
  constexpr int RAW = in_loads(IN, 16);     // loads per 16 activations
  FloatPiece<IN, 16> raw[NA];
  (void)raw;
  const unsigned chan_stride = in_apart(IN) ? (unsigned)(o.H * o.W) : 1u;
  auto issue = [&](int s) {  // step s of this wave's slice into its slot s & 1 (floating activations: into raw)
    const int slot = (s & 1) * SLOT_BYTES;
    unsigned k[2], koff[2];
    int dy[2], dx[2];
    bool ok[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      k[h] = (unsigned)((first + s) * BKB + (chunk0 ^ (4 * h)) * 16);
      ok[h] = k[h] < (unsigned)o.K;
      koff[h] = k[h];
      dy[h] = dx[h] = 0;
      if constexpr (!DENSE) {
        const unsigned tap = div_magic(k[h], o.magic_ci, o.mask_ci), ci = k[h] - tap * (unsigned)o.Ci;
        const unsigned r = div_magic(tap, o.magic_kw, o.mask_kw), q = tap - r * (unsigned)o.kw;
        dy[h] = (int)r * o.dh;
        dx[h] = (int)q * o.dw;
        koff[h] = (unsigned)dy[h] * o.row_stride + (unsigned)dx[h] * o.pix_stride + ci * chan_stride;
      }
    }
    // (the filters first: loads complete in order, so a wave that has its activations has its filters)
#pragma unroll
    for (int j = 0; j < NA; ++j) {
      const int h = j & 1;
      unsigned voff = ok[h] ? b_base[j] + k[h] : OOB;
      asm volatile("" : "+v"(voff));  // one select and one load, not two loads under complementary masks
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, (lds_ptr_t)(my + slot + (NA + j) * 1024), 16, (int)voff, 0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < NA; ++j) {
      const int h = j & 1;
      bool in = ok[h];
      if constexpr (!DENSE)
        in = in & ((unsigned)(a_hi[j] + dy[h]) < (unsigned)o.H) & ((unsigned)(a_wi[j] + dx[h]) < (unsigned)o.W);
      if constexpr (DENSE) in = in & (a_base[j] != OOB);
      unsigned voff = in ? (a_base[j] + koff[h]) * (unsigned)ES : OOB;
      asm volatile("" : "+v"(voff));
      if constexpr (IN == IN_I8) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_ptr_t)(my + slot + j * 1024), 16, (int)voff, 0, 0, 0);
      } else {
        raw[j].load(rsrc_a, voff, chan_stride * (unsigned)ES);
      }
    }
  };

  // ---- K loop: this wave's slice -------------------------------------------------------------------------------------
  typedef typename std::conditional<T == 32, v16i, v4i>::type acc_t;
  acc_t acc = {};
  if (mine > 0) {
    const int frow = lane & (T - 1), fk = lane / T;  // row of the fragment, 16-byte piece within a sub-step
    const unsigned my_addr = (unsigned)(uintptr_t)(__attribute__((address_space(3))) int8_t *)my;
    const unsigned a_addr = my_addr + (unsigned)(frow * BKB);
    const unsigned sw = (unsigned)((frow >> 1) & 7);
    issue(0);
    if (IN == IN_I8 && mine > 1) issue(1);
    for (int s = 0; s < mine; ++s) {
      if constexpr (IN == IN_I8) {
        if (s + 1 < mine) CATCHQ_SMALL_VMCNT(NI);
        else CATCHQ_SMALL_VMCNT(0);
      } else {
        // the step's activations have arrived, and with them its filters: quantized into the slot, as a transfer
        // would have left them; then the next step's loads
        v4i q[NA];
#pragma unroll
        for (int j = 0; j < NA; ++j) q[j] = quantize_piece<IN>(raw[j], p.x_neg_pos);
#pragma unroll
        for (int j = 0; j < NA; ++j)
          small_ds_write(my_addr + (unsigned)((s & 1) * SLOT_BYTES + j * 1024 + lane * 16), q[j]);
        if (s + 1 < mine) {
          issue(s + 1);
          CATCHQ_SMALL_VMCNT(NA + NA * RAW < 63 ? NA + NA * RAW : 63);  // (what the counter holds)
        } else {
          CATCHQ_SMALL_VMCNT(0);
        }
      }
      const unsigned base = a_addr + (unsigned)((s & 1) * SLOT_BYTES);
      v4i fa[SUB], fb[SUB];
#pragma unroll
      for (int u = 0; u < SUB; ++u) {
        const unsigned piece = (((unsigned)(u * (64 / T) + fk)) ^ sw) * 16;
        fa[u] = small_ds_read(base + piece);
        fb[u] = small_ds_read(base + T * BKB + piece);
      }
#pragma unroll
      for (int u = 0; u < SUB; ++u) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(fa[u]), "+v"(fb[u])::"memory");
      if (IN == IN_I8 && s + 2 < mine) issue(s + 2);  // the slot has been read
      // operands swapped (weights as A): a lane ends up with four consecutive channels of one pixel
#pragma unroll
      for (int u = 0; u < SUB; ++u) {
        if constexpr (T == 32) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb[u], fa[u], acc, 0, 0, 0);
        else acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(fb[u], fa[u], acc, 0, 0, 0);
      }
    }
    int *part = reinterpret_cast<int *>(my) + frow * PITCH + fk * 4;
    if constexpr (T == 32) {
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<v4i *>(part + 8 * g) = v4i{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
    } else {
      *reinterpret_cast<v4i *>(part) = acc;
    }
  }
  if (!epi_wave) {
    __syncthreads();
    return;
  }

  // ---- partial sums -> outputs ---------------------------------------------------------------------------------------
  auto steps_of = [&](int K) { return (K + BKB - 1) / BKB; };
  const int main_group = DUAL ? p.main_waves : NW;
  const int main_active = min(steps_of(p.side[0].K), main_group);
  const int second_active = DUAL ? min(steps_of(p.side[1].K), NW - main_group) : 0;
  // main and shortcut sums of lane t, four channels of a pixel: every wave's slot at once, also of those without a step (one after
  // the other they cost 100 clocks each)
  auto sums_of = [&](int t, v4i &a, v4i &a2) {
    const int *part = reinterpret_cast<const int *>(lds) + t / CPR * PITCH + t % CPR * 4;
    v4i parts[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) parts[w] = *reinterpret_cast<const v4i *>(part + w * (WAVE_BYTES / 4));
    a = a2 = v4i{0, 0, 0, 0};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      if (w < main_active) a += parts[w];
      if (DUAL && w >= main_group && w < main_group + second_active) a2 += parts[w];
    }
  };
  EpiLane ls;  // the shortcut's constants
  if constexpr (DUAL) {
    EpiDev es = {};
    es.exp2 = p.sc.exp2; es.chan_div = p.sc.chan_div; es.chan_rcp = p.sc.chan_rcp; es.bias = p.sc.bias;
    ls = epi_lane_finish<EpiGeneric>(s_div, s_rcp, s_bias, es);
  }
  auto residual = [&](int r, const v4i &a2) {
    v4f res = c_res[r];
    if constexpr (DUAL) {
#pragma unroll
      for (int u = 0; u < 4; ++u) res[u] = epi_dequant1((float)a2[u], u, ls, p.sc.exp2);
    }
    return res;
  };
  auto run = [&](auto spec) {
    typedef decltype(spec) S;
    EpiLane L = epi_lane_finish<S>(c_div, c_rcp, HALF_BIAS ? half4_values(c_bias16) : c_bias, e);  // (in front of the barrier)
    if constexpr (DUAL) {
      L.use_res = true;
      L.res_after = e.resid_after != 0;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
      const int t = threadIdx.x + r * 64 * NW, m = m0 + t / CPR;
      if (t >= EPI_LANES) break;
      v4i a, a2;
      sums_of(t, a, a2);
      if (m < p.M && ec < p.N) epi_vec4<S>(a, residual(r, a2), L, (int64_t)m * p.N + ec, e);
    }
  };
  switch (p.epi) {
    case EPI_Q8_RELU: run(EpiOf<EPI_Q8_RELU>::type{}); break;
    case EPI_RES_Y_Q8: run(EpiOf<EPI_RES_Y_Q8>::type{}); break;
    case EPI_Y32: run(EpiOf<EPI_Y32>::type{}); break;
    case EPI_RES_Q8: run(EpiOf<EPI_RES_Q8>::type{}); break;
    case EPI_Q8_RELU6: run(EpiOf<EPI_Q8_RELU6>::type{}); break;
    case EPI_Y16: run(EpiOf<EPI_Y16>::type{}); break;
    case EPI_Y16_STEPS: run(EpiOf<EPI_Y16_STEPS>::type{}); break;
    case EPI_SCALAR:
      __syncthreads();
#pragma unroll
      for (int r = 0; r < ROUNDS; ++r) {
        const int t = threadIdx.x + r * 64 * NW, m = m0 + t / CPR;
        if (t >= EPI_LANES) break;
        v4i a, a2;
        sums_of(t, a, a2);
        const int64_t idx = (int64_t)m * p.N + ec;
        if (m < p.M) {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            if (ec + u >= p.N) break;
            if (e.acc_out) e.acc_out[idx + u] = a[u];
            epi_store(epi_value((float)a[u], idx + u, ec + u, e), idx + u, e);
          }
        }
      }
      break;
    default: run(EpiGeneric{}); break;
  }
}

static void magic(unsigned d, unsigned *m, unsigned *mask) {
  *m = d <= 1 ? 0u : (unsigned)(((1ull << 32) + d - 1) / d);
  *mask = d <= 1 ? ~0u : 0u;
}

template <int T, int NW, bool DENSE, int IN, bool DUAL, bool HALF_BIAS>
static int launch_small(SmallParams p, const EpiDev &e, hipStream_t s) {
  constexpr int LDS_BYTES = NW * 2 * 2 * T * 128;
  static_assert(LDS_BYTES <= 128 * 1024, "slots of all waves");
  auto kern = small_i8_kernel<T, NW, DENSE, IN, DUAL, HALF_BIAS>;
  if (LDS_BYTES > 64 * 1024) {
    static std::atomic<bool> raised[64];
    if (raise_lds_limit((const void *)kern, LDS_BYTES, raised) != CATCHQ_OK) return CATCHQ_ERR_LAUNCH;
  }
  p.tiles_m = (p.M + T - 1) / T;
  p.tiles_n = (p.N + T - 1) / T;
  p.nblocks = p.tiles_m * p.tiles_n;
  magic(p.m_fastest ? p.tiles_m : p.tiles_n, &p.magic_t, &p.mask_t);
  if (DUAL) {
    const int s1 = (p.side[0].K + 127) / 128, s2 = (p.side[1].K + 127) / 128;
    p.main_waves = (NW * s1 + (s1 + s2) / 2) / (s1 + s2);
    p.main_waves = p.main_waves < 1 ? 1 : (p.main_waves > NW - 1 ? NW - 1 : p.main_waves);
  }
  kern<<<p.nblocks, 64 * NW, LDS_BYTES, s>>>(p, e);
  return launch_status();
}

// One side's constants; false where the kernel's 32-bit arithmetic does not cover the shape.  x_ci: channels of the activations
// (Ci and more of them make no sense), apart: their order is [N, channel, H, W].
static bool small_side(SmallSide *o, const void *x, int x_size, const void *w, int N_img, int H, int W, int Ci, int Co, int kh,
                       int kw, int ph, int pw, int sh, int sw, int dh, int dw, int Ho, int Wo, bool dense, int x_ci, bool apart) {
  const int64_t M = (int64_t)N_img * Ho * Wo, K = (int64_t)kh * kw * Ci;
  const int64_t a_bytes = ((int64_t)N_img * H * W * x_ci * x_size + 3) / 4 * 4, b_bytes = (int64_t)Co * K;  // (whole dwords)
  // (no offset wraps: one past the last channel stays below 2^32, one of 2^31 and a piece's channels behind it too)
  if (apart && (int64_t)H * W * x_size * (Ci - x_ci + 16) >= (1ll << 30)) return false;
  if (Ci % 16 != 0 || x_ci > Ci || M >= (1 << 20) || K >= (1 << 20) || a_bytes >= (1ll << 31) || b_bytes >= (1ll << 31)) return false;
  // the divisions through multiplication: dividend * divisor < 2^32
  if (!dense && (M * Wo >= (1ll << 32) || M * Ho >= (1ll << 32) || K * Ci >= (1ll << 32) || (int64_t)kh * kw * kw >= (1ll << 32) ||
                 (int64_t)dh * kh >= (1 << 20) || (int64_t)dw * kw >= (1 << 20) || H >= (1 << 20) || W >= (1 << 20)))
    return false;
  o->x = x; o->w = (const int8_t *)w;
  o->K = (int)K;
  o->H = H; o->W = W; o->Ci = Ci; o->kw = kw; o->ph = ph; o->pw = pw; o->sh = sh; o->sw = sw; o->dh = dh; o->dw = dw;
  o->img_stride = (unsigned)((int64_t)H * W * x_ci);
  o->row_stride = (unsigned)(apart ? W : (int64_t)W * x_ci);
  o->pix_stride = apart ? 1u : (unsigned)x_ci;
  magic(Ci, &o->magic_ci, &o->mask_ci);
  magic(kw, &o->magic_kw, &o->mask_kw);
  o->a_bytes = (unsigned)a_bytes; o->b_bytes = (unsigned)b_bytes;
  return true;
}

// Tile and waves (T * 100 + NW) for M x N outputs over `steps` 128-byte K steps, 0: not this kernel's shape.
//
// Measured with the launch repeated in a graph (us, this kernel / the tiled ones; MI355X):
//   16 x 16 tiles while the device holds two per compute unit: 7x7 512->512 3x3 4.6 / 10.6, 14x14 256->256 3x3 4.0 / 7.7,
//     14x14/2 512->512 3x3 4.6 / 18.6, 1 x 3072 -> 768 3.4 / 7.0, 1 x 4096 -> 4096 3.8 / 8.5, 6x6x14 960->160 4.0 / 5.0
//   32 x 32 tiles up to one per unit: 784 x 256 x 512 3.4 / 3.7, 4 x 14x14 256->256 3x3 (200 tiles) 5.3 / 7.7
//     (K = 192 ties, K <= 128 loses: those launches are all set-up); to 1.75 per unit from K = 1024 on
//     (4 x 28x28 128->128 3x3, 392 tiles, 5.4 / 6.0; K = 512 loses, 4.3 / 3.7); more for the longest K
//     (197 x 4096 x 4096, 896 tiles, 13.8 / 16.8), up to three per unit where there are more rows (with a quantizer in
//     front: 2048 x 3072 x 384, 768 tiles, 18.4 / 19.4, but 784 x 3072 x 1120, 875 tiles, 18.7 / 17.8 and
//     2048 x 3072 x 416, 832 tiles, 20.5 / 19.7)
// Four waves share K (one wave's transfers and arithmetic run under another's wait; eight cost more set-up than they
// hide), eight where a step's tap arithmetic is long and the blocks do not fill the device.
static int small_plan(int64_t M, int64_t N, int64_t K, bool dense, int cus) {
  const int64_t tiles32 = ((M + 31) / 32) * ((N + 31) / 32), tiles16 = ((M + 15) / 16) * ((N + 15) / 16);
  const int steps = (int)((K + 127) / 128);
  int plan = 0;
  if (tiles16 <= 2 * cus && K >= 64)
    plan = (!dense && steps >= 16 && tiles16 <= cus) ? 1608 : 1604;
  else if ((tiles32 <= cus && K >= 256) || (tiles32 * 4 <= 7 * cus && K >= 1024) || (tiles32 * 2 <= (M <= 512 ? 7 : 6) * cus && K >= 3072))
    plan = (!dense && steps >= 32 && tiles32 <= cus) ? 3208 : 3204;
  if (const char *f = tuning_env("CATCHQ_SMALL")) plan = std::atoi(f);
  return plan;
}

template <bool DENSE, int IN, bool DUAL, bool HALF_BIAS>
static int launch_small_bias(int plan, const SmallParams &p, const EpiDev &e, hipStream_t s) {
  switch (plan) {
    case 3204: return launch_small<32, 4, DENSE, IN, DUAL, HALF_BIAS>(p, e, s);
    case 3208: return launch_small<32, 8, DENSE, IN, DUAL, HALF_BIAS>(p, e, s);
    case 1604: return launch_small<16, 4, DENSE, IN, DUAL, HALF_BIAS>(p, e, s);
    case 1608: return launch_small<16, 8, DENSE, IN, DUAL, HALF_BIAS>(p, e, s);
    default: return -1;
  }
}

template <bool DENSE, int IN, bool DUAL>
static int launch_small_plan(int plan, const SmallParams &p, const EpiDev &e, hipStream_t s) {
  if constexpr (!DUAL) {
    if (e.bias_f16) return launch_small_bias<DENSE, IN, DUAL, true>(plan, p, e, s);
  }
  return launch_small_bias<DENSE, IN, DUAL, false>(plan, p, e, s);
}

static void small_common(SmallParams *p, int64_t M, int Co, int Ho, int Wo, const EpiDev &pick) {
  p->M = (int)M; p->N = Co; p->Ho = Ho; p->Wo = Wo;
  magic(Wo, &p->magic_wo, &p->mask_wo);
  magic(Ho, &p->magic_ho, &p->mask_ho);
  p->m_fastest = p->side[0].b_bytes > p->side[0].a_bytes;
  p->epi = pick_epilogue(Co, pick);
}

// The shapes this kernel takes from the tiled ones.  kh = kw = 1, stride 1, no padding: a GEMM of M rows.  -1: not one.
int contract_small_i8(const void *x, const void *w, int N_img, int H, int W, int Ci, int Co, int kh, int kw, int ph, int pw,
                      int sh, int sw, int dh, int dw, int Ho, int Wo, const EpiDev &e, hipStream_t s) {
  const bool dense = kh == 1 && kw == 1 && sh == 1 && sw == 1 && ph == 0 && pw == 0;
  const int64_t M = (int64_t)N_img * Ho * Wo;
  const int plan = small_plan(M, Co, (int64_t)kh * kw * Ci, dense, e.cus);
  if (!plan) return -1;
  SmallParams p = {};
  if (!small_side(&p.side[0], x, 1, w, N_img, H, W, Ci, Co, kh, kw, ph, pw, sh, sw, dh, dw, Ho, Wo, dense, Ci, false)) return -1;
  small_common(&p, M, Co, Ho, Wo, e);
  return dense ? launch_small_plan<true, IN_I8, false>(plan, p, e, s) : launch_small_plan<false, IN_I8, false>(plan, p, e, s);
}

// A residual block's last convolution with its 1x1 projection shortcut (arguments as conv2d_dual_i8).  -1: not one.
int contract_small_dual_i8(const void *x, const void *w, int N_img, int H, int W, int Ci, int Co, int kh, int kw, int ph, int pw,
                           int sh, int sw, int dh, int dw, int Ho, int Wo, const void *xs, const void *ws, int Hs, int Ws,
                           int Cs, int ss, const EpiDev &e, const ShortcutDev &sc, hipStream_t s) {
  if (e.exp2_a || e.exp2_b || e.resid || e.acc_out || !vec_epilogue_ok(Co, e) || !aligned16(sc.chan_div) ||
      !aligned16(sc.chan_rcp) || !aligned16(sc.bias))
    return -1;
  const int64_t M = (int64_t)N_img * Ho * Wo;
  const int plan = small_plan(M, Co, (int64_t)kh * kw * Ci + Cs, false, e.cus);
  if (!plan) return -1;
  SmallParams p = {};
  if (!small_side(&p.side[0], x, 1, w, N_img, H, W, Ci, Co, kh, kw, ph, pw, sh, sw, dh, dw, Ho, Wo, false, Ci, false) ||
      !small_side(&p.side[1], xs, 1, ws, N_img, Hs, Ws, Cs, Co, 1, 1, 0, 0, ss, ss, 1, 1, Ho, Wo, false, Cs, false))
    return -1;
  EpiDev probe = e;
  probe.resid = reinterpret_cast<const float *>(e.y ? e.y : e.q);  // any 16-byte aligned non-null pointer
  small_common(&p, M, Co, Ho, Wo, probe);
  p.sc = sc;
  return launch_small_plan<false, IN_I8, true>(plan, p, e, s);
}

// Activations still in floating point (NHWC), quantized at 2^position on their way into LDS: whether one launch serves
// the shape, and that launch.
//
// Every block converts its rows again for every filter tap and every column of tiles, which costs a wave more than the
// step's multiplications; a quantizer's launch costs about 1 us in front of it on the device (and 2.5 us of the host).
// So the one launch pays while a wave has few K steps.  Measured (one launch / two, us, half activations): 32 x 32 tiles,
// two steps a wave 5.1 / 5.7 (512 x 768 x 512) and 6.6 / 7.2 (384 x 1024 x 768), three 6.1 / 6.3 (256 x 1280 x 768), five
// 8.6 / 7.6 (4 x 14x14 256 -> 256 3x3), nine 37.7 / 19.0 (32 x 7x7 512 -> 512 3x3); 16 x 16 tiles, three steps 5.4 / 6.0
// (14x14 256 -> 256 3x3), four 4.6 / 5.3 (8 x 2048 x 1000), six 5.5 / 5.3 (1 x 3072 x 768), eight 9.8 / 7.0
// (32 x 4096 x 3072), thirteen 16.2 / 9.4 (2 x 14x14 256 -> 256 5x5).  Float activations lie within 1 us of these.
//
// Activations whose channels lie apart ([N, channel, H, W]) cost a load a value, against a quantizer that transposes (a call's time, us,
// two launches / one, 3 x 3 and 1 x 1 layers of 16 to 512 channels): 16 x 16 tiles on four waves, one step a wave 10.5 / 7.0, two 10.6 /
// 7.1, three and four 10.6 / 7.8 to 10.0 with up to a tile per unit and 11 / 13 to 17 with two; on eight waves two 11.9 / 10.3, three
// 11 / 12; 32 x 32 tiles one 10.5 / 6.8, two 11.8 / 9.1 up to a tile per unit, three 10.6 / 13.9.  Rows of any length in halfs, read in
// whole dwords, lie within 1 us of aligned ones: linears of an unaligned K 9.2 / 5.6, pixels of padded channels 10 / 7.  But rows that
// start off their pieces cost a wave more, and with more than a tile per unit a step less is what pays: 32 x 32 tiles on three steps, 310,
// 364 and 448 of them 8.5 / 11.9, 8.3 / 10.7 and 9.0 / 11.7, up to 256 8.3 / 7.9; 16 x 16 tiles on six, 306 to 498 of them 8.3 to 9.0 /
// 8.7 to 10.1, up to 256 8.5 / 7.1, on five 8.2 to 9.4 / 8.0 to 8.6.
//
// The plan (as small_plan) and the kernel's constants; 0: not the one launch.  The question and the launch ask it both.
static int small_float_plan(SmallSide *o, const void *x, bool half, const void *w, int N_img, int H, int W, int Ci, int Co, int kh,
                            int kw, int ph, int pw, int sh, int sw, int dh, int dw, int Ho, int Wo, bool dense, int x_ci, bool apart,
                            int cus) {
  const int64_t K = (int64_t)kh * kw * Ci;
  const int plan = small_plan((int64_t)N_img * Ho * Wo, Co, K, dense, cus);
  if (!plan) return 0;
  const int waves = plan % 100;
  const int64_t per_wave = ((K + 127) / 128 + waves - 1) / waves;
  const int64_t M = (int64_t)N_img * Ho * Wo, T = plan / 100, tiles = ((M + T - 1) / T) * ((Co + T - 1) / T);
  int most = T == 32 ? 3 : 6;
  if (apart) {
    if (T == 32) most = waves == 4 ? (tiles <= cus ? 2 : 1) : 0;
    else most = waves == 4 && tiles <= cus ? 4 : 2;
  } else if (x_ci != Ci && tiles > cus) {
    most -= 1;
  }
  if (per_wave > most) return 0;
  return small_side(o, x, half ? 2 : 4, w, N_img, H, W, Ci, Co, kh, kw, ph, pw, sh, sw, dh, dw, Ho, Wo, dense, x_ci, apart) ? plan : 0;
}
bool contract_small_float_ok(bool half, int N_img, int H, int W, int Ci, int Co, int kh, int kw, int ph, int pw, int sh, int sw,
                             int dh, int dw, int Ho, int Wo, int cus) {
  SmallSide o;
  const bool dense = kh == 1 && kw == 1 && sh == 1 && sw == 1 && ph == 0 && pw == 0;
  return small_float_plan(&o, nullptr, half, nullptr, N_img, H, W, Ci, Co, kh, kw, ph, pw, sh, sw, dh, dw, Ho, Wo, dense, Ci, false,
                          cus) != 0;
}
// x_ci channels in the activations, Ci in the filters (a multiple of 16, zeros where the activations have none); apart: [N, channel,
// H, W] activations.  Halfs of rows that start on any element are read in whole dwords and shifted.
int contract_small_float(const void *x, bool half, int position, const void *w, int N_img, int H, int W, int x_ci, bool apart, int Ci,
                         int Co, int kh, int kw, int ph, int pw, int sh, int sw, int dh, int dw, int Ho, int Wo, const EpiDev &e,
                         hipStream_t s) {
  const bool dense = kh == 1 && kw == 1 && sh == 1 && sw == 1 && ph == 0 && pw == 0 && !apart;
  SmallParams p = {};
  const int plan = small_float_plan(&p.side[0], x, half, w, N_img, H, W, Ci, Co, kh, kw, ph, pw, sh, sw, dh, dw, Ho, Wo, dense, x_ci,
                                    apart, e.cus);
  if (!plan) return -1;
  small_common(&p, (int64_t)N_img * Ho * Wo, Co, Ho, Wo, e);
  p.x_neg_pos = -position;
  if (apart)
    return half ? launch_small_plan<false, IN_F16_APART, false>(plan, p, e, s) : launch_small_plan<false, IN_F32_APART, false>(plan, p, e, s);
  if (half && x_ci % 2 != 0)
    return dense ? launch_small_plan<true, IN_F16_ANY, false>(plan, p, e, s) : launch_small_plan<false, IN_F16_ANY, false>(plan, p, e, s);
  if (half) return dense ? launch_small_plan<true, IN_F16, false>(plan, p, e, s) : launch_small_plan<false, IN_F16, false>(plan, p, e, s);
  return dense ? launch_small_plan<true, IN_F32, false>(plan, p, e, s) : launch_small_plan<false, IN_F32, false>(plan, p, e, s);
}

}  // namespace catchq
