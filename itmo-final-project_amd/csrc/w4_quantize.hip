// Group-wise asymmetric RTN int4 quantize/pack and the exact dequantize, for
// gfx950.  Semantics follow the reference's torch implementation
// (int4_triton/quantize.py:102-135) bit for bit; the kernel structure is this
// library's own: up to eight waves per (group, 64-column) tile, a lane per packed
// word, extremes by DPP steps across the lanes of a group, packing through the
// reciprocal with the rare doubtful words redone exactly, and an LDS transpose so
// that every qweight row segment is written as one coalesced 256-byte store.
// Groups above 512 take a statistics pass and a packing pass.
#include <hip/hip_runtime.h>

#include <climits>

#include "w4_common.hpp"

namespace w4 {

__device__ __forceinline__ float max_nan(float a, float b) { return (a > b || a != a) ? a : b; }
__device__ __forceinline__ float min_nan(float a, float b) { return (a < b || a != a) ? a : b; }
// torch.clamp keeps NaN (quantize.py:108-113); fminf/fmaxf would drop it.
__device__ __forceinline__ float clamp_nan(float x, float lo, float hi) {
  return (x != x) ? x : fminf(fmaxf(x, lo), hi);
}

// NaN-propagating maximum / minimum (v_maximum3_f32 / v_minimum3_f32 on
// gfx950): a NaN anywhere in a group reaches the reduced extremes, as with
// torch's amax / amin (quantize.py:108-109); no input canonicalization.
__device__ __forceinline__ float fmax_p(float a, float b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ float fmin_p(float a, float b) { return __builtin_elementwise_minimum(a, b); }

// One DPP step of a maximum and a minimum (values without NaN).  Written in
// assembly: the compiler puts a quieting v_max_f32 x, x before each, and the
// NaN-propagating forms have no DPP encoding, so a step took four or six
// instructions.  s_nop 1: a DPP operand written by the instruction before
// needs two wait states.
#define W4_MINMAX_DPP(CTRL)                                                     \
  asm("s_nop 1\n\t"                                                            \
      "v_max_f32_dpp %0, %0, %0 " CTRL " row_mask:0xf bank_mask:0xf\n\t"       \
      "v_min_f32_dpp %1, %1, %1 " CTRL " row_mask:0xf bank_mask:0xf\n\t"       \
      "s_nop 0"                                                                 \
      : "+v"(mx), "+v"(mn))

// Maximum and minimum over aligned groups of L lanes (L a power of two up to
// 64): DPP steps inside rows of 16 lanes (swap neighbours, swap pairs,
// half-row mirror, row mirror), lane shuffles across rows.
template <int L>
__device__ __forceinline__ void group_minmax(float& mx, float& mn) {
  if constexpr (L >= 2) W4_MINMAX_DPP("quad_perm:[1,0,3,2]");
  if constexpr (L >= 4) W4_MINMAX_DPP("quad_perm:[2,3,0,1]");
  if constexpr (L >= 8) W4_MINMAX_DPP("row_half_mirror");
  if constexpr (L >= 16) W4_MINMAX_DPP("row_mirror");
  if constexpr (L >= 32) {
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mn = fminf(mn, __shfl_xor(mn, 16, 64));
  }
  if constexpr (L >= 64) {
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    mn = fminf(mn, __shfl_xor(mn, 32, 64));
  }
}
#undef W4_MINMAX_DPP

struct QStats {
  float scale;  // fp16-representable (or 0/inf/NaN in degenerate groups)
  float zero;
};

// Fast form of group_stats, plus rcp(scale): bit-identical to it unless *bad.
//  - scale: for x = wmax - wmin in [2^-90, 2^126], y = x * fl(1/15) followed
//    by one fma correction with the exact residual fma(-y, 15, x) is the
//    correctly rounded x / 15 (checked for every float in that range by
//    tests/div15_exhaustive.c); every x whose scale is a positive finite fp16
//    lies in that range, so *bad covers the rest (infinite and NaN, quotients that
//    fp16 rounds to zero).  x = 0 is common, not rare (pruned weights, the rows past
//    N, which read zeros): its scale 1 and zero point 0 take one select here (all
//    redone, a zero 8192 x 2048 weight took 18.4 us at G = 128 instead of 10.9, 1 x 1024 at 512
//    10.8 instead of 6.2).
//  - zero: -wmin / scale <= 22.5 (scale >= x / 15 up to the fp16 rounding,
//    which for a subnormal scale >= 2^-24 is at most 2^-25), so with
//    v_rcp_f32 within 1 ulp t0 = fma(-wmin, rcp(scale), 0.5) is within 6e-6
//    of the reference's fl(fl(-wmin / scale) + 0.5) and the floors agree
//    unless fract(t0) is within 2^-15 of 0 or 1, which sets *bad.
// No branch: the caller redoes the rare bad groups with group_stats.
__device__ __forceinline__ QStats group_stats_fast(float rmax, float rmin, float* rcp, bool* bad) {
#pragma clang fp contract(off)
  const float wmax = __builtin_elementwise_maximum(rmax, 0.0f);
  const float wmin = __builtin_elementwise_minimum(rmin, 0.0f);
  const float x = wmax - wmin;
  constexpr float C15 = 1.0f / 15.0f;
  const float y = x * C15;
  QStats st;
  float q = __builtin_fmaf(__builtin_fmaf(-y, 15.0f, x), C15, y);
  q = x == 0.0f ? 1.0f : q;
  asm("" : "+v"(q));  // the fp32 quotient is rounded first, then to fp16: no fused fma-and-convert
  st.scale = (float)(_Float16)q;
  const float r = __builtin_amdgcn_rcpf(st.scale);
  const float t0 = __builtin_fmaf(-wmin, r, 0.5f);
  const float f0 = __builtin_amdgcn_fractf(t0);
  st.zero = __builtin_amdgcn_fmed3f(floorf(t0), 0.0f, 15.0f);
  *rcp = r;
  *bad = !__builtin_amdgcn_classf(st.scale, 0x100) ||  // positive normal
         !(__builtin_fabsf(f0 - 0.5f) <= 0.5f - 0x1p-15f);
  return st;
}

// quantize.py:108-112, in the same fp32 op order (true IEEE division).
__device__ __forceinline__ QStats group_stats(float rmax, float rmin) {
#pragma clang fp contract(off)
  const float wmax = max_nan(rmax, 0.0f);
  const float wmin = min_nan(rmin, 0.0f);
  float scale = (wmax - wmin) / 15.0f;
  if (scale == 0.0f) scale = 1.0f;
  scale = (float)(_Float16)scale;
  const float zero = clamp_nan(floorf(-wmin / scale + 0.5f), 0.0f, 15.0f);
  QStats r;
  r.scale = scale;
  r.zero = zero;
  return r;
}

// quantize.py:113-116: q = clamp(floor(w/scale + 0.5) + zero, 0, 15) -> int32
// (NaN converts to INT32_MIN like the reference's CPU cast), packed with
// int32 wrap-around.
__device__ __forceinline__ uint32_t quantize_pack8(const float v[8], QStats st) {
#pragma clang fp contract(off)
  uint32_t word = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float qf = clamp_nan(floorf(v[i] / st.scale + 0.5f) + st.zero, 0.0f, 15.0f);
    const uint32_t q = (qf != qf) ? 0x80000000u : (uint32_t)(int)qf;
    word += q << (4 * i);
  }
  return word;
}

// Fast form of quantize_pack8 for finite weights and a finite nonzero scale
// (group_stats' scale is then in [2^-24, 65504]).  m = 128 + t with t = w *
// rcp(scale) + 0.5 + zero, in one fma: between 128 and 256 a float's low 16
// bits are the fraction of t in units of 2^-16 and the bits above them its
// integer part.  v_rcp_f32 is within 1 ulp and the fma rounds by at most half
// a unit, so while |w / scale| < 32, t lies within one unit of the reference's
// fl(fl(w / scale) + 0.5) + zero, and both floors agree unless the fraction is
// within two units of 0 or 1; beyond that range, as for every t below 0.5 or
// above 15.5, both clamp to the same end (m is clamped to 128.5 .. 143.5,
// which gives 0 and 15 and a harmless fraction).  Returns true in *near when
// some fraction is that close: the caller then repacks the word with
// quantize_pack8.  Otherwise the word is bit-identical to quantize_pack8's.
// Two elements share each 32-bit operation after the clamp (39 vector
// instructions a word; a fract, two extremes, a conversion and a shift per
// element were 49).
__device__ __forceinline__ uint32_t quantize_pack8_fast(const float v[8], QStats st, float rcp, bool* near) {
  typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
  const float c = 128.5f + st.zero;
  uint32_t m[8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
    m[i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_fmed3f(__builtin_fmaf(v[i], rcp, c), 128.5f, 143.5f));
  // 0x4300 | q of elements i (low half) and i + 4 (high half)
  constexpr uint32_t kExp = 0x43004300u * 0x1111u;
  uint32_t word = 0u - kExp;
  u16x2 lo = u16x2{0xFFFF, 0xFFFF};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    word += __builtin_amdgcn_perm(m[i + 4], m[i], 0x07060302u) << (4 * i);
    const u16x2 f = __builtin_bit_cast(u16x2, __builtin_amdgcn_perm(m[i + 4], m[i], 0x05040100u));
    lo = __builtin_elementwise_min(lo, (u16x2)(f + (uint16_t)2));
  }
  *near = lo[0] < 4 || lo[1] < 4;
  return word;
}

// Stored fp16 patterns.  A NaN zero point is written as 0xFE00, the x86
// "default NaN" that the reference's CPU path produces for -0/0 and for
// negated NaN inputs; a NaN scale (NaN weights) as 0x7E00.
__device__ __forceinline__ uint16_t scale_bits(float s) {
  return (s != s) ? (uint16_t)0x7E00 : __builtin_bit_cast(uint16_t, (_Float16)s);
}
__device__ __forceinline__ uint16_t zero_bits(float z) {
  return (z != z) ? (uint16_t)0xFE00 : __builtin_bit_cast(uint16_t, (_Float16)z);
}

constexpr int QROWS = 64;  // columns n per tile (= lanes, for the stores)
constexpr int QSWAVES = 8;  // waves per workgroup

// Waves sharing one (group, 64-column) tile: 64 rows split between up to eight
// waves, each taking whole iterations of 512 / G rows (a lone wave per tile
// runs one long dependent chain per SIMD and leaves most of the chip idle).
constexpr int quantize_waves_per_tile(int G) { return G / 8 < QSWAVES ? G / 8 : QSWAVES; }

// Single-pass kernel for G <= 512: lanes_per_row = G/8 lanes each own one
// packed word of a row; 64/lanes_per_row rows are processed per iteration.
// Bound by HBM (154 MB for the block of 1B-model weights at G = 128: 33.0 us =
// 4.7 TB/s, a large copy reaches 5.2; 37.5 us before the statistics lost their
// branches, the packing its per-element boundary tests and the tiles their order
// along N).
// One weight of a quantize launch (w4_quantize_grouped puts several in one).
struct QuantArgs {
  const uint16_t* w;
  int32_t* qw;
  uint16_t* sc;
  uint16_t* ze;
  int64_t N, K, swn, swk;
  int64_t tiles_n, tiles_total;
  int gshift;  // G > 512: log2(G)
  int wpr;     // statistics pass of G > 512: waves per row
};

constexpr int kQuantMaxGrouped = 8;
struct QuantGroupedArgs {
  QuantArgs prob[kQuantMaxGrouped];
  int wg_start[kQuantMaxGrouped + 1];
  int count;
};

// The tiles of workgroup `blk` of one weight (see quantize_small_group_kernel).
// GIVEN: pack pass of a group size above 512; G is then only the tile's width
// in k, and the scale and zero point of each row are read from sc and ze, where
// the statistics pass has put them (both are exact in fp16).
template <int DT, int G, bool VEC, bool GIVEN = false>
__device__ __forceinline__ void quantize_small_group_tiles(const QuantArgs& qa, int blk) {
  const uint16_t* __restrict__ w = qa.w;
  int32_t* __restrict__ qw = qa.qw;
  uint16_t* __restrict__ sc = qa.sc;
  uint16_t* __restrict__ ze = qa.ze;
  const int64_t N = qa.N, K = qa.K, swn = qa.swn, swk = qa.swk, tiles_n = qa.tiles_n, tiles_total = qa.tiles_total;
  constexpr int L = G / 8;            // lanes per row (1..64)
  constexpr int RPI = 64 / L;         // rows per iteration
  constexpr int WPT = quantize_waves_per_tile(G);
  constexpr int TPB = QSWAVES / WPT;  // tiles per workgroup
  constexpr int RW = QROWS / WPT;     // rows per wave
  static_assert(RW % RPI == 0 && L % WPT == 0, "wave split of a tile");
  __shared__ uint32_t tile[TPB][L][QROWS + 1];
  __shared__ uint16_t st_s[TPB][QROWS];
  __shared__ uint16_t st_z[TPB][QROWS];

  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform: tile math stays scalar
  const int ts = wv / WPT, sub = wv % WPT;  // tile slot, row slice of this wave
  // the host keeps tile counts below 2^31, so the tile index math is 32-bit
  const int t = blk * TPB + ts;
  const bool active = t < (int)tiles_total;
  const int groups = (int)((uint32_t)K / (uint32_t)G);
  // Tiles in order along K, so that the workgroups running at one time read whole
  // rows.  Groups of 8 and 16 write as many bytes of scales and zero points as of
  // codes, 128 at a time, and from 2^24 weights on are faster along N, where those
  // meet in lines (8192 x 8192: 84.9 against 89.4 us at 8, 58.3 against 64.4 at 16;
  // 4096 x 2048: 11.8 against 11.5 and 9.4 against 9.0; G = 32, 8192 x 8192: 53.3
  // against 48.1).
  const bool along_n = G <= 16 && !GIVEN && N * K >= (int64_t)1 << 24;
  const int tn = !active ? 0 : along_n ? t % (int)tiles_n : t / groups;
  const int g = !active ? 0 : along_n ? t / (int)tiles_n : t - tn * groups;
  const int64_t n0 = (int64_t)tn * QROWS;
  const int seg = lane % L;
  const int rsub = lane / L;

  // Rows are loaded in batches of up to 16 per lane before any is used, so a
  // wave keeps 16 row segments in flight instead of one.
  constexpr int IT = RW / RPI;
  constexpr int B = IT < 16 ? IT : 16;
  const uint32_t w_bytes = VEC ? (uint32_t)(((N - 1) * swn + K) * 2) : 0u;
  const __amdgpu_buffer_rsrc_t rw =
      __builtin_amdgcn_make_buffer_rsrc((void*)w, (short)0, (int)w_bytes, 0x00020000);
  if (active) {
    for (int b0 = 0; b0 < IT; b0 += B) {
      u32x4 raw[B];
      uint16_t gs[B], gz[B];
      if constexpr (GIVEN) {
#pragma unroll
        for (int i = 0; i < B; ++i) {
          const int64_t n = n0 + sub * RW + (b0 + i) * RPI + rsub;
          const int64_t at = (((int64_t)g * G) >> qa.gshift) * N + n;
          gs[i] = n < N ? sc[at] : (uint16_t)0x3C00;
          gz[i] = n < N ? ze[at] : (uint16_t)0;
        }
      }
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const int row = sub * RW + (b0 + i) * RPI + rsub;
        const int64_t n = n0 + row;
        if constexpr (VEC) {
          // rows past N read zeros (buffer range check)
          // 32-bit offsets: the host routes only weights below 2^31 bytes here
          const uint32_t off = n < N ? ((uint32_t)n * (uint32_t)swn + (uint32_t)(g * G + seg * 8)) * 2u
                                     : 0x80000000u;
          // non-temporal (cache policy bit 1): every weight byte is read
          // once (block 64.4 -> 61.8 us against the default policy)
          raw[i] = __builtin_amdgcn_raw_buffer_load_b128(rw, off, 0, 2);
        } else {
          uint16_t e[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) e[j] = n < N ? w[n * swn + (g * G + seg * 8 + j) * swk] : (uint16_t)0;
          raw[i] = u32x4{e[0] | ((uint32_t)e[1] << 16), e[2] | ((uint32_t)e[3] << 16),
                         e[4] | ((uint32_t)e[5] << 16), e[6] | ((uint32_t)e[7] << 16)};
        }
      }
      // every word takes the reciprocal packing and the rare flagged ones are
      // redone exactly, a group with a NaN among them: the NaN-propagating
      // extremes of its lanes give it NaN extremes and so a NaN scale (the
      // sign of a zero extreme does not reach group_stats' result)
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const int row = sub * RW + (b0 + i) * RPI + rsub;
        float v[8];
        unpack8<DT>(raw[i], v);
        float rcp;
        bool bad, near;
        QStats st;
        float mx, mn;
        if constexpr (GIVEN) {
          st.scale = half_bits_to_float(gs[i]);
          st.zero = half_bits_to_float(gz[i]);
          rcp = __builtin_amdgcn_rcpf(st.scale);
          bad = !__builtin_amdgcn_classf(st.scale, 0x100) || st.zero != st.zero;  // positive normal
        } else {
          mx = fmax_p(v[0], v[1]), mn = fmin_p(v[0], v[1]);
#pragma unroll
          for (int j = 2; j < 8; ++j) {
            mx = fmax_p(mx, v[j]);
            mn = fmin_p(mn, v[j]);
          }
          const uint64_t nan_lanes = __ballot(mx != mx);
          group_minmax<L>(mx, mn);
          if (nan_lanes != 0) {  // rare, wave-uniform: a NaN reaches both extremes of its whole group
            if constexpr (L == 64)
              mx = mn = __builtin_nanf("");
            else if ((nan_lanes >> (lane & ~(L - 1))) & ((1ull << L) - 1))
              mx = mn = __builtin_nanf("");
          }
          st = group_stats_fast(mx, mn, &rcp, &bad);
        }
        uint32_t word = quantize_pack8_fast(v, st, rcp, &near);
        // a word near a rounding boundary, or a group whose statistics are:
        // infinite, NaN or underflowing scale, zero point near one
        if (near || bad) {
          if constexpr (!GIVEN) {
            if (bad) st = group_stats(mx, mn);  // (a chain of divisions that a near word need not wait for)
          }
          word = quantize_pack8(v, st);
        }
        tile[ts][seg][row] = word;
        if (!GIVEN && seg == 0) {
          st_s[ts][row] = scale_bits(st.scale);
          st_z[ts][row] = zero_bits(st.zero);
        }
      }
    }
  }
  __syncthreads();
  if (active) {
    const int64_t n = n0 + lane;
    if (n < N) {
      const int64_t k8_0 = g * L;
#pragma unroll 4
      // non-temporal stores: nothing here reads the packed outputs again
      // (3.5 % on the block against cached stores)
      for (int kk = sub; kk < L; kk += WPT)
        __builtin_nontemporal_store((int32_t)tile[ts][kk][lane], &qw[(k8_0 + kk) * N + n]);
      if (!GIVEN && sub == 0) {
        __builtin_nontemporal_store(st_s[ts][lane], &sc[g * N + n]);
        __builtin_nontemporal_store(st_z[ts][lane], &ze[g * N + n]);
      }
    }
  }
}

template <int DT, int G, bool VEC>
__global__ __launch_bounds__(QSWAVES * 64) void quantize_small_group_kernel(QuantArgs qa) {
  quantize_small_group_tiles<DT, G, VEC>(qa, (int)blockIdx.x);
}

// Several weights in one launch: workgroup b belongs to the weight whose
// workgroup range holds it (the ranges follow each other in order).
template <int DT, int G>
__global__ __launch_bounds__(QSWAVES * 64) void quantize_small_group_grouped_kernel(QuantGroupedArgs ga) {
  const int b = blockIdx.x;
  int p = 0;
#pragma unroll
  for (int i = 1; i < kQuantMaxGrouped; ++i)
    if (i < ga.count && b >= ga.wg_start[i]) p = i;
  quantize_small_group_tiles<DT, G, true>(ga.prob[p], b - ga.wg_start[p]);
}

// Group sizes above 512 (per-channel G = K included) take two passes, because a
// group of 64 columns no longer fits a workgroup's registers: the statistics
// of every (column, group) row, then the packing in tiles of 128 k.  The
// second read comes mostly from the Infinity Cache.  The one-kernel form they
// replace (a wave looping over 64 rows, twice) had N / 64 x K / G waves, 32 for
// a per-channel 2048 x 8192 weight: the block's seven weights per channel took
// 2703 us, these 57 us.
constexpr int QPACK = 128;  // k per tile of the packing pass

// Statistics: `wpr` waves (a power of two, chosen so that few rows still spread
// over the chip) reduce one row of G weights, eight waves per workgroup.
template <int DT, bool VEC>
__device__ __forceinline__ void quantize_stats_rows(const QuantArgs& qa, int blk) {
  __shared__ float part[2][QSWAVES];
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wpr = qa.wpr, rows = QSWAVES / wpr;  // rows per workgroup
  const int64_t G = 1ll << qa.gshift;
  // rows of one group are adjacent columns
  const int64_t per_group = (qa.N + rows - 1) / rows;
  const int64_t g = blk / per_group;
  const int64_t n0 = (blk - g * per_group) * rows;
  const int64_t n = n0 + wv / wpr;
  float mx = 0.f, mn = 0.f;
  if (n < qa.N) {
    const uint16_t* row = qa.w + n * qa.swn;
    const int64_t step = 512ll * wpr, k0 = g * G + (wv % wpr) * 512 + lane * 8;
    bool first = true;
    for (int64_t k = k0; k < (g + 1) * G; k += 4 * step) {
      u32x4 raw[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        // past the group: the row's first load again, which changes no extreme
        const int64_t ku = k + u * step < (g + 1) * G ? k + u * step : k;
        if constexpr (VEC) {
          raw[u] = *reinterpret_cast<const u32x4*>(row + ku);
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            raw[u][j] = row[(ku + 2 * j) * qa.swk] | ((uint32_t)row[(ku + 2 * j + 1) * qa.swk] << 16);
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        float v[8];
        unpack8<DT>(raw[u], v);
        if (first) mx = mn = v[0];
        first = false;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          mx = fmax_p(mx, v[j]);
          mn = fmin_p(mn, v[j]);
        }
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      mx = fmax_p(mx, __shfl_xor(mx, off, 64));
      mn = fmin_p(mn, __shfl_xor(mn, off, 64));
    }
  }
  if (lane == 0) part[0][wv] = mx, part[1][wv] = mn;
  __syncthreads();
  const int r = threadIdx.x;
  if (r < rows && n0 + r < qa.N) {
    float a = part[0][r * wpr], b = part[1][r * wpr];
    for (int w = 1; w < wpr; ++w) {
      a = fmax_p(a, part[0][r * wpr + w]);
      b = fmin_p(b, part[1][r * wpr + w]);
    }
    const QStats st = group_stats(a, b);
    qa.sc[g * qa.N + n0 + r] = scale_bits(st.scale);
    qa.ze[g * qa.N + n0 + r] = zero_bits(st.zero);
  }
}

template <int DT, bool VEC>
__global__ __launch_bounds__(QSWAVES * 64) void quantize_stats_kernel(QuantGroupedArgs ga) {
  const int b = blockIdx.x;
  int p = 0;
#pragma unroll
  for (int i = 1; i < kQuantMaxGrouped; ++i)
    if (i < ga.count && b >= ga.wg_start[i]) p = i;
  quantize_stats_rows<DT, VEC>(ga.prob[p], b - ga.wg_start[p]);
}

template <int DT, bool VEC>
__global__ __launch_bounds__(QSWAVES * 64) void quantize_pack_kernel(QuantGroupedArgs ga) {
  const int b = blockIdx.x;
  int p = 0;
#pragma unroll
  for (int i = 1; i < kQuantMaxGrouped; ++i)
    if (i < ga.count && b >= ga.wg_start[i]) p = i;
  quantize_small_group_tiles<DT, QPACK, VEC, true>(ga.prob[p], b - ga.wg_start[p]);
}

// W_hat[N, K] = round_once((q - z) * s): tiles of 64 columns x 64 words,
// transposed through LDS so that both the qweight reads (256-byte rows) and the
// W_hat row writes (1 KB in bf16 / fp16) are whole lines.
//
// What bounds it: HBM, four fifths of the bytes being writes.  Eight waves per
// tile, every wave's eight word loads and the tile's scales and zeros (staged
// once, two 16-bit values in one LDS word) in flight before the barrier: with
// four waves that fetched a scale and a zero per word from memory between the
// writes, the 8192 x 2048 weight took 14.3 us, this 8.4 us (5.0 TB/s,
// what a large copy reaches).  16-bit rows are stored non-temporal (9.7 us
// cached); fp32 lanes store two 16-byte halves 32 bytes apart, where partial
// lines made that slower (26 against 16.5 us).
//
// NT: the codes are loaded non-temporal, for fp32 output of whole 128-byte lines
// (N % 32 == 0).  Its writes are eight times the codes and fill the Infinity
// Cache, which the codes then leave to them (inputs not in the cache: 8192 x 2048
// 16.0 against 17.2 us, 12032 x 4096 46.1 against 48.4).  16-bit output leaves
// room for them (8192 x 4096: 15.1 us, non-temporal 17.4; again on the same input
// 14.7 against 17.9), and lines that two tiles share are fetched twice without the
// cache (12001 x 4096: 22.6 against 27.4, fp32 48.3 against 49.2).
template <int ODT, bool NT>
__global__ __launch_bounds__(512) void dequantize_kernel(const int32_t* __restrict__ qw,
                                                         const uint16_t* __restrict__ sc,
                                                         const uint16_t* __restrict__ ze,
                                                         int64_t N, int64_t K8, int gshift,
                                                         void* __restrict__ out) {
#pragma clang fp contract(off)
  __shared__ uint32_t tile[64][65];
  __shared__ uint32_t sz[64][65];  // [group of the tile][column]: scale | zero << 16
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t n0 = (int64_t)blockIdx.x * 64;
  const int64_t k80 = (int64_t)blockIdx.y * 64;
  const int64_t n = n0 + lane;
  const int rows = (int)(K8 - k80 < 64 ? K8 - k80 : 64);  // words per column of this tile
  uint32_t w[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int kk = i * 8 + wv;
    const int32_t* at = &qw[(k80 + kk) * N + n];
    w[i] = 0u;
    if (kk < rows && n < N) w[i] = (uint32_t)(NT ? __builtin_nontemporal_load(at) : *at);
  }
  // groups first .. first + groups - 1 (a group size below 512 divides the tile's 512 k)
  const int64_t first = (k80 * 8) >> gshift;
  const int groups = (int)(((k80 + rows) * 8 - 1) >> gshift) - (int)first + 1;
  for (int g = wv; g < groups; g += 8)
    if (n < N) sz[g][lane] = (uint32_t)sc[(first + g) * N + n] | ((uint32_t)ze[(first + g) * N + n] << 16);
#pragma unroll
  for (int i = 0; i < 8; ++i) tile[i * 8 + wv][lane] = w[i];
  __syncthreads();
  const int64_t K = K8 * 8;
  const int64_t k8 = k80 + lane;
  const int g = (int)(((k8 * 8) >> gshift) - first);
  if (lane >= rows) return;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int nn = i * 8 + wv;
    if (n0 + nn >= N) break;
    const uint32_t word = tile[lane][nn];
    const uint32_t c = sz[g][nn];
    const float s = half_bits_to_float((uint16_t)(c & 0xFFFFu));
    const float z = half_bits_to_float((uint16_t)(c >> 16));
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[j] = ((float)((word >> (4 * j)) & 0xFu) - z) * s;
      // Materialize the fp32 product: without this the backend folds
      // multiply + fp16 cast into one mixed fma with a +0 addend, which
      // turns a -0 product (q < z, s = 0) into +0.
      asm volatile("" : "+v"(v[j]));
    }
    if constexpr (ODT == W4_DTYPE_FP32) {
      float* o = reinterpret_cast<float*>(out) + (n0 + nn) * K + k8 * 8;
      f32x4 a, b;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        a[j] = v[j];
        b[j] = v[4 + j];
      }
      *reinterpret_cast<f32x4*>(o) = a;
      *reinterpret_cast<f32x4*>(o + 4) = b;
    } else {
      uint16_t* o = reinterpret_cast<uint16_t*>(out) + (n0 + nn) * K + k8 * 8;
      u32x4 p;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        p[j] = (uint32_t)float_to_act_bits<ODT>(v[2 * j]) |
               ((uint32_t)float_to_act_bits<ODT>(v[2 * j + 1]) << 16);
      __builtin_nontemporal_store(p, reinterpret_cast<u32x4*>(o));
    }
  }
}

}  // namespace w4

using namespace w4host;

// Both passes of `count` weights with group sizes above 512 (gshift set).
template <int DT, bool VEC>
static void launch_large(w4::QuantGroupedArgs ga, int count, hipStream_t st) {
  // waves per row: eight, four, ... while there are fewer rows than give every
  // CU (256) two workgroups, and at least 512 weights (a load per lane) each
  int64_t rows = 0;
  for (int i = 0; i < count; ++i) rows += ga.prob[i].N * (ga.prob[i].K >> ga.prob[i].gshift);
  int wpr = 1;
  while (wpr < w4::QSWAVES && rows * wpr * 2 <= 512 * w4::QSWAVES) wpr *= 2;
  int64_t wgs = 0, packs = 0;
  w4::QuantGroupedArgs gp = ga;
  for (int i = 0; i < count; ++i) {
    w4::QuantArgs& a = ga.prob[i];
    a.wpr = wpr;
    while (a.wpr > 1 && 512ll * a.wpr > (1ll << a.gshift)) a.wpr /= 2;
    const int64_t per_wg = w4::QSWAVES / a.wpr;
    ga.wg_start[i] = (int)wgs;
    wgs += (a.N + per_wg - 1) / per_wg * (a.K >> a.gshift);
    gp.wg_start[i] = (int)packs;
    const int64_t tpb = w4::QSWAVES / w4::quantize_waves_per_tile(w4::QPACK);
    packs += (a.tiles_total + tpb - 1) / tpb;
  }
  for (int i = count; i <= w4::kQuantMaxGrouped; ++i) ga.wg_start[i] = (int)wgs, gp.wg_start[i] = (int)packs;
  ga.count = gp.count = count;
  const dim3 block(w4::QSWAVES * 64);
  hipLaunchKernelGGL((w4::quantize_stats_kernel<DT, VEC>), dim3((unsigned)wgs), block, 0, st, ga);
  hipLaunchKernelGGL((w4::quantize_pack_kernel<DT, VEC>), dim3((unsigned)packs), block, 0, st, gp);
}

template <int DT, bool VEC>
static void launch_quantize(const uint16_t* w, int64_t N, int64_t K, int64_t swn, int64_t swk,
                            int G, int32_t* qw, uint16_t* sc, uint16_t* ze, hipStream_t st) {
  const int64_t tiles_n = (N + w4::QROWS - 1) / w4::QROWS;
  if (G > 512) {
    w4::QuantGroupedArgs ga{};
    ga.prob[0] = w4::QuantArgs{w, qw, sc, ze, N, K, swn, swk, tiles_n, tiles_n * (K / w4::QPACK), ilog2(G), 1};
    launch_large<DT, VEC>(ga, 1, st);
    return;
  }
  const int64_t tiles_total = tiles_n * (K / G);
  const int64_t tpb = w4::QSWAVES / w4::quantize_waves_per_tile(G);
  const dim3 grid((unsigned)((tiles_total + tpb - 1) / tpb));
  const dim3 block(w4::QSWAVES * 64);
  const w4::QuantArgs qa{w, qw, sc, ze, N, K, swn, swk, tiles_n, tiles_total, 0, 1};
#define W4_QS(GG)                                                                                  \
  case GG:                                                                                         \
    hipLaunchKernelGGL((w4::quantize_small_group_kernel<DT, GG, VEC>), grid, block, 0, st, qa); \
    return;
  switch (G) {
    W4_QS(8)
    W4_QS(16)
    W4_QS(32)
    W4_QS(64)
    W4_QS(128)
    W4_QS(256)
    W4_QS(512)
    default:
      break;
  }
#undef W4_QS
}

extern "C" int w4_quantize(const void* w, int w_dtype, int64_t N, int64_t K, int64_t stride_wn,
                           int64_t stride_wk, int group_size, int32_t* qweight, uint16_t* scales,
                           uint16_t* zeros, void* stream) {
  clear_error();
  if (w_dtype != W4_DTYPE_BF16 && w_dtype != W4_DTYPE_FP16)
    return fail(W4_ERR_INVALID, "w4_quantize: weight dtype must be bf16 or fp16 (got code %d)", w_dtype);
  if (N < 0 || K <= 0) return fail(W4_ERR_INVALID, "w4_quantize: bad shape N=%lld K=%lld", (long long)N, (long long)K);
  const int64_t G = group_size == -1 ? K : group_size;
  if (G <= 0 || K % G != 0 || G % 8 != 0 || !is_pow2(G))
    return fail(W4_ERR_INVALID,
                "w4_quantize: group_size must be a power of two, a multiple of 8 and divide K "
                "(K=%lld, group_size=%d)", (long long)K, group_size);
  if (G > (int64_t)1 << 30) return fail(W4_ERR_UNSUPPORTED, "w4_quantize: group_size too large");
  if (N == 0) return W4_OK;
  if (!w || !qweight || !scales || !zeros) return fail(W4_ERR_INVALID, "w4_quantize: null pointer");
  // (the tiles of the kernel that runs, and the rows of its statistics pass)
  if (((N + 63) / 64) * (K / (G > 512 ? w4::QPACK : G)) >= (int64_t)1 << 31 ||
      (G > 512 && N * (K / G) >= (int64_t)1 << 31))
    return fail(W4_ERR_UNSUPPORTED, "w4_quantize: %lld x %lld weight has too many tiles", (long long)N,
                (long long)K);
  const uint16_t* wp = static_cast<const uint16_t*>(w);
  // 128-bit buffer loads: dense rows, 16-byte aligned, whole tensor within 2 GiB
  const bool vec = stride_wk == 1 && (stride_wn % 8) == 0 && ((uintptr_t)wp % 16) == 0 &&
                   ((N - 1) * stride_wn + K) * 2 < (1LL << 31);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (w_dtype == W4_DTYPE_BF16) {
    if (vec) launch_quantize<W4_DTYPE_BF16, true>(wp, N, K, stride_wn, stride_wk, (int)G, qweight, scales, zeros, st);
    else launch_quantize<W4_DTYPE_BF16, false>(wp, N, K, stride_wn, stride_wk, (int)G, qweight, scales, zeros, st);
  } else {
    if (vec) launch_quantize<W4_DTYPE_FP16, true>(wp, N, K, stride_wn, stride_wk, (int)G, qweight, scales, zeros, st);
    else launch_quantize<W4_DTYPE_FP16, false>(wp, N, K, stride_wn, stride_wk, (int)G, qweight, scales, zeros, st);
  }
  return check_launch("w4_quantize");
}

// One grouped launch when every weight takes the single-pass 128-bit path
// with the same group size; otherwise one w4_quantize per weight, in order.
extern "C" int w4_quantize_grouped(const w4_quantize_problem* problems, int count, int w_dtype, void* stream) {
  clear_error();
  if (count < 1 || count > W4_MAX_GROUPED)
    return fail(W4_ERR_INVALID, "w4_quantize_grouped: count must be in [1, %d]", W4_MAX_GROUPED);
  if (!problems) return fail(W4_ERR_INVALID, "w4_quantize_grouped: null problem list");
  if (w_dtype != W4_DTYPE_BF16 && w_dtype != W4_DTYPE_FP16)
    return fail(W4_ERR_INVALID, "w4_quantize_grouped: weight dtype must be bf16 or fp16 (got code %d)", w_dtype);
  static_assert(W4_MAX_GROUPED <= w4::kQuantMaxGrouped, "grouped quantize capacity");
  w4::QuantGroupedArgs ga{};
  int64_t G0 = -1, wgs = 0;
  bool one_launch = true;
  for (int i = 0; i < count; ++i) {
    const w4_quantize_problem& q = problems[i];
    if (q.N < 0 || q.K <= 0)
      return fail(W4_ERR_INVALID, "w4_quantize_grouped: bad shape in problem %d (N=%lld K=%lld)", i,
                  (long long)q.N, (long long)q.K);
    const int64_t G = q.group_size == -1 ? q.K : q.group_size;
    if (G <= 0 || q.K % G != 0 || G % 8 != 0 || !is_pow2(G))
      return fail(W4_ERR_INVALID, "w4_quantize_grouped: bad group size %d in problem %d (K=%lld)", q.group_size, i,
                  (long long)q.K);
    if (q.N > 0 && (!q.w || !q.qweight || !q.scales || !q.zeros))
      return fail(W4_ERR_INVALID, "w4_quantize_grouped: null pointer in problem %d", i);
    const bool vec = q.stride_wk == 1 && (q.stride_wn % 8) == 0 && ((uintptr_t)q.w % 16) == 0 &&
                     ((q.N - 1) * q.stride_wn + q.K) * 2 < (1LL << 31) && ((q.N + 63) / 64) * (q.K / G) < (1LL << 30);
    // all of one group size up to 512, or all above it (each its own: -1 is K)
    one_launch = one_launch && q.N > 0 && vec && (G0 < 0 || G == G0 || (G > 512 && G0 > 512));
    G0 = G;
    if (!one_launch) continue;
    const int64_t tile_k = G > 512 ? w4::QPACK : G;
    const int64_t tiles_n = (q.N + w4::QROWS - 1) / w4::QROWS, tiles_total = tiles_n * (q.K / tile_k);
    const int64_t tpb = w4::QSWAVES / w4::quantize_waves_per_tile((int)tile_k);
    ga.prob[i] = w4::QuantArgs{static_cast<const uint16_t*>(q.w), q.qweight, q.scales, q.zeros, q.N, q.K,
                               q.stride_wn, q.stride_wk, tiles_n, tiles_total, ilog2(G), 1};
    ga.wg_start[i] = (int)wgs;
    wgs += (tiles_total + tpb - 1) / tpb;
    one_launch = wgs < (1LL << 30);
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (!one_launch) {
    for (int i = 0; i < count; ++i) {
      const w4_quantize_problem& q = problems[i];
      const int rc = w4_quantize(q.w, w_dtype, q.N, q.K, q.stride_wn, q.stride_wk, q.group_size, q.qweight,
                                 q.scales, q.zeros, stream);
      if (rc != W4_OK) return rc;
    }
    return W4_OK;
  }
  if (G0 > 512) {
    if (w_dtype == W4_DTYPE_BF16) launch_large<W4_DTYPE_BF16, true>(ga, count, st);
    else launch_large<W4_DTYPE_FP16, true>(ga, count, st);
    return check_launch("w4_quantize_grouped");
  }
  for (int i = count; i <= w4::kQuantMaxGrouped; ++i) ga.wg_start[i] = (int)wgs;
  ga.count = count;
  const dim3 grid((unsigned)wgs), block(w4::QSWAVES * 64);
#define W4_QG(DT, GG)                                                                                \
  case GG:                                                                                           \
    hipLaunchKernelGGL((w4::quantize_small_group_grouped_kernel<DT, GG>), grid, block, 0, st, ga); \
    break;
  if (w_dtype == W4_DTYPE_BF16) {
    switch (G0) { W4_QG(W4_DTYPE_BF16, 8) W4_QG(W4_DTYPE_BF16, 16) W4_QG(W4_DTYPE_BF16, 32) W4_QG(W4_DTYPE_BF16, 64)
                  W4_QG(W4_DTYPE_BF16, 128) W4_QG(W4_DTYPE_BF16, 256) W4_QG(W4_DTYPE_BF16, 512) default: break; }
  } else {
    switch (G0) { W4_QG(W4_DTYPE_FP16, 8) W4_QG(W4_DTYPE_FP16, 16) W4_QG(W4_DTYPE_FP16, 32) W4_QG(W4_DTYPE_FP16, 64)
                  W4_QG(W4_DTYPE_FP16, 128) W4_QG(W4_DTYPE_FP16, 256) W4_QG(W4_DTYPE_FP16, 512) default: break; }
  }
#undef W4_QG
  return check_launch("w4_quantize_grouped");
}

extern "C" int w4_dequantize(const int32_t* qweight, const uint16_t* scales, const uint16_t* zeros,
                             int64_t N, int64_t K, int group_size, int out_dtype, void* out,
                             void* stream) {
  clear_error();
  if (N < 0 || K <= 0 || K % 8 != 0)
    return fail(W4_ERR_INVALID, "w4_dequantize: bad shape N=%lld K=%lld", (long long)N, (long long)K);
  const int64_t G = group_size == -1 ? K : group_size;
  if (G <= 0 || K % G != 0 || G % 8 != 0 || !is_pow2(G))
    return fail(W4_ERR_INVALID, "w4_dequantize: bad group_size %d for K=%lld", group_size, (long long)K);
  if (N == 0) return W4_OK;
  if (!qweight || !scales || !zeros || !out) return fail(W4_ERR_INVALID, "w4_dequantize: null pointer");
  if (((uintptr_t)out % 16) != 0) return fail(W4_ERR_INVALID, "w4_dequantize: output must be 16-byte aligned");
  const int64_t K8 = K / 8;
  const dim3 grid((unsigned)((N + 63) / 64), (unsigned)((K8 + 63) / 64));
  const int gshift = ilog2(G);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(512), 0, st, qweight, scales, zeros, N, K8, gshift, out);
  };
  switch (out_dtype) {
    case W4_DTYPE_BF16:
      launch(w4::dequantize_kernel<W4_DTYPE_BF16, false>);
      break;
    case W4_DTYPE_FP16:
      launch(w4::dequantize_kernel<W4_DTYPE_FP16, false>);
      break;
    case W4_DTYPE_FP32:
      if (N % 32 == 0) launch(w4::dequantize_kernel<W4_DTYPE_FP32, true>);
      else launch(w4::dequantize_kernel<W4_DTYPE_FP32, false>);
      break;
    default:
      return fail(W4_ERR_INVALID, "w4_dequantize: bad out dtype %d", out_dtype);
  }
  return check_launch("w4_dequantize");
}
