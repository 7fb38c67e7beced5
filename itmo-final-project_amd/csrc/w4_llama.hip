// Kernels of a Llama-style decoder layer between its W4A16 linears
// (int4_hip/llama.py): the attention of one decode step and of a prompt, RMSNorm
// (with the residual addition before it) and the gated activation of the MLP.
//
// One token's attention is a handful of tiny operations (rotary embedding of
// q and k, two cache writes, q.K, softmax, p.V), so as separate launches it is
// bound by launch latency; here it is one launch.
#include <hip/hip_runtime.h>

#include "w4_common.hpp"

namespace w4 {

constexpr int kAttnThreads = 256;
constexpr int kAttnWaves = kAttnThreads / 64;
constexpr int kAttnMaxChunks = 64;  // position chunks per key-value head
constexpr int kAttnHeads = 4;       // query heads per workgroup
constexpr float kLog2e = 1.4426950408889634f;

struct AttnDecodeArgs {
  const uint16_t* q;  // [nh * D]
  const uint16_t* k;  // [nkv * D]
  const uint16_t* v;  // [nkv * D]
  const float* cos;   // [D / 2], the row of the position
  const float* sin;
  float* kc;          // [nkv, D, max_len]
  float* vc;          // [nkv, max_len, D]
  const int64_t* pos;
  uint16_t* out;      // [nh * D]
  unsigned* cnt;      // one arrival counter per key-value head and head slice
  float* part;        // [nkv, slices, chunks, kAttnHeads * (D + 2)]
  float qscale;       // softmax scale * log2(e)
  int g, max_len, chunk, chunks;
};

// Rotates the pair (x1, x2) = (x[d], x[d + D/2]); products and sums rounded
// separately, as the torch-op version does.
__device__ __forceinline__ void rope_pair(float x1, float x2, float c, float s, float* r1, float* r2) {
#pragma clang fp contract(off)
  *r1 = x1 * c - x2 * s;
  *r2 = x2 * c + x1 * s;
}

// Reductions over the 64 lanes (all active), the result in every lane: four DPP
// steps within the rows of 16, then the four rows through scalar registers (a
// shuffle through LDS per step is ten times the latency).
template <int CTRL>
__device__ __forceinline__ float lane_perm(float v) {
  return __builtin_bit_cast(float, dpp_mov<CTRL>(__builtin_bit_cast(uint32_t, v)));
}
__device__ __forceinline__ float lane_read(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}
__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, lane_perm<0xB1>(v));   // lane ^ 1
  v = fmaxf(v, lane_perm<0x4E>(v));   // lane ^ 2
  v = fmaxf(v, lane_perm<0x141>(v));  // half rows mirrored
  v = fmaxf(v, lane_perm<0x140>(v));  // rows mirrored
  return fmaxf(fmaxf(lane_read(v, 0), lane_read(v, 16)), fmaxf(lane_read(v, 32), lane_read(v, 48)));
}
__device__ __forceinline__ float wave_sum(float v) {
  v += lane_perm<0xB1>(v);
  v += lane_perm<0x4E>(v);
  v += lane_perm<0x141>(v);
  v += lane_perm<0x140>(v);
  return (lane_read(v, 0) + lane_read(v, 16)) + (lane_read(v, 32) + lane_read(v, 48));
}

// One workgroup = one key-value head x one chunk of cache positions (a
// multiple of 64) x up to four of its query heads (eight would need 256
// registers), fp32 throughout.
//
// What bounds it: the latency of a chain of trips to memory (at 576 positions a
// head's keys and values are 288 KB).  So positions are cut into chunks over
// workgroups (9 x 8 heads there), each lane issues its D/4 key loads (lane =
// position, the cache keeps K transposed, so a wave reads 256 contiguous
// bytes) and its value loads before the position itself has arrived, and the
// chunks of a head meet without a second launch: each publishes (max, sum,
// unnormalised output), and the last to arrive joins them in chunk order (same
// bits every run), their outputs loaded together with their maxima and sums.
// The chunk that holds the position writes the new key and value to the cache
// and uses them from LDS.  A decode step of the 1B model (16 layers, position
// 575, fp16): 1559 us with the torch operations, 848 us with the first form of
// this kernel alone.  There a layer's launch takes 6.2 us; 8.7 us with the keys
// loaded after the position and the query, the outputs to join after their
// weights, a branch per element for the new key and value, and reductions by
// LDS shuffles.
//
// What that costs on long caches: a workgroup past the position has loaded its
// first block for nothing (32 / 8 heads of 64, position 100: 5.6 us in a cache of
// 648, 6.3 in one of 4096), and the chunks follow the cache, so that a position of
// 1500 is 24 chunks in a cache of 4096 (8.9 us), three in one of 32768 (16.7) and
// one, block after block, in one of 131072 (37; a layer with torch's operations
// took 470 us there, with this kernel 94).
template <int DT, int D, int GP>
__global__ __launch_bounds__(kAttnThreads) void attn_decode_kernel(AttnDecodeArgs a) {
  constexpr int DW = D / kAttnWaves;   // head elements per wave (keys)
  constexpr int PW = 64 / kAttnWaves;  // positions per wave (values)
  constexpr int VE = D / 64;           // value elements per lane
  constexpr int HW = (GP + kAttnWaves - 1) / kAttnWaves;
  __shared__ __attribute__((aligned(16))) float q_s[GP][D];
  __shared__ __attribute__((aligned(16))) float k_s[D];
  __shared__ __attribute__((aligned(16))) float v_s[D];
  __shared__ __attribute__((aligned(16))) float p_s[GP][64];
  __shared__ float alpha_s[GP];
  __shared__ float m_s[GP], l_s[GP];
  // cross-wave sums: scores [wave][head][position], then outputs [wave][head][d]
  __shared__ __attribute__((aligned(16))) float red[kAttnWaves][GP][D];
  __shared__ float w_s[kAttnMaxChunks][GP];
  __shared__ unsigned arrived;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = blockIdx.x, kvh = blockIdx.y, z = blockIdx.z;
  const int h0 = kvh * a.g + z * kAttnHeads;  // first query head
  const int g = min(a.g - z * kAttnHeads, GP);
  const int c0 = c * a.chunk;
  const float* __restrict__ kc = a.kc + (int64_t)kvh * D * a.max_len;
  const float* __restrict__ vc = a.vc + (int64_t)kvh * a.max_len * D;

  const int64_t pos64 = *a.pos;
  // Everything the chunk's first block needs, in the order of its use.  Clamped
  // to the cache and not to the position, so that nothing waits for the
  // position: what lies past it is not used below.
  static_assert(GP * (D / 2) <= kAttnThreads && kAttnThreads % D == 0, "one rotary pair per thread");
  const int qh = tid / (D / 2), qd = tid % (D / 2);
  const uint16_t* const qp = a.q + (int64_t)(h0 + min(qh, g - 1)) * D + qd;
  const uint16_t q1 = qp[0], q2 = qp[D / 2];
  const float rc = a.cos[qd], rs = a.sin[qd];
  const uint16_t* const kp = a.k + (int64_t)kvh * D + qd;
  const uint16_t k1 = kp[0], k2 = kp[D / 2], v1 = a.v[(int64_t)kvh * D + tid % D];
  float kr[DW], vr[PW][VE];
  auto load_k = [&](int p0) {
    const int p = min(p0 + lane, a.max_len - 1);
#pragma unroll
    for (int i = 0; i < DW; ++i) kr[i] = kc[(int64_t)(wv * DW + i) * a.max_len + p];
  };
  auto load_v = [&](int p0) {
#pragma unroll
    for (int i = 0; i < PW; ++i) {
      const float* vp = vc + (int64_t)min(p0 + wv * PW + i, a.max_len - 1) * D + lane * VE;
#pragma unroll
      for (int e = 0; e < VE; ++e) vr[i][e] = vp[e];
    }
  };
  __builtin_amdgcn_sched_barrier(0);
  load_k(c0);
  load_v(c0);
  __builtin_amdgcn_sched_barrier(0);

  // A position the cache does not hold: nothing is written to it, and a NaN query gives
  // a NaN output (at position 0; a branch of its own cost 0.1 us at D = 128).
  const bool in_cache = (uint64_t)pos64 < (uint64_t)a.max_len;
  const int pos = in_cache ? (int)pos64 : 0;
  const float qscale = in_cache ? a.qscale : __builtin_nanf("");
  const int active = pos / a.chunk + 1;
  if (c >= active) return;
  const int c1 = min(c0 + a.chunk, pos + 1);

  if (tid < GP * (D / 2)) {
    float r1, r2;
    rope_pair(act_bits_to_float(q1, DT), act_bits_to_float(q2, DT), rc, rs, &r1, &r2);
    q_s[qh][qd] = qh < g ? r1 * qscale : 0.f;
    q_s[qh][qd + D / 2] = qh < g ? r2 * qscale : 0.f;
  }
  if (c == active - 1) {
    if (tid < D / 2) {
      float r1, r2;
      rope_pair(act_bits_to_float(k1, DT), act_bits_to_float(k2, DT), rc, rs, &r1, &r2);
      k_s[tid] = r1;
      k_s[tid + D / 2] = r2;
      if (z == 0 && in_cache) {
        a.kc[((int64_t)kvh * D + tid) * a.max_len + pos] = r1;
        a.kc[((int64_t)kvh * D + tid + D / 2) * a.max_len + pos] = r2;
      }
    } else if (tid >= 128 && tid < 128 + D) {
      const float v = act_bits_to_float(v1, DT);
      v_s[tid - 128] = v;
      if (z == 0 && in_cache) a.vc[((int64_t)kvh * a.max_len + pos) * D + tid - 128] = v;
    }
  }
  __syncthreads();

  float m[HW], l[HW];
#pragma unroll
  for (int j = 0; j < HW; ++j) m[j] = -__builtin_inff(), l[j] = 0.f;
  float o[GP][VE];
#pragma unroll
  for (int h = 0; h < GP; ++h)
#pragma unroll
    for (int e = 0; e < VE; ++e) o[h][e] = 0.f;

  for (int p0 = c0; p0 < c1; p0 += 64) {
    const int p = p0 + lane;
    if (p0 + 64 > pos) {  // uniform: the block of the position
#pragma unroll
      for (int i = 0; i < DW; i += 4) {
        const f32x4 kn = *reinterpret_cast<const f32x4*>(&k_s[wv * DW + i]);
#pragma unroll
        for (int e = 0; e < 4; ++e) kr[i + e] = p == pos ? kn[e] : kr[i + e];
      }
      // Rows past the position get its value too, whose weight is 0 there: one select
      // a row.  An infinity or NaN must not meet those weights; it is put into its row
      // alone (rare, uniform).
      float vn[VE];
      bool odd = false;
#pragma unroll
      for (int e = 0; e < VE; ++e) {
        vn[e] = v_s[lane * VE + e];
        const bool finite = __builtin_fabsf(vn[e]) < __builtin_inff();
        const float fill = finite ? vn[e] : 0.f;
        odd = odd || !finite;
#pragma unroll
        for (int i = 0; i < PW; ++i) vr[i][e] = p0 + wv * PW + i >= pos ? fill : vr[i][e];
      }
      if (__builtin_expect(__ballot(odd) != 0, 0)) {
#pragma unroll
        for (int i = 0; i < PW; ++i)
#pragma unroll
          for (int e = 0; e < VE; ++e) vr[i][e] = p0 + wv * PW + i == pos ? vn[e] : vr[i][e];
      }
    }
    float s[GP];
#pragma unroll
    for (int h = 0; h < GP; ++h) s[h] = 0.f;
#pragma unroll
    for (int i = 0; i < DW; i += 4) {
#pragma unroll
      for (int h = 0; h < GP; ++h) {
        const f32x4 qv = *reinterpret_cast<const f32x4*>(&q_s[h][wv * DW + i]);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[h] = __builtin_fmaf(qv[e], kr[i + e], s[h]);
      }
    }
#pragma unroll
    for (int h = 0; h < GP; ++h) red[wv][h][lane] = s[h];
    if (p0 + 64 < c1) load_k(p0 + 64);  // the next block's, under this one's softmax
    __syncthreads();
#pragma unroll
    for (int j = 0; j < HW; ++j) {
      const int h = wv + j * kAttnWaves;
      if (h < GP) {
        float t = (red[0][h][lane] + red[1][h][lane]) + (red[2][h][lane] + red[3][h][lane]);
        if (p > pos) t = -__builtin_inff();
        const float mn = fmaxf(m[j], wave_max(t));
        // a chunk of -inf scores has no weight; a NaN score stays NaN
        const float pe = (mn == -__builtin_inff() && t == t) ? 0.f : __builtin_amdgcn_exp2f(t - mn);
        const float al = m[j] == mn ? 1.f : __builtin_amdgcn_exp2f(m[j] - mn);
        l[j] = l[j] * al + wave_sum(pe);
        m[j] = mn;
        p_s[h][lane] = pe;
        if (lane == 0) alpha_s[h] = al;
      }
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < GP; ++h) {
      const float al = alpha_s[h];
#pragma unroll
      for (int e = 0; e < VE; ++e) o[h][e] *= al;
#pragma unroll
      for (int i = 0; i < PW; i += 4) {
        const f32x4 pv = *reinterpret_cast<const f32x4*>(&p_s[h][wv * PW + i]);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int e = 0; e < VE; ++e) o[h][e] = __builtin_fmaf(pv[u], vr[i + u][e], o[h][e]);
      }
    }
    if (p0 + 64 < c1) load_v(p0 + 64);
    // red is next written after every wave has passed the barrier above
  }
#pragma unroll
  for (int j = 0; j < HW; ++j) {
    const int h = wv + j * kAttnWaves;
    if (h < GP && lane == 0) m_s[h] = m[j], l_s[h] = l[j];
  }
#pragma unroll
  for (int h = 0; h < GP; ++h)
#pragma unroll
    for (int e = 0; e < VE; ++e) red[wv][h][lane * VE + e] = o[h][e];
  __syncthreads();

  const int n = g * D;
  constexpr int stride = kAttnHeads * (D + 2);
  const int64_t slice = (int64_t)kvh * gridDim.z + z;
  if (active == 1) {
    for (int i = tid; i < n; i += kAttnThreads) {
      const int h = i / D, d = i % D;
      const float t = (red[0][h][d] + red[1][h][d]) + (red[2][h][d] + red[3][h][d]);
      a.out[(int64_t)h0 * D + i] = float_to_act_bits<DT>(t / l_s[h]);
    }
    return;
  }
  // publish (device-coherent stores, waited for), then count the arrival
  float* const mine = a.part + (slice * a.chunks + c) * stride;
  for (int i = tid; i < n; i += kAttnThreads) {
    const int h = i / D, d = i % D;
    const float t = (red[0][h][d] + red[1][h][d]) + (red[2][h][d] + red[3][h][d]);
    __hip_atomic_store(mine + i, t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (tid < g) {
    __hip_atomic_store(mine + n + tid, m_s[tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(mine + n + g + tid, l_s[tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __builtin_amdgcn_s_waitcnt(0);  // the stores have reached the level all XCDs share
  __syncthreads();
  if (tid == 0) arrived = __hip_atomic_fetch_add(a.cnt + slice, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (arrived != (unsigned)(active - 1)) return;
  if (tid == 0) __hip_atomic_store(a.cnt + slice, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const float* const all = a.part + slice * a.chunks * stride;
  // The first chunks' outputs travel with the maxima and sums.  Twelve: ten chunks
  // (cache 648) 6.19 us a launch, 6.45 with four ahead, 6.51 with eight, 6.29 with
  // sixteen; two chunks 5.56, 5.46 with four.
  constexpr int AHEAD = 12;
  auto part_at = [&](int cc, int i) {
    return __hip_atomic_load(all + min(cc, active - 1) * stride + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  float first[AHEAD];
#pragma unroll
  for (int u = 0; u < AHEAD; ++u) first[u] = part_at(u, min(tid, n - 1));
  // lane = chunk (at most 64): its weight relative to the head's maximum
#pragma unroll
  for (int j = 0; j < HW; ++j) {
    const int h = wv + j * kAttnWaves;
    if (h < g) {
      float mc = -__builtin_inff(), lc = 0.f;
      if (lane < active) {
        mc = __hip_atomic_load(all + lane * stride + n + h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        lc = __hip_atomic_load(all + lane * stride + n + g + h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      const float mx = wave_max(mc);
      const float w = lane < active ? __builtin_amdgcn_exp2f(mc - mx) : 0.f;
      const float sum = wave_sum(lane < active ? w * lc : 0.f);
      if (lane < active) w_s[lane][h] = w;
      if (lane == 0) l_s[h] = sum;
    }
  }
  __syncthreads();
  for (int i = tid; i < n; i += kAttnThreads) {
    const int h = i / D;
    float t = 0.f;
    if (i != tid) {
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) first[u] = part_at(u, i);
    }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
      if (u < active) t = __builtin_fmaf(w_s[u][h], first[u], t);
    for (int cc = AHEAD; cc < active; cc += 8) {
      float r[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) r[u] = part_at(cc + u, i);
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (cc + u < active) t = __builtin_fmaf(w_s[cc + u][h], r[u], t);
    }
    a.out[(int64_t)h0 * D + i] = float_to_act_bits<DT>(t / l_s[h]);
  }
}

// ---------------------------------------------------------------- prompt
struct AttnPrefillArgs {
  const uint16_t* q;  // [T, nkv * g * D]
  const uint16_t* k;  // [T, nkv * D]
  const uint16_t* v;
  const float* cos;   // [T, D / 2]
  const float* sin;
  float* kc;          // [nkv, D, max_len]
  float* vc;          // [nkv, max_len, D]
  uint16_t* out;      // [T, nkv * g * D]
  float qscale;
  int g, nkv, T, pos0, max_len;
};

// Keys (rotated) and values of T tokens into the caches at pos0..: one workgroup
// per 64 tokens of one head, the keys transposed through LDS so that cache rows
// are written 256 bytes at a time.
template <int DT, int D>
__global__ __launch_bounds__(256) void rope_cache_kernel(AttnPrefillArgs a) {
  __shared__ float tile[D][65];
  const int tid = threadIdx.x, t0 = blockIdx.x * 64, h = blockIdx.y;
  const int64_t ld = (int64_t)a.nkv * D;
  constexpr int CH = D / 16;  // pairs of 8-element chunks per token
#pragma unroll
  for (int it = 0; it < CH / 4; ++it) {
    const int i = tid + it * 256, tl = i / CH, d = (i % CH) * 8, t = t0 + tl;
    if (t < a.T) {
      const uint16_t* kp = a.k + t * ld + (int64_t)h * D + d;
      float x1[8], x2[8];
      unpack8<DT>(*reinterpret_cast<const u32x4*>(kp), x1);
      unpack8<DT>(*reinterpret_cast<const u32x4*>(kp + D / 2), x2);
      const float *cp = a.cos + (int64_t)t * (D / 2) + d, *sp = a.sin + (int64_t)t * (D / 2) + d;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float r1, r2;
        rope_pair(x1[j], x2[j], cp[j], sp[j], &r1, &r2);
        tile[d + j][tl] = r1;
        tile[d + D / 2 + j][tl] = r2;
      }
    }
  }
#pragma unroll
  for (int it = 0; it < D / 32; ++it) {
    const int i = tid + it * 256, t = t0 + i / (D / 8), d = (i % (D / 8)) * 8;
    if (t < a.T) {
      float x[8];
      unpack8<DT>(*reinterpret_cast<const u32x4*>(a.v + t * ld + (int64_t)h * D + d), x);
      float* vp = a.vc + ((int64_t)h * a.max_len + a.pos0 + t) * D + d;
      *reinterpret_cast<f32x4*>(vp) = f32x4{x[0], x[1], x[2], x[3]};
      *reinterpret_cast<f32x4*>(vp + 4) = f32x4{x[4], x[5], x[6], x[7]};
    }
  }
  __syncthreads();
  const int lane = tid & 63, t = t0 + lane;
  if (t < a.T)
    for (int d = tid >> 6; d < D; d += 4)
      a.kc[((int64_t)h * D + d) * a.max_len + a.pos0 + t] = tile[d][lane];
}

// Causal attention of a prompt over the fp32 caches (rope_cache_kernel has
// filled them up to pos0 + T), online softmax, fp32 MFMA 16x16x4 for both
// products, one rounding of the output.
//
// One workgroup = two column tiles of 16 queries (two heads that share a
// key-value head, or 32 tokens of one head where their number per key-value
// head is odd); its four waves take every fourth block of 64 positions and join
// through LDS, which fills the chip at prompts of a few hundred tokens (500
// tokens x 32 heads: 512 workgroups).  Both products are computed transposed:
//   S^T[pos][query] = K[pos][d] Q[query][d],  O^T[n][query] = V[pos][n] P[query][pos]
// so that the softmax statistics of a query sit in its lane (4 lanes per
// query), and the four accumulator registers of S^T are, as they stand, the B
// operands of the second product: the order of positions within a block is
// free, so row 4j + r of the S^T tile c is position 16j + 4r + c (a lane's
// 128-bit key load covers four tiles), and the r-th step over tile c multiplies
// by V rows 16j + 4r + c.  What bounds it: the matrix cores' fp32 rate (157
// TFLOP/s) and the latency that stays visible: half of a block's values travel
// under its softmax, the rest and half of the next block's keys under its second
// product (all of it would not fit the registers of two waves per SIMD).  Four
// layers of the 1B model and its head on 500 tokens: 1764 us with torch's batched
// fp32 products, masks and copies; this kernel takes 21.7 us of a layer there (29 us
// with each load next to its use) and the cache kernel 5.1.  Head size 128 takes all
// 512 registers, one wave per SIMD, without scratch (an attention module of 16 / 4
// heads on 500 tokens 75 us, 194 with torch's operations; 4096 tokens 786 and 3079).
template <int DT, int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 64 ? 2 : 1))) void attn_prefill_kernel(
    AttnPrefillArgs a) {
  constexpr int DQ = D / 4;   // head elements per lane (keys and queries)
  constexpr int NT = D / 16;  // row tiles of O^T
  constexpr int VH = D / 64;  // 128-bit value loads per position
  constexpr int DH = DQ / 2;
  __shared__ __attribute__((aligned(16))) float o_s[4][2][16][D + 4];
  __shared__ float m_s[4][2][16], l_s[4][2][16];

  const int tid = threadIdx.x, lane = tid & 63, i = lane & 15, j = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kvh = blockIdx.x % a.nkv, pair = blockIdx.x / a.nkv;
  const int tile = gridDim.y - 1 - blockIdx.y;  // the longest rows first
  const bool two_heads = (a.g & 1) == 0;
  const int head0 = kvh * a.g + (two_heads ? 2 * pair : pair);
  const int tb = tile * (two_heads ? 16 : 32);
  const int64_t ld = (int64_t)a.nkv * a.g * D;

  float qf[2][DQ];
  int qpos[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int t = min(tb + (two_heads ? 0 : 16 * c) + i, a.T - 1);
    qpos[c] = a.pos0 + tb + (two_heads ? 0 : 16 * c) + i;
    const uint16_t* qp = a.q + t * ld + (int64_t)(head0 + (two_heads ? c : 0)) * D;
    const int d0 = j * DQ, dc = (j & 1) * DQ;  // own elements; their place in a half
    const float *cp = a.cos + (int64_t)t * (D / 2) + dc, *sp = a.sin + (int64_t)t * (D / 2) + dc;
#pragma unroll
    for (int u = 0; u < DQ; u += 8) {
      float x[8], y[8];
      unpack8<DT>(*reinterpret_cast<const u32x4*>(qp + d0 + u), x);
      unpack8<DT>(*reinterpret_cast<const u32x4*>(qp + (j ^ 2) * DQ + u), y);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
#pragma clang fp contract(off)
        const float xc = x[e] * cp[u + e], ys = y[e] * sp[u + e];
        qf[c][u + e] = (j < 2 ? xc - ys : xc + ys) * a.qscale;
      }
    }
  }

  // the head's keys, and its values up to the prompt's end (below 2 GiB each, the host checks)
  const int L = a.pos0 + a.T;
  const int64_t head = (int64_t)kvh * D * a.max_len;
  const __amdgpu_buffer_rsrc_t rk =
      __builtin_amdgcn_make_buffer_rsrc((void*)(a.kc + head), (short)0, D * a.max_len * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t rv =
      __builtin_amdgcn_make_buffer_rsrc((void*)(a.vc + head), (short)0, D * L * 4, 0x00020000);
  const int blocks = (min(a.pos0 + tb + (two_heads ? 15 : 31), L - 1) >> 6) + 1;
  float m[2], l[2];
  f32x4 o[2][NT];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    m[c] = -__builtin_inff(), l[c] = 0.f;
#pragma unroll
    for (int n = 0; n < NT; ++n) o[c][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // Keys of a block, lane i of part j: positions p0 + 4 i .. + 3 of elements
  // j DQ + d.  The last block of a cache whose end lies inside it is read
  // element by element, clamped.
  // (Buffer loads: the element enters through the scalar offset, so the 16 or 32
  // rows need no address registers of their own.)
  const uint32_t k_lane = (uint32_t)(j * DQ) * (uint32_t)a.max_len * 4u;
  // half h: elements [h DQ / 2, + DQ / 2)
  auto load_k = [&](int p0, int h, f32x4* kk) {
    const uint32_t row = (uint32_t)a.max_len * 4u;
    if (p0 + 64 <= a.max_len) {
      const uint32_t vo = k_lane + (uint32_t)(p0 + 4 * i) * 4u;
#pragma unroll
      for (int d = h * DH; d < (h + 1) * DH; ++d)
        kk[d] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rk, vo, (uint32_t)d * row, 0));
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t vo = k_lane + (uint32_t)min(p0 + 4 * i + u, a.max_len - 1) * 4u;
#pragma unroll
        for (int d = h * DH; d < (h + 1) * DH; ++d)
          kk[d][u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rk, vo, (uint32_t)d * row, 0));
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // values of a block, r in {2 h, 2 h + 1}; rows past the prompt hold nothing yet and
  // lie past the resource's range, which reads zeros (a row of the prompt in their
  // place would add 0 x infinity where it holds one)
  f32x4 vv[2][8][VH];
  auto load_v = [&](int p0, int h) {
#pragma unroll
    for (int x = 0; x < 8; ++x) {
      const uint32_t vo = (uint32_t)((p0 + 16 * j + 8 * h + x) * D + 4 * i) * 4u;
#pragma unroll
      for (int hh = 0; hh < VH; ++hh)
        vv[h][x][hh] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rv, vo, 256u * (uint32_t)hh, 0));
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  f32x4 kk[DQ];
  if (wv < blocks) {
    load_k(wv * 64, 0, kk);
    load_k(wv * 64, 1, kk);
  }
  for (int b = wv; b < blocks; b += 4) {
    const int p0 = b * 64;
    f32x4 s[2][4];
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int u = 0; u < 4; ++u) s[c][u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < DQ; ++d)
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int c = 0; c < 2; ++c)
          s[c][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[d][u], qf[c][d], s[c][u], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    load_v(p0, 0);  // in flight under the softmax
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      float mx = -__builtin_inff();
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (p0 + 16 * j + 4 * r + u > qpos[c]) s[c][u][r] = -__builtin_inff();
          mx = fmaxf(mx, s[c][u][r]);
        }
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float mn = fmaxf(m[c], mx);
      const float al = m[c] == mn ? 1.f : __builtin_amdgcn_exp2f(m[c] - mn);
      m[c] = mn;
      float sum = 0.f;
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float t = s[c][u][r];
          // -inf scores before any finite one weigh nothing; a NaN score stays NaN
          const float p = (mn == -__builtin_inff() && t == t) ? 0.f : __builtin_amdgcn_exp2f(t - mn);
          s[c][u][r] = p;
          sum += p;
        }
      l[c] = l[c] * al + sum;
#pragma unroll
      for (int n = 0; n < NT; ++n) o[c][n] *= al;
    }
    __builtin_amdgcn_sched_barrier(0);
    auto product = [&](int h) {
#pragma unroll
      for (int x = 0; x < 8; ++x)
#pragma unroll
        for (int hh = 0; hh < VH; ++hh)
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int c = 0; c < 2; ++c)
              o[c][4 * hh + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                  vv[h][x][hh][e], s[c][x & 3][2 * h + (x >> 2)], o[c][4 * hh + e], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    };
    // each half of the loads ahead goes out as soon as registers for it are free
    load_v(p0, 1);
    product(0);
    if (b + 4 < blocks) load_k(p0 + 256, 0, kk);
    product(1);
    if (b + 4 < blocks) load_k(p0 + 256, 1, kk);
  }
  // join the four waves: lane (j, i) holds O[query i][64 hh + 16 j + 4 r + e]
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    l[c] += __shfl_xor(l[c], 16, 64);
    l[c] += __shfl_xor(l[c], 32, 64);
    if (j == 0) m_s[wv][c][i] = m[c], l_s[wv][c][i] = l[c];
#pragma unroll
    for (int hh = 0; hh < VH; ++hh)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        *reinterpret_cast<f32x4*>(&o_s[wv][c][i][64 * hh + 16 * j + 4 * r]) =
            f32x4{o[c][4 * hh][r], o[c][4 * hh + 1][r], o[c][4 * hh + 2][r], o[c][4 * hh + 3][r]};
  }
  __syncthreads();
  constexpr int VPQ = D / 8;  // 8-element chunks per query
#pragma unroll
  for (int it = 0; it < 2 * 16 * VPQ / 256; ++it) {
    const int x = tid + it * 256, c = x / (16 * VPQ), qi = (x / VPQ) % 16, n = (x % VPQ) * 8;
    const int t = tb + (two_heads ? 0 : 16 * c) + qi;
    const float mx = fmaxf(fmaxf(m_s[0][c][qi], m_s[1][c][qi]), fmaxf(m_s[2][c][qi], m_s[3][c][qi]));
    float sum = 0.f, acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = __builtin_amdgcn_exp2f(m_s[w][c][qi] - mx);
      sum = __builtin_fmaf(f, l_s[w][c][qi], sum);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = __builtin_fmaf(f, o_s[w][c][qi][n + e], acc[e]);
    }
    if (t < a.T) {
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] /= sum;
      *reinterpret_cast<u32x4*>(a.out + t * ld + (int64_t)(head0 + (two_heads ? c : 0)) * D + n) = pack8<DT>(acc);
    }
  }
}

constexpr int kNormThreads = 256;
constexpr int kNormMaxVecs = 8;  // 16-byte vectors per thread: rows of up to 16384

// The same words, which the compiler takes for others if ON.  It computes what
// follows a conditional load inside the condition and keeps values that two passes
// unpack, so that all of a row's fp16 conversions live at once.
template <bool ON>
__device__ __forceinline__ u32x4 opaque(u32x4 v) {
  if constexpr (ON) asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
  return v;
}

// y = x / sqrt(mean(x^2) + eps) * weight, rows of n values, fp32 inside and one
// rounding; with a delta the row is first x + delta, rounded to the dtype (the
// residual stream) and written to sum.  One workgroup per row, the row held in
// registers (VPT vectors per thread) between the two passes over it.  For one
// row it is bound by launch and one trip to memory, for many by HBM: fusing
// the addition saves a launch and a read and write of the row.  With
// silu_mul_kernel, the 1B model's decode step went from 848 to 728 us.
template <int DT, int VPT, bool ADD>
__global__ __launch_bounds__(kNormThreads) void rmsnorm_kernel(const uint16_t* __restrict__ x,
                                                               const uint16_t* __restrict__ delta,
                                                               const uint16_t* __restrict__ weight, int n, float eps,
                                                               uint16_t* __restrict__ sum, uint16_t* __restrict__ y) {
  // fp16 rows above 4096: 8 vectors with a delta took 502 registers and 772 bytes of
  // scratch a lane, 111 registers so (2048 x 16384: 393 -> 43 us, without a delta 51 ->
  // 23).  Narrower rows fit either way and are 2-3 % faster converted under the
  // condition; bf16 unpacks by shifts, which the compiler repeats by itself.
  constexpr bool OQ = DT == W4_DTYPE_FP16 && VPT >= 4;
  __shared__ float part[kNormThreads / 64];
  const uint32_t tid = threadIdx.x, vecs = (uint32_t)n / 8;
  const int64_t row = (int64_t)blockIdx.x * n;
  x += row, y += row;
  if constexpr (ADD) delta += row, sum += row;
  u32x4 xr[VPT], dr[VPT], wr[VPT];
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const uint32_t v = tid + i * kNormThreads;
    xr[i] = dr[i] = wr[i] = u32x4{0u, 0u, 0u, 0u};
    if (v < vecs) {
      xr[i] = *reinterpret_cast<const u32x4*>(x + v * 8);
      if constexpr (ADD) dr[i] = *reinterpret_cast<const u32x4*>(delta + v * 8);
      wr[i] = *reinterpret_cast<const u32x4*>(weight + v * 8);
    }
  }
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    float xv[8];
    unpack8<DT>(opaque<OQ>(xr[i]), xv);
    if constexpr (ADD) {
      float dv[8];
      unpack8<DT>(opaque<OQ>(dr[i]), dv);
#pragma unroll
      for (int j = 0; j < 8; ++j) xv[j] += dv[j];
      xr[i] = pack8<DT>(xv);
      const uint32_t v = tid + i * kNormThreads;
      if (v < vecs) *reinterpret_cast<u32x4*>(sum + v * 8) = xr[i];
      unpack8<DT>(xr[i], xv);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) sq = __builtin_fmaf(xv[j], xv[j], sq);
  }
  sq = wave_sum(sq);
  if ((tid & 63) == 0) part[tid >> 6] = sq;
  __syncthreads();
  const float r = 1.0f / sqrtf(((part[0] + part[1]) + (part[2] + part[3])) / (float)n + eps);
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const uint32_t v = tid + i * kNormThreads;
    float xv[8], wv[8], o[8];
    unpack8<DT>(opaque<OQ>(xr[i]), xv);
    unpack8<DT>(opaque<OQ>(wr[i]), wv);
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = xv[j] * r * wv[j];
    if (v < vecs) *reinterpret_cast<u32x4*>(y + v * 8) = pack8<DT>(o);
  }
}

// Logits of one token: y = rmsnorm(x + delta) * W^T, W [N, K] 16-bit, fp32 sums,
// one rounding of the norm's output and of y.
//
// What bounds it: HBM, and only reads.  A wave holds the normalized row in its
// lanes and takes a few rows of W at a time, 16 bytes a lane and load, the next
// rows' loads issued before the sums across lanes; it computes the norm itself
// while its first rows travel, so there is no barrier and no launch before it.
// Past the caches (non-temporal): 128256 x 2048 in bf16 79 us (6.6 TB/s; 92 us
// cached), where the norm's launch and the library's product take 103-121;
// 32000 x 2048 21.7 us (cached 23.5, library 33.5), 1024 x 2048 3.3 (10.2).
// A decode step of the 1B model, fp16: 588 -> 534 us.
struct NormHeadArgs {
  const uint16_t* x;      // [K]
  const uint16_t* delta;  // [K], may be null
  const uint16_t* norm;   // [K]
  const uint16_t* w;      // [N, K]
  uint16_t* y;            // [N]
  int N, K;
  float eps;
};
constexpr int kHeadMaxChunks = 8;  // rows of up to 8 * 512 values
constexpr int head_rows(int chunks) { return chunks <= 2 ? 4 : 2; }

template <int DT, int NC>
__global__ __launch_bounds__(256) void norm_head_kernel(NormHeadArgs a) {
  // rows a wave takes at a time: twice as many measured 1-4 % slower (fewer waves fit)
  constexpr int R = head_rows(NC);
  // fp16 rows above 2048: with every conversion of the norm's operands alive at once,
  // rows above 3584 took 296 registers, one wave per SIMD (8000 x 4096: 24.0 us, now
  // 14.2; 32000 x 4096 48.6, now 40.6; 128256 x 3072 117.5, now 117.3).
  constexpr bool OQ = DT == W4_DTYPE_FP16 && NC >= 5;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int waves = (int)gridDim.x * 4;
  int n0 = ((int)blockIdx.x * 4 + wv) * R;
  // the last chunk's lanes past K load its first values and count as zero
  const bool in = (NC - 1) * 512 + lane * 8 < a.K;
  auto col = [&](int c) { return c * 512 + (c < NC - 1 || in ? lane * 8 : 0); };
  u32x4 xr[NC], dr[NC], nr[NC], w[R][NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    xr[c] = *reinterpret_cast<const u32x4*>(a.x + col(c));
    dr[c] = u32x4{0u, 0u, 0u, 0u};
    if (a.delta) dr[c] = *reinterpret_cast<const u32x4*>(a.delta + col(c));
    nr[c] = *reinterpret_cast<const u32x4*>(a.norm + col(c));
  }
  __builtin_amdgcn_sched_barrier(0);
  auto load = [&](int n) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint16_t* row = a.w + (int64_t)min(n + r, a.N - 1) * a.K;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const u32x4* at = reinterpret_cast<const u32x4*>(row + col(c));
        w[r][c] = __builtin_nontemporal_load(at);
      }
    }
  };
  load(n0);
  __builtin_amdgcn_sched_barrier(0);
  // every wave normalizes the row for itself: no barrier
  float x[NC][8], sq = 0.f;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    unpack8<DT>(opaque<OQ>(xr[c]), x[c]);
    if (a.delta) {
      float d[8];
      unpack8<DT>(opaque<OQ>(dr[c]), d);
#pragma unroll
      for (int j = 0; j < 8; ++j) x[c][j] += d[j];
      unpack8<DT>(pack8<DT>(x[c]), x[c]);
    }
    if (c == NC - 1 && !in) {
#pragma unroll
      for (int j = 0; j < 8; ++j) x[c][j] = 0.f;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) sq = __builtin_fmaf(x[c][j], x[c][j], sq);
  }
  const float rms = 1.0f / sqrtf(wave_sum(sq) / (float)a.K + a.eps);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    float g[8];
    unpack8<DT>(opaque<OQ>(nr[c]), g);
#pragma unroll
    for (int j = 0; j < 8; ++j) x[c][j] = x[c][j] * rms * g[j];
    unpack8<DT>(pack8<DT>(x[c]), x[c]);
  }
  for (; n0 < a.N;) {
    float y[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float t0 = 0.f, t1 = 0.f;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        if (c == NC - 1 && !in) w[r][c] = u32x4{0u, 0u, 0u, 0u};
        float v[8];
        unpack8<DT>(w[r][c], v);
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
          t0 = __builtin_fmaf(v[j], x[c][j], t0);
          t1 = __builtin_fmaf(v[j + 1], x[c][j + 1], t1);
        }
      }
      y[r] = t0 + t1;
    }
    const int n = n0;
    n0 += waves * R;
    if (n0 < a.N) load(n0);
    uint32_t bits = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint16_t b = float_to_act_bits<DT>(wave_sum(y[r]));
      bits = lane == r ? b : bits;
    }
    if (lane < R && n + lane < a.N) a.y[n + lane] = (uint16_t)bits;
  }
}

// y = silu(gate) * up, fp32 inside and one rounding (the separate operations
// round silu(gate) too).  Eight values per thread: HBM-bound once it fills the
// chip, a launch and a trip to memory below that.  One launch and pass less
// than silu and multiply: an MLP of 2048 x 2048 x 8192 from 222 to 205 us.
template <int DT>
__global__ __launch_bounds__(256) void silu_mul_kernel(const uint16_t* __restrict__ gate,
                                                       const uint16_t* __restrict__ up, int64_t vecs,
                                                       uint16_t* __restrict__ y) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= vecs) return;
  float g[8], u[8];
  unpack8<DT>(reinterpret_cast<const u32x4*>(gate)[i], g);
  unpack8<DT>(reinterpret_cast<const u32x4*>(up)[i], u);
#pragma unroll
  for (int j = 0; j < 8; ++j) u[j] *= g[j] / (1.0f + __expf(-g[j]));
  reinterpret_cast<u32x4*>(y)[i] = pack8<DT>(u);
}

}  // namespace w4

using namespace w4host;

namespace {

// Positions per chunk: 64, more for caches past 4096 positions so that a head
// has at most 64 chunks (its last workgroup reads one lane per chunk).
int attn_chunk(int64_t max_len) {
  return 64 * (int)((max_len + 64 * w4::kAttnMaxChunks - 1) / (64 * w4::kAttnMaxChunks));
}

int64_t attn_slices(int64_t nh, int64_t nkv) { return (nh / nkv + w4::kAttnHeads - 1) / w4::kAttnHeads; }

bool attn_decode_shape_ok(int64_t nh, int64_t nkv, int64_t head_dim, int64_t max_len) {
  return nkv >= 1 && nh >= nkv && nh % nkv == 0 &&
         (head_dim == 64 || head_dim == 128) && max_len >= 1 && max_len < (1LL << 24) &&
         nkv * attn_slices(nh, nkv) <= (int64_t)(W4_WORKSPACE_COUNTER_BYTES / 4);
}

template <int DT, int D>
void launch_decode(const w4::AttnDecodeArgs& a, int nkv, hipStream_t st) {
  const dim3 grid((unsigned)a.chunks, (unsigned)nkv, (unsigned)attn_slices((int64_t)a.g * nkv, nkv));
  const dim3 block(w4::kAttnThreads);
  if (a.g == 1) hipLaunchKernelGGL((w4::attn_decode_kernel<DT, D, 1>), grid, block, 0, st, a);
  else if (a.g == 2) hipLaunchKernelGGL((w4::attn_decode_kernel<DT, D, 2>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((w4::attn_decode_kernel<DT, D, 4>), grid, block, 0, st, a);
}

}  // namespace

namespace {

template <int DT, int D>
void launch_prefill(const w4::AttnPrefillArgs& a, hipStream_t st) {
  hipLaunchKernelGGL((w4::rope_cache_kernel<DT, D>), dim3((unsigned)((a.T + 63) / 64), (unsigned)a.nkv), dim3(256), 0,
                     st, a);
  const bool two_heads = a.g % 2 == 0;
  const int pairs = a.nkv * (two_heads ? a.g / 2 : a.g), rows = two_heads ? 16 : 32;
  hipLaunchKernelGGL((w4::attn_prefill_kernel<DT, D>), dim3((unsigned)pairs, (unsigned)((a.T + rows - 1) / rows)),
                     dim3(256), 0, st, a);
}

}  // namespace

extern "C" int w4_attention_prefill(const void* q, const void* k, const void* v, int dtype, int64_t tokens,
                                    int64_t num_heads, int64_t num_kv_heads, int64_t head_dim, const float* cos,
                                    const float* sin, float* k_cache, float* v_cache, int64_t max_len, int64_t pos0,
                                    void* out, void* stream) {
  clear_error();
  if (dtype != W4_DTYPE_BF16 && dtype != W4_DTYPE_FP16)
    return fail(W4_ERR_INVALID, "w4_attention_prefill: dtype must be bf16 or fp16 (got code %d)", dtype);
  if (num_kv_heads < 1 || num_kv_heads > 65535 || num_heads < num_kv_heads || num_heads % num_kv_heads != 0 ||
      num_heads >= (1LL << 24) || (head_dim != 64 && head_dim != 128) || max_len >= (1LL << 22))
    return fail(W4_ERR_UNSUPPORTED,
                "w4_attention_prefill: %lld query / %lld key-value heads of %lld over %lld positions "
                "(heads of 64 or 128)",
                (long long)num_heads, (long long)num_kv_heads, (long long)head_dim, (long long)max_len);
  if (tokens < 0 || pos0 < 0 || pos0 > max_len || tokens > max_len - pos0 || tokens > 65535 * 16)
    return fail(W4_ERR_INVALID, "w4_attention_prefill: %lld tokens at %lld in a cache of %lld", (long long)tokens,
                (long long)pos0, (long long)max_len);
  if (tokens == 0) return W4_OK;
  if (!q || !k || !v || !cos || !sin || !k_cache || !v_cache || !out)
    return fail(W4_ERR_INVALID, "w4_attention_prefill: null pointer");
  if ((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)v_cache | (uintptr_t)out) % 16) != 0)
    return fail(W4_ERR_INVALID, "w4_attention_prefill: operands must be 16-byte aligned");
  w4::AttnPrefillArgs a{};
  a.q = static_cast<const uint16_t*>(q);
  a.k = static_cast<const uint16_t*>(k);
  a.v = static_cast<const uint16_t*>(v);
  a.cos = cos;
  a.sin = sin;
  a.kc = k_cache;
  a.vc = v_cache;
  a.out = static_cast<uint16_t*>(out);
  a.qscale = w4::kLog2e / sqrtf((float)head_dim);
  a.g = (int)(num_heads / num_kv_heads);
  a.nkv = (int)num_kv_heads;
  a.T = (int)tokens;
  a.pos0 = (int)pos0;
  a.max_len = (int)max_len;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == W4_DTYPE_BF16) {
    if (head_dim == 64) launch_prefill<W4_DTYPE_BF16, 64>(a, st);
    else launch_prefill<W4_DTYPE_BF16, 128>(a, st);
  } else {
    if (head_dim == 64) launch_prefill<W4_DTYPE_FP16, 64>(a, st);
    else launch_prefill<W4_DTYPE_FP16, 128>(a, st);
  }
  return check_launch("w4_attention_prefill");
}

extern "C" size_t w4_attention_decode_workspace_bytes(int64_t num_heads, int64_t num_kv_heads, int64_t head_dim,
                                                      int64_t max_len) {
  if (!attn_decode_shape_ok(num_heads, num_kv_heads, head_dim, max_len)) return 0;
  const int64_t chunk = attn_chunk(max_len), chunks = (max_len + chunk - 1) / chunk;
  return W4_WORKSPACE_COUNTER_BYTES + (size_t)(num_kv_heads * attn_slices(num_heads, num_kv_heads) * chunks *
                                             w4::kAttnHeads * (head_dim + 2)) * 4;
}

extern "C" int w4_attention_decode(const void* q, const void* k, const void* v, int dtype, int64_t num_heads,
                                   int64_t num_kv_heads, int64_t head_dim, const float* cos, const float* sin,
                                   float* k_cache, float* v_cache, int64_t max_len, const int64_t* pos, void* out,
                                   void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  if (dtype != W4_DTYPE_BF16 && dtype != W4_DTYPE_FP16)
    return fail(W4_ERR_INVALID, "w4_attention_decode: dtype must be bf16 or fp16 (got code %d)", dtype);
  if (!attn_decode_shape_ok(num_heads, num_kv_heads, head_dim, max_len))
    return fail(W4_ERR_UNSUPPORTED,
                "w4_attention_decode: %lld query / %lld key-value heads of %lld over %lld positions "
                "(heads of 64 or 128)",
                (long long)num_heads, (long long)num_kv_heads, (long long)head_dim, (long long)max_len);
  if (!q || !k || !v || !cos || !sin || !k_cache || !v_cache || !pos || !out)
    return fail(W4_ERR_INVALID, "w4_attention_decode: null pointer");
  const size_t need = w4_attention_decode_workspace_bytes(num_heads, num_kv_heads, head_dim, max_len);
  if (workspace == nullptr || workspace_bytes < need || ((uintptr_t)workspace % 256) != 0)
    return fail(W4_ERR_WORKSPACE, "w4_attention_decode: needs a 256-byte aligned workspace of %zu bytes (got %zu)",
                need, workspace_bytes);
  w4::AttnDecodeArgs a{};
  a.q = static_cast<const uint16_t*>(q);
  a.k = static_cast<const uint16_t*>(k);
  a.v = static_cast<const uint16_t*>(v);
  a.cos = cos;
  a.sin = sin;
  a.kc = k_cache;
  a.vc = v_cache;
  a.pos = pos;
  a.out = static_cast<uint16_t*>(out);
  a.cnt = static_cast<unsigned*>(workspace);
  a.part = reinterpret_cast<float*>(static_cast<char*>(workspace) + W4_WORKSPACE_COUNTER_BYTES);
  a.qscale = w4::kLog2e / sqrtf((float)head_dim);
  a.g = (int)(num_heads / num_kv_heads);
  a.max_len = (int)max_len;
  a.chunk = attn_chunk(max_len);
  a.chunks = (int)((max_len + a.chunk - 1) / a.chunk);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int nkv = (int)num_kv_heads;
  if (dtype == W4_DTYPE_BF16) {
    if (head_dim == 64) launch_decode<W4_DTYPE_BF16, 64>(a, nkv, st);
    else launch_decode<W4_DTYPE_BF16, 128>(a, nkv, st);
  } else {
    if (head_dim == 64) launch_decode<W4_DTYPE_FP16, 64>(a, nkv, st);
    else launch_decode<W4_DTYPE_FP16, 128>(a, nkv, st);
  }
  return check_launch("w4_attention_decode");
}

namespace {

// HIP refuses launches of 2^32 threads and more.
constexpr int64_t kMaxGrid256 = 0xFFFFFFFFll / 256;

template <int DT, bool ADD>
void launch_rmsnorm(const uint16_t* x, const uint16_t* delta, const uint16_t* weight, int64_t rows, int n, float eps,
                    uint16_t* sum, uint16_t* y, hipStream_t st) {
  const dim3 grid((unsigned)rows), block(w4::kNormThreads);
  const int vpt = (n / 8 + w4::kNormThreads - 1) / w4::kNormThreads;
#define W4_NORM(V) \
  hipLaunchKernelGGL((w4::rmsnorm_kernel<DT, V, ADD>), grid, block, 0, st, x, delta, weight, n, eps, sum, y)
  if (vpt <= 1) W4_NORM(1);
  else if (vpt <= 2) W4_NORM(2);
  else if (vpt <= 4) W4_NORM(4);
  else W4_NORM(8);
#undef W4_NORM
}

}  // namespace

extern "C" int w4_rmsnorm(const void* x, const void* delta, const void* weight, int dtype, int64_t rows, int64_t n,
                          float eps, void* sum, void* y, void* stream) {
  clear_error();
  if (dtype != W4_DTYPE_BF16 && dtype != W4_DTYPE_FP16)
    return fail(W4_ERR_INVALID, "w4_rmsnorm: dtype must be bf16 or fp16 (got code %d)", dtype);
  if (rows < 0 || rows > kMaxGrid256 || n < 8 || n % 8 != 0 || n > 8 * w4::kNormThreads * w4::kNormMaxVecs)
    return fail(W4_ERR_UNSUPPORTED, "w4_rmsnorm: %lld rows of %lld (a multiple of 8, at most %d)", (long long)rows,
                (long long)n, 8 * w4::kNormThreads * w4::kNormMaxVecs);
  if (rows == 0) return W4_OK;
  if (!x || !weight || !y || (delta != nullptr) != (sum != nullptr))
    return fail(W4_ERR_INVALID, "w4_rmsnorm: null pointer");
  if ((((uintptr_t)x | (uintptr_t)delta | (uintptr_t)weight | (uintptr_t)sum | (uintptr_t)y) % 16) != 0)
    return fail(W4_ERR_INVALID, "w4_rmsnorm: operands must be 16-byte aligned");
  const uint16_t *xp = static_cast<const uint16_t*>(x), *dp = static_cast<const uint16_t*>(delta),
                 *wp = static_cast<const uint16_t*>(weight);
  uint16_t *sp = static_cast<uint16_t*>(sum), *yp = static_cast<uint16_t*>(y);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == W4_DTYPE_BF16) {
    if (dp) launch_rmsnorm<W4_DTYPE_BF16, true>(xp, dp, wp, rows, (int)n, eps, sp, yp, st);
    else launch_rmsnorm<W4_DTYPE_BF16, false>(xp, dp, wp, rows, (int)n, eps, sp, yp, st);
  } else {
    if (dp) launch_rmsnorm<W4_DTYPE_FP16, true>(xp, dp, wp, rows, (int)n, eps, sp, yp, st);
    else launch_rmsnorm<W4_DTYPE_FP16, false>(xp, dp, wp, rows, (int)n, eps, sp, yp, st);
  }
  return check_launch("w4_rmsnorm");
}

extern "C" int w4_silu_mul(const void* gate, const void* up, int dtype, int64_t count, void* y, void* stream) {
  clear_error();
  if (dtype != W4_DTYPE_BF16 && dtype != W4_DTYPE_FP16)
    return fail(W4_ERR_INVALID, "w4_silu_mul: dtype must be bf16 or fp16 (got code %d)", dtype);
  if (count < 0 || count % 8 != 0 || count / 8 > kMaxGrid256 * 256)
    return fail(W4_ERR_UNSUPPORTED, "w4_silu_mul: %lld values (a multiple of 8, below 2^35)", (long long)count);
  if (count == 0) return W4_OK;
  if (!gate || !up || !y) return fail(W4_ERR_INVALID, "w4_silu_mul: null pointer");
  if ((((uintptr_t)gate | (uintptr_t)up | (uintptr_t)y) % 16) != 0)
    return fail(W4_ERR_INVALID, "w4_silu_mul: operands must be 16-byte aligned");
  const int64_t vecs = count / 8;
  const dim3 grid((unsigned)((vecs + 255) / 256)), block(256);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uint16_t *gp = static_cast<const uint16_t*>(gate), *up16 = static_cast<const uint16_t*>(up);
  uint16_t* yp = static_cast<uint16_t*>(y);
  if (dtype == W4_DTYPE_BF16)
    hipLaunchKernelGGL((w4::silu_mul_kernel<W4_DTYPE_BF16>), grid, block, 0, st, gp, up16, vecs, yp);
  else
    hipLaunchKernelGGL((w4::silu_mul_kernel<W4_DTYPE_FP16>), grid, block, 0, st, gp, up16, vecs, yp);
  return check_launch("w4_silu_mul");
}

namespace {

template <int DT>
void launch_norm_head(const w4::NormHeadArgs& a, hipStream_t st) {
  const int nc = (a.K + 511) / 512, rows = 4 * w4::head_rows(nc);
  // Eight workgroups per CU, each going through its rows; four above 2048 values,
  // where each pays more for the norm: up to about 32000 rows they are faster
  // (16000 x 4096 22.6 against 26.1 us, 12000 x 2560 12.5 against 13.2), above that
  // slower or equal (50257 x 2560 42.1 against 39.0, 128256 x 3072 117.7 against
  // 114.4).  At 2048 values the line is less clear (fp16, eight against four:
  // 16000 rows 14.5 and 12.7, 128256 rows 80.2 and 82.1).
  const int64_t wgs = ((int64_t)a.N + rows - 1) / rows;
  const int64_t most = nc <= 4 ? 2048 : 1024;
  const dim3 grid((unsigned)(wgs < most ? wgs : most)), block(256);
  switch (nc) {
    case 1: hipLaunchKernelGGL((w4::norm_head_kernel<DT, 1>), grid, block, 0, st, a); break;
    case 2: hipLaunchKernelGGL((w4::norm_head_kernel<DT, 2>), grid, block, 0, st, a); break;
    case 3: hipLaunchKernelGGL((w4::norm_head_kernel<DT, 3>), grid, block, 0, st, a); break;
    case 4: hipLaunchKernelGGL((w4::norm_head_kernel<DT, 4>), grid, block, 0, st, a); break;
    case 5: hipLaunchKernelGGL((w4::norm_head_kernel<DT, 5>), grid, block, 0, st, a); break;
    case 6: hipLaunchKernelGGL((w4::norm_head_kernel<DT, 6>), grid, block, 0, st, a); break;
    case 7: hipLaunchKernelGGL((w4::norm_head_kernel<DT, 7>), grid, block, 0, st, a); break;
    default: hipLaunchKernelGGL((w4::norm_head_kernel<DT, 8>), grid, block, 0, st, a); break;
  }
}

}  // namespace

extern "C" int w4_norm_head(const void* x, const void* delta, const void* norm_weight, float eps, const void* weight,
                            int dtype, int64_t N, int64_t K, void* y, void* stream) {
  clear_error();
  if (dtype != W4_DTYPE_BF16 && dtype != W4_DTYPE_FP16)
    return fail(W4_ERR_INVALID, "w4_norm_head: dtype must be bf16 or fp16 (got code %d)", dtype);
  if (K < 8 || K % 8 != 0 || K > 512 * w4::kHeadMaxChunks || N < 0 || N >= (1LL << 30))
    return fail(W4_ERR_UNSUPPORTED, "w4_norm_head: %lld x %lld (rows a multiple of 8 long, at most %d)", (long long)N,
                (long long)K, 512 * w4::kHeadMaxChunks);
  if (N == 0) return W4_OK;
  if (!x || !norm_weight || !weight || !y) return fail(W4_ERR_INVALID, "w4_norm_head: null pointer");
  if ((((uintptr_t)x | (uintptr_t)delta | (uintptr_t)norm_weight | (uintptr_t)weight) % 16) != 0 ||
      (uintptr_t)y % 2 != 0)
    return fail(W4_ERR_INVALID, "w4_norm_head: operands must be 16-byte aligned");
  const w4::NormHeadArgs a{static_cast<const uint16_t*>(x),           static_cast<const uint16_t*>(delta),
                           static_cast<const uint16_t*>(norm_weight), static_cast<const uint16_t*>(weight),
                           static_cast<uint16_t*>(y),                 (int)N, (int)K, eps};
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == W4_DTYPE_BF16) launch_norm_head<W4_DTYPE_BF16>(a, st);
  else launch_norm_head<W4_DTYPE_FP16>(a, st);
  return check_launch("w4_norm_head");
}
