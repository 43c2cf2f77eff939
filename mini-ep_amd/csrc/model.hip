// The transformer around the MoE block (gfx950): residual adds and RMSNorm,
// rotary embedding with the KV cache, causal attention, the projections of small
// batches, and q, k and v of larger ones.
//
// Replaces, in the reference's model (modeling.py):
//   RMSNorm                                      :55-63
//   rotate-half RoPE                             :66-80
//   GQA attention over the KV cache, fp32        :146-185
//   the scaled residual adds of Block.forward    :186-197
//   q/k/v/o projections and the LM head          :160-185, :249-254
// Activations are bf16 or fp32; scores, softmax and the attention sums are
// fp32, keys and values are kept in fp32.  Every rounding of the layer-by-layer
// computation is kept where a tensor of the model's dtype is defined: x after
// the norm, a projection's output, the scaled residual term, the residual sum.
#include "../../include/miniep_amd_model.h"
#include "common.h"
#include "ring_gemm.h"

#include <initializer_list>
#include <type_traits>

namespace mep {
namespace {

constexpr float kLog2e = 1.4426950408889634f;

template <int DT>
__device__ __forceinline__ void unpack_chunk(const u32x4& v, float* f) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  if constexpr (DT == MEP_DTYPE_BF16) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      f[2 * q] = bf16_to_f32(static_cast<uint16_t>(w[q] & 0xffffu));
      f[2 * q + 1] = bf16_to_f32(static_cast<uint16_t>(w[q] >> 16));
    }
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) f[q] = __uint_as_float(w[q]);
  }
}

template <int DT>
__device__ __forceinline__ u32x4 pack_chunk(const float* f) {
  u32x4 o;
  if constexpr (DT == MEP_DTYPE_BF16) {
    o.x = pack_bf16x2(f[0], f[1]);
    o.y = pack_bf16x2(f[2], f[3]);
    o.z = pack_bf16x2(f[4], f[5]);
    o.w = pack_bf16x2(f[6], f[7]);
  } else {
    o.x = __float_as_uint(f[0]);
    o.y = __float_as_uint(f[1]);
    o.z = __float_as_uint(f[2]);
    o.w = __float_as_uint(f[3]);
  }
  return o;
}

// f rounded to the storage type and back
template <int DT>
__device__ __forceinline__ float rounded(float f) {
  if constexpr (DT == MEP_DTYPE_BF16) return bf16_to_f32(f32_to_bf16(f));
  else return f;
}

// h + round(delta * mult), the residual step (no contraction: the product is
// a tensor of its own in the layer-by-layer computation)
template <int DT>
__device__ __forceinline__ float residual(float h, float delta, float mult) {
#pragma clang fp contract(off)
  const float step = rounded<DT>(delta * mult);
  return rounded<DT>(h + step);
}

// ============================================================================
// Residual add + RMSNorm: h_out = h + round(delta * mult) (delta NULL: h), x =
// weight * (h_out / sqrt(mean(h_out^2) + eps)).  One wave per row, the row in
// registers (NCH 16-byte chunks per lane), so h and delta are read once and
// h_out and x written once.  Bound by those bytes for many rows (2048 rows of
// 1024 in bf16: 16.8 MB in 5.6 us; 16384 rows of 1024, 2048 and 4096: 21, 43 and
// 102 us, 5.3 to 6.3 TB/s), by the launch for a few (8 rows: 2.4 to 3.8 us);
// as torch operations the same step was nine launches.  fp32 rows of 1028 to
// 2048 elements are the slow width: their instance (<F32, 8>) holds part of the
// row in accumulator registers, moves it back and forth and runs one wave per
// SIMD (16384 rows of 2048 in 163 us, 3.3 TB/s; of 1024 47 us and 5.7, of 4096
// 190 us and 5.6).
// ============================================================================
constexpr int kNormWaves = 4;

template <int DT, int NCH>
__global__ __launch_bounds__(kNormWaves * 64) void add_norm_kernel(const typename Elem<DT>::T* __restrict__ h,
                                                                   const typename Elem<DT>::T* __restrict__ delta,
                                                                   float mult,
                                                                   const typename Elem<DT>::T* __restrict__ weight,
                                                                   float eps, int64_t n, int hidden,
                                                                   typename Elem<DT>::T* __restrict__ h_out,
                                                                   typename Elem<DT>::T* __restrict__ x_out) {
  constexpr int EPC = 16 / Elem<DT>::kBytes;
  const int lane = lane_id();
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kNormWaves + (threadIdx.x >> 6);
  if (row >= n) return;
  const int64_t base = row * hidden;
  const int chunks = hidden / EPC;
  u32x4 hv[NCH], dv[NCH], wv[NCH];
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int q = c * 64 + lane;
    if (q >= chunks) continue;
    hv[c] = *reinterpret_cast<const u32x4*>(h + base + q * EPC);
    if (delta != nullptr) dv[c] = *reinterpret_cast<const u32x4*>(delta + base + q * EPC);
    wv[c] = *reinterpret_cast<const u32x4*>(weight + q * EPC);
  }
  float ss = 0.0f;
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int q = c * 64 + lane;
    if (q >= chunks) continue;
    float f[EPC];
    unpack_chunk<DT>(hv[c], f);
    if (delta != nullptr) {
      float d[EPC];
      unpack_chunk<DT>(dv[c], d);
#pragma unroll
      for (int i = 0; i < EPC; ++i) f[i] = residual<DT>(f[i], d[i], mult);
      hv[c] = pack_chunk<DT>(f);
      *reinterpret_cast<u32x4*>(h_out + base + q * EPC) = hv[c];
    }
#pragma unroll
    for (int i = 0; i < EPC; ++i) ss += f[i] * f[i];
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) ss += __shfl_xor(ss, d, 64);
  const float r = rsqrtf(ss / static_cast<float>(hidden) + eps);
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int q = c * 64 + lane;
    if (q >= chunks) continue;
    float f[EPC], w[EPC];
    unpack_chunk<DT>(hv[c], f);
    unpack_chunk<DT>(wv[c], w);
#pragma unroll
    for (int i = 0; i < EPC; ++i) f[i] = w[i] * (f[i] * r);
    *reinterpret_cast<u32x4*>(x_out + base + q * EPC) = pack_chunk<DT>(f);
  }
}

// ============================================================================
// Rotary embedding and attention, head size 64.
// ============================================================================
constexpr int kHead = 64;

struct AttnParams {
  const void* q;            // (batch * t, hq * 64) projections, before RoPE
  const void* k;            // (batch * t, hk * 64)
  const void* v;            // (batch * t, hk * 64)
  const float* cos;         // (max positions, 64), the two halves equal
  const float* sin;
  float* kc;                // (batch, hk, max_len, 64): keys after RoPE
  float* vc;                // (batch, hk, max_len, 64)
  void* out;                // (batch * t, hq * 64)
  int batch, t, hq, hk;
  int start;                // positions in the cache before this call; token i is position start + i
  int64_t max_len;
  float scale;
  int n_cu;                 // compute units of the device
};

// The rotated value of element c of a head whose projections start at `head`:
// element c pairs with c +- 32, the first half with the negative sign.
template <int DT>
__device__ __forceinline__ float rope(const typename Elem<DT>::T* head, int c, const float* cos, const float* sin) {
  const float x = Elem<DT>::to_f32(head[c]);
  const float y = Elem<DT>::to_f32(head[c < kHead / 2 ? c + kHead / 2 : c - kHead / 2]);
  return x * cos[c] + (c < kHead / 2 ? -y : y) * sin[c];
}

// Four elements of a head from an address that is a multiple of them.
template <int DT>
__device__ __forceinline__ f32x4 load4(const typename Elem<DT>::T* src) {
  if constexpr (DT == MEP_DTYPE_BF16) {
    const uint2 w = *reinterpret_cast<const uint2*>(src);
    return f32x4{bf16_to_f32(static_cast<uint16_t>(w.x & 0xffffu)), bf16_to_f32(static_cast<uint16_t>(w.x >> 16)),
                 bf16_to_f32(static_cast<uint16_t>(w.y & 0xffffu)), bf16_to_f32(static_cast<uint16_t>(w.y >> 16))};
  } else {
    return *reinterpret_cast<const f32x4*>(src);
  }
}

// Start of a running softmax's maximum: finite, so that keys whose scores are
// -inf (an overflow, or -inf in a key) weigh 0 also while no other score has been
// seen (-inf - -inf would be NaN for good).
constexpr float kLowest = -3.402823466e38f;

// Keys (rotated) and values of the call's tokens into the cache: one thread
// per 4 elements of a (token, kv head).
template <int DT>
__global__ __launch_bounds__(256) void kv_write_kernel(AttnParams p) {
  typedef typename Elem<DT>::T T;
  constexpr int C4 = kHead / 4;
  const int64_t q = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t total = static_cast<int64_t>(p.batch) * p.t * p.hk * C4;
  if (q >= total) return;
  const int c = static_cast<int>(q % C4) * 4;
  const int64_t th = q / C4;                              // token * hk + head
  const int head = static_cast<int>(th % p.hk);
  const int64_t tok = th / p.hk;
  const int b = static_cast<int>(tok / p.t), i = static_cast<int>(tok % p.t);
  const int64_t src = th * kHead, pos = p.start + i;
  const T* const k = static_cast<const T*>(p.k) + src;
  const T* const v = static_cast<const T*>(p.v) + src;
  const f32x4 cs = *reinterpret_cast<const f32x4*>(p.cos + pos * kHead + c);
  const f32x4 sn = *reinterpret_cast<const f32x4*>(p.sin + pos * kHead + c);
  const f32x4 x = load4<DT>(k + c), y = load4<DT>(k + (c < kHead / 2 ? c + kHead / 2 : c - kHead / 2));
  const f32x4 vr = load4<DT>(v + c);
  f32x4 kr;
#pragma unroll
  for (int j = 0; j < 4; ++j) kr[j] = x[j] * cs[j] + (c < kHead / 2 ? -y[j] : y[j]) * sn[j];
  const int64_t dst = ((static_cast<int64_t>(b) * p.hk + head) * p.max_len + pos) * kHead + c;
  *reinterpret_cast<f32x4*>(p.kc + dst) = kr;
  *reinterpret_cast<f32x4*>(p.vc + dst) = vr;
}

// Attention of more than one query per sequence, causal and aligned to the
// last key (query i of the call sees keys 0 .. start + i), fp32 on the matrix
// cores.  A workgroup is 64 queries of one head, 4 waves of 16; keys and
// values pass through LDS 64 at a time, the next block's loads in flight
// during a block's MFMAs.  With S^T = K Q^T a lane holds 4 keys of one query
// (C layout: rows 4 g + i, column r), which is the B operand that O^T =
// V^T P^T wants when MFMA i takes keys 4 g + i: the probabilities never leave
// their lane.  LDS rows are padded to 68 floats, which spreads both the
// 16-byte key reads and the 4-byte value reads over all banks.  Bound by the
// fp32 MFMAs (32 per wave, 16 keys and 16 queries) and the waits around the
// two barriers of a block.  8 sequences of 256 tokens, 16 heads: 20.3 us (512
// tokens: 56), and 4.6 us for the cache write, against 49 us for torch's fp32
// attention after a dozen launches of rotation, cache copy and head
// repetition.  (With the query tile as the fastest grid index the longest
// tiles all fall on two XCDs: 27 and 90 us.)
constexpr int kFlashQ = 64, kFlashK = 64, kFlashRow = kHead + 4;

template <int DT>
__global__ __launch_bounds__(256) void attention_kernel(AttnParams p) {
  typedef typename Elem<DT>::T T;
  __shared__ __attribute__((aligned(16))) float s_k[kFlashK * kFlashRow];
  __shared__ __attribute__((aligned(16))) float s_v[kFlashK * kFlashRow];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, g = lane >> 4;
  // workgroup -> (query tile, sequence, head of the group, kv head), kv head
  // fastest: the heads and tiles of a kv head share an XCD's L2, and the tiles
  // with the most keys come first on every XCD
  int id = static_cast<int>(blockIdx.x);
  const int kv = id % p.hk;
  id /= p.hk;
  const int G = p.hq / p.hk;
  const int head = kv * G + id % G;
  id /= G;
  // (tile, sequence) pairs of one round of the CUs; the second round, which
  // joins the first on the same CUs, is taken backwards: a CU gets a long and
  // a short tile
  const int per = p.n_cu / p.hq, pairs = (p.t + kFlashQ - 1) / kFlashQ * p.batch;
  if (id >= per && id < 2 * per) id = per + min(2 * per, pairs) - 1 - id;
  const int b = id % p.batch;
  const int q0 = ((p.t + kFlashQ - 1) / kFlashQ - 1 - id / p.batch) * kFlashQ;
  const int S = p.start + p.t;
  const float* const kc = p.kc + (static_cast<int64_t>(b) * p.hk + kv) * p.max_len * kHead;
  const float* const vc = p.vc + (static_cast<int64_t>(b) * p.hk + kv) * p.max_len * kHead;

  // this lane's query: elements 16 j + 4 g .. + 3, rotated and scaled (rows
  // past the end repeat the last query and are not stored)
  const int qi = q0 + wave * 16 + r;
  const int qrow = min(qi, p.t - 1);
  const int qpos = p.start + qrow;
  f32x4 q[4];
  {
    const T* const src = static_cast<const T*>(p.q) + (static_cast<int64_t>(b) * p.t + qrow) * p.hq * kHead + head * kHead;
    const float* const cs = p.cos + static_cast<int64_t>(qpos) * kHead;
    const float* const sn = p.sin + static_cast<int64_t>(qpos) * kHead;
    f32x4 x[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = load4<DT>(src + 16 * j + 4 * g);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4 c = *reinterpret_cast<const f32x4*>(cs + 16 * j + 4 * g);
      const f32x4 s = *reinterpret_cast<const f32x4*>(sn + 16 * j + 4 * g);
#pragma unroll
      for (int i = 0; i < 4; ++i) q[j][i] = x[j][i] * c[i] + (j < 2 ? -x[j + 2][i] : x[j - 2][i]) * s[i];
    }
  }
  const float sc = p.scale * kLog2e;

  // block of 64 keys: thread moves 16 floats of row tid / 4 (K and V)
  const int lrow = tid >> 2, lcol = (tid & 3) * 16;
  f32x4 kr[4], vr[4];
  auto load = [&](int k0) {
    const int64_t row = min(k0 + lrow, S - 1);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      kr[j] = *reinterpret_cast<const f32x4*>(kc + row * kHead + lcol + 4 * j);
      vr[j] = *reinterpret_cast<const f32x4*>(vc + row * kHead + lcol + 4 * j);
    }
  };
  const int k_end = min(S, p.start + q0 + kFlashQ);       // keys the workgroup's last query sees
  float m = kLowest, l = 0.0f;
  f32x4 o[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  load(0);
  for (int k0 = 0; k0 < k_end; k0 += kFlashK) {
    __syncthreads();                                      // the previous block's reads are done
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      *reinterpret_cast<f32x4*>(s_k + lrow * kFlashRow + lcol + 4 * j) = kr[j];
      *reinterpret_cast<f32x4*>(s_v + lrow * kFlashRow + lcol + 4 * j) = vr[j];
    }
    __syncthreads();
    if (k0 + kFlashK < k_end) load(k0 + kFlashK);
    f32x4 s[4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) s[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f32x4 kf[4];
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
        kf[kt] = *reinterpret_cast<const f32x4*>(s_k + (16 * kt + r) * kFlashRow + 16 * j + 4 * g);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
          s[kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[kt][i], q[j][i], s[kt], 0, 0, 0);
    }
    float mb = m;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[kt][i] = k0 + 16 * kt + 4 * g + i <= qpos ? s[kt][i] * sc : -__builtin_inff();
        mb = fmaxf(mb, s[kt][i]);
      }
    mb = fmaxf(mb, __shfl_xor(mb, 16, 64));
    mb = fmaxf(mb, __shfl_xor(mb, 32, 64));
    const float alpha = __builtin_amdgcn_exp2f(m - mb);
    m = mb;
    l *= alpha;
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int i = 0; i < 4; ++i) o[d][i] *= alpha;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[kt][i] = __builtin_amdgcn_exp2f(s[kt][i] - m);
        l += s[kt][i];
      }
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int d = 0; d < 4; ++d)
          o[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(s_v[(16 * kt + 4 * g + i) * kFlashRow + 16 * d + r], s[kt][i], o[d],
                                                     0, 0, 0);
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (qi >= p.t) return;
  T* const dst = static_cast<T*>(p.out) + (static_cast<int64_t>(b) * p.t + qi) * p.hq * kHead + head * kHead;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const float v[4] = {o[d][0] / l, o[d][1] / l, o[d][2] / l, o[d][3] / l};
    if constexpr (DT == MEP_DTYPE_BF16)
      *reinterpret_cast<uint2*>(dst + 16 * d + 4 * g) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
    else
      *reinterpret_cast<f32x4*>(dst + 16 * d + 4 * g) = f32x4{v[0], v[1], v[2], v[3]};
  }
}

// Attention of one new token per sequence (decode).  A workgroup of 16 waves
// is one (sequence, kv head) with its G query heads, so keys and values are
// read once for the group.  It rotates the new key, writes it and the value
// to the cache, and walks the cached positions kDecKeys at a time: scores to
// LDS (16 lanes per key, 16 bytes each, so a wave reads four whole keys per
// instruction), the chunk's maximum and sum, then the values with the same
// lane layout.  The sums of the 64 key groups meet in LDS in a fixed order.
// Two batches of loads are kept in flight, from the first keys (before the
// rotation) through the softmax's barrier to the last values.  Bound by one
// CU's loads: 8 sequences of 513 positions, 8 kv heads (16.8 MB of cache), two
// query heads each: 11.0 us (14.1 with one batch at a time and the sums of 16
// lanes through LDS), against 46 us for torch's fp32 attention alone.  With one
// and four query heads each (back to back, where two take 9.2): 7.7 and 12.0;
// one sequence of 4000 positions 25, 30 and 47.
constexpr int kDecWaves = 16, kDecKeys = 2048;

// The sum over a row of 16 lanes, in every lane: the tree of xor 1, 2, 4, 8 (a
// mirrored lane holds what the xor partner holds once the steps before agree).
__device__ __forceinline__ float sum16(float v) {
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));    // quad_perm 1 0 3 2
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, true));    // quad_perm 2 3 0 1
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xF, 0xF, true));   // row_half_mirror
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x140, 0xF, 0xF, true));   // row_mirror
  return v;
}

template <int DT, int G>
__global__ __launch_bounds__(kDecWaves * 64) void attention_decode_kernel(AttnParams p) {
  typedef typename Elem<DT>::T T;
  __shared__ __attribute__((aligned(16))) float s_q[G][kHead];
  __shared__ __attribute__((aligned(16))) float s_new[2][kHead];     // the new token's key and value
  __shared__ float s_p[G][kDecKeys];
  __shared__ float s_red[kDecWaves][G];
  __shared__ __attribute__((aligned(16))) float s_o[kDecWaves][G][kHead];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c = lane & 15, g = lane >> 4;
  const int kv = static_cast<int>(blockIdx.x) % p.hk, b = static_cast<int>(blockIdx.x) / p.hk;
  const int pos = p.start, S = pos + 1;
  float* const kc = p.kc + (static_cast<int64_t>(b) * p.hk + kv) * p.max_len * kHead;
  float* const vc = p.vc + (static_cast<int64_t>(b) * p.hk + kv) * p.max_len * kHead;
  // a batch: kDecUnroll cached positions per lane group, 16 bytes of each per
  // lane (past the end, and in place of the new token: the last one again)
  constexpr int kDecUnroll = G == 4 ? 2 : 4;               // G = 4 has no registers for more
  constexpr int kStep = kDecWaves * 4, kBatch = kStep * kDecUnroll;
  f32x4 ra[kDecUnroll], rb[kDecUnroll];
  auto fetch = [&](f32x4 (&r)[kDecUnroll], const float* cache, int c0, int s0) {   // positions c0 + s0 ..
    const char* const base = reinterpret_cast<const char*>(cache + static_cast<int64_t>(c0) * kHead);
    const int last = max(pos - 1 - c0, 0);
#pragma unroll
    for (int u = 0; u < kDecUnroll; ++u) {
      const int s = min(s0 + u * kStep + wave * 4 + g, last);
      r[u] = *reinterpret_cast<const f32x4*>(base + static_cast<uint32_t>(s * (kHead * 4) + 16 * c));
    }
  };
  fetch(ra, kc, 0, 0);
  {
    const float* const cs = p.cos + static_cast<int64_t>(pos) * kHead;
    const float* const sn = p.sin + static_cast<int64_t>(pos) * kHead;
    if (tid < G * kHead) {
      const T* const src = static_cast<const T*>(p.q) + (static_cast<int64_t>(b) * p.hq + kv * G + tid / kHead) * kHead;
      s_q[tid / kHead][tid % kHead] = rope<DT>(src, tid % kHead, cs, sn) * (p.scale * kLog2e);
    } else if (tid < (G + 1) * kHead) {
      const int e = tid - G * kHead;
      const float k = rope<DT>(static_cast<const T*>(p.k) + (static_cast<int64_t>(b) * p.hk + kv) * kHead, e, cs, sn);
      s_new[0][e] = k;
      kc[static_cast<int64_t>(pos) * kHead + e] = k;
    } else if (tid < (G + 2) * kHead) {
      const int e = tid - (G + 1) * kHead;
      const float v = Elem<DT>::to_f32(static_cast<const T*>(p.v)[(static_cast<int64_t>(b) * p.hk + kv) * kHead + e]);
      s_new[1][e] = v;
      vc[static_cast<int64_t>(pos) * kHead + e] = v;
    }
  }
  lds_barrier();
  f32x4 q[G], fresh[2];                                    // the queries; the new token's key and value
#pragma unroll
  for (int h = 0; h < G; ++h) q[h] = *reinterpret_cast<const f32x4*>(&s_q[h][4 * c]);
#pragma unroll
  for (int i = 0; i < 2; ++i) fresh[i] = *reinterpret_cast<const f32x4*>(&s_new[i][4 * c]);
  float m[G], l[G], mx[G];
  f32x4 o[G];
#pragma unroll
  for (int h = 0; h < G; ++h) {
    m[h] = mx[h] = kLowest;
    l[h] = 0.0f;
    o[h] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  for (int c0 = 0; c0 < S; c0 += kDecKeys) {
    const int n = min(kDecKeys, S - c0);
    const int nb = (n + kBatch - 1) / kBatch, pairs = (nb + 1) / 2;
    if (c0 != 0) fetch(ra, kc, c0, 0);
    auto scores = [&](const f32x4 (&kr)[kDecUnroll], int bt) {
      if (bt >= nb) return;
#pragma unroll
      for (int u = 0; u < kDecUnroll; ++u) {
        const int s = bt * kBatch + u * kStep + wave * 4 + g;
        const f32x4 k = c0 + s == pos ? fresh[0] : kr[u];
#pragma unroll
        for (int h = 0; h < G; ++h) {
          const float d = sum16(k.x * q[h].x + k.y * q[h].y + k.z * q[h].z + k.w * q[h].w);
          if (s < n) {
            mx[h] = fmaxf(mx[h], d);
            if (c == 0) s_p[h][s] = d;
          }
        }
      }
    };
    for (int i = 0; i < pairs; ++i) {
      fetch(rb, kc, c0, (2 * i + 1) * kBatch);
      scores(ra, 2 * i);
      // after the last keys, the first values
      fetch(ra, i + 1 < pairs ? kc : vc, c0, i + 1 < pairs ? (2 * i + 2) * kBatch : 0);
      scores(rb, 2 * i + 1);
    }
#pragma unroll
    for (int h = 0; h < G; ++h) {
      float v = mx[h];
      v = fmaxf(v, __shfl_xor(v, 16, 64));
      v = fmaxf(v, __shfl_xor(v, 32, 64));
      if (lane == 0) s_red[wave][h] = v;
    }
    lds_barrier();                                         // the values' loads stay in flight
#pragma unroll
    for (int h = 0; h < G; ++h) {
      float v = s_red[0][h];
#pragma unroll
      for (int w = 1; w < kDecWaves; ++w) v = fmaxf(v, s_red[w][h]);
      const float alpha = __builtin_amdgcn_exp2f(m[h] - v);   // (in the first chunk l and o are 0)
      m[h] = mx[h] = v;
      l[h] *= alpha;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[h][i] *= alpha;
    }
    auto values = [&](const f32x4 (&vr)[kDecUnroll], int bt) {
      if (bt >= nb) return;
#pragma unroll
      for (int u = 0; u < kDecUnroll; ++u) {
        const int s = bt * kBatch + u * kStep + wave * 4 + g;
        if (s >= n) continue;
        const f32x4 v = c0 + s == pos ? fresh[1] : vr[u];
#pragma unroll
        for (int h = 0; h < G; ++h) {
          const float e = __builtin_amdgcn_exp2f(s_p[h][s] - m[h]);
          l[h] += e;
#pragma unroll
          for (int i = 0; i < 4; ++i) o[h][i] += e * v[i];
        }
      }
    };
    for (int i = 0; i < pairs; ++i) {
      fetch(rb, vc, c0, (2 * i + 1) * kBatch);
      values(ra, 2 * i);
      if (i + 1 == pairs) break;
      fetch(ra, vc, c0, (2 * i + 2) * kBatch);
      values(rb, 2 * i + 1);
    }
    values(rb, 2 * pairs - 1);
    lds_barrier();                                         // scores and maxima are read before the next chunk's
  }
#pragma unroll
  for (int h = 0; h < G; ++h) {
#pragma unroll
    for (int x = 16; x < 64; x <<= 1) {
      l[h] += __shfl_xor(l[h], x, 64);
#pragma unroll
      for (int i = 0; i < 4; ++i) o[h][i] += __shfl_xor(o[h][i], x, 64);
    }
    if (g == 0) *reinterpret_cast<f32x4*>(&s_o[wave][h][4 * c]) = o[h];
    if (lane == 0) s_red[wave][h] = l[h];
  }
  __syncthreads();
  if (tid < G * kHead) {
    const int h = tid / kHead, e = tid % kHead;
    float sum = 0.0f, den = 0.0f;
#pragma unroll
    for (int w = 0; w < kDecWaves; ++w) {
      sum += s_o[w][h][e];
      den += s_red[w][h];
    }
    static_cast<T*>(p.out)[(static_cast<int64_t>(b) * p.hq + kv * G + h) * kHead + e] = Elem<DT>::from_f32(sum / den);
  }
}

template <int DT>
hipError_t launch_attention(const AttnParams& p, hipStream_t stream) {
  if (p.t == 1) {
    const dim3 grid(static_cast<unsigned>(p.batch * p.hk));
    switch (p.hq / p.hk) {
      case 1: attention_decode_kernel<DT, 1><<<grid, kDecWaves * 64, 0, stream>>>(p); break;
      case 2: attention_decode_kernel<DT, 2><<<grid, kDecWaves * 64, 0, stream>>>(p); break;
      default: attention_decode_kernel<DT, 4><<<grid, kDecWaves * 64, 0, stream>>>(p); break;
    }
    return hipGetLastError();
  }
  const int64_t chunks = static_cast<int64_t>(p.batch) * p.t * p.hk * (kHead / 4);
  kv_write_kernel<DT><<<dim3(static_cast<unsigned>((chunks + 255) / 256)), 256, 0, stream>>>(p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const dim3 grid(static_cast<unsigned>((p.t + kFlashQ - 1) / kFlashQ) * static_cast<unsigned>(p.batch * p.hq));
  AttnParams pf = p;
  pf.n_cu = device_cu_count();
  attention_kernel<DT><<<grid, 256, 0, stream>>>(pf);
  return hipGetLastError();
}

// ============================================================================
// Projections of a small batch (at most 32 rows, bf16): out = x W^T for up to
// three weight matrices in one launch.
//
// There the time goes to reading W once, so the work is split for loads in
// flight, not for reuse: a workgroup is 16 output columns at a time, its 8
// waves an eighth of K each (KS steps of 32), every weight load of a tile
// issued at once, straight into the MFMA's registers, and the next tile's
// before the current one's MFMAs.  x (all rows) stays in registers across the
// workgroup's tiles.  The 8 partial tiles meet in LDS and are summed in wave
// order.
//
// NORM: x = rms_norm(h + round(delta * mult)) is computed by every workgroup
// from h in those registers (16 KB of reads that hit the L2, against a launch
// and a round trip of x); workgroup 0 stores the residual sum.
//
// Measured with 8 rows, hidden 1024: norm + q, k and v (4.2 MB) 6.7 us, against
// 3.8 us for the norm and three library GEMMs of 7.6 us; the output projection
// with its residual (2.1 MB) 4.2 us against 7.6 us; the head (49155 columns,
// 101 MB) 22.9 us, against 46 us for a library GEMM over an fp32 copy of it.
// ============================================================================
constexpr int kRowsMax = 32, kLinWaves = 8, kLinCols = 16, kLinPad = 20;

enum LinearOut { kLinPlain, kLinResidual, kLinScaled };   // bf16; bf16 onto a residual; fp32 / scale

struct LinearParams {
  const uint16_t* x;          // (n, K); NORM: h
  const uint16_t* delta;      // NORM: (n, K) or NULL
  const uint16_t* norm_w;     // NORM: (K,)
  uint16_t* h_out;            // NORM: (n, K) = h + round(delta * mult), or NULL
  float mult, eps;
  const uint16_t* w[3];       // (cols[i], K)
  void* out[3];               // (n, cols[i])
  int cols[3];
  int tiles[3];               // 16-column tiles of matrices 0 .. i together
  const uint16_t* res;        // kLinResidual: (n, cols[0])
  float out_mult;             // kLinResidual: residual multiplier; kLinScaled: divisor
  int n;
};

template <int KS, int MFC, bool NORM, int OUT>
__global__ __launch_bounds__(kLinWaves * 64) void linear_rows_kernel(LinearParams p) {
  constexpr int K = kLinWaves * KS * 32;
  __shared__ __attribute__((aligned(16))) float s_acc[2][kLinWaves][MFC][16 * kLinPad];
  __shared__ float s_ss[kLinWaves][16 * MFC];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lr = lane & 15, lg = lane >> 4;
  const int k0 = wave * KS * 32 + 8 * lg;                  // this lane's first K element of a step
  const int total = p.tiles[2];

  int mat = 0, col0 = 0;
  auto locate = [&](int tile, int& m, int& c) {
    m = tile < p.tiles[0] ? 0 : (tile < p.tiles[1] ? 1 : 2);
    c = (tile - (m == 0 ? 0 : p.tiles[m - 1])) * kLinCols;
  };
  u32x4 wq[KS], wn[KS];
  auto load_w = [&](int tile, u32x4 (&w)[KS]) {
    int m, c;
    locate(tile, m, c);
    const uint16_t* const row = p.w[m] + static_cast<int64_t>(min(c + lr, p.cols[m] - 1)) * K + k0;
#pragma unroll
    for (int s = 0; s < KS; ++s) w[s] = *reinterpret_cast<const u32x4*>(row + 32 * s);
  };
  int tile = blockIdx.x;                                   // the grid has at most `total` workgroups
  load_w(tile, wq);

  u32x4 xa[MFC][KS];
#pragma unroll
  for (int f = 0; f < MFC; ++f) {
    const int64_t row = static_cast<int64_t>(min(16 * f + lr, p.n - 1)) * K + k0;
#pragma unroll
    for (int s = 0; s < KS; ++s) xa[f][s] = *reinterpret_cast<const u32x4*>(p.x + row + 32 * s);
  }
  if constexpr (NORM) {
    float ss[MFC];
#pragma unroll
    for (int f = 0; f < MFC; ++f) {
      ss[f] = 0.0f;
      const int64_t row = static_cast<int64_t>(min(16 * f + lr, p.n - 1)) * K + k0;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        float v[8];
        unpack_chunk<MEP_DTYPE_BF16>(xa[f][s], v);
        if (p.delta != nullptr) {
          float d[8];
          unpack_chunk<MEP_DTYPE_BF16>(*reinterpret_cast<const u32x4*>(p.delta + row + 32 * s), d);
#pragma unroll
          for (int i = 0; i < 8; ++i) v[i] = residual<MEP_DTYPE_BF16>(v[i], d[i], p.mult);
          xa[f][s] = pack_chunk<MEP_DTYPE_BF16>(v);
          if (blockIdx.x == 0 && p.h_out != nullptr && 16 * f + lr < p.n)
            *reinterpret_cast<u32x4*>(p.h_out + row + 32 * s) = xa[f][s];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) ss[f] += v[i] * v[i];
      }
      ss[f] += __shfl_xor(ss[f], 16, 64);
      ss[f] += __shfl_xor(ss[f], 32, 64);
      if (lg == 0) s_ss[wave][16 * f + lr] = ss[f];
    }
    __syncthreads();
#pragma unroll
    for (int f = 0; f < MFC; ++f) {
      float sum = 0.0f;
#pragma unroll
      for (int w = 0; w < kLinWaves; ++w) sum += s_ss[w][16 * f + lr];
      const float r = rsqrtf(sum / static_cast<float>(K) + p.eps);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        float v[8], w[8];
        unpack_chunk<MEP_DTYPE_BF16>(xa[f][s], v);
        unpack_chunk<MEP_DTYPE_BF16>(*reinterpret_cast<const u32x4*>(p.norm_w + k0 + 32 * s), w);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = w[i] * (v[i] * r);
        xa[f][s] = pack_chunk<MEP_DTYPE_BF16>(v);
      }
    }
  }

  for (int buf = 0; tile < total; tile += gridDim.x, buf ^= 1) {
    const bool more = tile + static_cast<int>(gridDim.x) < total;
    if (more) load_w(tile + gridDim.x, wn);
    // weight fragment first: lane (lr, lg) gets columns 4 lg .. + 3 of row lr
#pragma unroll
    for (int f = 0; f < MFC; ++f) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wq[s]),
                                                      __builtin_bit_cast(bf16x8, xa[f][s]), acc, 0, 0, 0);
      *reinterpret_cast<f32x4*>(&s_acc[buf][wave][f][lr * kLinPad + 4 * lg]) = acc;
    }
    // one barrier a tile: the other buffer's readers are past it by the next one
    __syncthreads();
    const int row = tid >> 4, c = tid & 15;
    locate(tile, mat, col0);
    const int col = col0 + c, N = p.cols[mat];
    if (row < p.n && row < 16 * MFC && col < N) {
      float sum = 0.0f;
#pragma unroll
      for (int w = 0; w < kLinWaves; ++w) sum += s_acc[buf][w][row >> 4][(row & 15) * kLinPad + c];
      const int64_t at = static_cast<int64_t>(row) * N + col;
      if constexpr (OUT == kLinScaled) {
        static_cast<float*>(p.out[mat])[at] = sum / p.out_mult;
      } else if constexpr (OUT == kLinResidual) {
        static_cast<uint16_t*>(p.out[mat])[at] = f32_to_bf16(
            residual<MEP_DTYPE_BF16>(bf16_to_f32(p.res[at]), rounded<MEP_DTYPE_BF16>(sum), p.out_mult));
      } else {
        static_cast<uint16_t*>(p.out[mat])[at] = f32_to_bf16(sum);
      }
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) wq[s] = wn[s];
  }
}

// (at 4096 the registers of a wave no longer hold its share of x and of two
// weight tiles)
bool linear_rows_k(int k) { return k == 1024 || k == 2048; }

template <bool NORM, int OUT>
hipError_t launch_linear_rows(LinearParams p, int k, hipStream_t stream) {
  int tiles = 0;
  for (int i = 0; i < 3; ++i) p.tiles[i] = tiles += (p.cols[i] + kLinCols - 1) / kLinCols;
  // two workgroups per CU cover the loads in flight of the largest matrices
  const int cap = 2 * device_cu_count();
  const dim3 grid(static_cast<unsigned>(tiles < cap ? tiles : cap));
  auto go = [&](auto ks) {
    constexpr int KS = decltype(ks)::value;
    if (p.n <= 16) linear_rows_kernel<KS, 1, NORM, OUT><<<grid, kLinWaves * 64, 0, stream>>>(p);
    else linear_rows_kernel<KS, 2, NORM, OUT><<<grid, kLinWaves * 64, 0, stream>>>(p);
  };
  if (k == 1024) go(std::integral_constant<int, 4>());
  else go(std::integral_constant<int, 8>());
  return hipGetLastError();
}

// ============================================================================
// Projections of more rows (bf16): out = x W^T for up to three weight matrices
// in one launch.
//
// Tiles of 16 MFC rows by 128 columns, the experts' mid-size K loop
// (ring_loop): q, k and v of one prompt batch fill the chip together where
// three launches of larger tiles leave it half empty, each paying its own ramp.
// Tiles are listed row chunk by row chunk and split into 8 contiguous ranges,
// one per XCD: a chunk's rows are read into one L2.
// us with q, k and v of 1024 + 512 + 512 columns, hidden 1024, three library
// GEMMs -> this: 64 rows 24.7 -> 8.9, 512: 25 -> 9.9, 1024: 26 -> 11.1, 2048:
// 28.5 -> 14.8, 4096: 33.2 -> 21.7, 8192: 45 -> 39; hidden 2048, 2048 + 512 +
// 512 columns: 1024 rows 34 -> 22, 2048: 42 -> 34, 3000: 51 -> 53, 4096: 60 ->
// 55.  (A single matrix is no faster than the library's: 2048 rows of 1024,
// 11.2.)  Bound by the LDS (756 cycles of reads and writes for 512 of MFMAs per
// block of K) and, with one workgroup on a CU, by the waits around a block's
// barrier; four blocks of loads ahead instead of two change nothing.
// ============================================================================
struct LinearTileParams {
  const uint16_t* x;          // (n, K)
  const uint16_t* w[3];       // (cols[i], K)
  uint16_t* out[3];           // (n, cols[i])
  int cols[3];                // multiples of 128
  int tiles[3];               // column tiles of matrices 0 .. i together
  int n, K;
};

template <int MFC>
__global__ __launch_bounds__(ring::NT, 2) void linear_tile_kernel(LinearTileParams p) {
  constexpr int DT = MEP_DTYPE_BF16, CH = 16 * MFC, AP = MFC / 2, WP = ring::WP;
  __shared__ __attribute__((aligned(16))) unsigned char s_ring[ring::lds_bytes(MFC)];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1, lr = lane & 15, lg = lane >> 4;
  const int units = (p.n + CH - 1) / CH * p.tiles[2];
  const int xcd = blockIdx.x & 7;
  const int u = static_cast<int>(static_cast<int64_t>(units) * xcd / 8) + static_cast<int>(blockIdx.x >> 3);
  if (u >= static_cast<int>(static_cast<int64_t>(units) * (xcd + 1) / 8)) return;
  const int row0 = u / p.tiles[2] * CH, tile = u % p.tiles[2];
  const int mat = tile < p.tiles[0] ? 0 : (tile < p.tiles[1] ? 1 : 2);
  const int col0 = (tile - (mat == 0 ? 0 : p.tiles[mat - 1])) * 128;
  const int row_bytes = p.K * 2, NB = row_bytes / 128;
  const unsigned char* const W = reinterpret_cast<const unsigned char*>(p.w[mat]);
  const unsigned char* const A = reinterpret_cast<const unsigned char*>(p.x);
  const ring::Copy cp;
  uint32_t w_off[WP], a_off[AP];                           // x and a matrix are below 4 GiB (the host checks)
  // weight fragment 4 wn + j of the tile: row m of the pair's half j & 1 is
  // column 8 (m / 4) + 4 (j & 1) + m % 4 of 32, so a lane's results across a
  // pair are 8 consecutive columns
#pragma unroll
  for (int i = 0; i < WP; ++i) {
    const int fr = 2 * i + cp.half, j = fr & 3;
    const int row = col0 + 64 * (fr >> 2) + 32 * (j >> 1) + 8 * (cp.row16 >> 2) + 4 * (j & 1) + (cp.row16 & 3);
    w_off[i] = static_cast<uint32_t>(row) * static_cast<uint32_t>(row_bytes) + cp.chunk * 16;
  }
#pragma unroll
  for (int i = 0; i < AP; ++i)
    a_off[i] = static_cast<uint32_t>(min(row0 + 32 * i + 16 * cp.half + cp.row16, p.n - 1)) *
                   static_cast<uint32_t>(row_bytes) + cp.chunk * 16;
  u32x4 wr[ring::AHEAD][WP], ar[ring::AHEAD][AP];
  auto line = [&](int b) { return ring::block_at(b, 0, NB) * 128; };
  auto load_w = [&](int b, int i) { return *reinterpret_cast<const u32x4*>(W + line(b) + w_off[i]); };
  auto load_a = [&](int b, int i) { return *reinterpret_cast<const u32x4*>(A + line(b) + a_off[i]); };
#pragma unroll
  for (int b = 0; b < ring::AHEAD; ++b) {
#pragma unroll
    for (int i = 0; i < WP; ++i) wr[b][i] = load_w(b, i);
#pragma unroll
    for (int i = 0; i < AP; ++i) ar[b][i] = load_a(b, i);
  }
  f32x4 acc[MFC / 2][4];
  ring_loop<DT, MFC>(NB, s_ring, wr, ar, load_w, load_a, acc);
  const int N = p.cols[mat];
#pragma unroll
  for (int i = 0; i < MFC / 2; ++i) {
    const int r = row0 + (wm * (MFC / 2) + i) * 16 + lr;
    if (r >= p.n) continue;
    const int64_t at = static_cast<int64_t>(r) * N + col0 + 64 * wn + 8 * lg;
#pragma unroll
    for (int jp = 0; jp < 2; ++jp) {
      float v[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) v[c] = acc[i][2 * jp + (c >> 2)][c & 3];
      *reinterpret_cast<u32x4*>(p.out[mat] + at + 32 * jp) = pack_chunk<DT>(v);
    }
  }
}

// Tiles of 128 rows read x and W through LDS less often, tiles of 64 rows are
// taken while they fit the chip at once (us, 64 against 128 rows a tile, by
// tiles of 64 per CU; hidden 1024, q + k + v of 2048 columns: 1.0 10.3 against
// 13.0, 1.12 14.5 against 13.2, 2.0 15.6 against 14.9, 4.0 27.5 against 23.3;
// hidden 2048, 3072 columns: 0.75 18.0 against 21.4, 1.12 25.5 against 22.1; hidden
// 512, 1024 columns: 1.0 7.0 against 8.8, 1.47 9.7 against 9.1).
hipError_t launch_linear_tile(const LinearTileParams& p, hipStream_t stream) {
  auto go = [&](auto mfc) {
    constexpr int MFC = decltype(mfc)::value;
    const int64_t units = static_cast<int64_t>((p.n + 16 * MFC - 1) / (16 * MFC)) * p.tiles[2];
    linear_tile_kernel<MFC><<<dim3(static_cast<unsigned>((units + 7) / 8 * 8)), ring::NT, 0, stream>>>(p);
  };
  if (static_cast<int64_t>((p.n + 63) / 64) * p.tiles[2] <= device_cu_count()) go(std::integral_constant<int, 4>());
  else go(std::integral_constant<int, 8>());
  return hipGetLastError();
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

}  // namespace
}  // namespace mep

using namespace mep;

namespace mep {
namespace {

hipError_t launch_add_norm(const void* h, const void* delta, float mult, const void* weight, float eps, int64_t n_rows,
                           int hidden, int dtype, void* h_out, void* x_out, hipStream_t s) {
  const int epc = 16 / dtype_bytes(dtype);
  const dim3 grid(static_cast<unsigned>((n_rows + kNormWaves - 1) / kNormWaves));
  const int nch = (hidden / epc + 63) / 64;
  auto go = [&](auto dt, auto c) {
    constexpr int DT = decltype(dt)::value, NCH = decltype(c)::value;
    typedef typename Elem<DT>::T T;
    add_norm_kernel<DT, NCH><<<grid, kNormWaves * 64, 0, s>>>(static_cast<const T*>(h), static_cast<const T*>(delta), mult,
                                                              static_cast<const T*>(weight), eps, n_rows, hidden,
                                                              static_cast<T*>(h_out), static_cast<T*>(x_out));
  };
  auto by_width = [&](auto dt) {
    if (nch <= 2) go(dt, std::integral_constant<int, 2>());
    else if (nch <= 4) go(dt, std::integral_constant<int, 4>());
    else if (nch <= 8) go(dt, std::integral_constant<int, 8>());
    else go(dt, std::integral_constant<int, 16>());
  };
  if (dtype == MEP_DTYPE_BF16) by_width(std::integral_constant<int, MEP_DTYPE_BF16>());
  else by_width(std::integral_constant<int, MEP_DTYPE_F32>());
  return hipGetLastError();
}

// What attention supports, for the entry points that run it.
int check_attention(const char* fn, int64_t n_positions, int batch, int t, int n_heads, int n_kv_heads, int head_dim,
                    int64_t start, int64_t max_len) {
  MEP_REQUIRE(batch >= 0 && t >= 0 && start >= 0 && n_heads >= 1 && n_kv_heads >= 1, MEP_ERR_INVALID_ARG,
              "%s: bad sizes", fn);
  MEP_REQUIRE(head_dim == kHead, MEP_ERR_UNSUPPORTED, "%s: head size %d, supported: 64", fn, head_dim);
  const int group = n_heads / n_kv_heads;
  MEP_REQUIRE(n_heads % n_kv_heads == 0 && (group == 1 || group == 2 || group == 4), MEP_ERR_UNSUPPORTED,
              "%s: %d query heads over %d kv heads (1, 2 or 4 each)", fn, n_heads, n_kv_heads);
  MEP_REQUIRE(start + t <= max_len && start + t <= n_positions, MEP_ERR_INVALID_ARG,
              "%s: positions up to %lld, the cache holds %lld and the rotary table %lld", fn,
              static_cast<long long>(start + t), static_cast<long long>(max_len), static_cast<long long>(n_positions));
  MEP_REQUIRE(max_len < (int64_t(1) << 31) && static_cast<int64_t>(batch) * n_heads <= 65535 &&
                  static_cast<int64_t>(batch) * t * n_heads * (kHead / 4) < (int64_t(1) << 37),
              MEP_ERR_UNSUPPORTED, "%s: batch or length too large", fn);
  return MEP_OK;
}

}  // namespace
}  // namespace mep

extern "C" int mep_add_norm(const void* h, const void* delta, float mult, const void* weight, float eps,
                            int64_t n_rows, int32_t hidden, int32_t dtype, void* h_out, void* x_out, void* stream) {
  clear_error();
  const char* fn = "mep_add_norm";
  MEP_REQUIRE(dtype == MEP_DTYPE_F32 || dtype == MEP_DTYPE_BF16, MEP_ERR_INVALID_ARG, "%s: unknown dtype %d", fn, dtype);
  MEP_REQUIRE(n_rows >= 0 && n_rows < (int64_t(1) << 31), MEP_ERR_INVALID_ARG, "%s: bad n_rows", fn);
  const int epc = 16 / dtype_bytes(dtype);
  MEP_REQUIRE(hidden > 0 && hidden % epc == 0 && hidden <= 4096, MEP_ERR_UNSUPPORTED,
              "%s: hidden %d must be a positive multiple of %d, at most 4096", fn, hidden, epc);
  if (n_rows == 0) return MEP_OK;
  MEP_REQUIRE(h && weight && x_out && (delta == nullptr || h_out != nullptr), MEP_ERR_INVALID_ARG, "%s: null pointer", fn);
  MEP_REQUIRE(aligned16(h) && aligned16(delta) && aligned16(weight) && aligned16(h_out) && aligned16(x_out),
              MEP_ERR_INVALID_ARG, "%s: buffers must be 16-byte aligned", fn);
  const hipError_t e = launch_add_norm(h, delta, mult, weight, eps, n_rows, hidden, dtype, h_out, x_out,
                                       static_cast<hipStream_t>(stream));
  MEP_REQUIRE(e == hipSuccess, MEP_ERR_HIP, "%s: launch failed: %s", fn, hipGetErrorString(e));
  return MEP_OK;
}

extern "C" int mep_attention(const void* q, const void* k, const void* v, const float* cos, const float* sin,
                             int64_t n_positions, int32_t batch, int32_t t, int32_t n_heads, int32_t n_kv_heads,
                             int32_t head_dim, int64_t start, int64_t max_len, float scale, int32_t dtype,
                             float* k_cache, float* v_cache, void* out, void* stream) {
  clear_error();
  const char* fn = "mep_attention";
  MEP_REQUIRE(dtype == MEP_DTYPE_F32 || dtype == MEP_DTYPE_BF16, MEP_ERR_INVALID_ARG, "%s: unknown dtype %d", fn, dtype);
  const int rc = check_attention(fn, n_positions, batch, t, n_heads, n_kv_heads, head_dim, start, max_len);
  if (rc != MEP_OK) return rc;
  if (batch == 0 || t == 0) return MEP_OK;
  MEP_REQUIRE(q && k && v && cos && sin && k_cache && v_cache && out, MEP_ERR_INVALID_ARG, "%s: null pointer", fn);
  for (const void* ptr : {q, k, v, static_cast<const void*>(cos), static_cast<const void*>(sin),
                          static_cast<const void*>(k_cache), static_cast<const void*>(v_cache),
                          static_cast<const void*>(out)})
    MEP_REQUIRE(aligned16(ptr), MEP_ERR_INVALID_ARG, "%s: buffers must be 16-byte aligned", fn);
  AttnParams p;
  p.q = q; p.k = k; p.v = v; p.cos = cos; p.sin = sin; p.kc = k_cache; p.vc = v_cache; p.out = out;
  p.batch = batch; p.t = t; p.hq = n_heads; p.hk = n_kv_heads;
  p.start = static_cast<int>(start); p.max_len = max_len; p.scale = scale;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const hipError_t e = dtype == MEP_DTYPE_BF16 ? launch_attention<MEP_DTYPE_BF16>(p, s) : launch_attention<MEP_DTYPE_F32>(p, s);
  MEP_REQUIRE(e == hipSuccess, MEP_ERR_HIP, "%s: launch failed: %s", fn, hipGetErrorString(e));
  return MEP_OK;
}

extern "C" size_t mep_attention_block_workspace(int64_t n_rows, int32_t hidden, int32_t n_heads, int32_t n_kv_heads,
                                                int32_t head_dim) {
  if (n_rows < 0 || hidden <= 0 || n_heads <= 0 || n_kv_heads <= 0 || head_dim <= 0) return 0;
  // q, k, v, attention output, residual sum in front of the attention
  return static_cast<size_t>(n_rows) * 2 * (hidden + (2 * static_cast<size_t>(n_heads) + 2 * n_kv_heads) * head_dim);
}

extern "C" int mep_attention_block(const void* h, const void* delta, float mult, const void* norm1, const void* norm2,
                                   float eps, const void* wq, const void* wk, const void* wv, const void* wo,
                                   const float* cos, const float* sin, int64_t n_positions, int32_t batch, int32_t t,
                                   int32_t hidden, int32_t n_heads, int32_t n_kv_heads, int32_t head_dim, int64_t start,
                                   int64_t max_len, float scale, float* k_cache, float* v_cache, void* workspace,
                                   size_t workspace_bytes, void* h_out, void* x_out, void* stream) {
  clear_error();
  const char* fn = "mep_attention_block";
  const int rc = check_attention(fn, n_positions, batch, t, n_heads, n_kv_heads, head_dim, start, max_len);
  if (rc != MEP_OK) return rc;
  const int64_t n = static_cast<int64_t>(batch) * t;
  const int q_cols = n_heads * head_dim, kv_cols = n_kv_heads * head_dim;
  MEP_REQUIRE(n <= kRowsMax && linear_rows_k(hidden) && linear_rows_k(q_cols), MEP_ERR_UNSUPPORTED,
              "%s: %lld rows (at most %d), hidden %d and %d query columns (1024 or 2048)", fn,
              static_cast<long long>(n), kRowsMax, hidden, q_cols);
  if (n == 0) return MEP_OK;
  MEP_REQUIRE(h && norm1 && norm2 && wq && wk && wv && wo && cos && sin && k_cache && v_cache && workspace && h_out && x_out,
              MEP_ERR_INVALID_ARG, "%s: null pointer", fn);
  const size_t need = mep_attention_block_workspace(n, hidden, n_heads, n_kv_heads, head_dim);
  MEP_REQUIRE(workspace_bytes >= need, MEP_ERR_WORKSPACE, "%s: workspace %zu B < required %zu B", fn, workspace_bytes, need);
  for (const void* ptr : {h, delta, norm1, norm2, wq, wk, wv, wo, static_cast<const void*>(cos),
                          static_cast<const void*>(sin), static_cast<const void*>(k_cache),
                          static_cast<const void*>(v_cache), static_cast<const void*>(workspace),
                          static_cast<const void*>(h_out), static_cast<const void*>(x_out)})
    MEP_REQUIRE(aligned16(ptr), MEP_ERR_INVALID_ARG, "%s: buffers must be 16-byte aligned", fn);
  MEP_REQUIRE(h != h_out, MEP_ERR_INVALID_ARG, "%s: h_out must not be h", fn);
  uint16_t* const q = static_cast<uint16_t*>(workspace);
  uint16_t* const k = q + n * q_cols;
  uint16_t* const v = k + n * kv_cols;
  uint16_t* const o = v + n * kv_cols;
  uint16_t* const h1 = o + n * q_cols;
  hipStream_t s = static_cast<hipStream_t>(stream);

  LinearParams lin{};
  lin.x = static_cast<const uint16_t*>(h);
  lin.delta = static_cast<const uint16_t*>(delta);
  lin.norm_w = static_cast<const uint16_t*>(norm1);
  lin.h_out = delta != nullptr ? h1 : nullptr;
  lin.mult = mult;
  lin.eps = eps;
  const void* const w[3] = {wq, wk, wv};
  uint16_t* const out[3] = {q, k, v};
  for (int i = 0; i < 3; ++i) {
    lin.w[i] = static_cast<const uint16_t*>(w[i]);
    lin.out[i] = out[i];
    lin.cols[i] = i == 0 ? q_cols : kv_cols;
  }
  lin.n = static_cast<int>(n);
  hipError_t e = launch_linear_rows<true, kLinPlain>(lin, hidden, s);
  MEP_REQUIRE(e == hipSuccess, MEP_ERR_HIP, "%s: launch failed: %s", fn, hipGetErrorString(e));

  AttnParams p;
  p.q = q; p.k = k; p.v = v; p.cos = cos; p.sin = sin; p.kc = k_cache; p.vc = v_cache; p.out = o;
  p.batch = batch; p.t = t; p.hq = n_heads; p.hk = n_kv_heads;
  p.start = static_cast<int>(start); p.max_len = max_len; p.scale = scale;
  e = launch_attention<MEP_DTYPE_BF16>(p, s);
  MEP_REQUIRE(e == hipSuccess, MEP_ERR_HIP, "%s: launch failed: %s", fn, hipGetErrorString(e));

  LinearParams proj{};
  proj.x = o;
  proj.w[0] = static_cast<const uint16_t*>(wo);
  proj.out[0] = h_out;
  proj.cols[0] = hidden;
  proj.res = delta != nullptr ? h1 : static_cast<const uint16_t*>(h);
  proj.out_mult = mult;
  proj.n = static_cast<int>(n);
  e = launch_linear_rows<false, kLinResidual>(proj, q_cols, s);
  MEP_REQUIRE(e == hipSuccess, MEP_ERR_HIP, "%s: launch failed: %s", fn, hipGetErrorString(e));
  e = launch_add_norm(h_out, nullptr, 1.0f, norm2, eps, n, hidden, MEP_DTYPE_BF16, nullptr, x_out, s);
  MEP_REQUIRE(e == hipSuccess, MEP_ERR_HIP, "%s: launch failed: %s", fn, hipGetErrorString(e));
  return MEP_OK;
}

extern "C" int mep_norm_head(const void* h, const void* delta, float mult, const void* norm, float eps, const void* w,
                             int64_t n_rows, int32_t hidden, int32_t vocab, float divisor, float* logits, void* stream) {
  clear_error();
  const char* fn = "mep_norm_head";
  MEP_REQUIRE(n_rows >= 0 && vocab >= 1, MEP_ERR_INVALID_ARG, "%s: bad sizes", fn);
  MEP_REQUIRE(n_rows <= kRowsMax && linear_rows_k(hidden), MEP_ERR_UNSUPPORTED,
              "%s: %lld rows (at most %d), hidden %d (1024 or 2048)", fn, static_cast<long long>(n_rows), kRowsMax,
              hidden);
  if (n_rows == 0) return MEP_OK;
  MEP_REQUIRE(h && norm && w && logits, MEP_ERR_INVALID_ARG, "%s: null pointer", fn);
  MEP_REQUIRE(aligned16(h) && aligned16(delta) && aligned16(norm) && aligned16(w), MEP_ERR_INVALID_ARG,
              "%s: buffers must be 16-byte aligned", fn);
  LinearParams lin{};
  lin.x = static_cast<const uint16_t*>(h);
  lin.delta = static_cast<const uint16_t*>(delta);
  lin.norm_w = static_cast<const uint16_t*>(norm);
  lin.mult = mult;
  lin.eps = eps;
  lin.w[0] = static_cast<const uint16_t*>(w);
  lin.out[0] = logits;
  lin.cols[0] = vocab;
  lin.out_mult = divisor;
  lin.n = static_cast<int>(n_rows);
  const hipError_t e = launch_linear_rows<true, kLinScaled>(lin, hidden, static_cast<hipStream_t>(stream));
  MEP_REQUIRE(e == hipSuccess, MEP_ERR_HIP, "%s: launch failed: %s", fn, hipGetErrorString(e));
  return MEP_OK;
}

extern "C" int mep_linear(const void* x, int64_t n_rows, int32_t k, const void* const* w, const int32_t* cols,
                          int32_t n_mats, void* const* out, void* stream) {
  clear_error();
  const char* fn = "mep_linear";
  MEP_REQUIRE(n_rows >= 0 && n_mats >= 1 && n_mats <= 3 && w && cols && out, MEP_ERR_INVALID_ARG, "%s: bad sizes", fn);
  MEP_REQUIRE(k >= 256 && k % 128 == 0 && k <= (1 << 20), MEP_ERR_UNSUPPORTED,
              "%s: K %d must be a multiple of 128, at least 256", fn, k);
  MEP_REQUIRE(n_rows * k < (int64_t(1) << 31) && n_rows < (int64_t(1) << 23), MEP_ERR_UNSUPPORTED, "%s: x too large", fn);
  LinearTileParams p{};
  int64_t tiles = 0;
  for (int i = 0; i < 3; ++i) {
    p.cols[i] = i < n_mats ? cols[i] : 0;
    MEP_REQUIRE(i >= n_mats || (p.cols[i] > 0 && p.cols[i] % 128 == 0 &&
                                static_cast<int64_t>(p.cols[i]) * k < (int64_t(1) << 31)), MEP_ERR_UNSUPPORTED,
                "%s: %d columns must be a multiple of 128", fn, p.cols[i]);
    tiles += p.cols[i] / 128;
    p.tiles[i] = static_cast<int>(tiles);
  }
  MEP_REQUIRE((n_rows + 63) / 64 * tiles < (int64_t(1) << 31), MEP_ERR_UNSUPPORTED, "%s: too many tiles", fn);
  if (n_rows == 0) return MEP_OK;
  MEP_REQUIRE(x != nullptr && aligned16(x), MEP_ERR_INVALID_ARG,
              "%s: buffers must be present and 16-byte aligned", fn);
  for (int i = 0; i < n_mats; ++i) {
    MEP_REQUIRE(w[i] && out[i] && aligned16(w[i]) && aligned16(out[i]), MEP_ERR_INVALID_ARG,
                "%s: buffers must be present and 16-byte aligned", fn);
    p.w[i] = static_cast<const uint16_t*>(w[i]);
    p.out[i] = static_cast<uint16_t*>(out[i]);
  }
  p.x = static_cast<const uint16_t*>(x);
  p.n = static_cast<int>(n_rows);
  p.K = k;
  const hipError_t e = launch_linear_tile(p, static_cast<hipStream_t>(stream));
  MEP_REQUIRE(e == hipSuccess, MEP_ERR_HIP, "%s: launch failed: %s", fn, hipGetErrorString(e));
  return MEP_OK;
}
