// arcq_attention.hip -- causal attention of whole prompts, bf16, head_dim 128, grouped query heads
// (model/qLlamaLayer.py:340-370: softmax(q k^T / sqrt(d)) v over a prompt's own keys).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "arcq_gemm_tile.h"

namespace arcq {
namespace {

struct AttentionParams {
  const uint16_t *q, *k, *v;  // rows of tokens, a head's 128 values contiguous
  uint16_t *o;
  int ldq, ldk, ldv, ldo;     // elements from token to token
  int batch, seq, heads, kv_heads;
  float scale;                // of q k^T, times log2 e
  const uint16_t *cos, *sin;  // [positions, 64], of queries that are not rotated yet
  int positions;
};

typedef short v4s __attribute__((ext_vector_type(4)));
typedef v4s __attribute__((address_space(3))) lds_v4s;

// ---------------------------------------------------------------------------------------------
// A workgroup of four waves takes 128 queries of one head, a wave 32 of them, and walks the keys in tiles of 64.
//
// Both products are formed transposed: S^T = K Q^T, then O^T += V^T P^T, with v_mfma_f32_32x32x16_bf16.  A lane then holds
// 32 scores of ONE query per tile (its partner lane, 32 away, the other 32), so that maxima and sums need one exchange
// between two lanes, and its scores, rounded to bf16, already are the second product's operand: a lane of half h has keys
// 8 i + 4 h .. + 3 of a 32-key tile in accumulator registers 4 i .. 4 i + 3, and which key sits in which place of a matrix
// instruction is free as long as V^T agrees.  V^T comes out of LDS by transposing reads (ds_read_b64_tr_b16: sixteen lanes read
// 4 keys x 16 channels and get a channel's four keys each).
//
// K and V tiles travel by LDS-direct loads into two stages; 64 KB and 256 registers a wave leave room for two workgroups per
// CU, and the softmax of one runs beside the products of the other.  Rows of 256 bytes, 16-byte chunks swizzled: K by the key's
// low four bits (sixteen keys on one chunk), V by its low two, in steps of 64 bytes (eight keys on 64 bytes).
//
// The running maximum is exact at every tile of 64 keys, and the weights' sum is taken before they are rounded to bf16: the
// rounding of every weight is then that of torch's kernel (one output in 3000 to 10000 differs, by a bf16 step), behind which a quantizer
// makes the same codes.  (Raising the maximum only beyond 2^8 saves 4 %, but a row's largest weight is then no longer exactly 1:
// error against 64 bits 2.1e-3 in norm, so 1.8e-3 as torch's, the bf16 output alone 1.66e-3.)  O is rescaled only when some query's
// maximum moves.  us, torch's scaled_dot_product_attention before, N(0, 1) operands: 8 x 2048 tokens, 32 heads, 8 KV heads 747 -> 361
// (763 TFLOP/s; 339 in a layer), 4 x 1024 163 -> 58, 3 x 777, 28 heads, 4 KV heads 108 -> 39, 1 x 100 22 -> 11.  (Sequences of one token, 28
// heads, 64 of them: 6.7 -> 16.9.)
//
// ROTATE: the queries come as the projection left them and take their rotary embedding in registers.  Channels c and c + 64 of a query
// are the same lane's, every (query, head) is some workgroup's once, and the products are rounded as rope_rows_kernel rounds them: the
// same bits, without q written and read again.  Rotary pass + attention, us, q in the pass / here: 8 x 2048 tokens, 32 heads, 8 KV heads
// 71 + 354 / 19 + 367, 4096 tokens 23 + 67 / 8 + 71; a layer of 8 x 2048 tokens 5672 / 5624, of 4096 (MXFP4) 650 / 638.
//
// XCDs get contiguous runs of (sequence, KV head) groups, whose K and V their L2 then holds, the longest query tiles first.
// ---------------------------------------------------------------------------------------------
constexpr int kQ = 128, kKeys = 64, kStage = kKeys * 256;

// two channels of a query and the two 64 further on, each a pair of bf16: x cos - y sin and y cos + x sin, every product and sum rounded
__device__ __forceinline__ void rotate(uint32_t &x, uint32_t &y, uint32_t cs, uint32_t sn) {
  const float x0 = u2f(x << 16), x1 = u2f(x & 0xffff0000u), y0 = u2f(y << 16), y1 = u2f(y & 0xffff0000u);
  const float c0 = u2f(cs << 16), c1 = u2f(cs & 0xffff0000u), s0 = u2f(sn << 16), s1 = u2f(sn & 0xffff0000u);
  x = add_bf16_pair(pack_bf16_rne(x0 * c0, x1 * c1), pack_bf16_rne(-y0 * s0, -y1 * s1));
  y = add_bf16_pair(pack_bf16_rne(y0 * c0, y1 * c1), pack_bf16_rne(x0 * s0, x1 * s1));
}

template <bool ROTATE>
__global__ __launch_bounds__(256, 2) void attention_prefill_kernel(AttentionParams p) {
  __shared__ uint4 smem[4 * kStage / 16];  // K and V, two stages each
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = p.heads / p.kv_heads, tiles = (p.seq + kQ - 1) / kQ;
  const int per_group = tiles * group, total = p.batch * p.kv_heads * per_group;
  const int lin = (blockIdx.x & 7) * ((total + 7) >> 3) + (blockIdx.x >> 3);
  if (lin >= total || (int)(blockIdx.x >> 3) >= ((total + 7) >> 3)) return;
  const int gi = lin / per_group, in_group = lin - gi * per_group;
  const int b = gi / p.kv_heads, kvh = gi - b * p.kv_heads;
  const int qt = tiles - 1 - in_group / group, head = kvh * group + in_group % group;
  const int q0 = qt * kQ, qw = q0 + 32 * wave;          // first query of the workgroup, of the wave
  const int n_tiles = (min(q0 + kQ, p.seq) + kKeys - 1) / kKeys;
  const size_t row0 = (size_t)b * p.seq;

  const int r = lane & 31, h = lane >> 5;
  // ---- queries: channels 16 c + 8 h .. + 7 of query qw + r
  v8bf qf[8];
  {
    const uint16_t *src = p.q + (row0 + min(qw + r, p.seq - 1)) * p.ldq + head * 128 + 8 * h;
#pragma unroll
    for (int c = 0; c < 8; ++c) qf[c] = __builtin_bit_cast(v8bf, *reinterpret_cast<const uint4 *>(src + 16 * c));
    if constexpr (ROTATE) {
      const int at = min(min(qw + r, p.seq - 1), p.positions - 1) * 64 + 8 * h;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const uint4 cs = *reinterpret_cast<const uint4 *>(p.cos + at + 16 * c), sn = *reinterpret_cast<const uint4 *>(p.sin + at + 16 * c);
        uint4 x = __builtin_bit_cast(uint4, qf[c]), y = __builtin_bit_cast(uint4, qf[c + 4]);
        rotate(x.x, y.x, cs.x, sn.x);
        rotate(x.y, y.y, cs.y, sn.y);
        rotate(x.z, y.z, cs.z, sn.z);
        rotate(x.w, y.w, cs.w, sn.w);
        qf[c] = __builtin_bit_cast(v8bf, x), qf[c + 4] = __builtin_bit_cast(v8bf, y);
      }
    }
  }

  // ---- global -> LDS: four instructions per wave, tile and operand, four keys each
  const uint8_t *kbase = reinterpret_cast<const uint8_t *>(p.k + row0 * p.ldk + kvh * 128);
  const uint8_t *vbase = reinterpret_cast<const uint8_t *>(p.v + row0 * p.ldv + kvh * 128);
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>(smem);
  const int d_key = 16 * wave + (lane >> 4), d_pos = lane & 15;
  auto request = [&](int j) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = d_key + 4 * i;
      const uint32_t at = (uint32_t)min(j * kKeys + key, p.seq - 1);
      const uint32_t dst = lds0 + (j & 1) * (2 * kStage) + (16 * wave + 4 * i) * 256;
      lds_dma16_at(kbase, at * (uint32_t)(2 * p.ldk) + ((d_pos ^ (key & 15)) << 4), dst);
      lds_dma16_at(vbase, at * (uint32_t)(2 * p.ldv) + ((d_pos ^ ((key & 3) << 2)) << 4), dst + kStage);
    }
  };

  // ---- LDS -> operands
  const uint8_t *lds = reinterpret_cast<const uint8_t *>(smem);
  int k_rd[8];  // chunk 2 c + h of key r
#pragma unroll
  for (int c = 0; c < 8; ++c) k_rd[c] = r * 256 + (((2 * c + h) ^ (r & 15)) << 4);
  // transposing read: lane s of sixteen fetches channels 4 (s & 3) .. + 3 of key s / 4 and gets four keys of channel s
  const int s16 = lane & 15, v_key = 4 * h + (s16 >> 2);
  int v_rd[4];  // by 32-channel tile: key v_key, channels 32 t + 16 (lane / 16 & 1) + 4 (s & 3)
#pragma unroll
  for (int t = 0; t < 4; ++t)
    v_rd[t] = v_key * 256 + (((4 * t + 2 * ((lane >> 4) & 1) + ((s16 & 3) >> 1)) ^ ((v_key & 3) << 2)) << 4) + (s16 & 1) * 8;

  v16f o[4];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[t][e] = 0.0f;
  float m = -__builtin_inff(), l = 0.0f;
  const float c = p.scale;

  auto tile = [&](int j) {
    const uint8_t *ks = lds + (j & 1) * (2 * kStage), *vs = ks + kStage;
    v16f s[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int d = 0; d < 8; ++d) {
        const v8bf kf = __builtin_bit_cast(v8bf, *reinterpret_cast<const uint4 *>(ks + k_rd[d] + u * (32 * 256)));
        s[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[d], d ? s[u] : v16f{}, 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);  // (operands of more than this are not held in registers at once)
    }
    if (j * kKeys + kKeys - 1 > qw) {  // some of the keys are behind some of the wave's queries
      const int first = j * kKeys + 4 * h - (qw + r);  // key 8 i + e of the lane's, behind its query
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (first + 32 * u + 8 * (e >> 2) + (e & 3) > 0) s[u][e] = -__builtin_inff();
    }
    float top = s[0][0];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int e = 0; e < 16; ++e) top = __builtin_fmaxf(top, s[u][e]);
    top = __builtin_fmaxf(top, __shfl_xor(top, 32));
    // (a query whose scores have all been -inf so far, by an infinity among its keys: weights of 0, not exp2(-inf + inf))
    if (__builtin_amdgcn_ballot_w64(top > m) != 0) {
      const float next = __builtin_fmaxf(m, top), down = next == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f((m - next) * c);
      m = next;
      l *= down;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[t][e] *= down;
    }
    const float mc = m == -__builtin_inff() ? 0.0f : m * c;
    v8bf pf[4];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        uint32_t w[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float a = __builtin_amdgcn_exp2f(__builtin_fmaf(s[u][8 * g + 2 * e], c, -mc));
          const float d = __builtin_amdgcn_exp2f(__builtin_fmaf(s[u][8 * g + 2 * e + 1], c, -mc));
          l += a + d;
          w[e] = pack_bf16_rne(a, d);
        }
        pf[2 * u + g] = __builtin_bit_cast(v8bf, make_uint4(w[0], w[1], w[2], w[3]));
      }
#pragma unroll
    for (int g = 0; g < 4; ++g)  // 16 keys
#pragma unroll
      for (int t = 0; t < 4; ++t) {  // 32 channels
        const uint8_t *at = vs + v_rd[t] + g * (16 * 256);
        const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s *)(uintptr_t)(uint32_t)(uintptr_t)at);
        const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s *)(uintptr_t)(uint32_t)(uintptr_t)(at + 8 * 256));
        typedef short v8s __attribute__((ext_vector_type(8)));
        const v8s both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, both), pf[g], o[t], 0, 0, 0);
        if (t == 3 && (g & 1)) __builtin_amdgcn_sched_barrier(0);
      }
  };

  request(0);
  for (int j = 0; j < n_tiles; ++j) {
    wait_dma_and_sync();  // tile j is there, and everyone is done with the stage of tile j - 1
    if (j + 1 < n_tiles) request(j + 1);
    if (j * kKeys <= qw + 31) tile(j);  // (else its keys are behind all of this wave's queries)
  }

  // ---- O^T / l -> bf16 rows, through LDS: 8 KB per wave
  l += __shfl_xor(l, 32);
  const float inv = 1.0f / l;
  wait_dma_and_sync();
  uint8_t *region = reinterpret_cast<uint8_t *>(smem) + wave * 8192;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // channels 32 t + 8 i + 4 h .. + 3 of query r
      const int c8 = 8 * t + 2 * i + h;
      *reinterpret_cast<uint2 *>(region + r * 256 + ((c8 ^ ((r & 15) << 1)) << 3)) =
          make_uint2(pack_bf16_rne(o[t][4 * i] * inv, o[t][4 * i + 1] * inv), pack_bf16_rne(o[t][4 * i + 2] * inv, o[t][4 * i + 3] * inv));
    }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup", "local");
  const int rr = lane >> 4, t16 = lane & 15;
#pragma unroll
  for (int it = 0; it < 8; ++it) {
    const int row = 4 * it + rr;
    if (qw + row >= p.seq) continue;
    const uint4 v = *reinterpret_cast<const uint4 *>(region + row * 256 + (((2 * t16) ^ ((row & 15) << 1)) << 3));
    *reinterpret_cast<uint4 *>(p.o + (row0 + qw + row) * p.ldo + head * 128 + 8 * t16) = v;
  }
}

// cos_t, sin_t: null for rotated queries
int attention_entry(const void *q, int ldq, bool rotate, const void *cos_t, const void *sin_t, int positions, const void *k, int ldk,
                    const void *v, int ldv, int batch, int seq, int num_qo_heads, int num_kv_heads, int head_dim, float sm_scale, void *o,
                    int ldo, void *stream) {
  const float scale = sm_scale * 1.44269504088896341f;
  if (!(scale > 0.0f) || std::isinf(scale)) return ARCQ_ERR_SHAPE;  // the maximum is taken, and masked, ahead of the scale
  if (batch < 0 || seq < 0 || head_dim != 128 || num_kv_heads < 1 || num_qo_heads < num_kv_heads || num_qo_heads % num_kv_heads != 0)
    return ARCQ_ERR_SHAPE;
  const int need_q = num_qo_heads * 128, need_kv = num_kv_heads * 128;
  if (rotate && (positions < 1 || positions > (1 << 24))) return ARCQ_ERR_SHAPE;
  if (ldq < need_q || ldo < need_q || ldk < need_kv || ldv < need_kv || (ldq | ldk | ldv | ldo) % 8 != 0) return ARCQ_ERR_SHAPE;
  // 32-bit byte offsets of a sequence's keys
  if ((size_t)seq * (size_t)std::max(ldk, ldv) * 2 >= ((size_t)1 << 32)) return ARCQ_ERR_SHAPE;
  if (batch == 0 || seq == 0) return ARCQ_OK;
  if (!q || !k || !v || !o || (rotate && (!cos_t || !sin_t))) return ARCQ_ERR_NULL;
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(o) || !aligned16(cos_t) || !aligned16(sin_t)) return ARCQ_ERR_ALIGN;
  const long total = (long)batch * num_qo_heads * ((seq + kQ - 1) / kQ);
  if (total > (1l << 30)) return ARCQ_ERR_SHAPE;
  AttentionParams p{static_cast<const uint16_t *>(q), static_cast<const uint16_t *>(k), static_cast<const uint16_t *>(v),
                    static_cast<uint16_t *>(o), ldq, ldk, ldv, ldo, batch, seq, num_qo_heads, num_kv_heads,
                    scale,  static_cast<const uint16_t *>(cos_t),  static_cast<const uint16_t *>(sin_t),  positions};
  const auto kernel = rotate ? attention_prefill_kernel<true> : attention_prefill_kernel<false>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)(((total + 7) / 8) * 8)), dim3(256), 0, static_cast<hipStream_t>(stream), p);
  ARCQ_HIP_TRY(hipGetLastError());
  return ARCQ_OK;
}

}  // namespace
}  // namespace arcq

extern "C" int arcq_attention_prefill(const void *q, int ldq, const void *k, int ldk, const void *v, int ldv, int batch, int seq,
                                      int num_qo_heads, int num_kv_heads, int head_dim, float sm_scale, void *o, int ldo, void *stream) {
  return arcq::attention_entry(q, ldq, false, nullptr, nullptr, 0, k, ldk, v, ldv, batch, seq, num_qo_heads, num_kv_heads, head_dim,
                               sm_scale, o, ldo, stream);
}

extern "C" int arcq_attention_prefill_rope(const void *q, int ldq, const void *cos_table, const void *sin_table, int max_positions,
                                           const void *k, int ldk, const void *v, int ldv, int batch, int seq, int num_qo_heads,
                                           int num_kv_heads, int head_dim, float sm_scale, void *o, int ldo, void *stream) {
  return arcq::attention_entry(q, ldq, true, cos_table, sin_table, max_positions, k, ldk, v, ldv, batch, seq, num_qo_heads, num_kv_heads,
                               head_dim, sm_scale, o, ldo, stream);
}
