// arcq_gemm_nv_stream.hip -- NVFP4 GEMM of decode batches (up to 64 rows, or experts of few rows each): one pass over the
// weights, all of whose bytes are on their way through many small workgroups; and of a few hundred rows where tiles do not fill the chip.
#include <hip/hip_runtime.h>
#include <limits.h>
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "arcq_gemm_tile.h"

namespace arcq {
namespace {

// At most n of this wave's loads may still be on their way (more than the instruction's cases here: a stricter wait).
__device__ __forceinline__ void wait_vmcnt(int n) {
  switch (n) {
    case 0: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
    case 1: asm volatile("s_waitcnt vmcnt(1)" ::: "memory"); break;
    case 2: asm volatile("s_waitcnt vmcnt(2)" ::: "memory"); break;
    case 3: asm volatile("s_waitcnt vmcnt(3)" ::: "memory"); break;
    case 4: asm volatile("s_waitcnt vmcnt(4)" ::: "memory"); break;
    case 5: asm volatile("s_waitcnt vmcnt(5)" ::: "memory"); break;
    case 6: asm volatile("s_waitcnt vmcnt(6)" ::: "memory"); break;
    case 7: asm volatile("s_waitcnt vmcnt(7)" ::: "memory"); break;
    case 8: asm volatile("s_waitcnt vmcnt(8)" ::: "memory"); break;
    case 9: asm volatile("s_waitcnt vmcnt(9)" ::: "memory"); break;
    case 10: asm volatile("s_waitcnt vmcnt(10)" ::: "memory"); break;
    default: asm volatile("s_waitcnt vmcnt(11)" ::: "memory"); break;
  }
}

// ---------------------------------------------------------------------------------------------
// A workgroup multiplies 16 NT WN weight rows with 16 MT activation rows.  Its WN x WK waves share the K steps of 64 WK
// elements: a wave takes 64 elements of every step and 16 NT rows, decodes both operands to fp16 in registers and feeds
// v_mfma_f32_16x16x32_f16.  The WK partial sums of a tile meet in LDS at the end.
//
// What bounds such a problem is the stream of the weights, and in front of it everything that keeps a CU from asking for
// more of them: waves that wait for one another, load instructions that touch a cache line for a few bytes, and the decoding,
// which costs 8 VALU instructions (a wave's takes 2 ns on its SIMD once two or more waves offer them, 4 ns alone) per 512
// codes and operand.  So (EK = 64 elements of a step per wave, or 128 where workgroups have a CU to themselves):
//  - NT is as large as the grid allows: the activations are decoded once per workgroup (WN = 1), whatever its rows.
//  - Codes travel by LDS-direct loads in whole rows of 128 to 512 bytes, scale bytes in 64-byte windows (1024 elements): with
//    16-byte windows, or straight to registers, the cache lines fetched for scale bytes outweigh the codes.
//  - Two stages (one step on its way) and small workgroups, two to four per CU, that wait independently: 28672 x 4352 with 16
//    rows 15.7 us (4.5 TB/s); three stages in the same shape 17.6, sixteen waves on 128 rows and four stages 20.3.
// Before (64x32 and 128x64 tiles, the latter's K cut in slices and added up by a second launch, or a lane's operands straight
// from global memory), us, weights from HBM, 16 / 32 / 64 rows: 28672 x 4352 23.2 / 25.7 / 28.2, now 15.7 / 18.5 / 24.7;
// 14336 x 4352 17.8 / 26 / 26.4, now 10.9 / 14 / 16.9; 6144 x 4352 10.0 / 14.6 / 17.1, now 7.8 / 8.8 / 11.5; 4096 x 4352 6.6 / 9.0 /
// 12.5, now 6.0 / 6.9 / 9.4; 4096 x 14592 16.9 / 20.8 / 22.2, now 12.1 / 15.3 / 21.3.
// ---------------------------------------------------------------------------------------------
template <int MT, int NT, int WN, int WK, int NS, int EK = 64>
struct StreamShape {
  static constexpr int NW = WN * WK, BN = 16 * NT * WN, BM = 16 * MT;
  static constexpr int RB = EK / 2 * WK;         // code bytes of a row in one step (EK elements per wave)
  static constexpr int SB = RB >= 512 ? 1 : 512 / RB;  // steps per scale window of 64 bytes
  static constexpr int NB = (NS + SB - 2) / SB + 1;  // windows on their way or in use
  static constexpr int kCodes = NS * (BN + BM) * RB, kScales = NB * (BN + BM) * 64;
  static constexpr int kLds = kCodes + kScales;
  // the waves' sums meet in LDS a few 16x16 tiles per wave at a time
  static constexpr int kBatches = (NW * NT * MT * 1024 + kLds - 1) / kLds, kBatch = (NT * MT + kBatches - 1) / kBatches;
  static_assert(NW * kBatch * 1024 <= kLds, "a batch of sums fits");
};

template <int MT, int NT, int WN, int WK, int NS, bool GROUPED, int EK = 64>
__device__ __forceinline__ void nv_stream_tile(const GemmParams &p, int n_base, int m_base, uint8_t *smem) {
  using S = StreamShape<MT, NT, WN, WK, NS, EK>;
  constexpr int NW = S::NW, BN = S::BN, BM = S::BM, RB = S::RB, SB = S::SB, NB = S::NB;
  constexpr int CPR = RB / 16, RPI = 64 / CPR;      // 16-byte chunks per row, rows per load instruction
  constexpr int WI = BN / RPI, NI = (BN + BM) / RPI;  // load instructions of the weights and of both operands per step
  constexpr int PW = (NI + NW - 1) / NW;            // per wave, at most
  constexpr int SI = (BN + BM) / 16;                // of a scale window: 16 rows of 64 bytes each
  static_assert(BN % RPI == 0 && BM % RPI == 0, "whole instructions");
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int kbytes = p.Kp >> 1, ksc = p.Kp >> 4;
  const int nk = (kbytes + RB - 1) / RB;
  const uint8_t *wc = p.b_codes + (size_t)n_base * kbytes, *ws = p.b_scales + (size_t)n_base * ksc;
  const uint8_t *xc = p.a_codes + (size_t)m_base * kbytes, *xs = p.a_scales + (size_t)m_base * ksc;
  const int rows_w = p.N - 1 - n_base, rows_x = p.M - 1 - m_base;  // last valid row of either tile
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>(smem);
  // position of chunk c of a row: the 16 rows of an operand read spread over all banks
  auto swizzle = [](int row) { return CPR == 8 ? (row >> 1) & 7 : row & 15; };

  uint32_t ro[PW];
  int co[PW];
#pragma unroll
  for (int i = 0; i < PW; ++i) {
    const int k = wave + i * NW;
    const bool x = k >= WI;
    const int row = (x ? k - WI : k) * RPI + lane / CPR;
    ro[i] = (uint32_t)min(row, x ? rows_x : rows_w) * (uint32_t)kbytes;
    co[i] = ((lane % CPR) ^ swizzle(row)) * 16;
  }
  constexpr int PS = (SI + NW - 1) / NW;
  uint32_t so[PS];
  const int sp = ((lane & 3) ^ ((lane >> 4) & 3)) * 16;  // piece of the window; rows 4 apart take turns
#pragma unroll
  for (int i = 0; i < PS; ++i) {
    const int k = wave + i * NW;
    const bool x = k >= BN / 16;
    const int row = (x ? k - BN / 16 : k) * 16 + (lane >> 2);
    so[i] = (uint32_t)min(row, x ? rows_x : rows_w) * (uint32_t)ksc;
  }

  auto request = [&](int kt, int st, int win) {
    if (kt % SB == 0) {
#pragma unroll
      for (int i = 0; i < PS; ++i) {
        const int k = wave + i * NW;
        if (k < SI)  // (pieces past the row's end: its last 16 bytes)
          lds_dma16_at(k >= BN / 16 ? xs : ws, so[i] + (uint32_t)min((kt / SB) * 64 + sp, ksc - 16),
                       lds0 + S::kCodes + win * ((BN + BM) * 64) + k * 1024);
      }
    }
#pragma unroll
    for (int i = 0; i < PW; ++i) {
      const int k = wave + i * NW;
      if (k < NI)
        lds_dma16_at(k >= WI ? xc : wc, ro[i] + (uint32_t)min(kt * RB + co[i], kbytes - 16), lds0 + st * ((BN + BM) * RB) + k * 1024);
    }
  };
  const int mine = (NI - wave + NW - 1) / NW;  // load instructions of this wave per step
  const int mine_s = (SI - wave + NW - 1) / NW;
  auto group = [&](int kt) { return mine + (kt % SB == 0 ? mine_s : 0); };

  const int wn = wave % WN, wk = wave / WN;
  v4f acc[NT][MT];
#pragma unroll
  for (auto &a : acc)
#pragma unroll
    for (auto &b : a) b = v4f{0.f, 0.f, 0.f, 0.f};
  const int w_row = 16 * NT * wn + r, x_row = BN + r;
  const int chunk = EK == 64 ? 2 * wk + (g >> 1) : 4 * wk + g, in_chunk = EK == 64 ? (g & 1) * 8 : 0;
  const int w_rd = w_row * RB + ((chunk ^ swizzle(w_row)) << 4) + in_chunk;
  const int x_rd = x_row * RB + ((chunk ^ swizzle(r)) << 4) + in_chunk;
  const int swz_s = (r >> 2) & 3;

  auto compute = [&](int kt, int st, int win) {
    const int c64 = kt * WK + wk;  // this wave's 64 elements
    if (c64 * 32 >= kbytes) return;
    const int piece = c64 >> 2;
    const int sb = (((piece & 3) ^ swz_s) << 4) + 4 * (c64 & 3) + g + ((ksc & 15) && piece == (ksc >> 4) ? 8 : 0);
    const uint8_t *cs = smem + st * ((BN + BM) * RB), *ss = smem + S::kCodes + win * ((BN + BM) * 64) + sb;
    uint2 wq[NT], xq[MT];
    uint32_t wsc[NT], xsc[MT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      wq[i] = *reinterpret_cast<const uint2 *>(cs + w_rd + i * (16 * RB));
      wsc[i] = ss[(w_row + 16 * i) * 64];
    }
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      xq[j] = *reinterpret_cast<const uint2 *>(cs + x_rd + j * (16 * RB));
      xsc[j] = ss[(x_row + 16 * j) * 64];
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) wsc[i] = (wsc[i] << 7) + 0x1800u;
#pragma unroll
    for (int j = 0; j < MT; ++j) xsc[j] = (xsc[j] << 7) + 0x1800u;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      v8h b[MT];
#pragma unroll
      for (int j = 0; j < MT; ++j) b[j] = decode8_nvfp4_f16<false>(h ? xq[j].y : xq[j].x, xsc[j]);
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const v8h a = decode8_nvfp4_f16<false>(h ? wq[i].y : wq[i].x, wsc[i]);
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b[j], acc[i][j], 0, 0, 0);
      }
    }
  };
  // The same with 128 elements of a step per wave (EK = 128): a lane's 32 codes are one 16-byte read, their two scale bytes another one, and
  // the products of one quarter run with the decoding of the next between them.
  struct Operands {
    v8h w[NT], x[MT];
  };
  Operands quarter[EK == 128 ? 2 : 1];
  if constexpr (EK == 128) {
#pragma unroll
    for (auto &v : quarter[1].w) v = v8h{};
#pragma unroll
    for (auto &v : quarter[1].x) v = v8h{};
  }
  auto multiply = [&](const Operands &o) {
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(o.w[i], o.x[j], acc[i][j], 0, 0, 0);
  };
  auto compute128 = [&](int kt, int st, int win) {
    const int c = kt * WK + wk;  // this wave's 128 elements
    const int piece = c >> 1;
    const int sb = (((piece & 3) ^ swz_s) << 4) + 8 * (c & 1) + 2 * g + ((ksc & 15) && piece == (ksc >> 4) ? 8 : 0);
    const uint8_t *cs = smem + st * ((BN + BM) * RB), *ss = smem + S::kCodes + win * ((BN + BM) * 64) + sb;
    uint4 wq[NT], xq[MT];
    uint32_t wsc[NT], xsc[MT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      wq[i] = *reinterpret_cast<const uint4 *>(cs + w_rd + i * (16 * RB));
      wsc[i] = *reinterpret_cast<const uint16_t *>(ss + (w_row + 16 * i) * 64);
    }
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      xq[j] = *reinterpret_cast<const uint4 *>(cs + x_rd + j * (16 * RB));
      xsc[j] = *reinterpret_cast<const uint16_t *>(ss + (x_row + 16 * j) * 64);
    }
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      multiply(quarter[(h & 1) ^ 1]);  // (the step before's last quarter first)
      Operands &next = quarter[h & 1];
      auto scale = [&](uint32_t &two) { return ((h < 2 ? two & 0xffu : two >> 8) << 7) + 0x1800u; };
      auto dword = [&](const uint4 &q) { return h == 0 ? q.x : h == 1 ? q.y : h == 2 ? q.z : q.w; };
#pragma unroll
      for (int j = 0; j < MT; ++j) next.x[j] = decode8_nvfp4_f16<false>(dword(xq[j]), scale(xsc[j]));
#pragma unroll
      for (int i = 0; i < NT; ++i) next.w[i] = decode8_nvfp4_f16<false>(dword(wq[i]), scale(wsc[i]));
      constexpr int kEach = (10 * (NT + MT) + NT * MT - 1) / (NT * MT);
#pragma unroll
      for (int k = 0; k < NT * MT; ++k) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, kEach, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto barrier = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };

#pragma unroll
  for (int a = 0; a < NS - 1; ++a)
    if (a < nk) request(a, a, a / SB);
  int st = 0, st_req = NS - 1, win = 0, win_req = ((NS - 1) / SB) % NB;  // stages and windows of step kt and of the step requested
  for (int kt = 0; kt < nk; ++kt) {
    int younger = 0;
#pragma unroll
    for (int a = 1; a < NS - 1; ++a)
      if (kt + a < nk) younger += group(kt + a);
    wait_vmcnt(younger);
    barrier();  // step kt is there, and everyone is done with the stage of step kt - 1
    if (kt + NS - 1 < nk) request(kt + NS - 1, st_req, win_req);
    if constexpr (EK == 64)
      compute(kt, st, win);
    else if ((kt * WK + wk) * 64 < kbytes)
      compute128(kt, st, win);
    st = st == NS - 1 ? 0 : st + 1;
    st_req = st_req == NS - 1 ? 0 : st_req + 1;
    if ((kt + 1) % SB == 0) win = win == NB - 1 ? 0 : win + 1;
    if ((kt + NS) % SB == 0) win_req = win_req == NB - 1 ? 0 : win_req + 1;
  }

  if constexpr (EK == 128) multiply(quarter[1]);

  // the sums of the waves that share a tile meet in LDS, added in the order of K
  float4 *red = reinterpret_cast<float4 *>(smem);
  // (a grouped launch has one alpha and a residual of C's shape; with the parts' code in it, too, a decode step
  // over eight experts of 28672 x 4224 and 4096 x 14464 takes 288 us instead of 253)
  const std::conditional_t<GROUPED, OneAlpha, Alpha> by_column(p);
  const size_t ld_residual = GROUPED ? p.N : p.ld_residual;
  uint32_t amax = 0u;
  constexpr int Q = NT * MT, QB = S::kBatch;
#pragma unroll
  for (int b0 = 0; b0 < Q; b0 += QB) {
    barrier();
#pragma unroll
    for (int q = 0; q < QB; ++q)
      if (b0 + q < Q) {
        const v4f a = acc[(b0 + q) / MT][(b0 + q) % MT];
        red[(wave * QB + q) * 64 + lane] = make_float4(a[0], a[1], a[2], a[3]);
      }
    barrier();
    for (int t = wave; t < WN * QB; t += NW) {
      const int tn = t / QB, q = b0 + t % QB;  // tile q of the waves at position tn along N
      if (q >= Q) continue;
      float4 v = red[(tn * QB + t % QB) * 64 + lane];
#pragma unroll
      for (int w = 1; w < WK; ++w) {
        const float4 u = red[((w * WN + tn) * QB + t % QB) * 64 + lane];
        v.x += u.x, v.y += u.y, v.z += u.z, v.w += u.w;
      }
      const int n_tile = n_base + 16 * (NT * tn + q / MT), m = m_base + 16 * (q % MT) + r, n = n_tile + 4 * g;
      const float alpha = by_column.at(p, n_tile);
      if (p.swiglu) {  // N is a multiple of 16: a quad is inside C or outside as a whole
        const uint32_t o = swiglu_pair(pack_bf16_rne(v.x * alpha, v.z * alpha), pack_bf16_rne(v.y * alpha, v.w * alpha));
        if (m < p.M && n < p.N) {
          amax = max(amax, max(o & 0x7fffu, (o >> 16) & 0x7fffu));
          *reinterpret_cast<uint32_t *>(p.c + (size_t)m * (p.N >> 1) + (n >> 1)) = o;
        }
        continue;
      }
      if (m >= p.M || n >= p.N) continue;
      uint16_t *dst = p.c + (size_t)m * p.N + n;
      const uint16_t *res = p.residual ? p.residual + (size_t)m * ld_residual + n : nullptr;
      if ((p.N & 3) == 0) {
        uint2 o = make_uint2(pack_bf16_rne(v.x * alpha, v.y * alpha), pack_bf16_rne(v.z * alpha, v.w * alpha));
        if (res) o = add_bf16_x4(o, *reinterpret_cast<const uint2 *>(res));
        *reinterpret_cast<uint2 *>(dst) = o;
        continue;
      }
      const float f[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < p.N) {
          uint32_t h = f32_to_bf16_bits(f[e] * alpha);
          if (res) h = f32_to_bf16_bits(bf16_bits_to_f32(h) + bf16_bits_to_f32(res[e]));
          dst[e] = (uint16_t)h;
        }
    }
  }
  if (p.swiglu && p.absmax_bits) {
    // All workgroups of an expert share one word, and atomics on one word are served one after the other (28672 x 4224, eight
    // experts, one from every wave: 190 us, the GEMM alone 135): one per workgroup, and only if its maximum is above what the
    // word, which never falls, was seen to hold.
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) amax = max(amax, (uint32_t)__shfl_xor((int)amax, o));
    barrier();
    uint32_t *top = reinterpret_cast<uint32_t *>(smem);
    if (lane == 0) top[wave] = amax;
    barrier();
    if (threadIdx.x == 0) {
#pragma unroll
      for (int w = 1; w < NW; ++w) amax = max(amax, top[w]);
      uint32_t *word = p.absmax_bits + p.seg_index;
      if ((amax << 16) > *const_cast<volatile uint32_t *>(word)) atomicMax(word, amax << 16);  // bf16 bits -> fp32 bits
    }
  }
}

template <int MT, int NT, int WN, int WK, int NS, bool GROUPED, int EK = 64>
__global__ __launch_bounds__(64 * WN * WK) void gemm_nvfp4_stream(GemmParams p) {
  using S = StreamShape<MT, NT, WN, WK, NS, EK>;
  __shared__ uint4 smem[S::kLds / 16];
  uint8_t *lds = reinterpret_cast<uint8_t *>(smem);
  int lin;
  if constexpr (GROUPED) {
    if (!enter_segment_in_twos<S::BM, S::BN, 16>(p, lin)) return;
  } else {
    const int total = ((p.M + S::BM - 1) / S::BM) * ((p.N + S::BN - 1) / S::BN);
    lin = (blockIdx.x & 7) * ((total + 7) >> 3) + (blockIdx.x >> 3);
    if (lin >= total) return;
  }
  const int tiles_m = (p.M + S::BM - 1) / S::BM;
  const int n_base = (lin / tiles_m) * S::BN, m_base = (lin % tiles_m) * S::BM;
  if constexpr (GROUPED && MT > 1) {  // experts of few rows: no matrix instructions for rows that are not there
    const int rows = p.M - m_base;
    if (rows <= 16) return nv_stream_tile<1, NT, WN, WK, NS, GROUPED>(p, n_base, m_base, lds);
    if (MT > 2 && rows <= 32) return nv_stream_tile<2, NT, WN, WK, NS, GROUPED>(p, n_base, m_base, lds);
    if (MT > 3 && rows <= 48) return nv_stream_tile<3, NT, WN, WK, NS, GROUPED>(p, n_base, m_base, lds);
  }
  nv_stream_tile<MT, NT, WN, WK, NS, GROUPED, EK>(p, n_base, m_base, lds);
}

template <int MT, int NT, int WN, int WK, int NS, bool GROUPED = false, int EK = 64>
int launch(const GemmParams &p, hipStream_t st) {
  using S = StreamShape<MT, NT, WN, WK, NS, EK>;
  const int total = ((p.M + S::BM - 1) / S::BM + (GROUPED ? p.n_seg : 0)) * ((p.N + S::BN - 1) / S::BN);
  hipLaunchKernelGGL((gemm_nvfp4_stream<MT, NT, WN, WK, NS, GROUPED, EK>), dim3(grid_in_turn<GROUPED ? 2 : 1>(total)), dim3(64 * S::NW), 0, st, p);
  ARCQ_HIP_TRY(hipGetLastError());
  return ARCQ_OK;
}

// Rows per workgroup.  Up to 12288 rows of weights make at most one workgroup per CU of 16, 32 or 48 rows, which then has
// sixteen waves, or eight that take 128 elements of a step each (us at 16 rows: 6144 x 4352 7.8, eight waves of 64 elements 8.9; 10240 x
// 8320 15.0 and 17.6; at 16, 32, 64 rows of 6144 x 4352 sixteen waves 6.8, 8.0, 11.0, eight of 128 elements 6.5, 7.7, 10.7; but 64 rows of a
// longer K' are decoded faster by sixteen: 8192 x 6272 14.4 / 14.8, 8192 x 8448 18.2 / 19.1, 6144 x 14592 27.1 / 29.3, 48 rows 16.0 /
// 15.7 and 23.7 / 23.3).  Beyond, eight waves, and the
// rows per workgroup by how many rounds of 256 workgroups they make: the rows and activation rows of a CU's workgroups
// together, a quarter more where up to 32 rows, or a K' of one or two steps, have a single workgroup per CU to themselves (nothing else
// asks for weights while it starts, waits and ends): 28672 rows take 64 per workgroup up to 32 rows and 112 above (64 rows, K' = 4352:
// 24.7 us against 25.4; K' = 512: 64 per workgroup 8.2 against 9.3), 18944 rows 48 and 80.
template <int MT>
int launch_plain(const GemmParams &p, hipStream_t st) {
  if (p.N <= 4096) return launch<MT, 1, 1, 16, (MT == 1 ? 3 : 2)>(p, st);
  if (MT == 4 && p.N <= 8192 && p.Kp >= 6144) return launch<MT, 2, 1, 16, 2>(p, st);
  if (p.N <= 8192) return launch<MT, 2, 1, 8, 2, false, 128>(p, st);
  if (p.N <= 12288) return launch<MT, 3, 1, 16, 2>(p, st);
  int best = 0;
  double least = 0;
  for (const int nt : {2, 3, 4, 5, 7}) {
    const int groups = (p.N + 16 * nt - 1) / (16 * nt);
    const double cost = (groups + 255) / 256 * (nt + 0.25 * MT) * (groups <= 256 && (MT <= 2 || p.Kp < 1024) ? 1.25 : 1.0);
    if (!best || cost < least) best = nt, least = cost;
  }
  switch (best) {
    case 2: return launch<MT, 2, 1, 8, 2>(p, st);
    case 3: return launch<MT, 3, 1, 8, 2>(p, st);
    case 4: return launch<MT, 4, 1, 8, 2>(p, st);
    case 5: return launch<MT, 5, 1, 8, 2>(p, st);
    default: return launch<MT, 7, 1, 8, 2>(p, st);
  }
}

}  // namespace

// What the kernel takes: whole 128s of K', one step at least, 32-bit offsets inside a workgroup's rows.
bool nvfp4_stream_able(int M, int Kp, int n_seg) { return Kp % 128 == 0 && Kp >= 512 && Kp <= (1 << 24) && (n_seg > 0 || M <= 64); }

// The shortest K' from which on plain problems of up to 64 rows run as such a stream.  Below, the kernel that reads its operands
// straight into registers, which has nothing to fill, wait for and add up, gets in and out faster (the stream's waves take 512 to 1024
// elements at a time, and a last step that is mostly empty costs as much as a whole one), and 64 rows of a short K' on 32769 to 49151 rows
// of weights are as fast in 128x64 tiles.  us as a stream and so: 16 rows, 2048 x 1152 4.4 / 3.3, 4096 x 2176 5.3 / 4.4, 4096 x 8320 8.0
// / 9.4, 8192 x 1152 4.9 / 4.3, 12288 x 1152 5.6 / 4.9; 32 rows, 4096 x 1152 4.8 / 4.4, 4096 x 4352 6.9 / 8.8; 8 rows, 2048 x 8320 8.5 / 7.1,
// 3584 x 14592 10.8 / 11.6; 4 rows, 18944 x 1152 6.7 / 5.5, 18944 x 4352 13.0 / 16.4; 64 rows, 37888 x 512 13.0 / 9.6, 37888 x 2176 26.7 / 28.4.
constexpr int kNever = 1 << 30;
constexpr int kStreamRows[7] = {4, 7, 8, 16, 32, 48, 64};
constexpr struct {
  int N;           // up to this many rows of weights
  int from[7];     // K', by activation rows
} kStreamFrom[] = {{2048, {kNever, kNever, kNever, 10240, 4096, 0, 0}},
                   {4096, {kNever, 10240, 10240, 8192, 4096, 0, 0}},
                   {8192, {kNever, 4096, 4096, 4096, 2048, 0, 0}},
                   {12288, {2560, 2560, 2560, 2560, 0, 0, 0}},
                   {16383, {2560, 2560, 2560, 1536, 0, 0, 0}},
                   {24576, {2560, 2048, 0, 0, 0, 0, 0}},
                   {32768, {2048, 2048, 0, 0, 0, 0, 0}},
                   {49151, {2048, 2048, 0, 0, 0, 0, 1536}},
                   {INT_MAX, {2048, 2048, 0, 0, 0, 0, 0}}};

bool nvfp4_stream_wanted(int M, int N, int Kp, int n_seg, bool swiglu) {
  if (!nvfp4_stream_able(M, Kp, n_seg)) return false;
  // Experts: few rows on average, so that the weights are the work; a workgroup has at most 48 rows of its expert, and what they
  // decode of the weights is decoded again for the next 48.  us as a stream and in 128x64 tiles, even and skewed sizes, eight experts of
  // 4096 x 14464: 40 rows each 61, 86 / 85, 126; 48 rows 68, 148 / 84, 129; 64 rows 80, 150 / 85, 133; 8192 x 2176, 40 rows 26, 31 / 27, 38; 64
  // rows 34, 45 / 28, 39.  Wide layers take workgroups of 96 weight rows there, which decode less: 28672 x 4224, 64 rows 185, 220 / 185,
  // 237, 95 rows 290, 299 / 321, 322; so do a few narrow experts, all of whose tiles together are less than a round: 8 of 2048 x 8320, 64
  // rows 45, 45 / 49, 49.  K' < 2048: 64 of 2048 x 1536, 24 rows 31, 40 / 34, 40, 40 rows 38, 47 / 34, 42; 8 of 1536 x 1536, 40 rows 8.4, 8.7 /
  // 12.4, 12.4.
  if (n_seg > 0) {
    const int rows = M / n_seg;
    const bool few = (long)n_seg * N <= 16384;
    if (Kp < 2048) return rows <= (few ? 40 : 32);
    return rows <= 40 || (rows < 96 && (N > 8192 || few));
  }
  // The kernels above have no SwiGLU epilogue: the 128x64 tiles, which would take 1.05 (4096 x 512) to 5 (1024 x 14592) times as long.
  if (swiglu) return true;
  // (64 rows of a long K' on a narrow layer: 128x64 tiles with K in eight slices, 2048 x 19072 25.6 / 23.0 us, 1024 x 14592 20.2 / 19.5)
  if (M > 48 && N <= 4096 && Kp >= (N <= 1024 ? 12288 : 16384)) return false;
  if (M <= 7 && N > 20480 && Kp <= 512) return true;  // one step: 4 rows, 28672 x 512 5.3 / 6.1
  int n = 0, m = 0;
  while (N > kStreamFrom[n].N) ++n;
  while (M > kStreamRows[m]) ++m;
  return Kp >= kStreamFrom[n].from[m];
}

// Beyond 64 rows the same kernel with 64 to 112 rows per workgroup: both operands are decoded in every workgroup, but only
// once (its waves split K), which is about what the matrix instructions take, and small workgroups fill the chip where 128x128 tiles
// do not.  A workgroup's time per K' = 4352 and its wait to start and end (6 us; less for the smallest shapes, as long as they make one
// round), measured, by shape; where workgroups have a CU to themselves, each of several rounds takes an eighth more (us; workgroups of 1
// to 14 per CU; 1900 problems of 65 to 1024 rows, 256 to 28672 weight rows and K' = 512 to 14592 to within 10 % in one round):
// The larger shapes, whose workgroups have a CU to themselves in one round anyway, then take 128 elements of a step per wave (`one`): half as
// many LDS reads, barriers and waits, twice the bytes on their way.  us, 64 elements and 128: 333 x 6144 x 4352 27.9 / 25.4, 400 x 4096 x
// 4352 25.1 / 22.4, 512 x 4096 x 4352 25.5 / 23.1, 300 x 4608 x 3712 26.4 / 23.8.  (In several rounds two of the workgroups of 64 share a CU.)
struct MidShape {
  int mt, nt, wn, wk;
  double us, rounds;
  double short_start, short_us;
  double one;
};
constexpr double kMidStart = 6;
constexpr MidShape kMid[] = {{4, 3, 1, 8, 8.2, 1.0, 4.0, 10.0, 8.2},    {4, 4, 1, 8, 9.8, 1.0, 4.7, 11.8, 9.8},    {5, 3, 1, 8, 9.2, 1.0, 4.7, 11.3, 9.2},
                             {6, 4, 1, 8, 14.8, 1.12, 6, 14.8, 14.8}, {7, 3, 1, 8, 13.8, 1.12, 6, 13.8, 13.8}, {5, 3, 2, 4, 16.6, 1.0, 6, 16.8, 16.8},
                             {4, 4, 2, 4, 18.0, 1.0, 6, 17.6, 17.6},  {6, 3, 2, 4, 22.5, 1.0, 6, 19.8, 19.8},  {5, 4, 2, 4, 25.0, 1.0, 6, 21.5, 21.5}};

// The shape for a problem that the plan would give to 128x64 (21, K in `slices`), 128x128 (22) or 256x128 tiles (42), -1 where those
// are faster by their own measured times (`always`: the best one whatever theirs are).  Over 1888 measured problems 0.81 of the tiles'
// time; where it is taken, at worst 1.09 of it.  us, before and now: 128 x 6144 x 4352 21.9 and 14.3, 333 rows 34.4 and 28.5, 512 rows 34.1
// (kept); 256 x 4096 x 4352 23.3 and 16.3; 128 x 4096 x 14592 31 (kept), 333 rows 73.8 and 55.7; 80 x 28672 x 4352 43.6 and
// 33, 256 rows 62 (kept).
int nvfp4_mid_shape(int M, int N, int Kp, int kernel, int slices, bool always) {
  if (M <= 64 || M > 1024 || Kp < 512 || Kp % 128 != 0 || Kp > (1 << 24)) return -1;
  const double k = Kp / 4352.0;
  auto rounds = [](long groups) { return (double)((groups + 255) / 256); };
  auto tiles = [&](int bm, int bn) { return (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  double tiled;
  if (kernel == 21) {
    const double r = rounds(tiles(64, 128) * slices);
    tiled = slices > 1 ? 12 + 20 * k / slices * r : std::min(7 + 20 * k * r, 3.6 + 26 * k * r);  // (a short K' is little but its first step)
  } else if (kernel == 22)
    tiled = 4 + (tiles(128, 128) <= 256 ? 30 : 27) * k * rounds(tiles(128, 128));
  else if (kernel == 42)
    tiled = 4 + 28 * k * (1 + rounds(tiles(128, 256)));  // (further rounds: half the first one's and more)
  else
    return -1;
  int best = -1;
  double least = always ? HUGE_VAL : 0.97 * tiled;
  for (int i = 0; i < (int)(sizeof(kMid) / sizeof(kMid[0])); ++i) {
    const MidShape &s = kMid[i];
    const double r = rounds(tiles(16 * s.mt, 16 * s.nt * s.wn));
    const double us = r > 1 ? kMidStart + s.us * k * r * s.rounds : std::min(kMidStart + s.one * k, s.short_start + s.short_us * k);
    if (us < least) best = i, least = us;
  }
  return best;
}

int run_nvfp4_mid(const GemmParams &p, int shape, hipStream_t st) {
  if (shape < 0 || shape >= (int)(sizeof(kMid) / sizeof(kMid[0]))) return ARCQ_ERR_SHAPE;
  const int bm = 16 * kMid[shape].mt, bn = 16 * kMid[shape].nt * kMid[shape].wn;
  if ((long)((p.M + bm - 1) / bm) * ((p.N + bn - 1) / bn) <= 256) switch (shape) {
      case 5: return launch<5, 3, 2, 4, 2, false, 128>(p, st);
      case 6: return launch<4, 4, 2, 4, 2, false, 128>(p, st);
      case 7: return launch<6, 3, 2, 4, 2, false, 128>(p, st);
      case 8: return launch<5, 4, 2, 4, 2, false, 128>(p, st);
      default: break;
    }
  switch (shape) {
    case 0: return launch<4, 3, 1, 8, 2>(p, st);
    case 1: return launch<4, 4, 1, 8, 2>(p, st);
    case 2: return launch<5, 3, 1, 8, 2>(p, st);
    case 3: return launch<6, 4, 1, 8, 2>(p, st);
    case 4: return launch<7, 3, 1, 8, 2>(p, st);
    case 5: return launch<5, 3, 2, 4, 2>(p, st);
    case 6: return launch<4, 4, 2, 4, 2>(p, st);
    case 7: return launch<6, 3, 2, 4, 2>(p, st);
    case 8: return launch<5, 4, 2, 4, 2>(p, st);
    default: return ARCQ_ERR_SHAPE;
  }
}

int run_nvfp4_stream(const GemmParams &p, hipStream_t st) {
  if (p.seg) {
    // Experts of very different sizes in one launch: a workgroup takes at most 48 rows of its expert (64 where the average is
    // above 40) and leaves out the 16-row tiles that it has none for.  Eight experts of 28672 x 4224 with the SwiGLU epilogue and
    // of 4096 x 14464, weights from HBM, us: 2 to 48 rows 139 and 70 (4.0 TB/s; 128x64 tiles: 186 and 101), 16 rows each 124 and
    // 56, 32 rows each 134 and 60, 10 to 250 rows 270 and 150 (307 and 143).
    if (p.M / p.n_seg > 40) return p.N > 8192 ? launch<4, 3, 2, 4, 2, true>(p, st) : launch<4, 4, 2, 4, 2, true>(p, st);
    return p.N > 8192 ? launch<3, 4, 2, 4, 2, true>(p, st) : launch<3, 4, 1, 8, 2, true>(p, st);
  }
  switch ((p.M + 15) / 16) {
    case 1: return launch_plain<1>(p, st);
    case 2: return launch_plain<2>(p, st);
    case 3: return launch_plain<3>(p, st);
    default: return launch_plain<4>(p, st);
  }
}

}  // namespace arcq
