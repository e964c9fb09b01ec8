// arcq_gemm_nv.hip -- NVFP4 GEMM for many rows: one operand decoded to fp16 ahead, the other one inside the kernel.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "arcq_gemm_tile.h"

namespace arcq {
namespace {

// codes + scale bytes -> fp16 values, row-major [rows, K'] (exact: at most six significant bits).  Codes, scale bytes and
// values are dense, so that row boundaries play no part: dword i holds codes 8i .. 8i+7, all of block i / 2.
__global__ __launch_bounds__(256) void nvfp4_decode_f16_kernel(const uint32_t *codes, const uint8_t *scales, uint4 *out,
                                                               size_t dwords) {
  constexpr int U = 4;
  const size_t base = (size_t)blockIdx.x * (256 * U) + threadIdx.x;
  uint32_t c[U], s[U];
#pragma unroll
  for (int k = 0; k < U; ++k) {
    const size_t i = base + 256 * k;
    c[k] = i < dwords ? codes[i] : 0u;
    s[k] = i < dwords ? scales[i >> 1] : 0u;
  }
#pragma unroll
  for (int k = 0; k < U; ++k) {
    const size_t i = base + 256 * k;
    if (i < dwords) out[i] = __builtin_bit_cast(uint4, decode8_nvfp4_f16<false>(c[k], nv_scale_pair_f16(s[k])));
  }
}

// ---------------------------------------------------------------------------------------------
// 256 rows of codes x 256 rows of fp16 per workgroup, K in steps of 64.
//
// Eight waves, two per SIMD, in two groups of four: a wave owns 64 rows of the codes side (wave & 3) and 128 rows of
// the fp16 side (wave >> 2).  A wave alternates between a memory phase (operand reads from LDS for the next 32 elements
// of K, decoding of its codes, requests of later stages) and a compute phase (32 MFMAs, nothing else).  The second
// group starts one phase late, so that at any time one wave of every SIMD multiplies while the other one reads and
// decodes; the barrier between phases keeps them in step.
//
// The matrix instruction is 16x16x32: the chip is power-limited under these kernels, and on decoded FP4 values a
// register-only loop of it sustains 2.1-2.2 PFLOP/s against 1.7-1.8 for 32x32x16 (8 waves per CU, all CUs); walking the
// fp16 tiles back and forth keeps one operand of every other pair of neighbours unchanged (another 5-10 %).
//
// LDS: three stages of the fp16 tile (64 elements of K: rows of 128 bytes), two of the codes (128 elements: rows of 64
// bytes) and of the scale bytes (8 per row).  A stage is requested two steps ahead of its first read by LDS-direct
// loads of all eight waves; chunks of 16 bytes are swizzled on the way (fp16: stage_swizzle, codes: chunk ^
// (row / 4 & 3)) so that the lanes of an operand read, 16 consecutive rows, spread over the banks.
//
// Which element of K a lane feeds to which MFMA is free as long as both operands agree: lanes 16 g .. 16 g + 15 take
// block g of the step, elements 16 g .. 16 g + 7 in the first phase and the other eight in the second, so that a lane's
// codes of a step are eight bytes under one scale byte.
// CODES_W: the weights are the codes side; they always take the MFMA's A slot (a lane then holds four consecutive output
// columns).  Requires K' % 128 == 0, K' >= 256.
// ---------------------------------------------------------------------------------------------
template <bool CODES_W>
__global__ __launch_bounds__(512) void gemm_nvfp4_f16(GemmParams p) {
  constexpr int TF = 8;  // 16-row tiles of the fp16 side per wave
  constexpr int BC = 256, BF = 32 * TF;
  constexpr int BM = CODES_W ? BF : BC, BN = CODES_W ? BC : BF;
  constexpr int FI = BF / 64;                       // fp16 load instructions per wave and step
  constexpr int kF = 3 * BF * 128, kC = 2 * BC * 64, kS = 2 * BC * 8;
  constexpr int kRegion = 64 * 16 * TF * 2;         // bytes per wave of the epilogue's transpose
  static_assert(8 * kRegion <= kF + kC, "the epilogue's transpose");
  __shared__ uint4 smem[(kF + kC + kS) / 16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cpos = wave & 3, group = wave >> 2;
  const int kbytes = p.Kp >> 1, ksc = p.Kp >> 4, fbytes = p.Kp << 1;

  int lin;
  if (p.seg) {
    if (!enter_segment<BM, BN, 16>(p, lin)) return;
  } else {
    const int total = ((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN);
    lin = (blockIdx.x & 7) * ((total + 7) >> 3) + (blockIdx.x >> 3);
    if (lin >= total) return;
  }
  const int rows_c = CODES_W ? p.N : p.M, rows_f = CODES_W ? p.M : p.N;
  const uint8_t *codes = CODES_W ? p.b_codes : p.a_codes, *scales = CODES_W ? p.b_scales : p.a_scales;
  // An XCD's 32 workgroups run at the same time on consecutive tiles: 4 tiles of the fp16 side x 8 of the codes, so that
  // both operands are shared in its L2 (an fp16 tile is four times the bytes of a codes tile)
  const int tc = (rows_c + BC - 1) / BC, tf = (rows_f + BF - 1) / BF;
  const int band = lin / (4 * tc), bw = min(4, tf - 4 * band), in_band = lin - band * 4 * tc;
  const int c_base = (in_band / bw) * BC, f_base = (4 * band + in_band % bw) * BF;

  const int nk = p.Kp >> 6;  // even

  // ---- global -> LDS: a wave-uniform base plus a 32-bit byte offset per lane
  uint32_t fvo[FI], cvo[2], svo;
#pragma unroll
  for (int i = 0; i < FI; ++i) {
    const int row = 64 * i + 8 * wave + (lane >> 3);
    fvo[i] = (uint32_t)min(f_base + row, rows_f - 1) * (uint32_t)fbytes + (((lane & 7) ^ stage_swizzle(row)) << 4);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = 128 * i + 16 * wave + (lane >> 2);
    cvo[i] = (uint32_t)min(c_base + row, rows_c - 1) * (uint32_t)kbytes + (((lane & 3) ^ ((row >> 2) & 3)) << 4);
  }
  svo = (uint32_t)min(c_base + 64 * cpos + lane, rows_c - 1) * (uint32_t)ksc + 4 * group;
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>(smem);
  const uint8_t *f16 = reinterpret_cast<const uint8_t *>(p.f16);
  // (requests behind the last step fetch it again, into stages that nobody reads any more: the number of loads on their
  // way is the same in every step)
  auto request_f = [&](int u, int st, int i) {
    lds_dma16_at(f16 + (size_t)min(u, nk - 1) * 128, fvo[i], lds0 + st * (BF * 128) + i * 8192 + wave * 1024);
  };
  auto request_c = [&](int j, int i) {  // codes (i = 0, 1) and scale bytes (2) of steps 2j, 2j + 1
    const int jf = min(j, (nk >> 1) - 1);
    if (i < 2)
      lds_dma16_at(codes + (size_t)jf * 64, cvo[i], lds0 + kF + (j & 1) * (BC * 64) + i * 8192 + wave * 1024);
    else
      lds_dma4_at(scales + (size_t)jf * 8, svo, lds0 + kF + kC + (j & 1) * (BC * 8) + group * (BC * 4) + cpos * 256);
  };

  // ---- LDS -> operands
  const int r = lane & 15, g = lane >> 4;
  const uint8_t *lds = reinterpret_cast<const uint8_t *>(smem);
  const int f_row = 16 * TF * group + r, c_row = 64 * cpos + r;
  const uint8_t *f_rd[2] = {lds + f_row * 128 + (((2 * g) ^ stage_swizzle(r)) << 4),
                            lds + f_row * 128 + (((2 * g + 1) ^ stage_swizzle(r)) << 4)};
  const uint8_t *c_rd[2] = {lds + kF + c_row * 64 + (((g >> 1) ^ ((r >> 2) & 3)) << 4) + (g & 1) * 8,
                            lds + kF + c_row * 64 + ((((g >> 1) + 2) ^ ((r >> 2) & 3)) << 4) + (g & 1) * 8};
  const uint8_t *s_rd = lds + kF + kC + c_row * 4 + g;

  uint2 cq[2][4];           // codes of an even and of an odd step, eight bytes per 16 rows
  uint32_t sq[2][4];        // their scale byte
  v8h cf[4];                // decoded operands of a phase
  v8h ff[TF];
  v4f acc[CODES_W ? 4 : TF][CODES_W ? TF : 4];
#pragma unroll
  for (auto &a : acc)
#pragma unroll
    for (auto &b : a) b = v4f{0.f, 0.f, 0.f, 0.f};

  auto read_codes = [&](int j, auto odd_t, int i) {  // of step 2j or 2j + 1, 16-row tile i
    constexpr int o = decltype(odd_t)::value ? 1 : 0;
    cq[o][i] = *reinterpret_cast<const uint2 *>(c_rd[o] + (j & 1) * (BC * 64) + i * 1024);
    sq[o][i] = s_rd[(j & 1) * (BC * 8) + o * (BC * 4) + i * 64];
  };
  auto barrier = [&]() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
  };
  auto read_f = [&](int st, int half, int t) {
    ff[t] = __builtin_bit_cast(v8h, *reinterpret_cast<const uint4 *>(f_rd[half] + st * (BF * 128) + t * 2048));
  };
  auto decode = [&](int half, auto odd_t, int i) {
    constexpr int o = decltype(odd_t)::value ? 1 : 0;
    if (half == 0) sq[o][i] = (sq[o][i] << 7) + 0x1800u;  // scale byte -> fp16
    cf[i] = decode8_nvfp4_f16<false>(half ? cq[o][i].y : cq[o][i].x, sq[o][i]);
    asm volatile("" : "+v"(cf[i]));  // here, not behind the barrier
  };
  auto multiply = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int s = 0; s < TF; ++s) {
        const int t = i & 1 ? TF - 1 - s : s;
        if constexpr (CODES_W)
          acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(cf[i], ff[t], acc[i][t], 0, 0, 0);
        else
          acc[t][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ff[t], cf[i], acc[t][i], 0, 0, 0);
      }
  };

#pragma unroll
  for (int i = 0; i < 3; ++i) request_c(0, i);
#pragma unroll
  for (int i = 0; i < FI; ++i) request_f(0, 0, i);
#pragma unroll
  for (int i = 0; i < 3; ++i) request_c(1, i);
#pragma unroll
  for (int i = 0; i < FI; ++i) request_f(1, 1, i);
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(FI + 3) : "memory");  // codes 0 and fp16 stage 0 of this wave
  barrier();
#pragma unroll
  for (int i = 0; i < 4; ++i) read_codes(0, std::false_type{}, i);
  if (group) barrier();  // the second group runs one phase behind

  int st = 0, st2 = 2;   // stages of step u and u + 2
  auto step = [&](int u, auto odd_t) {
    constexpr bool ODD = decltype(odd_t)::value;
    // A memory phase goes tile by tile: LDS reads, decoding and requests take turns, so that none of the three queues
    // holds the other two up.
    // first phase
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int t = i * TF / 4; t < (i + 1) * TF / 4; ++t) read_f(st, 0, t);
      decode(0, odd_t, i);
      if (i < FI / 2) request_f(u + 2, st2, i);  // its stage was last read in step u - 1
      __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    barrier();
    multiply();
    barrier();
    // second phase; the codes read are the next step's (behind the last one: not used)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int t = i * TF / 4; t < (i + 1) * TF / 4; ++t) read_f(st, 1, t);
      read_codes((u + 1) >> 1, std::integral_constant<bool, !ODD>{}, i);
      decode(1, odd_t, i);
      if (i < FI / 2) request_f(u + 2, st2, FI / 2 + i);
      if (ODD && i > 0) request_c((u + 3) >> 1, i - 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    // the next step's fp16 stage (and everything older) has to be there behind this barrier; what this step has
    // requested may stay on its way
    asm volatile("s_waitcnt lgkmcnt(0) vmcnt(%0)" : : "n"(ODD ? FI + 3 : FI) : "memory");
    barrier();
    multiply();
    barrier();
    st = st == 2 ? 0 : st + 1;
    st2 = st2 == 2 ? 0 : st2 + 1;
  };
  for (int u = 0; u < nk; u += 2) {
    step(u, std::false_type{});
    step(u + 1, std::true_type{});
  }
  if (!group) barrier();

  const bool whole = c_base + BC <= rows_c && f_base + BF <= rows_f;
  uint8_t *region = reinterpret_cast<uint8_t *>(smem) + wave * kRegion;
  if constexpr (CODES_W)
    store_wave_tile(p, Acc16<4, TF>{acc}, region, f_base + 16 * TF * group, c_base + 64 * cpos, whole, lane);
  else
    store_wave_tile(p, Acc16<TF, 4>{acc}, region, c_base + 64 * cpos, f_base + 16 * TF * group, whole, lane);
}

template <bool CODES_W>
int launch(const GemmParams &p, hipStream_t st) {
  const int total = ((p.M + 255) / 256 + (p.seg ? p.n_seg : 0)) * ((p.N + 255) / 256);
  hipLaunchKernelGGL((gemm_nvfp4_f16<CODES_W>), dim3(((total + 7) / 8) * 8), dim3(512), 0, st, p);
  ARCQ_HIP_TRY(hipGetLastError());
  return ARCQ_OK;
}

}  // namespace

size_t nvfp4_f16_bytes(int M, int N, int Kp, bool grouped) {
  return (size_t)(grouped || M <= N ? M : N) * Kp * 2;
}

int run_nvfp4_f16(GemmParams p, void *workspace, hipStream_t st) {
  const bool codes_w = p.seg || p.M <= p.N;
  const int rows = codes_w ? p.M : p.N;
  const size_t dwords = (size_t)rows * (p.Kp >> 3);
  hipLaunchKernelGGL(nvfp4_decode_f16_kernel, dim3((unsigned)((dwords + 1023) / 1024)), dim3(256), 0, st,
                     reinterpret_cast<const uint32_t *>(codes_w ? p.a_codes : p.b_codes), codes_w ? p.a_scales : p.b_scales,
                     static_cast<uint4 *>(workspace), dwords);
  ARCQ_HIP_TRY(hipGetLastError());
  p.f16 = static_cast<const uint16_t *>(workspace);
  return codes_w ? launch<true>(p, st) : launch<false>(p, st);
}

}  // namespace arcq
