// arcq_gemm_nv.hip -- NVFP4 GEMM for many rows: one operand decoded to fp16 ahead, the other one inside the kernel.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "arcq_gemm_tile.h"

namespace arcq {
namespace {

// When the last round of tiles is cut along K: behind at least one whole round, and where the CUs without a tile times its steps are
// worth more than the sums' way through memory and the second launch (30 to 35 us; what is left idle is not all lost, the
// others run at a higher clock).  NVFP4, us, uncut and cut: 3000 x 6144 x 10240 (288 tiles) 391 and 292, 6000 x 4096 x 14592 (384) 560
// and 512; 2331 x 4096 x 14592 (160, no whole round) 260 and 292, 2048 x 4096 x 8320 (128) 116 and 122.
__host__ __device__ inline bool last_round_cut(long tiles, int pairs) {
  const int rest = (int)(tiles & 255);
  return tiles > 256 && rest > 0 && (256 - rest) * pairs > 6500;
}
constexpr int kSplitPairs = 12;   // pairs of steps that a workgroup has at least, about

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
// 256 rows of codes x 32 TF rows of fp16 per workgroup (TF = 8, 6, 4 or 2), K in steps of 64.
//
// Eight waves, two per SIMD, in two groups of four: a wave owns 64 rows of the codes side (wave & 3) and 16 TF rows of
// the fp16 side (wave >> 2).  A wave alternates between a memory phase (operand reads from LDS for the next 32 elements
// of K, requests of later stages) and a compute phase (4 TF MFMAs, and between them the decoding of its codes for the next
// phase).  The second group starts one phase late, so that at any time one wave of every SIMD multiplies while the other one
// reads; the barrier between phases keeps them in step.
//
// What bounds it is the longer of the two phases: 512 cycles of MFMAs (TF = 8), and in the other one what a lone wave can issue, an
// instruction every 5 to 9 cycles.  Decoding in the memory phase (32 instructions) made that 63 to 84 instructions long, and the phase
// of an odd step that also requests codes and scale bytes the longest of all; so the decoding goes between the MFMAs, which leave
// room for one VALU instruction each, and the requests are spread (4 of 8 KB or less per phase at most).  us, decoding and the requests of
// codes in the memory phases, and so: 2331 x 3584 x 19072 with TF = 6 316 and 262; 2048 x 2048 x 14592 with TF = 8 266 and 244
// (its MFMAs and barriers alone: 216), 16384 x 28672 x 4352 2715 and 2645, where all CUs are busy and the clock gives way.  Neither more
// stages on their way nor lines fetched into L2 ahead nor requests between the MFMAs, fewer barriers or raised wave
// priority are faster.
//
// The matrix instruction is 16x16x32: the chip is power-limited under these kernels, and on decoded FP4 values a
// register-only loop of it sustains 2.00 PFLOP/s against 1.83 for 32x32x16 (two waves per SIMD, all CUs), 2.08 when the fp16
// tiles are walked back and forth, which keeps one operand of neighbours unchanged at the turns too (arcq_mfma_rate_probe).
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
template <bool CODES_W, int TF_ = 8>
struct F16Shape {
  static constexpr int TF = TF_;  // 16-row tiles of the fp16 side per wave
  static constexpr int BC = 256, BF = 32 * TF;
  static constexpr int BM = CODES_W ? BF : BC, BN = CODES_W ? BC : BF;
  static constexpr int FI = BF / 64, FA = (FI + 1) / 2;    // fp16 load instructions per wave and step, and in its first phase
  static constexpr int kF = 3 * BF * 128, kC = 2 * BC * 64, kS = 2 * BC * 8;
  static constexpr int kRegion = 64 * 16 * TF * 2;         // bytes per wave of the epilogue's transpose
  static_assert(8 * kRegion <= kF + kC, "the epilogue's transpose");
  static constexpr int kQuads = 4 * TF;                    // accumulator quads of a lane
  static constexpr size_t kSlot = (size_t)512 * kQuads;    // of a workgroup, where its sums leave as they are
};

// Rows of either side where tile lin begins.
// An XCD's 32 workgroups run at the same time on consecutive tiles: 4 tiles of the fp16 side x 8 of the codes, so that
// both operands are shared in its L2 (an fp16 tile is four times the bytes of a codes tile)
template <bool CODES_W, int TF>
__device__ __forceinline__ void f16_tile_at(const GemmParams &p, int lin, int &c_base, int &f_base) {
  using S = F16Shape<CODES_W, TF>;
  const int rows_c = CODES_W ? p.N : p.M, rows_f = CODES_W ? p.M : p.N;
  const int tc = (rows_c + S::BC - 1) / S::BC, tf = (rows_f + S::BF - 1) / S::BF;
  const int band = lin / (4 * tc), bw = min(4, tf - 4 * band), in_band = lin - band * 4 * tc;
  c_base = (in_band / bw) * S::BC, f_base = (4 * band + in_band % bw) * S::BF;
}

// The tile at (c_base, f_base), nk steps of 64 elements from step u0 on (both even): the tile of C, or with `partial` the fp32 sums.
template <bool CODES_W, int TF, bool HALVES>
__device__ __forceinline__ void f16_tile_of(const GemmParams &p, int c_base, int f_base, int u0, int nk, float4 *partial, uint8_t *smem, int tid) {
  using S = F16Shape<CODES_W, TF>;
  constexpr int BC = S::BC, BF = S::BF, FI = S::FI, FA = S::FA, kF = S::kF, kC = S::kC, kRegion = S::kRegion;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cpos = wave & 3, group = wave >> 2;
  const int kbytes = p.Kp >> 1, ksc = p.Kp >> 4, fbytes = p.Kp << 1;
  const int rows_c = CODES_W ? p.N : p.M, rows_f = CODES_W ? p.M : p.N;
  const uint8_t *codes = (CODES_W ? p.b_codes : p.a_codes) + u0 * 32, *scales = (CODES_W ? p.b_scales : p.a_scales) + u0 * 4;

  // ---- global -> LDS: a wave-uniform base plus a 32-bit byte offset per lane
  uint32_t fvo[FI], cvo[2], svo;
#pragma unroll
  for (int i = 0; i < FI; ++i) {
    const int row = 64 * i + 8 * wave + (lane >> 3);
    fvo[i] = (uint32_t)(CODES_W ? min(f_base + row, rows_f - 1) : weight_row<16 * TF, HALVES>(p, f_base, row)) * (uint32_t)fbytes + (((lane & 7) ^ stage_swizzle(row)) << 4);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = 128 * i + 16 * wave + (lane >> 2);
    cvo[i] = (uint32_t)(CODES_W ? weight_row<64, HALVES>(p, c_base, row) : min(c_base + row, rows_c - 1)) * (uint32_t)kbytes + (((lane & 3) ^ ((row >> 2) & 3)) << 4);
  }
  svo = (uint32_t)(CODES_W ? weight_row<64, HALVES>(p, c_base, 64 * cpos + lane) : min(c_base + 64 * cpos + lane, rows_c - 1)) * (uint32_t)ksc + 4 * group;
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>(smem);
  const uint8_t *f16 = reinterpret_cast<const uint8_t *>(p.f16) + (size_t)u0 * 128;
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

  uint2 cq[4];              // codes of a step, eight bytes per 16 rows
  uint32_t sq[4];           // their scale byte
  v8h cf[2][4];             // decoded operands of either phase
  v8h ff[TF];
  v4f acc[CODES_W ? 4 : TF][CODES_W ? TF : 4];
#pragma unroll
  for (auto &a : acc)
#pragma unroll
    for (auto &b : a) b = v4f{0.f, 0.f, 0.f, 0.f};

  auto read_codes = [&](int j, auto odd_t, int i) {  // of step 2j or 2j + 1, 16-row tile i
    constexpr int o = decltype(odd_t)::value ? 1 : 0;
    cq[i] = *reinterpret_cast<const uint2 *>(c_rd[o] + (j & 1) * (BC * 64) + i * 1024);
    sq[i] = s_rd[(j & 1) * (BC * 8) + o * (BC * 4) + i * 64];
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
  auto decode = [&](int half, int i) {
    if (half == 0) sq[i] = (sq[i] << 7) + 0x1800u;  // scale byte -> fp16
    cf[half][i] = decode8_nvfp4_f16<false>(half ? cq[i].y : cq[i].x, sq[i]);
  };
  // the products of a phase, and between them the decoding of the next phase's codes (the last step's: of codes that nobody uses)
  auto multiply = [&](auto half_t) {
    constexpr int h = decltype(half_t)::value;
#pragma unroll
    for (int i = 0; i < 4; ++i) decode(1 - h, i);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int s = 0; s < TF; ++s) {
        const int t = i & 1 ? TF - 1 - s : s;
        if constexpr (CODES_W)
          acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(cf[h][i], ff[t], acc[i][t], 0, 0, 0);
        else
          acc[t][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ff[t], cf[h][i], acc[t][i], 0, 0, 0);
      }
#pragma unroll
    for (int k = 0; k < 4 * TF; ++k) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, (8 + TF - 1) / TF, 0);
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
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int i = 0; i < 4; ++i) decode(0, i);
  if (group) barrier();  // the second group runs one phase behind

  int st = 0, st2 = 2;   // stages of step u and u + 2
  auto step = [&](int u, auto odd_t) {
    constexpr bool ODD = decltype(odd_t)::value;
    // A memory phase goes tile by tile: LDS reads and requests take turns, so that neither queue holds the other up.
    // first phase; the stage of the codes requested here was last read in step u - 1
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int t = i * TF / 4; t < (i + 1) * TF / 4; ++t) read_f(st, 0, t);
      if (i < FA) request_f(u + 2, st2, i);  // its stage was last read in step u - 1
      if (ODD && (i == 2 || i == 3)) request_c((u + 3) >> 1, i - 2);
      __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    barrier();
    multiply(std::integral_constant<int, 0>{});
    barrier();
    // second phase; the codes read are the next step's (behind the last one: not used)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int t = i * TF / 4; t < (i + 1) * TF / 4; ++t) read_f(st, 1, t);
      read_codes((u + 1) >> 1, std::integral_constant<bool, !ODD>{}, i);
      if (i < FI - FA) request_f(u + 2, st2, FA + i);
      if (ODD && i == 3) request_c((u + 3) >> 1, 2);
      __builtin_amdgcn_sched_barrier(0);
    }
    // the next step's fp16 stage (and everything older) has to be there behind this barrier; what this step has
    // requested may stay on its way
    asm volatile("s_waitcnt lgkmcnt(0) vmcnt(%0)" : : "n"(ODD ? FI + 3 : FI) : "memory");
    barrier();
    multiply(std::integral_constant<int, 1>{});
    barrier();
    st = st == 2 ? 0 : st + 1;
    st2 = st2 == 2 ? 0 : st2 + 1;
  };
  for (int u = 0; u < nk; u += 2) {
    step(u, std::false_type{});
    step(u + 1, std::true_type{});
  }
  if (!group) barrier();

  if (partial) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int t = 0; t < TF; ++t) {
        const v4f a = CODES_W ? acc[i][t] : acc[t][i];
        partial[(wave * S::kQuads + i * TF + t) * 64 + lane] = make_float4(a[0], a[1], a[2], a[3]);
      }
    return;
  }
  uint8_t *region = smem + wave * kRegion;
  if constexpr (CODES_W)
    store_wave_tile<HALVES>(p, Acc16<4, TF>{acc}, region, f_base + 16 * TF * group, c_base + 64 * cpos, lane);
  else
    store_wave_tile<HALVES>(p, Acc16<TF, 4>{acc}, region, c_base + 64 * cpos, f_base + 16 * TF * group, lane);
}

// The last rows of a problem or of an expert's: a tile of fewer fp16 rows, whose phases are shorter (the sums are the same).  Zipf-like
// experts, 8192 rows over eight of 28672 x 4224 with the SwiGLU epilogue: 1616 us with whole tiles alone, 1595 so; 333 x 28672 x 4352:
// 96 and 85.
template <bool CODES_W, int TF, bool HALVES, bool SMALL>
__device__ __forceinline__ void f16_tile(const GemmParams &p, int lin, int u0, int nk, float4 *partial, uint8_t *smem, int tid) {
  int c_base, f_base;
  f16_tile_at<CODES_W, TF>(p, lin, c_base, f_base);
  if constexpr (CODES_W && SMALL) {
    const int left = p.M - f_base;
    if (TF > 2 && left <= 64) return f16_tile_of<CODES_W, 2, HALVES>(p, c_base, f_base, u0, nk, partial, smem, tid);
    if (TF > 4 && left <= 128) return f16_tile_of<CODES_W, 4, HALVES>(p, c_base, f_base, u0, nk, partial, smem, tid);
    if (TF > 6 && left <= 192) return f16_tile_of<CODES_W, 6, HALVES>(p, c_base, f_base, u0, nk, partial, smem, tid);
  }
  f16_tile_of<CODES_W, TF, HALVES>(p, c_base, f_base, u0, nk, partial, smem, tid);
}

// HALVES, and SMALL (a problem with rows for a smaller last tile, or experts, which may have some): what a launch does not need is not in its
// kernel, 39 KB of code for 256 rows with neither, against 177 KB with every epilogue and height in one.  us, that one and so: 2048 x 16384 x 512 44.1,
// 43.0, 4096 x 16384 x 640 90.8, 88.7, 640 x 28672 x 1152 48.2, 47.7.
template <bool CODES_W, int TF, bool HALVES, bool SMALL>
__global__ __launch_bounds__(512) void gemm_nvfp4_f16(GemmParams p) {
  using S = F16Shape<CODES_W, TF>;
  __shared__ uint4 smem[(S::kF + S::kC + S::kS) / 16];
  int lin;
  if (p.seg) {
    if (!enter_segment_in_runs<S::BM, S::BN, 16>(p, lin)) return;
  } else {
    const int total = ((p.M + S::BM - 1) / S::BM) * ((p.N + S::BN - 1) / S::BN);
    lin = (blockIdx.x & 7) * ((total + 7) >> 3) + (blockIdx.x >> 3);
    if (lin >= total) return;
  }
  f16_tile<CODES_W, TF, HALVES, SMALL>(p, lin, 0, p.Kp >> 6, nullptr, reinterpret_cast<uint8_t *>(smem), threadIdx.x);
}

// ---------------------------------------------------------------------------------------------
// The same with its last round of tiles cut along K.  A round takes its time however few tiles it has, and with a long K that is
// most of what a problem of one or two rounds costs.  The tiles of whole rounds run first, a workgroup each; the steps of
// the other R tiles, one tile's behind the other's, are dealt out evenly to up to 256 workgroups.  A workgroup whose steps end
// inside a tile, or begin there, leaves its fp32 sums in a slot of the workspace (two at most); a second launch adds a tile's up in
// the order of K and stores it.  Every sum has a fixed place: the result does not depend on who is first.
// The split and its edges follow from the number of tiles alone, which grouped launches only know on the device.
// ---------------------------------------------------------------------------------------------
struct LastRound {
  int full, rest, groups;  // tiles of whole rounds, the other ones, workgroups that share those
  int pairs;               // of steps, per tile
  __device__ __forceinline__ LastRound(int total, int Kp) {
    pairs = Kp >> 7;
    full = total & ~255;
    rest = total - full;
    if (!last_round_cut(total, pairs)) full = total, rest = 0;
    groups = min(256, rest * max(1, pairs / kSplitPairs));
  }
  __device__ __forceinline__ int begin(int w) const { return (int)((long)rest * pairs * w / groups); }
  __device__ __forceinline__ int holder(int pair) const {  // the workgroup that has this pair
    int w = (int)((long)pair * groups / ((long)rest * pairs));
    while (begin(w + 1) <= pair) ++w;
    return w;
  }
};

// Tiles of the whole problem; with segments, p becomes the problem of the one that tile lin belongs to and lin its number there.
template <bool CODES_W>
__device__ __forceinline__ int f16_tiles(const GemmParams &p) {
  using S = F16Shape<CODES_W>;
  if (p.seg) return Segments<S::BM, S::BN, 16>(p).total;
  return ((p.M + S::BM - 1) / S::BM) * ((p.N + S::BN - 1) / S::BN);
}
template <bool CODES_W>
__device__ __forceinline__ bool f16_enter(GemmParams &p, int &lin) {
  using S = F16Shape<CODES_W>;
  if (!p.seg) return true;
  Segments<S::BM, S::BN, 16> segments(p);
  return segments.enter(p, lin);
}

template <bool CODES_W, bool HALVES>
__global__ __launch_bounds__(512) void gemm_nvfp4_f16_split(GemmParams p) {
  using S = F16Shape<CODES_W>;
  __shared__ uint4 smem[(S::kF + S::kC + S::kS) / 16];
  const LastRound r(f16_tiles<CODES_W>(p), p.Kp);
  const int full_grid = (r.full + 7) & ~7;
  int at, end, w = -1;  // pairs of steps of the rest; a whole tile of the full rounds: its pairs, as if those were all
  if ((int)blockIdx.x < full_grid) {
    const int lin = (blockIdx.x & 7) * (full_grid >> 3) + (blockIdx.x >> 3);
    if (lin >= r.full) return;
    at = (lin - r.full) * r.pairs;  // negative: in front of the rest
    end = at + r.pairs;
  } else {
    const int id = (int)blockIdx.x - full_grid;
    if (id >= 256) return;
    w = (id & 7) * 32 + (id >> 3);  // neighbours on one XCD
    if (w >= r.groups) return;
    at = r.begin(w);
    end = r.begin(w + 1);
  }
  while (at < end) {
    const int tile = (at + r.full * r.pairs) / r.pairs, first = at - (tile - r.full) * r.pairs, n = min(end - at, r.pairs - first);
    GemmParams q = p;
    int lin = tile;
    if (!f16_enter<CODES_W>(q, lin)) return;
    float4 *partial = n == r.pairs ? nullptr : p.split + (2 * w + (first + n == r.pairs ? 0 : 1)) * S::kSlot;
    wait_dma_and_sync();  // the LDS of the part before this one
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // what follows from it is formed per part: hoisted out of this loop it would be spilled
    f16_tile<CODES_W, 8, HALVES, true>(q, lin, 2 * first, 2 * n, partial, reinterpret_cast<uint8_t *>(smem), tid);
    at += n;
  }
}

// a wave per eighth of a tile
template <bool CODES_W, int TF, bool HALVES>
__device__ __forceinline__ void f16_add_parts(const GemmParams &p, const LastRound &r, int w0, int w1, int c_base, int f_base, uint8_t *region) {
  using S = F16Shape<CODES_W, TF>;
  const int lane = threadIdx.x, wave = blockIdx.x & 7, cpos = wave & 3, group = wave >> 2;
  v4f acc[CODES_W ? 4 : TF][CODES_W ? TF : 4];
#pragma unroll
  for (auto &a : acc)
#pragma unroll
    for (auto &b : a) b = v4f{0.f, 0.f, 0.f, 0.f};
  for (int w = w0; w <= w1; ++w) {
    if (r.begin(w) == r.begin(w + 1)) continue;
    const float4 *src = p.split + (2 * w + (w == w1 ? 0 : 1)) * F16Shape<CODES_W>::kSlot + (size_t)wave * S::kQuads * 64 + lane;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int t = 0; t < TF; ++t) {
        const float4 v = src[(i * TF + t) * 64];
        (CODES_W ? acc[i][t] : acc[t][i]) += v4f{v.x, v.y, v.z, v.w};
      }
  }
  if constexpr (CODES_W)
    store_wave_tile<HALVES>(p, Acc16<4, TF>{acc}, region, f_base + 16 * TF * group, c_base + 64 * cpos, lane);
  else
    store_wave_tile<HALVES>(p, Acc16<TF, 4>{acc}, region, c_base + 64 * cpos, f_base + 16 * TF * group, lane);
}

template <bool CODES_W, bool HALVES>
__global__ __launch_bounds__(64) void f16_split_add_kernel(GemmParams p) {
  using S = F16Shape<CODES_W>;
  __shared__ uint4 smem[S::kRegion / 16];
  const int tile = blockIdx.x >> 3;
  const LastRound r(f16_tiles<CODES_W>(p), p.Kp);
  if (tile >= r.rest) return;
  const int w0 = r.holder(tile * r.pairs), w1 = r.holder((tile + 1) * r.pairs - 1);
  int lin = r.full + tile;
  if (w0 == w1 || !f16_enter<CODES_W>(p, lin)) return;  // (one workgroup had the whole tile and stored it)
  int c_base, f_base;
  f16_tile_at<CODES_W, 8>(p, lin, c_base, f_base);
  uint8_t *region = reinterpret_cast<uint8_t *>(smem);
  if constexpr (CODES_W) {  // as f16_tile
    const int left = p.M - f_base;
    if (left <= 64) return f16_add_parts<CODES_W, 2, HALVES>(p, r, w0, w1, c_base, f_base, region);
    if (left <= 128) return f16_add_parts<CODES_W, 4, HALVES>(p, r, w0, w1, c_base, f_base, region);
    if (left <= 192) return f16_add_parts<CODES_W, 6, HALVES>(p, r, w0, w1, c_base, f_base, region);
  }
  f16_add_parts<CODES_W, 8, HALVES>(p, r, w0, w1, c_base, f_base, region);
}

template <bool CODES_W, int TF, bool HALVES>
int launch_tiles(const GemmParams &p, hipStream_t st) {
  using S = F16Shape<CODES_W, TF>;
  const int total = ((p.M + S::BM - 1) / S::BM + (p.seg ? p.n_seg : 0)) * ((p.N + S::BN - 1) / S::BN), left = p.M % S::BM;
  const bool small = CODES_W && (p.seg || (left > 0 && left <= S::BM - 64));
  const auto kernel = small ? gemm_nvfp4_f16<CODES_W, TF, HALVES, CODES_W> : gemm_nvfp4_f16<CODES_W, TF, HALVES, false>;
  hipLaunchKernelGGL(kernel, dim3(p.seg ? grid_in_turn<32>(total) : grid_in_turn<1>(total)), dim3(512), 0, st, p);
  ARCQ_HIP_TRY(hipGetLastError());
  return ARCQ_OK;
}

template <bool CODES_W, bool HALVES>
int launch_split(const GemmParams &p, hipStream_t st) {
  const int total = ((p.M + 255) / 256 + (p.seg ? p.n_seg : 0)) * ((p.N + 255) / 256);
  const int grid = ((total + 7) / 8) * 8;
  hipLaunchKernelGGL((gemm_nvfp4_f16_split<CODES_W, HALVES>), dim3(grid + 256), dim3(512), 0, st, p);
  ARCQ_HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL((f16_split_add_kernel<CODES_W, HALVES>), dim3(8 * std::min(total, 255)), dim3(64), 0, st, p);
  ARCQ_HIP_TRY(hipGetLastError());
  return ARCQ_OK;
}

// Which operand is decoded ahead, and the tile: the fewest rounds of 256 tiles, a round with 192 rows of activations counting 0.82 of one
// with 256 rows, and with 128 rows 0.70 (a round takes more than its share of rows: codes and their decoding are the same; partly
// empty ones less).  On 400 problems of 65 to 16384 rows, 2048 to 57344 columns and K' = 512 to 8064 that is 0.1 % above the fastest tile
// on average, 6 % at most, and nowhere more than 3 % above 256 rows (with 0.78 and 0.62: 0.4, 11 and 11 %).  us with 256, 192 and 128 rows: 2331
// x 3584 x 3712 71, 62, 99; 1300 x 6144 x 4352 79, 68, 112; 640 x 28672 x 4352 164, 134, 170; 300 x 37888 x 3712 133, 117, 101; 1024 x 28672
// x 4352 184, 213, 229; 4096 x 6144 x 4352 175, 215, 185; 600 x 37888 x 3712 147, 174, 159; 6144 x 28672 x 1152 326, 363, 393.
// The smaller tiles need the activations decoded; decoding a row takes 2.4e-5 of a round (about 5 TB/s, whatever K').
struct F16Plan {
  bool codes_w;
  int tf;
};
F16Plan f16_plan(int M, int N, bool grouped) {
  F16Plan plan{grouped || M <= N, 8};
  if (grouped) return plan;
  auto rounds = [&](long rows) { return (double)(((M + rows - 1) / rows * ((N + 255L) / 256) + 255) / 256); };
  double least = rounds(256) - 2.4e-5 * std::max(0, M - N);
  const struct { int tf; double weight; } smaller[] = {{6, 0.82}, {4, 0.70}};
  for (const auto &s : smaller)
    if (const double cost = rounds(32 * s.tf) * s.weight; cost < least) least = cost, plan = {true, s.tf};
  return plan;
}

}  // namespace

size_t nvfp4_f16_bytes(int M, int N, int Kp, bool grouped) {
  return (size_t)(f16_plan(M, N, grouped).codes_w ? M : N) * Kp * 2;
}

// (Experts: the tiles are known on the device alone; from 512 rows per expert on, and where the most tiles that the rows can make are
// more than a round -- with no more of them nothing is ever cut, and 256x256 tiles leave CUs idle: 4096 x 14464, four experts of 512
// rows 274 us, two 240, the kernels without a workspace 242 and 126.  Eight of 4096 x 14464, 8192 rows skewed 912 -> 825 us against
// 128x128 tiles, even 840 -> 732; 4096 rows skewed 496 -> 464, even (256 tiles: one round) 439 -> 386; 5000 rows skewed 598 -> 552, but
// even (625 rows each, three tiles) 539 -> 564; 64 of 2048 x 8320, 600 rows each, would lose 5 %.)
size_t nvfp4_split_bytes(int M, int N, int Kp, int n_seg) {
  if (Kp < 8192 || Kp % 128 != 0 || M <= 64) return 0;
  if (n_seg == 0) {
    const long total = (long)((M + 255) / 256) * ((N + 255) / 256);
    if (!last_round_cut(total, Kp >> 7) || total > 6 * 256) return 0;
  } else {
    const long tiles_n = (N + 255) / 256, tiles_m = (M + 255) / 256;
    if (N <= 2048 || M / n_seg < 512 || (tiles_m + n_seg) * tiles_n <= 256 || (tiles_m + n_seg / 2) * tiles_n > 6 * 256) return 0;
  }
  return 512 * F16Shape<true>::kSlot * sizeof(float4);
}

size_t nvfp4_split_operand_bytes(int M, int N, int Kp, bool grouped) { return (size_t)(grouped || M <= N ? M : N) * Kp * 2; }

int run_nvfp4_f16(GemmParams p, void *workspace, hipStream_t st, bool split) {
  const F16Plan plan = split ? F16Plan{p.seg || p.M <= p.N, 8} : f16_plan(p.M, p.N, p.seg != nullptr);
  const int rows = plan.codes_w ? p.M : p.N;
  const size_t dwords = (size_t)rows * (p.Kp >> 3);
  hipLaunchKernelGGL(nvfp4_decode_f16_kernel, dim3((unsigned)((dwords + 1023) / 1024)), dim3(256), 0, st,
                     reinterpret_cast<const uint32_t *>(plan.codes_w ? p.a_codes : p.b_codes), plan.codes_w ? p.a_scales : p.b_scales,
                     static_cast<uint4 *>(workspace), dwords);
  ARCQ_HIP_TRY(hipGetLastError());
  p.f16 = static_cast<const uint16_t *>(workspace);
  if (split) p.split = reinterpret_cast<float4 *>(static_cast<uint8_t *>(workspace) + nvfp4_split_operand_bytes(p.M, p.N, p.Kp, p.seg != nullptr));
  auto launch = [&](auto halves) {
    constexpr bool HALVES = decltype(halves)::value;
    if (split) return plan.codes_w ? launch_split<true, HALVES>(p, st) : launch_split<false, HALVES>(p, st);
    if (!plan.codes_w) return launch_tiles<false, 8, HALVES>(p, st);
    return plan.tf == 8 ? launch_tiles<true, 8, HALVES>(p, st) : plan.tf == 6 ? launch_tiles<true, 6, HALVES>(p, st) : launch_tiles<true, 4, HALVES>(p, st);
  };
  return p.swiglu == kSwigluHalves ? launch(std::true_type{}) : launch(std::false_type{});
}

}  // namespace arcq
