// arcq_gemm_mx.hip -- MXFP4 GEMM for many rows: 256x256 tiles, ping-pong waves, 16x16x128 scaled MFMAs.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "arcq_gemm_tile.h"

namespace arcq {
namespace {

// ---------------------------------------------------------------------------------------------
// 256x256 tile, K in stages of 256.
//
// Eight waves, two per SIMD, in two groups of four: a wave owns 128 rows of the weights (wave >> 2) and 64 of the
// activations (wave & 3).  It alternates between memory phases (operand reads from LDS, requests of later stages) and
// compute phases (32 MFMAs, nothing else); the second group starts one phase late, so that one wave of every SIMD
// multiplies while the other one reads, with a barrier between phases.
//
// What bounds it is the longer of the two phases: 512 cycles of MFMAs, and in the other one what a lone wave can issue, an
// instruction every 5 to 9 cycles.  So a memory phase holds LDS reads and requests and next to nothing else: scale bytes are read a
// stage ahead, two tiles per instruction, and taken apart between the MFMAs, addresses are formed there too, and stages come in
// pairs so that their places in LDS are constants.  (With scale bytes read and taken apart where they are used, and addresses formed
// where the requests are, 30 scalar and 12 vector instructions more: 2048 x 2048 x 14592, 64 workgroups, 84 us, so 69.5, the MFMAs and
// barriers alone 57; 4096 x 4096 x 14592 111 / 102.5, 16384 x 28672 x 4352 1144 / 1066.)
//
// The matrix instruction is 16x16x128: a register-only loop of it sustains 7.0-7.2 PFLOP/s on random codes against 5.8-6.3 for
// 32x32x64 (one and two waves per SIMD, arcq_mfma_rate_probe), the upper figure when the tiles are walked back and forth, so
// that neighbouring instructions share an operand.  4096 x 4096 x 14592, one round of tiles: 102-107 us, 4.6-4.8 PFLOP/s, once the
// clock is up; 110-120 us in the first milliseconds after a pause.
//
// A stage has two phases: all activations with weight rows 0-63 of the wave, then with rows 64-127.  The activations and
// the first half of the weights leave LDS in the first phase, so their buffers are requested again in the second one: two
// stages of LDS (128 KB) hold requests for six phases ahead.  (Stages of 128 elements would do the same in four buffers,
// but a row is then fetched in pieces of 64 bytes: twice the requests to L2.)
//
// LDS rows are 128 bytes of codes = 8 chunks, swizzled as the fp16 tile of the NVFP4 kernel (chunk ^ stage_swizzle(row)), and
// windows of 16 scale bytes for two stages, the last of which ends with the row.  Lanes 16 g .. 16 g + 15 hold K blocks 2 g
// and 2 g + 1 of the stage: their two scale bytes are half of a dword and picked by op_sel.
// Requires K' % 128 == 0, K' >= 512.
// ---------------------------------------------------------------------------------------------
template <bool HALVES>
__global__ __launch_bounds__(512) void gemm_mxfp4_pingpong(GemmParams p) {
  constexpr int BT = 256;
  constexpr int kCodes = 2 * BT * 128, kScales = 2 * 2 * BT * 16;
  constexpr int kRegion = 128 * 64 * 2;
  static_assert(8 * kRegion <= 2 * kCodes, "the epilogue's transpose");
  // weights, activations, scale bytes (512 rows per window; those read behind the last stage may begin 12 bytes past their row)
  __shared__ uint4 smem[(2 * kCodes + kScales) / 16 + 1];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int pos = wave & 3, group = wave >> 2;
  const int kbytes = p.Kp >> 1, ksc = p.Kp >> 5;

  int lin;
  if (p.seg) {
    if (!enter_segment_in_runs<BT, BT, 32>(p, lin)) return;
  } else {
    const int total = ((p.M + BT - 1) / BT) * ((p.N + BT - 1) / BT);
    lin = (blockIdx.x & 7) * ((total + 7) >> 3) + (blockIdx.x >> 3);
    if (lin >= total) return;
  }
  const int tm = (p.M + BT - 1) / BT, tn = (p.N + BT - 1) / BT;
  const int band = lin / (4 * tn), bw = min(4, tm - 4 * band), in_band = lin - band * 4 * tn;
  const int n_base = (in_band / bw) * BT, m_base = (4 * band + in_band % bw) * BT;

  const int ns = (p.Kp + 255) >> 8;                 // stages
  const bool short_last = (p.Kp & 255) != 0;        // the last one then has blocks 4..7 only
  const int nw = (ns + 1) >> 1, s_shift = 16 * nw - ksc;

  // ---- global -> LDS
  uint32_t wvo[4], xvo[4];
  const int ld_row = 8 * wave + (lane >> 3);
  const uint32_t ld_q = (lane & 7) ^ stage_swizzle(ld_row);   // (the swizzle has a period of 16 rows)
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    wvo[i] = (uint32_t)weight_row<128, HALVES>(p, n_base, 64 * i + ld_row) * (uint32_t)kbytes + ld_q * 16;
    xvo[i] = (uint32_t)min(m_base + 64 * i + ld_row, p.M - 1) * (uint32_t)kbytes + ld_q * 16;
  }
  const uint8_t *sbase = group ? p.a_scales : p.b_scales;
  const uint32_t svo = (uint32_t)(group ? min(m_base + 64 * pos + lane, p.M - 1) : weight_row<128, HALVES>(p, n_base, 64 * pos + lane)) * (uint32_t)ksc;
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>(smem);
  // requests behind the last stage fetch it again into buffers that nobody reads any more: the number of loads on their
  // way is the same in every stage.  A short last stage is the row's last 256 elements, the first half of which the stage before it has.
  const int last_at = kbytes - 128;
  auto stage_at = [&](int s) { return min(s * 128, last_at); };
  auto request_x = [&](const uint8_t *x, int odd, int i) { lds_dma16_at(x, xvo[i], lds0 + wave * 1024, kCodes + odd * (BT * 128) + i * 8192); };
  // i even: first phase's rows, odd: second's
  auto request_w = [&](const uint8_t *w, int odd, int i) { lds_dma16_at(w, wvo[i], lds0 + wave * 1024, odd * (BT * 128) + i * 8192); };
  auto window_at = [&](int w) { return min(w * 16, ksc - 16); };  // the last window ends with the row
  auto request_scales = [&](const uint8_t *window, uint32_t at) { lds_dma16_at(window, svo, at, 2 * kCodes); };

  // ---- LDS -> operands
  const int r = lane & 15, g = lane >> 4;
  const uint8_t *lds = reinterpret_cast<const uint8_t *>(smem);
  const uint8_t *w_rd[2], *x_rd[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int c = ((2 * g + h) ^ stage_swizzle(r)) << 4;
    w_rd[h] = lds + (128 * group + r) * 128 + c;
    x_rd[h] = lds + kCodes + (64 * pos + r) * 128 + c;
  }
  const uint32_t ws_rd = 2 * kCodes + (128 * group + r) * 16 + 4 * (g >> 1);
  const uint32_t xs_rd = 2 * kCodes + BT * 16 + (64 * pos + r) * 16 + 4 * (g >> 1);
  const int s_half = 16 * (g & 1);

  uint4 wq[4][2], xq[4][2];
  int wr[8], xr[4];          // scale bytes of a stage as they are in LDS
  int ws[2][4], xs[4];       // and this lane's two of each, by half of the weights
  v4f acc[8][4];
#pragma unroll
  for (auto &a : acc)
#pragma unroll
    for (auto &b : a) b = v4f{0.f, 0.f, 0.f, 0.f};

  auto barrier = [&]() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
  };
  auto scale_offset = [&](int s) {
    return ((s >> 1) & 1) * (2 * BT * 16) + 8 * (s & 1) + ((s >> 1) == nw - 1 ? s_shift : 0) - (short_last && s == ns - 1 ? 4 : 0);
  };
  auto read_w = [&](int odd, int t, int i) {
    wq[i][0] = *reinterpret_cast<const uint4 *>(w_rd[0] + odd * (BT * 128) + t * 2048);
    wq[i][1] = *reinterpret_cast<const uint4 *>(w_rd[1] + odd * (BT * 128) + t * 2048);
  };
  auto read_scales = [&](uint32_t ws_at, uint32_t xs_at, int part) {  // of the activations and of the two halves of the weights: four tiles each
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (part == 0)
        xr[i] = *reinterpret_cast<const int *>(lds + xs_at + i * 256);
      else
        wr[4 * part - 4 + i] = *reinterpret_cast<const int *>(lds + ws_at + (4 * part - 4 + i) * 256);
    }
  };
  // lanes without blocks (g < 2 of a short last stage): both scales 2^-127, so that whatever codes they hold multiply to
  // less than half the smallest number
  auto present = [&](int s) { return short_last && s == ns - 1 && g < 2 ? 0 : 16; };
  auto multiply = [&](auto half_t) {
    constexpr int W0 = decltype(half_t)::value * 4;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int i = j & 1 ? 3 - t : t;
        acc[W0 + i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fp4_operand(wq[i][0]), fp4_operand(xq[j][0]), acc[W0 + i][j],
                                                                         4, 4, 0, ws[W0 >> 2][i], 0, xs[j]);
      }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int i = j & 1 ? 3 - t : t;
        acc[W0 + i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fp4_operand(wq[i][1]), fp4_operand(xq[j][1]), acc[W0 + i][j],
                                                                         4, 4, 1, ws[W0 >> 2][i], 1, xs[j]);
      }
  };

  // in the order of the steady state, so that the same wait counts apply
  request_scales(sbase, lds0 + wave * 1024);
  request_w(p.b_codes, 0, 1);
  request_w(p.b_codes, 0, 3);
#pragma unroll
  for (int i = 0; i < 4; ++i) request_x(p.a_codes, 0, i);
  request_w(p.b_codes, 0, 0);
  request_w(p.b_codes, 0, 2);
  const uint8_t *x_next = p.a_codes + stage_at(1), *w_next = p.b_codes + stage_at(1);  // of the stage requested next
#pragma unroll
  for (int i = 0; i < 4; ++i) request_x(x_next, 1, i);
  request_w(w_next, 1, 0);
  request_w(w_next, 1, 2);
  asm volatile("s_waitcnt vmcnt(6)" ::: "memory");  // stage 0
  barrier();
#pragma unroll
  for (int i = 0; i < 3; ++i) read_scales(ws_rd + scale_offset(0), xs_rd + scale_offset(0), i);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    xs[i] = __builtin_amdgcn_ubfe(xr[i], s_half, 16);
    ws[0][i] = __builtin_amdgcn_ubfe(wr[i], s_half, 16);
  }
  if (group) barrier();  // the second group runs one phase behind

  const uint8_t *scales_next = sbase + window_at(1);   // of the window requested next, and its place
  uint32_t scales_to = lds0 + wave * 1024 + 2 * BT * 16;
  // What a memory phase needs of scalars is formed in the compute phase before it: there they are free.
  auto stage = [&](int s, auto odd_t) {
    constexpr int ODD = decltype(odd_t)::value;
    // first phase: activations and the first half of the weights
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      xq[i][0] = *reinterpret_cast<const uint4 *>(x_rd[0] + ODD * (BT * 128) + i * 2048);
      xq[i][1] = *reinterpret_cast<const uint4 *>(x_rd[1] + ODD * (BT * 128) + i * 2048);
      read_w(ODD, i, i);
      if (i == 0 && !ODD) request_scales(scales_next, scales_to);
      if (i == 1) request_w(w_next, 1 - ODD, 1);
      if (i == 2) request_w(w_next, 1 - ODD, 3);
      __builtin_amdgcn_sched_barrier(0);
    }
    // the second half of this stage's weights has to be there behind this barrier (the counts leave out the scale load of an
    // even stage, which then may be waited for a little early)
    asm volatile("s_waitcnt lgkmcnt(0) vmcnt(8)" ::: "memory");
    barrier();
    multiply(std::integral_constant<int, 0>{});
    const int here = present(s);
    const uint32_t so = scale_offset(s + 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) ws[1][i] = __builtin_amdgcn_ubfe(wr[4 + i], s_half, here);  // the scales of the second half
    x_next = p.a_codes + stage_at(s + 2), w_next = p.b_codes + stage_at(s + 2);
    uint32_t ws_at = ws_rd + so, xs_at = xs_rd + so;
#pragma unroll
    for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(ws[1][i]));
    asm volatile("" : "+s"(x_next), "+s"(w_next), "+v"(ws_at), "+v"(xs_at));
    barrier();
    // second phase: the second half of the weights, and the next stage's scale bytes (behind the last stage: not used)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      read_w(ODD, 4 + i, i);
      if (i < 3) read_scales(ws_at, xs_at, i);
      request_x(x_next, ODD, i);
      if (i & 1) request_w(w_next, ODD, i - 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    // the next stage's activations and first half of the weights
    asm volatile("s_waitcnt lgkmcnt(0) vmcnt(8)" ::: "memory");
    barrier();
    multiply(std::integral_constant<int, 1>{});
    const int next = present(s + 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      ws[0][i] = __builtin_amdgcn_ubfe(wr[i], s_half, next);
      xs[i] = __builtin_amdgcn_ubfe(xr[i], s_half, next);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(ws[0][i]), "+v"(xs[i]));
    if (ODD) {
      scales_next = sbase + window_at((s + 3) >> 1);
      scales_to = lds0 + wave * 1024 + ((s + 3) >> 1 & 1) * (2 * BT * 16);
      asm volatile("" : "+s"(scales_next), "+s"(scales_to));
    }
    barrier();
  };
  int s = 0;
  for (; s + 1 < ns; s += 2) {
    stage(s, std::integral_constant<int, 0>{});
    stage(s + 1, std::integral_constant<int, 1>{});
  }
  if (s < ns) stage(s, std::integral_constant<int, 0>{});
  if (!group) barrier();
  store_wave_tile<HALVES>(p, Acc16<8, 4>{acc}, reinterpret_cast<uint8_t *>(smem) + wave * kRegion, m_base + 64 * pos, n_base + 128 * group, lane);
}

}  // namespace

int run_mxfp4_pingpong(const GemmParams &p, hipStream_t st) {
  const int total = ((p.M + 255) / 256 + (p.seg ? p.n_seg : 0)) * ((p.N + 255) / 256);
  const auto kernel = p.swiglu == kSwigluHalves ? gemm_mxfp4_pingpong<true> : gemm_mxfp4_pingpong<false>;
  hipLaunchKernelGGL(kernel, dim3(p.seg ? grid_in_turn<32>(total) : grid_in_turn<1>(total)), dim3(512), 0, st, p);
  ARCQ_HIP_TRY(hipGetLastError());
  return ARCQ_OK;
}

}  // namespace arcq
