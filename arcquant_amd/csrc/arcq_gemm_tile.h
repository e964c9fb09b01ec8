// arcq_gemm_tile.h -- what the GEMM kernels share: the problem, the mapping of workgroups to expert segments, LDS-direct
// loads, NVFP4 decoding to fp16, and the epilogues.
#ifndef ARCQ_GEMM_TILE_H_
#define ARCQ_GEMM_TILE_H_

#include <hip/hip_runtime.h>

#include "arcq_internal.h"
#include "arcq_math.h"
#include "arcq_swiglu.h"

namespace arcq {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

constexpr int kMaxParts = ARCQ_MAX_PARTS;

constexpr int kSwigluPairs = 1, kSwigluHalves = 2;

struct GemmParams {
  const uint8_t *a_codes, *a_scales;  // activations, M rows
  const uint8_t *b_codes, *b_scales;  // weights, N rows
  uint16_t *c;                        // bf16 [M,N]
  const float *d_alpha_a, *d_alpha_b;
  float alpha;
  int M, N, Kp;
  // split-K (tiled kernels): blockIdx.y selects one of k_slices ranges of K steps and the workgroup
  // writes its fp32 partial tile to partial[slice][M][N] instead of C; splitk_reduce_kernel adds them
  float *partial = nullptr;
  int k_slices = 1;
  // optional residual, bf16 [M,N]: C = bf16(bf16(alpha * acc) + residual), what a bf16 add of the
  // rounded GEMM output and the residual gives
  const uint16_t *residual = nullptr;
  int ld_residual = 0;  // elements from one of its rows to the next: N, or 0 for one row that is added to all (a bias)
  // grouped GEMM (tiled kernels): rows seg[e] .. seg[e+1]-1 of A and C belong to segment e, whose weights
  // start seg_b_codes / seg_b_scales bytes after those of segment e-1; d_alpha_a / d_alpha_b are arrays
  // indexed by segment.  A workgroup rewrites its copy of these parameters to its segment's sub-problem.
  const int *seg = nullptr;
  int n_seg = 0;
  size_t seg_b_codes = 0, seg_b_scales = 0;
  // fused SwiGLU epilogue (tiled kernels): the weight rows alternate gate, up, gate, up ..., so that output
  // columns 2j and 2j+1 are gate_j and up_j of one token and sit in one lane; c then is bf16 [M, N/2] and
  // receives act_fn(gate) * up formed from the bf16-rounded GEMM outputs, exactly what the unfused sequence
  // (GEMM, then silu and multiply in bf16) gives.  absmax_bits: NULL, or one word per segment (one word when
  // not grouped) that collects max |output| as the bits of a non-negative float (zeroed by the caller).
  // kSwigluHalves: the first N/2 weight rows are the gates, the others the ups; a tile takes half of its rows from either (weight_row), so
  // that gate_j and up_j are kN / 2 apart in a wave's accumulators (gemm_nvfp4_f16 and gemm_mxfp4_pingpong, plain launches).
  int swiglu = 0;
  uint32_t *absmax_bits = nullptr;
  int seg_index = 0;
  // gemm_nvfp4_f16: one operand decoded to fp16 [rows, K'] ahead of the launch
  const uint16_t *f16 = nullptr;
  // gemm_nvfp4_f16 with its last round of tiles cut along K: the workgroups' fp32 sums of parts of tiles, two slots each
  float4 *split = nullptr;
  // weights made of several parts with a tensor scale each (q | k | v): rows part_end[k - 1] .. part_end[k] - 1 have *part_alpha[k]
  // in the place of *d_alpha_b.  Multiples of 32: a 16- or 32-column tile of accumulators lies in one part.
  int parts = 0;
  int part_end[kMaxParts - 1] = {};
  const float *part_alpha[kMaxParts] = {};
};

// arcq_gemm_nv.hip: bytes of the decoded operand, and the GEMM on it
size_t nvfp4_f16_bytes(int M, int N, int Kp, bool grouped);
int run_nvfp4_f16(GemmParams p, void *workspace, hipStream_t st, bool split);
// scratch of the same with its last round cut along K behind the decoded operand, 0 where that does not pay
size_t nvfp4_split_bytes(int M, int N, int Kp, int n_seg);
size_t nvfp4_split_operand_bytes(int M, int N, int Kp, bool grouped);

// arcq_gemm_nv_stream.hip: decode batches, plain (n_seg = 0, M <= 64) and grouped
bool nvfp4_stream_able(int M, int Kp, int n_seg);
bool nvfp4_stream_wanted(int M, int N, int Kp, int n_seg, bool swiglu);
int run_nvfp4_stream(const GemmParams &p, hipStream_t st);
// 65 to 1024 rows: a shape of the same kernel in the place of the plan's tiles, or -1
int nvfp4_mid_shape(int M, int N, int Kp, int kernel, int slices, bool always);
int run_nvfp4_mid(const GemmParams &p, int shape, hipStream_t st);

// arcq_gemm_mx.hip
int run_mxfp4_pingpong(const GemmParams &p, hipStream_t st);

namespace {

// Inclusive prefix over the lanes of a wave: sum, or maximum of values that are not negative.  (DPP: lanes shifted in from
// outside a row, and rows that a step leaves out, read 0.)
template <bool MAX>
__device__ __forceinline__ int wave_prefix(int v) {
#define ARCQ_PREFIX_STEP(ctrl, rows)                                                  \
  {                                                                                   \
    const int o = __builtin_amdgcn_update_dpp(0, v, ctrl, rows, 0xf, false);          \
    v = MAX ? max(v, o) : v + o;                                                      \
  }
  ARCQ_PREFIX_STEP(0x111, 0xf)  // row_shr:1
  ARCQ_PREFIX_STEP(0x112, 0xf)
  ARCQ_PREFIX_STEP(0x114, 0xf)
  ARCQ_PREFIX_STEP(0x118, 0xf)
  ARCQ_PREFIX_STEP(0x142, 0xa)  // row_bcast:15 into rows 1 and 3
  ARCQ_PREFIX_STEP(0x143, 0xc)  // row_bcast:31 into rows 2 and 3
#undef ARCQ_PREFIX_STEP
  return v;
}

// Grouped launches: maps the workgroup to (segment, tile) and turns p into that segment's problem (M = its
// rows, operand pointers moved to its first row and its weights).  lin: tile number inside the segment, in
// the order the ungrouped kernels use.  The launch holds an upper bound of the tile count; workgroups
// beyond the real count return false.  G: elements per scale byte.
// Every lane reads one offset, 64 segments at a time: a walk from segment to segment is a chain of dependent scalar loads in
// front of every tile (MXFP4, 64 experts of 2048 x 1536, 256 skewed rows each: 78 us with one walk, 104 with another one to count
// the tiles, 68 so; NVFP4, 1024 rows: 457, 470, 426).
template <int BM, int BN, int G>
struct Segments {
  int tiles_n, rows, lane, first;
  int end, beg, tiles, upto;  // of segment e0 + lane: its rows, its tiles, the tiles up to its end
  int total;                  // tiles of all segments

  __device__ __forceinline__ void read(const GemmParams &p, int e0, int from) {
    const int e = e0 + lane;
    // offsets that do not grow or leave the tensor: empty segments
    end = min(wave_prefix<true>(max(e < p.n_seg ? p.seg[e + 1] : 0, from)), rows);
    beg = __shfl_up(end, 1);
    if (lane == 0) beg = from;
    tiles = ((end - beg + BM - 1) / BM) * tiles_n;
    upto = wave_prefix<false>(tiles);
  }

  __device__ __forceinline__ explicit Segments(const GemmParams &p) {
    tiles_n = (p.N + BN - 1) / BN;
    rows = p.M, lane = threadIdx.x & 63;
    first = min(max(p.seg[0], 0), rows);
    total = 0;
    for (int e0 = 0, from = first; e0 < p.n_seg; e0 += 64) {
      read(p, e0, from);
      total += __builtin_amdgcn_readlane(upto, 63);
      from = __builtin_amdgcn_readlane(end, 63);
    }
  }

  // (up to 64 segments) much the same rows in each: one 16-row tile of an MFMA at most, or no more than one and a half times the average
  __device__ __forceinline__ bool even(int n_seg) const {
    const int most = __builtin_amdgcn_readlane(wave_prefix<true>(end - beg), 63);
    return most <= 16 || 2l * most * n_seg <= 3l * (__builtin_amdgcn_readlane(end, 63) - first);
  }

  // Turns p into the problem of the segment that tile lin belongs to, lin into the tile's number inside it; false past the end.
  // (Up to 64 segments the constructor's one read still holds; beyond, p is read anew, so it has to be the launch's own.)
  __device__ __forceinline__ bool enter(GemmParams &p, int &lin) {
    if (lin >= total) return false;
    int e0 = 0;
    if (p.n_seg > 64) {
      for (int from = first; e0 < p.n_seg; e0 += 64) {
        read(p, e0, from);
        const int here = __builtin_amdgcn_readlane(upto, 63);
        if (lin < here) break;
        lin -= here;
        from = __builtin_amdgcn_readlane(end, 63);
      }
      if (e0 >= p.n_seg) return false;
    }
    const int l = __builtin_ctzll(__builtin_amdgcn_ballot_w64(lin < upto));  // the first segment that ends behind lin
    lin -= __builtin_amdgcn_readlane(upto, l) - __builtin_amdgcn_readlane(tiles, l);
    const int row0 = __builtin_amdgcn_readlane(beg, l), e = e0 + l;
    const size_t kbytes = p.Kp >> 1, ksc = p.Kp / G;
    p.a_codes += (size_t)row0 * kbytes;
    p.a_scales += (size_t)row0 * ksc;
    if (p.f16) p.f16 += (size_t)row0 * p.Kp;
    p.c += (size_t)row0 * (p.swiglu ? p.N >> 1 : p.N);
    if (p.residual) p.residual += (size_t)row0 * p.ld_residual;
    p.b_codes += (size_t)e * p.seg_b_codes;
    p.b_scales += (size_t)e * p.seg_b_scales;
    if (p.d_alpha_a) p.d_alpha_a += e;
    if (p.d_alpha_b) p.d_alpha_b += e;
    p.M = __builtin_amdgcn_readlane(end, l) - row0;
    p.seg_index = e;
    return true;
  }
};

template <int BM, int BN, int G>
__device__ __forceinline__ bool enter_segment(GemmParams &p, int &lin) {
  Segments<BM, BN, G> segments(p);
  // contiguous runs of tiles per XCD, of the tiles that there are: cut from the upper bound, the last XCD would get the
  // surplus workgroups and the others its tiles (8192 rows over 8 experts: 36 of 40 rows of tiles are real)
  const int per_xcd = (segments.total + 7) >> 3;
  if ((int)(blockIdx.x >> 3) >= per_xcd) return false;
  lin = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  return segments.enter(p, lin);
}

// The same in shorter runs that go to the XCDs in turn, for kernels whose tiles take less time for fewer rows: with one run per XCD,
// the XCD that has the experts of most rows, or none of those that end in a small tile, is the last one.  The grid is a multiple of
// 8 RUN (grid_in_turn).
template <int RUN>
inline int grid_in_turn(int tiles) { return (tiles + 8 * RUN - 1) / (8 * RUN) * (8 * RUN); }

// Large tiles: runs of at most 32 tiles, as many for every XCD and all of one length (whole runs of 32 for some XCDs and none for
// others: 2048 even rows over eight of 4096 x 14464, 128 tiles, 135 us, so 129).  More than 32 experts keep one run per XCD: a shorter run
// ends inside an expert, whose operands another XCD's L2 then fetches again, as often as it evens anything out.  us, one run per XCD, runs of 32
// wherever they end, and runs of one length, each for even sizes, Zipf-like ones and those in reverse: gemm_nvfp4_f16, 8192 rows over eight of
// 14336 x 4224 672, 733, 735 / 668, 723, 736 / 670, 712, 724, 20800 over 16 of 6144 x 4224 864, 840, 838 / 870, 833, 824 / 858, 803, 820, 83200 over 64
// of 2816 x 2176 969, 881, 909 / 998, 916, 933 / 1001, 893, 884; gemm_mxfp4_pingpong, 2048 over eight of 4096 x 14464 130, 130, 128 / 135, 129, 134 /
// 129, 130, 128, 8192 241, 343, 336 / 247, 328, 322 / 245, 331, 298, 24576 over 16 of 2048 x 14464 382, 458, 451 / 374, 455, 430 / 375, 435, 418.
template <int BM, int BN, int G>
__device__ __forceinline__ bool enter_segment_in_runs(GemmParams &p, int &lin) {
  constexpr int kMost = 32;
  Segments<BM, BN, G> segments(p);
  if (segments.total == 0) return false;
  const int runs = p.n_seg > 32 ? 1 : (segments.total + 8 * kMost - 1) / (8 * kMost);  // of an XCD
  const int run = (segments.total + 8 * runs - 1) / (8 * runs), of_xcd = blockIdx.x >> 3;
  lin = (of_xcd / run * 8 + (blockIdx.x & 7)) * run + of_xcd % run;  // (of_xcd >= run * runs: behind the last tile)
  return segments.enter(p, lin);
}

// Small tiles: in twos (those of an expert's first and second rows, which share their weights).  A few narrow experts with a long K' and much
// the same rows keep one run per XCD, which then has an expert or two and their activations to itself.  us, one run per XCD, in twos, and so, even
// sizes, Zipf-like ones, those in reverse and top-2 of skewed scores: 128 rows over eight of 28672 x 4224 118, 129, 129, 139 / 117, 123, 126, 120, of 4096 x
// 14464 55.2, 84.1, 84.3, 68.7 / 55.8, 82.2, 92.2, 57.3 / 55.3, 82.3, 92.1, 57.5, of 8192 x 14464 99.6, 132, 132, 134 / 109, 127, 145, 113 / 99.9, 127, 146, 114.
// (Sizes that grow from expert to expert are the ones that lose: their longest tiles come last.  With the experts sorted, 7 to 10 % are lost on
// 16 even ones, whose XCDs then share all of them.)
template <int BM, int BN, int G>
__device__ __forceinline__ bool enter_segment_in_twos(GemmParams &p, int &lin) {
  Segments<BM, BN, G> segments(p);
  const int of_xcd = blockIdx.x >> 3, xcd = blockIdx.x & 7;
  if (p.Kp >= 8192 && p.N <= 8192 && p.n_seg <= 16 && segments.even(p.n_seg)) {
    const int per_xcd = (segments.total + 7) >> 3;
    if (of_xcd >= per_xcd) return false;
    lin = xcd * per_xcd + of_xcd;
  } else {
    lin = (of_xcd / 2 * 8 + xcd) * 2 + of_xcd % 2;
  }
  return segments.enter(p, lin);
}

// two bf16 pairs + two bf16 pairs, each sum rounded to bf16
__device__ __forceinline__ uint32_t add_bf16_pair(uint32_t a, uint32_t b) {
  return pack_bf16_rne(u2f(a << 16) + u2f(b << 16), u2f(a & 0xffff0000u) + u2f(b & 0xffff0000u));
}
__device__ __forceinline__ uint2 add_bf16_x4(uint2 a, uint2 b) {
  return make_uint2(add_bf16_pair(a.x, b.x), add_bf16_pair(a.y, b.y));
}

__device__ __forceinline__ float effective_alpha(const GemmParams &p) {
  float a = p.alpha;
  if (p.d_alpha_a && p.d_alpha_b) {
    a *= (*p.d_alpha_a) * (*p.d_alpha_b);
  } else if (p.d_alpha_a) {
    a *= *p.d_alpha_a;
  } else if (p.d_alpha_b) {
    a *= *p.d_alpha_b;
  }
  return a;
}

// What a sum is multiplied by, by the tile of columns that it belongs to (n: the tile's first column, the same for the wave).
struct Alpha {
  float a[kMaxParts];
  __device__ __forceinline__ explicit Alpha(const GemmParams &p) {
    if (!p.parts) {
      a[0] = effective_alpha(p);
      return;
    }
#pragma unroll
    for (int k = 0; k < kMaxParts; ++k)
      if (k < p.parts) a[k] = p.alpha * (p.d_alpha_a ? *p.d_alpha_a * *p.part_alpha[k] : *p.part_alpha[k]);
  }
  __device__ __forceinline__ float at(const GemmParams &p, int n) const {
    if (!p.parts) return a[0];
    float v = a[0];
#pragma unroll
    for (int k = 1; k < kMaxParts; ++k)
      if (k < p.parts && n >= p.part_end[k - 1]) v = a[k];
    return v;
  }
};

struct OneAlpha {
  float a;
  __device__ __forceinline__ explicit OneAlpha(const GemmParams &p) : a(effective_alpha(p)) {}
  __device__ __forceinline__ float at(const GemmParams &, int) const { return a; }
};

// These write M0.  The compiler reserves M0 and refuses it on a clobber list ("may lead to undefined
// behaviour"), so the contract is kept by hand: the kernels that use these helpers contain nothing for
// which the compiler would set or read M0 itself (no LDS-direct builtins, no indirect register
// indexing, no s_sendmsg), and every helper sets M0 before its load.
__device__ __forceinline__ void lds_dma16(const void *g, uint32_t lds_wave_base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               :
               : "s"(lds_wave_base), "v"(g)
               : "memory");
}

// The same with a wave-uniform base address and a 32-bit byte offset per lane.
__device__ __forceinline__ void lds_dma16_at(const void *base, uint32_t lane_offset, uint32_t lds_wave_base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(lds_wave_base), "v"(lane_offset), "s"(base)
               : "memory");
}

// And with a constant part of the LDS address: one scalar instruction forms M0.
__device__ __forceinline__ void lds_dma16_at(const void *base, uint32_t lane_offset, uint32_t lds_wave_base, int lds_offset) {
  asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(lds_wave_base), "v"(lane_offset), "s"(base), "i"(lds_offset)
               : "memory", "scc");
}

__device__ __forceinline__ void lds_dma4_at(const void *base, uint32_t lane_offset, uint32_t lds_wave_base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
               :
               : "s"(lds_wave_base), "v"(lane_offset), "s"(base)
               : "memory");
}

__device__ __forceinline__ void wait_dma_and_sync() {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The accumulator tiles of a wave, by matrix instruction.  In both a lane holds quads: four consecutive output columns n of
// one row m (the weights sit in the instruction's A slot).
//   quads / rows of tiles: kQuads along n, kTiles along m; columns and rows of the wave tile: kN, kM
//   one tile: kSide rows and columns, kTileQuads quads; n of quad q = a constant of q + a term of the lane
typedef float v4f __attribute__((ext_vector_type(4)));

template <int WN, int WM>
struct Acc32 {  // v_mfma_*_32x32x*: element 4 q + e of a lane is n = 8 q + 4 (lane / 32) + e, m = lane % 32
  static constexpr int kQuads = 4 * WN, kTiles = WM, kN = 32 * WN, kM = 32 * WM, kSide = 32, kTileQuads = 4;
  v16f (&a)[WN][WM];
  static __device__ __forceinline__ constexpr int quad_n(int q) { return 32 * (q >> 2) + 8 * (q & 3); }
  static __device__ __forceinline__ int lane_n(int lane) { return 4 * (lane >> 5); }
  static __device__ __forceinline__ int n(int q, int lane) { return quad_n(q) + lane_n(lane); }
  static __device__ __forceinline__ int m(int j, int lane) { return 32 * j + (lane & 31); }
  __device__ __forceinline__ float4 quad(int q, int j) const {
    const v16f &t = a[q >> 2][j];
    const int e = 4 * (q & 3);
    return make_float4(t[e], t[e + 1], t[e + 2], t[e + 3]);
  }
};

template <int NT, int MT>
struct Acc16 {  // v_mfma_*_16x16x*: element e of a lane is n = 4 (lane / 16) + e, m = lane % 16
  static constexpr int kQuads = NT, kTiles = MT, kN = 16 * NT, kM = 16 * MT, kSide = 16, kTileQuads = 1;
  v4f (&a)[NT][MT];
  static __device__ __forceinline__ constexpr int quad_n(int q) { return 16 * q; }
  static __device__ __forceinline__ int lane_n(int lane) { return 4 * (lane >> 4); }
  static __device__ __forceinline__ int n(int q, int lane) { return quad_n(q) + lane_n(lane); }
  static __device__ __forceinline__ int m(int j, int lane) { return 16 * j + (lane & 15); }
  __device__ __forceinline__ float4 quad(int q, int j) const { return make_float4(a[q][j][0], a[q][j][1], a[q][j][2], a[q][j][3]); }
};

// Row of the weights that local row `row` of the tile at n_base holds, kN of them to a wave.
template <int kN, bool HALVES>
__device__ __forceinline__ int weight_row(const GemmParams &p, int n_base, int row) {
  if (!HALVES) return min(n_base + row, p.N - 1);
  const int o = row % kN, F = p.N >> 1;
  return min((n_base >> 1) + row / kN * (kN / 2) + o % (kN / 2), F - 1) + (o >= kN / 2 ? F : 0);
}

// max |output| of a wave's lanes (bf16 bits without the sign) into its segment's word.  One atomic per wave, and only if its maximum is above
// what the word, which never falls, is seen to hold: atomics on one word are served one after the other (16384 x 28672 x 4352, a
// word for 57344 waves: 2852 us, so 2800; MXFP4 4096 rows 357 / 310).
__device__ __forceinline__ void collect_absmax(const GemmParams &p, uint32_t amax, int lane) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint32_t v = (uint32_t)__shfl_xor((int)amax, o);
    amax = v > amax ? v : amax;
  }
  uint32_t *word = p.absmax_bits + p.seg_index;
  if (lane == 0 && (amax << 16) > *const_cast<volatile uint32_t *>(word)) atomicMax(word, amax << 16);  // bf16 bits -> fp32 bits
}

// kSwigluHalves: quads q and q + kQuads / 2 of a lane are the gates and the ups of the same four output columns.  m0: first row of C of the
// wave's tile, n0: first output column.
template <class Acc>
__device__ __forceinline__ void store_wave_tile_halves(const GemmParams &p, const Acc &acc, uint8_t *region, int m0, int n0, int lane) {
  constexpr int kNo = Acc::kN / 2, RB = 2 * kNo, LPR = RB / 16;  // output columns, bytes per row, lanes per row when reading 16 bytes each
  static_assert((LPR & (LPR - 1)) == 0 && RB <= 256, "the swizzle needs a power of two");
  const int F = p.N >> 1;
  const Alpha by_column(p);
  const float ag = by_column.at(p, 0), au = by_column.at(p, F);
  // rows 256 bytes apart (all banks once) take turns
  auto swizzle = [](int m) { return ((m / (256 / RB)) & (LPR - 1)) << 1; };
  wait_dma_and_sync();  // every wave is done reading operands
  const int rows = p.M - m0;
  if (rows <= 0) return;
  uint32_t amax = 0u;
#pragma unroll
  for (int q = 0; q < Acc::kQuads / 2; ++q)
#pragma unroll
    for (int j = 0; j < Acc::kTiles; ++j) {
      const float4 g = acc.quad(q, j), u = acc.quad(q + Acc::kQuads / 2, j);
      const uint2 t = swiglu_quad(make_uint2(pack_bf16_rne(g.x * ag, g.y * ag), pack_bf16_rne(g.z * ag, g.w * ag)),
                                  make_uint2(pack_bf16_rne(u.x * au, u.y * au), pack_bf16_rne(u.z * au, u.w * au)));
      const int m = Acc::m(j, lane), n = Acc::n(q, lane);
      if (m < rows && n0 + n < F) amax = max(max(amax, max(t.x & 0x7fffu, (t.x >> 16) & 0x7fffu)), max(t.y & 0x7fffu, (t.y >> 16) & 0x7fffu));
      *reinterpret_cast<uint2 *>(region + m * RB + (((n >> 2) ^ swizzle(m)) << 3)) = t;
    }
  const int rr = lane / LPR, tq = lane % LPR, col = n0 + 8 * tq;
  uint16_t *cbase = p.c + (size_t)m0 * F + col;
  const int lane_rows = col < F ? rows : 0;  // (F is a multiple of 8)
#pragma unroll
  for (int it = 0; it < (Acc::kM * LPR) / 64; ++it) {
    const int m = it * (64 / LPR) + rr;
    const uint4 v = *reinterpret_cast<const uint4 *>(region + m * RB + (((2 * tq) ^ swizzle(m)) << 3));
    if (m < lane_rows) *reinterpret_cast<uint4 *>(cbase + (size_t)m * F) = v;
  }
  if (p.absmax_bits) collect_absmax(p, amax, lane);
}

// Fused SwiGLU epilogue of the tiled kernels (p.swiglu; N is a multiple of 16): a lane's four consecutive columns of one row are
// (gate_j, up_j, gate_j+1, up_j+1); each is rounded to bf16 as the plain epilogue would store it, and the two
// products act_fn(gate) * up leave through LDS, so that every store instruction writes 16 bytes per lane along output rows.
template <class Acc>
__device__ __forceinline__ void store_wave_tile_swiglu(const GemmParams &p, const Acc &acc, uint8_t *region, int m0, int n0, int lane) {
  const float alpha = effective_alpha(p);
  const int No = p.N >> 1;  // output columns
  uint32_t amax = 0u;       // max |t| of this lane as bf16 bits without the sign
  auto products = [&](int q, int j) {  // of quads q and q + 1; the hardware's RNE convert: the bits f32_to_bf16_bits gives
    const float4 v = acc.quad(q, j), w = acc.quad(q + 1, j);
    return swiglu_quad(make_uint2(pack_bf16_rne(v.x * alpha, v.z * alpha), pack_bf16_rne(w.x * alpha, w.z * alpha)),
                       make_uint2(pack_bf16_rne(v.y * alpha, v.w * alpha), pack_bf16_rne(w.y * alpha, w.w * alpha)));
  };
  wait_dma_and_sync();  // every wave is done reading operands
  const int rows = p.M - m0;  // of this wave's tile inside C
  if (rows <= 0) return;
  constexpr int RB = Acc::kN;        // bytes per row of the wave tile: kN / 2 products
  constexpr int LPR = Acc::kN / 16;  // lanes per row when reading 16 bytes each
  static_assert((LPR & (LPR - 1)) == 0, "the swizzle needs a power of two");
#pragma unroll
  for (int q2 = 0; q2 < Acc::kQuads; q2 += 2)
#pragma unroll
    for (int j = 0; j < Acc::kTiles; ++j) {
      const uint2 two = products(q2, j);  // (every lane: the special-value test of the activation is a vote of the whole wave)
#pragma unroll
      for (int q = q2; q < q2 + 2; ++q) {
        const int m = Acc::m(j, lane), c = Acc::n(q, lane) >> 2;  // row and dword of the row
        const int sw = m & (LPR - 1);                             // swizzle of the row's 16-byte groups
        const uint32_t t = q == q2 ? two.x : two.y;
        if (m < rows && n0 + Acc::n(q, lane) < p.N) {
          const uint32_t lo = t & 0x7fffu, hi = (t >> 16) & 0x7fffu;
          amax = lo > amax ? lo : amax;
          amax = hi > amax ? hi : amax;
        }
        *reinterpret_cast<uint32_t *>(region + m * RB + ((((c >> 2) ^ sw) << 2) | (c & 3)) * 4) = t;
      }
    }
  const int rr = lane / LPR, tq = lane % LPR, col = (n0 >> 1) + 8 * tq;
  uint16_t *cbase = p.c + (size_t)m0 * No + col;
  const int lane_rows = col < No ? rows : 0;
#pragma unroll
  for (int it = 0; it < (Acc::kM * LPR) / 64; ++it) {
    const int m = it * (64 / LPR) + rr;
    const int sw = m & (LPR - 1);
    const uint4 v = *reinterpret_cast<const uint4 *>(region + m * RB + ((tq ^ sw) << 4));
    if (m < lane_rows) *reinterpret_cast<uint4 *>(cbase + (size_t)m * No) = v;
  }
  if (p.absmax_bits) collect_absmax(p, amax, lane);
}

// Tile (i, j) of the wave's accumulators with bounds checks: the row is tested once per tile, the columns once per tile
// where it ends inside C, and the address is formed once.  (Both per quad, here and in the store of split-K's partial
// tiles: 64 x 6144 x 4352, four slices, 17.4 us against 16.3; MXFP4 64 x 4096 x 14592, eight slices, 16.0 against 15.0.)
template <class Acc>
__device__ __forceinline__ void store_tile(const GemmParams &p, const Acc &acc, int i, int j, int m0, int n0, int lane, const Alpha &by_column) {
  const int m = m0 + Acc::m(j, lane);
  if (m >= p.M) return;
  const int n_tile = n0 + Acc::kSide * i;
  const float alpha = by_column.at(p, n_tile);
  const size_t at = (size_t)m * p.N + n_tile + Acc::lane_n(lane);
  uint16_t *dst = p.c + at;
  const uint16_t *res = p.residual ? p.residual + (size_t)m * p.ld_residual + n_tile + Acc::lane_n(lane) : nullptr;
  const bool quads = (p.N & 3) == 0;  // a quad is 8-byte aligned, and inside C or outside as a whole
  auto store = [&](int q) {
    const float4 v = acc.quad(Acc::kTileQuads * i + q, j);
    uint2 w = make_uint2(pack_bf16_rne(v.x * alpha, v.y * alpha), pack_bf16_rne(v.z * alpha, v.w * alpha));
    if (res) w = add_bf16_x4(w, *reinterpret_cast<const uint2 *>(res + Acc::quad_n(q)));
    *reinterpret_cast<uint2 *>(dst + Acc::quad_n(q)) = w;
  };
  if (quads && n_tile + Acc::kSide <= p.N) {
#pragma unroll
    for (int q = 0; q < Acc::kTileQuads; ++q) store(q);
    return;
  }
#pragma unroll
  for (int q = 0; q < Acc::kTileQuads; ++q) {
    const int c = Acc::quad_n(q), n = n_tile + Acc::lane_n(lane) + c;
    if (quads) {
      if (n < p.N) store(q);
      continue;
    }
    const float4 v = acc.quad(Acc::kTileQuads * i + q, j);
    const float f[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < p.N) {
        uint32_t h = f32_to_bf16_bits(f[e] * alpha);
        if (res) h = f32_to_bf16_bits(bf16_bits_to_f32(h) + bf16_bits_to_f32(res[c + e]));
        dst[c + e] = (uint16_t)h;
      }
  }
}

// Epilogue shared by the tiled kernels, called by every wave of the workgroup (there is a barrier in it).  m0 / n0: first row /
// column of C of this wave's tile.  region: 2 * kM * kN bytes of LDS of this wave's own, free for reuse once every wave is done
// reading operands.
template <bool HALVES = false, class Acc>
__device__ __forceinline__ void store_wave_tile(const GemmParams &p, const Acc &acc, uint8_t *region, int m0, int n0, int lane) {
  if constexpr (HALVES) return store_wave_tile_halves(p, acc, region, m0, n0 >> 1, lane);
  if (p.swiglu) return store_wave_tile_swiglu(p, acc, region, m0, n0, lane);
  if (Acc::kSide == 32 && p.partial) {  // split-K: the unscaled fp32 tile of this K range
    float *part = p.partial + (size_t)blockIdx.y * p.M * p.N;
    const bool quads = (p.N & 3) == 0, inside = quads && n0 + Acc::kN <= p.N;
#pragma unroll
    for (int j = 0; j < Acc::kTiles; ++j) {
      const int m = m0 + Acc::m(j, lane);
      if (m >= p.M) continue;
      const int n = n0 + Acc::lane_n(lane);
      float *dst = part + (size_t)m * p.N + n;
      if (inside) {
#pragma unroll
        for (int q = 0; q < Acc::kQuads; ++q) *reinterpret_cast<float4 *>(dst + Acc::quad_n(q)) = acc.quad(q, j);
        continue;
      }
#pragma unroll
      for (int q = 0; q < Acc::kQuads; ++q) {
        const float4 v = acc.quad(q, j);
        const int c = Acc::quad_n(q);
        if (quads) {
          if (n + c < p.N) *reinterpret_cast<float4 *>(dst + c) = v;
          continue;
        }
        const float f[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + c + e < p.N) dst[c + e] = f[e];
      }
    }
    return;
  }
  // Each wave's tile is transposed through LDS (free now) so that every store instruction writes whole rows of the wave tile, 16
  // bytes per lane; what lies behind C's last row or column is left out there.  (Tiles that reach
  // beyond C stored from the registers, 8 bytes per lane and with tests per quad: 1500 x 6144 x 4352 MXFP4 37.0 us, so 32.7; 4090
  // rows 78.0, so 73.0; NVFP4 192.0, so 187.2.  And that code made half of each kernel: 112 KB of <4,2,2>, more than the
  // instruction cache holds.)
  constexpr int RB = 2 * Acc::kN;   // bytes per row of the wave tile
  constexpr int LPR = Acc::kN / 8;  // lanes per row when reading 16 bytes each
  constexpr int IT = (Acc::kM * LPR) / 64;
  static_assert((LPR & (LPR - 1)) == 0, "the swizzle needs a power of two");
  float alpha[Acc::kQuads / Acc::kTileQuads];
  {
    const Alpha by_column(p);
#pragma unroll
    for (int i = 0; i < Acc::kQuads / Acc::kTileQuads; ++i) alpha[i] = by_column.at(p, n0 + Acc::kSide * i);
  }
  wait_dma_and_sync();  // every wave is done reading operands
  if (m0 >= p.M) return;
#pragma unroll
  for (int q = 0; q < Acc::kQuads; ++q)
#pragma unroll
    for (int j = 0; j < Acc::kTiles; ++j) {
      const int m = Acc::m(j, lane), c = Acc::n(q, lane) >> 2;  // row and 8-byte chunk of the row
      const int sw = (m & (LPR - 1)) << 1;                      // even: keeps 8-byte chunk pairs adjacent
      const float4 v = acc.quad(q, j);                          // the hardware's round-to-nearest-even convert
      const float a = alpha[q / Acc::kTileQuads];
      *reinterpret_cast<uint2 *>(region + m * RB + ((c ^ sw) << 3)) = make_uint2(pack_bf16_rne(v.x * a, v.y * a), pack_bf16_rne(v.z * a, v.w * a));
    }
  const int rr = lane / LPR, n = n0 + 8 * (lane % LPR);
  const int rows = n < p.N ? p.M - m0 : 0;  // of this lane's columns inside C
  uint16_t *cbase = p.c + (size_t)m0 * p.N + n;
  const uint16_t *rbase = p.residual ? p.residual + (size_t)m0 * p.ld_residual + n : nullptr;
  auto row = [&](int it) { return it * (64 / LPR) + rr; };
  auto piece = [&](int it) {
    const int m = row(it), sw = (m & (LPR - 1)) << 1;
    return *reinterpret_cast<const uint4 *>(region + m * RB + (((2 * (lane % LPR)) ^ sw) << 3));
  };
  auto put = [&](int it, const uint4 &v) {
    if (row(it) < rows) *reinterpret_cast<uint4 *>(cbase + (size_t)row(it) * p.N) = v;
  };
  if ((p.N & 7) != 0) {  // rows of C that are not 16-byte aligned, and columns that end inside a lane's eight
#pragma unroll 1
    for (int it = 0; it < IT; ++it) {
      if (row(it) >= rows) continue;
      const uint4 v = piece(it);
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
      uint16_t *dst = cbase + (size_t)row(it) * p.N;
      const uint16_t *res = rbase ? rbase + (size_t)row(it) * p.ld_residual : nullptr;
      if ((p.N & 3) == 0) {  // quads are 8-byte aligned, and inside C or outside as a whole
#pragma unroll
        for (int h = 0; h < 2; ++h)
          if (n + 4 * h < p.N) {
            uint2 x = make_uint2(w[2 * h], w[2 * h + 1]);
            if (res) x = add_bf16_x4(x, reinterpret_cast<const uint2 *>(res)[h]);
            reinterpret_cast<uint2 *>(dst)[h] = x;
          }
        continue;
      }
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (n + e < p.N) {
          uint32_t h = (w[e >> 1] >> (16 * (e & 1))) & 0xffffu;
          if (res) h = f32_to_bf16_bits(bf16_bits_to_f32(h) + bf16_bits_to_f32(res[e]));
          dst[e] = (uint16_t)h;
        }
    }
    return;
  }
  if (!rbase) {
#pragma unroll
    for (int it = 0; it < IT; ++it) put(it, piece(it));
    return;
  }
  // The residual is asked for sixteen pieces per lane at a time: one by one, each is a round trip to memory that the store
  // before it holds up (16384 x 4096 x 4352 with a residual, four rounds of tiles: 439 us, so 397).
  constexpr int RI = IT < 16 ? IT : 16;
#pragma unroll
  for (int it0 = 0; it0 < IT; it0 += RI) {
    uint4 res[RI];
#pragma unroll
    for (int k = 0; k < RI; ++k)
      if (row(it0 + k) < rows) res[k] = *reinterpret_cast<const uint4 *>(rbase + (size_t)row(it0 + k) * p.ld_residual);
#pragma unroll
    for (int k = 0; k < RI; ++k) {
      const uint4 v = piece(it0 + k);
      put(it0 + k, make_uint4(add_bf16_pair(v.x, res[k].x), add_bf16_pair(v.y, res[k].y), add_bf16_pair(v.z, res[k].z),
                              add_bf16_pair(v.w, res[k].w)));
    }
  }
}

// The same for the kernels whose waves form a 2 (along N) x NWM (along M) grid, wave = n + 2 * m, of 32x32 tiles.
// ldsA / ldsB: two LDS areas of at least NWM*32*WM*64*WN bytes each.
template <int WN, int WM, int NWM = 2>
__device__ __forceinline__ void store_workgroup_tile(const GemmParams &p, v16f (&acc)[WN][WM], uint8_t *ldsA,
                                                     uint8_t *ldsB, int m_base, int n_base, int wave, int lane) {
  uint8_t *region = (wave < NWM ? ldsA : ldsB) + (wave % NWM) * (32 * WM * 64 * WN);
  store_wave_tile(p, Acc32<WN, WM>{acc}, region, m_base + (wave >> 1) * 32 * WM, n_base + (wave & 1) * 32 * WN, lane);
}

// Swizzle of staged rows of eight 16-byte chunks for the 16x16 matrix instructions.  A 16-byte LDS read is served in groups of 16 lanes that are not
// consecutive: lanes 0-3 and 12-15 of one 16-lane quarter with lanes 4-11 of its neighbour, and the rest of the two.  Here
// neighbouring quarters read chunks two apart, so rows 0-3, 12-15 get even numbers and rows 4-11 odd ones (chunk ^ row / 2,
// which suits 32 rows on one chunk, costs a conflict cycle for every other group: NVFP4 4096 x 28672 x 4352 691 us instead of 682,
// MXFP4 16384 x 4096 x 14592 458 instead of 435).
__device__ __forceinline__ int stage_swizzle(int row) {
  const int q = (row >> 1) & 7;
  return (((q >> 2) ^ (q >> 1)) & 1) | ((q & 1) << 1) | (q & 4);
}

// An FP4 operand of the scaled MFMA is 4 registers; the builtin's type has 8, the upper 4 unused.
__device__ __forceinline__ v8i fp4_operand(uint4 q) {
  const v4i v = {(int)q.x, (int)q.y, (int)q.z, (int)q.w};
  return __builtin_shufflevector(v, v, 0, 1, 2, 3, -1, -1, -1, -1);
}

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

// fp16 bits of two NVFP4 scale bytes sitting in bits 7:0 and 23:16: (1+m/8)*2^(e-9) = (b<<7) + 0x1800
__device__ __forceinline__ uint32_t nv_scale_pair_f16(uint32_t two_bytes) { return (two_bytes << 7) + 0x18001800u; }

// packed fp16 multiply of both halves of a by the LOW (HI=false) or HIGH half of s.  Plain vector
// code, not inline asm: the compiler folds the broadcast into op_sel and, unlike with asm, keeps
// the wait states the matrix pipe needs between a VALU write and an MFMA reading that register.
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
template <bool HI>
__device__ __forceinline__ uint32_t pk_mul_f16_bcast(uint32_t a, uint32_t s) {
  const v2h av = __builtin_bit_cast(v2h, a), sv = __builtin_bit_cast(v2h, s);
  const _Float16 k = HI ? sv[1] : sv[0];
  const v2h kv = {k, k};
  return __builtin_bit_cast(uint32_t, av * kv);
}

template <bool HI>
__device__ __forceinline__ v8h decode8_nvfp4_f16(uint32_t codes, uint32_t scale_pair) {
  // hardware FP4 -> fp16 conversion, two codes per instruction (low nibble first), then one packed
  // multiply by the block scale: 8 VALU instructions per 8 values
  v4u d;
  d[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(codes, 1.0f, 0));
  d[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(codes, 1.0f, 1));
  d[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(codes, 1.0f, 2));
  d[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(codes, 1.0f, 3));
#pragma unroll
  for (int k = 0; k < 4; ++k) d[k] = pk_mul_f16_bcast<HI>(d[k], scale_pair);
  return __builtin_bit_cast(v8h, d);
}

}  // namespace
}  // namespace arcq
#endif  // ARCQ_GEMM_TILE_H_
