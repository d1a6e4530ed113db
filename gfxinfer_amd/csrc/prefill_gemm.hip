// The low-bit GEMM of a wide prefill pass (more than 32 tokens at once) for gfx950, and
// the expansion of its activations.
//
// A 32-token block reads every weight once per 32 tokens and spends most of its vector
// instructions on widening codes; over a whole prompt the same products are a compute
// problem.  Here a workgroup holds 128 weight rows x up to 128 tokens: each weight chunk
// is read and widened once per 128 tokens and reaches the waves through LDS.
//
// Products run on v_mfma_f32_16x16x128_f8f6f4 with both operands in FP6 (e2m3), twice the
// rate of the int8 MFMA: the FP6 codes 0..15 are the numbers 0/8 .. 15/8 (subnormals and
// the first binade are one linear scale), so an unsigned nibble is an FP6 number as it
// stands and a 4-bit activation is its magnitude with a sign bit.  Weights go in as
// u = w + 8 (W4), w + 4 (W3) or w + 3 (W2); the offset times the token's code sum is the
// MFMA's initial accumulator, so the result is the group's exact integer dot over 64 (all
// terms are multiples of 1/64 below 2^9: every fp32 sum is exact).  The epilogue is the
// canonical one (gemm_common.hpp): v = fmaf(P, ws * as, v) group by group with the 64
// folded into as, ranges added in order, so outputs equal the block kernels' bit for bit.
#include <algorithm>
#include <limits>
#include <string>
#include <type_traits>
#include <utility>

#include "common.hpp"
#include "gemm_common.hpp"
#include "prefill.hpp"

namespace gfx950 {
namespace {

using i32x8 = int __attribute__((ext_vector_type(8)));
using f32x4 = float __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// FP6 operands.  A lane's 32 columns are four dwords of eight nibbles (column 8 j + i in
// nibble i of dword j); two dwords x, y make three dwords of 6-bit slots.  The slots hold,
// in order, x0 x1 x3 x4 x6 x7 y1 y2 y4 y5 y7 y0 x2 y3 x5 y6: the order in which shifts by
// 0 and 2 bring whole nibbles to multiples of six.  Weights and activations use the same
// order, so the dot product does not see it.
// ---------------------------------------------------------------------------

__device__ __forceinline__ void fp6_pack(unsigned x, unsigned y, unsigned& d0, unsigned& d1, unsigned& d2) {
  d0 = (x & 0x0F00F00Fu) | ((x << 2) & 0xC03C03C0u);
  d1 = (y & 0xF00F00F0u) | ((y << 2) & 0x03C03C00u) | (x >> 30);
  d2 = ((y << 2) & 0x3C03C03Cu) | (x & 0x00F00F00u);
}

// The nibbles u = w + offset of a lane chunk (common.hpp's layouts), in column order.
template <int Format>
constexpr float kWeightOffset = Format == GFXI_W4G128 ? 8.0F : (Format == GFXI_W3G128 ? 4.0F : 3.0F);

template <int Format>
__device__ __forceinline__ void weight_nibbles(const unsigned* w, unsigned (&n)[4]) {
  if constexpr (Format == GFXI_W4G128) {
#pragma unroll
    for (int d = 0; d < 4; ++d) n[d] = w[d] ^ 0x88888888u;
  } else if constexpr (Format == GFXI_W3G128) {
    constexpr unsigned X = 0x44444444u;
#pragma unroll
    for (int d = 0; d < 3; ++d) n[d] = ((w[d] & 0x07070707u) | ((w[d] << 1) & 0x70707070u)) ^ X;
    n[3] = (((w[0] >> 5) & 0x06060606u) | ((w[1] >> 6) & 0x01010101u) | ((w[2] >> 1) & 0x60606060u) |
            ((w[1] >> 3) & 0x10101010u)) ^ X;
  } else {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      n[2 * h] = ((w[h] << 1) & 0x06060606u) | ((w[h] << 3) & 0x60606060u);
      n[2 * h + 1] = ((w[h] >> 3) & 0x06060606u) | ((w[h] >> 1) & 0x60606060u);
    }
  }
}

// ---------------------------------------------------------------------------
// Activation expansion: one wave per (16-token tile, group).  Memory-bound: reads the A4
// codes once and writes 1.5 times their bytes.
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(256) void prefill_expand_kernel(const uint8_t* __restrict__ codes,
                                                             const __half* __restrict__ scales,
                                                             PrefillOperand out, uint32_t groups, uint32_t tokens) {
  const uint32_t linear = blockIdx.x * 4u + (threadIdx.x >> 6);
  const uint32_t tile = linear % out.tiles, g = linear / out.tiles;
  if (g >= groups) return;
  const unsigned lane = threadIdx.x & 63u, n = lane & 15u, kb = lane >> 4;
  const uint32_t token = tile * 16u + n;
  u32x4 x = u32x4{0u, 0u, 0u, 0u};
  float scale = 0.0F;
  if (token < tokens) {
    x = *reinterpret_cast<const u32x4*>(codes + (static_cast<std::size_t>(token) * groups + g) * 64u + kb * 16u);
    scale = __half2float(scales[static_cast<std::size_t>(token) * groups + g]);
  }
  int sum = 0;
  unsigned magnitude[4], sign[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    sum = __builtin_amdgcn_sdot8(static_cast<int>(x[d]), 0x11111111, sum, false);
    const unsigned one = (x[d] >> 3) & 0x11111111u;   // 1 in every negative nibble
    sign[d] = one << 3;
    magnitude[d] = (x[d] ^ (one * 15u)) + one;        // two's complement: at most 8, no carry
  }
  unsigned d[6], s[6];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    fp6_pack(magnitude[2 * h], magnitude[2 * h + 1], d[3 * h], d[3 * h + 1], d[3 * h + 2]);
    fp6_pack(sign[2 * h], sign[2 * h + 1], s[3 * h], s[3 * h + 1], s[3 * h + 2]);
    // the sign bits, packed at bit 3 of their slots, two up to bit 5
    d[3 * h] |= s[3 * h] << 2;
    d[3 * h + 1] |= (s[3 * h + 1] << 2) | (s[3 * h] >> 30);
    d[3 * h + 2] |= (s[3 * h + 2] << 2) | (s[3 * h + 1] >> 30);
  }
  sum += __shfl_xor(sum, 16);
  sum += __shfl_xor(sum, 32);
  uint8_t* fragment = out.fragments + (static_cast<std::size_t>(g) * out.tiles + tile) * kFragmentBytes;
  *reinterpret_cast<u32x4*>(fragment + lane * 16u) = u32x4{d[0], d[1], d[2], d[3]};
  *reinterpret_cast<u32x2*>(fragment + 1024u + lane * 8u) = u32x2{d[4], d[5]};
  if (kb == 0) {
    out.meta[(static_cast<std::size_t>(g) * out.tiles + tile) * 16u + n] =
        float2{scale * 64.0F, static_cast<float>(sum) * (1.0F / 64.0F)};
  }
}

// ---------------------------------------------------------------------------
// GEMM.  Workgroup = WR x WT waves, wave = RT row tiles x CT token tiles of 16 x 16: 128 rows
// x 128 tokens.
// One group of K per step.  The token side arrives by DMA (buffer_load ... lds) in operand
// order, three steps ahead through four LDS stages; the row side is loaded into one of
// two register sets three steps ahead and widened one step ahead, each wave an equal share
// of the tiles, into one of two LDS buffers.  Every step issues the same loads in the same order (past
// the end of K its last group again), so that its waits count loads and drain none early.
// ---------------------------------------------------------------------------

struct PrefillArgs {
  GemmMatrix matrix[4];
  uint32_t unit_begin[5];  // (row block, split) units before each matrix
  const uint8_t* fragments;
  const float2* meta;
  uint32_t tiles;         // 16-token tiles of the operand
  uint32_t tokens;
  uint32_t groups;
  uint32_t splits;
  uint32_t token_blocks;
};

constexpr int RT = 4, CT = 4;       // 16-row / 16-token tiles of a wave
constexpr unsigned WR = 2, WT = 2;  // waves of a workgroup

template <int Format, bool HalfOut>
__global__ __launch_bounds__(64 * WR * WT, 2) void prefill_gemm_kernel(PrefillArgs args) {
  constexpr unsigned LB = lane_bytes(Format), WD = LB / 4;
  constexpr unsigned kRows = WR * RT, kCols = WT * CT, kWaves = WR * WT;  // 16-row / 16-token tiles
  constexpr unsigned kOwn = kRows / kWaves;                               // row tiles a wave widens
  constexpr unsigned kDma = (kCols * kFragmentBytes / 1024 + kWaves - 1) / kWaves;  // 64 x 16-byte pieces per wave
  constexpr unsigned kStages = 4;                  // token stages in LDS
  constexpr unsigned kSets = 2;                    // weight register sets
  constexpr unsigned kMetaDma = (kCols + 2 * kWaves - 1) / (2 * kWaves);  // 64 x 4-byte pieces of the meta rows per wave
  constexpr unsigned kTokenLoads = kDma + kMetaDma;    // vector-memory instructions of load_tokens
  constexpr unsigned kLoads = kOwn + 1;            // ... and of load_weights
  static_assert(kRows % kWaves == 0 && kOwn == 2 && CT == 4, "two row tiles widened between four token tiles");
  constexpr unsigned kOut = 0x80000000u;
  __shared__ __align__(16) uint8_t row_side[2][kRows * kFragmentBytes];
  // One object per stage, so that the compiler sees which DMA a read can meet: from one
  // array of stages it makes every read wait for the DMA of the same step (1.1 us a step).
  constexpr unsigned kTokenBytes = kDma * kWaves * 1024;
  __shared__ __align__(16) uint8_t tokens0[kTokenBytes], tokens1[kTokenBytes], tokens2[kTokenBytes], tokens3[kTokenBytes];
  __shared__ __align__(16) float row_scales[2][kRows * 16 + 64];
  constexpr unsigned kMetaRows = kMetaDma * kWaves * 32;
  __shared__ __align__(16) float2 meta0[kMetaRows], meta1[kMetaRows], meta2[kMetaRows], meta3[kMetaRows];
  auto token_side = [&](auto stage) __attribute__((always_inline)) -> uint8_t* {
    constexpr unsigned k = decltype(stage)::value;
    if constexpr (k == 0) return tokens0;
    else if constexpr (k == 1) return tokens1;
    else if constexpr (k == 2) return tokens2;
    else return tokens3;
  };
  auto token_meta = [&](auto stage) __attribute__((always_inline)) -> float2* {
    constexpr unsigned k = decltype(stage)::value;
    if constexpr (k == 0) return meta0;
    else if constexpr (k == 1) return meta1;
    else if constexpr (k == 2) return meta2;
    else return meta3;
  };

  // Units in XCD-major order: workgroup b runs on XCD b % 8, and the token blocks of one
  // unit (which read the same weights) follow each other there, so they share its L2.
  const unsigned lane = threadIdx.x & 63u;
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned order = blockIdx.x / 8u;
  unsigned unit = (order / args.token_blocks) * 8u + blockIdx.x % 8u;
  const unsigned token_block = order % args.token_blocks;
  if (unit >= args.unit_begin[4]) return;  // whole workgroup: padding of the XCD-major grid
  unsigned index = 0;
#pragma unroll
  for (unsigned i = 1; i < 4; ++i) {
    if (unit >= args.unit_begin[i]) index = i;
  }
  const GemmMatrix matrix = args.matrix[index];
  unit -= args.unit_begin[index];
  const unsigned split = unit % args.splits;
  const unsigned tile0 = unit / args.splits * kRows;
  const uint32_t groups = args.groups;
  const unsigned valid_rows = min(kRows, matrix.tiles - tile0);
  const unsigned col0 = token_block * kCols;
  const unsigned valid_cols = min(kCols, args.tiles - col0);
  const uint32_t rows = matrix.tiles * 16u;
  const uint32_t tile_bytes = groups * 64u * LB;
  const auto weights =
      buffer(matrix.weights + static_cast<std::size_t>(tile0) * tile_bytes, valid_rows * tile_bytes);
  const auto weight_scales =
      buffer(matrix.scales + static_cast<std::size_t>(tile0) * groups * 16u, valid_rows * groups * 32u);
  const auto fragments = buffer(args.fragments, groups * args.tiles * static_cast<uint32_t>(kFragmentBytes));
  const auto meta = buffer(args.meta, groups * args.tiles * 128u);

  const unsigned n = lane & 15u, kb = lane >> 4;
  const unsigned wr = wave / WT, wt = wave % WT;
  const GroupRange own = split_groups(groups, split, args.splits);
  const unsigned ranges = range_count(own.end - own.begin);

  unsigned wregs[kSets][kOwn][WD];
  unsigned short sregs[kSets];
  auto load_weights = [&](unsigned g, unsigned (&wreg)[kOwn][WD], unsigned short& sreg) __attribute__((always_inline)) {
    g = min(g, own.end - 1u);
#pragma unroll
    for (unsigned j = 0; j < kOwn; ++j) {
      // a tile past the matrix loads the block's last one (widened, never stored)
      const unsigned at = (min(wave * kOwn + j, valid_rows - 1u) * groups + g) * 64u * LB;
      if constexpr (Format == GFXI_W2G128) {
        const u32x2 w = __builtin_amdgcn_raw_buffer_load_b64(weights, lane * LB, at, 0);
        wreg[j][0] = w[0];
        wreg[j][1] = w[1];
      } else if constexpr (Format == GFXI_W3G128) {
        const u32x3 w = __builtin_amdgcn_raw_buffer_load_b96(weights, lane * LB, at, 0);
        wreg[j][0] = w[0];
        wreg[j][1] = w[1];
        wreg[j][2] = w[2];
      } else {
        const u32x4 w = __builtin_amdgcn_raw_buffer_load_b128(weights, lane * LB, at, 0);
        wreg[j][0] = w[0];
        wreg[j][1] = w[1];
        wreg[j][2] = w[2];
        wreg[j][3] = w[3];
      }
    }
    const unsigned tile = min(wave * kOwn + lane / 16u, valid_rows - 1u);
    sreg = __builtin_amdgcn_raw_buffer_load_b16(
        weight_scales, lane < kOwn * 16u ? (tile * groups * 16u + n) * 2u : kOut, g * 32u, 0);
  };
  auto widen_tile = [&](unsigned j, unsigned buf, const unsigned (&wreg)[kOwn][WD]) __attribute__((always_inline)) {
    unsigned u[4], d[6];
    weight_nibbles<Format>(wreg[j], u);
    fp6_pack(u[0], u[1], d[0], d[1], d[2]);
    fp6_pack(u[2], u[3], d[3], d[4], d[5]);
    uint8_t* at = row_side[buf] + (wave * kOwn + j) * kFragmentBytes;
    *reinterpret_cast<u32x4*>(at + lane * 16u) = u32x4{d[0], d[1], d[2], d[3]};
    *reinterpret_cast<u32x2*>(at + 1024u + lane * 8u) = u32x2{d[4], d[5]};
  };
  // The lanes past the scales of the wave's tiles write a row that nothing reads.
  auto widen_scales = [&](unsigned buf, unsigned short sreg) __attribute__((always_inline)) {
    row_scales[buf][lane < kOwn * 16u ? wave * kOwn * 16u + lane : kRows * 16u + lane] =
        __half2float(__ushort_as_half(sreg));
  };
  auto load_tokens = [&](unsigned g, auto stage) __attribute__((always_inline)) {
    g = min(g, own.end - 1u);
    const unsigned first = g * args.tiles + col0;
#pragma unroll
    for (unsigned p = 0; p < kDma; ++p) {
      const unsigned piece = p * kWaves + wave, at = piece * 1024u + lane * 16u;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          fragments, (lds_void*)(token_side(stage) + piece * 1024u), 16,
          at < valid_cols * kFragmentBytes ? at : kOut, first * static_cast<unsigned>(kFragmentBytes), 0, 0);
    }
#pragma unroll
    for (unsigned p = 0; p < kMetaDma; ++p) {
      const unsigned at = (p * kWaves + wave) * 256u + lane * 4u;  // past the block: zeros
      __builtin_amdgcn_raw_ptr_buffer_load_lds(meta, (lds_void*)(token_meta(stage) + (p * kWaves + wave) * 32u), 4,
                                               at < valid_cols * 128u ? at : kOut, first * 128u, 0, 0);
    }
    // Nothing moves above the DMA: the step's wait counts the loads issued after it.
    __builtin_amdgcn_sched_barrier(0);
  };
  // Ends a step: this wave's LDS writes are done and all but its youngest `Younger` loads
  // have arrived; then the same of every wave.
  auto step_barrier = [&](auto younger) __attribute__((always_inline)) {
    constexpr unsigned Y = decltype(younger)::value;
    static_assert(Y <= 63, "vmcnt holds at most 63");
    // One asm block, not a fence and a barrier: a release fence waits for every DMA.
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(Y) : "memory");
  };

  auto fragment = [&](const uint8_t* at) __attribute__((always_inline)) {
    const u32x4 lo = *reinterpret_cast<const u32x4*>(at + lane * 16u);
    const u32x2 hi = *reinterpret_cast<const u32x2*>(at + 1024u + lane * 8u);
    return i32x8{static_cast<int>(lo[0]), static_cast<int>(lo[1]), static_cast<int>(lo[2]), static_cast<int>(lo[3]),
                 static_cast<int>(hi[0]), static_cast<int>(hi[1]), 0, 0};
  };
  float acc[RT][CT][4], total[RT][CT][4];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[r][t][i] = total[r][t][i] = 0.0F;

  // Loads in issue order: T(0) W(0) T(1) W(1) T(2) W(2), then T(g + 3) W(g + 3) in step g
  // (T the tokens, W the weights of a group).
  load_tokens(own.begin, std::integral_constant<unsigned, 0>{});
  load_weights(own.begin, wregs[0], sregs[0]);
  load_tokens(own.begin + 1, std::integral_constant<unsigned, 1>{});
  load_weights(own.begin + 1, wregs[1], sregs[1]);
  __builtin_amdgcn_sched_barrier(0);
  load_tokens(own.begin + 2, std::integral_constant<unsigned, 2>{});
#pragma unroll
  for (unsigned j = 0; j < kOwn; ++j) widen_tile(j, 0, wregs[0]);
  widen_scales(0, sregs[0]);
  load_weights(own.begin + 2, wregs[0], sregs[0]);
  step_barrier(std::integral_constant<unsigned, 2 * kTokenLoads + 3 * kLoads>{});

  unsigned range = 0;
  unsigned range_end = canonical_range(groups, split, args.splits, 0, ranges).end;
  auto step = [&](unsigned g, auto stage_constant) __attribute__((always_inline)) {
    constexpr unsigned stage = decltype(stage_constant)::value, buf = stage & 1u;
    // Stage (g + 3) % 4 was last read in step g - 1; the weight set of group g + 1 takes
    // group g + 3 once it is widened.
    load_tokens(g + 3u, std::integral_constant<unsigned, (stage + 3u) % kStages>{});
    // The products ws * as of all 64 x 64 (row, token) pairs, 16 tokens at a time, by
    // v_mfma_f32_16x16x1_4b_f32: lane l holds row l's scale and token l's, block b of the
    // result pairs row tile b with the token tile that blgp broadcasts.  One product per
    // output: exact, as the two fp16 scales have 22 significant bits between them.
    const float ws = row_scales[buf][wr * RT * 16u + lane];
    const float as = token_meta(stage_constant)[wt * CT * 16u + lane].x;
    i32x8 a[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) a[r] = fragment(row_side[buf] + (wr * RT + r) * kFragmentBytes);
    auto token_tile = [&](auto tile) __attribute__((always_inline)) {
      constexpr int t = decltype(tile)::value;
      const i32x8 b = fragment(token_side(stage_constant) + (wt * CT + t) * kFragmentBytes);
      const float o = token_meta(stage_constant)[(wt * CT + t) * 16u + n].y * -kWeightOffset<Format>;
      const f32x4 offset = f32x4{o, o, o, o};
      const f32x16 scale = __builtin_amdgcn_mfma_f32_16x16x1f32(ws, as, f32x16{}, 0, 0, 4 + t);
      f32x4 c[RT];
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        c[r] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a[r], b, offset, 2, 2, 0, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[r][t][i] = fmaf(c[r][i], scale[4 * r + i], acc[r][t][i]);
    };
    // The next group's tiles are widened between the token tiles, in the shadow of their
    // matrix instructions (before the first token tile, with the expansion: W3 34816 x 5120 x
    // 512 tokens 158 us against 149, W3 12288 x 5120 64.7 against 63, W3 5120 x 17408 in four
    // planes 90.7 against 85, W4 5120 x 5120 36.4 against 34.0).
    token_tile(std::integral_constant<int, 0>{});
    widen_tile(0, buf ^ 1u, wregs[buf ^ 1u]);
    token_tile(std::integral_constant<int, 1>{});
    widen_tile(1, buf ^ 1u, wregs[buf ^ 1u]);
    token_tile(std::integral_constant<int, 2>{});
    widen_scales(buf ^ 1u, sregs[buf ^ 1u]);
    load_weights(g + 3u, wregs[buf ^ 1u], sregs[buf ^ 1u]);
    token_tile(std::integral_constant<int, 3>{});
    if (g + 1 == range_end) {  // workgroup-uniform: the range's value joins the split's
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < CT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            total[r][t][i] = range == 0 ? acc[r][t][i] : total[r][t][i] + acc[r][t][i];
            acc[r][t][i] = 0.0F;
          }
      ++range;
      if (range < ranges) range_end = canonical_range(groups, split, args.splits, range, ranges).end;
    }
    // the tokens of group g + 1 have arrived: younger are W(g + 1), T W (g + 2), T W (g + 3)
    step_barrier(std::integral_constant<unsigned, 2 * kTokenLoads + 3 * kLoads>{});
  };
  static_assert(kStages == 4 && kSets == 2, "the step loop is unrolled by four");
  for (unsigned g = own.begin; g < own.end; g += 4) {
    step(g, std::integral_constant<unsigned, 0>{});
    if (g + 1 >= own.end) break;
    step(g + 1, std::integral_constant<unsigned, 1>{});
    if (g + 2 >= own.end) break;
    step(g + 2, std::integral_constant<unsigned, 2>{});
    if (g + 3 >= own.end) break;
    step(g + 3, std::integral_constant<unsigned, 3>{});
  }

  const std::size_t plane = static_cast<std::size_t>(split) * args.tokens * rows;
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const unsigned tile = wr * RT + r;
    if (tile >= valid_rows) break;  // wave-uniform
#pragma unroll
    for (int t = 0; t < CT; ++t) {
      const unsigned token = (col0 + wt * CT + t) * 16u + n;
      if (token >= args.tokens) continue;
      const std::size_t out = plane + static_cast<std::size_t>(token) * rows + (tile0 + tile) * 16u + 4u * kb;
      if constexpr (HalfOut) {
        __half* o = reinterpret_cast<__half*>(matrix.output) + out;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = to_half(total[r][t][i]);
      } else {
        *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(matrix.output) + out) =
            f32x4{total[r][t][0], total[r][t][1], total[r][t][2], total[r][t][3]};
      }
    }
  }
}

template <int Format, bool HalfOut>
void launch(PrefillArgs& args, hipStream_t stream) {
  uint32_t units = 0;
  for (unsigned i = 0; i < 4; ++i) {
    args.unit_begin[i] = units;
    if (args.matrix[i].weights != nullptr) units += (args.matrix[i].tiles + WR * RT - 1) / (WR * RT) * args.splits;
  }
  args.unit_begin[4] = units;
  args.token_blocks = (args.tiles + WT * CT - 1) / (WT * CT);
  hipLaunchKernelGGL((prefill_gemm_kernel<Format, HalfOut>), dim3((units + 7) / 8 * 8 * args.token_blocks),
                     dim3(64 * WR * WT), 0, stream, args);
}

}  // namespace

int32_t prefill_expand(const uint8_t* codes, const uint16_t* scales, const PrefillOperand& out,
                       std::size_t columns, uint32_t tokens, hipStream_t stream) {
  const auto groups = static_cast<uint32_t>(columns / kGroup);
  hipLaunchKernelGGL(prefill_expand_kernel, dim3((groups * out.tiles + 3) / 4), dim3(256), 0, stream, codes,
                     reinterpret_cast<const __half*>(scales), out, groups, tokens);
  return launch_status("prefill activation expansion launch failed");
}

int32_t prefill_gemm(int32_t format, const PrefillMatrix* matrices, std::size_t count,
                     const PrefillOperand& in, std::size_t columns, uint32_t tokens, uint32_t splits,
                     bool half_output, hipStream_t stream) {
  if (!valid_weight_format(format) || count == 0 || count > 4 || columns == 0 || columns % kGroup != 0 ||
      tokens == 0 || in.tiles != (tokens + 15) / 16 || splits == 0 || splits > columns / kGroup ||
      (splits > 1 && count > 1) ||
      prefill_fragment_bytes(columns, tokens) > std::numeric_limits<int32_t>::max()) {
    return fail(GFXI_INVALID_ARGUMENT, "invalid prefill GEMM arguments");
  }
  PrefillArgs args{};
  for (std::size_t i = 0; i < count; ++i) {
    const PrefillMatrix& m = matrices[i];
    if (m.weights == nullptr || m.scales == nullptr || m.output == nullptr || m.rows == 0 || m.rows % 16 != 0 ||
        m.rows > std::numeric_limits<uint32_t>::max() / 16) {
      return fail(GFXI_INVALID_ARGUMENT, "invalid prefill GEMM matrix");
    }
    args.matrix[i] = {m.weights, reinterpret_cast<const __half*>(m.scales), m.output,
                      static_cast<uint32_t>(m.rows / 16)};
  }
  args.fragments = in.fragments;
  args.meta = in.meta;
  args.tiles = in.tiles;
  args.tokens = tokens;
  args.groups = static_cast<uint32_t>(columns / kGroup);
  args.splits = splits;
  switch (format) {
    case GFXI_W2G128:
      half_output ? launch<GFXI_W2G128, true>(args, stream) : launch<GFXI_W2G128, false>(args, stream);
      break;
    case GFXI_W3G128:
      half_output ? launch<GFXI_W3G128, true>(args, stream) : launch<GFXI_W3G128, false>(args, stream);
      break;
    default:
      half_output ? launch<GFXI_W4G128, true>(args, stream) : launch<GFXI_W4G128, false>(args, stream);
      break;
  }
  return launch_status("prefill GEMM launch failed");
}

}  // namespace gfx950

using namespace gfx950;

extern "C" size_t gfxinfer_debug_gemm_prefill_workspace_bytes(size_t columns, uint32_t tokens) {
  return columns % kGroup != 0 ? 0 : prefill_fragment_bytes(columns, tokens) + prefill_meta_bytes(columns, tokens);
}

extern "C" int32_t gfxinfer_debug_gemm_prefill(int32_t format, const uint8_t* tiled_weights,
                                               const uint16_t* tiled_weight_scales,
                                               const uint8_t* packed_activations,
                                               const uint16_t* activation_scales, void* output,
                                               int32_t half_output, size_t rows, size_t columns, uint32_t tokens,
                                               uint32_t splits, void* workspace, size_t workspace_bytes,
                                               void* stream) {
  if (packed_activations == nullptr || activation_scales == nullptr || workspace == nullptr || tokens == 0 ||
      columns == 0 || columns % kGroup != 0 || reinterpret_cast<std::uintptr_t>(workspace) % 16 != 0 ||
      reinterpret_cast<std::uintptr_t>(packed_activations) % 16 != 0 ||
      reinterpret_cast<std::uintptr_t>(tiled_weights) % 16 != 0 ||
      reinterpret_cast<std::uintptr_t>(output) % 16 != 0 ||
      workspace_bytes < gfxinfer_debug_gemm_prefill_workspace_bytes(columns, tokens)) {
    return fail(GFXI_INVALID_ARGUMENT, "invalid prefill GEMM debug arguments");
  }
  auto* base = static_cast<uint8_t*>(workspace);
  const PrefillOperand operand{base, reinterpret_cast<float2*>(base + prefill_fragment_bytes(columns, tokens)),
                               (tokens + 15) / 16};
  const auto s = static_cast<hipStream_t>(stream);
  if (const int32_t e = prefill_expand(packed_activations, activation_scales, operand, columns, tokens, s);
      e != GFXI_OK) {
    return e;
  }
  const PrefillMatrix m{tiled_weights, tiled_weight_scales, output, rows};
  return prefill_gemm(format, &m, 1, operand, columns, tokens, splits, half_output != 0, s);
}
