// What the low-bit GEMM kernels share: vector types, buffer descriptors, the matrix
// binding and the canonical order of the sum over K.
#pragma once

#include "common.hpp"

namespace gfx950 {

using i32x4 = int __attribute__((ext_vector_type(4)));
using u32x4 = unsigned __attribute__((ext_vector_type(4)));
using u32x3 = unsigned __attribute__((ext_vector_type(3)));
using u32x2 = unsigned __attribute__((ext_vector_type(2)));
using f32x16 = float __attribute__((ext_vector_type(16)));

// Buffer descriptors: one SGPR resource per stream, a lane-constant VGPR offset
// and a wave-uniform SGPR offset per access, so a load costs no address VGPRs.
// Reads past num_records return zeros (used for a missing last group).
constexpr int kBufferWord3 = 0x00020000;  // gfx9-family raw buffer, 32-bit data format
constexpr int kStreaming = 2;             // nt: weights are read exactly once

typedef __attribute__((address_space(3))) void lds_void;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes),
                                           kBufferWord3);
}

struct GemmMatrix {
  const uint8_t* weights;
  const __half* scales;
  void* output;
  uint32_t tiles;
};

// Canonical summation over K.  Every GEMM variant adds the int32 group partials the
// same way, so an output depends only on (row, token, K, splits): not on the batch,
// the kernel family or the launch shape, and a block of tokens gives each token
// exactly what a one-token step gives it (as the reference's sequential epilogue does).
//   * split s of S owns groups [G s / S, G (s + 1) / S) of the G groups;
//   * a split of n groups [b, b + n) is cut into R = range_count(n) ranges, range r
//     holding groups [b + n r / R, b + n (r + 1) / R);
//   * a range's value is v = fmaf(float(partial_g), ws_g * as_g, v) over its groups g
//     in increasing order, from v = 0 (partial_g: the group's exact int32 MFMA sum;
//     ws_g, as_g: the row's fp16 weight scale and the token's activation scale times
//     1/F, as fp32);
//   * a split's output is ((range_0 + range_1) + range_2) + ... in range order.
// A kernel may give a wave several consecutive ranges.  Load chunks start at the
// range's first group and hold CH packs of GP groups; the MFMA pair of a pack leaves
// group pg + w in the lanes of token window w, and add_pack folds the pack's groups
// into the value held by the window-0 lanes in group order.  Groups past the range's
// end are skipped.
struct GroupRange {
  unsigned begin, end;  // groups [begin, end)
};

__host__ __device__ inline GroupRange split_groups(unsigned groups, unsigned split, unsigned splits) {
  return {groups * split / splits, groups * (split + 1u) / splits};
}

__host__ __device__ inline unsigned range_count(unsigned groups_in_split) {
  const unsigned r = (groups_in_split + 9u) / 10u;  // about ten groups per range
  return r < 1u ? 1u : (r > 16u ? 16u : r);
}

__host__ __device__ inline GroupRange canonical_range(unsigned groups, unsigned split, unsigned splits,
                                                      unsigned range, unsigned ranges) {
  const GroupRange own = split_groups(groups, split, splits);
  const unsigned n = own.end - own.begin;
  return {own.begin + n * range / ranges, own.begin + n * (range + 1u) / ranges};
}

}  // namespace gfx950
