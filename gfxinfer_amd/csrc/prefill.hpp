// Launches of the wide prefill pass: more than 32 tokens at once, for the session only
// (the public launchers keep their 32-token blocks).  Every value they compute equals the
// block launchers' bit for bit.
#pragma once

#include "common.hpp"

namespace gfx950 {

// A wide activation block as the prefill GEMM reads it: per (group of 128 columns, tile of
// 16 tokens) the B operand of one 16x16x128 MFMA in FP6 (e2m3), and per (group, token) the
// activation scale and the sum of its codes.  `tiles` 16-token tiles; tokens past the last
// one hold zeros.
constexpr std::size_t kFragmentBytes = 1536;  // 64 lanes x 24 bytes
struct PrefillOperand {
  uint8_t* fragments;  // [groups][tiles][kFragmentBytes]
  float2* meta;        // [groups][tiles * 16] (scale * 64, sum of codes / 64)
  uint32_t tiles;
};
inline std::size_t prefill_fragment_bytes(std::size_t columns, std::size_t tokens) {
  return columns / kGroup * ((tokens + 15) / 16) * kFragmentBytes;
}
inline std::size_t prefill_meta_bytes(std::size_t columns, std::size_t tokens) {
  return columns / kGroup * ((tokens + 15) / 16) * 16 * sizeof(float2);
}

// A4 codes [tokens][columns / 2] and scales [tokens][columns / 128] -> operand.
int32_t prefill_expand(const uint8_t* codes, const uint16_t* scales, const PrefillOperand& out,
                       std::size_t columns, uint32_t tokens, hipStream_t stream);

// gfxinfer_launch_gfx950_i4_gemm[_fused | _split | _half] over a wide operand: 1..4 matrices
// of one format and column count; splits > 1 (one matrix) writes fp32 planes.
struct PrefillMatrix {
  const uint8_t* weights;
  const uint16_t* scales;
  void* output;  // fp32 or fp16 [splits][tokens][rows]
  std::size_t rows;
};
int32_t prefill_gemm(int32_t format, const PrefillMatrix* matrices, std::size_t count,
                     const PrefillOperand& in, std::size_t columns, uint32_t tokens, uint32_t splits,
                     bool half_output, hipStream_t stream);

// gfxinfer_launch_gdn_conv_window over any number of tokens, without logs.  Rows 16-byte
// aligned; conv and recurrent states are not updated in place.
struct GdnPrefillPass {
  const float* projected;         // [tokens][channels]
  const uint16_t* conv_weight;    // bf16 [channels][4]
  const uint16_t* conv_initial;   // fp16 [channels][4]
  uint16_t* conv_final;
  const float* a;                 // [tokens][value_heads]
  const float* b;
  const uint16_t* a_log;          // bf16 [value_heads]
  const uint16_t* dt_bias;
  float* convolved;               // scratch [tokens][channels]
  float* gates;                   // scratch [2][tokens][value_heads]
  const float* initial_state;     // [value_heads][128][128]
  float* final_state;
  float* mixed;                   // [tokens][value_heads * 128]
  uint32_t tokens, key_heads, value_heads;
};
int32_t gdn_prefill(const GdnPrefillPass& pass, hipStream_t stream);

// gfxinfer_launch_gated_attention_decode_block_quantize_i4 over any number of tokens: token
// t at position + t, each 32-token block with the splits and the arithmetic of a launch of
// its own.  The workspace holds at least one block's partial results
// (gfxinfer_attention_workspace_bytes(32, ..., position + tokens)).
struct PrefillAttention {
  const uint16_t* query;        // [tokens][q_heads * head_size]
  const float* gate;            // [tokens][q_heads][2 * head_size]
  const uint16_t* key_cache;
  const uint16_t* value_cache;
  uint16_t* output;             // [tokens][q_heads * head_size]
  uint8_t* codes;
  uint16_t* scales;
  uint64_t position;
  std::size_t capacity;
  uint32_t tokens, q_heads, kv_heads, head_size;
  float* workspace;
  std::size_t workspace_bytes;
};
int32_t prefill_attention(const PrefillAttention& attention, hipStream_t stream);

// The block launchers' kernels over any number of rows.
int32_t quantize_activation_rows(const uint16_t* input, uint8_t* codes, uint16_t* scales, std::size_t columns,
                                 uint32_t rows, hipStream_t stream);
int32_t silu_multiply_quantize_rows(const float* gate, const float* up, uint8_t* codes, uint16_t* scales,
                                    std::size_t columns, uint32_t rows, hipStream_t stream);
int32_t gdn_output_quantize_rows(const float* mixed, const float* z, const uint16_t* norm_weight, uint8_t* codes,
                                 uint16_t* scales, uint32_t rows, uint32_t value_heads, hipStream_t stream);

}  // namespace gfx950
