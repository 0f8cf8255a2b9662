// A few prompt tokens at once, with the decode step's arithmetic.
//
// A prompt chunk too short for the MFMA GEMMs of prefill used to run through
// the decode step token by token, streaming every weight once per token. These
// kernels stream them once for the chunk and give each token the bits the
// decode step gives it: the projections keep the summation order of
// gemv_core.h, attention is attention_decode.h's block per (token, query
// head), and norms, RoPE and SwiGLU are the unfused kernels' (whose bits are
// the fused step's).
#pragma once

#include "decode_step.h"

namespace lcr {

// Most tokens of one call.
constexpr int kShortPromptMaxTokens = 64;

// Where element k of token t's projection input lies. The inputs are kept in
// the order the projections' MFMA operands take them, so that a wave reads 1 KB
// pieces of them: by 2048-element slice, 512-element chunk, quad (of the
// chunk's 64 lane chains, those equal modulo 16), 16-token fragment, MFMA block
// (chain / 16) and token of the fragment, eight elements each.
__host__ __device__ inline int short_fragment_index(int k, int t, int tokens) {
  const int chunk = k >> 9;  // over all slices
  const int chain = (k >> 3) & 63;
  const int fragments = (tokens + 15) >> 4;
  return (((chunk * 16 + (chain & 15)) * fragments + (t >> 4)) << 9) + ((chain >> 4) << 7) + ((t & 15) << 3) + (k & 7);
}
// Elements of such an input.
inline size_t short_fragment_elements(int tokens, int k) {
  return static_cast<size_t>((tokens + 15) / 16 * 16) * static_cast<size_t>(k);
}

// The activations of a chunk; `position` is that of its first token, and every
// one of its tokens attends with a single split.
struct ShortPromptArgs {
  int tokens, position;
  int num_heads, num_kv_heads, head_dim;
  int hidden, ffn;
  int compute_units;
  bool paged;
  const float2* rope_table;  // [max_seq][head_dim / 2]
  elem_t* x;       // [tokens][hidden] residual stream
  elem_t* q;       // [tokens][num_heads * head_dim]
  elem_t* normed;  // fragment order, hidden elements a token
  elem_t* attn;    // fragment order, num_heads * head_dim elements a token
  elem_t* act;     // fragment order, ffn elements a token
  float* partial;  // [slices][tokens][hidden] sums of o_proj (one slice) or down (short_down_slices)
};

int short_down_slices(int ffn);
// Floats of ShortPromptArgs::partial for a chunk of `tokens`.
inline size_t short_partial_floats(int tokens, int hidden, int ffn) {
  return static_cast<size_t>(short_down_slices(ffn)) * tokens * hidden;
}

// The steps of a chunk, for the geometries of decode_step_supported.
// x = the ids' embedding rows, normed = RMSNorm(x) * weight.
void enqueue_short_embed_norm(const ShortPromptArgs& a, const elem_t* table, const int32_t* ids,
                              const elem_t* weight, float eps, hipStream_t stream);
// q/k/v + RoPE + KV append, then attention: normed -> q, cache, attn.
void enqueue_short_qkv_attention(const ShortPromptArgs& a, const LayerDevicePtrs& w, const KvCacheView& view,
                                 hipStream_t stream);
// o_proj: attn -> partial, one slice.
void enqueue_short_oproj(const ShortPromptArgs& a, const LayerDevicePtrs& w, hipStream_t stream);
// gate/up + SwiGLU, then down: normed -> act -> partial, short_down_slices().
void enqueue_short_mlp(const ShortPromptArgs& a, const LayerDevicePtrs& w, hipStream_t stream);
// x += the slices' sum (added in slice order, rounded), normed = RMSNorm(x) * weight.
void enqueue_short_residual_norm(const ShortPromptArgs& a, const elem_t* weight, int slices, float eps,
                                 hipStream_t stream);
// resid = x + the last down projection of the chunk's last token, unrounded:
// the output head's input.
void enqueue_short_residual(const ShortPromptArgs& a, float* resid, hipStream_t stream);

}  // namespace lcr
