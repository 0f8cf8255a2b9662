// Short prompt chunks with the decode step's arithmetic (short_prompt.h).
#include <algorithm>
#include <cmath>

#include "../hip_utils.h"
#include "attention_decode.h"
#include "gemv_core.h"
#include "row_norm.h"
#include "short_prompt.h"

namespace lcr {
namespace {

// ---------------------------------------------------------------------------
// Projections
// ---------------------------------------------------------------------------
//
// A decode GEMV row (gemv_core.h) is, per 2048 elements, 64 chains of 32
// fused multiply-adds, one per lane, added by a butterfly. For T tokens the
// chains are independent small products of rows and tokens, which is what
// v_mfma_f32_16x16x1_4b_f32 computes: four separate 16 x 16 outer products
// (blocks), each accumulated with one fused multiply-add per element and
// instruction. On gfx950 that accumulation is fmaf's to the bit (checked over
// 1.2 million sums with denormal, cancelling and infinite operands), so the
// results are the decode step's bits at up to twice the rate of VALU fmas,
// 127 TFLOP/s measured.
//
// A block owns 16 FT tokens of one 2048-element slice of K and walks row tiles
// of 16. Its tokens' values stay in registers, widened, for all of them; the
// weights go through a ring of LDS stages of 1024 elements of 16 rows, filled
// by direct global-to-LDS loads of whole 1 KB row pieces that run three stages
// ahead. In a 512-element chunk (elements 8 l .. 8 l + 7 are lane l's), MFMA
// block b of a wave's quad l holds chain l + 16 b, and wave w has quads w and
// w + 8: the butterfly's offsets 32 and 16 pair MFMA blocks and offset 8 the
// quads, in registers; offsets 4, 2, 1 pair the eight waves through LDS.
// Slices of a longer row leave fp32 sums, which the residual norm adds from
// left to right.
//
// Bound by the fp32 matrix rate above 16 tokens (gate/up at 32: 17 us, against
// 9.6 us for its weights from HBM), by the weights below. On gfx950 these
// MFMAs and VALU instructions do not overlap, so what is left of the loop is
// one widening per weight pair and tile. A 27-token prompt went from 14.6 to
// 1.31 ms; per layer at 27 tokens gate/up takes 29.7 us, down 18.4, q/k/v
// 11.0, o_proj 7.5. Weights and tokens loaded straight to registers by the
// waves that use them (64-byte row pieces) took 33 us for gate/up, both
// staged in LDS and widened for every tile 34.
enum class ShortOut { kPartial, kRope, kSwiglu };

typedef float mfma_acc16 __attribute__((ext_vector_type(16)));

struct ShortProjection {
  const elem_t* w;
  const elem_t* x;  // [tokens][k] in fragment order (short_fragment_index)
  void* out;        // kPartial float [slices][tokens][rows], kRope q [tokens][q_dim],
                    // kSwiglu act [tokens][rows / 2] in fragment order
  int rows;         // of w, a multiple of 128
  int k;            // a multiple of 2048; 2048 unless kPartial
  int tokens;
  int token_tiles;
  int lanes;        // slices x token_tiles: a block keeps one (slice, token tile)
  // kRope
  const float2* rope_table;
  KvCacheView view;
  int position;
  int q_dim;
};

constexpr int kShortWaves = 8;
constexpr int kShortThreads = 64 * kShortWaves;
constexpr int kShortChunk = 512;       // elements of a row piece
constexpr int kShortStageChunks = 2;   // chunks per ring stage
constexpr int kShortStages = 4;        // 128 KiB
constexpr int kShortTileStages = kGemvLaneChunks / kShortStageChunks;
constexpr int kShortLoads = 16 * kShortStageChunks / kShortWaves;  // 1 KB loads per wave and stage

template <int FT>
struct ShortShared {
  elem_t stage[kShortStages][kShortStageChunks][16 * kShortChunk];
  float red[kShortWaves][FT][4][64];
};

template <ShortOut kOut, bool kPaged, int FT>
__global__ __launch_bounds__(kShortThreads, 2) void short_projection_kernel(ShortProjection p) {
  constexpr int HD = 64;
  __shared__ __attribute__((aligned(1024))) ShortShared<FT> sh;

  const int lane = lane_id();
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int sub = lane & 15;
  const int chain = lane >> 4;

  // XCD x (block id mod 8) has row tiles x, x + 8, ...; its blocks share them
  // out, and the blocks of a tile's slices and token tiles run side by side
  // there, so its weights come from HBM once.
  const int xcd = static_cast<int>(blockIdx.x) & 7;
  const int in_xcd = static_cast<int>(blockIdx.x) >> 3;
  const int mine = in_xcd % p.lanes;
  const int slice = mine / p.token_tiles;
  const int t0 = (mine % p.token_tiles) * (16 * FT);
  const int step = (static_cast<int>(gridDim.x) >> 3) / p.lanes;
  const int first = in_xcd / p.lanes;
  const int tiles = (p.rows / 128 - first + step - 1) / step;
  const int stages = tiles * kShortTileStages;
  auto tile_of = [&](int n) { return xcd + 8 * (first + n * step); };
  // Rows of a tile. Rope: pairs i0 .. i0 + 7 of a head; SwiGLU: gate and up
  // of eight activations; each so that a lane's four results (tile rows
  // 4 g + v) are two pairs, v and v + 2.
  auto row_of = [&](int tile, int i) -> int {
    if constexpr (kOut == ShortOut::kRope) {
      return (tile >> 2) * HD + 8 * (tile & 3) + 2 * (i >> 2) + (i & 1) + ((i & 2) ? HD / 2 : 0);
    } else if constexpr (kOut == ShortOut::kSwiglu) {
      return 8 * tile + 2 * (i >> 2) + (i & 1) + ((i & 2) ? p.rows / 2 : 0);
    } else {
      return 16 * tile + i;
    }
  };

  // Stage g: half g % 2 of this block's (g / 2)-th tile's slice. Row r of a
  // chunk holds 16-byte piece c at slot c ^ (r & 15), so the fragment reads of
  // 16 rows spread over all banks; a load's lane takes the piece of its slot.
  // Stages are issued in order: `src` walks a tile's chunks and is set anew at
  // the next tile's first.
  const uint32_t ring_base = lds_address_of(sh.stage) + static_cast<uint32_t>(w * kShortChunk * 2);
  const elem_t* src[16 / kShortWaves];
  auto issue = [&](int g) {
    if (g % kShortTileStages == 0) {
      const int tile = tile_of(g / kShortTileStages);
#pragma unroll
      for (int i = 0; i < 16 / kShortWaves; ++i) {
        const int r = kShortWaves * i + w;
        src[i] = p.w + static_cast<size_t>(row_of(tile, r)) * p.k + slice * kGemvBlock + 8 * (lane ^ r);
      }
    }
    const uint32_t base = ring_base + static_cast<uint32_t>((g % kShortStages) * kShortStageChunks * 16 * kShortChunk * 2);
#pragma unroll
    for (int c = 0; c < kShortStageChunks; ++c) {
#pragma unroll
      for (int i = 0; i < 16 / kShortWaves; ++i) {
        load_to_lds16(src[i], base + static_cast<uint32_t>((c * 16 + i * kShortWaves) * kShortChunk * 2));
        src[i] += kShortChunk;
      }
    }
  };
  for (int g = 0; g < kShortStages - 1 && g < stages; ++g) issue(g);

  // This wave's token values: quads w and w + 8 of the slice's four chunks.
  float xr[kGemvLaneChunks][2][FT][8];
  {
    const int frags = (p.tokens + 15) / 16;
#pragma unroll
    for (int c = 0; c < kGemvLaneChunks; ++c) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
#pragma unroll
        for (int f = 0; f < FT; ++f) {
          const int frag = min(t0 / 16 + f, frags - 1);
          unpack8(load16(p.x + ((static_cast<size_t>(slice * kGemvLaneChunks + c) * 16 + w + 8 * q) * frags + frag) * 512 +
                         8 * lane),
                  xr[c][q][f]);
        }
      }
    }
  }

  for (int n = 0; n < tiles; ++n) {
    mfma_acc16 acc[2][FT];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
#pragma unroll
      for (int f = 0; f < FT; ++f) acc[q][f] = mfma_acc16(0.0f);
    }
#pragma unroll
    for (int half = 0; half < kShortTileStages; ++half) {
      // This wave's loads of stage g have landed (at most the younger stages'
      // remain) and its reads of stage g - 1 have returned; after the barrier
      // that holds for every wave, and stage g - 1's buffer is free.
      const int g = n * kShortTileStages + half;
      if (g + kShortStages - 2 < stages) {
        wait_stage_landed<kShortLoads * (kShortStages - 2)>();
      } else {
        wait_stage_landed<0>();
      }
      plain_barrier();
      if (g + kShortStages - 1 < stages) issue(g + kShortStages - 1);
#pragma unroll
      for (int cc = 0; cc < kShortStageChunks; ++cc) {
        const int c = half * kShortStageChunks + cc;
        const elem_t* rows = sh.stage[g % kShortStages][cc] + sub * kShortChunk;
        vec16 wv[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) wv[q] = load16(rows + 8 * (16 * chain + ((w + 8 * q) ^ sub)));
#pragma unroll
        for (int e = 0; e < 8; ++e) {
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const float wf = (e & 1) ? elem_hi(wv[q].w[e / 2]) : elem_lo(wv[q].w[e / 2]);
#pragma unroll
            for (int f = 0; f < FT; ++f) {
              acc[q][f] = __builtin_amdgcn_mfma_f32_16x16x1f32(wf, xr[c][q][f][e], acc[q][f], 0, 0, 0);
            }
          }
        }
      }
    }
    // Register 4 b + v of lane l: MFMA block b, tile row 4 (l / 16) + v, token
    // l % 16 of the fragment. `red` was last read two barriers ago.
#pragma unroll
    for (int f = 0; f < FT; ++f) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float a = (acc[0][f][v] + acc[0][f][8 + v]) + (acc[0][f][4 + v] + acc[0][f][12 + v]);
        const float b = (acc[1][f][v] + acc[1][f][8 + v]) + (acc[1][f][4 + v] + acc[1][f][12 + v]);
        sh.red[w][f][v][lane] = a + b;
      }
    }
    // LDS writes only: a full barrier would wait for the stage loads in flight.
    wait_lds();
    plain_barrier();
    const int tile = tile_of(n);
    auto total = [&](int f, int v, int l) -> float {
      const float s0 = sh.red[0][f][v][l] + sh.red[4][f][v][l];
      const float s1 = sh.red[1][f][v][l] + sh.red[5][f][v][l];
      const float s2 = sh.red[2][f][v][l] + sh.red[6][f][v][l];
      const float s3 = sh.red[3][f][v][l] + sh.red[7][f][v][l];
      return (s0 + s2) + (s1 + s3);
    };
    const int tid = static_cast<int>(threadIdx.x);
    if constexpr (kOut == ShortOut::kPartial) {
      float* out = static_cast<float*>(p.out) + static_cast<size_t>(slice) * p.tokens * p.rows;
      for (int item = tid; item < FT * 256; item += kShortThreads) {
        const int l = item & 63, v = (item >> 6) & 3, f = item >> 8;
        const int t = t0 + 16 * f + (l & 15);
        if (t < p.tokens) {
          out[static_cast<size_t>(t) * p.rows + row_of(tile, 4 * (l >> 4) + v)] = total(f, v, l);
        }
      }
    } else if (tid < FT * 128) {
      const int l = tid & 63, v = (tid >> 6) & 1, f = tid >> 7;
      const int t = t0 + 16 * f + (l & 15);
      if (t < p.tokens) {
        const float lo = elem_to_float(float_to_elem(total(f, v, l)));
        const float hi = elem_to_float(float_to_elem(total(f, v + 2, l)));
        const int row = row_of(tile, 4 * (l >> 4) + v);
        elem_t* out = static_cast<elem_t*>(p.out);
        if constexpr (kOut == ShortOut::kSwiglu) {
          out[short_fragment_index(row, t, p.tokens)] = float_to_elem(lcr_silu(lo) * hi);
        } else {
          const int i = row % HD;
          const int kv_dim = p.view.num_kv_heads * HD;
          const int position = p.position + t;
          elem_t* dst;
          float a = lo, b = hi;
          if (row < p.q_dim + kv_dim) {
            const float2 r = rope_rotate(lo, hi, p.rope_table[static_cast<size_t>(position) * (HD / 2) + i]);
            a = r.x;
            b = r.y;
            dst = row < p.q_dim ? out + static_cast<size_t>(t) * p.q_dim + row
                                : p.view.keys + p.view.offset<kPaged>((row - p.q_dim) / HD, position) + i;
          } else {
            dst = p.view.values + p.view.offset<kPaged>((row - p.q_dim - kv_dim) / HD, position) + i;
          }
          dst[0] = float_to_elem(a);
          dst[HD / 2] = float_to_elem(b);
        }
      }
    }
  }
}

template <ShortOut kOut, bool kPaged, int FT>
void launch_tiles(ShortProjection p, int compute_units, hipStream_t s) {
  p.token_tiles = (p.tokens + 16 * FT - 1) / (16 * FT);
  p.lanes = p.k / kGemvBlock * p.token_tiles;
  // One block per compute unit (its ring fills the LDS), as many for each
  // (slice, token tile), in whole XCD rounds.
  const int per_xcd = std::max(1, std::min(p.rows / 128, compute_units / 8 / p.lanes));
  const unsigned blocks = static_cast<unsigned>(8 * per_xcd * p.lanes);
  short_projection_kernel<kOut, kPaged, FT><<<blocks, kShortThreads, 0, s>>>(p);
  HIP_CHECK_LAUNCH();
}

// 16 tokens per block while that leaves compute units without a tile, else 32
// (fewer reads and widenings of the weights).
template <ShortOut kOut, bool kPaged>
void launch_projection(const ShortProjection& p, int compute_units, hipStream_t s) {
  LCR_CHECK(p.rows % 128 == 0 && p.k % kGemvBlock == 0 && p.tokens > 0,
            "short projection of " << p.rows << " x " << p.k);
  if (p.rows / 16 * (p.k / kGemvBlock) * ((p.tokens + 15) / 16) > compute_units && p.tokens > 16) {
    launch_tiles<kOut, kPaged, 2>(p, compute_units, s);
  } else {
    launch_tiles<kOut, kPaged, 1>(p, compute_units, s);
  }
}

// ---------------------------------------------------------------------------
// Norms, into fragment order
// ---------------------------------------------------------------------------

// x = the embedding rows, normed = RMSNorm(x) * weight.
__global__ __launch_bounds__(kNormThreads) void short_embed_norm_kernel(elem_t* __restrict__ normed,
                                                                        elem_t* __restrict__ x,
                                                                        const elem_t* __restrict__ table,
                                                                        const int32_t* __restrict__ ids,
                                                                        const elem_t* __restrict__ weight,
                                                                        int tokens, float eps) {
  __shared__ float scratch[9];
  const int t = static_cast<int>(blockIdx.x);
  const elem_t* row = table + static_cast<size_t>(ids[t]) * kGemvBlock;
  elem_t* xrow = x + static_cast<size_t>(t) * kGemvBlock;
  const int c = static_cast<int>(threadIdx.x);  // a row is one chunk per thread
  store16(xrow + 8 * c, load16(row + 8 * c));
  norm_row_vec<false, 1>([&](int chunk) { return normed + short_fragment_index(8 * chunk, t, tokens); }, xrow, weight,
                         kGemvBlock, eps, [](int, float*) {}, scratch);
}

// x += the rounded sum of the projection's slices, left to right;
// normed = RMSNorm(x) * weight.
__global__ __launch_bounds__(kNormThreads) void short_residual_norm_kernel(elem_t* __restrict__ normed,
                                                                           elem_t* __restrict__ x,
                                                                           const float* __restrict__ partial,
                                                                           int slices,
                                                                           const elem_t* __restrict__ weight,
                                                                           int tokens, float eps) {
  __shared__ float scratch[9];
  const int t = static_cast<int>(blockIdx.x);
  const size_t base = static_cast<size_t>(t) * kGemvBlock;
  const size_t count = static_cast<size_t>(tokens) * kGemvBlock;
  norm_row_vec<true, 1>(
      [&](int chunk) { return normed + short_fragment_index(8 * chunk, t, tokens); }, x + base, weight, kGemvBlock,
      eps,
      [&](int c, float* df) {
        const float* at = partial + base + 8 * c;
        float sum[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) sum[j] = at[j];
        for (int sl = 1; sl < slices; ++sl) {
#pragma unroll
          for (int j = 0; j < 8; ++j) sum[j] += at[sl * count + j];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) df[j] = elem_to_float(float_to_elem(sum[j]));
      },
      scratch);
}

// ---------------------------------------------------------------------------
// Attention
// ---------------------------------------------------------------------------

// One block per (token, query head), in waves enough for the longest token's
// tiles up to eight; blocks of one kv head share an XCD when there are eight.
template <bool kPaged, int kWaves>
__global__ __launch_bounds__(64 * kWaves) void short_attention_kernel(elem_t* __restrict__ out,
                                                                      const elem_t* __restrict__ q, KvCacheView view,
                                                                      int num_heads, int tokens, int position,
                                                                      float scale) {
  constexpr int HD = 64;
  __shared__ AttnShared<kPaged, HD, 1, kWaves> sh;
  const int kv = static_cast<int>(blockIdx.x) % view.num_kv_heads;
  const int rest = static_cast<int>(blockIdx.x) / view.num_kv_heads;
  const int group = num_heads / view.num_kv_heads;
  const int head = kv * group + rest % group;
  const int t = rest / group;
  const size_t row = static_cast<size_t>(t) * num_heads * HD;
  decode_attention_block<kPaged, HD, 1, false, NoPreWait, kWaves>(
      sh, [&](int i) -> elem_t& { return out[short_fragment_index(i, t, tokens)]; }, nullptr, q + row, view, kv, head,
      0, 1, position + t + 1, scale);
}

template <bool kPaged>
void launch_attention(const ShortPromptArgs& a, const KvCacheView& view, hipStream_t s) {
  const unsigned blocks = static_cast<unsigned>(a.num_heads * a.tokens);
  const float scale = 1.0f / std::sqrt(static_cast<float>(a.head_dim));
  const int tiles = (a.position + a.tokens + kAttnTile - 1) / kAttnTile;
  if (tiles <= 1) {
    short_attention_kernel<kPaged, 1><<<blocks, 64, 0, s>>>(a.attn, a.q, view, a.num_heads, a.tokens, a.position,
                                                            scale);
  } else if (tiles <= 2) {
    short_attention_kernel<kPaged, 2><<<blocks, 128, 0, s>>>(a.attn, a.q, view, a.num_heads, a.tokens, a.position,
                                                             scale);
  } else if (tiles <= 4) {
    short_attention_kernel<kPaged, 4><<<blocks, 256, 0, s>>>(a.attn, a.q, view, a.num_heads, a.tokens, a.position,
                                                             scale);
  } else {
    short_attention_kernel<kPaged, kAttnWaves><<<blocks, kAttnThreads, 0, s>>>(a.attn, a.q, view, a.num_heads,
                                                                             a.tokens, a.position, scale);
  }
  HIP_CHECK_LAUNCH();
}

// The residual join of the chunk's last token, unrounded (the output head's
// input).
__global__ __launch_bounds__(256) void short_residual_kernel(float* __restrict__ resid, const elem_t* __restrict__ x,
                                                             const float* __restrict__ partial, int slices,
                                                             int tokens, int hidden) {
  const int i = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
  if (i >= hidden) return;
  const size_t at = static_cast<size_t>(tokens - 1) * hidden + i;
  float sum = partial[at];
  for (int s = 1; s < slices; ++s) sum += partial[static_cast<size_t>(s) * tokens * hidden + at];
  resid[i] = elem_to_float(x[at]) + elem_to_float(float_to_elem(sum));
}

}  // namespace

void enqueue_short_qkv_attention(const ShortPromptArgs& a, const LayerDevicePtrs& w, const KvCacheView& view,
                                 hipStream_t s) {
  LCR_CHECK(a.tokens > 0 && a.tokens <= kShortPromptMaxTokens, "short prompt of " << a.tokens << " tokens");
  ShortProjection p{};
  p.w = w.qkv;
  p.x = a.normed;
  p.out = a.q;
  p.rows = (a.num_heads + 2 * a.num_kv_heads) * a.head_dim;
  p.k = a.hidden;
  p.tokens = a.tokens;
  p.rope_table = a.rope_table;
  p.view = view;
  p.position = a.position;
  p.q_dim = a.num_heads * a.head_dim;
  if (a.paged) {
    launch_projection<ShortOut::kRope, true>(p, a.compute_units, s);
    launch_attention<true>(a, view, s);
  } else {
    launch_projection<ShortOut::kRope, false>(p, a.compute_units, s);
    launch_attention<false>(a, view, s);
  }
}

void enqueue_short_oproj(const ShortPromptArgs& a, const LayerDevicePtrs& w, hipStream_t s) {
  ShortProjection p{};
  p.w = w.o;
  p.x = a.attn;
  p.out = a.partial;
  p.rows = a.hidden;
  p.k = a.num_heads * a.head_dim;
  p.tokens = a.tokens;
  launch_projection<ShortOut::kPartial, false>(p, a.compute_units, s);
}

void enqueue_short_mlp(const ShortPromptArgs& a, const LayerDevicePtrs& w, hipStream_t s) {
  ShortProjection gate_up{};
  gate_up.w = w.gate_up;
  gate_up.x = a.normed;
  gate_up.out = a.act;
  gate_up.rows = 2 * a.ffn;
  gate_up.k = a.hidden;
  gate_up.tokens = a.tokens;
  ShortProjection down{};
  down.w = w.down;
  down.x = a.act;
  down.out = a.partial;
  down.rows = a.hidden;
  down.k = a.ffn;
  down.tokens = a.tokens;
  launch_projection<ShortOut::kSwiglu, false>(gate_up, a.compute_units, s);
  launch_projection<ShortOut::kPartial, false>(down, a.compute_units, s);
}

void enqueue_short_embed_norm(const ShortPromptArgs& a, const elem_t* table, const int32_t* ids,
                              const elem_t* weight, float eps, hipStream_t s) {
  LCR_CHECK(a.hidden == kGemvBlock, "short prompt norms are compiled for " << kGemvBlock << " columns");
  short_embed_norm_kernel<<<static_cast<unsigned>(a.tokens), kNormThreads, 0, s>>>(a.normed, a.x, table, ids, weight,
                                                                                   a.tokens, eps);
  HIP_CHECK_LAUNCH();
}

void enqueue_short_residual_norm(const ShortPromptArgs& a, const elem_t* weight, int slices, float eps,
                                 hipStream_t s) {
  LCR_CHECK(a.hidden == kGemvBlock, "short prompt norms are compiled for " << kGemvBlock << " columns");
  short_residual_norm_kernel<<<static_cast<unsigned>(a.tokens), kNormThreads, 0, s>>>(
      a.normed, a.x, a.partial, slices, weight, a.tokens, eps);
  HIP_CHECK_LAUNCH();
}

int short_down_slices(int ffn) { return ffn / kGemvBlock; }

void enqueue_short_residual(const ShortPromptArgs& a, float* resid, hipStream_t s) {
  short_residual_kernel<<<static_cast<unsigned>((a.hidden + 255) / 256), 256, 0, s>>>(
      resid, a.x, a.partial, short_down_slices(a.ffn), a.tokens, a.hidden);
  HIP_CHECK_LAUNCH();
}

}  // namespace lcr
