// Paged attention of items with several tokens (prompt portions) in true 32-bit.
//
// A block of four waves per (32 queries, head); the waves take the request's keys 32 at a time in turn, each
// with a softmax of its own that runs online in float with the library's expf (reference:
// src/kernels/triton_paged_attention.py:219-223,275-331), and the four results are merged through LDS at the end.
// Scores and weighted values are v_mfma_f32_32x32x2_f32: true 32-bit products and sums.
//
// The scores are made transposed (keys x queries), so that a lane holds 16 keys of one query: the softmax
// needs one exchange with the lane of the other half, its correction is one factor per lane, and the
// probabilities are, where they lie, the operand of the product with the values (also transposed:
// dimensions x queries), since instruction e takes keys 8 (e / 4) + e % 4 + {0, 4} from the lane halves.
// Keys and values come straight from their pages into registers, a row of a key in pieces of 16 bytes,
// a value 128 bytes of a row at a time; the next tile's keys are on their way during softmax and values,
// its values during the scores.
//
// What bounds it: a tile of 32 x 32 at 64 dimensions is 64 matrix instructions of 64 cycles beside some 800
// others, 4.5 us for a wave alone on its SIMD; a portion of a few hundred tokens is a dozen blocks per head, so
// that what counts is the longest chain.  With tiles of 64 queries, plain multiply-adds and one run over the
// keys per block a portion of 300 tokens at 12 heads of 64 took 55 us, now 17; 512 tokens 86 and 21, 2 x 1,024
// tokens 179 and 64 (a third of the time the matrix cores are busy).
//
// The tiles are those of the bfloat16 kernel (`tile_item`, `tile_q0`: the item of each tile and its first query within
// the item's tokens of this step), of 32 queries or of 64, which are two blocks or one (ops/kernels.py says where), and so
// are the rules: query i of an
// item whose cached length after the step is L and which brings n tokens stands at position
// L - n + i and sees keys first_visible_key(position, window) .. position.
//
// Head sizes that are multiples of 4 up to 128; others stay with the one-wave-per-token
// kernel.
#include <math.h>

#include "common.h"
#include "pagedserve_hip.h"

#define AF_TILE 64       // queries of a listed tile
#define AF_ROWS 32       // queries of a block, and keys per turn of a wave's loop
#define AF_WAVES 4
#define AF_MAX_DIM 128

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float af_f32x4;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float af_f32x16;

// DF: 32 head dimensions each; RAGGED: the head size is not 32 DF; PAIRS: one block takes the 64 queries of a tile,
// two waves to 32 of them; `parts`: else, blocks to a listed tile (of 32 queries each)
template <int DF, bool RAGGED, bool PAIRS>
__global__ __launch_bounds__(64 * AF_WAVES) void attention_tiled_f32_kernel(
    const float* __restrict__ q, int64_t q_stride, const float* __restrict__ k_pool,
    const float* __restrict__ v_pool, float* __restrict__ out, int64_t out_stride,
    const int* __restrict__ tile_item, const int* __restrict__ tile_q0,
    const int* __restrict__ cu_tokens, const int* __restrict__ kv_lens,
    const int* __restrict__ tables, int table_width, int heads, int kv_heads, int head_dim,
    int page_size, int num_pages, float scale, int window, int parts, const AttnExtras extra) {
  constexpr int STEPS = 4 * DF;                 // pieces of 2 x 4 dimensions of a score
  constexpr int STRIDE = 32 * DF + 4;           // floats from query to query of a wave's result
  __shared__ __attribute__((aligned(16))) float s_out[AF_WAVES * AF_ROWS * STRIDE];
  __shared__ float s_max[AF_WAVES * AF_ROWS], s_sum[AF_WAVES * AF_ROWS];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int column = lane & 31;                 // the lane's query, and its key when keys are read
  const int half = lane >> 5;
  // (the lists begin with the tiles that see the most keys, and so do the blocks, the later half of a tile first: with the
  // longest at the end prompts of 500, 20, 35, 800 and 64 tokens at 16 heads of 64 take 56 us, this way 40)
  const int index = blockIdx.x;
  const int tile_index = index / (parts * heads);
  const int part = parts - 1 - (index - tile_index * parts * heads) / heads;   // which 32 queries of the listed tile
  const int head = index % heads;
  const int kv_head = head / (heads / kv_heads);

  const int item = tile_item[tile_index];
  const int tile_q = tile_q0[tile_index];
  const int tok0 = cu_tokens[item];
  const int count = cu_tokens[item + 1] - tok0;
  const int start = kv_lens[item] - count;      // position of the portion's first token
  const int* table = tables + (int64_t)item * table_width;
  constexpr int TURNS = PAIRS ? 2 : AF_WAVES;   // waves that share the keys of 32 queries
  const int turn = PAIRS ? wave & 1 : wave;     // which of them this one is
  const int first_q = tile_q + part * AF_ROWS;  // of the block
  if (first_q >= count) return;                 // (the whole block)
  const int q0 = PAIRS ? first_q + (wave >> 1) * AF_ROWS : first_q;
  const int last_q = q0 + AF_ROWS - 1 < count ? q0 + AF_ROWS - 1 : count - 1;
  const int key_begin = first_visible_key(start + q0, window);
  const int key_end = q0 < count ? start + last_q + 1 : key_begin;

  const int q_pos = q0 + column < count ? start + q0 + column : -1;
  const int q_first = q_pos < 0 ? 0 : first_visible_key(q_pos, window);

  // the lane's query: dimensions 8 s + 4 half ..; rows beyond the item's tokens are zeros and never stored
  af_f32x4 query[STEPS];
#pragma unroll
  for (int s = 0; s < STEPS; ++s) {
    const int dim = 8 * s + 4 * half;
    query[s] = af_f32x4{0.f, 0.f, 0.f, 0.f};
    if (q_pos >= 0 && (!RAGGED || dim < head_dim))
      query[s] = *reinterpret_cast<const af_f32x4*>(q + (int64_t)(tok0 + q0 + column) * q_stride +
                                                    (int64_t)head * head_dim + dim);
  }

  // The page of key k0 + column as the table names it (read without a branch: a wait for it then leaves the
  // loads behind it on their way), and the first value of the key's row in the pools, or -1.
  auto page_of = [&](int k0) {
    const int logical = (k0 + column) / page_size;
    return table[logical < table_width ? logical : table_width - 1];
  };
  auto row_of = [&](int k0, int page) -> int64_t {
    const int key = k0 + column;
    const int logical = key / page_size;
    const bool there = key < key_end && logical < table_width && page >= 0 && page < num_pages;
    const int64_t row = (((int64_t)page * kv_heads + kv_head) * page_size + (key - logical * page_size)) * head_dim;
    return there ? row : -1;
  };
  af_f32x4 key_values[STEPS];
  float values[DF][16];
  // (rows that are not there are read from the pool's first row and not used)
  auto load_keys = [&](int64_t row) {
    const float* source = k_pool + (row < 0 ? 0 : row);
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const int dim = 8 * s + 4 * half;
      key_values[s] = *reinterpret_cast<const af_f32x4*>(source + (!RAGGED || dim < head_dim ? dim : 0));
    }
  };
  auto load_values = [&](int64_t row) {
    const int64_t from = row < 0 ? 0 : row;
    const int low = (int)from, high = (int)(from >> 32);
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      // key 8 (e / 4) + e % 4 for the lower half of the lanes, four further on for the upper one
      const int key = (e >> 2) * 8 + (e & 3);
      const int low_0 = __builtin_amdgcn_readlane(low, key), low_1 = __builtin_amdgcn_readlane(low, key + 4);
      const int high_0 = __builtin_amdgcn_readlane(high, key), high_1 = __builtin_amdgcn_readlane(high, key + 4);
      const int64_t base = ((int64_t)(half ? high_1 : high_0) << 32) | (unsigned int)(half ? low_1 : low_0);
#pragma unroll
      for (int f = 0; f < DF; ++f) {
        const int dim = 32 * f + column;
        values[f][e] = v_pool[base + (!RAGGED || dim < head_dim ? dim : 0)];
      }
    }
  };

  // (a sink is a score without key or value: it starts the denominator, in one lane half of one wave)
  const bool starts = turn == 0 && extra.sink != nullptr;
  float run_max = starts ? extra.sink[head] : -INFINITY;
  float run_sum = starts && half == 0 ? 1.f : 0.f;     // of the lane's own keys
  af_f32x16 acc[DF];
#pragma unroll
  for (int f = 0; f < DF; ++f)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[f][e] = 0.f;

  int k0 = key_begin + turn * AF_ROWS;
  if (k0 < key_end) {
    constexpr int TURN = TURNS * AF_ROWS;
    int64_t row = row_of(k0, page_of(k0));
    load_keys(row);
    int next_page = page_of(k0 + TURN);
    load_values(row);
    for (; k0 < key_end; k0 += TURN) {
      // two chains of half the length: no instruction waits for the one before, half the rounding
      af_f32x16 sums[2];
#pragma unroll
      for (int e = 0; e < 16; ++e) sums[0][e] = sums[1][e] = 0.f;
#pragma unroll
      for (int s = 0; s < STEPS; ++s) {
        af_f32x4 piece = key_values[s];
        if (RAGGED && 8 * s + 4 * half >= head_dim) piece = af_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i)
          sums[i & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(piece[i], query[s][i], sums[i & 1], 0, 0, 0);
      }
      const int64_t next_row = row_of(k0 + TURN, next_page);
      load_keys(next_row);
      next_page = page_of(k0 + 2 * TURN);
      __builtin_amdgcn_sched_barrier(0);   // (these loads stay in front of the softmax)

      // the lane's 16 scores: query `column`, keys k0 + 8 (e / 4) + 4 half + e % 4
      const unsigned long long there = __ballot(row >= 0);
      float p[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) p[e] = (sums[0][e] + sums[1][e]) * scale;
      if (extra.softcap > 0.f) {
#pragma unroll
        for (int e = 0; e < 16; ++e) p[e] = capped_score(p[e], extra.softcap);
      }
      const unsigned int mine = (unsigned int)(there >> (4 * half));
      float tile_max = -INFINITY;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int offset = (e >> 2) * 8 + (e & 3);
        const int key = k0 + 4 * half + offset;
        const bool visible = ((mine >> offset) & 1u) != 0 && key <= q_pos && key >= q_first;
        p[e] = visible ? p[e] : -INFINITY;
        tile_max = fmaxf(tile_max, p[e]);
      }
      if (extra.logistic != nullptr) {
        const float shift = extra.logistic[head];
#pragma unroll
        for (int e = 0; e < 16; ++e) p[e] = 1.0f / (1.0f + expf(-(p[e] + shift)));   // 0 where p is -inf
      } else {
        tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 32));
        const float new_max = fmaxf(run_max, tile_max);
        // new_max is -inf only while no key has been visible: zeros then
        const float base = new_max == -INFINITY ? 0.f : new_max;
        const float correction = expf(run_max - base);
        float tile_sum = 0.f;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          p[e] = expf(p[e] - base);
          tile_sum += p[e];
        }
        run_sum = run_sum * correction + tile_sum;
        run_max = new_max;
#pragma unroll
        for (int f = 0; f < DF; ++f)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[f][e] *= correction;
      }
      if (there != ~0ull) {
        // (nothing of rows that are not there: a weight of zero would keep what is not a number)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const bool here = ((mine >> ((e >> 2) * 8 + (e & 3))) & 1u) != 0;
#pragma unroll
          for (int f = 0; f < DF; ++f) values[f][e] = here ? values[f][e] : 0.f;
        }
      }
#pragma unroll
      for (int e = 0; e < 16; ++e)
#pragma unroll
        for (int f = 0; f < DF; ++f)
          acc[f] = __builtin_amdgcn_mfma_f32_32x32x2f32(values[f][e], p[e], acc[f], 0, 0, 0);
      load_values(next_row);
      row = next_row;
    }
  }

  // ---- the four waves' results: dimension 32 f + 8 (e / 4) + 4 half + e % 4 of query `column`
  run_sum += __shfl_xor(run_sum, 32);
  float* mine = s_out + (wave * AF_ROWS + column) * STRIDE;
#pragma unroll
  for (int f = 0; f < DF; ++f)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<float4*>(mine + 32 * f + 8 * g + 4 * half) =
          make_float4(acc[f][4 * g], acc[f][4 * g + 1], acc[f][4 * g + 2], acc[f][4 * g + 3]);
  if (half == 0) {
    s_max[wave * AF_ROWS + column] = run_max;
    s_sum[wave * AF_ROWS + column] = run_sum;
  }
  __syncthreads();
  // eight threads to a query, four where the block has 64 of them
  constexpr int SHARE = PAIRS ? 4 : 8;
  const int row = tid / SHARE;
  const int first = PAIRS ? (row >> 5) * 2 * AF_ROWS + (row & 31) : row;   // the query in its first wave's results
  if (first_q + row >= count) return;
  float total_max = -INFINITY;
#pragma unroll
  for (int w = 0; w < TURNS; ++w) total_max = fmaxf(total_max, s_max[w * AF_ROWS + first]);
  float factor[TURNS], total = 0.f;
#pragma unroll
  for (int w = 0; w < TURNS; ++w) {
    const float wave_max = s_max[w * AF_ROWS + first];
    factor[w] = wave_max == -INFINITY ? 0.f : expf(wave_max - total_max);
    total += s_sum[w * AF_ROWS + first] * factor[w];
  }
  if (extra.logistic != nullptr) {
#pragma unroll
    for (int w = 0; w < TURNS; ++w) factor[w] = 1.f;
    total = extra.logistic_norm;
  }
  const float inverse = (total != 0.f ? 1.f / total : 0.f) * gate_factor(extra, tok0 + first_q + row, head);
  float* to = out + (int64_t)(tok0 + first_q + row) * out_stride + (int64_t)head * head_dim;
#pragma unroll
  for (int v = 0; v < 8 * DF / SHARE; ++v) {
    const int dim = 4 * (tid % SHARE) + 4 * SHARE * v;
    if (RAGGED && dim >= head_dim) continue;
    float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int w = 0; w < TURNS; ++w) {
      const float4 value = *reinterpret_cast<const float4*>(s_out + (w * AF_ROWS + first) * STRIDE + dim);
      sum.x = fmaf(factor[w], value.x, sum.x);
      sum.y = fmaf(factor[w], value.y, sum.y);
      sum.z = fmaf(factor[w], value.z, sum.z);
      sum.w = fmaf(factor[w], value.w, sum.w);
    }
    *reinterpret_cast<float4*>(to + dim) =
        make_float4(sum.x * inverse, sum.y * inverse, sum.z * inverse, sum.w * inverse);
  }
}

extern "C" int ps_attention_tiled_f32_supported(int head_dim) {
  return head_dim >= 4 && head_dim <= AF_MAX_DIM && head_dim % 4 == 0;
}

extern "C" int ps_attention_tiled_f32_tile() { return AF_TILE; }

extern "C" int ps_attention_tiled_f32(const void* q, int64_t q_stride, const void* k_pool,
                                      const void* v_pool, void* out, int64_t out_stride,
                                      const int* tile_item, const int* tile_q0, int tiles,
                                      const int* cu_tokens, const int* kv_lens, const int* tables,
                                      int table_width, int heads, int kv_heads, int head_dim,
                                      int page_size, int num_pages, float scale, int window,
                                      const float* sink, const float* gate, int64_t gate_ld,
                                      float softcap, const float* logistic, float logistic_norm,
                                      int query_tile, int paired, void* stream) {
  PS_REQUIRE(tiles >= 0 && heads > 0 && kv_heads > 0 && page_size > 0 && num_pages > 0 &&
                 table_width > 0,
             "ps_attention_tiled_f32: bad sizes");
  PS_REQUIRE(ps_attention_tiled_f32_supported(head_dim),
             "ps_attention_tiled_f32: head_dim %d must be a multiple of 4 up to %d "
             "(ps_attention_rowwise takes every size)", head_dim, AF_MAX_DIM);
  PS_REQUIRE(heads % kv_heads == 0,
             "ps_attention_tiled_f32: heads (%d) must be a multiple of kv_heads (%d)", heads, kv_heads);
  PS_REQUIRE(scale > 0.f, "ps_attention_tiled_f32: the score scale must be positive, got %g", scale);
  PS_REQUIRE((q_stride % 4) == 0 && (out_stride % 4) == 0 && ((uintptr_t)q % 16) == 0 &&
                 ((uintptr_t)out % 16) == 0 && ((uintptr_t)k_pool % 16) == 0 &&
                 ((uintptr_t)v_pool % 16) == 0,
             "ps_attention_tiled_f32: rows of q, out and the pools must allow 16-byte accesses");
  PS_REQUIRE(query_tile == AF_TILE || query_tile == AF_ROWS,
             "ps_attention_tiled_f32: tiles of %d or %d queries, not %d", AF_TILE, AF_ROWS, query_tile);
  PS_REQUIRE(!paired || query_tile == AF_TILE, "ps_attention_tiled_f32: one block takes a tile of %d queries, not of %d",
             AF_TILE, query_tile);
  const int parts = paired ? 1 : query_tile / AF_ROWS;
  const int64_t blocks = (int64_t)tiles * heads * parts;
  PS_REQUIRE(blocks < ((int64_t)1 << 31), "ps_attention_tiled_f32: too many blocks");
  if (blocks == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const AttnExtras extra = {sink, gate, gate_ld, softcap, logistic, logistic_norm};
#define PS_LAUNCH_AF(DF)                                                                          \
  do {                                                                                            \
    if (head_dim == 32 * DF && paired) PS_LAUNCH_AF_FORM(DF, false, true);                        \
    else if (head_dim == 32 * DF) PS_LAUNCH_AF_FORM(DF, false, false);                            \
    else if (paired) PS_LAUNCH_AF_FORM(DF, true, true);                                           \
    else PS_LAUNCH_AF_FORM(DF, true, false);                                                      \
  } while (0)
#define PS_LAUNCH_AF_FORM(DF, RAGGED, PAIRS)                                                      \
  hipLaunchKernelGGL((attention_tiled_f32_kernel<DF, RAGGED, PAIRS>), dim3((unsigned)blocks),     \
                     dim3(64 * AF_WAVES), 0, s,                                                   \
                     (const float*)q, q_stride, (const float*)k_pool, (const float*)v_pool,       \
                     (float*)out, out_stride, tile_item, tile_q0, cu_tokens, kv_lens, tables,     \
                     table_width, heads, kv_heads, head_dim, page_size, num_pages, scale, window, parts, extra)
  switch ((head_dim + 31) / 32) {
    case 1: PS_LAUNCH_AF(1); break;
    case 2: PS_LAUNCH_AF(2); break;
    case 3: PS_LAUNCH_AF(3); break;
    default: PS_LAUNCH_AF(4); break;
  }
#undef PS_LAUNCH_AF_FORM
#undef PS_LAUNCH_AF
  PS_CHECK_LAUNCH("ps_attention_tiled_f32");
  return 0;
}
