// Decode attention and output projection in one launch, for steps of up to 64 single-token items
// over contexts of some hundreds of keys (bfloat16, heads of 64 or 128):
//
//   residual[t, :] += concat_h(attention of head h of token t) W^T + bias
//
// As two launches each of them is a chain of trips to memory: position and block table, keys and values,
// the exchange between the waves; then the rows of the context, the weights, the exchange, the add.  The
// second chain mostly repeats waits of the first.  Here block (t, h, p) computes head h of token t over all
// its keys (attention_decode_block.h) and multiplies it with the piece of W that belongs to head h
// and to the p-th part of the columns, out of the packed copy of W (pagedserve_hip.h).  The piece is asked for
// beside the keys and travels with them.  Blocks that differ in p repeat the attention: while the keys are few that costs
// less than leaving compute units idle, since a unit takes in some 55 KB/us and what it has to take in (its
// keys and its piece of W) is what the launch waits for beside the chain.  The sum over heads is made
// by float atomic adds into the residual rows, in an order that differs from run to run within float
// rounding, as for every product here whose k range is split over blocks.
//
// One row of the matrix core's operand holds the head's context, the other fifteen are zero: the
// instructions are few and free beside the loads, and with the context as row operand the sixteen
// results of a tile lie in sixteen consecutive lanes, whose adds fall into one 64-byte piece.
//
// Measured (us, keys and weights from memory, attention + projection in two launches before): one request of
// 12 heads over 144 keys 8.6 -> 5.9, 8 over 540 keys 13.6 -> 10.5, 16 over 540 keys 16.4 -> 12.3; 8 of 16
// heads over 270 keys 11.8 -> 9.8.  parts/attention.py says where the lines lie.
#include <math.h>

#include "attention_decode_block.h"
#include "common.h"
#include "pagedserve_hip.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

// STEPS: head_dim / 64; AHEAD: tiles of 16 columns per wave whose weights are asked for beside the keys
// (further ones follow behind the attention): right behind the first keys and values, or FIRST, in front of the
// attention, where they hold back the block table and with it the keys, but nothing of a wave's later turns
// (parts/attention.py says where the line lies).  Heads of 128 hold twice the weights, which the first turn over the keys has
// no registers left for (16 waves spill 16 of them; 8 requests of 8 heads over 250 keys 9.5 us with the weights in front,
// 11.7 behind; one of 16 heads over 400 keys 10.6 and 12.1): always in front.
template <int STEPS, int AD_WAVES, int AD_UNROLL, int AHEAD, bool FIRST>
__global__ __launch_bounds__(64 * AD_WAVES) void attention_decode_linear_kernel(
    const bf16_t* __restrict__ q, int64_t q_stride, const bf16_t* __restrict__ k_pool,
    const bf16_t* __restrict__ v_pool, const int* __restrict__ tok_pos,
    const int* __restrict__ tables, int table_width, int heads, int kv_heads, int page_size,
    int page_shift, int num_pages, float scale_log2, int window, const AttnExtras extra,
    const bf16_t* __restrict__ wp, const float* __restrict__ bias, float* __restrict__ residual,
    int64_t ld_res, int n, int tiles_per_block) {
  constexpr int HEAD_DIM = STEPS * 64;
  __shared__ DecodeLds<AD_WAVES> lds;
  __shared__ __attribute__((aligned(16))) bf16_t context[HEAD_DIM];
  const int token = blockIdx.x;
  const int head = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // the same in every lane: scalar
  const int tiles_n = (n + 15) / 16;
  const int first_tile = blockIdx.z * tiles_per_block;
  const int end_tile = first_tile + tiles_per_block < tiles_n ? first_tile + tiles_per_block : tiles_n;

  // element ((tile * k_steps + step) * 2 + h) * 512 + lane * 8 of the packed copy
  const int k_steps = heads * STEPS;
  const bf16_t* w_head = wp + (int64_t)head * STEPS * 1024 + lane * 8;
  uint4 w_raw[AHEAD][STEPS][2];
  auto load_weights = [&](int round) {
#pragma unroll
    for (int c = 0; c < AHEAD; ++c) {
      int tile = first_tile + (round * AHEAD + c) * AD_WAVES + wave;
      if (tile >= end_tile) tile = end_tile - 1;      // never stored
      const bf16_t* w_tile = w_head + (int64_t)tile * k_steps * 1024;
#pragma unroll
      for (int st = 0; st < STEPS; ++st)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          w_raw[c][st][h] = *reinterpret_cast<const uint4*>(w_tile + (st * 2 + h) * 512);
    }
  };

  auto attend = [&](auto ahead) {
    attention_decode_block<bf16_t, 8 * STEPS, AD_WAVES, AD_UNROLL, false>(
        lds, token, head, 0, q, q_stride, k_pool, v_pool, (bf16_t*)nullptr, 0, nullptr, nullptr, nullptr,
        tok_pos, tables, table_width, heads, kv_heads, HEAD_DIM, page_size, page_shift, num_pages,
        scale_log2, window, 1, extra, context, ahead);
  };
  if constexpr (FIRST) {
    load_weights(0);
    attend(NothingAhead());
  } else {
    attend([&] { load_weights(0); });
  }
  __syncthreads();

  // row operand: row 0 is the head's context, the other fifteen are zero; lane l holds row l % 16,
  // k values 64 st + 16 (l / 16) + 8 h ..., the order of the packed copy
  bf16x8 x[STEPS][2];
#pragma unroll
  for (int st = 0; st < STEPS; ++st)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint4 raw = *reinterpret_cast<const uint4*>(context + st * 64 + (lane >> 4) * 16 + h * 8);
      const uint4 zero = {0u, 0u, 0u, 0u};
      x[st][h] = __builtin_bit_cast(bf16x8, (lane & 15) == 0 ? raw : zero);
    }
  const int rounds = (end_tile - first_tile + AHEAD * AD_WAVES - 1) / (AHEAD * AD_WAVES);
  for (int round = 0; round < rounds; ++round) {
    if (round > 0) load_weights(round);
#pragma unroll
    for (int c = 0; c < AHEAD; ++c) {
      const int tile = first_tile + (round * AHEAD + c) * AD_WAVES + wave;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int st = 0; st < STEPS; ++st)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[st][h], __builtin_bit_cast(bf16x8, w_raw[c][st][h]),
                                                        acc, 0, 0, 0);
      // row 0 of the tile lies in the first element of lanes 0 to 15, a column each
      const int col = tile * 16 + lane;
      if (tile < end_tile && lane < 16 && col < n) {
        float v = acc[0];
        if (head == 0 && bias != nullptr) v += bias[col];
        unsafeAtomicAdd(residual + (int64_t)token * ld_res + col, v);
      }
    }
  }
}

extern "C" int ps_attention_decode_linear(const void* q, int64_t q_stride, const void* k_pool,
                                          const void* v_pool, const int* tok_pos, const int* tables,
                                          int table_width, int count, int heads, int kv_heads,
                                          int head_dim, int page_size, int num_pages, float scale,
                                          int window, const float* sink, const float* gate,
                                          int64_t gate_ld, float softcap, const float* logistic,
                                          float logistic_norm, const void* w_packed,
                                          const float* bias, float* residual, int64_t ld_res, int n,
                                          int parts, int waves, int weights_first, void* stream) {
  PS_REQUIRE(count >= 0 && count <= 64 && heads > 0 && heads <= 65535 && kv_heads > 0 &&
                 heads % kv_heads == 0 && page_size > 0 && num_pages > 0 && table_width > 0,
             "ps_attention_decode_linear: bad sizes (count %d, heads %d, kv_heads %d)", count, heads,
             kv_heads);
  PS_REQUIRE(head_dim == 64 || head_dim == 128,
             "ps_attention_decode_linear: heads of 64 or 128, not %d", head_dim);
  PS_REQUIRE(n > 0 && ld_res >= n, "ps_attention_decode_linear: residual rows shorter than %d columns", n);
  const int tiles_n = (n + 15) / 16;
  PS_REQUIRE(parts >= 1 && parts <= tiles_n && parts <= 65535,
             "ps_attention_decode_linear: %d parts of %d tiles of columns", parts, tiles_n);
  PS_REQUIRE(waves == 4 || waves == 8 || waves == 16,
             "ps_attention_decode_linear: blocks have 4, 8 or 16 waves, not %d", waves);
  PS_REQUIRE(q && k_pool && v_pool && tok_pos && tables && w_packed && residual &&
                 (reinterpret_cast<uintptr_t>(w_packed) & 15u) == 0,
             "ps_attention_decode_linear: null or unaligned operand");
  if (count == 0) return 0;
  int page_shift = -1;
  if ((page_size & (page_size - 1)) == 0) {
    page_shift = 0;
    while ((1 << page_shift) < page_size) ++page_shift;
  }
  const int tiles_per_block = (tiles_n + parts - 1) / parts;
  const AttnExtras extra{sink, gate, gate_ld, softcap, logistic, logistic_norm};
  dim3 grid(count, heads, (tiles_n + tiles_per_block - 1) / tiles_per_block);
  hipStream_t s = (hipStream_t)stream;
#define PS_LAUNCH_ADL(STEPS, WAVES, UNROLL, AHEAD, FIRST)                                          \
  hipLaunchKernelGGL((attention_decode_linear_kernel<STEPS, WAVES, UNROLL, AHEAD, FIRST>), grid,   \
                     dim3(64 * WAVES), 0, s, (const bf16_t*)q, q_stride, (const bf16_t*)k_pool,    \
                     (const bf16_t*)v_pool, tok_pos, tables, table_width, heads, kv_heads,         \
                     page_size, page_shift, num_pages, scale * 1.4426950408889634f, window, extra, \
                     (const bf16_t*)w_packed, bias, residual, ld_res, n, tiles_per_block)
  if (head_dim == 64) {
    // (eight waves are behind with the weights in front everywhere)
    if (waves == 4 && weights_first) PS_LAUNCH_ADL(1, 4, 4, 4, true);
    else if (waves == 4) PS_LAUNCH_ADL(1, 4, 4, 4, false);
    else if (waves == 8) PS_LAUNCH_ADL(1, 8, 8, 4, false);
    else if (weights_first) PS_LAUNCH_ADL(1, 16, 8, 3, true);
    else PS_LAUNCH_ADL(1, 16, 8, 3, false);
  } else {
    if (waves == 4) PS_LAUNCH_ADL(2, 4, 4, 4, true);
    else if (waves == 8) PS_LAUNCH_ADL(2, 8, 8, 4, true);
    else PS_LAUNCH_ADL(2, 16, 8, 2, true);
  }
#undef PS_LAUNCH_ADL
  PS_CHECK_LAUNCH("ps_attention_decode_linear");
  return 0;
}
