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
// Measured (us, keys and weights from memory; while every load had an address and a block-table exchange of its own, now):
// one request of 12 heads over 100, 250 and 540 keys 4.36 -> 3.63, 5.75 -> 4.71 and 8.31 -> 6.78, 8 requests 6.30 -> 5.10,
// 6.81 -> 6.15 and 10.06 -> 8.49, 16 over 540 keys 11.5 -> 10.7; 8 of 8 heads of 128 over 400 keys 11.8 -> 11.2.
// parts/attention.py says where the lines lie.
#include <math.h>

#include "attention_decode_block.h"
#include "common.h"
#include "pagedserve_hip.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

// STEPS: head_dim / 64; AHEAD: tiles of 16 columns per wave whose weights are asked for beside the keys
// (further ones follow behind the attention): right behind the first keys and values, or FIRST, in front of the
// attention, where they hold back the block table and with it the keys, but nothing of a wave's later turns
// (parts/attention.py says where the line lies).
template <int STEPS, int AD_WAVES, int AD_UNROLL, int AHEAD, bool FIRST>
__global__ __launch_bounds__(64 * AD_WAVES) void attention_decode_linear_kernel(
    const int* __restrict__ tables, const int* __restrict__ tok_pos, const bf16_t* __restrict__ q, int64_t q_stride,
    const bf16_t* __restrict__ wp, int table_width, int form, int heads, int n, int tiles_per_block, int kv_group,
    int page_size, int kv_heads, int num_pages, const bf16_t* __restrict__ k_pool, const bf16_t* __restrict__ v_pool,
    float scale_log2, int window, const float* __restrict__ bias, float* __restrict__ residual, int64_t ld_res,
    const AttnExtras extra) {
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
  float b[AHEAD];       // lane l < 16: the bias of column l of the tile (added by the blocks of head 0)
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
    if (bias != nullptr && head == 0) {
#pragma unroll
      for (int c = 0; c < AHEAD; ++c) {
        const int col = (first_tile + (round * AHEAD + c) * AD_WAVES + wave) * 16 + (lane & 15);
        b[c] = bias[col < n ? col : n - 1];
      }
    } else {
#pragma unroll
      for (int c = 0; c < AHEAD; ++c) b[c] = 0.f;
    }
  };

  auto attend = [&](auto ahead) {
    attention_decode_block<bf16_t, 8 * STEPS, AD_WAVES, AD_UNROLL, false>(
        lds, token, head, 0, q, q_stride, k_pool, v_pool, (bf16_t*)nullptr, 0, nullptr, nullptr, nullptr,
        tok_pos, tables, table_width, heads, kv_heads, kv_group,
        (form & 0xffff) | (HEAD_DIM << 16), page_size, num_pages,
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
        unsafeAtomicAdd(residual + (int64_t)token * ld_res + col, acc[0] + b[c]);
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
  const int tiles_per_block = (tiles_n + parts - 1) / parts;
  const int form = decode_form(head_dim, page_size, kv_heads, window == 0);
  const AttnExtras extra{sink, gate, gate_ld, softcap, logistic, logistic_norm};
  dim3 grid(count, heads, (tiles_n + tiles_per_block - 1) / tiles_per_block);
  hipStream_t s = (hipStream_t)stream;
#define PS_LAUNCH_ADL(STEPS, WAVES, UNROLL, AHEAD, FIRST)                                          \
  hipLaunchKernelGGL((attention_decode_linear_kernel<STEPS, WAVES, UNROLL, AHEAD, FIRST>), grid,   \
                     dim3(64 * WAVES), 0, s, tables, tok_pos, (const bf16_t*)q, q_stride,          \
                     (const bf16_t*)w_packed, table_width, form, heads, n, tiles_per_block,        \
                     heads / kv_heads, page_size, kv_heads, num_pages, (const bf16_t*)k_pool,      \
                     (const bf16_t*)v_pool, scale * 1.4426950408889634f, window, bias, residual,   \
                     ld_res, extra)
  // (sixteen waves leave a wave 128 registers, too few for the keys and the weights of a turn: over 800 keys 8 requests of
  // 12 heads 12.3 us, with eight waves and two turns 10.8.  Who asks for them gets eight.)
  if (head_dim == 64) {
    if (waves == 4 && weights_first) PS_LAUNCH_ADL(1, 4, 4, 4, true);
    else if (waves == 4) PS_LAUNCH_ADL(1, 4, 4, 4, false);
    else PS_LAUNCH_ADL(1, 8, 8, 4, false);
  } else {
    if (waves == 4) PS_LAUNCH_ADL(2, 4, 4, 4, false);
    else PS_LAUNCH_ADL(2, 8, 8, 4, false);
  }
#undef PS_LAUNCH_ADL
  PS_CHECK_LAUNCH("ps_attention_decode_linear");
  return 0;
}
