// What the tiled products share: vector types, a step of the matrix cores, the fast GELU of a
// bfloat16 result, and the epilogue that takes a wave's 32 x 32 accumulators to memory.
#pragma once

#include "common.h"
#include "linear.h"
#include "pagedserve_hip.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;

#define TB_BK 64     // bfloat16 values of k per stage
#define TB_ROW 128   // bytes per row and stage

typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4_t;

// One step of the matrix cores on 16 bytes of k per lane, into ACCS accumulators whose sum is the
// result.  bfloat16: the operand of one v_mfma_f32_32x32x16_bf16.  float: the four values feed four
// v_mfma_f32_32x32x2_f32, true 32-bit products and sums (both operands use the same assignment of k
// to lanes and instructions, which is all a dot product needs), which take turns in the accumulators:
// with four of them the chains are a quarter as long and have half the rounding error, and no
// instruction waits for the one before.
template <int ACCS>
__device__ inline void mma_step(bf16_t, const u32x4_t& a, const u32x4_t& w, f32x16 (&acc)[ACCS]) {
  static_assert(ACCS == 1, "one instruction per step");
  acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, w), acc[0], 0, 0, 0);
}
template <int ACCS>
__device__ inline void mma_step(float, const u32x4_t& a, const u32x4_t& w, f32x16 (&acc)[ACCS]) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    acc[i % ACCS] = __builtin_amdgcn_mfma_f32_32x32x2f32(
        __builtin_bit_cast(float, (uint32_t)a[i]), __builtin_bit_cast(float, (uint32_t)w[i]),
        acc[i % ACCS], 0, 0, 0);
}

typedef const __attribute__((address_space(1))) void* global_ptr_t;
typedef __attribute__((address_space(3))) void* lds_ptr_t;

// gelu_tanh(u) = u * sigmoid(2 z), z = sqrt(2/pi) (u + 0.044715 u^3), with the hardware
// exponential: its error (about 1e-6 relative) is far below the rounding of a bfloat16 result, which is the
// only place where it is used.  The reciprocal is the hardware's and one step of Newton's method, four instructions
// where a division takes ten (a tile of 256 x 256 spent 17 us in this function with that); the two agree for every d up to
// 2^126, beyond it this one is 0 where the division's is subnormal.  Where d is infinite, the step is no number
// without the maximum, with it the reciprocal stays 0.
__device__ inline float gelu_tanh_fast(float u) {
  const float z2 = 1.5957691216057308f * (u + 0.044715f * u * u * u);
  const float d = 1.0f + __expf(-z2);
  const float r = __builtin_amdgcn_rcpf(d);
  const float e = fmaxf(fmaf(-d, r, 1.0f), -1.0f);
  return u * fmaf(r, e, r);
}

template <int EPI, typename TOut>
__device__ inline float finish_value(float v) {
  if (EPI == PS_EPI_GELU_TANH && sizeof(TOut) == 2) return gelu_tanh_fast(v);
  return apply_activation<EPI>(v);
}

// Eight finished values to eight consecutive outputs (16-byte aligned).
__device__ inline void store8(float* out, const float* v) {
  *reinterpret_cast<float4*>(out) = make_float4(v[0], v[1], v[2], v[3]);
  *reinterpret_cast<float4*>(out + 4) = make_float4(v[4], v[5], v[6], v[7]);
}
__device__ inline void store8(bf16_t* out, const float* v) {
  uint4 packed;
  packed.x = pack2_bf16(v[0], v[1]);
  packed.y = pack2_bf16(v[2], v[3]);
  packed.z = pack2_bf16(v[4], v[5]);
  packed.w = pack2_bf16(v[6], v[7]);
  *reinterpret_cast<uint4*>(out) = packed;
}

// The accumulators acc[WM][WN] of one wave (32 x 32 each, rows row_base + 32 i ..., columns
// col_base + 32 j ...) to C, through `region`, an area of LDS of 32 x (32 WN + 8) floats that
// belongs to this wave alone: bias, activation, residual add into the float stream, key/value
// columns into cache pages.  `split` / `k_splits`: partial sums of a k range are added with
// atomics, the bias by split 0 only.
template <int WM, int WN, typename TOut, int EPI>
__device__ inline void store_wave_tile(f32x16 (&acc)[WM][WN], float* region, int lane, int row_base,
                                       int col_base, int m, int n, int ldc, TOut* __restrict__ c,
                                       const float* __restrict__ bias, int split, int k_splits,
                                       const KvScatter& scatter) {
  // ---- epilogue.  Element e of a 32 x 32 accumulator is row (e / 4) * 8 + (lane / 32) * 4 +
  // e % 4, column lane % 32: a lane holds one column.  Each wave turns 32 rows at a time
  // through a region of LDS of its own, after which a lane holds eight consecutive columns of
  // one row: bias and activation are applied there and rows leave in pieces of 16 or 32
  // bytes, eight (or more) lanes to a row.
  constexpr int EP_STRIDE = WN * 32 + 8;          // floats; 4 rows further is 32 banks further
  constexpr int EP_CHUNKS = WN * 4;               // pieces of eight columns per row
  constexpr int EP_ROWS = 64 / EP_CHUNKS;         // rows per pass of the wave
  // The callers read operands by assembly and wait for them just in front of this.  What is worked out of the lane here
  // must not be moved in front of that wait, into a register that such a read may still be filling.
  asm volatile("" : "+v"(lane));
  const int chunk = lane % EP_CHUNKS;
  const int row_in_pass = lane / EP_CHUNKS;
  // The piece that the end of the rows lies in begins further left where that is aligned and within the wave's columns
  // (float rows of whole fours): both pieces then write the same values to the columns that they share.
  const bool reaches_back = sizeof(TOut) == 4 && (n & 3) == 0 && n - col_base >= 8;
  const int first = col_base + chunk * 8;
  const int col0 = reaches_back && first < n && first + 8 > n ? n - 8 : first;
  const bool vec_c = ldc % (16 / (int)sizeof(TOut)) == 0 && (reinterpret_cast<uintptr_t>(c) & 15u) == 0;
  constexpr bool PLAIN = EPI == PS_EPI_NONE;
  const bool full = col0 + 8 <= n;
  // eight key or value columns lie in one head (then n is whole pieces too)
  const bool whole_kv = !PLAIN || scatter.k_pool == nullptr ||
                        ((scatter.head_dim | scatter.q_cols | scatter.kv_cols) & 7) == 0;
  const bool by_column = !vec_c || !whole_kv || k_splits > 1;
  float b[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) b[q] = (bias && split == 0 && col0 + q < n) ? bias[col0 + q] : 0.f;
  // otherwise the columns behind the last whole piece go eight rows at a time
  const bool ends_inside =
      !reaches_back && (n & 7) != 0 && (n & ~7) >= col_base && (n & ~7) < col_base + WN * 32;
  const int last_col = (n & ~7) + (lane & 7);
  const float last_bias = bias && split == 0 && ends_inside && last_col < n ? bias[last_col] : 0.f;
  // key and value columns also go into cache pages
  TOut* pool = nullptr;
  int64_t pool_offset = 0;
  if (PLAIN && !by_column && scatter.k_pool != nullptr && full && col0 >= scatter.q_cols)
    pool = kv_scatter_col<TOut>(scatter, col0, &pool_offset);

  // What the whole pieces need from memory is asked for before the first of them: the residual rows, and
  // where each token's keys and values lie (two dependent reads a row).  One trip each, not one per pass.
  constexpr int PASSES = 32 / EP_ROWS;
  constexpr bool RESIDUAL = EPI == PS_EPI_RESIDUAL;
  float4 old[RESIDUAL ? WM : 1][RESIDUAL ? PASSES : 1][2];
  if (RESIDUAL && !by_column && full) {
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int pass = 0; pass < PASSES; ++pass) {
        const int row = row_base + i * 32 + pass * EP_ROWS + row_in_pass;
        const float* sum = reinterpret_cast<const float*>(c) + (int64_t)(row < m ? row : m - 1) * ldc + col0;
        old[RESIDUAL ? i : 0][RESIDUAL ? pass : 0][0] = *reinterpret_cast<const float4*>(sum);
        old[RESIDUAL ? i : 0][RESIDUAL ? pass : 0][1] = *reinterpret_cast<const float4*>(sum + 4);
      }
  }
  int64_t slots[PLAIN ? WM : 1][PLAIN ? PASSES : 1];
  if (PLAIN && pool != nullptr) {
    int pos[PLAIN ? WM : 1][PLAIN ? PASSES : 1], item[PLAIN ? WM : 1][PLAIN ? PASSES : 1];
#pragma unroll
    for (int i = 0; i < (PLAIN ? WM : 0); ++i)
#pragma unroll
      for (int pass = 0; pass < PASSES; ++pass) {
        const int row = row_base + i * 32 + pass * EP_ROWS + row_in_pass;
        pos[i][pass] = scatter.tok_pos[row < m ? row : m - 1];
        item[i][pass] = scatter.tok_item[row < m ? row : m - 1];
      }
#pragma unroll
    for (int i = 0; i < (PLAIN ? WM : 0); ++i)
#pragma unroll
      for (int pass = 0; pass < PASSES; ++pass)
        slots[i][pass] = kv_scatter_slot(scatter, pos[i][pass], &item[i][pass]);
  }

#pragma unroll
  for (int i = 0; i < WM; ++i) {
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e)
        region[((e >> 2) * 8 + (lane >> 5) * 4 + (e & 3)) * EP_STRIDE + j * 32 + (lane & 31)] =
            acc[i][j][e];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (by_column) {
      // rows that cannot leave in aligned pieces, heads that are no whole pieces, and partial sums of a split k: a
      // wave's lanes take consecutive columns of one row
#pragma unroll 8
      for (int r = 0; r < 32; ++r) {
        const int row = row_base + i * 32 + r;
        if (row >= m) continue;
#pragma unroll
        for (int half = 0; half < (WN + 1) / 2; ++half) {
          const int within = half * 64 + lane;
          const int col = col_base + within;
          if (within >= WN * 32 || col >= n) continue;
          const float bias_here = (bias && split == 0) ? bias[col] : 0.f;
          const float v = finish_value<EPI, TOut>(region[r * EP_STRIDE + within] + bias_here);
          TOut* out = c + (int64_t)row * ldc + col;
          if (EPI == PS_EPI_RESIDUAL) {
            float* sum = reinterpret_cast<float*>(out);
            if (k_splits > 1) unsafeAtomicAdd(sum, v);
            else *sum += v;
          } else {
            *out = from_float<TOut>(v);
            if (EPI == PS_EPI_NONE) kv_scatter_store<TOut>(scatter, row, col, v);
          }
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      continue;
    }
#pragma unroll
    for (int pass = 0; pass < PASSES; ++pass) {
      const int r = pass * EP_ROWS + row_in_pass;
      const int row = row_base + i * 32 + r;
      const float4 lo = *reinterpret_cast<const float4*>(region + r * EP_STRIDE + col0 - col_base);
      const float4 hi = *reinterpret_cast<const float4*>(region + r * EP_STRIDE + col0 - col_base + 4);
      if (row >= m || !full) continue;
      float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = finish_value<EPI, TOut>(v[q] + b[q]);
      TOut* out = c + (int64_t)row * ldc + col0;
      if constexpr (RESIDUAL) {
        float* sum = reinterpret_cast<float*>(out);
        float4 o0 = old[i][pass][0], o1 = old[i][pass][1];
        o0.x += v[0]; o0.y += v[1]; o0.z += v[2]; o0.w += v[3];
        o1.x += v[4]; o1.y += v[5]; o1.z += v[6]; o1.w += v[7];
        *reinterpret_cast<float4*>(sum) = o0;
        *reinterpret_cast<float4*>(sum + 4) = o1;
      } else {
        // (eight key or value columns that go to their page and that nobody reads from c)
        if (!(PLAIN && pool != nullptr && scatter.cache_only)) store8(out, v);
        if constexpr (PLAIN)
          if (pool != nullptr && slots[i][pass] >= 0) store8(pool + slots[i][pass] + pool_offset, v);
      }
    }
    if (ends_inside) {
      // (in the passes this code would stand in every one)
#pragma unroll 1
      for (int t = 0; t < 4; ++t) {
        const int r = t * 8 + (lane >> 3);
        const int row = row_base + i * 32 + r;
        if (row >= m || last_col >= n) continue;
        const float v = finish_value<EPI, TOut>(region[r * EP_STRIDE + last_col - col_base] + last_bias);
        TOut* out = c + (int64_t)row * ldc + last_col;
        if constexpr (RESIDUAL) *reinterpret_cast<float*>(out) += v;
        else *out = from_float<TOut>(v);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
}
