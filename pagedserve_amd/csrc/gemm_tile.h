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

// How a wave's 32-column blocks leave for memory.  Element e of a 32 x 32 accumulator is row (e / 4) * 8 + (lane / 32)
// * 4 + e % 4, column lane % 32: a lane holds one column.  Each wave turns 32 rows at a time through a region of LDS of
// its own, after which a lane holds eight consecutive columns of one row: bias and activation are applied there and
// rows leave in pieces of 16 or 32 bytes, eight (or more) lanes to a row.
template <int WM, int WN>
struct TilePieces {
  static constexpr int STRIDE = WN * 32 + 8;      // floats of LDS; 4 rows further is 32 banks further
  static constexpr int CHUNKS = WN * 4;           // pieces of eight columns per row
  static constexpr int ROWS = 64 / CHUNKS;        // rows per pass of the wave
  static constexpr int PASSES = 32 / ROWS;
  static constexpr int COUNT = WM * PASSES;       // pieces of a lane
  // (the last piece that lies in m rows, for those beyond)
  __device__ static int row(int lane, int row_base, int piece, int m) {
    const int at = row_base + piece / PASSES * 32 + piece % PASSES * ROWS + lane / CHUNKS;
    return at < m ? at : m - 1;
  }
};

// Pieces of eight columns cannot be stored: rows that are not aligned, heads that are no whole pieces (eight key or
// value columns lie in one head; then n is whole pieces too), and partial sums of a split k.
template <typename TOut, int EPI>
__device__ inline bool tile_by_column(const TOut* c, int ldc, int k_splits, const KvScatter& scatter) {
  const bool vec_c = ldc % (16 / (int)sizeof(TOut)) == 0 && (reinterpret_cast<uintptr_t>(c) & 15u) == 0;
  const bool whole_kv = EPI != PS_EPI_NONE || scatter.k_pool == nullptr ||
                        ((scatter.head_dim | scatter.q_cols | scatter.kv_cols) & 7) == 0;
  return !vec_c || !whole_kv || k_splits > 1;
}

// First column of a lane's pieces.  The piece that the end of the rows lies in begins further left where that is
// aligned and within the wave's columns (float rows of whole fours): both pieces then write the same values to the
// columns that they share.
template <typename TOut>
__device__ inline bool tile_reaches_back(int col_base, int n) {
  return sizeof(TOut) == 4 && (n & 3) == 0 && n - col_base >= 8;
}
template <int WN, typename TOut>
__device__ inline int tile_first_col(int lane, int col_base, int n) {
  const int first = col_base + lane % (WN * 4) * 8;
  return tile_reaches_back<TOut>(col_base, n) && first < n && first + 8 > n ? n - 8 : first;
}

// The pages of a wave's rows: two dependent reads for each.  They are the same for all its columns, so that a kernel
// asks for all of them at once (where a row's check in front of its read made one trip per row and slice of columns),
// and before its last products: with this 4096 x 4800 x 1600 with 3200 key and value columns, 256 x 320 to a tile, went
// from 70.4 to 64.0 us in a prefill, 2048 x 2304 x 768 from 17.8 to 16.0, 544 x 3072 x 1024 from 10.2 to 9.2.
template <int WM, int WN>
struct TilePages {
  using Pieces = TilePieces<WM, WN>;
  int pos[Pieces::COUNT], page[Pieces::COUNT];
  // `wanted` (the same for the whole wave): some of its columns are keys or values
  __device__ static bool wanted(const KvScatter& s, int col_end) {
    return s.k_pool != nullptr && s.table_width > 0 && col_end > s.q_cols;
  }
  __device__ void ask_rows(const KvScatter& s, int lane, int row_base, int m) {
#pragma unroll
    for (int p = 0; p < Pieces::COUNT; ++p) {
      const int row = Pieces::row(lane, row_base, p, m);
      pos[p] = s.tok_pos[row];
      page[p] = s.tok_item[row];
    }
  }
  __device__ void ask_pages(const KvScatter& s) {
    int64_t entry[Pieces::COUNT];
#pragma unroll
    for (int p = 0; p < Pieces::COUNT; ++p) entry[p] = (int64_t)page[p] * s.table_width;
    int logical[Pieces::COUNT];
    if (s.page_shift >= 0) {
#pragma unroll
      for (int p = 0; p < Pieces::COUNT; ++p) logical[p] = pos[p] >> s.page_shift;
    } else {
#pragma unroll
      for (int p = 0; p < Pieces::COUNT; ++p) logical[p] = pos[p] / s.page_size;
    }
#pragma unroll
    for (int p = 0; p < Pieces::COUNT; ++p) page[p] = s.tables[logical[p] < s.table_width ? entry[p] + logical[p] : 0];
#pragma unroll
    for (int p = 0; p < Pieces::COUNT; ++p) pos[p] = logical[p] < s.table_width ? pos[p] : -1;
  }
  __device__ bool holds(const KvScatter& s, int p) const {
    return s.table_width > 0 && pos[p] >= 0 && page[p] >= 0 && page[p] < s.num_pages;
  }
};

// What a wave's whole pieces need from memory: bias, and the rows that are added to.  The bias is read without a
// branch, as zeros from memory where there is none: behind a branch, or in front of a choice, the compiler waits for it.
static __device__ const float tile_no_bias[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)), aligned(4))) float f32x4_any;
typedef const __attribute__((address_space(1))) f32x4* global_f32x4_t;
typedef const __attribute__((address_space(1))) f32x4_any* global_f32x4_any_t;
template <int WM, int WN, typename TOut, int EPI>
struct TileEnds {
  using Pieces = TilePieces<WM, WN>;
  static constexpr bool RESIDUAL = EPI == PS_EPI_RESIDUAL;
  f32x4 bias[2], old[RESIDUAL ? Pieces::COUNT : 1][2];
  __device__ void ask(int lane, int row_base, int col_base, int m, int n, int ldc, const TOut* c, const float* b,
                      int split, bool by_column) {
    const int col0 = tile_first_col<WN, TOut>(lane, col_base, n);
    const bool full = col0 + 8 <= n;
    const bool biased = b != nullptr && split == 0 && n >= 8;
    const float* from = biased ? b : tile_no_bias;
    const int col = biased && full ? col0 : 0;
    // (through pointers that the compiler does not know: it would choose between values instead, and move the reads of
    // c to where they are used)
    const float* rows = reinterpret_cast<const float*>(c);
    asm volatile("" : "+v"(from), "+v"(rows));
    bias[0] = *(global_f32x4_any_t)(from + col);
    bias[1] = *(global_f32x4_any_t)(from + col + 4);
    if (RESIDUAL && !by_column && full) {
#pragma unroll
      for (int p = 0; p < (RESIDUAL ? Pieces::COUNT : 0); ++p) {
        const float* sum = rows + (int64_t)Pieces::row(lane, row_base, p, m) * ldc + col0;
        old[p][0] = *(global_f32x4_t)sum;
        old[p][1] = *(global_f32x4_t)(sum + 4);
      }
    }
  }
};

// The accumulators acc[WM][WN] of one wave (32 x 32 each, rows row_base + 32 i ..., columns
// col_base + 32 j ...) to C, through `region`, an area of LDS of 32 x (32 WN + 8) floats that
// belongs to this wave alone: bias, activation, residual add into the float stream, key/value
// columns into cache pages.  `split` / `k_splits`: partial sums of a k range are added with
// atomics, the bias by split 0 only.  `ends`, `pages`: what the caller has asked for (the pages
// where TilePages::wanted says so).  Inlined whatever it costs: the compiler made it a function of its own behind
// the GELU of tiles of 128 x 64, its arrays in scratch memory (float rows, us: 2048 x 3072 x 768 92.6, inlined 90.0,
// 4096 x 3072 x 768 176.7 and 170.8, 2048 x 6400 x 1600 391 and 384).
template <int WM, int WN, typename TOut, int EPI>
__device__ __forceinline__ void store_wave_tile(f32x16 (&acc)[WM][WN], float* region, int lane, int row_base,
                                                int col_base, int m, int n, int ldc, TOut* __restrict__ c,
                                                const float* __restrict__ bias, int split, int k_splits,
                                                const KvScatter& scatter,
                                                const TileEnds<WM, WN, TOut, EPI>& ends,
                                                const TilePages<WM, WN>& pages) {
  using Pieces = TilePieces<WM, WN>;
  constexpr int EP_STRIDE = Pieces::STRIDE, EP_ROWS = Pieces::ROWS, PASSES = Pieces::PASSES;
  // The callers read operands by assembly and wait for them just in front of this.  What is worked out of the lane here
  // must not be moved in front of that wait, into a register that such a read may still be filling.
  asm volatile("" : "+v"(lane));
  const int row_in_pass = lane / Pieces::CHUNKS;
  const bool reaches_back = tile_reaches_back<TOut>(col_base, n);
  const int col0 = tile_first_col<WN, TOut>(lane, col_base, n);
  constexpr bool PLAIN = EPI == PS_EPI_NONE, RESIDUAL = EPI == PS_EPI_RESIDUAL;
  const bool full = col0 + 8 <= n;
  const bool by_column = tile_by_column<TOut, EPI>(c, ldc, k_splits, scatter);
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
      for (int q = 0; q < 8; ++q) v[q] = finish_value<EPI, TOut>(v[q] + ends.bias[q / 4][q % 4]);
      TOut* out = c + (int64_t)row * ldc + col0;
      if constexpr (RESIDUAL) {
        float* sum = reinterpret_cast<float*>(out);
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] += ends.old[i * PASSES + pass][q / 4][q % 4];
        store8(sum, v);
      } else {
        // (eight key or value columns that go to their page and that nobody reads from c)
        if (!(PLAIN && pool != nullptr && scatter.cache_only)) store8(out, v);
        if constexpr (PLAIN) {
          const int p = i * PASSES + pass;
          if (pool != nullptr && pages.holds(scatter, p))
            store8(pool + kv_page_slot(scatter, pages.pos[p], pages.page[p]) + pool_offset, v);
        }
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

// The same for a kernel that has asked for nothing yet.
template <int WM, int WN, typename TOut, int EPI>
__device__ __forceinline__ void store_wave_tile(f32x16 (&acc)[WM][WN], float* region, int lane, int row_base,
                                                int col_base, int m, int n, int ldc, TOut* __restrict__ c,
                                                const float* __restrict__ bias, int split, int k_splits,
                                                const KvScatter& scatter) {
  asm volatile("" : "+v"(lane));
  const bool by_column = tile_by_column<TOut, EPI>(c, ldc, k_splits, scatter);
  TileEnds<WM, WN, TOut, EPI> ends;
  TilePages<WM, WN> pages;
  const bool paged = EPI == PS_EPI_NONE && !by_column && pages.wanted(scatter, col_base + WN * 32);
  if (paged) pages.ask_rows(scatter, lane, row_base, m);
  ends.ask(lane, row_base, col_base, m, n, ldc, c, bias, split, by_column);
  if (paged) pages.ask_pages(scatter);
  store_wave_tile<WM, WN, TOut, EPI>(acc, region, lane, row_base, col_base, m, n, ldc, c, bias, split, k_splits,
                                     scatter, ends, pages);
}
