// What the skinny matrix products (gemm_mfma.hip, gemm_skinny_norm.hip) share: the shape of a
// block and the epilogue that sums the waves' partial tiles.
#pragma once

#include "common.h"
#include "linear.h"
#include "pagedserve_hip.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

#define SK_WAVES 4
#define SK_UNROLL 4   // 64-k steps whose loads are issued together

// What the epilogue needs beside the sums: a column's bias, the residual values that it adds to, the page slots of
// its rows.  All of it is asked for beside the weights; behind the sums each would be a trip to memory of its own, 0.5
// us (a page slot two) at the end of a kernel of 3 us.  Thread t finishes column t % 16 of row t / 16 of each 16 x 16
// accumulator, so that 16 consecutive threads store one run of 16 columns.
template <typename TOut, int EPI, int MB>
struct SkinnyEnds {
  float bias;
  float before[MB];    // residual values (k not split)
  int pos[MB], item[MB], page[MB];
  bool there[MB];      // the row's position lies in the block table
  TOut* pool;          // of the column, null for a query's
  int64_t pool_offset;

  // In front of the weights: positions and items of the rows (tok_pos null: no scatter).
  __device__ inline void ask_rows(const int* __restrict__ tok_pos, const int* __restrict__ tok_item, int m, int row0) {
    if (EPI != PS_EPI_NONE || tok_pos == nullptr) return;
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      const int wanted = row0 + b * 16 + ((int)threadIdx.x >> 4);
      const int row = wanted < m ? wanted : m - 1;
      pos[b] = tok_pos[row];
      item[b] = tok_item[row];
    }
  }
  // Behind the loads of the weights.
  __device__ inline void ask(const float* __restrict__ bias_row, const TOut* c, int m, int n, int ldc, int n0, int row0,
                             int split, int k_splits, const KvScatter& scatter, const int* tok_pos,
                             int c_packed = 0) {
    const int col = n0 + ((int)threadIdx.x & 15) < n ? n0 + ((int)threadIdx.x & 15) : n - 1;
    bias = 0.f;
    if (bias_row != nullptr && split == 0) bias = bias_row[col];
    pool = nullptr;
    if (EPI == PS_EPI_NONE && tok_pos != nullptr)
      pool = kv_scatter_col<TOut>(scatter, n0 + ((int)threadIdx.x & 15), &pool_offset);
    if (EPI != PS_EPI_RESIDUAL) return;
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      const int wanted = row0 + b * 16 + ((int)threadIdx.x >> 4);
      const int row = wanted < m ? wanted : m - 1;
      before[b] = 0.f;
      if (k_splits == 1)
        before[b] = to_float<TOut>(c[c_packed ? packed_offset(row, col, n) : (int64_t)row * ldc + col]);
    }
  }
  // Once the positions are there: the block-table entries.
  __device__ inline void ask_pages(const KvScatter& scatter, const int* tok_pos, int n0) {
    if (EPI != PS_EPI_NONE || tok_pos == nullptr || n0 + 16 <= scatter.q_cols) return;
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      const int logical = scatter.page_shift >= 0 ? (pos[b] >> scatter.page_shift) : pos[b] / scatter.page_size;
      // a row without a page reads the first entry in its place
      there[b] = logical < scatter.table_width;
      page[b] = scatter.tables[there[b] ? (int64_t)item[b] * scatter.table_width + logical : 0];
    }
  }
};

// Sum the four waves' partial tiles and finish the block's 16 columns of MB x 16 rows.
// Element i of lane l of an accumulator is column (l / 16) * 4 + i of row l % 16.
template <typename TOut, int EPI, int MB>
__device__ inline void skinny_epilogue(float (*partial)[MB][4][64], const SkinnyEnds<TOut, EPI, MB>& ends, TOut* c,
                                       int m, int n, int ldc, int n0, int row0, int k_splits,
                                       const KvScatter& scatter, int c_packed = 0) {
  const int col_in = threadIdx.x & 15;
  const int row_in = threadIdx.x >> 4;
  const int col = n0 + col_in;
  if (col >= n) return;
  const int i = col_in & 3;
  const int lane = (col_in >> 2) * 16 + row_in;
#pragma unroll
  for (int b = 0; b < MB; ++b) {
    const int row = row0 + b * 16 + row_in;
    if (row >= m) continue;
    float v = partial[0][b][i][lane] + partial[1][b][i][lane] + partial[2][b][i][lane] +
              partial[3][b][i][lane] + ends.bias;
    // (c_packed: the output is the operand of another skinny product and is written in the
    // order in which that one reads it)
    TOut* dst = c_packed ? c + packed_offset(row, col, n) : c + (int64_t)row * ldc + col;
    if (EPI == PS_EPI_RESIDUAL) {
      if (k_splits > 1) {
        unsafeAtomicAdd(reinterpret_cast<float*>(dst), v);
      } else {
        *dst = from_float<TOut>(v + ends.before[b]);
      }
    } else {
      v = apply_activation<EPI>(v);
      *dst = from_float<TOut>(v);
      if (EPI == PS_EPI_NONE && ends.pool != nullptr && ends.there[b] && ends.page[b] >= 0 &&
          ends.page[b] < scatter.num_pages)
        ends.pool[ends.pool_offset + kv_page_slot(scatter, ends.pos[b], ends.page[b])] = from_float<TOut>(v);
    }
  }
}
