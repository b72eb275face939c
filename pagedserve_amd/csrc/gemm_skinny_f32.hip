// Matrix product of few float rows (decode steps and short prompt portions of the 32-bit path) on
// the matrix cores of gfx950, in true 32-bit (v_mfma_f32_16x16x4_f32):
//   C[m, n] = epi(sum_k A[m, k] W[n, k] + b[n]),   k a multiple of 4, any m and n.
//
// Bound by reading W once, and at these sizes by the one trip to memory that this takes: like the
// bfloat16 product for few rows, a block owns 16 NT weight rows and MB blocks of 16 rows of A, its
// waves take turns along k in steps of 32 values (128 bytes of every row), operands go straight from
// memory to the matrix cores, UNROLL steps asked for together (8 x 4096 x 1024 8.8 us where the compiler orders
// the loads, 7.4 so), and the waves' partial tiles are summed in LDS in a fixed order.  Rows of A beyond MB blocks go to further blocks (grid z), which read the
// same weights out of the L2.  k may be split over blocks; those partial sums are added with float
// atomics into the stream (residual epilogue only).  A lane's 16 bytes of k are the same for both
// operands, so that which four values an instruction multiplies does not matter.
//
// Measured with weights from memory, before (the plain kernel, or up to 16 rows one dot product per
// wave and column) and after, in us: 64 x 2304 x 768 88 / 9.7, 64 x 768 x 3072 338 / 9.5, 32 x 768 x
// 768 89 / 5.4, 200 x 768 x 768 34 / 9.7, 16 x 3072 x 768 8.6 / 5.6, 8 x 768 x 3072 7.1 / 5.0,
// 16 x 50257 x 768 68 / 46 (its weights alone are 30 at the rate of a copy).  Relative error against 64 bits: 16 x
// 2304 x 768 9.3e-8 (the dot products 9.3e-8; with one accumulator per value of k 1.1e-7), 64 x 768 x 3072 1.0e-6 / 1.2e-7.
#include "common.h"
#include "linear.h"
#include "pagedserve_hip.h"

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

#define SF_STEP 32    // values of k per step of a wave: 128 bytes of every row

// The sum of N numbers in pairs, the pairs in pairs and so on.
template <int N>
__device__ inline float sum_in_pairs(float (&v)[N]) {
#pragma unroll
  for (int span = 1; span < N; span *= 2)
#pragma unroll
    for (int p = 0; p + span < N; p += 2 * span) v[p] += v[p + span];
  return v[0];
}

// What the epilogue needs beside the sums (bias, residual values, page slots), asked for behind the weights' loads and
// there when they are: behind the sums each would be a trip of its own (as SkinnyEnds, gemm_skinny.h).  Thread t
// finishes elements t, t + 64 WAVES, ... of the block's 16 NT columns of 16 MB rows: element i of a 16 x 16 accumulator is
// weight row (lane / 16) * 4 + i, activation row lane % 16, and 16 consecutive threads finish one run of 16 columns.
template <int EPI, int MB, int NT, int WAVES>
struct FloatEnds {
  static constexpr int ELEMENTS = NT * MB * 256, COUNT = (ELEMENTS + 64 * WAVES - 1) / (64 * WAVES);
  float bias[COUNT], before[COUNT];
  int pos[COUNT], item[COUNT], page[COUNT];
  bool there[COUNT];

  __device__ static inline int column(int e) { return (e >> 8) / MB * 16 + (e & 15); }
  __device__ static inline int row(int e) { return (e >> 8) % MB * 16 + ((e >> 4) & 15); }
  __device__ inline void ask(const float* __restrict__ bias_row, const float* c, int m, int n, int ldc, int n0, int row0,
                             int split, int k_splits, const KvScatter& scatter) {
#pragma unroll
    for (int it = 0; it < COUNT; ++it) {
      const int e = threadIdx.x + it * 64 * WAVES;
      const int col = n0 + column(e) < n ? n0 + column(e) : n - 1;
      const int at = row0 + row(e) < m ? row0 + row(e) : m - 1;
      bias[it] = 0.f;
      if (bias_row != nullptr && split == 0) bias[it] = bias_row[col];
      if (EPI == PS_EPI_RESIDUAL) {
        before[it] = 0.f;
        if (k_splits == 1) before[it] = c[(int64_t)at * ldc + col];
      }
      if (EPI == PS_EPI_NONE && scatter.k_pool != nullptr) {
        pos[it] = scatter.tok_pos[at];
        item[it] = scatter.tok_item[at];
      }
    }
  }
  __device__ inline void ask_pages(const KvScatter& scatter, int n0) {
    if (EPI != PS_EPI_NONE || scatter.k_pool == nullptr || n0 + 16 * NT <= scatter.q_cols) return;
#pragma unroll
    for (int it = 0; it < COUNT; ++it) {
      const int logical = scatter.page_shift >= 0 ? (pos[it] >> scatter.page_shift) : pos[it] / scatter.page_size;
      // a row without a page reads the first entry in its place
      there[it] = logical < scatter.table_width;
      page[it] = scatter.tables[there[it] ? (int64_t)item[it] * scatter.table_width + logical : 0];
    }
  }
};

// Sum the waves' partial tiles in a fixed order and finish the block's 16 NT columns of 16 MB rows.
template <int EPI, int MB, int NT, int WAVES>
__device__ inline void skinny_f32_epilogue(float (&partial)[NT][WAVES][MB][4][64],
                                           const FloatEnds<EPI, MB, NT, WAVES>& ends, float* c,
                                           int m, int n, int ldc, int n0, int row0, int k_splits,
                                           const KvScatter& scatter) {
  typedef FloatEnds<EPI, MB, NT, WAVES> Ends;
#pragma unroll
  for (int it = 0; it < Ends::COUNT; ++it) {
    const int e = threadIdx.x + it * 64 * WAVES;
    const int col = n0 + Ends::column(e);
    const int row = row0 + Ends::row(e);
    if (e >= Ends::ELEMENTS || col >= n || row >= m) continue;
    const int j = (e >> 8) / MB, b = (e >> 8) % MB;
    const int i = e & 3;
    const int at = ((e & 15) >> 2) * 16 + ((e >> 4) & 15);
    float of_wave[WAVES];
#pragma unroll
    for (int p = 0; p < WAVES; ++p) of_wave[p] = partial[j][p][b][i][at];
    float v = sum_in_pairs(of_wave) + ends.bias[it];
    float* dst = c + (int64_t)row * ldc + col;
    if (EPI == PS_EPI_RESIDUAL) {
      if (k_splits > 1) unsafeAtomicAdd(dst, v);
      else *dst = ends.before[it] + v;
    } else {
      v = apply_activation<EPI>(v);
      *dst = v;
      if (EPI == PS_EPI_NONE && scatter.k_pool != nullptr && col >= scatter.q_cols) {
        int64_t offset;
        float* pool = kv_scatter_col<float>(scatter, col, &offset);
        if (ends.there[it] && ends.page[it] >= 0 && ends.page[it] < scatter.num_pages)
          pool[offset + kv_page_slot(scatter, ends.pos[it], ends.page[it])] = v;
      }
    }
  }
}

// (the arguments in front of the scatter come with the launch)
template <int EPI, int MB, int NT, int UNROLL, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void gemm_nt_skinny_f32_kernel(
    const float* __restrict__ a, const float* __restrict__ w, const float* __restrict__ bias,
    float* __restrict__ c, int m, int n, int k, int lda, int k_chunk, int ldc, int k_splits,
    KvScatter scatter) {
  __shared__ float partial[NT][WAVES][MB][4][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // the same in every lane: scalar
  const int n0 = blockIdx.x * 16 * NT;
  const int split = blockIdx.y;
  const int row0 = blockIdx.z * (MB * 16);
  const int k_begin = split * k_chunk;
  const int k_end = k_begin + k_chunk < k ? k_begin + k_chunk : k;
  const int sub = lane & 15;
  const int group = lane >> 4;
  const float* w_ptr[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int row = n0 + j * 16 + sub < n ? n0 + j * 16 + sub : n - 1;
    w_ptr[j] = w + (int64_t)row * k;
  }
  const float* a_ptr[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b) {
    const int row = row0 + b * 16 + sub < m ? row0 + b * 16 + sub : m - 1;
    a_ptr[b] = a + (int64_t)row * lda;
  }
  // an accumulator for each of a lane's four values of k, and for up to 16 rows two such fours that take
  // turns: short chains, whose rounding errors stay small (with the sums in pairs behind them those of one dot
  // product to a wave's 64 lanes) and whose instructions do not wait for each other
  constexpr int SETS = MB == 1 ? 2 : 1;
  f32x4 acc[NT][MB][4 * SETS];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
      for (int i = 0; i < 4 * SETS; ++i) acc[j][b][i] = f32x4{0.f, 0.f, 0.f, 0.f};

  f32x4 wf[UNROLL][NT][2], xf[UNROLL][MB][2];
  auto load = [&](int k0) {
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int kk = k0 + u * WAVES * SF_STEP + h * 16 + group * 4;
        const bool there = kk < k_end;      // (k is a multiple of 4: a piece is whole or absent)
        // unconditional loads from a clamped place, zeroed afterwards: loads under a branch
        // would not be issued together
        const int at = there ? kk : k_begin;
#pragma unroll
        for (int j = 0; j < NT; ++j) wf[u][j][h] = *reinterpret_cast<const f32x4*>(w_ptr[j] + at);
#pragma unroll
        for (int b = 0; b < MB; ++b) xf[u][b][h] = *reinterpret_cast<const f32x4*>(a_ptr[b] + at);
      }
    // (without this the compiler asks for a few at a time, to use fewer registers)
    __builtin_amdgcn_sched_barrier(0);
  };
  auto multiply = [&](int k0) {
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const bool there = k0 + u * WAVES * SF_STEP + h * 16 + group * 4 < k_end;
        if (!there) {
#pragma unroll
          for (int j = 0; j < NT; ++j) wf[u][j][h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int b = 0; b < MB; ++b) xf[u][b][h] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int b = 0; b < MB; ++b)
              acc[j][b][(2 * u + h) % SETS * 4 + i] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                  wf[u][j][h][i], xf[u][b][h][i], acc[j][b][(2 * u + h) % SETS * 4 + i], 0, 0, 0);
      }
  };
  // wave `wave` takes the steps wave, wave + WAVES, ... of the block's range; UNROLL of them are
  // asked for together, the first ones in front of what the epilogue needs.  (A wave without a step, of a short k, asks
  // for nothing and leaves the matrix cores to the others: 32 x 192 x 64 7.05 us when it multiplied zeros, now 3.8, 16 x
  // 320 x 96 4.95 and 3.5.)
  FloatEnds<EPI, MB, NT, WAVES> ends;
  int k0 = k_begin + wave * SF_STEP;
  const bool works = k0 < k_end;
  if (works) load(k0);
  if (EPI == PS_EPI_NONE && scatter.k_pool != nullptr) read_scatter(scatter);
  ends.ask(bias, c, m, n, ldc, n0, row0, split, k_splits, scatter);
  if (works) multiply(k0);
  for (k0 += WAVES * UNROLL * SF_STEP; k0 < k_end; k0 += WAVES * UNROLL * SF_STEP) {
    load(k0);
    multiply(k0);
  }
  ends.ask_pages(scatter, n0);
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float sums[4 * SETS];
#pragma unroll
        for (int p = 0; p < 4 * SETS; ++p) sums[p] = acc[j][b][p][i];
        partial[j][wave][b][i][lane] = sum_in_pairs(sums);
      }
  __syncthreads();

  skinny_f32_epilogue<EPI, MB, NT, WAVES>(partial, ends, c, m, n, ldc, n0, row0, k_splits, scatter);
}

// A value of the lane N places on within its run of 16.
template <int N>
__device__ inline float row_turned(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 + N, 0xf, 0xf, false));
}

// The same for up to 16 rows with the norm of its input fused in front (whole k in one round of loads): while the
// weights travel, each wave normalises up to two rows in registers (as norm_wave_kernel, elementwise.hip)
// and leaves them in LDS, where the product reads its column operand.  One launch and one trip to memory
// instead of two launches, in us: 1 x 2304 x 768 7.4 -> 5.3, 8 x 2304 x 768 8.7 -> 5.9, 16 x 2304 x 768
// 11.6 -> 6.7, 8 x 4096 x 1024 16.9 -> 8.7.  (The arguments in front of the bias come with the launch.)
#define SF_ROW_BITS 16  // of the number of rows; behind it
#define SF_RMS 1
#define SF_SHIFT 2      // (without a shift the argument is gamma)
template <int EPI, int UNROLL>
__global__ __launch_bounds__(512) void gemm_nt_skinny_norm_f32_kernel(
    const float* __restrict__ h_rows, const float* __restrict__ gamma, const float* __restrict__ shift,
    const float* __restrict__ w, const int* __restrict__ rows_of, int ldh, int rows_and_flags, int n, int k,
    const float* __restrict__ bias, float* __restrict__ c, int ldc, float eps, KvScatter scatter) {
  const int m = rows_and_flags & ((1 << SF_ROW_BITS) - 1);
  const bool rms = (rows_and_flags >> SF_ROW_BITS) & SF_RMS, shifts = (rows_and_flags >> SF_ROW_BITS) & SF_SHIFT;
  constexpr int WAVES = 8;
  constexpr int MOST = WAVES * UNROLL * SF_STEP;     // the longest k
  constexpr int STRIDE = MOST + 4;                   // floats; the next row is four banks further
  constexpr int PIECES = MOST / 256;
  __shared__ __attribute__((aligned(16))) float rows[16 * STRIDE];
  __shared__ float partial[1][WAVES][1][4][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // the same in every lane: scalar
  const int n0 = blockIdx.x * 16;
  const int sub = lane & 15;
  const int group = lane >> 4;
  const float* w_row = w + (int64_t)(n0 + sub < n ? n0 + sub : n - 1) * k;
  // The rows and the norm's scale and shift are asked for in front of the weights: a wave's loads come back in
  // the order of issue, and the norm works while the weights travel.
  const bool two = m > WAVES;                        // a second row per wave
  float v[2][PIECES][4], g[PIECES][4], b[PIECES][4];
  auto load_row = [&](int half) {
    const int r = wave + half * WAVES < m ? wave + half * WAVES : m - 1;
    const float* src = h_rows + (int64_t)(rows_of ? rows_of[r] : r) * ldh;
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int col = (lane + i * 64) * 4;
      *reinterpret_cast<float4*>(v[half][i]) = *reinterpret_cast<const float4*>(src + (col < k ? col : k - 4));
    }
  };
  f32x4 wf[UNROLL][2];
  FloatEnds<EPI, 1, 1, WAVES> ends;
  auto load_scale = [&] {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int col = (lane + i * 64) * 4;
      const int safe = col < k ? col : k - 4;
      *reinterpret_cast<float4*>(g[i]) = *reinterpret_cast<const float4*>(gamma + safe);
      *reinterpret_cast<float4*>(b[i]) = *reinterpret_cast<const float4*>(shift + safe);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto load_weights = [&] {
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int kk = (u * WAVES + wave) * SF_STEP + h * 16 + group * 4;
        wf[u][h] = *reinterpret_cast<const f32x4*>(w_row + (kk < k ? kk : 0));
      }
    read_arguments(bias, c, ldc, eps);
    if (EPI == PS_EPI_NONE && scatter.k_pool != nullptr) read_scatter(scatter);
    ends.ask(bias, c, m, n, ldc, n0, 0, 0, 1, scatter);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto finish_row = [&](int half) {
    const int r = wave + half * WAVES;
    if (r >= m) return;
    float mean = 0.f;
    if (!rms) {
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < PIECES; ++i)
        if ((lane + i * 64) * 4 < k) sum += (v[half][i][0] + v[half][i][1]) + (v[half][i][2] + v[half][i][3]);
      mean = wave_sum(sum) / (float)k;
    }
    float sq = 0.f;
#pragma unroll
    for (int i = 0; i < PIECES; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[half][i][j] = (lane + i * 64) * 4 < k ? v[half][i][j] - mean : 0.f;
        sq = fmaf(v[half][i][j], v[half][i][j], sq);
      }
    const float inv_std = 1.0f / sqrtf(wave_sum(sq) / (float)k + eps);
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int col = (lane + i * 64) * 4;
      if (col >= k) continue;
      f32x4 y;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        y[j] = shifts ? fmaf(v[half][i][j] * inv_std, g[i][j], b[i][j]) : v[half][i][j] * inv_std * g[i][j];
      *reinterpret_cast<f32x4*>(rows + r * STRIDE + col) = y;
    }
  };
  // (paths of their own, so that the waits of each know how many loads are behind the ones they wait for; a wave
  // without a row asks for weights alone: 4 x 6144 x 1000, where units have more than one block, 10.3 and 9.7 us)
  if (two) {
    load_row(0);
    load_row(1);
    load_scale();
    load_weights();
    finish_row(0);
    finish_row(1);
  } else if (wave < m) {
    load_row(0);
    load_scale();
    load_weights();
    finish_row(0);
  } else {
    load_weights();
  }
  ends.ask_pages(scatter, n0);
#pragma unroll
  for (int u = 0; u < UNROLL; ++u)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      if ((u * WAVES + wave) * SF_STEP + h * 16 + group * 4 >= k) wf[u][h] = f32x4{0.f, 0.f, 0.f, 0.f};
  __syncthreads();
  // (rows of LDS beyond m stay as they are: they only feed outputs that are never stored)
  constexpr int SETS = 3;     // (as above; the normed rows carry a rounding of their own)
  f32x4 acc[4 * SETS];
#pragma unroll
  for (int i = 0; i < 4 * SETS; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < UNROLL; ++u)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int kk = (u * WAVES + wave) * SF_STEP + h * 16 + group * 4;
      f32x4 x = *reinterpret_cast<const f32x4*>(rows + sub * STRIDE + (kk < k ? kk : 0));
      if (kk >= k) x = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i)
        acc[(2 * u + h) % SETS * 4 + i] =
            __builtin_amdgcn_mfma_f32_16x16x4f32(wf[u][h][i], x[i], acc[(2 * u + h) % SETS * 4 + i], 0, 0, 0);
    }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float sums[4 * SETS];
#pragma unroll
    for (int p = 0; p < 4 * SETS; ++p) sums[p] = acc[p][i];
    partial[0][wave][0][i][lane] = sum_in_pairs(sums);
  }
  __syncthreads();
  skinny_f32_epilogue<EPI, 1, 1, WAVES>(partial, ends, c, m, n, ldc, n0, 0, 1, scatter);
}

// The same for up to eight rows.  Instructions of 16 x 16 spend half of their time and more on rows that are not there
// (0.55 of 5.4 us, 8 x 3072 x 768), and blocks of 16 columns leave 112 units without one at 2304 columns.  Here four
// waves take a quarter of k each and blocks have 4 GROUPS columns: an instruction of 4 x 4 multiplies four columns by
// four rows in 16 places of k, whose sums meet at the end.  A lane's 16 bytes are those of column lane % 4 and k piece
// lane / 4, so that a load takes 256 bytes of four rows of W.  Up to four rows, or eight, which use W's operand twice.
// Bound by the launch and the trip of the weights from memory (without them 3.7 us).  In us, 16 x 16 and this one: 1 x
// 2304 x 768 5.1 / 4.35, 4 rows 4.95 / 4.25, 8 rows 5.5 / 4.9, 1 x 3072 x 768 5.35 / 4.6, 8 rows 5.7 / 5.1.  In blocks of
// 16 columns 8 x 2304 x 768 takes 5.5, 8 x 3072 x 768 5.5: 12 wherever that is no more blocks than units.
#define SF_FEW_ROWS 8
#define SF_FEW_PIECE 64      // values of k that the 16 places take
template <int EPI, int PIECES, int GROUPS, int ROWS>
__global__ __launch_bounds__(256) void gemm_nt_few_norm_f32_kernel(
    const float* __restrict__ h_rows, const float* __restrict__ gamma, const float* __restrict__ shift,
    const float* __restrict__ w, const int* __restrict__ rows_of, int ldh, int rows_and_flags, int n, int k,
    const float* __restrict__ bias, float* __restrict__ c, int ldc, float eps, KvScatter scatter) {
  const int m = rows_and_flags & ((1 << SF_ROW_BITS) - 1);
  const bool rms = (rows_and_flags >> SF_ROW_BITS) & SF_RMS, shifts = (rows_and_flags >> SF_ROW_BITS) & SF_SHIFT;
  constexpr int WAVES = 4, SETS = ROWS / 4, HELD = ROWS / WAVES;     // rows that a wave normalises
  constexpr int MOST = WAVES * PIECES * SF_FEW_PIECE;                // the longest k
  constexpr int STRIDE = MOST + 8;                   // the four rows of two places then lie in 32 different banks
  constexpr int COLS = 4 * GROUPS, ELEMENTS = COLS * ROWS;
  static_assert(ROWS == 4 || ROWS == 8, "one or two sets of four rows");
  static_assert(ELEMENTS <= 64 * WAVES && MOST % 256 == 0, "a thread finishes one element, a wave reads whole rows");
  __shared__ __attribute__((aligned(16))) float rows[ROWS * STRIDE];
  __shared__ float partial[4 * WAVES][ELEMENTS];     // of a wave's four runs of 16 lanes
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // the same in every lane: scalar
  const int n0 = blockIdx.x * COLS;
  const int sub = lane & 3, place = lane >> 2;
  // (rows, scale, shift and weights in this order, as above)
  constexpr int PARTS = MOST / 256;
  float v[HELD][PARTS][4], g[PARTS][4], b[PARTS][4];
  f32x4 wf[PIECES][GROUPS];
  int src_row[HELD];
#pragma unroll
  for (int half = 0; half < HELD; ++half) {
    const int r = wave + half * WAVES < m ? wave + half * WAVES : m - 1;
    src_row[half] = rows_of ? scalar_load(rows_of + r) : r;
  }
#pragma unroll
  for (int half = 0; half < HELD; ++half) {
    const float* src = h_rows + (int64_t)src_row[half] * ldh;
#pragma unroll
    for (int i = 0; i < PARTS; ++i) {
      const int col = (lane + i * 64) * 4;
      *reinterpret_cast<float4*>(v[half][i]) = *reinterpret_cast<const float4*>(src + (col < k ? col : k - 4));
    }
  }
#pragma unroll
  for (int i = 0; i < PARTS; ++i) {
    const int col = (lane + i * 64) * 4;
    const int safe = col < k ? col : k - 4;
    *reinterpret_cast<float4*>(g[i]) = *reinterpret_cast<const float4*>(gamma + safe);
    *reinterpret_cast<float4*>(b[i]) = *reinterpret_cast<const float4*>(shift + safe);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int p = 0; p < PIECES; ++p)
#pragma unroll
    for (int j = 0; j < GROUPS; ++j) {
      const int col = n0 + j * 4 + sub < n ? n0 + j * 4 + sub : n - 1;
      const int kk = (p * WAVES + wave) * SF_FEW_PIECE + place * 4;
      wf[p][j] = *reinterpret_cast<const f32x4*>(w + (int64_t)col * k + (kk < k ? kk : 0));
    }
  read_arguments(bias, c, ldc, eps);
  if (EPI == PS_EPI_NONE && scatter.k_pool != nullptr) read_scatter(scatter);
  // what the epilogue needs: element e is column e % COLS of row e / COLS
  const int element = threadIdx.x;
  const int out_col = n0 + element % COLS, out_row = element / COLS;
  const int col_read = out_col < n ? out_col : n - 1, row_read = out_row < m ? out_row : m - 1;
  const bool scatters = EPI == PS_EPI_NONE && scatter.k_pool != nullptr;
  float own_bias = 0.f;
  int pos = 0, item = 0, page = -1;
  bool there = false;
  if (bias != nullptr) own_bias = bias[col_read];
  if (scatters) {
    pos = scatter.tok_pos[row_read];
    item = scatter.tok_item[row_read];
  }
  __builtin_amdgcn_sched_barrier(0);

  float mean[HELD], inv_std[HELD];      // (a wave's rows side by side: their sums do not wait for each other)
#pragma unroll
  for (int half = 0; half < HELD; ++half) mean[half] = 0.f;
  if (!rms) {
#pragma unroll
    for (int half = 0; half < HELD; ++half) {
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < PARTS; ++i)
        if ((lane + i * 64) * 4 < k) sum += (v[half][i][0] + v[half][i][1]) + (v[half][i][2] + v[half][i][3]);
      mean[half] = sum;
    }
#pragma unroll
    for (int half = 0; half < HELD; ++half) mean[half] = wave_sum(mean[half]) / (float)k;
  }
#pragma unroll
  for (int half = 0; half < HELD; ++half) {
    float sq = 0.f;
#pragma unroll
    for (int i = 0; i < PARTS; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[half][i][j] = (lane + i * 64) * 4 < k ? v[half][i][j] - mean[half] : 0.f;
        sq = fmaf(v[half][i][j], v[half][i][j], sq);
      }
    inv_std[half] = sq;
  }
#pragma unroll
  for (int half = 0; half < HELD; ++half) inv_std[half] = 1.0f / sqrtf(wave_sum(inv_std[half]) / (float)k + eps);
  // (rows beyond m are the last one again, places beyond k zeros)
#pragma unroll
  for (int half = 0; half < HELD; ++half)
#pragma unroll
    for (int i = 0; i < PARTS; ++i) {
      const int col = (lane + i * 64) * 4;
      f32x4 y;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        y[j] = shifts ? fmaf(v[half][i][j] * inv_std[half], g[i][j], b[i][j]) : v[half][i][j] * inv_std[half] * g[i][j];
      if (col >= k) y = f32x4{0.f, 0.f, 0.f, 0.f};
      *reinterpret_cast<f32x4*>(rows + (wave + half * WAVES) * STRIDE + col) = y;
    }
  __syncthreads();

  // an accumulator for each of a lane's four values of k: chains of PIECES
  f32x4 acc[GROUPS][SETS][4];
#pragma unroll
  for (int j = 0; j < GROUPS; ++j)
#pragma unroll
    for (int t = 0; t < SETS; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[j][t][i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int p = 0; p < PIECES; ++p) {
    const int kk = (p * WAVES + wave) * SF_FEW_PIECE + place * 4;
    f32x4 x[SETS];
#pragma unroll
    for (int t = 0; t < SETS; ++t) x[t] = *reinterpret_cast<const f32x4*>(rows + (t * 4 + sub) * STRIDE + kk);
#pragma unroll
    for (int j = 0; j < GROUPS; ++j) {
      f32x4 weights = wf[p][j];
      asm volatile("" : "+v"(weights));      // (or the choice below is made, and waited for, in front of the norm)
      if (kk >= k) weights = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < SETS; ++t)
          acc[j][t][i] = __builtin_amdgcn_mfma_f32_4x4x1f32(weights[i], x[t][i], acc[j][t][i], 0, 0, 0);
    }
  }
  if (scatters && n0 + COLS > scatter.q_cols) {
    const int logical = scatter.page_shift >= 0 ? (pos >> scatter.page_shift) : pos / scatter.page_size;
    // a row without a page reads the first entry in its place
    there = logical < scatter.table_width;
    page = scatter.tables[there ? (int64_t)item * scatter.table_width + logical : 0];
  }
  // lane l holds columns 4 j .. 4 j + 3 of row 4 t + l % 4 for place l / 4
#pragma unroll
  for (int j = 0; j < GROUPS; ++j)
#pragma unroll
    for (int t = 0; t < SETS; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float sum = (acc[j][t][0][i] + acc[j][t][1][i]) + (acc[j][t][2][i] + acc[j][t][3][i]);
        sum += row_turned<4>(sum);
        sum += row_turned<8>(sum);
        if ((lane & 15) < 4) partial[wave * 4 + (lane >> 4)][(t * 4 + sub) * COLS + j * 4 + i] = sum;
      }
  __syncthreads();
  if (element >= ELEMENTS || out_col >= n || out_row >= m) return;
  float of_run[4 * WAVES];
#pragma unroll
  for (int p = 0; p < 4 * WAVES; ++p) of_run[p] = partial[p][element];
  const float value = apply_activation<EPI>(sum_in_pairs(of_run) + own_bias);
  c[(int64_t)out_row * ldc + out_col] = value;
  if (scatters && out_col >= scatter.q_cols) {
    int64_t offset;
    float* pool = kv_scatter_col<float>(scatter, out_col, &offset);
    if (there && page >= 0 && page < scatter.num_pages) pool[offset + kv_page_slot(scatter, pos, page)] = value;
  }
}

// Up to eight rows added to, without a norm in front, four columns to a block: the operands as in
// gemm_nt_few_norm_f32_kernel, the rows' straight from memory, all asked for at once, and each block reads them once
// (the waves of the plain kernel, gemm_simple.hip, read all of them each: that, and not the weights, is what a unit then
// waits for).  Where it is taken (few_rows_take) both sides are measured.
template <int PIECES, int ROWS>
__global__ __launch_bounds__(256) void gemm_nt_few_f32_kernel(
    const float* __restrict__ a, const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ c,
    int m, int n, int k, int lda, int ldc) {
  constexpr int WAVES = 4, SETS = ROWS / 4, ELEMENTS = 4 * ROWS;
  __shared__ float partial[4 * WAVES][ELEMENTS];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // the same in every lane: scalar
  const int n0 = blockIdx.x * 4;
  const int sub = lane & 3, place = lane >> 2;
  const float* w_row = w + (int64_t)(n0 + sub < n ? n0 + sub : n - 1) * k;
  const float* a_row[SETS];
#pragma unroll
  for (int t = 0; t < SETS; ++t) a_row[t] = a + (int64_t)(t * 4 + sub < m ? t * 4 + sub : m - 1) * lda;
  f32x4 wf[PIECES], xf[PIECES][SETS];
#pragma unroll
  for (int p = 0; p < PIECES; ++p) {
    const int kk = (p * WAVES + wave) * SF_FEW_PIECE + place * 4;
    const int at = kk < k ? kk : 0;
    wf[p] = *reinterpret_cast<const f32x4*>(w_row + at);
#pragma unroll
    for (int t = 0; t < SETS; ++t) xf[p][t] = *reinterpret_cast<const f32x4*>(a_row[t] + at);
  }
  const int element = threadIdx.x;
  const int out_col = n0 + (element & 3), out_row = element >> 2;
  float* dst = c + (int64_t)(out_row < m ? out_row : m - 1) * ldc + (out_col < n ? out_col : n - 1);
  const float before = *dst;
  float own_bias = 0.f;
  if (bias != nullptr) own_bias = bias[out_col < n ? out_col : n - 1];
  __builtin_amdgcn_sched_barrier(0);
  f32x4 acc[SETS][4];
#pragma unroll
  for (int t = 0; t < SETS; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[t][i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int p = 0; p < PIECES; ++p) {
    const bool beyond = (p * WAVES + wave) * SF_FEW_PIECE + place * 4 >= k;
    if (beyond) wf[p] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < SETS; ++t)
      if (beyond) xf[p][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int t = 0; t < SETS; ++t)
        acc[t][i] = __builtin_amdgcn_mfma_f32_4x4x1f32(wf[p][i], xf[p][t][i], acc[t][i], 0, 0, 0);
  }
#pragma unroll
  for (int t = 0; t < SETS; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float sum = (acc[t][0][i] + acc[t][1][i]) + (acc[t][2][i] + acc[t][3][i]);
      sum += row_turned<4>(sum);
      sum += row_turned<8>(sum);
      if ((lane & 15) < 4) partial[wave * 4 + (lane >> 4)][(t * 4 + sub) * 4 + i] = sum;
    }
  __syncthreads();
  if (element >= ELEMENTS || out_col >= n || out_row >= m) return;
  float of_run[4 * WAVES];
#pragma unroll
  for (int p = 0; p < 4 * WAVES; ++p) of_run[p] = partial[p][element];
  *dst = before + (sum_in_pairs(of_run) + own_bias);
}

// --------------------------------------------------------------------------------- host
// Whether this kernel takes the product (a row of either operand in pieces of 16 bytes), and is the
// fastest that does.  The lines, with weights from memory, in us:
// - Up to 16 rows one dot product per wave and column (gemm_simple.hip) is ahead while the weights
//   are few (8 x 768 x 768 4.2 against 4.7, 16 x 768 x 768 5.0 against 5.9, 16 x 64 x 256 3.1 against 5.3, 16 x
//   1024 x 1024 5.6 against 6.8, 16 x 320 x 1280 4.7 against 5.6), and up to 8 level at very many columns; up to 4 rows
//   always but where k is long and can be split (4 x 1024 x 4096 8.6 against 7.1), or where rows are added to (see
//   few_rows_take).  Nine rows and more with the
//   plain epilogue come here all the same: with a key/value scatter behind it the other kernel needs a second launch
//   (2.5), and a product is the same bits with and without (16 x 192 x 64 3.3 here, 2.8 there).
// - Residual epilogue, k split: 200 x 768 x 3072 24.3 against 25.2 for the tiled kernel, 300 rows 33 against
//   28; 300 x 768 x 768 11.4 against 11.5; wide models sooner (32 x 1600 x 6400 25.4 against 25.2).
// - Otherwise up to 64 rows and one round of loads (32 x 4096 x 1024 12.2 against 17.3, 64 rows 17.1
//   against 17.4; 32 x 4800 x 1600 24.0 against 22.7; 100 x 2304 x 768 13.1 against 11.8), and not
//   the output head beyond 16 rows (32 x 50257 x 768 71 against 68).
// - A k that is no multiple of 32, which the tiled kernel does not take, up to 768 rows: there it
//   meets the one that does (gemm_mfma.hip).
// (few_rows_take) Rows added to, four columns to a block.  In us with weights from memory, the kernels that would take
// them otherwise and this one:
// - Up to three rows of a k above 1024, where the other is a dot product per wave: 1 x 256 x 1280 3.4 / 3.2, 1 x 1024 x
//   3072 6.05 / 4.75, 2 x 1600 x 1600 6.55 / 5.35, 2 x 2048 x 3584 10.9 / 9.75, 3 x 1600 x 1600 6.55 / 5.75, 3 x 1280 x 3584 9.4 / 9.75.
// - Four rows where a block's rounds of loads are nearly full: 4 x 256 x 1280 3.4 / 3.9, 4 x 1600 x 1280 5.5 / 6.2, but 4 x 1024 x
//   1600 4.55 / 4.4, 4 x 1600 x 1600 6.6 / 6.25, 4 x 2048 x 3072 9.8 / 9.35; 4 x 1280 x 3584 9.6 / 10.7.
// - k = 4096, up to four rows: the other splits k, and its blocks are many however few the columns are.  Where the last round
//   of this kernel's blocks leaves half of the units empty it is behind, of three or four rows a quarter: 1 x 512 x 4096 4.5 / 5.4, 4 rows 4.85 / 6.6, 2 x
//   1280 x 4096 7.55 / 8.8, 4 x 1600 x 4096 9.8 / 11.05, but 1 x 1600 x 4096 9.25 / 8.7, 2 x 768 x 4096 6.55 / 6.35, 1 x 1024 x 4096 6.85 / 6.0, 4 rows 7.4 / 7.45,
//   1 x 2048 x 4096 11.5 / 8.85, 4 rows 12.4 / 12.05.
// - Five to eight rows of 512 to 1024: 5 x 512 x 512 3.2 / 2.75, 5 x 2048 x 1024 5.85 / 4.85, 8 x 1024 x 1024 4.05 / 4.0, 8 x 2048 x
//   768 5.35 / 4.7, 8 x 256 x 1024 3.45 / 3.6; beyond, 8 x 1600 x 1600 7.0 / 8.3 and 5 x 768 x 3072, whose k is split, 4.85 / 6.2.
// - Up to 2,048 columns, two rounds of blocks, the line of eight rows (8 x 2304 x 768 4.9 / 5.6, 8 x 4096 x 1024 6.8 / 8.3).  Up to
//   three rows would gain from it further on (1 x 2304 x 2048 8.7 / 6.3, 3 x 4096 x 2048 11.4 / 9.0, 4 x 6400 x 1600 12.85 / 15.1).
static bool few_rows_take(int m, int n, int k, int epilogue) {
  const int units = ps_compute_units();
  if (epilogue != PS_EPI_RESIDUAL || m > 8 || n > 8 * units) return false;
  if (m > 4) return k >= 512 && k <= 1024;
  const int last_round = ((n + 3) / 4 - 1) % units + 1;
  if (k == 4096) return m <= 2 ? 2 * last_round > units : 4 * last_round >= 3 * units;
  return m < 4 ? k > 1024 && k < 4096 : k >= 1536 && k <= 3072;
}

bool ps_gemm_nt_f32_skinny_takes(const void* a, const void* w, int m, int n, int k, int lda,
                                 int epilogue) {
  if (k % 4 != 0 || lda % 4 != 0 || (reinterpret_cast<uintptr_t>(a) & 15u) != 0 ||
      (reinterpret_cast<uintptr_t>(w) & 15u) != 0)
    return false;
  if (few_rows_take(m, n, k, epilogue)) return true;
  const bool residual = epilogue == PS_EPI_RESIDUAL;
  const int64_t weights = (int64_t)n * k;
  if (m <= 4) return residual && k >= 4096;
  if (m <= 8) return weights > (1 << 20) && n < 64 * 256;
  if (m <= 16) return weights > (1 << 20) || epilogue == PS_EPI_NONE;
  if (k % SF_STEP != 0) return m < 768;
  if (residual) return (int64_t)m * n <= 160000 && weights < 6000000;
  return n < 64 * 256 && (k <= 768 ? m <= 64 : k <= 1024 && m <= 32);
}

// The fused norm: up to 16 rows, a k of one round, and not so many columns that each of their blocks
// normalising the rows again costs more than a launch (the output head).  With a k that leaves most of the
// waves idle two small launches are over sooner (3 x 192 x 64: 4.2 against 4.6 us).
bool ps_norm_gemm_f32_fusable(const void* w, const NormPrologue& norm, int m, int n, int k) {
  const uintptr_t all = reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(norm.h) |
                        reinterpret_cast<uintptr_t>(norm.gamma) | reinterpret_cast<uintptr_t>(norm.beta);
  return m <= 16 && n <= 8192 && k % 4 == 0 && k >= 256 && k <= 8 * 4 * SF_STEP && norm.ldh % 4 == 0 && (all & 15u) == 0;
}

int ps_norm_gemm_f32_fused(const NormPrologue& norm, const void* w, const float* bias, void* c, int m,
                           int n, int k, int ldc, int epilogue, const KvScatter& scatter, hipStream_t s) {
  const bool shift = norm.rms == 0 && norm.beta != nullptr;
  const int rows_and_flags = m | ((norm.rms ? SF_RMS : 0) | (shift ? SF_SHIFT : 0)) << SF_ROW_BITS;
  const bool narrow = n <= 12 * ps_compute_units();      // blocks of 12 columns are at most one to a unit
#define PS_LAUNCH_SNF(EPI, UNROLL)                                                                     \
  hipLaunchKernelGGL((gemm_nt_skinny_norm_f32_kernel<EPI, UNROLL>), dim3((n + 15) / 16), dim3(512), 0, \
                     s, norm.h, norm.gamma, shift ? norm.beta : norm.gamma, (const float*)w, norm.rows, norm.ldh, \
                     rows_and_flags, n, k, bias, (float*)c, ldc, norm.eps, scatter)
#define PS_LAUNCH_FNF(EPI, PIECES, GROUPS, ROWS)                                                                    \
  hipLaunchKernelGGL((gemm_nt_few_norm_f32_kernel<EPI, PIECES, GROUPS, ROWS>), dim3((n + 4 * GROUPS - 1) / (4 * GROUPS)), \
                     dim3(256), 0, s, norm.h, norm.gamma, shift ? norm.beta : norm.gamma, (const float*)w, norm.rows,  \
                     norm.ldh, rows_and_flags, n, k, bias, (float*)c, ldc, norm.eps, scatter)
#define PS_FNF_ROWS(EPI, PIECES, GROUPS)               \
  do {                                                 \
    if (m <= 4) PS_LAUNCH_FNF(EPI, PIECES, GROUPS, 4); \
    else PS_LAUNCH_FNF(EPI, PIECES, GROUPS, 8);        \
  } while (0)
#define PS_SNF_CASE(EPI)                                                         \
  case EPI:                                                                      \
    if (m <= SF_FEW_ROWS && narrow && k <= 768) PS_FNF_ROWS(EPI, 3, 3);          \
    else if (m <= SF_FEW_ROWS && narrow) PS_FNF_ROWS(EPI, 4, 3);                 \
    else if (m <= SF_FEW_ROWS && k <= 768) PS_FNF_ROWS(EPI, 3, 4);               \
    else if (m <= SF_FEW_ROWS) PS_FNF_ROWS(EPI, 4, 4);                           \
    else if (k <= 8 * 3 * SF_STEP) PS_LAUNCH_SNF(EPI, 3);                        \
    else PS_LAUNCH_SNF(EPI, 4);                                                  \
    break
  switch (epilogue) {
    PS_SNF_CASE(PS_EPI_NONE);
    PS_SNF_CASE(PS_EPI_GELU_TANH);
    PS_SNF_CASE(PS_EPI_GELU_ERF);
    PS_SNF_CASE(PS_EPI_RELU2);
    default: ps_set_error("ps_linear: unknown epilogue %d", epilogue); return 1;
  }
#undef PS_SNF_CASE
#undef PS_FNF_ROWS
#undef PS_LAUNCH_FNF
#undef PS_LAUNCH_SNF
  PS_CHECK_LAUNCH("ps_linear(skinny, norm, float)");
  return 0;
}

template <int EPI>
static int launch_skinny_f32(const void* a, const void* w, const float* bias, void* c, int m, int n,
                             int k, int lda, int ldc, const KvScatter& scatter, hipStream_t s) {
  const int row_blocks = (m + 15) / 16;
  int k_splits = 1, k_chunk = k;
#define PS_LAUNCH_SF(MB, NT, UNROLL, WAVES)                                                         \
  hipLaunchKernelGGL((gemm_nt_skinny_f32_kernel<EPI, MB, NT, UNROLL, WAVES>),                       \
                     dim3((n + 16 * NT - 1) / (16 * NT), k_splits, (row_blocks + MB - 1) / MB),     \
                     dim3(64 * WAVES), 0, s, (const float*)a, (const float*)w, bias, (float*)c, m,  \
                     n, k, lda, k_chunk, ldc, k_splits, scatter)
  if (EPI == PS_EPI_RESIDUAL && m > 16) {
    // ranges of one round of four waves' loads (32 x 768 x 3072: 7.2 us with ranges of 384, 8.7 with 768)
    k_splits = (k + 4 * 3 * SF_STEP - 1) / (4 * 3 * SF_STEP);
    k_chunk = ((k + k_splits - 1) / k_splits + SF_STEP - 1) / SF_STEP * SF_STEP;
    k_splits = (k + k_chunk - 1) / k_chunk;
    PS_LAUNCH_SF(2, 1, 3, 4);
  } else if (m <= 16) {
    // (up to 1,024 k stay in one block: no atomics)
    if (EPI == PS_EPI_RESIDUAL && k > 1024) {
      k_splits = (k + 8 * 3 * SF_STEP - 1) / (8 * 3 * SF_STEP);
      k_chunk = ((k + k_splits - 1) / k_splits + SF_STEP - 1) / SF_STEP * SF_STEP;
      k_splits = (k + k_chunk - 1) / k_chunk;
    }
    if (k_chunk <= 8 * 3 * SF_STEP) PS_LAUNCH_SF(1, 1, 3, 8);
    else PS_LAUNCH_SF(1, 1, 4, 8);
  } else if (k > 8 * 3 * SF_STEP) PS_LAUNCH_SF(1, 1, 4, 8);
  else if (m <= 32) PS_LAUNCH_SF(2, 1, 3, 8);
  else PS_LAUNCH_SF(2, 2, 3, 8);
#undef PS_LAUNCH_SF
  PS_CHECK_LAUNCH("ps_linear(skinny, float)");
  return 0;
}

int ps_gemm_nt_f32_skinny(const void* a, const void* w, const float* bias, void* c, int m, int n,
                          int k, int lda, int ldc, int epilogue, const KvScatter& scatter,
                          hipStream_t s) {
  if (few_rows_take(m, n, k, epilogue)) {
#define PS_LAUNCH_FEW(PIECES, ROWS)                                                                       \
  hipLaunchKernelGGL((gemm_nt_few_f32_kernel<PIECES, ROWS>), dim3((n + 3) / 4), dim3(256), 0, s,          \
                     (const float*)a, (const float*)w, bias, (float*)c, m, n, k, lda, ldc)
    if (m > 4) {
      if (k <= 512) PS_LAUNCH_FEW(2, 8);
      else if (k <= 768) PS_LAUNCH_FEW(3, 8);
      else PS_LAUNCH_FEW(4, 8);
    } else if (k <= 2048) PS_LAUNCH_FEW(8, 4);
    else if (k <= 3072) PS_LAUNCH_FEW(12, 4);
    else PS_LAUNCH_FEW(16, 4);
#undef PS_LAUNCH_FEW
    PS_CHECK_LAUNCH("ps_linear(few rows, float)");
    return 0;
  }
#define PS_SKINNY_CASE(EPI) \
  case EPI: return launch_skinny_f32<EPI>(a, w, bias, c, m, n, k, lda, ldc, scatter, s)
  switch (epilogue) {
    PS_SKINNY_CASE(PS_EPI_NONE);
    PS_SKINNY_CASE(PS_EPI_GELU_TANH);
    PS_SKINNY_CASE(PS_EPI_GELU_ERF);
    PS_SKINNY_CASE(PS_EPI_RELU2);
    PS_SKINNY_CASE(PS_EPI_RESIDUAL);
    default: ps_set_error("ps_linear: unknown epilogue %d", epilogue); return 1;
  }
#undef PS_SKINNY_CASE
}
