// True 32-bit matrix product of many rows in tiles of 32 x 64 to 64 x 96:
//   C[m, n] = epi(sum_k A[m, k] W[n, k] + b[n]),   k a multiple of 32.
//
// The matrix cores bound it (16,384 products per cycle and chip where bfloat16 has sixteen times as many), so two things
// count: that every SIMD gets about as many products, and that nothing stands between them.
//
// Fragments are 16 x 16 (v_mfma_f32_16x16x4_f32, as many products per cycle as 32 x 32 x 2), four waves to a block, so
// that tiles come in steps of 16 rows and one that fills the units evenly is chosen (even_time below): 193 x 3072 is 240 blocks of 48 x
// 64, 2500 x 3072 six blocks of 80 x 64 to every unit, 2048 x 768 and 544 x 2304 go in 32 x 64, three blocks to a unit and up to three,
// where 64 x 64 leaves some units two and others one.
//
// A wave alone on its SIMD has to issue a product every 32 cycles, seven instructions at most.  With pointers of 64 bits
// and places in the ring by division a load to LDS took nine by itself and the matrix cores stood still: 544 x 768 x 3072
// in 64 x 64 took 57.5 us, 47.6 with neither loads nor reads.  So operands are buffers (one scalar addition per load), the
// place in the ring is stepped, and reads and loads go one by one between the products: 52.7 us.
//
// Stages hold 32 values of k of every row, three or four in a ring, in the order of gemm_tiled.hip (piece c of row r in slot
// c ^ ((r >> 1) & 7): the 16 lanes that read one piece of 16 rows touch every bank once).  The second step of a stage
// meets the other waves in front of its products: the stage has then been read by all of them and the next one has landed.
//
// Four accumulators per fragment take turns and are added to a total every 128 values of k, between the products of the
// steps around: no chain is longer than 32 products.  Against float64, over 150 products of 17 to 2,300 rows and k of 256
// to 6,400: 0.8 to 1.3e-7, where the kernel that took them before was 0.8 to 2.7e-7.
//
// With weights from memory, each product by itself, that kernel (tiles of 64 x 64 to 128 x 128) and this one, us: 2048 x 2304 x 768 70 /
// 61, x 3072 with GELU 95 / 85, 2048 x 768 x 768 added to rows 31 / 22, x 3072 94 / 76 (127 TFLOP/s), 544 x 2304 x 768 30 / 22, 544 x
// 768 x 3072 38 / 31, 193 x 3072 x 1024 23.6 / 17.0, 4101 x 1600 x 1600 211 / 176, 4102 x 3072 x 1024 240 / 204, 4096 x 6400 x 1600 with
// GELU 728 / 656; the output head, 50257 x 768, at 17 rows 60 / 36, 64 64 / 55, 96 106 / 75, 128 107 / 94.  1,001 products of 17 to 8,192
// rows take 0.83 of the time, the most 1.05 (6000 x 512 x 128 12.0 / 12.5).  In a pass, between a layer's other launches, the gain is
// less: 2048 x 2304 x 768 74, x 3072 with GELU 99, the two added to rows 59 on average (97 to 103 TFLOP/s; 77 to 103 and 61 at another
// time), where the kernel before took 103 for the second.
#include <type_traits>

#include "common.h"
#include "linear.h"
#include "pagedserve_hip.h"

#include "gemm_tile.h"

#define GE_BK 32         // values of k per stage: 128 bytes of every row
#define GE_WAVES 4

template <int PENDING>
__device__ __forceinline__ void ge_wait_and_sync() {
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(PENDING) : "memory");
}

template <int I, int N, typename F>
__device__ __forceinline__ void ge_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    ge_for<I + 1, N>(f);
  }
}

#if defined(__HIP_DEVICE_COMPILE__)
// `rows` rows of k values as a buffer: no load reaches beyond them
__device__ __forceinline__ __amdgpu_buffer_rsrc_t ge_operand(const float* first, int rows, int stride, int k) {
  const uint32_t bytes = ((uint32_t)(rows - 1) * (uint32_t)stride + (uint32_t)k) * 4u;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(first), 0, (int)bytes, 0x00027000);
}
#endif

// By assembly, as in gemm_tiled.hip: the step that uses the operands waits first, and touches each of them behind the wait.
template <int OFFSET>
__device__ __forceinline__ void ge_read(u32x4_t& to, uint32_t address) {
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(to) : "v"(address), "n"(OFFSET) : "memory");
}

// WAVES_M of the four waves lie along m; a wave owns FM x FN fragments.  ADDED: a range of k per block, whose sums are
// added to C by atomics.  `form`: bit 0, tiles run along the rows of C; above it the number of ranges of `range` values.
template <int WAVES_M, int FM, int FN, int STAGES, int EPI, bool ADDED>
__global__ __launch_bounds__(64 * GE_WAVES, FM * FN < 4 ? 3 : 2) void gemm_nt_even_f32_kernel(
    const float* __restrict__ a, const float* __restrict__ w, int m, int n, int k, int lda, int ldc, int form,
    float* __restrict__ c, const float* __restrict__ bias, int range, KvScatter scatter) {
#if defined(__HIP_DEVICE_COMPILE__)      // (the host's pass knows no buffer resources)
  constexpr int WAVES_N = GE_WAVES / WAVES_M;
  constexpr int BM = 16 * FM * WAVES_M, BN = 16 * FN * WAVES_N;
  constexpr int STAGE_BYTES = (BM + BN) * TB_ROW;
  constexpr int GROUPS = (BM + BN) / 8;                  // load instructions of a stage, eight rows each
  constexpr int LOADS = (GROUPS + GE_WAVES - 1) / GE_WAVES;
  static_assert(STAGES >= 2 && STAGES <= 8 && BM % 16 == 0 && BN % 16 == 0, "tiles of whole fragments");
  static_assert(LOADS * (STAGES - 1) < 64, "the load counter has six bits");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[STAGES * STAGE_BYTES];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave_m = wave % WAVES_M, wave_n = wave / WAVES_M;
  // every XCD works on a contiguous run of tiles, along the rows of C or down its columns (see gemm_tiled.hip)
  const bool row_major = form & 1;
  const int ranges = form >> 1;
  const int tiles_m = (m + BM - 1) / BM, tiles_n = (n + BN - 1) / BN;
  const int per_xcd = tiles_m * tiles_n * ranges / 8;
  int tile = blockIdx.x;
  if (blockIdx.x < per_xcd * 8) tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  int k_begin = 0, k_tiles = k / GE_BK;
  if constexpr (ADDED) {
    const int which = tile / (tiles_m * tiles_n);
    tile -= which * tiles_m * tiles_n;
    k_begin = which * range;
    k_tiles = min(range, k - k_begin) / GE_BK;
    if (which > 0) bias = nullptr;
  }
  const int line = row_major ? tiles_n : tiles_m;
  const int outer = tile / line, inner = tile - outer * line;
  const int m0 = (row_major ? outer : inner) * BM;
  const int n0 = (row_major ? inner : outer) * BN;

  // ---- loads: lane l of an instruction fills slot l % 8 of row l / 8 of its eight rows.  Where the groups do not go
  // round, the last waves fetch the last group once more.
  const __amdgpu_buffer_rsrc_t from_a = ge_operand(a + (int64_t)m0 * lda + k_begin, min(BM, m - m0), lda, k_tiles * GE_BK);
  const __amdgpu_buffer_rsrc_t from_w = ge_operand(w + (int64_t)n0 * k + k_begin, min(BN, n - n0), k, k_tiles * GE_BK);
  uint32_t offset[LOADS];
  int target[LOADS];
  bool of_a[LOADS];
#pragma unroll
  for (int j = 0; j < LOADS; ++j) {
    const int group = j * GE_WAVES + wave < GROUPS ? j * GE_WAVES + wave : GROUPS - 1;
    const int row = group * 8 + (lane >> 3);
    const int piece = (lane & 7) ^ ((row >> 1) & 7);
    of_a[j] = group * 8 < BM;
    offset[j] = (of_a[j] ? (uint32_t)min(row, m - 1 - m0) * (uint32_t)lda : (uint32_t)min(row - BM, n - 1 - n0) * (uint32_t)k) * 4u +
                piece * 16;
    target[j] = group * 8 * TB_ROW;
  }
  // `k_at`: bytes along the rows, `fill`: the stage in the ring
  auto load = [&](uint32_t k_at, uint32_t fill, int j) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(of_a[j] ? from_a : from_w, (lds_ptr_t)(lds + fill + target[j]), 16, offset[j],
                                             k_at, 0, 0);
  };

  // Four accumulators take turns in a fragment's products.  Every RUN stages they are added to each other and then to a
  // total, and start anew, so that no chain is longer than 32 products.
  constexpr int ACCS = 4, RUN = 4, FRAGMENTS = FM * FN;
  f32x4 sums[FRAGMENTS][ACCS], total[FRAGMENTS], pair[FRAGMENTS];
#pragma unroll
  for (int f = 0; f < FRAGMENTS; ++f) {
#pragma unroll
    for (int p = 0; p < ACCS; ++p) sums[f][p] = f32x4{0.f, 0.f, 0.f, 0.f};
    total[f] = pair[f] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // ---- operands: lane l reads the 16 bytes of k piece 4 s + l / 16 of row l % 16
  const int key = (lane >> 1) & 7;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_ptr_t)lds;
  uint32_t row_at[2][2];     // of a and w, in each step
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const uint32_t slot = (uint32_t)(((4 * q + (lane >> 4)) ^ key) << 4);
    row_at[0][q] = lds_base + (wave_m * FM * 16 + (lane & 15)) * TB_ROW + slot;
    row_at[1][q] = lds_base + (BM + wave_n * FN * 16 + (lane & 15)) * TB_ROW + slot;
  }
  constexpr int READS = FM + FN, PRODUCTS = 4 * FM * FN;
  u32x4_t operands[2][READS];
  auto read = [&](uint32_t stage_at, auto step, auto index, u32x4_t* to) {
    constexpr int R = decltype(index)::value, S = decltype(step)::value;
    ge_read<(R < FM ? R : R - FM) * 16 * TB_ROW>(to[R], stage_at + row_at[R < FM ? 0 : 1][S]);
  };
  // Step S of a stage: the products of operands[S], the reads of the next step's operands and half of a stage's loads
  // between them.  LOAD: the stage that is asked for exists; AHEAD: how many stages behind the next one may be on their
  // way when that one has to be there, -1: there is no next step.
  constexpr int FIRST_PART = (LOADS + 1) / 2;
  uint32_t here = 0, k_next = (uint32_t)(STAGES - 1) * TB_ROW;      // the stage that is multiplied, in the ring
  auto around = [](uint32_t at) { return at + STAGE_BYTES < STAGES * STAGE_BYTES ? at + STAGE_BYTES : 0u; };
  auto back = [](uint32_t at) { return at >= STAGE_BYTES ? at - STAGE_BYTES : (STAGES - 1) * STAGE_BYTES; };
  auto step = [&](auto which, auto loads, auto ahead, auto begins, auto ends) {
    constexpr int S = decltype(which)::value, AHEAD = decltype(ahead)::value;
    constexpr bool LOAD = decltype(loads)::value, NEXT = AHEAD >= 0, LAST = S == 1;
    constexpr bool BEGINS = decltype(begins)::value, ENDS = decltype(ends)::value;
    constexpr int FROM = LAST ? 0 : FIRST_PART, COUNT = LAST ? FIRST_PART : LOADS - FIRST_PART;
    // (the first part of a stage's loads goes where the stage at hand lay, the other one where the one before did)
    const uint32_t next_stage = LAST ? around(here) : here, fill = LAST ? here : back(here);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if constexpr (LAST && NEXT) ge_wait_and_sync<(AHEAD > 0 ? AHEAD : 0) * LOADS>();
#pragma unroll
    for (int r = 0; r < READS; ++r) asm volatile("" : "+v"(operands[S][r]));   // used only behind the wait
    ge_for<0, PRODUCTS>([&](auto product) {
      constexpr int Q = decltype(product)::value;
      constexpr int V = Q / FRAGMENTS, F = Q % FRAGMENTS, I = F / FN, J = F % FN;
      // Rows of the result are columns of C: a lane then holds four consecutive columns of one row, the lanes of an
      // instruction 64 bytes of 16 rows each.  Where sums are added by atomics they are rows: 16 lanes side by side.
      const float x = __builtin_bit_cast(float, (uint32_t)operands[S][I][V]);
      const float y = __builtin_bit_cast(float, (uint32_t)operands[S][FM + J][V]);
      const f32x4 before = BEGINS ? f32x4{0.f, 0.f, 0.f, 0.f} : sums[F][V];
      sums[F][V] = ADDED ? __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, before, 0, 0, 0)
                         : __builtin_amdgcn_mfma_f32_16x16x4f32(y, x, before, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      // a run ends: the first two accumulators behind their last product, the others in front of their next one
      if constexpr (ENDS && V == 2) pair[F] = sums[F][0] + sums[F][1];
      if constexpr (BEGINS && V == 0) pair[F] += sums[F][2] + sums[F][3];
      if constexpr (BEGINS && V == 1) total[F] += pair[F];
      if constexpr (NEXT)
        ge_for<(Q * READS * 2 / PRODUCTS < READS ? Q * READS * 2 / PRODUCTS : READS),
               ((Q + 1) * READS * 2 / PRODUCTS < READS ? (Q + 1) * READS * 2 / PRODUCTS : READS)>([&](auto index) {
          read(next_stage, std::integral_constant<int, 1 - S>{}, index, operands[1 - S]);
        });
      if constexpr (LOAD)
        ge_for<0, COUNT>([&](auto index) {
          constexpr int L = decltype(index)::value;
          if constexpr (Q == (2 * L + 1) * PRODUCTS / (2 * COUNT)) load(k_next, fill, FROM + L);
        });
      __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (LAST) here = next_stage;
    else k_next += TB_ROW;
  };
  using Zero = std::integral_constant<int, 0>;
  using One = std::integral_constant<int, 1>;
  using Yes = std::true_type;
  using No = std::false_type;
  // stages 0 .. STAGES - 2, and the first part of stage STAGES - 1 (the host sends no product of fewer stages)
#pragma unroll
  for (int d = 0; d < STAGES - 1; ++d)
#pragma unroll
    for (int j = 0; j < LOADS; ++j) load(d * TB_ROW, d * STAGE_BYTES, j);
#pragma unroll
  for (int j = 0; j < FIRST_PART; ++j) load((STAGES - 1) * TB_ROW, (STAGES - 1) * STAGE_BYTES, j);
  ge_wait_and_sync<(STAGES - 2) * LOADS + FIRST_PART>();
  ge_for<0, READS>([&](auto index) { read(0, Zero{}, index, operands[0]); });
  using Full = std::integral_constant<int, STAGES - 2>;
  // The stages that make no whole run, whole runs, and the last STAGES stages as a run of their own; the first of those
  // still asks for the other part of the last one.
  const int ahead_of_last = k_tiles - STAGES;
  for (int stage = 0; stage < ahead_of_last % RUN; ++stage) {
    step(Zero{}, Yes{}, Full{}, No{}, No{});
    step(One{}, Yes{}, Full{}, No{}, No{});
  }
#pragma unroll
  for (int f = 0; f < FRAGMENTS; ++f) pair[f] = sums[f][0] + sums[f][1];
  for (int run = 0; run < ahead_of_last / RUN; ++run) {
    ge_for<0, RUN>([&](auto index) {
      constexpr int T = decltype(index)::value;
      step(Zero{}, Yes{}, Full{}, std::integral_constant<bool, T == 0>{}, No{});
      step(One{}, Yes{}, Full{}, No{}, std::integral_constant<bool, T == RUN - 1>{});
    });
  }
  ge_for<0, STAGES>([&](auto index) {
    constexpr int T = decltype(index)::value;
    step(Zero{}, std::integral_constant<bool, T == 0>{}, Full{}, std::integral_constant<bool, T == 0>{}, No{});
    step(One{}, No{}, std::integral_constant<int, T == STAGES - 1 ? -1 : (STAGES - 2 - T > 0 ? STAGES - 2 - T : 0)>{}, No{},
         No{});
  });
  auto result = [&](int f) { return total[f] + ((sums[f][0] + sums[f][1]) + (sums[f][2] + sums[f][3])); };

  if constexpr (ADDED) {
    const int row0 = m0 + wave_m * FM * 16 + (lane >> 4) * 4;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int col = n0 + (wave_n * FN + j) * 16 + (lane & 15);
      const float shift = bias != nullptr && col < n ? bias[col] : 0.f;
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const f32x4 v = result(i * FN + j) + shift;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = row0 + i * 16 + e;
          if (row < m && col < n) unsafeAtomicAdd(c + (int64_t)row * ldc + col, v[e]);
        }
      }
    }
    return;
  }

  // ---- epilogue: lane l holds columns 4 (l / 16) .. + 3 of row l % 16 of every fragment
  const bool whole = ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(c) & 15u) == 0 &&
                     (EPI != PS_EPI_NONE || scatter.k_pool == nullptr ||
                      ((scatter.head_dim | scatter.q_cols | scatter.kv_cols) & 3) == 0);
  const int row0 = m0 + wave_m * FM * 16 + (lane & 15);
  const int col0 = n0 + wave_n * FN * 16 + (lane >> 4) * 4;
  int64_t slots[FM];
  const bool paged = EPI == PS_EPI_NONE && scatter.k_pool != nullptr && n0 + BN > scatter.q_cols;
  if (paged) {
#pragma unroll
    for (int i = 0; i < FM; ++i) slots[i] = kv_scatter_row(scatter, min(row0 + i * 16, m - 1));
  }
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int col = col0 + j * 16;
    const bool full = whole && col + 4 <= n;
    f32x4 shift = {0.f, 0.f, 0.f, 0.f};
    if (bias != nullptr) {
#pragma unroll
      for (int e = 0; e < 4; ++e) shift[e] = col + e < n ? bias[col + e] : 0.f;
    }
    f32x4 v[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      v[i] = result(i * FN + j) + shift;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[i][e] = apply_activation<EPI>(v[i][e]);
    }
    if (full) {
      float* pool = nullptr;
      int64_t pool_offset = 0;
      if (paged) pool = kv_scatter_col<float>(scatter, col, &pool_offset);
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const int row = row0 + i * 16;
        if (row >= m) continue;
        f32x4* to = reinterpret_cast<f32x4*>(c + (int64_t)row * ldc + col);
        if constexpr (EPI == PS_EPI_RESIDUAL) v[i] += *to;
        if (!(pool != nullptr && scatter.cache_only)) *to = v[i];
        if (pool != nullptr && slots[i] >= 0) *reinterpret_cast<f32x4*>(pool + slots[i] + pool_offset) = v[i];
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (col + e >= n) continue;
        float* pool = nullptr;
        int64_t pool_offset = 0;
        if (paged) pool = kv_scatter_col<float>(scatter, col + e, &pool_offset);
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          const int row = row0 + i * 16;
          if (row >= m) continue;
          float* to = c + (int64_t)row * ldc + col + e;
          if constexpr (EPI == PS_EPI_RESIDUAL) *to += v[i][e];
          else *to = v[i][e];
          if (pool != nullptr && slots[i] >= 0) pool[slots[i] + pool_offset] = v[i][e];
        }
      }
    }
  }
#endif
}

// --------------------------------------------------------------------------------- host
template <int WAVES_M, int FM, int FN, int STAGES>
static int launch_even(const void* a, const void* w, const float* bias, void* c, int m, int n, int k, int lda, int ldc,
                       int epilogue, int ranges, const KvScatter& scatter, hipStream_t s) {
  constexpr int BM = 16 * FM * WAVES_M, BN = 16 * FN * (GE_WAVES / WAVES_M);
  const int tiles_m = (m + BM - 1) / BM, tiles_n = (n + BN - 1) / BN;
  const int range = (k / GE_BK + ranges - 1) / ranges * GE_BK;
  ranges = (k + range - 1) / range;
  PS_REQUIRE((k - (ranges - 1) * range) / GE_BK >= STAGES, "ps_linear: k of %d in %d ranges is too short for these tiles", k, ranges);
  PS_REQUIRE((int64_t)tiles_m * tiles_n * ranges < ((int64_t)1 << 30), "ps_linear: too many tiles");
  // what one XCD's run of tiles fetches into its L2, in rows of k values
  const int run = (tiles_m * tiles_n + 7) / 8;
  const int64_t rows_along = (int64_t)((run + tiles_n - 1) / tiles_n) * BM + n;
  const int64_t rows_down = (int64_t)((run + tiles_m - 1) / tiles_m) * BN + m;
  const int form = (rows_along < rows_down ? 1 : 0) + 2 * ranges;
  dim3 grid(tiles_m * tiles_n * ranges);
#define PS_LAUNCH_GE(EPI, ADDED)                                                                           \
  hipLaunchKernelGGL((gemm_nt_even_f32_kernel<WAVES_M, FM, FN, STAGES, EPI, ADDED>), grid,                 \
                     dim3(64 * GE_WAVES), 0, s, (const float*)a, (const float*)w, m, n, k, lda, ldc, form, \
                     (float*)c, bias, range, scatter)
  switch (epilogue) {
    case PS_EPI_NONE: PS_LAUNCH_GE(PS_EPI_NONE, false); break;
    case PS_EPI_GELU_TANH: PS_LAUNCH_GE(PS_EPI_GELU_TANH, false); break;
    case PS_EPI_GELU_ERF: PS_LAUNCH_GE(PS_EPI_GELU_ERF, false); break;
    case PS_EPI_RELU2: PS_LAUNCH_GE(PS_EPI_RELU2, false); break;
    case PS_EPI_RESIDUAL:
      if (ranges > 1) PS_LAUNCH_GE(PS_EPI_RESIDUAL, true);
      else PS_LAUNCH_GE(PS_EPI_RESIDUAL, false);
      break;
    default: ps_set_error("ps_linear: unknown epilogue %d", epilogue); return 1;
  }
#undef PS_LAUNCH_GE
  PS_CHECK_LAUNCH("ps_linear(even tiles, float)");
  return 0;
}

// The tiles by number.  `resident`: how many blocks share a compute unit, by registers and LDS.
static const struct {
  int rows, columns, stages, resident;
} even_tiles[] = {{32, 64, 4, 3}, {48, 64, 4, 2}, {64, 64, 3, 2}, {80, 64, 3, 2}, {64, 96, 3, 2}};
#define GE_TILES ((int)(sizeof(even_tiles) / sizeof(even_tiles[0])))
#define GE_SHORTEST_RANGE 256

#define PS_EVEN_ARGUMENTS                                                                                           \
  const void *a, const void *w, const float *bias, void *c, int m, int n, int k, int lda, int ldc, int epilogue,    \
      int tile, int ranges, const KvScatter &scatter, hipStream_t s

static int launch_even_tile(PS_EVEN_ARGUMENTS) {
#define PS_EVEN(...) launch_even<__VA_ARGS__>(a, w, bias, c, m, n, k, lda, ldc, epilogue, ranges, scatter, s)
  switch (tile) {
    case 0: return PS_EVEN(1, 2, 1, 4);
    case 1: return PS_EVEN(1, 3, 1, 4);
    case 2: return PS_EVEN(1, 4, 1, 3);
    case 3: return PS_EVEN(1, 5, 1, 3);
    default: return PS_EVEN(2, 2, 3, 3);
  }
#undef PS_EVEN
}

// Microseconds, about: what it takes to begin and end a tile, for every stage the products of the unit with the most
// tiles and 0.08 us that its blocks do not hide from each other, and the atomic additions of several ranges.  Fitted to
// 1,300 timings (17 to 2,300 rows, 15 pairs of n and k, every tile and 1 to 12 ranges; 6 % off in the mean): the tile that
// it picks takes 1.012 of the fastest one's time on average, 1.26 at most.
static float even_time(int m, int n, int k, int tile, int ranges, int units) {
  const auto& t = even_tiles[tile];
  const int64_t blocks = (int64_t)((m + t.rows - 1) / t.rows) * ((n + t.columns - 1) / t.columns) * ranges;
  const float area = t.rows * t.columns / 1024.f;
  const float fullest = (float)((blocks + units - 1) / units);
  const int stages = (k / GE_BK + ranges - 1) / ranges;
  const float added = ranges > 1 ? 2.4f + 1.8e-6f * (float)m * (float)n * (float)ranges : 0.f;
  return 1.05f * area + stages * (0.109f * area * fullest + 0.08f * ceilf(fullest / t.resident)) + added;
}

// Ranges of k only where C is added to anyway, over a k of more than 1,024 and with at most one and a half tiles of 64 x 64 to
// a unit.  Elsewhere sums keep an order that does not change from call to call; ranges would gain there (us, one range and
// several: 224 x 768 x 768 10.1 / 7.7, 160 x 1024 x 1024 12.1 / 8.3, 256 x 1024 x 1024 12.4 / 10.1, 1024 x 1600 x 6400 199 / 178).
static void choose_even(int m, int n, int k, int epilogue, int* best_tile, int* best_ranges) {
  const int units = ps_compute_units();
  const int64_t tiles_64 = (int64_t)((m + 63) / 64) * ((n + 63) / 64);
  const int most = epilogue == PS_EPI_RESIDUAL && k > 1024 && 2 * tiles_64 <= 3 * units ? 12 : 1;
  float least = INFINITY;
  *best_tile = 0;
  *best_ranges = 1;
  for (int tile = 0; tile < GE_TILES; ++tile)
    for (int ranges = 1; ranges <= most; ++ranges) {
      const int stages = (k / GE_BK + ranges - 1) / ranges;
      const int shortest = k / GE_BK - (ranges - 1) * stages;
      if (ranges > 1 && shortest * GE_BK < GE_SHORTEST_RANGE) continue;
      const float time = even_time(m, n, k, tile, ranges, units);
      if (time < least) {
        least = time;
        *best_tile = tile;
        *best_ranges = ranges;
      }
    }
}

// (a tile's rows lie within 32-bit offsets; the ring of four stages wants as many)
bool ps_gemm_nt_f32_even_takes(int m, int n, int k, int lda) {
  return m > 0 && n > 0 && k % GE_BK == 0 && k >= 4 * GE_BK && k <= (1 << 22) && lda <= (1 << 22);
}

int ps_gemm_nt_f32_even(const void* a, const void* w, const float* bias, void* c, int m, int n, int k, int lda, int ldc,
                        int epilogue, const KvScatter& scatter, hipStream_t s) {
  int tile, ranges;
  choose_even(m, n, k, epilogue, &tile, &ranges);
  return launch_even_tile(a, w, bias, c, m, n, k, lda, ldc, epilogue, tile, ranges, scatter, s);
}

// The tile and number of ranges that a product gets, tile + 16 * ranges, -1: not this kernel; for tests.
extern "C" int ps_gemm_nt_even_choice(int m, int n, int k, int epilogue) {
  if (!ps_gemm_nt_f32_even_takes(m, n, k, k)) return -1;
  int tile, ranges;
  choose_even(m, n, k, epilogue, &tile, &ranges);
  return tile + 16 * ranges;
}

// The product in a given tile and number of ranges, for tests and measurements.
extern "C" int ps_gemm_nt_even(const void* a, const void* w, const float* bias, void* c, int m, int n, int k, int lda,
                               int ldc, int epilogue, int tile, int ranges, void* stream) {
  PS_REQUIRE(a && w && c && ps_gemm_nt_f32_even_takes(m, n, k, lda) && lda >= k && lda % 4 == 0 && ldc >= n &&
                 ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(w)) & 15u) == 0,
             "ps_gemm_nt_even: bad sizes or unaligned operand (m %d, n %d, k %d, lda %d, ldc %d)", m, n, k, lda, ldc);
  PS_REQUIRE(tile >= 0 && tile < GE_TILES && ranges >= 1 && (ranges == 1 || epilogue == PS_EPI_RESIDUAL),
             "ps_gemm_nt_even: no tile %d in %d ranges", tile, ranges);
  KvScatter none = {};
  return launch_even_tile(a, w, bias, c, m, n, k, lda, ldc, epilogue, tile, ranges, none, (hipStream_t)stream);
}
