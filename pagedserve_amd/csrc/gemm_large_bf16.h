// bfloat16 matrix product of hundreds to thousands of rows in tiles of 128 x 64 to 256 x 320:
//   C[m, n] = epi(sum_k A[m, k] W[n, k] + b[n]),   k a multiple of 32.
//
// Eight waves, four along m and two along n, one block per compute unit; a wave owns 32 FM rows x 32 FN columns,
// FM being 1 or 2 and FN 1 to 5.  Both operands go from global memory straight into LDS in stages of ROW bytes of
// every row, three to six of them in a ring.  Two things bound such a block.
//
// What it takes in: a compute unit gets 45 KB/us of stages of 64-byte rows and 60 to 75 of 128-byte rows, which are
// whole lines of the L2 (2048 x 2304 x 3072 in tiles of 128 x 192: 48 us with 64 bytes, 38 with 128; 256 x 128 at
// 4096 x 1600 x 6400: 115 and 98).  Tiles up to 256 x 128 therefore have rows of 128 bytes.
//
// LDS, at the larger tiles: loads fill it at 64 bytes per cycle and reads take 128, one after the other (a lone block
// of 64 x 64 takes 500 cycles for a k tile of 64, 250 of each, however many stages or operands are fetched ahead).
// A block of 256 x BN therefore needs 2 (256 + BN) + 512 + 4 BN cycles per 64 values of k where its products take
// 8 BN: the tiles are as large as registers and LDS allow.  There the number of stages counts for more than the
// lines (256 x 320 at 4096 x 4800 x 1600: four of 64 bytes 65 us, two of 128 bytes 70; 256 x 256 at 4096 x 6400 x
// 1600 104 and 109; 256 x 192 at 4096 x 2304 x 768 23.6 and 25.4).
//
// A load instruction blocks its wave until the address unit takes it.  Eight in a row kept the matrix cores idle at
// the head of every stage (8,192 cubed: 1.21 PFLOP/s with the loads in a row, 1.98 with none, which is the
// clock's limit), so each step issues its share of loads and its reads of the next step's operands between its
// products.  A step is 16 values of k, SUB = 2 or 4 steps to a stage.  The last step of stage s meets the other waves
// in front of its products: stage s has then been read by all of them, and stage s + 1 has landed.  It asks for the
// first part of stage s + RING, the steps of stage s + 1 but the last for the other parts.
//
// A stage holds 64 or 128 bytes of every row; piece c (16 bytes) of row r lies in slot c ^ ((r >> 2) & 3) or
// c ^ ((r >> 1) & 7), so that the 16 lanes that read one piece of 16 consecutive rows touch every bank once.
//
// Measured with weights from memory, in us, against the kernels that these products went to before (64 x 256 with
// the weights past LDS, and the ring of 128 x 128): 4096 x 4800 x 1600 75 / 88, 4096 x 6400 x 1600 107 / 118,
// 8192 x 2304 x 768 45 / 51, 8192 x 3072 x 768 58 / 67, 4096 x 4096 x 1024 44 / 55, 2048 x 6400 x 1600 57 / 73.  In tiles
// of up to 256 x 128, against the same: 4096 x 1600 x 6400 98 / 131, 2048 x 3072 x 768 18.0 / 19.9, 2048 x 2304 x 768
// 13.9 / 16.7, 2048 x 3072 x 1024 20 / 24, 544 x 4096 x 1024 13.6 / 14.9, 544 x 3072 x 1024 9.9 / 11.7.  In a
// prefill that lasts 0.2 s the card's power sets the clock and 4096 x 6400 x 1600 is level (104 / 102).  What is
// left beside the products is the ends of the tiles, in which a unit that holds one block multiplies nothing.  They
// waited for memory one trip after the other: for the arguments behind the preloaded ones in front of the first load,
// then, all products done, for the bias, the rows added to and the pages.  Tile numbers now come of the preloaded
// arguments and the rest is asked for in the last two stages: 4096 x 6400 x 1600 107 to 101 us in that prefill, 4096 x
// 1600 x 1600 and 6400 (their mean) 62.1 to 58.0, 544 x 4096 x 1024 14.4 to 13.9.
#pragma once
#include <type_traits>

#include "gemm_tile.h"

#define GL_WAVES_M 4
#define GL_WAVES_N 2

template <int I, int N, typename F>
__device__ __forceinline__ void gl_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    gl_for<I + 1, N>(f);
  }
}

// By assembly, as in gemm_tiled.hip: the compiler would wait for every load in flight before an LDS read.  The step
// that uses the operands waits first, and touches each of them behind the wait.  (The compiler does not know that they
// are on their way until then: a test of the built code looks for registers that are used before.)
template <int OFFSET>
__device__ __forceinline__ void gl_read(u32x4_t& to, uint32_t address) {
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(to) : "v"(address), "n"(OFFSET) : "memory");
}

template <int PENDING>
__device__ __forceinline__ void gl_wait_and_sync() {
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(PENDING) : "memory");
}

// The columns of a wave in slices of SLICE fragments: the region of LDS that a slice is turned through is smaller.
// `first`: what has been asked for of the first slice; `pages`, `tail`: the rows' pages, as whole slices and as a
// narrower last one hold them.
template <int FM, int FN, int SLICE, int FIRST, typename TOut, int EPI>
__device__ __forceinline__ void gl_store(f32x16 (&acc)[FM][FN], float* region, int lane, int row, int col,
                                         int m, int n, int ldc, TOut* c, const float* bias,
                                         const KvScatter& scatter, const TileEnds<FM, SLICE, TOut, EPI>& first,
                                         const TilePages<FM, SLICE>& pages,
                                         const TilePages<FM, FN % SLICE ? FN % SLICE : SLICE>& tail) {
  if constexpr (FIRST < FN) {
    constexpr int COUNT = FIRST + SLICE <= FN ? SLICE : FN - FIRST;
    f32x16 slice[FM][COUNT];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < COUNT; ++j) slice[i][j] = acc[i][FIRST + j];
    auto store = [&](const auto& ends, const auto& rows) {
      store_wave_tile<FM, COUNT, TOut, EPI>(slice, region, lane, row, col + FIRST * 32, m, n, ldc, c, bias, 0, 1,
                                            scatter, ends, rows);
    };
    if constexpr (FIRST == 0) {
      store(first, pages);
    } else {
      TileEnds<FM, COUNT, TOut, EPI> ends;
      ends.ask(lane, row, col + FIRST * 32, m, n, ldc, c, bias, 0, tile_by_column<TOut, EPI>(c, ldc, 1, scatter));
      if constexpr (COUNT == SLICE) store(ends, pages);
      else store(ends, tail);
    }
    gl_store<FM, FN, SLICE, FIRST + COUNT, TOut, EPI>(acc, region, lane, row, col, m, n, ldc, c, bias, scatter,
                                                      first, pages, tail);
  }
}

// What a block of 8 waves does: tile `block` of `blocks` of C.  `lds`: RING stages.
template <int FM, int FN, int ROW, int RING, typename TOut, int EPI>
__device__ __forceinline__ void gl_tile(unsigned char* lds, const int block, const int blocks, const bf16_t* __restrict__ a,
                                        const bf16_t* __restrict__ w, const int m, const int n, const int k, const int lda,
                                        const int panel, const int ldc, TOut* __restrict__ c,
                                        const float* __restrict__ bias, const KvScatter& scatter) {
  constexpr int WAVES = GL_WAVES_M * GL_WAVES_N;
  constexpr int BM = 32 * FM * GL_WAVES_M, BN = 32 * FN * GL_WAVES_N;
  static_assert(ROW == 64 || ROW == 128, "rows of half a line or of a whole one");
  constexpr int SUB = ROW / 32;                          // steps of a stage
  constexpr int PIECES = ROW / 16, SHIFT = ROW == 64 ? 2 : 1;
  constexpr int GROUP = 1024 / ROW;                      // rows of a stage that a load instruction fills
  constexpr int STAGE_BYTES = (BM + BN) * ROW;
  constexpr int GROUPS = (BM + BN) / GROUP;
  constexpr int LOADS = (GROUPS + WAVES - 1) / WAVES;
  constexpr int FIRST_PART = (LOADS + SUB - 1) / SUB;    // part p: the loads from p LOADS / SUB on, rounded up
  constexpr int READS = FM + FN, PRODUCTS = FM * FN;
  static_assert((RING - 1) * LOADS + FIRST_PART < 64, "the load counter has six bits");

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // the same in every lane: scalar
  const int wave_m = wave % GL_WAVES_M, wave_n = wave / GL_WAVES_M;
  // every XCD works on a contiguous run of tiles (see gemm_tiled.hip): panels of `panel` rows of tiles, walked
  // column by column, so that what runs at one time on an XCD is about as many rows as columns
  const int tiles_m = (m + BM - 1) / BM, tiles_n = (n + BN - 1) / BN;
  const int per_xcd = blocks / 8;
  int tile = block;
  if (block < per_xcd * 8) tile = (block & 7) * per_xcd + (block >> 3);
  const int first_row = tile / (panel * tiles_n) * panel;
  const int within = tile - first_row * tiles_n;
  const int panel_rows = min(panel, tiles_m - first_row);
  const int m0 = (first_row + within % panel_rows) * BM;
  const int n0 = within / panel_rows * BN;
  const int stages = k / (ROW / 2);

  // ---- loads: lane l of an instruction fills slot l % PIECES of row l / PIECES of its rows.  Rows beyond m or n are
  // fetched from the last valid one (they feed outputs that are never stored).  Where the groups do not go
  // round, the last waves fetch the last group once more.
  const char* base_a = reinterpret_cast<const char*>(a + (int64_t)m0 * lda);
  const char* base_w = reinterpret_cast<const char*>(w + (int64_t)n0 * k);
  uint32_t offset[LOADS];
  int target[LOADS];
  bool of_a[LOADS];
#pragma unroll
  for (int j = 0; j < LOADS; ++j) {
    const int group = j * WAVES + wave < GROUPS ? j * WAVES + wave : GROUPS - 1;
    const int row = group * GROUP + lane / PIECES;
    const int piece = (lane & (PIECES - 1)) ^ ((row >> SHIFT) & (PIECES - 1));
    of_a[j] = group * GROUP < BM;
    offset[j] = of_a[j] ? (uint32_t)min(row, m - 1 - m0) * (uint32_t)lda * 2u + piece * 16
                        : (uint32_t)min(row - BM, n - 1 - n0) * (uint32_t)k * 2u + piece * 16;
    target[j] = group * GROUP * ROW;
  }
  auto load = [&](int stage, int j) {
    const char* base = (of_a[j] ? base_a : base_w) + (int64_t)stage * ROW;
    __builtin_amdgcn_global_load_lds((global_ptr_t)(base + offset[j]),
                                     (lds_ptr_t)(lds + (stage % RING) * STAGE_BYTES + target[j]), 16, 0, 0);
  };

  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // ---- operands: lane l reads the 16 bytes of k piece 2 s + l / 32 of row l % 32
  const int key = (lane >> SHIFT) & (PIECES - 1);
  const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_ptr_t)lds;
  const uint32_t a_row = lds_base + (wave_m * FM * 32 + (lane & 31)) * ROW;
  const uint32_t w_row = lds_base + (BM + wave_n * FN * 32 + (lane & 31)) * ROW;
  uint32_t slot[SUB];
#pragma unroll
  for (int q = 0; q < SUB; ++q) slot[q] = (uint32_t)(((2 * q + (lane >> 5)) ^ key) << 4);
  u32x4_t operands[2][READS];
  auto read = [&](uint32_t stage_offset, auto step, auto index, u32x4_t* to) {
    constexpr int R = decltype(index)::value;
    const uint32_t at = stage_offset + slot[decltype(step)::value] + (R < FM ? a_row : w_row);
    gl_read<(R < FM ? R : R - FM) * 32 * ROW>(to[R], at);
  };
  // Step S of a stage: the products of operands[S % 2], the reads of the next step's operands and a part of a stage's
  // loads between them.  LOAD: the stage that is asked for exists; AHEAD: how many stages behind the next one may
  // be on their way when that one has to be there, -1: there is no next step.
  auto step = [&](int stage, auto which, auto loads, auto ahead) {
    constexpr int S = decltype(which)::value, AHEAD = decltype(ahead)::value;
    constexpr bool LOAD = decltype(loads)::value, NEXT = AHEAD >= 0;
    constexpr bool LAST = S == SUB - 1;
    constexpr int PART = (S + 1) % SUB;
    constexpr int FROM = (PART * LOADS + SUB - 1) / SUB, COUNT = ((PART + 1) * LOADS + SUB - 1) / SUB - FROM;
    const uint32_t next_stage = (uint32_t)(((LAST ? stage + 1 : stage) % RING) * STAGE_BYTES);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if constexpr (LAST && NEXT) gl_wait_and_sync<(AHEAD > 0 ? AHEAD : 0) * LOADS>();
#pragma unroll
    for (int r = 0; r < READS; ++r) asm volatile("" : "+v"(operands[S & 1][r]));   // used only behind the wait
    gl_for<0, PRODUCTS>([&](auto product) {
      constexpr int Q = decltype(product)::value;
      constexpr int I = Q / FN, J = Q % FN;
      acc[I][J] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, operands[S & 1][I]),
                                                          __builtin_bit_cast(bf16x8, operands[S & 1][FM + J]),
                                                          acc[I][J], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (NEXT)
        gl_for<Q * READS / PRODUCTS, (Q + 1) * READS / PRODUCTS>([&](auto index) {
          read(next_stage, std::integral_constant<int, PART>{}, index, operands[(S + 1) & 1]);
        });
      if constexpr (LOAD)
        gl_for<0, COUNT>([&](auto index) {
          constexpr int L = decltype(index)::value;
          if constexpr (Q == (2 * L + 1) * PRODUCTS / (2 * COUNT))
            load(LAST ? stage + RING : stage + RING - 1, FROM + L);
        });
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  using Zero = std::integral_constant<int, 0>;
  using Last = std::integral_constant<int, SUB - 1>;
  using Yes = std::true_type;
  using No = std::false_type;

  // stages 0 .. RING - 2, and the first part of stage RING - 1 (the host sends no product of fewer than RING stages)
#pragma unroll
  for (int d = 0; d < RING - 1; ++d)
#pragma unroll
    for (int j = 0; j < LOADS; ++j) load(d, j);
#pragma unroll
  for (int j = 0; j < FIRST_PART; ++j) load(RING - 1, j);
  gl_wait_and_sync<(RING - 2) * LOADS + FIRST_PART>();
  gl_for<0, READS>([&](auto index) { read(0, Zero{}, index, operands[0]); });
  using Full = std::integral_constant<int, RING - 2>;
  int stage = 0;
  for (; stage + RING < stages; ++stage) {
    gl_for<0, SUB>([&](auto which) { step(stage, which, Yes{}, Full{}); });
  }
  // the last RING stages; the first of them still asks for the other parts of the last one.  The last two ask for what
  // the ends need from memory: the rows' positions in front of the wait for the last stage, which leaves nothing on
  // its way, and behind it the pages and, where there are registers for it, the first slice's bias and rows.
  constexpr int SLICE = FN > 1 && FN < 5 ? 2 : 1;      // (FN = 5 has registers for one fragment's residual rows)
  constexpr bool EARLY = FM * FN <= 4 || EPI != PS_EPI_RESIDUAL;
  const int row_base = m0 + wave_m * FM * 32, col_base = n0 + wave_n * FN * 32;
  const bool by_column = tile_by_column<TOut, EPI>(c, ldc, 1, scatter);
  TileEnds<FM, SLICE, TOut, EPI> ends;
  TilePages<FM, SLICE> pages;
  constexpr int REST = FN % SLICE;
  TilePages<FM, REST ? REST : SLICE> tail;
  const bool paged = EPI == PS_EPI_NONE && !by_column && pages.wanted(scatter, col_base + FN * 32);
  gl_for<0, RING>([&](auto index) {
    constexpr int T = decltype(index)::value;
    if constexpr (T == RING - 2) {
      if (paged) {
        pages.ask_rows(scatter, lane, row_base, m);
        if constexpr (REST) tail.ask_rows(scatter, lane, row_base, m);
      }
    }
    if constexpr (T == RING - 1) {
      if (paged) {
        pages.ask_pages(scatter);
        if constexpr (REST) tail.ask_pages(scatter);
      }
      if constexpr (EARLY) ends.ask(lane, row_base, col_base, m, n, ldc, c, bias, 0, by_column);
    }
    gl_for<0, SUB - 1>([&](auto which) { step(stage + T, which, std::integral_constant<bool, T == 0>{}, Full{}); });
    step(stage + T, Last{}, No{},
         std::integral_constant<int, T == RING - 1 ? -1 : (RING - 2 - T > 0 ? RING - 2 - T : 0)>{});
  });

  // ---- epilogue: no load of a stage and no read is on its way, and every wave is past its last operand
  static_assert(WAVES * 32 * (SLICE * 32 + 8) * 4 <= RING * STAGE_BYTES, "the epilogue reuses the stages");
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  if constexpr (!EARLY) ends.ask(lane, row_base, col_base, m, n, ldc, c, bias, 0, by_column);
  gl_store<FM, FN, SLICE, 0, TOut, EPI>(acc, reinterpret_cast<float*>(lds) + wave * 32 * (SLICE * 32 + 8), lane,
                                        row_base, col_base, m, n, ldc, c, bias, scatter, ends, pages, tail);
}

template <int FM, int FN, int ROW>
constexpr int gl_stage_bytes() { return 32 * (FM * GL_WAVES_M + FN * GL_WAVES_N) * ROW; }

template <int FM, int FN, int ROW, int RING, typename TOut, int EPI>
__global__ __launch_bounds__(512) void gemm_nt_bf16_large_kernel(
    const bf16_t* __restrict__ a, const bf16_t* __restrict__ w, int m, int n, int k, int lda, int panel, int ldc,
    TOut* __restrict__ c, const float* __restrict__ bias, KvScatter scatter) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds[RING * gl_stage_bytes<FM, FN, ROW>()];
  constexpr int BM = 32 * FM * GL_WAVES_M, BN = 32 * FN * GL_WAVES_N;
  gl_tile<FM, FN, ROW, RING, TOut, EPI>(lds, blockIdx.x, ((m + BM - 1) / BM) * ((n + BN - 1) / BN), a, w, m, n, k, lda, panel,
                                        ldc, c, bias, scatter);
}

// --------------------------------------------------------------------------------- host
#define PS_LARGE_ARGUMENTS                                                                                          \
  const void *a, const void *w, const float *bias, void *c, int m, int n, int k, int lda, int ldc, int c_dtype,     \
      int epilogue, const KvScatter &scatter, int shape, hipStream_t s
int ps_gemm_nt_bf16_large_lines(PS_LARGE_ARGUMENTS);
int ps_gemm_nt_bf16_large_half_lines(PS_LARGE_ARGUMENTS);

// `most_rows`: rows of tiles to a panel.
template <int FM, int FN, int ROW, int RING, typename TOut>
static int launch_large(const void* a, const void* w, const float* bias, void* c, int m, int n, int k, int lda,
                        int ldc, int epilogue, int most_rows, const KvScatter& scatter, hipStream_t s) {
  constexpr int BM = 32 * FM * GL_WAVES_M, BN = 32 * FN * GL_WAVES_N;
  PS_REQUIRE(k % (ROW / 2) == 0 && k / (ROW / 2) >= RING, "ps_linear: k of %d is not whole stages of these tiles", k);
  const int tiles_m = (m + BM - 1) / BM, tiles_n = (n + BN - 1) / BN;
  const int panel = tiles_m < most_rows ? tiles_m : most_rows;
  PS_REQUIRE((int64_t)tiles_m * tiles_n < ((int64_t)1 << 31), "ps_linear: too many tiles");
  dim3 grid(tiles_m * tiles_n);
#define PS_LAUNCH_GL(EPI)                                                                                       \
  hipLaunchKernelGGL((gemm_nt_bf16_large_kernel<FM, FN, ROW, RING, TOut, EPI>), grid, dim3(512), 0, s,          \
                     (const bf16_t*)a, (const bf16_t*)w, m, n, k, lda, panel, ldc, (TOut*)c, bias, scatter)
  switch (epilogue) {
    case PS_EPI_NONE: PS_LAUNCH_GL(PS_EPI_NONE); break;
    case PS_EPI_GELU_TANH: PS_LAUNCH_GL(PS_EPI_GELU_TANH); break;
    case PS_EPI_GELU_ERF: PS_LAUNCH_GL(PS_EPI_GELU_ERF); break;
    case PS_EPI_RELU2: PS_LAUNCH_GL(PS_EPI_RELU2); break;
    case PS_EPI_RESIDUAL:      // (ps_linear takes it with float outputs only)
      if constexpr (sizeof(TOut) == 4) {
        PS_LAUNCH_GL(PS_EPI_RESIDUAL);
        break;
      }
      [[fallthrough]];
    default: ps_set_error("ps_linear: unknown epilogue %d", epilogue); return 1;
  }
#undef PS_LAUNCH_GL
  PS_CHECK_LAUNCH("ps_linear(large, bfloat16)");
  return 0;
}

#define PS_LARGE(FM, FN, ROW, RING, PANEL)                                                                          \
  (c_dtype == PS_F32                                                                                                \
       ? launch_large<FM, FN, ROW, RING, float>(a, w, bias, c, m, n, k, lda, ldc, epilogue, PANEL, scatter, s)      \
       : launch_large<FM, FN, ROW, RING, bf16_t>(a, w, bias, c, m, n, k, lda, ldc, epilogue, PANEL, scatter, s))
