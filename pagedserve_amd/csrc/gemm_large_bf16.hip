// bfloat16 matrix product of thousands of rows in tiles of 256 x 128 to 256 x 320:
//   C[m, n] = epi(sum_k A[m, k] W[n, k] + b[n]),   k a multiple of 32.
//
// Eight waves, four along m and two along n, one block per compute unit; a wave owns 64 rows x 32 FN columns,
// FN being 2 to 5.  Both operands go from global memory straight into LDS in stages of 32 values of k,
// four to six of them in a ring.  What such a block can do is bounded by LDS: loads fill it at 64 bytes per
// cycle and reads take 128, one after the other (a lone block of 64 x 64 takes 500 cycles for a k tile of 64,
// 250 of each, however many stages or operands are fetched ahead).  A block of BM x BN therefore needs
// 2 (BM + BN) + 2 BM + 4 BN cycles per 64 values of k where its products take BM BN / 32: the tiles are as
// large as registers and LDS allow.
//
// A load instruction blocks its wave until the address unit takes it.  Eight in a row kept the matrix cores idle at
// the head of every stage (8,192 cubed: 1.21 PFLOP/s with the loads in a row, 1.98 with none, which is the
// clock's limit), so each step issues its share of loads and its reads of the next step's operands between its
// products.  A step is 16 values of k, two steps to a stage.  Step 1 of stage s meets the other waves in front of
// its products: stage s has then been read by all of them, and stage s + 1 has landed.  It asks for the first half
// of stage s + RING, step 0 of stage s + 1 for the second half.
//
// A stage holds 64 bytes of every row; piece c (16 bytes) of row r lies in slot c ^ ((r >> 2) & 3), so that the 16
// lanes that read one piece of 16 consecutive rows touch every bank once.
//
// Measured with weights from memory, in us, against the kernels that these products went to before (64 x 256 with
// the weights past LDS, and the ring of 128 x 128): 4096 x 4800 x 1600 75 / 88, 4096 x 6400 x 1600 107 / 118,
// 8192 x 2304 x 768 45 / 51, 8192 x 3072 x 768 58 / 67, 4096 x 4096 x 1024 44 / 55, 2048 x 6400 x 1600 57 / 73.  In a
// prefill that lasts 0.2 s the card's power sets the clock and 4096 x 6400 x 1600 is level (104 / 102).  What is
// left beside the products is the ends of the tiles, 10 us a round, in which a unit that holds one block
// multiplies nothing.
#include <type_traits>

#include "gemm_tile.h"

#define GL_ROW 64          // bytes of a row and stage
#define GL_WAVES_M 4
#define GL_WAVES_N 2
#define GL_BM 256
#define GL_FM 2            // 32-row fragments of a wave

template <int I, int N, typename F>
__device__ __forceinline__ void gl_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    gl_for<I + 1, N>(f);
  }
}

// By assembly, as in gemm_tiled.hip: the compiler would wait for every load in flight before an LDS read.  The step
// that uses the operands waits first, and touches each of them behind the wait.
template <int OFFSET>
__device__ __forceinline__ void gl_read(u32x4_t& to, uint32_t address) {
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(to) : "v"(address), "n"(OFFSET) : "memory");
}

template <int PENDING>
__device__ __forceinline__ void gl_wait_and_sync() {
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(PENDING) : "memory");
}

// The columns of a wave in slices of SLICE fragments: the region of LDS that a slice is turned through is smaller.
template <int FN, int SLICE, int FIRST, typename TOut, int EPI>
__device__ __forceinline__ void gl_store(f32x16 (&acc)[GL_FM][FN], float* region, int lane, int row, int col,
                                         int m, int n, int ldc, TOut* c, const float* bias,
                                         const KvScatter& scatter) {
  if constexpr (FIRST < FN) {
    constexpr int COUNT = FIRST + SLICE <= FN ? SLICE : FN - FIRST;
    f32x16 slice[GL_FM][COUNT];
#pragma unroll
    for (int i = 0; i < GL_FM; ++i)
#pragma unroll
      for (int j = 0; j < COUNT; ++j) slice[i][j] = acc[i][FIRST + j];
    store_wave_tile<GL_FM, COUNT, TOut, EPI>(slice, region, lane, row, col + FIRST * 32, m, n, ldc, c, bias, 0, 1,
                                             scatter);
    gl_store<FN, SLICE, FIRST + COUNT, TOut, EPI>(acc, region, lane, row, col, m, n, ldc, c, bias, scatter);
  }
}

template <int FN, int RING, typename TOut, int EPI>
__global__ __launch_bounds__(512) void gemm_nt_bf16_large_kernel(
    const bf16_t* __restrict__ a, const bf16_t* __restrict__ w, const float* __restrict__ bias,
    TOut* __restrict__ c, int m, int n, int k, int lda, int ldc, int tiles_m, int tiles_n, int panel,
    KvScatter scatter) {
  constexpr int WAVES = GL_WAVES_M * GL_WAVES_N;
  constexpr int BN = 32 * FN * GL_WAVES_N;
  constexpr int STAGE_BYTES = (GL_BM + BN) * GL_ROW;
  constexpr int GROUPS = (GL_BM + BN) / 16;              // a load instruction fills 16 rows of a stage
  constexpr int LOADS = (GROUPS + WAVES - 1) / WAVES;
  constexpr int FIRST_HALF = (LOADS + 1) / 2;
  constexpr int READS = GL_FM + FN, PRODUCTS = GL_FM * FN;
  static_assert((RING - 1) * LOADS + FIRST_HALF < 64, "the load counter has six bits");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[RING * STAGE_BYTES];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // the same in every lane: scalar
  const int wave_m = wave % GL_WAVES_M, wave_n = wave / GL_WAVES_M;
  // every XCD works on a contiguous run of tiles (see gemm_tiled.hip): panels of `panel` rows of tiles, walked
  // column by column, so that what runs at one time on an XCD is about as many rows as columns
  const int per_xcd = gridDim.x / 8;
  int tile = blockIdx.x;
  if (blockIdx.x < per_xcd * 8) tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  const int first_row = tile / (panel * tiles_n) * panel;
  const int within = tile - first_row * tiles_n;
  const int panel_rows = min(panel, tiles_m - first_row);
  const int m0 = (first_row + within % panel_rows) * GL_BM;
  const int n0 = within / panel_rows * BN;
  const int stages = k / 32;

  // ---- loads: lane l of an instruction fills slot l % 4 of row l / 4 of its 16 rows.  Rows beyond m or n are
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
    const int row = group * 16 + (lane >> 2);
    const int piece = (lane & 3) ^ ((row >> 2) & 3);
    of_a[j] = group * 16 < GL_BM;
    offset[j] = of_a[j] ? (uint32_t)min(row, m - 1 - m0) * (uint32_t)lda * 2u + piece * 16
                        : (uint32_t)min(row - GL_BM, n - 1 - n0) * (uint32_t)k * 2u + piece * 16;
    target[j] = group * 16 * GL_ROW;
  }
  auto load = [&](int stage, int j) {
    const char* base = (of_a[j] ? base_a : base_w) + (int64_t)stage * GL_ROW;
    __builtin_amdgcn_global_load_lds((global_ptr_t)(base + offset[j]),
                                     (lds_ptr_t)(lds + (stage % RING) * STAGE_BYTES + target[j]), 16, 0, 0);
  };

  f32x16 acc[GL_FM][FN];
#pragma unroll
  for (int i = 0; i < GL_FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // ---- operands: lane l reads the 16 bytes of k piece 2 s + l / 32 of row l % 32
  const int key = (lane >> 2) & 3;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_ptr_t)lds;
  const uint32_t a_row = lds_base + (wave_m * GL_FM * 32 + (lane & 31)) * GL_ROW;
  const uint32_t w_row = lds_base + (GL_BM + wave_n * FN * 32 + (lane & 31)) * GL_ROW;
  const uint32_t slot[2] = {(uint32_t)(((lane >> 5) ^ key) << 4), (uint32_t)(((2 + (lane >> 5)) ^ key) << 4)};
  u32x4_t operands[2][READS];
  auto read = [&](uint32_t stage_offset, auto step, auto index, u32x4_t* to) {
    constexpr int R = decltype(index)::value;
    const uint32_t at = stage_offset + slot[decltype(step)::value] + (R < GL_FM ? a_row : w_row);
    gl_read<(R < GL_FM ? R : R - GL_FM) * 32 * GL_ROW>(to[R], at);
  };
  // Step S of a stage: the products of operands[S], the reads of the next step's operands and half of a stage's
  // loads between them.  LOAD: the stage that is asked for exists; AHEAD: how many stages behind the next one may
  // be on their way when that one has to be there, -1: there is no next step.
  auto step = [&](int stage, auto which, auto loads, auto ahead) {
    constexpr int S = decltype(which)::value, AHEAD = decltype(ahead)::value;
    constexpr bool LOAD = decltype(loads)::value, NEXT = AHEAD >= 0;
    constexpr int FROM = S == 1 ? 0 : FIRST_HALF, COUNT = S == 1 ? FIRST_HALF : LOADS - FIRST_HALF;
    const uint32_t next_stage = (uint32_t)(((S == 1 ? stage + 1 : stage) % RING) * STAGE_BYTES);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if constexpr (S == 1 && NEXT) gl_wait_and_sync<(AHEAD > 0 ? AHEAD : 0) * LOADS>();
#pragma unroll
    for (int r = 0; r < READS; ++r) asm volatile("" : "+v"(operands[S][r]));   // used only behind the wait
    gl_for<0, PRODUCTS>([&](auto product) {
      constexpr int Q = decltype(product)::value;
      constexpr int I = Q / FN, J = Q % FN;
      acc[I][J] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, operands[S][I]),
                                                          __builtin_bit_cast(bf16x8, operands[S][GL_FM + J]),
                                                          acc[I][J], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (NEXT)
        gl_for<Q * READS / PRODUCTS, (Q + 1) * READS / PRODUCTS>([&](auto index) {
          read(next_stage, std::integral_constant<int, S ^ 1>{}, index, operands[S ^ 1]);
        });
      if constexpr (LOAD)
        gl_for<0, COUNT>([&](auto index) {
          constexpr int L = decltype(index)::value;
          if constexpr (Q == (2 * L + 1) * PRODUCTS / (2 * COUNT))
            load(S == 1 ? stage + RING : stage + RING - 1, FROM + L);
        });
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  using Zero = std::integral_constant<int, 0>;
  using One = std::integral_constant<int, 1>;
  using Yes = std::true_type;
  using No = std::false_type;

  // stages 0 .. RING - 2, and the first half of stage RING - 1 (the host sends no product of fewer than RING stages)
#pragma unroll
  for (int d = 0; d < RING - 1; ++d)
#pragma unroll
    for (int j = 0; j < LOADS; ++j) load(d, j);
#pragma unroll
  for (int j = 0; j < FIRST_HALF; ++j) load(RING - 1, j);
  gl_wait_and_sync<(RING - 2) * LOADS + FIRST_HALF>();
  gl_for<0, READS>([&](auto index) { read(0, Zero{}, index, operands[0]); });
  using Full = std::integral_constant<int, RING - 2>;
  int stage = 0;
  for (; stage + RING < stages; ++stage) {
    step(stage, Zero{}, Yes{}, Full{});
    step(stage, One{}, Yes{}, Full{});
  }
  // the last RING stages; the first of them still asks for the second half of the last one
  gl_for<0, RING>([&](auto index) {
    constexpr int T = decltype(index)::value;
    step(stage + T, Zero{}, std::integral_constant<bool, T == 0>{}, Full{});
    step(stage + T, One{}, No{},
         std::integral_constant<int, T == RING - 1 ? -1 : (RING - 2 - T > 0 ? RING - 2 - T : 0)>{});
  });

  // ---- epilogue: no load or read is on its way, and every wave is past its last operand
  constexpr int SLICE = FN < 5 ? 2 : 1;      // (FN = 5 has registers for one fragment's residual rows)
  static_assert(WAVES * 32 * (SLICE * 32 + 8) * 4 <= RING * STAGE_BYTES, "the epilogue reuses the stages");
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  gl_store<FN, SLICE, 0, TOut, EPI>(acc, reinterpret_cast<float*>(lds) + wave * 32 * (SLICE * 32 + 8), lane,
                                    m0 + wave_m * GL_FM * 32, n0 + wave_n * FN * 32, m, n, ldc, c, bias, scatter);
}

// --------------------------------------------------------------------------------- host
// Which width (FN) a product takes, 0: not this kernel.  A block has its compute unit to itself, so that time goes
// in rounds: `share` is the part of the rounds' outputs that the product needs.  At a full chip a tile's outputs per
// time stand as 0.70, 0.87, 0.95 and 1 for FN of 2 to 5 (256 x 128 44 us for 1600 values of k where 256 x 320
// takes 78).  Against the other kernels the line lies at 0.6 of a full chip of the widest tiles: 2048 x 4800 x 1600
// (0.68) 44 us where they take 50, 4096 x 3072 x 768 (0.87) 31 and 39; 4096 x 1600 x 1600 (0.55) 38 and 36,
// 8192 x 768 x 3072 (0.52) 57 and 58, 4096 x 1024 x 4096 (0.35) 57 and 50.  Short products are left to them: with k
// under 768 the ends of a tile take longer than its products.
static int large_width(int m, int n, int k) {
  static const float rate[] = {0.f, 0.f, 0.70f, 0.87f, 0.95f, 1.f};
  if (m < 1024 || n < 256 || k < 768) return 0;
  const int units = ps_compute_units();
  const int64_t tiles_m = (m + GL_BM - 1) / GL_BM;
  int best = 0;
  float best_value = 0.6f;
  for (int width = 2; width <= 5; ++width) {
    const int bn = 32 * width * GL_WAVES_N;
    const int64_t tiles = tiles_m * ((n + bn - 1) / bn);
    const int64_t rounds = (tiles + units - 1) / units;
    const float share = (float)m * (float)n / ((float)(rounds * units) * GL_BM * bn);
    if (share * rate[width] > best_value) {
      best_value = share * rate[width];
      best = width;
    }
  }
  return best;
}

// (k a multiple of 32 for whole stages; a tile's rows lie within 32-bit offsets)
static bool large_takes(const void* a, const void* w, int m, int n, int k, int lda) {
  return m > 0 && n > 0 && k >= 8 * 32 && k % 32 == 0 && lda >= k && lda % 8 == 0 && lda <= (1 << 22) &&
         (reinterpret_cast<uintptr_t>(a) & 15u) == 0 && (reinterpret_cast<uintptr_t>(w) & 15u) == 0;
}

bool ps_gemm_nt_bf16_large_supported(const void* a, const void* w, int m, int n, int k, int lda) {
  return large_takes(a, w, m, n, k, lda) && large_width(m, n, k) != 0;
}

template <int FN, int RING, typename TOut>
static int launch_large(const void* a, const void* w, const float* bias, void* c, int m, int n, int k, int lda,
                        int ldc, int epilogue, const KvScatter& scatter, hipStream_t s) {
  constexpr int BN = 32 * FN * GL_WAVES_N;
  const int tiles_m = (m + GL_BM - 1) / GL_BM, tiles_n = (n + BN - 1) / BN;
  const int panel = tiles_m < 8 ? tiles_m : 8;
  PS_REQUIRE((int64_t)tiles_m * tiles_n < ((int64_t)1 << 31), "ps_linear: too many tiles");
  dim3 grid(tiles_m * tiles_n);
#define PS_LAUNCH_GL(EPI)                                                                                      \
  hipLaunchKernelGGL((gemm_nt_bf16_large_kernel<FN, RING, TOut, EPI>), grid, dim3(512), 0, s, (const bf16_t*)a, \
                     (const bf16_t*)w, bias, (TOut*)c, m, n, k, lda, ldc, tiles_m, tiles_n, panel, scatter)
  switch (epilogue) {
    case PS_EPI_NONE: PS_LAUNCH_GL(PS_EPI_NONE); break;
    case PS_EPI_GELU_TANH: PS_LAUNCH_GL(PS_EPI_GELU_TANH); break;
    case PS_EPI_GELU_ERF: PS_LAUNCH_GL(PS_EPI_GELU_ERF); break;
    case PS_EPI_RELU2: PS_LAUNCH_GL(PS_EPI_RELU2); break;
    case PS_EPI_RESIDUAL: PS_LAUNCH_GL(PS_EPI_RESIDUAL); break;
    default: ps_set_error("ps_linear: unknown epilogue %d", epilogue); return 1;
  }
#undef PS_LAUNCH_GL
  PS_CHECK_LAUNCH("ps_linear(large, bfloat16)");
  return 0;
}

// width: FN, 0: by the rule.  Stages as many as LDS holds (160 KB).
int ps_gemm_nt_bf16_large(const void* a, const void* w, const float* bias, void* c, int m, int n, int k, int lda,
                          int ldc, int c_dtype, int epilogue, const KvScatter& scatter, int width, hipStream_t s) {
  if (width == 0) width = large_width(m, n, k);
#define PS_LARGE(FN, RING)                                                                                      \
  (c_dtype == PS_F32 ? launch_large<FN, RING, float>(a, w, bias, c, m, n, k, lda, ldc, epilogue, scatter, s)    \
                     : launch_large<FN, RING, bf16_t>(a, w, bias, c, m, n, k, lda, ldc, epilogue, scatter, s))
  if (width == 2) return PS_LARGE(2, 6);
  if (width == 3) return PS_LARGE(3, 5);
  if (width == 4) return PS_LARGE(4, 4);
  if (width == 5) return PS_LARGE(5, 4);
#undef PS_LARGE
  ps_set_error("ps_linear: the large product has tiles of 2 to 5 fragments, not %d", width);
  return 1;
}

// The large product on its own, for tests and measurements of its tile shapes.
extern "C" int ps_gemm_nt_large(const void* a, const void* w, const float* bias, void* c, int m, int n, int k,
                                int lda, int ldc, int c_dtype, int epilogue, int width, void* stream) {
  PS_REQUIRE(a && w && c && large_takes(a, w, m, n, k, lda) && ldc >= n,
             "ps_gemm_nt_large: bad sizes or unaligned operand (m %d, n %d, k %d, lda %d, ldc %d)", m, n, k, lda, ldc);
  PS_REQUIRE(c_dtype == PS_F32 || c_dtype == PS_BF16, "ps_gemm_nt_large: unknown output dtype");
  PS_REQUIRE(epilogue != PS_EPI_RESIDUAL || c_dtype == PS_F32,
             "ps_gemm_nt_large: the residual epilogue needs a float output");
  KvScatter none = {};
  return ps_gemm_nt_bf16_large(a, w, bias, c, m, n, k, lda, ldc, c_dtype, epilogue, none, width, (hipStream_t)stream);
}
