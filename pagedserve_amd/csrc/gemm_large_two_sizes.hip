// bfloat16 products of which whole rounds of blocks in tiles of 256 x 320 leave a rest of the columns: the rest in tiles of 128 x
// 192 by the same launch (gemm_large_bf16.h has the tiles).
//
// A unit holds one block, so that time goes in rounds.  4096 x 6400 is 400 tiles of 256 x 256 on 256 units, two rounds of which
// the second is 56 % full; 5,120 of its columns are one full round of 256 x 320, the other 1,280 224 tiles of 128 x 192,
// which begin as the units become free.  Every output keeps its bits: both kinds of tiles add up k in the same order.
//
// With weights from memory, one size of tiles and two, us: 4096 x 6400 x 1600 with GELU 100 / 91 (two launches 93), 8192 x
// 6400 x 1600 186 / 175, 2048 x 12800 x 1600 92 / 83.  In a batch of 64 prompts of 768 and 12 steps (GPT-2 XL) 105 to 93 a layer
// and budget of 4,096 tokens.
#include "gemm_large_bf16.h"

#define TS_FIRST 2, 5, 64, 4      // 256 x 320
#define TS_REST 1, 3, 128, 4      // 128 x 192
#define TS_FIRST_ROWS 256
#define TS_FIRST_COLUMNS 320
#define TS_REST_ROWS 128
#define TS_REST_COLUMNS 192
#define TS_PANEL_FIRST 8           // rows of tiles to a panel, as the kernels of one size have them
#define TS_PANEL_REST 4

template <typename TOut, int EPI>
__global__ __launch_bounds__(512) void gemm_nt_bf16_two_sizes_kernel(
    const bf16_t* __restrict__ a, const bf16_t* __restrict__ w, int m, int n, int k, int lda, int first_columns, int panels,
    int ldc, TOut* __restrict__ c, const float* __restrict__ bias) {
  constexpr int FIRST_BYTES = 4 * gl_stage_bytes<2, 5, 64>(), REST_BYTES = 4 * gl_stage_bytes<1, 3, 128>();
  __shared__ __attribute__((aligned(1024))) unsigned char lds[FIRST_BYTES > REST_BYTES ? FIRST_BYTES : REST_BYTES];
  const KvScatter none = {};
  const int first = ((m + TS_FIRST_ROWS - 1) / TS_FIRST_ROWS) * (first_columns / TS_FIRST_COLUMNS);
  if ((int)blockIdx.x < first) {
    gl_tile<TS_FIRST, TOut, EPI>(lds, blockIdx.x, first, a, w, m, first_columns, k, lda, panels & 0xff, ldc, c, bias, none);
  } else {
    const int rest = n - first_columns;
    const int blocks = ((m + TS_REST_ROWS - 1) / TS_REST_ROWS) * ((rest + TS_REST_COLUMNS - 1) / TS_REST_COLUMNS);
    gl_tile<TS_REST, TOut, EPI>(lds, blockIdx.x - first, blocks, a, w + (int64_t)first_columns * k, m, rest, k, lda, panels >> 8,
                                ldc, c + first_columns, bias != nullptr ? bias + first_columns : nullptr, none);
  }
}

// How many columns go in the first tiles, 0: not this kernel.  The rest is as 0.75 of the rate of the first tiles (4096 x 1280
// x 1600 26 us).  Of 54 products of 1,500 to 8,192 rows, 4,800 to 12,800 columns and k of 1,600 and 2,048 the six that the
// rule takes are 0.91 to 0.98 of one size; where it expects less than a twentieth, two sizes were 0.94 to 1.20 of it (6000 x 6400 x
// 1600 128 and 144).  A shorter k leaves little: in two launches 8192 x 3072 x 768 56.9 and 54.8, 6000 x 4096 x 1024 66.7 and 68.4.
int ps_gemm_nt_bf16_two_sizes_columns(int m, int n, int k, int c_dtype, int epilogue, const KvScatter& scatter) {
  if (c_dtype != PS_BF16 || epilogue == PS_EPI_RESIDUAL || scatter.k_pool != nullptr || m < 1024 || k < 1536 || k % 64 != 0) return 0;
  const int units = ps_compute_units();
  const int64_t rows_first = (m + TS_FIRST_ROWS - 1) / TS_FIRST_ROWS, rows_rest = (m + TS_REST_ROWS - 1) / TS_REST_ROWS;
  if (rows_first > units) return 0;
  // rounds as they would be in one size of tiles, in outputs at the rate of the widest (as in gemm_large_bf16.hip)
  float least = INFINITY;
  const float rate[] = {0.f, 0.f, 0.85f, 0.87f, 0.95f, 1.f};
  for (int width = 2; width <= 5; ++width) {
    const int64_t tiles = rows_first * ((n + 64 * width - 1) / (64 * width));
    least = fminf(least, (float)((tiles + units - 1) / units) * 256.f * 64.f * width / rate[width]);
  }
  int best = 0;
  for (int rounds = 1; rounds <= 4; ++rounds) {
    const int64_t columns = rounds * units / rows_first * TS_FIRST_COLUMNS;
    if (columns + 64 > n) break;
    const int64_t tiles = rows_rest * ((n - columns + TS_REST_COLUMNS - 1) / TS_REST_COLUMNS);
    const float time = rounds * 256.f * 320.f + (float)((tiles + units - 1) / units) * 128.f * 192.f / 0.75f;
    if (time < (best ? 1.f : 0.95f) * least) {
      least = time;
      best = (int)columns;
    }
  }
  return best;
}

int ps_gemm_nt_bf16_two_sizes(const void* a, const void* w, const float* bias, void* c, int m, int n, int k, int lda, int ldc,
                              int epilogue, int first_columns, hipStream_t s) {
  PS_REQUIRE(first_columns > 0 && first_columns % TS_FIRST_COLUMNS == 0 && first_columns < n && k % 64 == 0 && k >= 8 * 64,
             "ps_linear: no two sizes of tiles of %d of %d columns, k %d", first_columns, n, k);
  const int64_t rows_first = (m + TS_FIRST_ROWS - 1) / TS_FIRST_ROWS, rows_rest = (m + TS_REST_ROWS - 1) / TS_REST_ROWS;
  const int64_t blocks = rows_first * (first_columns / TS_FIRST_COLUMNS) +
                         rows_rest * ((n - first_columns + TS_REST_COLUMNS - 1) / TS_REST_COLUMNS);
  PS_REQUIRE(blocks < ((int64_t)1 << 30), "ps_linear: too many tiles");
  const int panels = (int)(rows_first < TS_PANEL_FIRST ? rows_first : TS_PANEL_FIRST) +
                     256 * (int)(rows_rest < TS_PANEL_REST ? rows_rest : TS_PANEL_REST);
#define PS_LAUNCH_TS(EPI)                                                                                            \
  case EPI:                                                                                                          \
    hipLaunchKernelGGL((gemm_nt_bf16_two_sizes_kernel<bf16_t, EPI>), dim3((unsigned)blocks), dim3(512), 0, s,        \
                       (const bf16_t*)a, (const bf16_t*)w, m, n, k, lda, first_columns, panels, ldc, (bf16_t*)c, bias); \
    break
  switch (epilogue) {
    PS_LAUNCH_TS(PS_EPI_NONE);
    PS_LAUNCH_TS(PS_EPI_GELU_TANH);
    PS_LAUNCH_TS(PS_EPI_GELU_ERF);
    PS_LAUNCH_TS(PS_EPI_RELU2);
    default: ps_set_error("ps_linear: no two sizes of tiles with epilogue %d", epilogue); return 1;
  }
#undef PS_LAUNCH_TS
  PS_CHECK_LAUNCH("ps_linear(two sizes of tiles, bfloat16)");
  return 0;
}

// The product in two sizes of tiles on its own, for tests and measurements.
bool ps_gemm_nt_bf16_large_operands(const void* a, const void* w, int m, int n, int k, int lda);
extern "C" int ps_gemm_nt_two_sizes(const void* a, const void* w, const float* bias, void* c, int m, int n, int k, int lda,
                                    int ldc, int epilogue, int first_columns, void* stream) {
  PS_REQUIRE(a && w && c && ps_gemm_nt_bf16_large_operands(a, w, m, n, k, lda) && ldc >= n,
             "ps_gemm_nt_two_sizes: bad sizes or unaligned operand (m %d, n %d, k %d, lda %d, ldc %d)", m, n, k, lda, ldc);
  return ps_gemm_nt_bf16_two_sizes(a, w, bias, c, m, n, k, lda, ldc, epilogue, first_columns, (hipStream_t)stream);
}
