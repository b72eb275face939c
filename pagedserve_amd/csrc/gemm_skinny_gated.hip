// The first product of a gated feed-forward for few rows (decode steps) with the gate in its epilogue, bfloat16:
//   C[m, c] = act(A W_gate^T)[m, c] * (A W_up^T)[m, c],   W the rows [gate | up] in their packed copy (pagedserve_hip.h).
//
// As two launches the product leaves 2 x inner floats per row and the gate reads them again, 2.9 us for a handful of
// rows whose every step waits for the one before.  A block owns 16 columns of both halves: the layout is that of the
// skinny product (gemm_mfma.hip) with two tiles of columns, the second one `inner` rows of W further, the four waves
// take k in turn and every load of a round is asked for before the first product.  Sums in the same order as in that
// kernel, so the result has the same bits as the two launches.
//
// Bound by the trip of the weights from memory.  In us, two launches and this one, with weights from memory: 8 x (2 x
// 3072) x 768 6.7 and 4.4 (4.2 since row scale and arguments are read beside the weights), 64 rows 10.7 and 6.9,
// 8 x (2 x 6400) x 1600 14.0 and 12.1, 8 x (2 x 512) x 256 4.4 and 2.8.
#include <type_traits>

#include "gemm_skinny.h"

template <int ACT, int UNROLL>
__global__ __launch_bounds__(64 * SK_WAVES) void gemm_nt_skinny_gated_kernel(
    const bf16_t* __restrict__ a, const bf16_t* __restrict__ wp, bf16_t* __restrict__ c, int m, int inner, int k,
    int lda, int64_t ldc, const float* __restrict__ row_scale, float limit, float slope, float shift) {
  __shared__ float partial[2][SK_WAVES][4][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // the same in every lane: scalar
  const int n0 = blockIdx.x * 16;
  const int row0 = blockIdx.y * 16;
  const int64_t tile_values = (int64_t)k * 16;       // of the packed copy: 16 columns, all of k
  const bf16_t* w_tile[2] = {wp + (n0 / 16) * tile_values, wp + ((inner + n0) / 16) * tile_values};
  const int row = row0 + (lane & 15) < m ? row0 + (lane & 15) : m - 1;
  const bf16_t* a_ptr = a + (int64_t)row * lda + (lane >> 4) * 16;
  f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
  const uint4 zero = {0u, 0u, 0u, 0u};
  uint4 wf[UNROLL][2][2], xf[UNROLL][2];
  // the steps k0, k0 + 4 x 64, ... of a wave
  auto load = [&](int k0, auto whole) {
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      // a step behind the end is fetched from the first one and zeroed: loads under a branch would not be issued
      // together
      const bool there = decltype(whole)::value || k0 + u * SK_WAVES * 64 < k;
      const int step = there ? k0 + u * SK_WAVES * 64 : 0;
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          wf[u][j][h] = *reinterpret_cast<const uint4*>(w_tile[j] + (int64_t)step * 16 + h * 512 + lane * 8);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        xf[u][h] = *reinterpret_cast<const uint4*>(a_ptr + step + h * 8);
        if (!there) xf[u][h] = wf[u][0][h] = wf[u][1][h] = zero;
      }
    }
  };
  auto load_steps = [&](int k0) {
    if (k0 + (UNROLL - 1) * SK_WAVES * 64 < k) load(k0, std::true_type{});
    else load(k0, std::false_type{});
  };
  // wave `wave` takes the steps of 64 values of k wave, wave + 4, ...
  int k0 = wave * 64;
  if (k0 < k) load_steps(k0);
  read_arguments(row_scale, limit, slope, shift);
  const int col_in = threadIdx.x & 15, row_in = threadIdx.x >> 4;
  const int out_row = row0 + row_in;
  float scale = 1.f;
  if (row_scale != nullptr) scale = row_scale[out_row < m ? out_row : m - 1];
  while (k0 < k) {
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(&wf[u][j][h]),
                                                           *reinterpret_cast<const bf16x8*>(&xf[u][h]), acc[j], 0, 0, 0);
    k0 += SK_WAVES * UNROLL * 64;
    if (k0 < k) load_steps(k0);
  }
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) partial[j][wave][i][lane] = acc[j][i];
  __syncthreads();
  // element i of lane l is column (l / 16) * 4 + i of row l % 16; thread t finishes column t % 16 of row t / 16
  const int from = (col_in >> 2) * 16 + row_in, i = col_in & 3;
  if (out_row >= m) return;
  float v[2];
#pragma unroll
  for (int j = 0; j < 2; ++j)
    v[j] = partial[j][0][i][from] + partial[j][1][i][from] + partial[j][2][i][from] + partial[j][3][i][from];
  float value = ACT == 1 ? gelu_tanh_f(v[0]) * v[1]
                         : (ACT == 2 ? fmaxf(v[0], 0.f) * v[1] : gated_unit(v[0], v[1], GateForm{limit, slope, shift}));
  if (row_scale != nullptr) value *= scale;
  c[out_row * ldc + n0 + col_in] = from_float<bf16_t>(value);
}

extern "C" int ps_linear_gated(const void* a, const void* w_packed, void* c, int m, int inner, int k, int lda, int64_t ldc,
                               int activation, float limit, float slope, float shift, const float* row_scale,
                               void* stream) {
  PS_REQUIRE(a && w_packed && c && m > 0 && inner > 0 && inner % 16 == 0 && k > 0 && k % 64 == 0 && lda >= k &&
                 lda % 8 == 0 && ldc >= inner && m <= 64,
             "ps_linear_gated: bad sizes (m %d, inner %d, k %d, lda %d, ldc %lld)", m, inner, k, lda, (long long)ldc);
  PS_REQUIRE((reinterpret_cast<uintptr_t>(a) & 15u) == 0 && (reinterpret_cast<uintptr_t>(w_packed) & 15u) == 0,
             "ps_linear_gated: unaligned operand");
  PS_REQUIRE(activation >= 0 && activation <= 2, "ps_linear_gated: activation %d (0: silu, 1: gelu_tanh, 2: relu)",
             activation);
  PS_REQUIRE(limit > 0.f, "ps_linear_gated: the limit must be positive");
  const dim3 grid(inner / 16, (m + 15) / 16);
#define PS_LAUNCH_GS(ACT, UNROLL)                                                                                 \
  hipLaunchKernelGGL((gemm_nt_skinny_gated_kernel<ACT, UNROLL>), grid, dim3(64 * SK_WAVES), 0, (hipStream_t)stream, \
                     (const bf16_t*)a, (const bf16_t*)w_packed, (bf16_t*)c, m, inner, k, lda, ldc, row_scale, limit, \
                     slope, shift)
  // (three steps per wave cover a k of 768; a step that is not there would still be fetched)
#define PS_LAUNCH_GS_ACT(ACT)                       \
  do {                                              \
    if (k <= SK_WAVES * 3 * 64) PS_LAUNCH_GS(ACT, 3); \
    else PS_LAUNCH_GS(ACT, SK_UNROLL);              \
  } while (0)
  if (activation == 1) PS_LAUNCH_GS_ACT(1);
  else if (activation == 2) PS_LAUNCH_GS_ACT(2);
  else PS_LAUNCH_GS_ACT(0);
#undef PS_LAUNCH_GS_ACT
#undef PS_LAUNCH_GS
  PS_CHECK_LAUNCH("ps_linear_gated");
  return 0;
}
