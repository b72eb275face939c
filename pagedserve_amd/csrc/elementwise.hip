// Embedding(+position table) add, LayerNorm / RMS norm with row gather, and the scatter of
// new keys and values into cache pages.  All arithmetic is float; storage may be bfloat16.
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include "common.h"
#include "linear.h"
#include "pagedserve_hip.h"

// ---------------------------------------------------------------- error channel
static thread_local char g_error[512] = "";

void ps_set_error(const char* fmt, ...) {
  va_list args;
  va_start(args, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, args);
  va_end(args);
}

extern "C" const char* ps_last_error(void) { return g_error; }

extern "C" int ps_device_info(int* compute_units, int* lds_bytes, char* arch, int arch_len) {
  int device = 0;
  hipError_t status = hipGetDevice(&device);
  PS_REQUIRE(status == hipSuccess, "ps_device_info: %s", hipGetErrorString(status));
  hipDeviceProp_t prop;
  status = hipGetDeviceProperties(&prop, device);
  PS_REQUIRE(status == hipSuccess, "ps_device_info: %s", hipGetErrorString(status));
  if (compute_units) *compute_units = prop.multiProcessorCount;
  if (lds_bytes) *lds_bytes = (int)prop.sharedMemPerBlock;
  if (arch && arch_len > 0) {
    strncpy(arch, prop.gcnArchName, arch_len - 1);
    arch[arch_len - 1] = 0;
  }
  return 0;
}

// Compute units of the current device, asked once per device: launch shapes follow it.
int ps_compute_units() {
  static int cached[64];
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) return 256;
  if (cached[device] == 0) {
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess || prop.multiProcessorCount <= 0) return 256;
    cached[device] = prop.multiProcessorCount;
  }
  return cached[device];
}

// ---------------------------------------------------------------- embedding
// h0[t] = scale * wte[id[t]] + wpe[pos[t]]  (reference: src/model/paged_decoder.py:306-314,
// where the scale is 1); with norm_gamma, the row is then RMS-normed in float in the same
// launch: h0 <- h0 / sqrt(mean(h0^2) + eps) * norm_gamma.  `copy`: the rows are written there too.
// The id of token t is ids[t], or carried[src[t]] where src[t] >= 0: a token that an earlier
// step chose on the device and that the host has not seen yet.
// (The chain: ids, sources and positions at once -> a carried token -> rows of both tables.  The arguments in front of
// `out` come with the launch.)  AT_ONCE: columns of a thread whose loads leave together, one where it has no more (2,048
// rows of 256 3.46 us with four, 3.25 with one).
template <typename T, int AT_ONCE>
__global__ void embed_kernel(const int* __restrict__ ids, const int* __restrict__ src,
                             const int* __restrict__ carried, const int* __restrict__ positions,
                             const T* __restrict__ table, const T* __restrict__ pos_table, int width, int vocab,
                             float* __restrict__ out, float* __restrict__ copy, float scale,
                             const float* __restrict__ norm_gamma, float norm_eps) {
  __shared__ __attribute__((aligned(16))) float scratch[16];
  const int t = blockIdx.x;
  int id = ids[t];
  const int from = src != nullptr ? src[t] : -1;
  const int position = pos_table != nullptr ? positions[t] : 0;
  read_arguments(out, copy, scale, norm_gamma);
  if (from >= 0) id = carried[from];
  id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);   // never a read outside the table
  const T* row = table + (int64_t)id * width;
  const T* prow = pos_table != nullptr ? pos_table + (int64_t)position * width : row;
  float* dst = out + (int64_t)t * width;
  const int threads = blockDim.x;
  float sum = 0.f;
  for (int first = threadIdx.x; first < width; first += AT_ONCE * threads) {
    T value[AT_ONCE], place[AT_ONCE];
#pragma unroll
    for (int j = 0; j < AT_ONCE; ++j) {
      const int i = first + j * threads < width ? first + j * threads : width - 1;
      value[j] = row[i];
      place[j] = prow[i];
    }
#pragma unroll
    for (int j = 0; j < AT_ONCE; ++j) {
      const int i = first + j * threads;
      float v = to_float<T>(value[j]) * scale;
      if (pos_table != nullptr) v += to_float<T>(place[j]);
      if (i >= width) continue;
      dst[i] = v;
      if (norm_gamma == nullptr && copy != nullptr) copy[(int64_t)t * width + i] = v;
      sum = fmaf(v, v, sum);
    }
  }
  if (norm_gamma == nullptr) return;
  // (each thread reads back what it wrote itself)
  const float inv = 1.0f / sqrtf(block_sum(sum, scratch) / (float)width + norm_eps);
  for (int first = threadIdx.x; first < width; first += AT_ONCE * threads)
#pragma unroll
    for (int j = 0; j < AT_ONCE; ++j) {
      const int i = first + j * threads;
      if (i >= width) continue;
      const float v = dst[i] * inv * norm_gamma[i];
      dst[i] = v;
      if (copy != nullptr) copy[(int64_t)t * width + i] = v;
    }
}

extern "C" int ps_embed(const void* table, const void* pos_table, const int* ids, const int* src,
                        const int* carried, const int* positions, float* out, float* copy, int tokens,
                        int width, int vocab, int max_positions, float scale,
                        const float* norm_gamma, float norm_eps, int dtype, void* stream) {
  PS_REQUIRE(tokens >= 0 && width > 0 && vocab > 0, "ps_embed: bad sizes (tokens %d, width %d)",
             tokens, width);
  PS_REQUIRE(dtype == PS_F32 || dtype == PS_BF16, "ps_embed: unknown dtype %d", dtype);
  PS_REQUIRE(pos_table == nullptr || max_positions > 0, "ps_embed: position table without rows");
  PS_REQUIRE(src == nullptr || carried != nullptr, "ps_embed: carried tokens are missing");
  PS_REQUIRE(norm_gamma == nullptr || norm_eps > 0.f, "ps_embed: a norm needs a positive eps");
  if (tokens == 0) return 0;
  const int threads = width >= 256 ? 256 : 64;
  hipStream_t s = (hipStream_t)stream;
#define PS_LAUNCH_EMBED(T, AT_ONCE)                                                                                       \
  hipLaunchKernelGGL((embed_kernel<T, AT_ONCE>), dim3(tokens), dim3(threads), 0, s, ids, src, carried, positions,         \
                     (const T*)table, (const T*)pos_table, width, vocab, out, copy, scale, norm_gamma, norm_eps)
  if (dtype == PS_F32) {
    if (width <= threads) PS_LAUNCH_EMBED(float, 1);
    else PS_LAUNCH_EMBED(float, 4);
  } else {
    if (width <= threads) PS_LAUNCH_EMBED(bf16_t, 1);
    else PS_LAUNCH_EMBED(bf16_t, 4);
  }
#undef PS_LAUNCH_EMBED
  PS_CHECK_LAUNCH("ps_embed");
  return 0;
}

// ---------------------------------------------------------------- norms
// mean, centred values, biased variance of the centred values, rsqrt(var + eps), scale and
// shift (reference: src/kernels/triton_residual_layernorm.py:25-39).
//
// norm_wave_kernel: one wave per row, the row held in registers (width <= 64 * VPT): one
// trip to memory, reductions by shuffles, no barrier.  norm_block_kernel: one block per row,
// the row read three times (it stays in cache), any width.
template <typename T, bool RMS, int VPT>
__global__ __launch_bounds__(256) void norm_wave_kernel(
    const float* __restrict__ x, const int* __restrict__ rows, const float* __restrict__ gamma,
    const float* __restrict__ beta, T* __restrict__ out, int n_rows, int width, float eps,
    int packed) {
  const int lane = threadIdx.x & 63;
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= n_rows) return;
  const float* src = x + (int64_t)(rows ? rows[r] : r) * width;
  // Loads are unconditional (index clamped, value selected afterwards): a load under a
  // branch would wait for the one before it, and the row would cost VPT trips to memory.
  float v[VPT], g[VPT], b[VPT];
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int col = lane + i * 64;
    const int safe = col < width ? col : width - 1;
    v[i] = src[safe];
    g[i] = gamma[safe];
    b[i] = (!RMS && beta != nullptr) ? beta[safe] : 0.f;
  }
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    if (lane + i * 64 >= width) v[i] = 0.f;
    sum += v[i];
  }
  float mean = 0.f;
  if (!RMS) mean = wave_sum(sum) / (float)width;
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int col = lane + i * 64;
    const float c = col < width ? v[i] - mean : 0.f;
    v[i] = c;
    sq += c * c;
  }
  const float inv_std = 1.0f / sqrtf(wave_sum(sq) / (float)width + eps);
  T* dst = out + (int64_t)r * width;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int col = lane + i * 64;
    if (col >= width) continue;
    const T y = from_float<T>(v[i] * inv_std * g[i] + b[i]);
    if (packed) out[packed_offset(r, col, width)] = y;
    else dst[col] = y;
  }
}

// norm_vec_kernel: the same for rows that can be read in pieces of four values (width a multiple of
// four, operands aligned): a lane reads and writes whole pieces, a quarter of the instructions.  WAVES
// waves share a row and meet through LDS: one where rows are many, four where they are few and what
// counts is the one trip to memory (then a thread holds one or two pieces).  Measured, in us, single
// values per lane before and now: 64 x 768 3.3 / 2.85, 544 x 1024 3.7 / 3.1, 2048 x 768 4.5 / 4.2, 4096 x
// 1600 11.9 / 10.6; with one barrier to a sum 64 x 768 in a decode step 3.0 -> 2.4.  Short rows, a handful of values per
// lane either way, stay with norm_wave_kernel (launch_norm says up to where).
template <typename T>
__device__ inline void store4(T* out, const float* v);
template <>
__device__ inline void store4<float>(float* out, const float* v) {
  *reinterpret_cast<float4*>(out) = make_float4(v[0], v[1], v[2], v[3]);
}
template <>
__device__ inline void store4<bf16_t>(bf16_t* out, const float* v) {
  *reinterpret_cast<uint2*>(out) = make_uint2(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]));
}

// In the packed order a line of 128 bytes holds 8 columns of 8 rows.  Blocks of those rows on different XCDs, each with
// an L2 of its own, would each write a sixteenth of it to memory: consecutive block ids run on different XCDs, so that
// every eighth block takes a row of the same 16 (64 x 768 in a decode step 2.6 us, in the order of the rows 3.95).
__device__ inline int norm_packed_row(int block) {
  const int xcd = block & 7, slot = block >> 3;
  return ((slot >> 4) * 8 + xcd) * 16 + (slot & 15);
}
static int norm_packed_blocks(int rows) { return (rows + 127) / 128 * 128; }

template <typename T, bool RMS, int PIECES, int WAVES>
__global__ __launch_bounds__(256) void norm_vec_kernel(
    const float* __restrict__ x, const int* __restrict__ rows, const float* __restrict__ gamma,
    const float* __restrict__ beta, T* __restrict__ out, int n_rows, int width, float eps,
    int packed) {
  __shared__ __attribute__((aligned(16))) float scratch[2][WAVES];    // a place for each of the two sums
  const int at = WAVES == 1 ? threadIdx.x & 63 : threadIdx.x;
  int r = WAVES == 1 ? blockIdx.x * 4 + (threadIdx.x >> 6) : blockIdx.x;
  if (WAVES > 1 && packed) r = norm_packed_row(blockIdx.x);
  if (r >= n_rows) return;
  const float* src = x + (int64_t)(rows ? rows[r] : r) * width;
  // loads are unconditional, as above; without a shift gamma stands in for it
  const float* shift = (!RMS && beta != nullptr) ? beta : gamma;
  float v[PIECES][4], g[PIECES][4], b[PIECES][4];
#pragma unroll
  for (int i = 0; i < PIECES; ++i) {
    const int col = (at + i * 64 * WAVES) * 4;
    const int safe = col < width ? col : width - 4;
    *reinterpret_cast<float4*>(v[i]) = *reinterpret_cast<const float4*>(src + safe);
    *reinterpret_cast<float4*>(g[i]) = *reinterpret_cast<const float4*>(gamma + safe);
    *reinterpret_cast<float4*>(b[i]) = *reinterpret_cast<const float4*>(shift + safe);
  }
  float mean = 0.f;
  if (!RMS) {
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < PIECES; ++i)
      if ((at + i * 64 * WAVES) * 4 < width) sum += (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);
    mean = (WAVES == 1 ? wave_sum(sum) : block_total(sum, scratch[0], WAVES)) / (float)width;
  }
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < PIECES; ++i) {
    const bool there = (at + i * 64 * WAVES) * 4 < width;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[i][j] = there ? v[i][j] - mean : 0.f;
      sq = fmaf(v[i][j], v[i][j], sq);
    }
  }
  const float total = WAVES == 1 ? wave_sum(sq) : block_total(sq, scratch[1], WAVES);
  const float inv_std = 1.0f / sqrtf(total / (float)width + eps);
#pragma unroll
  for (int i = 0; i < PIECES; ++i) {
    const int col = (at + i * 64 * WAVES) * 4;
    if (col >= width) continue;
    float y[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      y[j] = v[i][j] * inv_std * g[i][j];
      if (!RMS && beta != nullptr) y[j] += b[i][j];
    }
    // (four columns from a multiple of four lie side by side in the packed order too)
    store4<T>(out + (packed ? packed_offset(r, col, width) : (int64_t)r * width + col), y);
  }
}

// norm_row_kernel: one block of four waves per row, the row held in registers (width <= 256 *
// VPT), the two sums met through LDS.  For few wide rows that cannot be read in pieces of four: a
// wave alone would hold 25 values per lane at 1,601 columns and ask for them one after the
// other, four waves ask for 7 each (16 x 1601 3.6 us, a wave to a row 4.8).
template <typename T, bool RMS, int VPT>
__global__ __launch_bounds__(256) void norm_row_kernel(
    const float* __restrict__ x, const int* __restrict__ rows, const float* __restrict__ gamma,
    const float* __restrict__ beta, T* __restrict__ out, int width, float eps, int packed) {
  __shared__ __attribute__((aligned(16))) float scratch[16];
  const int r = blockIdx.x;
  const float* src = x + (int64_t)(rows ? rows[r] : r) * width;
  float v[VPT], g[VPT], b[VPT];
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int col = threadIdx.x + i * 256;
    const int safe = col < width ? col : width - 1;
    v[i] = src[safe];
    g[i] = gamma[safe];
    b[i] = (!RMS && beta != nullptr) ? beta[safe] : 0.f;
  }
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    if ((int)threadIdx.x + i * 256 >= width) v[i] = 0.f;
    sum += v[i];
  }
  float mean = 0.f;
  if (!RMS) mean = block_sum(sum, scratch) / (float)width;
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int col = threadIdx.x + i * 256;
    const float c = col < width ? v[i] - mean : 0.f;
    v[i] = c;
    sq += c * c;
  }
  const float inv_std = 1.0f / sqrtf(block_sum(sq, scratch) / (float)width + eps);
  T* dst = out + (int64_t)r * width;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int col = threadIdx.x + i * 256;
    if (col >= width) continue;
    const T y = from_float<T>(v[i] * inv_std * g[i] + b[i]);
    if (packed) out[packed_offset(r, col, width)] = y;
    else dst[col] = y;
  }
}

template <typename T, bool RMS>
__global__ void norm_block_kernel(const float* __restrict__ x, const int* __restrict__ rows,
                                  const float* __restrict__ gamma, const float* __restrict__ beta,
                                  T* __restrict__ out, int width, float eps) {
  __shared__ __attribute__((aligned(16))) float scratch[16];
  const int r = blockIdx.x;
  const float* src = x + (int64_t)(rows ? rows[r] : r) * width;
  T* dst = out + (int64_t)r * width;
  float mean = 0.f;
  if (!RMS) {
    float partial = 0.f;
    for (int i = threadIdx.x; i < width; i += blockDim.x) partial += src[i];
    mean = block_sum(partial, scratch) / (float)width;
  }
  float partial = 0.f;
  for (int i = threadIdx.x; i < width; i += blockDim.x) {
    const float c = src[i] - mean;
    partial += c * c;
  }
  const float variance = block_sum(partial, scratch) / (float)width;
  const float inv_std = 1.0f / sqrtf(variance + eps);
  for (int i = threadIdx.x; i < width; i += blockDim.x) {
    float v = (src[i] - mean) * inv_std * gamma[i];
    if (!RMS && beta != nullptr) v += beta[i];
    dst[i] = from_float<T>(v);
  }
}

#define NORM_FEW_ROWS 256    // up to here a block of four waves per row, from the width on where that
#define NORM_FEW_WIDTH 512   // is no slower than a wave that reads single values (64 x 320 3.2 against 3.0 us,
                             // 64 x 512 3.15 against 3.25, 64 x 768 3.2 against 3.6)
#define NORM_MANY_WIDTH 320  // the same for more rows, a wave to a row (300 x 260 3.15 against 3.05, 300 x 320 3.05
                             // against 3.1, 300 x 768 3.2 against 3.6)

template <typename T, bool RMS>
static void launch_norm(const float* x, const int* rows, const float* gamma, const float* beta,
                        void* out, int n_rows, int width, float eps, int packed, hipStream_t s) {
  const int per_lane = (width + 63) / 64;
  const dim3 grid((n_rows + 3) / 4);
  const uintptr_t all = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(gamma) |
                        reinterpret_cast<uintptr_t>(beta) | reinterpret_cast<uintptr_t>(out);
  if (width % 4 == 0 && width >= (n_rows <= NORM_FEW_ROWS ? NORM_FEW_WIDTH : NORM_MANY_WIDTH) && width <= 2048 &&
      (all & 15u) == 0) {
#define PS_LAUNCH_NV(PIECES, WAVES)                                                               \
  hipLaunchKernelGGL((norm_vec_kernel<T, RMS, PIECES, WAVES>),                                    \
                     WAVES == 1 ? grid : dim3(packed ? norm_packed_blocks(n_rows) : n_rows),      \
                     dim3(256), 0, s, x, rows, gamma, beta, (T*)out, n_rows, width, eps, packed)
    if (n_rows <= NORM_FEW_ROWS) {
      if (width <= 1024) PS_LAUNCH_NV(1, 4);
      else PS_LAUNCH_NV(2, 4);
    } else if (width <= 512) PS_LAUNCH_NV(2, 1);
    else if (width <= 768) PS_LAUNCH_NV(3, 1);
    else if (width <= 1024) PS_LAUNCH_NV(4, 1);
    else if (width <= 1536) PS_LAUNCH_NV(6, 1);
    else PS_LAUNCH_NV(8, 1);
#undef PS_LAUNCH_NV
    return;
  }
  if (n_rows <= 64 && per_lane > 12 && per_lane <= 32) {
#define PS_LAUNCH_NR(VPT)                                                                          \
  hipLaunchKernelGGL((norm_row_kernel<T, RMS, VPT>), dim3(n_rows), dim3(256), 0, s, x, rows, gamma, \
                     beta, (T*)out, width, eps, packed)
    if (per_lane <= 16) PS_LAUNCH_NR(4);
    else PS_LAUNCH_NR(8);
#undef PS_LAUNCH_NR
    return;
  }
#define PS_LAUNCH_NW(VPT)                                                                       \
  hipLaunchKernelGGL((norm_wave_kernel<T, RMS, VPT>), grid, dim3(256), 0, s, x, rows, gamma, beta, \
                     (T*)out, n_rows, width, eps, packed)
  if (per_lane <= 2) PS_LAUNCH_NW(2);
  else if (per_lane <= 4) PS_LAUNCH_NW(4);
  else if (per_lane <= 8) PS_LAUNCH_NW(8);
  else if (per_lane <= 12) PS_LAUNCH_NW(12);
  else if (per_lane <= 16) PS_LAUNCH_NW(16);
  else if (per_lane <= 32) PS_LAUNCH_NW(32);
  else
    hipLaunchKernelGGL((norm_block_kernel<T, RMS>), dim3(n_rows), dim3(256), 0, s, x, rows, gamma,
                       beta, (T*)out, width, eps);
#undef PS_LAUNCH_NW
}

// The norm with its rows written row by row (packed == 0) or in the operand order of the
// skinny product (packed_offset in linear.h; needs width a multiple of 64 up to 2048 and room
// for the row count rounded up to 16).
int ps_norm_layout(const float* x, const int* rows, const float* gamma, const float* beta,
                   void* out, int n_rows, int width, float eps, int rms, int out_dtype,
                   int packed, hipStream_t s) {
  PS_REQUIRE(n_rows >= 0 && width > 0, "ps_norm: bad sizes (rows %d, width %d)", n_rows, width);
  PS_REQUIRE(out_dtype == PS_F32 || out_dtype == PS_BF16, "ps_norm: unknown dtype %d", out_dtype);
  PS_REQUIRE(eps > 0.f, "ps_norm: eps must be positive");
  PS_REQUIRE(!packed || (width % 64 == 0 && width <= 2048),
             "ps_norm: the packed layout needs a width that is a multiple of 64 up to 2048");
  if (n_rows == 0) return 0;
  if (out_dtype == PS_F32) {
    if (rms) launch_norm<float, true>(x, rows, gamma, beta, out, n_rows, width, eps, packed, s);
    else launch_norm<float, false>(x, rows, gamma, beta, out, n_rows, width, eps, packed, s);
  } else {
    if (rms) launch_norm<bf16_t, true>(x, rows, gamma, beta, out, n_rows, width, eps, packed, s);
    else launch_norm<bf16_t, false>(x, rows, gamma, beta, out, n_rows, width, eps, packed, s);
  }
  PS_CHECK_LAUNCH("ps_norm");
  return 0;
}

extern "C" int ps_norm(const float* x, const int* rows, const float* gamma, const float* beta,
                       void* out, int n_rows, int width, float eps, int rms, int out_dtype,
                       void* stream) {
  return ps_norm_layout(x, rows, gamma, beta, out, n_rows, width, eps, rms, out_dtype, 0,
                        (hipStream_t)stream);
}

// ---------------------------------------------------------------- key/value scatter
// Token t of request r at position p is stored at (page = table[r][p / page], offset =
// p % page) (reference: src/model/kv_manager.py:303-308,403-404).
template <typename T>
__global__ void kv_write_kernel(const T* __restrict__ k, const T* __restrict__ v, int64_t stride,
                                T* __restrict__ k_pool, T* __restrict__ v_pool,
                                const int* __restrict__ tok_item, const int* __restrict__ tok_pos,
                                const int* __restrict__ tables, int table_width, int kv_heads,
                                int head_dim, int page_size, int num_pages) {
  const int t = blockIdx.x;
  const int pos = tok_pos[t];
  const int logical = pos / page_size;
  if (logical >= table_width) return;
  const int page = tables[(int64_t)tok_item[t] * table_width + logical];
  if (page < 0 || page >= num_pages) return;
  const int offset = pos - logical * page_size;
  const int row = kv_heads * head_dim;
  for (int i = threadIdx.x; i < row; i += blockDim.x) {
    const int head = i / head_dim;
    const int dim = i - head * head_dim;
    const int64_t dst = (((int64_t)page * kv_heads + head) * page_size + offset) * head_dim + dim;
    k_pool[dst] = k[(int64_t)t * stride + i];
    v_pool[dst] = v[(int64_t)t * stride + i];
  }
}

extern "C" int ps_kv_write(const void* k, const void* v, int64_t stride, void* k_pool,
                           void* v_pool, const int* tok_item, const int* tok_pos,
                           const int* tables, int table_width, int tokens, int kv_heads,
                           int head_dim, int page_size, int num_pages, int dtype, void* stream) {
  PS_REQUIRE(tokens >= 0 && kv_heads > 0 && head_dim > 0 && page_size > 0 && num_pages > 0 &&
                 table_width > 0,
             "ps_kv_write: bad sizes");
  PS_REQUIRE(stride >= (int64_t)kv_heads * head_dim, "ps_kv_write: row stride too small");
  PS_REQUIRE(dtype == PS_F32 || dtype == PS_BF16, "ps_kv_write: unknown dtype %d", dtype);
  if (tokens == 0) return 0;
  const int row = kv_heads * head_dim;
  const int threads = row >= 256 ? 256 : 64;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == PS_F32)
    hipLaunchKernelGGL(kv_write_kernel<float>, dim3(tokens), dim3(threads), 0, s, (const float*)k,
                       (const float*)v, stride, (float*)k_pool, (float*)v_pool, tok_item, tok_pos,
                       tables, table_width, kv_heads, head_dim, page_size, num_pages);
  else
    hipLaunchKernelGGL(kv_write_kernel<bf16_t>, dim3(tokens), dim3(threads), 0, s,
                       (const bf16_t*)k, (const bf16_t*)v, stride, (bf16_t*)k_pool,
                       (bf16_t*)v_pool, tok_item, tok_pos, tables, table_width, kv_heads, head_dim,
                       page_size, num_pages);
  PS_CHECK_LAUNCH("ps_kv_write");
  return 0;
}

// logits <- cap * tanh(logits / cap); a row is shared by blocks of 256 columns so that a
// handful of rows still fills the chip
__global__ void softcap_kernel(float* __restrict__ logits, int64_t ld, int vocab, float cap) {
  const int i = blockIdx.y * blockDim.x + threadIdx.x;
  if (i < vocab) {
    float* p = logits + (int64_t)blockIdx.x * ld + i;
    *p = cap * tanhf(*p / cap);
  }
}

extern "C" int ps_softcap(float* logits, int64_t ld, int rows, int vocab, float cap, void* stream) {
  PS_REQUIRE(rows >= 0 && vocab > 0 && ld >= vocab && cap > 0.f, "ps_softcap: bad sizes");
  PS_REQUIRE((vocab + 255) / 256 <= 65535, "ps_softcap: vocabulary too large");
  if (rows == 0) return 0;
  hipLaunchKernelGGL(softcap_kernel, dim3(rows, (vocab + 255) / 256), dim3(256), 0,
                     (hipStream_t)stream, logits, ld, vocab, cap);
  PS_CHECK_LAUNCH("ps_softcap");
  return 0;
}

// ---- words between pinned host memory and the device, by a kernel.  From some 16 KB on the copy
// engine's path holds a step up: with its indices (19 KB at 64 requests) through it a decode step
// took 37 us longer than its graph alone (493 against 456 us, GPT-2 small over 160 keys), with a kernel that
// reads the host's memory itself 18 us.  Below, either way costs a step the same (engine's path less kernel's, us a
// step: 28 words 0.1, 109 0.3, 217 0.1, 433 -0.4, 1,201 0.6, 2,401 1.1; 4,185 14.0, 4,801 11.5, 16,737 12.8), so there is no
// line between them.
__global__ __launch_bounds__(256) void copy_words_kernel(const uint32_t* __restrict__ src,
                                                         uint32_t* __restrict__ dst, int64_t words,
                                                         int pieces) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (pieces && i + 4 <= words) {
    *reinterpret_cast<uint4*>(dst + i) = *reinterpret_cast<const uint4*>(src + i);
    return;
  }
  for (int64_t at = i; at < i + 4 && at < words; ++at) dst[at] = src[at];
}

extern "C" int ps_copy_words(const void* src, void* dst, int64_t words, void* stream) {
  PS_REQUIRE(words >= 0 && words < ((int64_t)1 << 38), "ps_copy_words: bad size");
  if (words == 0) return 0;
  const uintptr_t a = reinterpret_cast<uintptr_t>(src), b = reinterpret_cast<uintptr_t>(dst);
  PS_REQUIRE(a != 0 && b != 0 && (a & 3u) == 0 && (b & 3u) == 0, "ps_copy_words: null or unaligned memory");
  const int pieces = ((a | b) & 15u) == 0;
  hipLaunchKernelGGL(copy_words_kernel, dim3((unsigned)((words + 1023) / 1024)), dim3(256), 0,
                     (hipStream_t)stream, (const uint32_t*)src, (uint32_t*)dst, words, pieces);
  PS_CHECK_LAUNCH("ps_copy_words");
  return 0;
}

// The address under which kernels reach pinned host memory.
extern "C" int ps_host_address(void* host, void** address) {
  PS_REQUIRE(host != nullptr && address != nullptr, "ps_host_address: null pointer");
  const hipError_t status = hipHostGetDevicePointer(address, host, 0);
  if (status != hipSuccess) {
    (void)hipGetLastError();   // (the error is reported here and must not be found by the next call)
    ps_set_error("ps_host_address: not pinned host memory (%s)", hipGetErrorString(status));
    return 1;
  }
  return 0;
}
