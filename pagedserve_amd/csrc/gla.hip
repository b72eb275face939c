// Gated linear attention: a recurrent mixer whose state is a matrix per head.
//
//   S_t = diag(alpha_t) S_(t-1) + k_t v_t^T        (S: [key_dim, value_dim], float, per request)
//   o_t = S_t^T q_t
//
// with a decay alpha in (0, 1) per key channel, alpha = sigmoid(z)^(1/tau), z a low-rank
// projection of the layer's input.  Three launches: the decays of the step's tokens, the
// recurrence, and the output's norm and gate.  The state, the decays and everything they are
// made from are 32-bit; q, k, v arrive as the float columns of the layer's projection.
#include <math.h>

#include "common.h"
#include "pagedserve_hip.h"

// alpha[t, c] = exp(log_sigmoid(z) / tau), z = bias[c] + sum_r low[t, r] w[c, r].
template <typename T>
__global__ __launch_bounds__(256) void gla_decay_kernel(
    const float* __restrict__ proj, int64_t ld, int low_col, int rank, const T* __restrict__ w,
    const float* __restrict__ bias, float inv_tau, float* __restrict__ alpha, int channels) {
  extern __shared__ float low[];
  const int t = blockIdx.x;
  for (int r = threadIdx.x; r < rank; r += blockDim.x) low[r] = proj[(int64_t)t * ld + low_col + r];
  __syncthreads();
  for (int c = threadIdx.x; c < channels; c += blockDim.x) {
    float z = bias ? bias[c] : 0.f;
    const T* w_row = w + (int64_t)c * rank;
    for (int r = 0; r < rank; ++r) z = fmaf(low[r], to_float<T>(w_row[r]), z);
    // log sigmoid(z) = min(z, 0) - log(1 + exp(-|z|))
    const float log_sigmoid = fminf(z, 0.f) - log1pf(expf(-fabsf(z)));
    alpha[(int64_t)t * channels + c] = expf(log_sigmoid * inv_tau);
  }
}

// The same for a rank of PIECES whole pieces of 16 bytes: a thread takes one channel and asks for all of its weights at
// once, and the scalar unit for the row (the loop above makes a trip for every few of them; the sums are in the same
// order).  8 tokens of 768 channels and a rank of 16 in a decode step: 5.45 -> 2.6 us.
template <typename T, int PIECES>
__global__ __launch_bounds__(256) void gla_decay_pieces_kernel(
    const float* __restrict__ low_rows, int64_t ld, const T* __restrict__ w, const float* __restrict__ bias,
    float* __restrict__ alpha, float inv_tau, int channels) {
  constexpr int EACH = 16 / (int)sizeof(T), RANK = PIECES * EACH;
  const int t = blockIdx.x;
  const int c = blockIdx.y * 256 + threadIdx.x;
  const int safe = c < channels ? c : channels - 1;
  uint4 raw[PIECES];
#pragma unroll
  for (int p = 0; p < PIECES; ++p) raw[p] = *reinterpret_cast<const uint4*>(w + (int64_t)safe * RANK + p * EACH);
  float low[RANK];
#pragma unroll
  for (int r = 0; r < RANK; ++r) low[r] = scalar_load(low_rows + (int64_t)t * ld + r);
  float z = bias ? bias[safe] : 0.f;
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int r = 0; r < RANK; ++r) argument_is_read(low[r]);
#pragma unroll
  for (int p = 0; p < PIECES; ++p) {
    const uint32_t words[4] = {raw[p].x, raw[p].y, raw[p].z, raw[p].w};
#pragma unroll
    for (int e = 0; e < EACH; ++e) {
      const uint32_t bits = sizeof(T) == 4 ? words[e & 3] : e & 1 ? words[e / 2 & 3] & 0xFFFF0000u : words[e / 2 & 3] << 16;
      const float weight = __builtin_bit_cast(float, bits);
      z = fmaf(low[p * EACH + e], weight, z);
    }
  }
  if (c >= channels) return;
  const float log_sigmoid = fminf(z, 0.f) - log1pf(expf(-fabsf(z)));
  alpha[(int64_t)t * channels + c] = expf(log_sigmoid * inv_tau);
}

// A block owns COLS columns of one head's state for one item of the step and walks the item's tokens in order:
// thread = row group * COLS + column.  The state's rows are dealt to the row groups, RPL rows per thread, in
// registers; o needs the sum over the row groups, which is taken through LDS once per chunk.  The tokens' q, k and
// decays come GLA_CHUNK at a time: a chunk's loads leave together into registers while the chunk before is being
// worked on from LDS.
//
// What bounds it: the walk is one dependent chain per token, so that a prompt waits for what a thread does per
// token (3 RPL multiply-adds, four LDS reads, one write) and for its part of the staging.  Prompts therefore
// take four waves to 16 columns, which stage q, k and decays for all of them; blocks of one wave and 4
// columns staged them four times as often, 57 KB of LDS each, two to a compute unit.  5 prompts of 400 tokens at
// 12 heads of 64: 151 -> 44 us, 16 of 128: 45 -> 27, one of 2,000: 350 -> 193.  Chunks of 32 let one block into
// a unit instead of three (16 prompts of 128 45 us, 5 of 400 49).  Steps of up to eight
// tokens an item take one wave: 16 columns in chunks of 8 where that gives blocks enough, else 4, in chunks of 8 or,
// of single tokens, of one.
#define GLA_LONG 16   // tokens of a chunk of a prompt

template <int RPL, int COLS, int GLA_CHUNK, int WAVES, bool HEAD_DECAY>
__global__ __launch_bounds__(64 * WAVES) void gla_scan_kernel(
    const int* __restrict__ cu_tokens, const int* __restrict__ slots, float* __restrict__ state,
    const float* __restrict__ proj, const float* __restrict__ alpha, int heads, int key_dim, int value_dim, int q_col,
    int64_t ld, int k_col, int v_col, float* __restrict__ out, float q_scale, int silu_inputs,
    const float* __restrict__ head_decay) {
  constexpr int THREADS = 64 * WAVES;
  constexpr int GROUPS = THREADS / COLS;                // row groups
  constexpr int ROWS = GROUPS * RPL;               // rows with padding up to the lanes' share
  constexpr int PAD = RPL + 4;                     // row groups start in different banks
  constexpr int PER = GLA_CHUNK * ROWS / THREADS;       // values of a chunk per lane and array
  constexpr int PER_V = (GLA_CHUNK * COLS + THREADS - 1) / THREADS;
  static_assert(GLA_CHUNK * ROWS % THREADS == 0 && PER >= 1, "a chunk's rows are dealt evenly to the lanes");
  __shared__ __attribute__((aligned(16))) float s_q[GLA_CHUNK][GROUPS * PAD];
  __shared__ __attribute__((aligned(16))) float s_k[GLA_CHUNK][GROUPS * PAD];
  __shared__ __attribute__((aligned(16))) float s_a[GLA_CHUNK][GROUPS * PAD];
  __shared__ float s_v[GLA_CHUNK][COLS];
  __shared__ float s_o[GLA_CHUNK][THREADS + 1];     // every thread's share of o_t (rows one bank apart)
  const int item = blockIdx.x, head = blockIdx.y;
  const int lane = threadIdx.x;
  const int col = blockIdx.z * COLS + (lane % COLS);
  const int group = lane / COLS;
  const bool has_col = col < value_dim;
  const int t0 = scalar_load(cu_tokens + item), t1 = scalar_load(cu_tokens + item + 1);
  const int slot = scalar_load(slots + item);
  read_arguments(t0, t1, slot, ld, k_col, v_col, out, q_scale, silu_inputs, head_decay);
  float* s_ptr = state + (((int64_t)slot * heads + head) * key_dim) * value_dim;
  float S[RPL];
#pragma unroll
  for (int i = 0; i < RPL; ++i) {
    // (unconditional, and masked as bits where they are used: nothing waits for a branch)
    const int r = group * RPL + i;
    S[i] = s_ptr[(int64_t)(r < key_dim ? r : 0) * value_dim + (has_col ? col : 0)];
  }
  const int channels = heads * key_dim;
  float rq[PER], rk[PER], ra[PER], rv[PER_V];
  // one decay per head for all key channels and tokens (then no array of decays is read)
  const float fixed_decay = HEAD_DECAY ? head_decay[head] : 0.f;
  // every load is unconditional from a clamped address; what lies outside is masked when stored
  auto fetch = [&](const int base) {
    const int count = (t1 - base) < GLA_CHUNK ? (t1 - base) : GLA_CHUNK;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int idx = lane + j * THREADS;
      const int tt = idx / ROWS;
      const int r = idx - tt * ROWS;
      const int64_t t = base + (tt < count ? tt : 0);
      const int c = head * key_dim + (r < key_dim ? r : 0);
      rq[j] = proj[t * ld + q_col + c];
      rk[j] = proj[t * ld + k_col + c];
      ra[j] = HEAD_DECAY ? fixed_decay : alpha[t * channels + c];
    }
#pragma unroll
    for (int j = 0; j < PER_V; ++j) {
      const int idx = (lane + j * THREADS) % (GLA_CHUNK * COLS);
      const int tt = idx / COLS;
      const int c = blockIdx.z * COLS + (idx - tt * COLS);
      const int64_t t = base + (tt < count ? tt : 0);
      rv[j] = proj[t * ld + v_col + head * value_dim + (c < value_dim ? c : 0)];
    }
  };
  auto stash = [&](const int base) {
    const int count = (t1 - base) < GLA_CHUNK ? (t1 - base) : GLA_CHUNK;
    if (silu_inputs) {
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        rq[j] = rq[j] / (1.0f + expf(-rq[j]));
        rk[j] = rk[j] / (1.0f + expf(-rk[j]));
      }
#pragma unroll
      for (int j = 0; j < PER_V; ++j) rv[j] = rv[j] / (1.0f + expf(-rv[j]));
    }
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int idx = lane + j * THREADS;
      const int tt = idx / ROWS;
      const int r = idx - tt * ROWS;
      const bool valid = tt < count && r < key_dim;
      const int at = (r / RPL) * PAD + (r % RPL);
      s_q[tt][at] = valid ? rq[j] * q_scale : 0.f;
      s_k[tt][at] = valid ? rk[j] : 0.f;
      s_a[tt][at] = valid ? ra[j] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < PER_V; ++j) {
      const int idx = lane + j * THREADS;
      if (idx < GLA_CHUNK * COLS) {
        const int tt = idx / COLS;
        const int c = blockIdx.z * COLS + (idx - tt * COLS);
        s_v[tt][idx - tt * COLS] = (tt < count && c < value_dim) ? rv[j] : 0.f;
      }
    }
  };
  if (t0 < t1) fetch(t0);
#pragma unroll
  for (int i = 0; i < RPL; ++i)
    S[i] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, S[i]) &
                                         (group * RPL + i < key_dim && has_col ? 0xFFFFFFFFu : 0u));
  for (int base = t0; base < t1; base += GLA_CHUNK) {
    const int count = (t1 - base) < GLA_CHUNK ? (t1 - base) : GLA_CHUNK;
    __syncthreads();      // the chunk before has been read
    stash(base);
    __syncthreads();
    if (base + GLA_CHUNK < t1) fetch(base + GLA_CHUNK);   // in flight during the work below
    // a lane's share of o_t
    auto token = [&](const int tt) -> float {
      const float v = s_v[tt][lane % COLS];
      float o = 0.f;
#pragma unroll
      for (int i = 0; i < RPL; ++i) {
        const int at = group * PAD + i;
        S[i] = fmaf(s_a[tt][at], S[i], s_k[tt][at] * v);
        o = fmaf(S[i], s_q[tt][at], o);
      }
      return o;
    };
    // The lanes' shares wait in LDS: the state's chain then holds no exchange between lanes,
    // and the sums over the row groups are taken for all tokens of the chunk at once.
    if (count == GLA_CHUNK) {
      // a whole chunk: unrolled, so that the reads of the next tokens run ahead of the chain
#pragma unroll
      for (int tt = 0; tt < GLA_CHUNK; ++tt) s_o[tt][lane] = token(tt);
    } else {
      for (int tt = 0; tt < count; ++tt) s_o[tt][lane] = token(tt);
    }
    __syncthreads();
    for (int idx = lane; idx < count * COLS; idx += THREADS) {
      const int tt = idx / COLS;
      const int c = idx - tt * COLS;
      float sum = 0.f;
#pragma unroll
      for (int g = 0; g < GROUPS; ++g) sum += s_o[tt][g * COLS + c];
      const int to = blockIdx.z * COLS + c;
      if (to < value_dim) out[(int64_t)(base + tt) * heads * value_dim + head * value_dim + to] = sum;
    }
  }
#pragma unroll
  for (int i = 0; i < RPL; ++i) {
    const int r = group * RPL + i;
    if (r < key_dim && has_col) s_ptr[(int64_t)r * value_dim + col] = S[i];
  }
}

// out[t, h, :] = o[t, h, :] / sqrt(mean(o[t, h, :]^2) + eps) * w * silu(gate[t, h, :]).
// DIMS values to a lane, asked for with their weights and gates in one trip (8 tokens of 12 heads of 64
// 4.45 -> 2.25 us); 0: any number, in two.
template <typename T, int DIMS>
__global__ __launch_bounds__(64) void gla_output_kernel(
    const float* __restrict__ o, const float* __restrict__ w, const float* __restrict__ gate, int64_t gate_ld,
    int heads, int value_dim, T* __restrict__ out, int64_t out_stride, float eps) {
  const int t = blockIdx.x, head = blockIdx.y, lane = threadIdx.x;
  const float* row = o + ((int64_t)t * heads + head) * value_dim;
  const float* gates = gate + (int64_t)t * gate_ld + head * value_dim;
  if constexpr (DIMS > 0) {
    float v[DIMS], g[DIMS], weight[DIMS];
#pragma unroll
    for (int i = 0; i < DIMS; ++i) {
      const int d = lane + i * 64 < value_dim ? lane + i * 64 : 0;
      v[i] = row[d];
      g[i] = gates[d];
      weight[i] = w[d];
    }
    read_arguments(out, out_stride, eps);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < DIMS; ++i)
      if (lane + i * 64 < value_dim) sum = fmaf(v[i], v[i], sum);
    const float inv = 1.0f / sqrtf(wave_sum(sum) / (float)value_dim + eps);
#pragma unroll
    for (int i = 0; i < DIMS; ++i) {
      const int d = lane + i * 64;
      const float silu = g[i] / (1.0f + expf(-g[i]));
      if (d < value_dim)
        out[(int64_t)t * out_stride + head * value_dim + d] = from_float<T>(v[i] * inv * weight[i] * silu);
    }
    return;
  }
  float sum = 0.f;
  for (int d = lane; d < value_dim; d += 64) sum = fmaf(row[d], row[d], sum);
  const float inv = 1.0f / sqrtf(wave_sum(sum) / (float)value_dim + eps);
  for (int d = lane; d < value_dim; d += 64) {
    const float g = gates[d];
    const float silu = g / (1.0f + expf(-g));
    out[(int64_t)t * out_stride + head * value_dim + d] = from_float<T>(row[d] * inv * w[d] * silu);
  }
}

// out[t, :] = o[t, :] / sqrt(mean(o[t, :]^2) + eps) * w * sigmoid(gate[t, :]): the norm over the
// whole row (all heads together), a block per token.
template <typename T>
__global__ __launch_bounds__(256) void row_norm_gate_kernel(
    const float* __restrict__ o, const float* __restrict__ w, float eps,
    const float* __restrict__ gate, int64_t gate_ld, T* __restrict__ out, int64_t out_stride,
    int columns) {
  __shared__ __attribute__((aligned(16))) float scratch[16];
  const int t = blockIdx.x;
  const float* row = o + (int64_t)t * columns;
  float sum = 0.f;
  for (int d = threadIdx.x; d < columns; d += blockDim.x) sum = fmaf(row[d], row[d], sum);
  const float inv = 1.0f / sqrtf(block_sum(sum, scratch) / (float)columns + eps);
  for (int d = threadIdx.x; d < columns; d += blockDim.x) {
    const float g = gate[(int64_t)t * gate_ld + d];
    out[(int64_t)t * out_stride + d] = from_float<T>(row[d] * inv * w[d] / (1.0f + expf(-g)));
  }
}

extern "C" int ps_row_norm_gate(const float* o, const float* w, float eps, const float* gate,
                                int64_t gate_ld, void* out, int64_t out_stride, int tokens,
                                int columns, int dtype, void* stream) {
  PS_REQUIRE(tokens >= 0 && columns > 0 && eps > 0.f, "ps_row_norm_gate: bad sizes");
  PS_REQUIRE(dtype == PS_F32 || dtype == PS_BF16, "ps_row_norm_gate: unknown dtype %d", dtype);
  if (tokens == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == PS_F32)
    hipLaunchKernelGGL(row_norm_gate_kernel<float>, dim3(tokens), dim3(256), 0, s, o, w, eps, gate,
                       gate_ld, (float*)out, out_stride, columns);
  else
    hipLaunchKernelGGL(row_norm_gate_kernel<bf16_t>, dim3(tokens), dim3(256), 0, s, o, w, eps, gate,
                       gate_ld, (bf16_t*)out, out_stride, columns);
  PS_CHECK_LAUNCH("ps_row_norm_gate");
  return 0;
}

// ---- long portions in pieces that run side by side (recurrences with one decay per head) ----
// The recurrence is linear in the state: a piece of n tokens takes S to d^n S + E, with E what
// it leaves from a zero state.  So the items of a step are cut into pieces, every piece runs
// the recurrence kernel as an item of its own with a state of its own (first from zero, which
// leaves E there; then, once ps_decay_join has put every piece's true start in E's place, again,
// now for the outputs).
//
// piece_cu[k] .. piece_cu[k + 1]: the tokens of piece k (empty behind the last piece);
// item_first[i]: the first piece of item i.  One thread: a step has a handful of items.
__global__ void scan_pieces_kernel(const int* __restrict__ cu_tokens, int items, int piece,
                                   int max_pieces, int* __restrict__ piece_cu,
                                   int* __restrict__ item_first) {
  if (blockIdx.x != 0 || threadIdx.x != 0) return;
  int at = 0;
  for (int i = 0; i < items; ++i) {
    item_first[i] = at;
    for (int t = cu_tokens[i]; t < cu_tokens[i + 1] && at < max_pieces; t += piece) piece_cu[at++] = t;
  }
  item_first[items] = at;
  for (int k = at; k <= max_pieces; ++k) piece_cu[k] = cu_tokens[items];
}

// A thread per number of an item's state: S <- the slot's; for the item's pieces in order:
// E <-> S's place (the piece's start), S <- d^n S + E; the last S goes to the slot.
__global__ __launch_bounds__(256) void decay_join_kernel(
    float* __restrict__ piece_states, float* __restrict__ state, const int* __restrict__ piece_cu,
    const int* __restrict__ item_first, const int* __restrict__ slots,
    const float* __restrict__ head_decay, int heads, int per_head) {
  const int item = blockIdx.x, head = blockIdx.y;
  const int e = blockIdx.z * 256 + threadIdx.x;
  if (e >= per_head) return;
  const int first = item_first[item], last = item_first[item + 1];
  if (first == last) return;
  const float d = head_decay[head];
  float* mine = state + ((int64_t)slots[item] * heads + head) * per_head + e;
  float s = *mine;
  for (int k = first; k < last; ++k) {
    float* record = piece_states + ((int64_t)k * heads + head) * per_head + e;
    const float left = *record;
    *record = s;
    s = fmaf(powf(d, (float)(piece_cu[k + 1] - piece_cu[k])), s, left);
  }
  *mine = s;
}

extern "C" int ps_scan_pieces(const int* cu_tokens, int items, int piece, int max_pieces,
                              int* piece_cu, int* item_first, void* stream) {
  PS_REQUIRE(items >= 0 && piece > 0 && max_pieces >= 0, "ps_scan_pieces: bad sizes");
  hipLaunchKernelGGL(scan_pieces_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, cu_tokens, items,
                     piece, max_pieces, piece_cu, item_first);
  PS_CHECK_LAUNCH("ps_scan_pieces");
  return 0;
}

extern "C" int ps_decay_join(float* piece_states, float* state, const int* piece_cu,
                             const int* item_first, const int* slots, const float* head_decay,
                             int items, int heads, int per_head, void* stream) {
  PS_REQUIRE(items >= 0 && heads > 0 && per_head > 0, "ps_decay_join: bad sizes");
  if (items == 0) return 0;
  hipLaunchKernelGGL(decay_join_kernel, dim3(items, heads, (per_head + 255) / 256), dim3(256), 0,
                     (hipStream_t)stream, piece_states, state, piece_cu, item_first, slots,
                     head_decay, heads, per_head);
  PS_CHECK_LAUNCH("ps_decay_join");
  return 0;
}

extern "C" int ps_gla_decay(const float* proj, int64_t ld, int low_col, int rank, const void* w,
                            const float* bias, float tau, float* alpha, int tokens, int channels,
                            int dtype, void* stream) {
  PS_REQUIRE(tokens >= 0 && rank > 0 && channels > 0 && tau > 0.f, "ps_gla_decay: bad sizes");
  PS_REQUIRE(rank <= 8192, "ps_gla_decay: rank %d above 8192", rank);
  PS_REQUIRE(dtype == PS_F32 || dtype == PS_BF16, "ps_gla_decay: unknown dtype %d", dtype);
  if (tokens == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const size_t lds = (size_t)rank * sizeof(float);
#define PS_LAUNCH_GD(T)                                                                                        \
  hipLaunchKernelGGL(gla_decay_kernel<T>, dim3(tokens), dim3(256), lds, s, proj, ld, low_col, rank, (const T*)w, \
                     bias, 1.0f / tau, alpha, channels)
#define PS_LAUNCH_GDP(T, PIECES)                                                                               \
  hipLaunchKernelGGL((gla_decay_pieces_kernel<T, PIECES>), dim3(tokens, (channels + 255) / 256), dim3(256), 0, \
                     s, proj + low_col, ld, (const T*)w, bias, alpha, 1.0f / tau, channels)
  const bool aligned = ((uintptr_t)w & 15u) == 0;
  if (dtype == PS_F32) {
    if (aligned && rank == 8) PS_LAUNCH_GDP(float, 2);
    else if (aligned && rank == 16) PS_LAUNCH_GDP(float, 4);
    else if (aligned && rank == 32) PS_LAUNCH_GDP(float, 8);
    else PS_LAUNCH_GD(float);
  } else {
    if (aligned && rank == 8) PS_LAUNCH_GDP(bf16_t, 1);
    else if (aligned && rank == 16) PS_LAUNCH_GDP(bf16_t, 2);
    else if (aligned && rank == 32) PS_LAUNCH_GDP(bf16_t, 4);
    else PS_LAUNCH_GD(bf16_t);
  }
#undef PS_LAUNCH_GD
#undef PS_LAUNCH_GDP
  PS_CHECK_LAUNCH("ps_gla_decay");
  return 0;
}

extern "C" int ps_gla_scan(const float* proj, int64_t ld, int q_col, int k_col, int v_col,
                           const float* alpha, float* state, float* out, const int* cu_tokens,
                           const int* slots, int items, int max_slots, int heads, int key_dim,
                           int value_dim, float q_scale, int longest, const float* head_decay,
                           int silu_inputs, void* stream) {
  PS_REQUIRE(alpha != nullptr || head_decay != nullptr, "ps_gla_scan: no decays given");
  PS_REQUIRE(items >= 0 && heads > 0 && key_dim > 0 && value_dim > 0 && max_slots > 0,
             "ps_gla_scan: bad sizes");
  PS_REQUIRE(key_dim <= 256, "ps_gla_scan: key head size %d above 256", key_dim);
  PS_REQUIRE(heads <= 65535 && (value_dim + 3) / 4 <= 65535, "ps_gla_scan: grid too large");
  if (items == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  // items of a few tokens at most (decode steps): chunks of 8 or fewer, which cost less to stage, and blocks of one
  // wave, narrow ones while wide ones would leave the chip's SIMDs (four to a compute unit) idle
  const int64_t wide_blocks = (int64_t)items * heads * ((value_dim + 15) / 16);
  const bool narrow = wide_blocks < 2 * (int64_t)ps_compute_units();
  const bool brief = longest > 0 && longest <= 8;
#define PS_LAUNCH_GLA_H(RPL, COLS, CHUNK, WAVES, HEAD)                                            \
  hipLaunchKernelGGL((gla_scan_kernel<RPL, COLS, CHUNK, WAVES, HEAD>),                            \
                     dim3(items, heads, (value_dim + COLS - 1) / COLS),                           \
                     dim3(64 * WAVES), 0, s, cu_tokens, slots, state, proj, alpha, heads,         \
                     key_dim, value_dim, q_col, ld, k_col, v_col, out, q_scale, silu_inputs, head_decay)
#define PS_LAUNCH_GLA(RPL, COLS, CHUNK, WAVES)                                                    \
  do {                                                                                            \
    if (head_decay != nullptr) PS_LAUNCH_GLA_H(RPL, COLS, CHUNK, WAVES, true);                    \
    else PS_LAUNCH_GLA_H(RPL, COLS, CHUNK, WAVES, false);                                         \
  } while (0)
  if (!brief) {
    if (key_dim <= 32) PS_LAUNCH_GLA(2, 16, GLA_LONG, 4);
    else if (key_dim <= 64) PS_LAUNCH_GLA(4, 16, GLA_LONG, 4);
    else if (key_dim <= 128) PS_LAUNCH_GLA(8, 16, GLA_LONG, 4);
    else PS_LAUNCH_GLA(16, 16, GLA_LONG / 2, 4);
  } else if (narrow && longest == 1) {
    // one token each: nothing is staged that is not there (8 items of 12 heads of 64: 5.45 -> 3.95 us; a chunk's rows
    // are dealt to the lanes whole, two tokens of up to 32 keys)
    if (key_dim <= 32) PS_LAUNCH_GLA(2, 4, 2, 1);
    else if (key_dim <= 64) PS_LAUNCH_GLA(4, 4, 1, 1);
    else if (key_dim <= 128) PS_LAUNCH_GLA(8, 4, 1, 1);
    else PS_LAUNCH_GLA(16, 4, 1, 1);
  } else if (narrow) {
    if (key_dim <= 32) PS_LAUNCH_GLA(2, 4, 8, 1);
    else if (key_dim <= 64) PS_LAUNCH_GLA(4, 4, 8, 1);
    else if (key_dim <= 128) PS_LAUNCH_GLA(8, 4, 8, 1);
    else PS_LAUNCH_GLA(16, 4, 8, 1);
  } else {
    if (key_dim <= 32) PS_LAUNCH_GLA(8, 16, 8, 1);
    else if (key_dim <= 64) PS_LAUNCH_GLA(16, 16, 8, 1);
    else if (key_dim <= 128) PS_LAUNCH_GLA(32, 16, 8, 1);
    else PS_LAUNCH_GLA(64, 16, 8, 1);
  }
#undef PS_LAUNCH_GLA
#undef PS_LAUNCH_GLA_H
  PS_CHECK_LAUNCH("ps_gla_scan");
  return 0;
}

extern "C" int ps_gla_output(const float* o, const float* w, float eps, const float* gate,
                             int64_t gate_ld, void* out, int64_t out_stride, int tokens, int heads,
                             int value_dim, int dtype, void* stream) {
  PS_REQUIRE(tokens >= 0 && heads > 0 && value_dim > 0 && eps > 0.f && heads <= 65535,
             "ps_gla_output: bad sizes");
  PS_REQUIRE(dtype == PS_F32 || dtype == PS_BF16, "ps_gla_output: unknown dtype %d", dtype);
  if (tokens == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
#define PS_LAUNCH_GO_AS(T, DIMS)                                                                              \
  hipLaunchKernelGGL((gla_output_kernel<T, DIMS>), dim3(tokens, heads), dim3(64), 0, s, o, w, gate, gate_ld,  \
                     heads, value_dim, (T*)out, out_stride, eps)
#define PS_LAUNCH_GO(T)                            \
  do {                                             \
    if (value_dim <= 64) PS_LAUNCH_GO_AS(T, 1);    \
    else if (value_dim <= 128) PS_LAUNCH_GO_AS(T, 2); \
    else if (value_dim <= 256) PS_LAUNCH_GO_AS(T, 4); \
    else PS_LAUNCH_GO_AS(T, 0);                    \
  } while (0)
  if (dtype == PS_F32) PS_LAUNCH_GO(float);
  else PS_LAUNCH_GO(bf16_t);
#undef PS_LAUNCH_GO
#undef PS_LAUNCH_GO_AS
  PS_CHECK_LAUNCH("ps_gla_output");
  return 0;
}
