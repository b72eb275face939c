// The decode attention's block (see attention_decode.hip for the method): shared by the kernel
// of that file and by the kernel of attention_mixed.hip, which runs such blocks beside the
// blocks of the tiled prefill attention in one launch.
#pragma once
#include <math.h>

#include <type_traits>

#include "common.h"

// 2^x (the arguments here are never positive).  Scores are kept in units of log 2, so that no
// multiplication precedes it.  The 32-bit path takes the library's exp2f, which is exact to an
// ulp over the whole range, tiny results included; bfloat16 storage takes the bare hardware
// instruction.
template <typename T>
__device__ inline float exp2_fast(float x) {
  if constexpr (sizeof(T) == 4) return exp2f(x);
  else return __builtin_amdgcn_exp2f(x);
}

// Over the lanes that hold the same head dimensions (l ^ LPK, l ^ 2 LPK, ... l ^ 32): the
// maximum, then the sums of the states scaled to it.
template <int LPK>
__device__ inline float groups_max(float v) {
  if (LPK <= 1) v = xor_max<1>(v);
  if (LPK <= 2) v = xor_max<2>(v);
  if (LPK <= 4) v = xor_max<4>(v);
  if (LPK <= 8) v = xor_max<8>(v);
  if (LPK <= 16) v = xor_max<16>(v);
  return xor_max<32>(v);
}
template <int LPK>
__device__ inline float groups_sum(float v) {
  if (LPK <= 1) v = xor_sum<1>(v);
  if (LPK <= 2) v = xor_sum<2>(v);
  if (LPK <= 4) v = xor_sum<4>(v);
  if (LPK <= 8) v = xor_sum<8>(v);
  if (LPK <= 16) v = xor_sum<16>(v);
  return xor_sum<32>(v);
}

// What a block of this kernel keeps in LDS, in floats: the waves' accumulators and their (m, l).
template <int AD_WAVES>
struct DecodeLds {
  __attribute__((aligned(16))) float acc[AD_WAVES][256];
  __attribute__((aligned(8))) float ml[AD_WAVES][2];
};

// The address in global memory that a lane holds, in scalar registers.
typedef const char __attribute__((address_space(1))) * global_bytes;
__device__ inline global_bytes read_address(uint64_t held, int lane) {
  const unsigned low = __builtin_amdgcn_readlane((int)(unsigned)held, lane);
  const unsigned high = __builtin_amdgcn_readlane((int)(unsigned)(held >> 32), lane);
  return reinterpret_cast<global_bytes>((uint64_t)high << 32 | low);
}

struct NothingAhead {
  __device__ void operator()() const {}
};

// How a launch's pages are walked, worked out on the host: a word that comes with the launch.
#define AD_SHIFT(form) (((form) & 63) - 1)     // log2 of the page size, -1: no power of two
#define AD_EVEN 64          // the keys of one load lie in one page, whose bytes are counted in 31 bits
#define AD_FROM_START 128   // token t is item t and its block walks all keys from the first: the first entries of the
                            // block table are known without the position
#define AD_HEAD_DIM(form) ((form) >> 16)
inline int decode_form(int head_dim, int page_size, int kv_heads, bool from_start) {
  int lanes = 1;            // to a key, eight values each: 64 / lanes keys to a load
  while (lanes * 8 < head_dim) lanes *= 2;
  int shift = -1;
  if ((page_size & (page_size - 1)) == 0) {
    shift = 0;
    while ((1 << shift) < page_size) ++shift;
  }
  const bool even = shift >= 0 && page_size >= 64 / lanes &&
                    (int64_t)page_size * kv_heads * head_dim < ((int64_t)1 << 29);
  return (shift + 1) | (even ? AD_EVEN : 0) | (from_start ? AD_FROM_START : 0) | (head_dim << 16);
}

// The work of one block: token n of the list, one head, one range of its keys.  The caller
// provides the block's LDS (the kernel below its own; a kernel that runs blocks of several
// kinds in one launch a share of what all of them need).  `context` (one split only): the head's
// finished values go there, into LDS, for the caller to go on with, instead of to `out`.
// `ahead` runs once in every wave, behind the first loads of keys and values: loads that the caller
// wants to travel beside them and needs later.  (A wave's loads come back in the order of issue; asked
// for earlier they would hold back the block table and with it the keys.)
//
// Where a block has a turn or two over its keys the launch is bound by the chain position and block table -> keys
// and values -> exchange, and by every instruction between them.  So the first trip asks for position, table
// entries, query and the kernel's remaining arguments at once.  Where the keys of one load lie in one page (AD_EVEN)
// lane r of a wave works out where the r-th page of its turn lies, once for all loads; a load reads that from the lane,
// adds the key's place in the scalar unit and a constant per lane, and the entries of the next turn travel beside
// the keys of this one.  The general form exchanges the entries through LDS and makes an address in every lane, some 30
// vector instructions and a wait per load.  (us, keys from memory, before and now: 64 requests of 12 heads of 64 over 144
// and 400 keys in bfloat16 10.4 and 9.0, 19.5 and 17.6, 16 over 400 keys 9.5 and 8.1; 16 over 400 in float 12.8 and
// 10.9; 538 shapes of both types 0.87 of the time, with the ranges of parts/attention.py 0.83.)
template <typename T, int LPK, int AD_WAVES, int AD_UNROLL, bool NT, typename Ahead = NothingAhead>
__device__ __forceinline__ void attention_decode_block(
    DecodeLds<AD_WAVES>& lds, const int n, const int head, const int split,
    const T* __restrict__ q, int64_t q_stride, const T* __restrict__ k_pool,
    const T* __restrict__ v_pool, T* __restrict__ out, int64_t out_stride,
    float* __restrict__ partial, const int* __restrict__ tok_list,
    const int* __restrict__ tok_item, const int* __restrict__ tok_pos,
    const int* __restrict__ tables, int table_width, int heads, int kv_heads, int kv_group, int form,
    int page_size, int num_pages, float scale_log2, int window, int splits,
    const AttnExtras extra, T* context = nullptr, Ahead ahead = Ahead()) {
  constexpr int GROUPS = 64 / LPK;               // keys per wave load
  constexpr int KEYS_PER_WAVE = GROUPS * AD_UNROLL;
  float (&s_acc)[AD_WAVES][256] = lds.acc;
  float (&s_ml)[AD_WAVES][2] = lds.ml;

  const int t = tok_list ? tok_list[n] : n;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // the same in every lane: scalar
  const int group = lane / LPK;
  const int dim0 = (lane % LPK) * 8;
  const int head_dim = AD_HEAD_DIM(form), page_shift = AD_SHIFT(form);
  const bool even = form & AD_EVEN;
  const bool has_dims = dim0 < head_dim;
  const int lane_dim = has_dims ? dim0 : 0;

  // tok_item == null: token t is item t (a step of single tokens only).  The row of the
  // block table is then known without a load, and its entries (the first ones, or in the general form all of
  // a short row) are asked for at once, beside the position, instead of behind it: one trip to memory less on the
  // way to the first keys.
  const bool direct = tok_item == nullptr;
  const bool prefetched = !even && direct && table_width <= 128;
  int held = 0, held1 = 0;
  if (prefetched) {
    // (lane l holds entries l and l + 64; the lanes hand them to each other)
    const int* row = tables + (int64_t)t * table_width;
    held = row[lane < table_width ? lane : table_width - 1];
    if (table_width > 64) held1 = row[lane + 64 < table_width ? lane + 64 : table_width - 1];
  }
  // (of a turn that begins at key `base` no lane beyond the first AD_UNROLL + 1 is asked; a token of a negative position,
  // which sees no key, has ranges that begin in front of the table)
  auto ask_entries = [&](const int* row, int base) {
    const int entry = ((base > 0 ? base : 0) >> page_shift) + (lane < AD_UNROLL ? lane : AD_UNROLL);
    held = row[entry < table_width ? entry : table_width - 1];
  };
  const bool from_start = even && (form & AD_FROM_START);
  if (from_start) ask_entries(tables + (int64_t)t * table_width, wave * KEYS_PER_WAVE);
  Raw8<T> query;
  query.load_anywhere(q + (int64_t)t * q_stride + (int64_t)head * head_dim + lane_dim);
  const int pos = tok_pos[t];
  const int* table = tables + (int64_t)(direct ? t : tok_item[t]) * table_width;
  read_arguments(pos, k_pool, v_pool, kv_heads, page_size, num_pages, scale_log2, window, extra.sink, extra.gate,
                 extra.logistic, extra.softcap);
  const int kv_head = kv_group == 1 ? head : head / kv_group;

  const int first_key = first_visible_key(pos, window);
  const int first_load = even ? first_key & ~(GROUPS - 1) : first_key;
  const int end_key = pos + 1;
  int range_begin = first_load, range_end = end_key;
  if (splits > 1) {
    int chunk = (end_key - first_load + splits - 1) / splits;
    chunk = (chunk + KEYS_PER_WAVE - 1) / KEYS_PER_WAVE * KEYS_PER_WAVE;
    range_begin = first_load + split * chunk;
    range_end = range_begin + chunk < end_key ? range_begin + chunk : end_key;
  }
  // (keys beyond the block table have no page)
  if (even && range_end > (int64_t)table_width << page_shift) range_end = table_width << page_shift;

  float m = -INFINITY, l = 0.f;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  Raw8<T> kr[AD_UNROLL], vr[AD_UNROLL];
  bool valid[AD_UNROLL];
  const bool logistic = extra.logistic != nullptr;
  float shift = 0.f, gate = 0.f;

  // Every load of a turn is unconditional from an address that exists and masked afterwards, so that the
  // table entries, then all keys and values of the turn, travel together.
  const unsigned page_values = (unsigned)kv_heads * page_size * head_dim;
  const unsigned head_values = (unsigned)kv_head * page_size * head_dim;
  const unsigned lane_bytes = (unsigned)(group * head_dim + lane_dim) * sizeof(T);
  auto load_even = [&](int base) {
    const int first = base >> page_shift, last = (range_end - 1) >> page_shift;
    const bool exists = (unsigned)held < (unsigned)num_pages;
    const uint64_t place = ((uint64_t)(exists ? (unsigned)held : 0u) * page_values + head_values) * sizeof(T);
    const uint64_t k_place = (uint64_t)k_pool + place, v_place = (uint64_t)v_pool + place;
    const int visible_end = exists ? range_end : 0;
    int ends[AD_UNROLL];
#pragma unroll
    for (int u = 0; u < AD_UNROLL; ++u) {
      const int key = base + u * GROUPS;
      // a load beyond the range stays in its last page
      const int logical = key >> page_shift;
      const int from = (logical < last ? logical : last) - first;
      const unsigned bytes = lane_bytes + (unsigned)((key & (page_size - 1)) * head_dim) * sizeof(T);
      kr[u].template load<NT>((const T*)(const char*)(read_address(k_place, from) + bytes));
      vr[u].template load<NT>((const T*)(const char*)(read_address(v_place, from) + bytes));
      ends[u] = __builtin_amdgcn_readlane(visible_end, from);
    }
#pragma unroll
    for (int u = 0; u < AD_UNROLL; ++u) {
      const int key = base + u * GROUPS + group;
      valid[u] = (key >= first_key) & (key < ends[u]);
    }
    if (base + AD_WAVES * KEYS_PER_WAVE < range_end) ask_entries(table, base + AD_WAVES * KEYS_PER_WAVE);
  };
  auto load_general = [&](int base) {
    int page[AD_UNROLL], within[AD_UNROLL];
#pragma unroll
    for (int u = 0; u < AD_UNROLL; ++u) {
      const int key = base + u * GROUPS + group;
      const int safe_key = key < range_end ? key : range_end - 1;
      const int logical = page_shift >= 0 ? (safe_key >> page_shift) : safe_key / page_size;
      within[u] = safe_key - logical * page_size;
      const int entry = logical < table_width ? logical : table_width - 1;
      if (prefetched) {
        const int low = __shfl(held, entry & 63, 64);
        page[u] = low;
        if (table_width > 64) {
          const int high = __shfl(held1, entry & 63, 64);
          page[u] = entry < 64 ? low : high;
        }
      } else {
        page[u] = table[entry];
      }
      valid[u] = key < range_end && logical < table_width;
    }
#pragma unroll
    for (int u = 0; u < AD_UNROLL; ++u) {
      valid[u] = valid[u] && page[u] >= 0 && page[u] < num_pages;
      const int safe_page = valid[u] ? page[u] : 0;
      const int64_t offset =
          (((int64_t)safe_page * kv_heads + kv_head) * page_size + within[u]) * head_dim + lane_dim;
      kr[u].template load<NT>(k_pool + offset);
      vr[u].template load<NT>(v_pool + offset);
    }
  };
  // A masked key was loaded from another key's place and may hold anything, also NaN.  (bfloat16 values are masked four
  // registers at a time in front of the sum, float sums behind it, which needs no register more.)
  auto add_values = [&](int u, float p) {
    float vf[8];
    if constexpr (sizeof(T) == 2) vr[u].widen_if(valid[u], vf);
    else vr[u].widen(vf);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float sum = fmaf(p, vf[i], acc[i]);
      acc[i] = sizeof(T) == 2 || valid[u] ? sum : acc[i];
    }
  };
  auto weigh = [&]() {
    float s[AD_UNROLL];
    float m_new = m;
#pragma unroll
    for (int u = 0; u < AD_UNROLL; ++u) {
      float dot = kr[u].dot(query);
      if (!has_dims) dot = 0.f;
      if (LPK <= 16) {
        dot = lanes_sum<(LPK <= 16 ? LPK : 16)>(dot);
      } else {
        dot = lanes_sum<16>(dot);
        dot += __shfl_xor(dot, 16, 64);
      }
      float score = dot * scale_log2;
      // (the cap in the scores' units of log 2)
      if (extra.softcap > 0.f) score = capped_score_as<T>(score, extra.softcap * 1.4426950408889634f);
      s[u] = valid[u] ? score : -INFINITY;
      m_new = fmaxf(m_new, s[u]);
    }
    if (logistic) {
#pragma unroll
      for (int u = 0; u < AD_UNROLL; ++u) {
        const float p = valid[u] ? logistic_weight_as<T>(s[u] + shift) : 0.f;
        add_values(u, p);
      }
    } else if (m_new != -INFINITY) {
      const float correction = (m == -INFINITY) ? 0.f : exp2_fast<T>(m - m_new);
      l *= correction;
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] *= correction;
#pragma unroll
      for (int u = 0; u < AD_UNROLL; ++u) {
        // (a masked key's score is minus infinity, and m_new is none)
        const float p = exp2_fast<T>(s[u] - m_new);
        l += p;
        add_values(u, p);
      }
      m = m_new;
    }
  };
  // behind the loads of the first turn: what the sums start from
  auto start = [&]() {
    if (extra.gate != nullptr) gate = extra.gate[(int64_t)t * extra.gate_ld + head];
    if (extra.sink != nullptr && split == 0 && wave == 0 && group == 0) {
      // a score without key or value (not scaled): it starts the denominator of one lane group
      m = extra.sink[head] * 1.4426950408889634f;
      l = 1.f;
    }
    if (logistic) {
      shift = extra.logistic[head] * 1.4426950408889634f;
      m = 0.f;
      if (split == 0 && wave == 0 && group == 0) l = extra.logistic_norm;
    }
  };
  auto walk = [&](auto load) {
    int base = range_begin + wave * KEYS_PER_WAVE;
    if (even && !from_start) ask_entries(table, base);
    if constexpr (!std::is_same<Ahead, NothingAhead>::value) {
      // a wave without keys apart, and the first turn on its own, so that its waits know which loads are behind its own
      if (base >= range_end) {
        ahead();
        start();
        return;
      }
      load(base);
      __builtin_amdgcn_sched_barrier(0);
      ahead();
      __builtin_amdgcn_sched_barrier(0);
      start();
      weigh();
      for (base += AD_WAVES * KEYS_PER_WAVE; base < range_end; base += AD_WAVES * KEYS_PER_WAVE) {
        load(base);
        weigh();
      }
    } else {
      if (base < range_end) load(base);
      start();
      while (base < range_end) {
        weigh();
        base += AD_WAVES * KEYS_PER_WAVE;
        if (base < range_end) load(base);
      }
    }
  };
  if (even) walk(load_even);
  else walk(load_general);
  if (!has_dims) {
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = 0.f;
  }

  // merge the lane groups of this wave: every state is scaled to the wave's maximum, then
  // the sums run over the lanes that hold the same head dimensions
  {
    const float wave_m = groups_max<LPK>(m);
    const float c = (m == -INFINITY) ? 0.f : exp2_fast<T>(m - wave_m);
    l = groups_sum<LPK>(l * c);
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = groups_sum<LPK>(acc[i] * c);
    m = wave_m;
  }
  if (group == 0 && has_dims) {
    *reinterpret_cast<float4*>(&s_acc[wave][dim0]) = make_float4(acc[0], acc[1], acc[2], acc[3]);
    *reinterpret_cast<float4*>(&s_acc[wave][dim0 + 4]) = make_float4(acc[4], acc[5], acc[6], acc[7]);
  }
  if (lane == 0) *reinterpret_cast<float2*>(s_ml[wave]) = make_float2(m, l);
  __syncthreads();

  // merge the waves: one thread per head dimension.  Lane w of every wave works out the share of wave w.
  const int d = threadIdx.x;
  if (d >= 256 || wave * 64 >= head_dim) return;
  float2 ml = make_float2(-INFINITY, 0.f);
  if (lane < AD_WAVES) ml = *reinterpret_cast<const float2*>(s_ml[lane]);
  float value[AD_WAVES];
#pragma unroll
  for (int w = 0; w < AD_WAVES; ++w) value[w] = s_acc[w][d];
  // (lanes from AD_WAVES on hold nothing: the row of 16 lanes is all that counts)
  const float block_m = read_lane(lanes_max<16>(ml.x), 0);
  const float share = (ml.x == -INFINITY) ? 0.f : exp2_fast<T>(ml.x - block_m);
  const float block_l = read_lane(lanes_sum<16>(ml.y * share), 0);
  float sum = 0.f;
#pragma unroll
  for (int w = 0; w < AD_WAVES; ++w) sum += value[w] * read_lane(share, w);
  if (context != nullptr || (splits == 1 && out != nullptr)) {
    float result = sum / block_l;
    if (extra.gate != nullptr) result *= 1.0f / (1.0f + expf(-gate));
    if (d < head_dim) {
      if (context != nullptr) context[d] = from_float<T>(result);
      else out[(int64_t)t * out_stride + (int64_t)head * head_dim + d] = from_float<T>(result);
    }
  } else {
    float* dst = partial + (((int64_t)n * heads + head) * splits + split) * (head_dim + 2);
    if (d < head_dim) dst[d] = sum;
    if (d == 0) {
      dst[head_dim] = block_m;
      dst[head_dim + 1] = block_l;
    }
  }
}

// (the arguments in front of `page_size` are what the first loads need: they come with the launch)
template <typename T, int LPK, int AD_WAVES, int AD_UNROLL, bool NT>
__global__ __launch_bounds__(64 * AD_WAVES) void attention_decode_kernel(
    const int* __restrict__ tables, const int* __restrict__ tok_pos, const int* __restrict__ tok_list,
    const int* __restrict__ tok_item, const T* __restrict__ q, int64_t q_stride, int table_width, int form,
    int page_size, int heads, int kv_heads, int kv_group, int num_pages,
    const T* __restrict__ k_pool, const T* __restrict__ v_pool, T* __restrict__ out, int64_t out_stride,
    float* __restrict__ partial, float scale_log2, int window, int splits, const AttnExtras extra) {
  __shared__ DecodeLds<AD_WAVES> lds;
  attention_decode_block<T, LPK, AD_WAVES, AD_UNROLL, NT>(
      lds, blockIdx.x, blockIdx.y, blockIdx.z, q, q_stride, k_pool, v_pool, out, out_stride, partial,
      tok_list, tok_item, tok_pos, tables, table_width, heads, kv_heads, kv_group, form, page_size,
      num_pages, scale_log2, window, splits, extra);
}
