// bfloat16 matrix product of a hundred to some thousands of rows whose waves share a tile and split its k:
//   C[m, n] = epi(sum_k A[m, k] W[n, k] + b[n]),   k a multiple of 64.
//
// A lone block of such a product is bound by LDS: loads fill it at 64 bytes a cycle, reads take 128, one after the
// other.  Four waves in a square, each with a quarter of 64 x 64, read every operand twice: 250 cycles of loads and 250 of
// reads for 64 values of k, of which the products take 64.  Here each of the four waves holds sums of the whole tile and
// multiplies one of a stage's four steps of 16 values, so that every operand is read once: 3 cycles a row of the tile
// instead of 4, and tiles that are no square of squares, 32 x 96 and 64 x 96, cost their rows and no more (measured: 430
// cycles a stage for 64 x 64, 510 for 64 x 96).  At the end the four waves' sums meet in LDS, 32 rows at a time, where a
// thread takes four columns of a row and adds them in a fixed order.  (Four chains of a quarter of k: error against float64 0.64e-7
// for a k of 768, 1.7e-7 for 6,400, in one chain 1.13 and 3.6e-7.)
// Every tile of every size adds a row's products in the same order, so that equal rows of a product give equal bits wherever they
// lie.  Blocks of an XCD that begin their k 256 bytes apart, round and round, ask for fewer rows of one channel at a time, but
// lose that: 667 products took 1.002 of the time on average (256 x 5120 x 1280 11.2 us and 12.2, 1024 x 1280 x 5120 29.7 and 32.5, but
// 1024 x 1024 x 4096 16.3 and 15.5); begun by the tile's column, which would keep it, 1.003 of what k from its start takes.
// Between the other launches of a pass, whose rows have just been written, it costs more: 512 rows of GPT-2 small 8.4 us for the
// mean of the two products added to rows and 9.6 for QKV, begun apart 7.5 and 8.9, by the column 8.4 and 9.6 in either order of
// tiles: what helps is that rows of tiles begin apart.
//
// With one block to a unit nothing hides its ends, so they are straight code: C and bias are buffers (what lies outside reads
// as zero and is not written), and what cannot go in pieces of four columns takes another branch in a loop of its own.
// With branches and single values beside every piece a tile of 64 x 160 spent 1.7 us more in them, in skipped code.
//
// Stages hold 64 values of k of every row, four to six in a ring, which two blocks of a unit have room for, in the order of
// gemm_tiled.hip (piece c of row r in slot c ^ ((r >> 1) & 7)).  A stage meets the other
// waves once: everyone has then read it and the next one has landed; its products run with the next stage's reads and the
// loads of the stage that takes its place between them.
//
// With weights from memory, the kernels that took these products before and this one, us: 2048 x 768 x 3072 added to rows
// 22.7 / 16.9, 2048 x 768 x 768 8.7 / 7.1, 544 x 1024 x 1024 7.3 / 5.3, 544 x 1024 x 4096 18.9 / 17.0, 800 x 1600 x 6400
// 51 / 36, 256 x 768 x 3072 11.7 / 8.2, 160 x 1024 x 4096 13.7 / 9.8; 256 x 2304 x 768 6.1 / 4.9, 544 x 2304 x 768 6.9 /
// 6.1, 256 x 4800 x 1600 16.5 / 11.5.  Between other kernels the gain is less (prefill of 2 x 1,024, GPT-2 small, a pair of products
// added to rows 30.2 to 26.1 us): requests beside prompt portions (GPT-2 medium) 78.8 to 77.2 ms, that prefill 808 to 804 us.
#include <type_traits>

#include "common.h"
#include "linear.h"
#include "pagedserve_hip.h"

#include "gemm_tile.h"

#define KW_WAVES 4       // one per step of 16 values of k of a stage

typedef __attribute__((__vector_size__(2 * sizeof(uint32_t)))) uint32_t u32x2_t;

template <int I, int N, typename F>
__device__ __forceinline__ void kw_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    kw_for<I + 1, N>(f);
  }
}

template <int PENDING>
__device__ __forceinline__ void kw_wait_and_sync() {
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(PENDING) : "memory");
}

#if defined(__HIP_DEVICE_COMPILE__)
// `rows` rows of k values as a buffer: no load reaches beyond them
__device__ __forceinline__ __amdgpu_buffer_rsrc_t kw_operand(const bf16_t* first, int rows, int stride, int k) {
  const uint32_t bytes = ((uint32_t)(rows - 1) * (uint32_t)stride + (uint32_t)k) * 2u;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(first), 0, (int)bytes, 0x00027000);
}
#endif

// By assembly, as in gemm_tiled.hip: the step that uses the operands waits first, and touches each of them behind the wait.
template <int OFFSET>
__device__ __forceinline__ void kw_read(u32x4_t& to, uint32_t address) {
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(to) : "v"(address), "n"(OFFSET) : "memory");
}

// Tiles of 32 FM x 32 FN.  `form`: bit 0, tiles run along the rows of C; above it the number of ranges of `range` values
// of k, whose sums are added to C by atomics where there are several (with the residual epilogue only).
template <int FM, int FN, int RING, typename TOut, int EPI>
__global__ __launch_bounds__(64 * KW_WAVES, 2) void gemm_nt_k_waves_kernel(
    const bf16_t* __restrict__ a, const bf16_t* __restrict__ w, int m, int n, int k, int lda, int ldc, int form,
    TOut* __restrict__ c, const float* __restrict__ bias, int range, KvScatter scatter) {
#if defined(__HIP_DEVICE_COMPILE__)      // (the host's pass knows no buffer resources)
  constexpr int BM = 32 * FM, BN = 32 * FN;
  constexpr int STAGE_BYTES = (BM + BN) * TB_ROW;
  constexpr int LOADS = FM + FN, READS = FM + FN, PRODUCTS = FM * FN;      // of a wave and stage
  constexpr int STRIDE = BN + 4;                                           // floats of a row that waves meet in
  constexpr bool PLAIN = EPI == PS_EPI_NONE, RESIDUAL = EPI == PS_EPI_RESIDUAL;
  static_assert(RING >= 3 && RING * LOADS < 64, "the load counter has six bits");
  static_assert(KW_WAVES * 32 * STRIDE * 4 <= RING * STAGE_BYTES, "the sums meet where the stages lay");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[RING * STAGE_BYTES];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // every XCD works on a contiguous run of tiles, along the rows of C or down its columns (see gemm_tiled.hip)
  const bool row_major = form & 1;
  const int ranges = form >> 1;
  const int tiles_m = (m + BM - 1) / BM, tiles_n = (n + BN - 1) / BN;
  const int per_xcd = tiles_m * tiles_n * ranges / 8;
  int tile = blockIdx.x;
  if (blockIdx.x < per_xcd * 8) tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  int k_begin = 0, stages = k / TB_BK;
  if constexpr (RESIDUAL) {
    const int which = tile / (tiles_m * tiles_n);
    tile -= which * tiles_m * tiles_n;
    k_begin = which * range;
    stages = min(range, k - k_begin) / TB_BK;
    if (which > 0) bias = nullptr;
  }
  const int line = row_major ? tiles_n : tiles_m;
  const int outer = tile / line, inner = tile - outer * line;
  const int m0 = (row_major ? outer : inner) * BM;
  const int n0 = (row_major ? inner : outer) * BN;

  // ---- loads: lane l of an instruction fills slot l % 8 of row l / 8 of its eight rows.  Rows beyond m or n are fetched
  // from the last valid one (they feed outputs that are never stored).
  const __amdgpu_buffer_rsrc_t from_a = kw_operand(a + (int64_t)m0 * lda + k_begin, min(BM, m - m0), lda, stages * TB_BK);
  const __amdgpu_buffer_rsrc_t from_w = kw_operand(w + (int64_t)n0 * k + k_begin, min(BN, n - n0), k, stages * TB_BK);
  uint32_t offset[LOADS];
#pragma unroll
  for (int j = 0; j < LOADS; ++j) {
    const int row = (j * KW_WAVES + wave) * 8 + (lane >> 3);
    const int piece = (lane & 7) ^ ((row >> 1) & 7);
    offset[j] = (j < FM ? (uint32_t)min(row, m - 1 - m0) * (uint32_t)lda : (uint32_t)min(row - BM, n - 1 - n0) * (uint32_t)k) * 2u +
                piece * 16;
  }
  const uint32_t own = wave * 8 * TB_ROW;
  // `k_at`: bytes along the rows, `fill`: the stage in the ring
  auto load = [&](uint32_t k_at, uint32_t fill, auto which) {
    constexpr int J = decltype(which)::value;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(J < FM ? from_a : from_w, (lds_ptr_t)(lds + fill + own + J * 32 * TB_ROW), 16,
                                             offset[J], k_at, 0, 0);
  };

  f32x16 sums[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) sums[i][j][e] = 0.f;

  // ---- operands: lane l reads the 16 bytes of k piece 2 wave + l / 32 of row l % 32
  const uint32_t reads_at = (uint32_t)(uintptr_t)(lds_ptr_t)lds + (lane & 31) * TB_ROW +
                            (uint32_t)(((2 * wave + (lane >> 5)) ^ ((lane >> 1) & 7)) << 4);
  u32x4_t operands[2][READS];
  uint32_t here = 0, k_next = 0;      // the stage that is multiplied, in the ring; the stage that is asked for
  auto around = [](uint32_t at) { return at + STAGE_BYTES < RING * STAGE_BYTES ? at + STAGE_BYTES : 0u; };
  auto arrived = [](u32x4_t* of) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int r = 0; r < READS; ++r) asm volatile("" : "+v"(of[r]));   // used only behind the wait
  };
  // A stage: the products of operands[S], the reads of the next stage's operands and the loads of the stage that takes
  // this one's place between them.  LOAD: that stage exists; AHEAD: how many stages behind the next one may be on their way
  // when that one has to be there, -1: there is no next one.  TO: the operands that are read into; S itself behind the
  // products.
  auto step = [&](auto which, auto to, auto loads, auto ahead) {
    constexpr int S = decltype(which)::value, TO = decltype(to)::value, AHEAD = decltype(ahead)::value;
    constexpr bool LOAD = decltype(loads)::value, NEXT = AHEAD >= 0;
    const uint32_t next = around(here), fill = here;
    if constexpr (NEXT) kw_wait_and_sync<AHEAD * LOADS>();
    kw_for<0, PRODUCTS>([&](auto product) {
      constexpr int Q = decltype(product)::value;
      constexpr int I = Q / FN, J = Q % FN;
      // rows of the result are columns of C: a lane then holds four consecutive columns of one row
      sums[I][J] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, operands[S][FM + J]),
                                                           __builtin_bit_cast(bf16x8, operands[S][I]), sums[I][J], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (NEXT && TO != S)
        kw_for<(Q * READS * 2 / PRODUCTS < READS ? Q * READS * 2 / PRODUCTS : READS),
               ((Q + 1) * READS * 2 / PRODUCTS < READS ? (Q + 1) * READS * 2 / PRODUCTS : READS)>([&](auto index) {
          constexpr int R = decltype(index)::value;
          kw_read<R * 32 * TB_ROW>(operands[TO][R], reads_at + next);
        });
      if constexpr (LOAD)
        kw_for<Q * LOADS / PRODUCTS, (Q + 1) * LOADS / PRODUCTS>([&](auto index) { load(k_next, fill, index); });
      __builtin_amdgcn_sched_barrier(0);
    });
    // (within the stage: no read is on its way where the compiler may move the operands to other registers)
    if constexpr (NEXT && TO == S)
      kw_for<0, READS>([&](auto index) {
        constexpr int R = decltype(index)::value;
        kw_read<R * 32 * TB_ROW>(operands[TO][R], reads_at + next);
      });
    if constexpr (NEXT) arrived(operands[TO]);
    here = next;
    if constexpr (LOAD) k_next += TB_ROW;
  };
  using Yes = std::true_type;
  using No = std::false_type;
  using Even = std::integral_constant<int, 0>;
  using Odd = std::integral_constant<int, 1>;
  using Full = std::integral_constant<int, RING - 2>;

  kw_for<0, RING>([&](auto stage) {      // (the host sends no product of fewer stages)
    kw_for<0, LOADS>([&](auto index) { load(k_next, decltype(stage)::value * STAGE_BYTES, index); });
    k_next += TB_ROW;
  });
  kw_wait_and_sync<(RING - 1) * LOADS>();
  kw_for<0, READS>([&](auto index) {
    constexpr int R = decltype(index)::value;
    kw_read<R * 32 * TB_ROW>(operands[0][R], reads_at);
  });
  arrived(operands[0]);
  int left = stages - RING;
  if (left & 1) step(Even{}, Even{}, Yes{}, Full{});
  for (left >>= 1; left > 0; --left) {
    step(Even{}, Odd{}, Yes{}, Full{});
    step(Odd{}, Even{}, Yes{}, Full{});
  }

  // ---- the ends.  32 rows at a time the four waves' sums meet in LDS; thread t finishes pieces of four columns there, t +
  // 256 p, where rows can be stored in such pieces, and single values else.  What the pieces need from memory is asked for in
  // the last two stages: the rows' positions, then their pages, bias and the rows added to.  C and bias are buffers, so
  // that no piece needs a branch: what lies outside reads as zero and is not written.
  constexpr int PER_ROW = BN / 4;
  const bool pieces = ((ldc | n) & 3) == 0 && (reinterpret_cast<uintptr_t>(c) & (4 * sizeof(TOut) - 1)) == 0 &&
                      (!RESIDUAL || ranges == 1) &&
                      (!PLAIN || scatter.k_pool == nullptr || ((scatter.head_dim | scatter.q_cols | scatter.kv_cols) & 3) == 0);
  const bool paged = PLAIN && pieces && scatter.k_pool != nullptr && n0 + BN > scatter.q_cols;
  const int64_t c_rows = min(BM, m - m0);
  const __amdgpu_buffer_rsrc_t to_c = __builtin_amdgcn_make_buffer_rsrc(
      c + (int64_t)m0 * ldc + n0, 0, (int)(((c_rows - 1) * ldc + n - n0) * (int)sizeof(TOut)), 0x00027000);
  const __amdgpu_buffer_rsrc_t from_bias =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(bias), 0, bias != nullptr ? n * 4 : 0, 0x00027000);
  constexpr uint32_t OUTSIDE = 0x7ffffff0u;
  int row_in[FN], col_in[FN];
  uint32_t c_at[FN];
  constexpr int HELD = PLAIN ? FM : 1;
  int position[HELD][FN], page[HELD][FN];
  u32x4_t shift[FN], old[RESIDUAL ? FM : 1][FN];
  auto ask_rows = [&] {
    kw_for<0, FN>([&](auto index) {
      constexpr int P = decltype(index)::value;
      const int at = P * 64 * KW_WAVES + tid;
      row_in[P] = at / PER_ROW;
      col_in[P] = (at - row_in[P] * PER_ROW) * 4;
      c_at[P] = n0 + col_in[P] < n ? (uint32_t)(row_in[P] * ldc + col_in[P]) * (uint32_t)sizeof(TOut) : OUTSIDE;
    });
    if (!paged) return;
    kw_for<0, HELD * FN>([&](auto index) {
      constexpr int I = decltype(index)::value / FN, P = decltype(index)::value % FN;
      const int row = min(m0 + I * 32 + row_in[P], m - 1);
      position[I][P] = scatter.tok_pos[row];
      page[I][P] = scatter.tok_item[row];
    });
  };
  auto ask_rest = [&] {
    if (paged) {
      kw_for<0, HELD * FN>([&](auto index) {
        constexpr int I = decltype(index)::value / FN, P = decltype(index)::value % FN;
        const int logical =
            scatter.page_shift >= 0 ? position[I][P] >> scatter.page_shift : position[I][P] / scatter.page_size;
        const bool in = logical < scatter.table_width;
        page[I][P] = scatter.tables[in ? (int64_t)page[I][P] * scatter.table_width + logical : 0];
        position[I][P] = in ? position[I][P] : -1;
      });
    }
    kw_for<0, FN>([&](auto index) {
      constexpr int P = decltype(index)::value;
      shift[P] = __builtin_amdgcn_raw_buffer_load_b128(from_bias, (uint32_t)(n0 + col_in[P]) * 4u, 0, 0);
    });
    if constexpr (RESIDUAL) {
      if (pieces)
        kw_for<0, FM * FN>([&](auto index) {
          constexpr int I = decltype(index)::value / FN, P = decltype(index)::value % FN;
          old[I][P] = __builtin_amdgcn_raw_buffer_load_b128(to_c, c_at[P] + (uint32_t)(I * 32 * ldc) * 4u, 0, 0);
        });
    }
  };
  kw_for<0, RING>([&](auto index) {
    constexpr int T = decltype(index)::value;
    if constexpr (T == RING - 2) ask_rows();
    if constexpr (T == RING - 1) ask_rest();
    step(std::integral_constant<int, T & 1>{}, std::integral_constant<int, 1 - (T & 1)>{}, No{},
         std::integral_constant<int, RING - 2 - T>{});
  });

  float* const mine = reinterpret_cast<float*>(lds) + wave * 32 * STRIDE + (lane & 31) * STRIDE + (lane >> 5) * 4;
  const float* const met = reinterpret_cast<const float*>(lds);
  auto meet = [&](auto rows) {
    constexpr int I = decltype(rows)::value;
    asm volatile("s_barrier" ::: "memory");      // every wave has read what lies here
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4*>(mine + j * 32 + g * 8) =
            f32x4{sums[I][j][4 * g], sums[I][j][4 * g + 1], sums[I][j][4 * g + 2], sums[I][j][4 * g + 3]};
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  if (pieces) {
    kw_for<0, FM>([&](auto rows) {
      constexpr int I = decltype(rows)::value;
      meet(rows);
      kw_for<0, FN>([&](auto piece) {
        constexpr int P = decltype(piece)::value;
        const float* from = met + row_in[P] * STRIDE + col_in[P];
        const f32x4 part[4] = {*reinterpret_cast<const f32x4*>(from), *reinterpret_cast<const f32x4*>(from + 32 * STRIDE),
                               *reinterpret_cast<const f32x4*>(from + 64 * STRIDE),
                               *reinterpret_cast<const f32x4*>(from + 96 * STRIDE)};
        f32x4 v = (part[0] + part[1]) + (part[2] + part[3]) + __builtin_bit_cast(f32x4, shift[P]);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = finish_value<EPI, TOut>(v[e]);
        if constexpr (RESIDUAL) v += __builtin_bit_cast(f32x4, old[RESIDUAL ? I : 0][P]);
        uint32_t at = c_at[P] + (uint32_t)(I * 32 * ldc) * (uint32_t)sizeof(TOut);
        const uint2 halves = make_uint2(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]));
        if constexpr (PLAIN) {
          if (paged) {
            int64_t pool_offset = 0;
            const int col = n0 + col_in[P], row = m0 + I * 32 + row_in[P];
            TOut* pool = col < n && row < m ? kv_scatter_col<TOut>(scatter, col, &pool_offset) : nullptr;
            if (pool != nullptr && scatter.cache_only) at = OUTSIDE;
            const int held = page[PLAIN ? I : 0][P], where = position[PLAIN ? I : 0][P];
            if (pool != nullptr && where >= 0 && held >= 0 && held < scatter.num_pages) {
              TOut* out = pool + kv_page_slot(scatter, where, held) + pool_offset;
              if constexpr (sizeof(TOut) == 4) *reinterpret_cast<f32x4*>(out) = v;
              else *reinterpret_cast<uint2*>(out) = halves;
            }
          }
        }
        if constexpr (sizeof(TOut) == 4)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), to_c, at, 0, 0);
        else
          __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2_t, halves), to_c, at, 0, 0);
      });
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    });
  } else {
    kw_for<0, FM>([&](auto rows) {
      constexpr int I = decltype(rows)::value;
      meet(rows);
      // (a wave's lanes take consecutive columns)
#pragma unroll 1
      for (int p = tid; p < 32 * BN; p += 64 * KW_WAVES) {
        const int row = m0 + I * 32 + p / BN, col = n0 + p % BN;
        const float* from = met + p / BN * STRIDE + p % BN;
        float v = (from[0] + from[32 * STRIDE]) + (from[64 * STRIDE] + from[96 * STRIDE]);
        if (row >= m || col >= n) continue;
        if (bias != nullptr) v += bias[col];
        v = finish_value<EPI, TOut>(v);
        TOut* to = c + (int64_t)row * ldc + col;
        if constexpr (RESIDUAL) {
          if (ranges > 1) unsafeAtomicAdd(to, v);
          else *to += v;
        } else {
          *to = from_float<TOut>(v);
          if constexpr (PLAIN) kv_scatter_store<TOut>(scatter, row, col, v);
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    });
  }
#endif
}

// --------------------------------------------------------------------------------- host
#define PS_K_WAVES_ARGUMENTS                                                                                        \
  const void *a, const void *w, const float *bias, void *c, int m, int n, int k, int lda, int ldc, int c_dtype,     \
      int epilogue, int tile, int ranges, const KvScatter &scatter, hipStream_t s

template <int FM, int FN, int RING, typename TOut>
static int launch_k_waves(const void* a, const void* w, const float* bias, void* c, int m, int n, int k, int lda, int ldc,
                          int epilogue, int ranges, const KvScatter& scatter, hipStream_t s) {
  constexpr int BM = 32 * FM, BN = 32 * FN;
  const int tiles_m = (m + BM - 1) / BM, tiles_n = (n + BN - 1) / BN;
  const int range = (k / TB_BK + ranges - 1) / ranges * TB_BK;
  ranges = (k + range - 1) / range;
  PS_REQUIRE((k - (ranges - 1) * range) / TB_BK >= RING, "ps_linear: k of %d in %d ranges is too short for these tiles", k, ranges);
  PS_REQUIRE((int64_t)tiles_m * tiles_n * ranges < ((int64_t)1 << 30), "ps_linear: too many tiles");
  // what one XCD's run of tiles fetches into its L2, in rows of k values
  const int run = (tiles_m * tiles_n + 7) / 8;
  const int64_t rows_along = (int64_t)((run + tiles_n - 1) / tiles_n) * BM + n;
  const int64_t rows_down = (int64_t)((run + tiles_m - 1) / tiles_m) * BN + m;
  const int form = (rows_along < rows_down ? 1 : 0) + 2 * ranges;
  dim3 grid(tiles_m * tiles_n * ranges);
#define PS_LAUNCH_KW(EPI)                                                                                           \
  hipLaunchKernelGGL((gemm_nt_k_waves_kernel<FM, FN, RING, TOut, EPI>), grid, dim3(64 * KW_WAVES), 0, s,  \
                     (const bf16_t*)a, (const bf16_t*)w, m, n, k, lda, ldc, form, (TOut*)c, bias, range, scatter)
  switch (epilogue) {
    case PS_EPI_NONE: PS_LAUNCH_KW(PS_EPI_NONE); break;
    case PS_EPI_GELU_TANH: PS_LAUNCH_KW(PS_EPI_GELU_TANH); break;
    case PS_EPI_GELU_ERF: PS_LAUNCH_KW(PS_EPI_GELU_ERF); break;
    case PS_EPI_RELU2: PS_LAUNCH_KW(PS_EPI_RELU2); break;
    case PS_EPI_RESIDUAL:      // (ps_linear takes it with float outputs only)
      if constexpr (sizeof(TOut) == 4) {
        PS_LAUNCH_KW(PS_EPI_RESIDUAL);
        break;
      }
      [[fallthrough]];
    default: ps_set_error("ps_linear: unknown epilogue %d", epilogue); return 1;
  }
#undef PS_LAUNCH_KW
  PS_CHECK_LAUNCH("ps_linear(waves along k, bfloat16)");
  return 0;
}

// The tiles by number.  Microseconds, about, of a product whose blocks come to one per compute unit at most: `ends` and, for
// every stage, `alone` and as much of `beside` as units have a block.  Where k goes in several ranges, `split` and `added` for
// every million atomic additions.  Fitted to 1,400 timings with weights from memory (65 to 3,000 rows, 23 pairs of n and k;
// 8 % off in the mean): the tile and ranges that it picks take 1.005 of the fastest ones' time on average, 1.38 at most.
#define KW_TILES 4
static const struct {
  int rows, columns, stages;
  float ends, alone, beside, split, added;
} k_waves_tiles[KW_TILES] = {{32, 64, 6, 2.24f, 0.120f, 0.050f, 2.4f, 1.34f},
                             {32, 96, 5, 2.26f, 0.163f, 0.079f, 4.1f, 0.17f},
                             {64, 64, 5, 2.53f, 0.165f, 0.076f, 5.3f, 0.27f},
                             {64, 96, 4, 3.02f, 0.217f, 0.104f, 8.2f, 0.f}};

int ps_gemm_nt_k_waves_tile(PS_K_WAVES_ARGUMENTS) {
#define PS_KW(...)                                                                                                  \
  (c_dtype == PS_F32                                                                                                \
       ? launch_k_waves<__VA_ARGS__, float>(a, w, bias, c, m, n, k, lda, ldc, epilogue, ranges, scatter, s)          \
       : launch_k_waves<__VA_ARGS__, bf16_t>(a, w, bias, c, m, n, k, lda, ldc, epilogue, ranges, scatter, s))
  switch (tile) {
    case 0: return PS_KW(1, 2, 6);
    case 1: return PS_KW(1, 3, 5);
    case 2: return PS_KW(2, 2, 5);
    default: return PS_KW(2, 3, 4);
  }
#undef PS_KW
}

// (a tile's rows lie within 32-bit offsets; the longest ring wants six stages)
bool ps_gemm_nt_k_waves_takes(const void* a, const void* w, int m, int n, int k, int lda, int ldc) {
  return m > 0 && n > 0 && k % TB_BK == 0 && k >= 6 * TB_BK && k <= (1 << 22) && lda >= k && lda % 8 == 0 && lda <= (1 << 22) &&
         ldc <= (1 << 22) &&
         ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(w)) & 15u) == 0;
}

// Rows added to that the kernel for few rows would take: from how many outputs on this one is ahead.  Its blocks read k in one round
// of loads and this one's walk it, so that it is behind until the other one's blocks outnumber what the units hold at a time.
// Of 2,389 products (97 to 224 rows, 64 to 2,048 columns, k of 512 to 8,192, in pieces) 981 were more than 3 % slower here, up to
// twice as slow; of those that this rule takes 13, up to 1.08, and they take 0.79 of the time on average.  us there and here:
// 128 x 512 x 768 3.5 / 4.1, 128 x 512 x 1024 3.8 / 4.7, 160 x 64 x 5120 3.7 / 7.3, but 144 x 512 x 1024 4.9 / 4.5, 128 x 768 x 3072 8.8 / 7.2;
// 128 x 768 x 1536 5.2 / 5.7 (two ranges of 768 there, which its waves read in three steps and not four).
static bool ahead_of_few_rows(int m, int n, int k) {
  const int64_t outputs = (int64_t)m * n;
  if (k <= 576) return true;
  if (k < 2048) return outputs >= (k > 1408 && k <= 1536 ? 100000 : 70000);
  return outputs * k >= 210000000;
}

// Products that go elsewhere although their tiles come to one round: those whose rows nearly fill their tiles (rows beyond m are read
// from one address, so that what is left of a tile costs little here and much in larger tiles).
//  - 64 x 96 in an odd number of rows of tiles, more than 7/8 full, over a k of 1,024 and more where the large kernel takes 128 x
//    64: the half of a row of tiles that it wastes is cheap there too.  532 products take 0.95 of the time there, 0.88 to 1.05 (us,
//    here and there: 293 x 3840 x 1280 11.4 / 10.0, 314 x 4096 x 1024 8.9 / 8.3, 805 x 1600 x 6400 35.5 / 32.5).  Less full they are level, in
//    an even number, or over a k of up to 960, behind there (544 x 2304 x 768 6.1 / 6.9), as are nine and more rows of tiles over a k of
//    less than 3,584 (821 x 1472 x 1600 1.18 of the time) or with plain float outputs (150 products 1.04).
//  - a long k where the ring kernel is left and 257 rows and more: 64 x 64 on up to 9/16 of the units, 19/20 full, which goes in
//    pairs of 64 x 32 there (33 products of a k of more than 4,096 0.92, 0.81 to 1.02 and one 1.14: 704 x 768 x 5120 25.5 / 21.8; but plain
//    float outputs 0.99 to 1.26, up to 512 columns 1.04 to 1.35, and a k of 2,048 to 4,096 0.88 to 1.30), and 64 x 96, 49/50 full, that
//    are up to 9/8 of the units in 64 x 64 and as many on every XCD (39 products of a k of more than 3,456 0.94, 0.87 to 1.08: 1071 x
//    1024 x 6400 36.7 / 32.2; not as many on every XCD 1.09).  Three and four rows of tiles are 1.0 to 1.3 there.
// `plain_float`: float outputs that are not added to what is there.
static bool behind_elsewhere(int tile, int m, int n, int k, bool added, bool plain_float, int large_shape, int units) {
  const int rows = (m + 63) / 64;
  const int64_t tiles_64 = (int64_t)rows * ((n + 63) / 64);
  if (tile == 3 && large_shape == 11)
    return rows % 2 == 1 && 8 * m > 7 * 64 * rows && k >= (rows > 7 ? 3584 : added ? 1088 : 1024) && !(plain_float && rows > 5);
  if (large_shape != 0 || m <= 256) return false;
  if (tile == 2)
    return k > 4096 && n > 512 && !plain_float && 2 * tiles_64 > units && 16 * tiles_64 <= 9 * units && 20 * m >= 19 * 64 * rows;
  return tile == 3 && k > 3456 && 8 * tiles_64 <= 9 * units && tiles_64 % 8 == 0 && 50 * m >= 49 * 64 * rows;
}

// Which tile and number of ranges a product takes, false: not this kernel.  `few`: it would go to the kernel for few rows.
// `large_shape`: the tile that the large kernel would take it in, 0: none.
// `pieces`: rows of C in aligned pieces of four columns; in single values the ends of rows added to cost 3 us more here, which
// few rows do not make up for (100 x 321 x 768 3.8 / 8.3, 130 x 1030 x 1600 9.2 / 9.5).
//
// One round of blocks: with more than one to a unit this kernel shares LDS as the others do and has longer ends (two rounds of
// 64 x 96 at 2048 x 2304 x 768 16.5 us, 13.9 in tiles of 128 x 192).  Where only larger tiles than 64 x 96 come to one round,
// the large kernel is ahead or level (64 x 128 to 96 x 96, 120 products: 0.94 to 1.04 on average, single ones up to
// 1.28).  Of 230 products in these four tiles all but nine took less than the kernel before (0.74 to 0.88 on average): those
// nine were 65 rows added to, which the kernel for few rows takes faster (768 x 768 3.2 and 3.9 us; 100 rows level, 160
// 4.1 and 4.3), and bfloat16 rows in 64 x 96 on nearly all units (500 x 3072 x 1024 8.4 and 9.2, 1400 x 1000 x 2560 15.8 and
// 18.0; on 216 of them 544 x 2304 x 768 6.9 and 6.1).  Three rows of 64 x 96 over a k of more than 1,024 are behind, whatever
// the outputs (180 products of 130 to 192 rows 0.88 to 1.10, 1.01 on average; 180 x 6400 x 1600 11.6 and 12.6), over a shorter one
// ahead (180 products 0.89 on average), as are one or two rows of them where smaller tiles do not come to one round (192 products
// 0.82 on average, bfloat16 110 x 9600 x 1024 11.4 and 9.5).  In single values rows added
// to in 64 x 96 are behind on nearly all units too (300 x 4097 x 768 17.8 and 19.7, on 172 of them 200 rows 0.76 to 0.86).
// Ranges of k only where the kernel for few rows adds ranges by atomics too: beyond, sums keep an order that does not
// change from call to call (256 x 1024 x 4096 15.1 us, in two ranges 11.8, before 16.4).
bool ps_gemm_nt_k_waves_choice(int m, int n, int k, int c_dtype, int epilogue, bool few, bool pieces, int large_shape,
                               int* best_tile, int* best_ranges) {
  if (m <= (few ? 96 : 64) || k < 512) return false;
  if (few && !(pieces && ahead_of_few_rows(m, n, k))) return false;
  const int units = ps_compute_units(), most = few && epilogue == PS_EPI_RESIDUAL && k > 1024 ? 6 : 1;
  float least = INFINITY;
  for (int tile = 0; tile < KW_TILES; ++tile) {
    const auto& t = k_waves_tiles[tile];
    const int64_t tiles = (int64_t)((m + t.rows - 1) / t.rows) * ((n + t.columns - 1) / t.columns);
    if (tile == KW_TILES - 1 && ((c_dtype != PS_F32 && 8 * tiles > 7 * units) || (m > 2 * t.rows && m <= 3 * t.rows && k > 1024) ||
                                 (epilogue == PS_EPI_RESIDUAL && !pieces && 4 * tiles > 3 * units)))
      continue;
    for (int ranges = 1; ranges <= most && tiles * ranges <= units; ++ranges) {
      const int stages = (k / TB_BK + ranges - 1) / ranges;
      if (k / TB_BK - (ranges - 1) * stages < 8) break;
      const float time = t.ends + stages * (t.alone + t.beside * (float)(tiles * ranges) / units) +
                         (ranges > 1 ? t.split + t.added * 1e-6f * (float)m * (float)n * (float)ranges : 0.f);
      if (time < least) {
        least = time;
        *best_tile = tile;
        *best_ranges = ranges;
      }
    }
  }
  const bool added = epilogue == PS_EPI_RESIDUAL, plain_float = c_dtype == PS_F32 && !added;
  return least < INFINITY && (few || !behind_elsewhere(*best_tile, m, n, k, added, plain_float, large_shape, units));
}

// The product in a given tile and number of ranges, for tests and measurements.
extern "C" int ps_gemm_nt_k_waves(const void* a, const void* w, const float* bias, void* c, int m, int n, int k, int lda,
                                  int ldc, int c_dtype, int epilogue, int tile, int ranges, void* stream) {
  PS_REQUIRE(a && w && c && ps_gemm_nt_k_waves_takes(a, w, m, n, k, lda, ldc) && ldc >= n,
             "ps_gemm_nt_k_waves: bad sizes or unaligned operand (m %d, n %d, k %d, lda %d, ldc %d)", m, n, k, lda, ldc);
  PS_REQUIRE(c_dtype == PS_F32 || c_dtype == PS_BF16, "ps_gemm_nt_k_waves: unknown output dtype");
  PS_REQUIRE(epilogue != PS_EPI_RESIDUAL || c_dtype == PS_F32,
             "ps_gemm_nt_k_waves: the residual epilogue needs a float output");
  PS_REQUIRE(tile >= 0 && tile < KW_TILES && ranges >= 1 && (ranges == 1 || epilogue == PS_EPI_RESIDUAL),
             "ps_gemm_nt_k_waves: no tile %d in %d ranges", tile, ranges);
  KvScatter none = {};
  return ps_gemm_nt_k_waves_tile(a, w, bias, c, m, n, k, lda, ldc, c_dtype, epilogue, tile, ranges, none, (hipStream_t)stream);
}
