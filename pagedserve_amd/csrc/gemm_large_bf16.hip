// Which bfloat16 products the large kernel (gemm_large_bf16.h) takes, and in which tiles.  Its instances are compiled in two
// files, gemm_large_lines.hip and gemm_large_half_lines.hip: the driver loads the code of a file when its first kernel is
// launched.
#include "gemm_large_bf16.h"

// The tiles by number: 10 x the fragments of a wave along m + those along n (12: 128 x 128); 2 to 5 are 256 x 128 to
// 256 x 320 in rows of 64 bytes.
static int tile_rows(int shape) { return 32 * GL_WAVES_M * (shape < 20 && shape > 9 ? 1 : 2); }
static int tile_columns(int shape) { return 32 * GL_WAVES_N * (shape % 10); }

// Tiles of up to 256 x 128, for a product that they cover in one round of blocks: the smallest of them that does, as a
// unit without a block does nothing and a second round takes as long as the first.  What 64 x 64 tiles cover in one
// round is left to them (1000 x 1024 x 1024 9.0 us, in 128 x 64 9.6; 300 x 3072 x 768 7.2 and 8.1).  In us, former kernel
// and this one: in 128 x 64 tiles 544 x 3072 x 1024 11.7 and 9.9, 300 x 4096 x 1024 11.5 and 10.0, 2048 x 1024 x 4096 33.5
// and 29.2; 128 x 128 1000 x 3072 x 768 13.3 and 11.9, 640 x 4096 x 1024 15.5 and 14.5, 2048 x 1600 x 6400 68 and 63, 2800
// x 768 x 3072 46 and 31; 128 x 192 2048 x 3072 x 1024 22.8 and 20.0, 2048 x 2304 x 768 16.7 and 14.5; 256 x 128 2048 x 4096
// x 1024 27.7 and 24.7, 8192 x 768 x 3072 53 and 46, 4096 x 1600 x 6400 116 and 95.
// 128 x 64 on few of the units are behind two blocks of 64 x 64 on each: on 132 of them 1400 x 768 x 3072 takes 18.6 us
// there and 20.5 here, on 144 330 x 3072 x 768 is level, on 180 544 x 2304 x 768 takes 8.3 and 7.9.  A residual product
// reads the rows that it adds to behind its last product, which two blocks hide from each other: on 192 units 2048 x 768 x
// 3072 takes 21.8 there and 22.7 here.  With k under 768 the ends of a tile take longer than its products (600 x 4096 x 512
// 8.9 there, 9.3 here).  Nor do larger tiles pay that lie half behind the product's ends: 259 x 6144 x 768 is 0.38 of what
// 256 tiles of 128 x 128 hold and takes 12.1 us in them, 11.0 in 64 x 64 (544 x 4096 x 1024, 0.53, 13.6 and 14.9).
static int medium_shape(int m, int n, int k, int epilogue) {
  if (m <= 128 || k < 768 || k % 64 != 0) return 0;
  const int units = ps_compute_units();
  if ((int64_t)((m + 63) / 64) * ((n + 63) / 64) <= units) return 0;
  static const int shapes[] = {11, 12, 13, 22};
  for (int shape : shapes) {
    const int rows = tile_rows(shape), columns = tile_columns(shape);
    const int64_t tiles = (int64_t)((m + rows - 1) / rows) * ((n + columns - 1) / columns);
    if (tiles > units) continue;
    if (shape != 11 && 100 * (int64_t)m * n < 45 * (int64_t)units * rows * columns) return 0;
    return shape == 11 && 8 * tiles <= (epilogue == PS_EPI_RESIDUAL ? 6 : 5) * units ? 0 : shape;
  }
  return 0;
}

// Which width (FN) a product of several rounds or of wider tiles takes, 0: not this kernel.  A block has its compute
// unit to itself, so that time goes in rounds: `share` is the part of the rounds' outputs that the product needs.  At a
// full chip a tile's outputs per time stand as 0.85, 0.87, 0.95 and 1 for FN of 2 to 5 (0.70 for FN = 2 in rows of 64
// bytes).  Against the other kernels the line lies at 0.6 of a full chip of the widest tiles: 2048 x 4800 x 1600
// (0.68) 44 us where they take 50, 4096 x 3072 x 768 (0.87) 31 and 39.  Short products are left to them: with k
// under 768 the ends of a tile take longer than its products.
static int large_width(int m, int n, int k) {
  const float rate[] = {0.f, 0.f, k % 64 == 0 ? 0.85f : 0.70f, 0.87f, 0.95f, 1.f};
  if (m < 1024 || n < 256 || k < 768) return 0;
  const int units = ps_compute_units();
  const int64_t tiles_m = (m + 255) / 256;
  int best = 0;
  float best_value = 0.6f;
  for (int width = 2; width <= 5; ++width) {
    const int bn = tile_columns(width);
    const int64_t tiles = tiles_m * ((n + bn - 1) / bn);
    const int64_t rounds = (tiles + units - 1) / units;
    const float share = (float)m * (float)n / ((float)(rounds * units) * 256 * bn);
    if (share * rate[width] > best_value) {
      best_value = share * rate[width];
      best = width;
    }
  }
  return best == 2 && k % 64 == 0 ? 22 : best;
}

// Outputs that the unit with the most tiles makes where the other kernels take the product (gemm_mfma.hip asks this one
// first): the wide one's blocks of 64 x 256, or tiles of 128 x 64 or 64 x 64.
static int64_t fullest_elsewhere(int m, int n, bool wide) {
  const int units = ps_compute_units();
  const int64_t tiles_128 = (int64_t)((m + 127) / 128) * ((n + 63) / 64);
  const int rows = !wide && 2 * tiles_128 >= 3 * units ? 128 : 64;
  const int columns = wide ? 256 : 64;
  const int64_t tiles = (int64_t)((m + rows - 1) / rows) * ((n + columns - 1) / columns);
  return (tiles + units - 1) / units * rows * columns;
}

// Which tiles a product takes, 0: not this kernel.  `wide`: the wide kernel would take it otherwise.
//
// Not where the fullest unit makes one and a half times the outputs that it would make elsewhere.  Of 350 products of 113
// to 4,116 rows those with a ratio of up to 1.33 take 0.57 to 0.998 of the other kernel's time with bfloat16 outputs or
// as residual (one with 1.2 1.02).  Beyond, one block of 64 x 256 per unit is ahead at any k (1300 x 3072 x 1024 14.5 us
// there and 15.7 here, x 2048 22.9 and 24.0, x 4096 level), two blocks of 64 x 64 up to a k of 1,600 (1294 x 1536 x 768 9.2
// and 9.8, as residual 9.7 and 11.2, x 1600 14.4 and 14.1, 15.0 and 16.0; x 2048 18.2 and 16.8, 18.3 and 18.7; 1568 x 1280 x
// 5120 40.5 and 35.9, 41.5 and 38.0).
//
// Float outputs that are not added to what is there are twice the bytes at the end of a tile, which blocks that
// share a unit hide from each other.  With k up to 1,024 they leave nothing to gain at 128 x 64 (515 x 3072 x 1024
// 10.5 there and 11.2 here, 26 products 0.98 to 1.07; k = 1280 0.90 to 0.93), at a ratio of 1.33 (0.97 to 1.02; k =
// 1280 0.87 to 0.93) and, against the wide kernel, at 256 x 128 and 256 x 192 where more than 6 % of the tiles lie behind the
// product's ends (785 x 8192 x 1024 24.0 and 27.0, 2596 x 4096 x 1024 35.8 and 38.2; with less 3292 x 3072 x 1024 37.7 and
// 34.4, 2048 x 4096 x 1024 28.5 and 27.0).
static int shape_for(int m, int n, int k, int c_dtype, int epilogue, bool wide) {
  const int medium = medium_shape(m, n, k, epilogue);
  const int shape = medium != 0 ? medium : large_width(m, n, k);
  if (shape == 0) return 0;
  const int rows = tile_rows(shape), columns = tile_columns(shape);
  const int units = ps_compute_units();
  const int64_t tiles = (int64_t)((m + rows - 1) / rows) * ((n + columns - 1) / columns);
  const int64_t here = (tiles + units - 1) / units * rows * columns, there = fullest_elsewhere(m, n, wide);
  if (2 * here >= 3 * there && (wide || k < 2048)) return 0;
  if (c_dtype == PS_F32 && epilogue != PS_EPI_RESIDUAL && k <= 1024) {
    const bool padded = 100 * (int64_t)m * n < 94 * tiles * rows * columns;
    if (shape == 11 || 10 * here > 13 * there || (wide && padded && (shape == 22 || shape == 3))) return 0;
  }
  return shape;
}

// (k a multiple of 32 for whole stages; a tile's rows lie within 32-bit offsets)
static bool large_takes(const void* a, const void* w, int m, int n, int k, int lda) {
  return m > 0 && n > 0 && k >= 8 * 32 && k % 32 == 0 && lda >= k && lda % 8 == 0 && lda <= (1 << 22) &&
         (reinterpret_cast<uintptr_t>(a) & 15u) == 0 && (reinterpret_cast<uintptr_t>(w) & 15u) == 0;
}

bool ps_gemm_nt_bf16_large_operands(const void* a, const void* w, int m, int n, int k, int lda) {
  return large_takes(a, w, m, n, k, lda);
}

int ps_gemm_nt_bf16_large_shape(const void* a, const void* w, int m, int n, int k, int lda, int c_dtype, int epilogue,
                                bool wide) {
  return large_takes(a, w, m, n, k, lda) ? shape_for(m, n, k, c_dtype, epilogue, wide) : 0;
}

// shape: a tile's number.
int ps_gemm_nt_bf16_large(PS_LARGE_ARGUMENTS) {
  return (shape > 9 ? ps_gemm_nt_bf16_large_lines : ps_gemm_nt_bf16_large_half_lines)(
      a, w, bias, c, m, n, k, lda, ldc, c_dtype, epilogue, scatter, shape, s);
}

// The large product on its own, for tests and measurements of its tile shapes.
extern "C" int ps_gemm_nt_large(const void* a, const void* w, const float* bias, void* c, int m, int n, int k,
                                int lda, int ldc, int c_dtype, int epilogue, int tile, void* stream) {
  PS_REQUIRE(a && w && c && large_takes(a, w, m, n, k, lda) && ldc >= n,
             "ps_gemm_nt_large: bad sizes or unaligned operand (m %d, n %d, k %d, lda %d, ldc %d)", m, n, k, lda, ldc);
  PS_REQUIRE(c_dtype == PS_F32 || c_dtype == PS_BF16, "ps_gemm_nt_large: unknown output dtype");
  PS_REQUIRE(epilogue != PS_EPI_RESIDUAL || c_dtype == PS_F32,
             "ps_gemm_nt_large: the residual epilogue needs a float output");
  KvScatter none = {};
  return ps_gemm_nt_bf16_large(a, w, bias, c, m, n, k, lda, ldc, c_dtype, epilogue, none, tile, (hipStream_t)stream);
}
