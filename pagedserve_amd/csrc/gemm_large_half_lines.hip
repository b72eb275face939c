// The large product (gemm_large_bf16.h) in tiles of 256 x 128 to 256 x 320, whose stages hold half a cache line of every row.
// Stages: as many as LDS holds (160 KB) less one of 256 x 256, of which five fit exactly and take 1 to 3 % longer than
// four (4088 x 3840 x 1280 44.2 and 43.4 us, 2581 x 4800 x 1600 48.0 and 46.7; level at 4,096 cubed).
#include "gemm_large_bf16.h"

int ps_gemm_nt_bf16_large_half_lines(PS_LARGE_ARGUMENTS) {
  switch (shape) {
    case 2: return PS_LARGE(2, 2, 64, 6, 8);
    case 3: return PS_LARGE(2, 3, 64, 5, 8);
    case 4: return PS_LARGE(2, 4, 64, 4, 8);
    case 5: return PS_LARGE(2, 5, 64, 4, 8);
  }
  ps_set_error("ps_linear: the large product has no tiles of number %d", shape);
  return 1;
}
