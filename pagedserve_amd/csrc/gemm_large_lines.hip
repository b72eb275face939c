// The large product (gemm_large_bf16.h) in tiles of 128 x 64 to 256 x 128, whose stages hold whole cache lines.  Stages: as
// many as LDS holds (160 KB); of 128 x 64 and 128 x 128 four, which measured no slower than five or six.
#include "gemm_large_bf16.h"

int ps_gemm_nt_bf16_large_lines(PS_LARGE_ARGUMENTS) {
  switch (shape) {
    case 11: return PS_LARGE(1, 1, 128, 4, 4);
    case 12: return PS_LARGE(1, 2, 128, 4, 4);
    case 13: return PS_LARGE(1, 3, 128, 4, 4);
    case 22: return PS_LARGE(2, 2, 128, 3, 4);
  }
  ps_set_error("ps_linear: the large product has no tiles of number %d", shape);
  return 1;
}
