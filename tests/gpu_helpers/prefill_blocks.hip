// Test helper: the routes per M block that a prefill call takes.
#include "kernels.h"

extern "C" int prefill_blocks(int fmt, int M, int k, int rows, int H, int I) {
  return ftmoe::prefill_block_size(fmt, M, k, rows, H, I);
}
