// Which kernel or schedule a call takes, as plain arithmetic on its sizes: no device code and no HIP header, so that a
// host compiler can build it by itself and the rules can be checked without a GPU.
#pragma once
#include <stdint.h>

namespace fm {

// Blocks of 256 threads, four 8-element chunks per thread, for scale_cast_rows_kernel's walk over a rows_p x cols_p matrix
// (cols_p a multiple of 8), or 0 where it does not take it: the walk's index is an int, and every thread's last step goes
// up to one grid beyond the last chunk.  Larger matrices run on scale_cast_kernel, whose blocks are 64x64 tiles.
inline int64_t scale_cast_rows_blocks(int64_t rows_p, int64_t cols_p) {
  const int64_t chunks = rows_p * (cols_p / 8), blocks = (chunks + 1023) / 1024;
  return chunks + blocks * 256 <= INT32_MAX ? blocks : 0;
}

}  // namespace fm
