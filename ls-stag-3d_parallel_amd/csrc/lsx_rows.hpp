// Rows of a reduction's blocks and threads.
#pragma once

#include <hip/hip_runtime.h>

namespace lsx {

// block b of nb takes rows [lo, hi) of n
__host__ __device__ inline void chunk_of(long n, int b, int nb, long* lo, long* hi) {
  const long per = (n + nb - 1) / nb;
  *lo = per * b;
  long h = *lo + per;
  *hi = h < n ? h : n;
}

// row i + k, or row i itself past the chunk's end: what a thread whose row i lies in the chunk may read
// ahead, since no other thread writes it
__host__ __device__ inline long row_ahead(long i, long k, long hi) { return i + k < hi ? i + k : i; }

}  // namespace lsx
