// Which softmax tensors are read through the caches, as functions that a host test compiles as well.
#pragma once
#include <stdint.h>

#ifdef __HIP__
#define MTRT_ROW_READS __host__ __device__ __forceinline__
#else
#define MTRT_ROW_READS inline
#endif

namespace mtrt_dev {

// Rows that are no whole cache lines, of 20 to 80 MiB together, go through the caches: the line that two rows share is fetched once, and what an earlier
// launch has left in the Infinity Cache comes from there.  Whole lines gain from the second alone, and a launch that has just made x, or memory, is the more
// common place for it to come from.  us, past and through, (rows, columns): three tensors in turn; each from memory; with a launch that makes x in front and one
// that reads y behind, all three.  No whole lines: f16 (17476, 1500) 19.8, 17.2; 20.7, 20.8; 64.2, 62.2; (8735, 3001) 21.3, 17.8; 22.3, 22.4; 64.7, 61.8; bf16
// (4368, 9001) 32.9, 26.3; 33.6, 34.1; 88.5, 84.4; f32 (12750, 1028) 19.5, 16.6; 20.3, 20.0; 58.1, 56.7; half lines (6553, 2000) 18.9, 16.4; 19.8, 20.3; 56.5, 57.0.
// Whole lines: f16 (25600, 1024) 17.7, 16.1; 18.7, 19.5; 54.7, 56.8; (4096, 4096) 11.4, 10.8; 12.8, 13.4; 37.1, 39.3; f32 (12800, 1024) 18.0, 16.5; 19.1, 19.7;
// 53.6, 56.7; (3268, 6016) 26.7, 23.4; 27.7, 28.8; 79.2, 80.6.  Smaller tensors of either kind: f16 (2097, 1500) 4.6, 4.4; 5.2, 5.3; 18.6, 18.9; f32 (698, 4501) 5.2,
// 5.6; 5.8, 6.3; 18.7, 19.0; larger ones: f16 (38447, 1500) 41.2, 41.0; 42.1, 42.0; f32 (6406, 4501) 40.5, 41.0; 41.5, 42.1.
constexpr int64_t kThroughAbove = int64_t(20) << 20, kThroughUpTo = int64_t(80) << 20;
MTRT_ROW_READS bool softmax_reads_past(int64_t rows, int64_t row_bytes) {
  const int64_t bytes = rows * row_bytes;
  return row_bytes % 128 == 0 || bytes <= kThroughAbove || bytes > kThroughUpTo;
}

}  // namespace mtrt_dev
