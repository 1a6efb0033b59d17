// Which bytes of an operand the unaligned vector loads of the BatchMatMul kernel touch.  An operand is stored [R, K] (k
// fastest, 16-byte loads along k) or [K, R] (r fastest, 4-byte loads along r), R being the rows or columns of the output that
// it feeds.  Plain C++: the CPU test of these offsets includes this file.
#ifndef ITEXHIP_QBMM_READS_HPP_
#define ITEXHIP_QBMM_READS_HPP_

#include <stdint.h>

#ifdef __HIP__
#define ITEXHIP_HD __host__ __device__ inline
#else
#define ITEXHIP_HD inline
#endif

namespace itexhip {

// Whether such loads find a place inside a row of the operand.  The kernel issues the first ones before it looks at K, so an
// empty reduction (whose operands may be null) must not come here.
ITEXHIP_HD bool vector_reads_fit(bool k_fastest, int64_t R, int64_t K) { return K > 0 && (k_fastest ? K >= 16 : R >= 4); }

// Byte offset of a load in the matrix.  Rows and k past the end repeat the last one; a load that would cross the end of its
// row starts at the last place inside it.
ITEXHIP_HD int64_t read_offset_k_fastest(int64_t row, int64_t k, int64_t R, int64_t K) {
  return (row < R ? row : R - 1) * K + (k < K - 16 ? k : K - 16);
}
ITEXHIP_HD int64_t read_offset_r_fastest(int64_t r, int64_t k, int64_t R, int64_t K) {
  return (k < K ? k : K - 1) * R + (r < R - 4 ? r : R - 4);
}

}  // namespace itexhip
#endif  // ITEXHIP_QBMM_READS_HPP_
