// Byte offsets of rows that are loaded by 32-bit offsets against a window: host code as well, so that they can be checked without a GPU.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define MPA_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define MPA_HOST_DEVICE inline
#endif

namespace mpa {

// An offset beyond every window below 2 GB, with a scalar offset on top as well (which the range check leaves out).
constexpr uint32_t kNoRow = 0x80000000u;
// Whether rows of whole tiles reach 2^32 bytes.  What is left of such a row's offset can lie within the window of the rows that there are; the
// offsets of all others beyond the last are beyond the window as they are.
MPA_HOST_DEVICE bool rows_wrap(int64_t rows, int64_t tile, int64_t pitch, int64_t element) {
    return (rows + tile - 1) / tile * tile * pitch * element >= (int64_t)1 << 32;
}
// Then: row `row` of `rows`, whose offset is `at` modulo 2^32.
MPA_HOST_DEVICE uint32_t row_offset(int row, int rows, uint32_t at) { return row < rows ? at : kNoRow; }

}  // namespace mpa
