// lq_extent.h -- the byte range a strided operand owns.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define LQ_HD __host__ __device__
#else
#define LQ_HD
#endif

namespace lq {

// Bytes from the start of a row-major operand to the end of its last row: rows of `width` bytes, `ld`
// apart.  The last row ends at its width, not at its leading dimension: an operand that is a column
// slice of a wider matrix owns nothing after it.
LQ_HD constexpr int64_t operand_bytes(int64_t rows, int64_t ld, int64_t width) {
    return rows > 0 ? (rows - 1) * ld + width : 0;
}

}  // namespace lq
