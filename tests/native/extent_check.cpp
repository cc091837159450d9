// CPU check of the LDS-DMA copies' address range (lucid_amd/csrc/lq_extent.h): the copies of the
// int8 GEMM's stages, enumerated for operands of several strides, against the bytes the operand
// owns.  A copy is in range if its vector offset is below num_records - scalar offset, as the
// hardware compares them; it then reads 16 bytes at their sum.
// Built and run by tests/test_operand_extent.py; prints "ok" and exits 0 on success.
#include <cstdint>
#include <cstdio>
#include <cstdlib>

#include "lq_extent.h"

namespace {

constexpr int BK = 128, TILE = 128;

// Copies that read a byte the operand does not own, or miss one that the product needs.
long faults(int64_t rows, int64_t ld, int64_t K, int64_t num_records) {
    long bad = 0;
    const int64_t owned = (rows - 1) * ld + K;  // the caller's bytes
    const int64_t padded = (rows + TILE - 1) / TILE * TILE;
    for (int64_t k0 = 0; k0 < K; k0 += BK)
        for (int64_t r = 0; r < padded; ++r)
            for (int64_t c = 0; c < BK; c += 16) {
                const int64_t voff = r * ld + c;
                const bool in = (uint32_t)voff < (uint32_t)num_records - (uint32_t)k0;
                if (in && voff + k0 + 16 > owned) ++bad;
                if (!in && r < rows && k0 + c < K) ++bad;
            }
    return bad;
}

}  // namespace

int main() {
    const int64_t shapes[][3] = {{300, 272, 144}, {300, 144, 144}, {1, 16, 16},     {1, 4096, 16},  {129, 512, 368},
                                 {256, 128, 128}, {257, 384, 128}, {2100, 640, 368}, {64, 1040, 1040}};
    for (const auto& s : shapes) {
        const int64_t rows = s[0], ld = s[1], K = s[2];
        if (const long n = faults(rows, ld, K, lq::operand_bytes(rows, ld, K))) {
            std::fprintf(stderr, "rows %lld ld %lld K %lld: %ld copies out of range\n", (long long)rows, (long long)ld,
                         (long long)K, n);
            return 1;
        }
        // rows * ld bytes let the last row's copies run past its end wherever K is shorter than a stage
        if (ld > K && K % BK != 0 && faults(rows, ld, K, rows * ld) == 0) return 1;
    }
    if (lq::operand_bytes(0, 128, 64) != 0) return 1;
    std::puts("ok");
    return 0;
}
