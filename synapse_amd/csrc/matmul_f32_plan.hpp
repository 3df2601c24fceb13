// matmul_f32_plan.hpp — which kernel a product with F32 weights takes and how
// many blocks it launches (matmul_f32.hip), apart so that a CPU test can walk
// the rule's edges.
#pragma once

#include <cstdint>

namespace syn {

// A launch takes fewer than 2^32 threads in one dimension; all blocks here
// are 256 threads.
constexpr uint64_t matmul_f32_max_blocks = uint64_t{1} << 24;

struct matmul_f32_plan {
    uint32_t bm = 0;        // activation and weight rows of a tile of the matrix-core kernel;
    uint32_t bn = 0;        //   0: one wave per weight row
    uint32_t blocks_x = 0;  // 0: no launch holds the product
    uint32_t blocks_y = 0;
};

// The matrix-core kernel's time for few rows is its stages' latency (6 ns per
// column), the other's grows with n rows cols (0.15 us per million): they
// meet at n rows = 40000. us per call, one wave per weight row against
// tiles: 768 x 3072 weights 12.9 / 23.4 at 32 rows, 23.5 / 23.5 at 64; 3072 x
// 768 5.8 / 7.6 at 8 and 9.4 / 8.0 at 16; 1152 x 588 7.4 / 8.1 at 32, 12.6 /
// 8.1 at 64; 1024 x 1024 20.9 / 10.6 at 128. Fewer than 8 rows would leave
// three quarters of a tile empty.
// The tiled kernel copies whole 16-byte chunks of a row, through 32-bit
// offsets below 2^31 over a tile's 64 rows.
constexpr bool matmul_f32_on_matrix_cores(uint32_t n, uint32_t rows, uint32_t cols) {
    return n >= 8 && uint64_t{n} * rows >= 40000 && cols % 4 == 0 && cols < (uint32_t{1} << 23);
}

constexpr matmul_f32_plan plan_matmul_f32(uint32_t n, uint32_t rows, uint32_t cols) {
    const auto tiles = [&](uint32_t bm, uint32_t bn) {
        return ((uint64_t{n} + bm - 1) / bm) * ((uint64_t{rows} + bn - 1) / bn);
    };
    if (matmul_f32_on_matrix_cores(n, rows, cols)) {
        // The largest tile whose count still fills the 256 CUs (the waves
        // then split the columns). us per call for 64 x 64, 32 x 64 and
        // 32 x 32 tiles: 1024 rows of 3072 x 768 46.6, 50.6, 64.7 (768 tiles
        // of 64 x 64); 512 rows 32.5, 26.5, 33.5 (384 and 768); 729 rows of
        // 768 x 3072 71.7, 62.6, 54.5 (144, 276, 552); 257 rows of 768 x 768
        // 21.0, 13.0, 8.8.
        const uint32_t bm = tiles(64, 64) >= 512 ? 64 : 32;
        const uint32_t bn = bm == 64 || tiles(32, 64) >= 384 ? 64 : 32;
        if (tiles(bm, bn) < matmul_f32_max_blocks) {
            return {bm, bn, static_cast<uint32_t>(tiles(bm, bn)), 1};
        }
    }
    // One row's bytes, and a trip of the loop past them, within 32 bits.
    const uint64_t blocks = (uint64_t{rows} + 3) / 4;
    if (blocks >= matmul_f32_max_blocks || cols >= (uint32_t{1} << 29)) {
        return {};
    }
    const uint32_t nr = n >= 4 ? 4 : (n >= 2 ? 2 : 1);
    return {0, 0, static_cast<uint32_t>(blocks), (n + nr - 1) / nr};
}

}  // namespace syn
