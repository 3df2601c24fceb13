// quant_plan.hpp — which kernel a product with quantized weights takes
// (quant.hip, quant_gemm.hip), apart so that a CPU test can walk the rule's
// edges. All figures are us per call, the activations' quantizer included.
#pragma once

#include <cstdint>

namespace syn {

// Quantized weights, ggml type numbers.
constexpr uint32_t qtype_q4_0 = 2, qtype_q5_0 = 6, qtype_q8_0 = 8, qtype_q4_k = 12, qtype_q6_k = 14;

enum class quant_kernel {
    gemv,   // passes over the weights for up to four activation rows each
    r16,    // 16 weight rows a block, up to 32 activation rows
    ks,     // 32 x 32 tiles, the columns split over the block's waves
    tiles,  // the larger tiles
};

// gemm_r16_kernel launches 32 threads per weight row, and a launch takes fewer
// than 2^32 of them (the GEMV's grid is a resident one).
constexpr uint32_t r16_max_rows = (1u << 27) - 16;

// The GEMV, where its blocks (8 weight rows, `per_pass` activation rows) are
// one per CU at most: it is one launch, and its time then hardly grows with
// the columns, while a 16-row tile's grows with the 2048-column units each of
// its waves walks (2 us each in the 32-block formats). GEMV against 16-row
// tiles, 512 weight rows: 3 rows of Q8_0, 2048 columns 6.1 / 6.7, 4096 6.5 /
// 8.0, 8192 7.1 / 10.6; Q5_0 7.6 / 7.2, 7.9 / 9.3, 8.8 / 13.0; Q4_0 8.2 / 6.7,
// 8.5 / 8.4, 9.3 / 11.5; Q6_K 6.9 / 6.9, 7.1 / 8.3, 9.5 / 10.5; Q4_K 7.1 / 6.8,
// 7.6 / 7.4, 8.3 / 9.2. 4 to 16 rows (two more passes' decode) of 8192 columns:
// Q5_0 12.1 / 13.2, Q4_0 13.3 / 11.6, Q8_0 10.2 / 10.6 (14336: 15.6 / 14.0). 31
// rows of 256 weight rows: Q8_0 4096 9.8 / 10.2, 8192 10.6 / 13.8; Q5_0 11.6 /
// 11.2, 12.6 / 16.2; Q4_0 12.6 / 10.4, 13.6 / 14.4.
constexpr bool quant_gemv_beats_r16(uint32_t t, uint32_t n, uint32_t per_pass, uint32_t rows, uint32_t cols,
                                    uint32_t cus) {
    if ((uint64_t{rows} + 7) / 8 * ((n + per_pass - 1) / per_pass) > cus) {
        return false;
    }
    const uint32_t units = (cols + 2047) / 2048;
    if (n == 3) {
        return t == qtype_q8_0 ? cols > 1024 : units >= (t == qtype_q5_0 || t == qtype_q6_k ? 2u : 3u);
    }
    if (n <= 16) {
        return units >= 4 && (t == qtype_q5_0 || (t == qtype_q8_0 && units < 6));
    }
    return t == qtype_q4_0 ? units >= 4 : (t == qtype_q5_0 || t == qtype_q8_0) && units >= 3;
}

// 32 activation rows: 16-row tiles run in rounds of one block per CU, each
// with its start; the larger tiles take a matrix of many weight rows and few
// columns in one. Both times fitted to 64 to 8192 columns of 4096 to 131072
// weight rows. Larger against 16-row tiles, 256 and 4096 columns: Q4_0 8192
// rows 11.3 / 9.6 and 73.7 / 16.2, 32768 11.5 / 24.8 and 75.8 / 52.3, 131072
// 17.1 / 87.9 and 143 / 218; Q4_K 8.7 / 8.4 and 28.7 / 13.9, 9.0 / 19.2 and
// 33.2 / 42.0, 16.2 / 63.9 and 101 / 175; Q6_K 16.9 / 8.7 and 42.5 / 15.4,
// 23.9 / 20.6 and 60.9 / 48.2, 37.9 / 69.7 and 196 / 208.
constexpr bool quant_r16_beats_tiles(uint32_t t, uint32_t rows, uint32_t cols, uint32_t cus) {
    const float c = static_cast<float>(cols);
    const float rounds = static_cast<float>((uint64_t{rows} + 16 * cus - 1) / (16 * cus));
    if (t == qtype_q4_k) {
        return 4.9f + rounds * (1.65f + 7.0e-4f * c) <= 7.3f + 5.2e-3f * c;
    }
    if (t == qtype_q6_k) {
        return 4.7f + rounds * (1.8f + 8.6e-4f * c) <= 23.0f + 2.8e-7f * static_cast<float>(rows) * c;
    }
    return 4.6f + rounds * (2.4f + 8.5e-4f * c) <= 7.5f + c / 60.0f;
}

// The columns from which 32 x 32 tiles with the columns split over the waves
// beat the larger tiles, which decode a weight for more activation rows but
// are fewer blocks (~0: never). Larger tiles against these, 64 activation
// rows: Q4_K 4096 weight rows (256 tiles) of 14336 columns 93 / 23; 14336 rows
// (896 tiles) of 1024, 2048 and 4096 columns 14.0 / 14.7, 19.2 / 18.9, 35 /
// 30; 4096 x 14336 at 256 rows (1024) 98 / 72, at 512 107 / 136. Q6_K 4096 x
// 4096 at 256 (1024) 51 / 44, at 512 67 / 81. Q4_0 14336 rows (896) of 64
// columns 9.7 / 8.9, 20480 (1280) of 192 and 256 12.3 / 10.5, 13.5 / 10.9,
// 32768 (2048) of 64, 256 and 512 9.9 / 12.3, 14.0 / 14.0, 19.0 / 17.5; Q8_0
// 12288 (768) of 64 9.3 / 8.3, with 33 rows 7.5 / 7.9, 20480 of 256 and 512
// 13.0 / 12.1, 17.0 / 14.2, 32768 of 64, 768 and 2048 9.8 / 13.8, 21 / 21.5,
// 40 / 37.5.
//
// K formats from 1024 columns on: up to three 256-blocks a row give a wave one
// block at most, and the larger tiles' one running sum is then as exact (768
// columns, error against 64 bits 5.1e-8 in those, 5.2e-8 in these; from four
// blocks on these have the smaller one).
constexpr uint32_t quant_ks_min_cols(uint32_t t, uint32_t n, uint64_t tiles) {
    if (t == qtype_q4_k || t == qtype_q6_k) {
        return tiles > 1024 ? ~0u : (t == qtype_q4_k && tiles > 768 ? 3072u : 1024u);
    }
    if (tiles > 2048) {
        return ~0u;
    }
    if (tiles <= 768) {
        return t == qtype_q8_0 && tiles > 512 && n < 64 ? 128 : 0;
    }
    if (t == qtype_q8_0 && tiles > 1792) {
        return 2048;
    }
    const uint32_t over = tiles > 1024 ? static_cast<uint32_t>(tiles - 1024) : 0;
    const uint32_t grown = t == qtype_q8_0 ? over * 4 / 3 : over / 2;
    return grown > 192 ? grown : 192;
}

// staged: the operands take the staged kernels' copies (quant_gemm.hip);
// per_pass: activation rows of a GEMV pass.
constexpr quant_kernel plan_matmul_q(uint32_t t, bool staged, uint32_t n, uint32_t per_pass, uint32_t rows,
                                     uint32_t cols, uint32_t cus) {
    // One and two rows: a GEMV pass against 16-row tiles (4096 x 14336, 14336
    // x 4096, 4096 x 4096) Q4_K 2 rows 16.8 / 12.8, 14.3 / 13.6, 7.9 / 7.9;
    // Q6_K 19.3 / 16.7, 16.5 / 17.8, 9.3 / 9.0; Q8_0 22.7 / 18.9, 16.9 / 19.5,
    // 11.0 / 9.3: which is faster hangs on the shape at two rows, the sums
    // take another order, and the GEMV keeps them.
    if (n < 3) {
        return quant_kernel::gemv;
    }
    // Up to 32: the weights are read and decoded once. At 24 rows, GEMV passes
    // against 16-row tiles: Q6_K 4096 x 14336 147 / 19, Q8_0 133 / 27.
    if (n < 32) {
        return staged && rows < r16_max_rows && !quant_gemv_beats_r16(t, n, per_pass, rows, cols, cus)
                   ? quant_kernel::r16
                   : quant_kernel::gemv;
    }
    if (!staged) {
        return quant_kernel::tiles;
    }
    if (n == 32 && rows < r16_max_rows && quant_r16_beats_tiles(t, rows, cols, cus)) {
        return quant_kernel::r16;
    }
    const uint64_t tiles = (uint64_t{rows} + 31) / 32 * ((n + 31) / 32);
    return cols >= quant_ks_min_cols(t, n, tiles) ? quant_kernel::ks : quant_kernel::tiles;
}

}  // namespace syn
