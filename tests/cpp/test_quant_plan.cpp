// The quantized product's rule (quant_plan.hpp): every kernel is given what it
// takes, launches stay in range, and the shapes of the GPU tests
// (test_gpu_quant.py, test_gpu_quant_few_rows.py) reach the kernels they are
// there for.
#include "quant_plan.hpp"

#include "check.hpp"

#include <initializer_list>

namespace {

using syn::quant_kernel;

constexpr std::uint32_t types[] = {syn::qtype_q4_0, syn::qtype_q5_0, syn::qtype_q8_0, syn::qtype_q4_k, syn::qtype_q6_k};

std::uint32_t per_pass(std::uint32_t n) {
    return n >= 4 ? 4 : n >= 2 ? 2 : 1;
}

quant_kernel plan(std::uint32_t t, std::uint32_t n, std::uint32_t rows, std::uint32_t cols, bool staged = true) {
    return syn::plan_matmul_q(t, staged, n, per_pass(n), rows, cols, 256);
}

void one(std::uint32_t t, bool staged, std::uint32_t n, std::uint32_t rows, std::uint32_t cols) {
    const quant_kernel k = plan(t, n, rows, cols, staged);
    const bool kq = t == syn::qtype_q4_k || t == syn::qtype_q6_k;
    if (n < 3) {
        CHECK(k == quant_kernel::gemv);
    } else if (!staged) {
        CHECK(k == (n < 32 ? quant_kernel::gemv : quant_kernel::tiles));
    } else if (n < 32) {
        CHECK(k == quant_kernel::gemv || k == quant_kernel::r16);
    } else {
        CHECK(k != quant_kernel::gemv);
    }
    if (k == quant_kernel::r16) {
        CHECK(n <= 32);
        CHECK((std::uint64_t{rows} + 15) / 16 * 512 < (std::uint64_t{1} << 32));
    }
    if (k == quant_kernel::ks) {
        // Tile counts are kept in 32 bits; K formats keep short rows' error.
        CHECK((std::uint64_t{rows} + 31) / 32 * ((n + 31) / 32) <= 2048);
        CHECK(!kq || cols >= 1024);
    }
}

}  // namespace

int main() {
    for (const std::uint32_t t : types) {
        for (const bool staged : {false, true}) {
            for (const std::uint32_t n : {1u, 2u, 3u, 4u, 16u, 17u, 31u, 32u, 33u, 64u, 65u, 512u, 65535u}) {
                for (const std::uint32_t cols : {64u, 256u, 768u, 1024u, 2048u, 4096u, 14336u, 119040u}) {
                    for (std::uint64_t rows = 1; rows < (std::uint64_t{1} << 32); rows *= 2) {
                        for (const int d : {rows == 1 ? 0 : -1, 0, 1}) {
                            one(t, staged, n, static_cast<std::uint32_t>(rows + static_cast<std::uint64_t>(d)), cols);
                        }
                    }
                }
            }
        }
        const bool kq = t == syn::qtype_q4_k || t == syn::qtype_q6_k;
        // test_large_tiles: past 1024 (2048) tiles of 32 x 32.
        CHECK(plan(t, kq ? 1025 : 2049, 1000, kq ? 2560 : 320) == quant_kernel::tiles);
        // test_few_rows' long rows of few weight rows: the GEMV takes 3 of them.
        CHECK(plan(t, 3, 40, 4160) == quant_kernel::gemv);
        // test_few_rows, test_gemm_at_model_size_matches_the_gemv.
        CHECK(plan(t, 16, 31, 4096) == quant_kernel::r16);
        CHECK(plan(t, 24, 65, 2048) == quant_kernel::r16);
        CHECK(plan(t, 16, 2048, 4096) == quant_kernel::r16);
        CHECK(plan(t, 128, 2048, 4096) == quant_kernel::ks);
        CHECK(plan(t, 2, 2048, 4096) == quant_kernel::gemv);
        CHECK(plan(t, 33, 9, kq ? 768 : 64) == (kq ? quant_kernel::tiles : quant_kernel::ks));
        CHECK(plan(t, 33, 20, 800, false) == quant_kernel::tiles);
        CHECK(plan(t, 3, (1u << 27) + 8, 64) == quant_kernel::gemv);
    }
    // test_tile_count_rule: each side of the columns that a tile count asks for.
    CHECK(plan(syn::qtype_q4_k, 33, 12288, 1024) == quant_kernel::ks);
    CHECK(plan(syn::qtype_q4_k, 33, 12289, 1024) == quant_kernel::tiles);
    CHECK(plan(syn::qtype_q4_k, 33, 12289, 3072) == quant_kernel::ks);
    CHECK(plan(syn::qtype_q6_k, 33, 16384, 1024) == quant_kernel::ks);
    CHECK(plan(syn::qtype_q6_k, 33, 16385, 1024) == quant_kernel::tiles);
    CHECK(plan(syn::qtype_q8_0, 33, 12288, 64) == quant_kernel::tiles);
    CHECK(plan(syn::qtype_q8_0, 64, 12288, 64) == quant_kernel::ks);
    CHECK(plan(syn::qtype_q8_0, 33, 8192, 64) == quant_kernel::ks);
    CHECK(plan(syn::qtype_q8_0, 33, 12289, 128) == quant_kernel::tiles);
    CHECK(plan(syn::qtype_q8_0, 33, 12289, 192) == quant_kernel::ks);
    CHECK(plan(syn::qtype_q4_0, 33, 12288, 64) == quant_kernel::ks);
    CHECK(plan(syn::qtype_q5_0, 33, 24576, 192) == quant_kernel::tiles);
    CHECK(plan(syn::qtype_q5_0, 33, 24576, 256) == quant_kernel::ks);
    CHECK(plan(syn::qtype_q4_0, 32, 32768, 64) == quant_kernel::tiles);
    CHECK(plan(syn::qtype_q4_k, 32, 32768, 256) == quant_kernel::tiles);
    CHECK(plan(syn::qtype_q6_k, 32, 131072, 256) == quant_kernel::tiles);
    CHECK_DONE();
}
