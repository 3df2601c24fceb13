// The F32 product's rule (matmul_f32_plan.hpp) at its edges: every launch
// stays below 2^32 threads, covers the product, and keeps the kernels' 32-bit
// offsets; products too large for the tiles keep the kernel they always had.
#include "matmul_f32_plan.hpp"

#include "check.hpp"

#include <initializer_list>

namespace {

void one(std::uint32_t n, std::uint32_t rows, std::uint32_t cols) {
    const syn::matmul_f32_plan p = syn::plan_matmul_f32(n, rows, cols);
    if (rows <= (1u << 26) - 4 && cols < (1u << 29)) {
        CHECK(p.blocks_x > 0);  // one wave per weight row always took these
    }
    if (p.blocks_x == 0) {
        return;
    }
    CHECK(std::uint64_t{p.blocks_x} * 256 < (std::uint64_t{1} << 32));
    CHECK(p.blocks_y <= 65535);
    if (p.bm != 0) {
        CHECK(p.blocks_y == 1);
        CHECK(std::uint64_t{p.blocks_x} == (std::uint64_t{n} + p.bm - 1) / p.bm * ((std::uint64_t{rows} + p.bn - 1) / p.bn));
        CHECK(64 * std::uint64_t{cols} * 4 < (std::uint64_t{1} << 31));
        CHECK(cols % 4 == 0);
    } else {
        CHECK(std::uint64_t{p.blocks_x} * 4 >= rows);
        CHECK(std::uint64_t{p.blocks_y} * (n >= 4 ? 4 : n >= 2 ? 2 : 1) >= n);
        CHECK(std::uint64_t{cols} * 4 + 4096 < (std::uint64_t{1} << 32));
    }
}

}  // namespace

int main() {
    // 64 x 64 tiles at and around 2^24 of them (256 GiB of outputs, which one card holds).
    CHECK(syn::plan_matmul_f32(65535, 1u << 20, 4).bm == 0);
    CHECK(syn::plan_matmul_f32(65535, (1u << 20) - 64, 4).bm == 64);
    for (const std::uint32_t n : {1u, 2u, 3u, 4u, 7u, 8u, 9u, 63u, 64u, 65u, 1000u, 65535u}) {
        for (const std::uint32_t cols : {1u, 4u, 63u, 64u, 768u, (1u << 23) - 4, 1u << 23, (1u << 29) - 1, 1u << 29, ~0u}) {
            for (std::uint64_t rows = 1; rows < (std::uint64_t{1} << 32); rows *= 2) {
                for (const int d : {rows == 1 ? 0 : -1, 0, 1}) {
                    one(n, static_cast<std::uint32_t>(rows + static_cast<std::uint64_t>(d)), cols);
                }
            }
        }
    }
    // The choices themselves.
    CHECK(syn::plan_matmul_f32(1024, 3072, 768).bm == 64);
    CHECK(syn::plan_matmul_f32(512, 3072, 768).bm == 32 && syn::plan_matmul_f32(512, 3072, 768).bn == 64);
    CHECK(syn::plan_matmul_f32(257, 768, 768).bm == 32 && syn::plan_matmul_f32(257, 768, 768).bn == 32);
    CHECK(syn::plan_matmul_f32(7, 1u << 20, 768).bm == 0);
    CHECK(syn::plan_matmul_f32(64, 577, 766).bm == 0);
    CHECK(syn::plan_matmul_f32(1, 1u << 26, 4).blocks_x == 0);
    CHECK_DONE();
}
