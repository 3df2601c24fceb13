// decode_lds.hpp — the split-KV decode kernel's LDS layout (decode.hip), apart
// so that a CPU test can walk its copies.
#pragma once

#include <cstddef>
#include <cstdint>

namespace syn {

// What one wave's direct copy (load16_lds) writes, whatever it was asked to
// fetch: 16 bytes for each of 64 lanes. Lanes past the end of their source
// re-read its first bytes and write them behind it.
constexpr uint32_t decode_copy_bytes = 1024;

// In order: the group's q as given (f32 size, the larger); the new K and V row
// of one head (likewise); the (max, sum) pairs, 4 waves and the new row, 16
// heads each, then the 4 waves' parts of the new row's scores; the waves'
// unscaled outputs (head rows padded by 4 floats); a fused step's RoPE table
// (hd/2 cos, hd/2 sin), frequency factors (one copy) and the pairs' angles.
//
// q takes whole copies: another wave's tail would otherwise land on the new
// row, which wave 0 copies at the same time, and whichever came last stayed
// (seen as a wrong new K row in a process's first step, 7 heads of 64 floats).
// The new row need not: its tail lands on the pairs and the outputs, which
// nothing writes before every copy has been waited for.
constexpr uint32_t q_lds_bytes(uint32_t group, uint32_t hd) {
    return (group * hd * 4 + decode_copy_bytes - 1) / decode_copy_bytes * decode_copy_bytes;
}
constexpr uint32_t new_lds_bytes(uint32_t hd) {
    return (2 * hd * 4 + 15) / 16 * 16;
}
constexpr uint32_t decode_ml_floats = 5 * 16 * 2 + 4 * 16;
constexpr uint32_t rope_lds_offset(uint32_t group, uint32_t hd) {
    return q_lds_bytes(group, hd) + new_lds_bytes(hd) + (decode_ml_floats + 4 * group * (hd + 4)) * 4;
}
constexpr uint32_t rope_max_pairs = 128;  // head_dim <= 256, as attention's
constexpr std::size_t decode_lds_bytes(uint32_t group, uint32_t hd) {
    return rope_lds_offset(group, hd) + std::size_t{hd} * sizeof(float) + decode_copy_bytes +
           rope_max_pairs * sizeof(float);
}

}  // namespace syn
