// The decode kernel's direct copies into LDS (decode.hip): four waves copy q
// and the new row at once, each copy writing decode_copy_bytes whatever is
// left of its source. For every head layout the kernel takes, no copy of q may
// reach the new row, and none of the new row the RoPE table, which is built
// while the copies are in flight.
#include "decode_lds.hpp"

#include "check.hpp"

#include <initializer_list>

int main() {
    for (std::uint32_t hd = 8; hd <= 256; hd += 8) {
        for (std::uint32_t group = 1; group <= 16; ++group) {
            const std::uint32_t new_at = syn::q_lds_bytes(group, hd);
            const std::uint32_t rope_at = syn::rope_lds_offset(group, hd);
            bool q_stays = true, new_stays = true;
            for (const std::uint32_t element : {2u, 4u}) {
                for (std::uint32_t c = 0; c < group * hd * element; c += syn::decode_copy_bytes) {
                    q_stays = q_stays && c + syn::decode_copy_bytes <= new_at;
                }
                for (std::uint32_t c = 0; c < 2 * hd * element; c += syn::decode_copy_bytes) {
                    new_stays = new_stays && new_at + c + syn::decode_copy_bytes <= rope_at;
                }
            }
            CHECK(q_stays);
            CHECK(new_stays);
            CHECK(new_at % 16 == 0 && rope_at % 16 == 0);
            CHECK(rope_at + 4 * hd + syn::decode_copy_bytes + 4 * (hd / 2) <= syn::decode_lds_bytes(group, hd));
            CHECK(syn::decode_lds_bytes(group, hd) <= 160 * 1024);
        }
    }
    CHECK_DONE();
}
