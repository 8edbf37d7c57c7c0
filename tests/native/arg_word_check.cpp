// CPU check of the words that carry a product's addresses and lengths in a
// launch's arguments (gpupi_amd/csrc/ragged.hpp): every word-aligned address
// that arg_packs accepts comes back with its length, and it refuses exactly
// those that would not.  Exit status 0 = all checks passed.
#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#include "../../gpupi_amd/csrc/ragged.hpp"

using namespace gpupi;

int main() {
    uint64_t seed = 88172645463325252ull;
    int accepted = 0, refused = 0;
    for (int i = 0; i < 200000; ++i) {
        seed ^= seed << 13, seed ^= seed >> 7, seed ^= seed << 17;
        const uint64_t address = (seed >> (seed % 61)) & ~(uint64_t)(i % 5 ? 3 : 0);
        for (const uint32_t length : {0u, 1u, 17u, 2044u, 4087u}) {
            const uint64_t w = arg_word(address, length);
            const bool kept = arg_address(w) == address && arg_length(w) == length;
            if (arg_packs(address) != (kept && (address & 3u) == 0)) {
                std::printf("address %llx length %u\n", (unsigned long long)address, length);
                return 1;
            }
        }
        ++(arg_packs(address) ? accepted : refused);
    }
    if (accepted < 1000 || refused < 1000) return 1;
    std::printf("arg words: ok\n");
    return 0;
}
