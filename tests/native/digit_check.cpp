// CPU check of the digit and run index rules (ntt_plan.hpp): digits read from
// at most two words of an operand, the words that the lanes of a run write,
// and the division of a limb index by a run's length.
#include <cstdio>
#include <random>
#include <vector>

#include "ntt_plan.hpp"

using namespace gpupi::ntt;

static int bit(const std::vector<uint32_t> &x, uint64_t i) { return i / 32 < x.size() ? x[i / 32] >> (i % 32) & 1 : 0; }

int main() {
    std::mt19937_64 rng(7);
    for (uint32_t q : {0u, 2u, 4u, 8u}) {
        const uint32_t d = 32 + q;
        // digits of an operand, and none past its last word
        for (uint32_t L : {1u, 2u, 3u, 8u, 9u, 10u, 31u, 257u}) {
            std::vector<uint32_t> x(L);
            for (auto &w : x) w = (uint32_t)rng();
            const uint64_t n = digits_of(L, d);
            if (n * d < 32ull * L || (n - 1) * d >= 32ull * L) return std::printf("digits_of %u %u\n", q, L), 1;
            for (uint64_t j = 0; j < n + 40; ++j) {
                const uint64_t w = digit_word(j, q);
                if ((w < L) != (j < n)) return std::printf("digit %llu of %u words, q %u\n", (unsigned long long)j, L, q), 1;
                const uint64_t lo = w < L ? x[w] : 0, hi = w + 1 < L ? x[w + 1] : 0;
                const uint64_t v = (hi << 32 | lo) >> digit_shift(j, q) & ((1ull << d) - 1);
                for (uint32_t b = 0; b < d; ++b)
                    if ((int)(v >> b & 1) != bit(x, j * d + b)) return std::printf("digit bits q %u\n", q), 1;
            }
        }
        // a step of 512 elements or more moves whole words
        for (uint64_t j = 0; j < 4096; j += 37)
            for (int s = 9; s < 26; ++s)
                if (digit_word(j + (3ull << s), q) != digit_word(j, q) + 3 * digit_word(1ull << s, q) ||
                    digit_shift(j + (3ull << s), q) != digit_shift(j, q))
                    return std::printf("step 2^%d q %u\n", s, q), 1;
        // the words of a run from its digits
        for (int rl : {3, 4}) {
            if (run_fits(rl, q) != ((d << rl) % 32 == 0)) return std::printf("run_fits\n"), 1;
            if (!run_fits(rl, q)) continue;
            const uint32_t words = run_words(rl, q);
            if (words * 32 != d << rl) return std::printf("run_words\n"), 1;
            std::vector<uint32_t> want(words), got(words);
            std::vector<int> seen(words);
            for (auto &w : want) w = (uint32_t)rng();
            for (uint32_t jr = 0; jr < 1u << rl; ++jr) {
                uint64_t f = 0;
                uint32_t nl = 0;
                for (uint32_t b = 0; b < d; ++b) f |= (uint64_t)bit(want, (uint64_t)jr * d + b) << b;
                for (uint32_t b = 0; b < 32; ++b) nl |= (uint32_t)bit(want, (uint64_t)(jr + 1) * d + b) << b;
                if (jr + 1 == 1u << rl) nl = (uint32_t)rng();  // another run's digit: not used
                const uint32_t next = (uint32_t)(f >> 32) | (uint32_t)((uint64_t)nl << q);
                const uint32_t t = lane_shift(jr, q), w = lane_word(jr, q);
                if (w >= words) return std::printf("lane_word\n"), 1;
                got[w] = (uint32_t)(((uint64_t)next << 32 | (uint32_t)f) >> t);
                ++seen[w];
                if (q != 0 && t == 0) {
                    got[w + 1] = next;
                    ++seen[w + 1];
                }
            }
            for (uint32_t w = 0; w < words; ++w)
                if (seen[w] != 1 || got[w] != want[w]) return std::printf("word %u of a run, rl %d q %u\n", w, rl, q), 1;
        }
    }
    for (uint32_t len = 2; len < 70; ++len) {
        const RunDivisor r = run_divisor(len);
        for (uint64_t j = 0; j < 0x80000000ull; j += j < 4096 ? 1 : 1 + rng() % 400000)
            if (r.run_of((uint32_t)j) != j / len) return std::printf("run_of %llu / %u\n", (unsigned long long)j, len), 1;
        for (uint32_t m = 0x7fffffffu / len, i = 0; i < 200; ++i, --m)
            if (r.run_of(m * len) != m || r.run_of(m * len - 1) != m - 1) return std::printf("run_of %u\n", len), 1;
    }
    std::printf("digit check: ok\n");
    return 0;
}
