// CPU check of the truncated transforms: the last inverse step (itft) against
// 128-bit modular arithmetic for every number of known values, and the tile
// and row counts of the first tau parts.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <random>

#include "ntt_arith.hpp"

using namespace gpupi::ntt;
typedef __int128 i128;

static const int64_t kP[2] = {562948879679489ll, 562941363486721ll};
static const int64_t kGen[2] = {3, 13};
static int64_t mulmod(int64_t a, int64_t b, int64_t p) { return (int64_t)((i128)a * b % p); }
static int64_t powmod(int64_t b, int64_t e, int64_t p) {
    int64_t r = 1;
    for (; e; e >>= 1, b = mulmod(b, b, p))
        if (e & 1) r = mulmod(r, b, p);
    return r;
}
static int64_t centred(int64_t v, int64_t p) {
    v %= p;
    if (v < 0) v += p;
    return v > p / 2 ? v - p : v;
}
static int fails = 0;
static void expect(bool ok, const char *what, int a, int b) {
    if (ok) return;
    if (++fails < 20) std::printf("failed: %s (%d, %d)\n", what, a, b);
}

static std::mt19937_64 rng(7);

template <int T>
static void check_itft(int q) {
    const int64_t p = kP[q], w = powmod(kGen[q], (p - 1) >> 4, p), wi = powmod(w, p - 2, p);
    const Mod m = mod_of(q);
    double w16[8], w16i[8];
    for (int e = 0; e < 8; ++e) {
        w16[e] = (double)centred(powmod(w, e, p), p);
        w16i[e] = (double)centred(powmod(wi, e, p), p);
    }
    const double inv2 = (double)centred((p + 1) / 2, p);
    for (int it = 0; it < 400; ++it) {
        int64_t x[16] = {};
        for (int u = 0; u < T; ++u) {
            const int kind = it % 4;
            x[u] = kind == 0 ? p / 2 : kind == 1 ? -(p / 2) : kind == 2 ? (u & 1 ? p / 2 : -(p / 2)) : centred((int64_t)(rng() >> 2), p);
        }
        double v[16];
        for (int j = 0; j < 16; ++j) {
            i128 s = 0;
            for (int u = 0; u < T; ++u) s += (i128)x[u] * centred(powmod(w, (int64_t)u * bitrev(j, 4) % 16, p), p) % p;
            int64_t y = centred((int64_t)(s % p), p);
            // the bounds of a last inverse step's inputs
            if (j == 0) y += (it % 3 - 1) * 6 * p;
            else if (it & 8) y += (rng() & 1) ? (y < -p / 16 ? 0 : (y < 0 ? 0 : (y < (int64_t)(0.46 * p) ? 0 : -p))) : 0;
            v[j] = j < T ? (double)y : 0.0;
        }
        itft<16, T>(v, w16, w16i, inv2, m);
        for (int u = 0; u < T; ++u) {
            expect(v[u] == std::rint(v[u]) && centred((int64_t)v[u], p) == centred(16 * (x[u] % p), p), "value", T, u);
            expect(std::fabs(v[u]) <= kRedBound * (double)p, "bound", T, u);
        }
    }
}

int main() {
    for (int q = 0; q < 2; ++q) {
        check_itft<9>(q);
        check_itft<10>(q);
        check_itft<11>(q);
        check_itft<12>(q);
        check_itft<13>(q);
        check_itft<14>(q);
        check_itft<15>(q);
        check_itft<16>(q);
    }
    for (int k = kTileLog2 + 1; k <= kMaxLog2; ++k) {
        const uint64_t K = 1ull << k;
        // parts needed by totals around every boundary
        for (uint32_t t = 1; t <= kTauMax; ++t)
            for (int d = -1; d <= 1; ++d) {
                const uint64_t total = K * t / 16 + d;
                if (total == 0 || total > K) continue;
                const uint32_t tau = tau_of(total, k);
                expect(tau * (K / 16) >= total && tau <= kTauMax && tau >= kTauMin && tau % 2 == 0, "parts", k, (int)t);
                expect(tau == kTauMin || (tau - 2) * (K / 16) < total, "parts not more than needed", k, (int)t);
            }
        for (int m0 = kColMinLog2; m0 <= kColMaxLog2; ++m0)
            for (uint32_t tau = kTauMin; tau <= kTauMax; tau += 2) {
                const Plan p = make_plan_split(k, m0, 0);
                if (!plan_ok(p)) continue;
                const uint64_t used = (uint64_t)tau_rows(m0, tau) << (k - m0);  // elements of the parts
                const uint32_t tiles = tau_tiles(tiles_per_product(p), tau);
                expect(used == K / 16 * tau, "rows of the parts", k, m0);
                expect((uint64_t)tiles * kTile >= used && (uint64_t)(tiles - 1) * kTile < used, "tiles of the parts", k, m0);
                // a paired deeper column level starts and ends on whole pairs
                expect(p.levels < 3 || tiles % 2 == 0, "whole tile pairs", k, m0);
            }
    }
    // the threads' last-step values: part of value k (rows in order)
    for (int m0 = kColMinLog2; m0 <= kColMaxLog2; ++m0)
        for (uint32_t tid = 0; tid < 256; ++tid)
            for (int k = 0; k < 16; ++k) {
                const int u = k >> col_last_lr(m0);
                const uint32_t row = col_last_row0(m0, tid) + col_last_row_delta(m0, k);
                const uint32_t first = col_last_row0(m0, tid) + col_last_row_delta(m0, u << col_last_lr(m0));
                expect(row >> (m0 - 4) == first >> (m0 - 4) && row < 1u << m0, "one part per small DFT", m0, k);
            }
    if (fails) {
        std::printf("itft check: %d failures\n", fails);
        return 1;
    }
    std::printf("itft check: ok\n");
    return 0;
}
