// Schoolbook products on the matrix cores, for products of at most
// kMulMfmaMaxTotal limbs.
//
// A product of big integers is a convolution of their digits.  With digits
// of one byte it is a matrix product: output digit 32 C + r (block C, row r)
// is the sum over blocks i and over k < 32 of
//     a[32 i + r - k] * b[32 (C - i) + k],
// so for a fixed i the 32 x 32 Toeplitz matrix T_i[r][k] = a[32 i + r - k]
// multiplies the matrix whose column c is block C - i of b: one
// v_mfma_i32_32x32x32_i8 adds block i's share to 32 output blocks (a tile of
// 1024 digits, 256 limbs; 16 accumulator registers).
//
// The instruction takes signed bytes, so both operands are recoded to
// balanced digits in [-128, 127]: x + 0x80..80 (with its carries), every byte
// minus 0x80, and a carry out as one more digit.  Column sums stay below
// 2^14 times the digits of the shorter operand, exact in 32 bits.
//
// A result register group of a lane holds four consecutive digits' columns,
// that is one limb: u = d0 + 2^8 d1 + 2^16 d2 + 2^24 (d3 - 1), |u| < 2^53.
// The -1 (it comes with the accumulator's start value) moves 2^24 from the
// limb itself to the part passed on, which is then hi(u) + 2^24 > 0: the
// limbs are lo(u), what each passes to the next is a positive 25-bit number,
// and adding the two rows of words is an ordinary addition whose carries the
// ballots resolve (resolve_carries).
//
// What bounds it: for rows of some hundred limbs the matrix pipe (16384
// products of 501 x 503 limbs: 85 us, 71 % of the CU cycles in MFMA; the
// one-tile NTT took 269 us), for short rows the VALU work around it (staging,
// fragment shifts, limbs: 261 instructions per product; 262144 products of
// 63 x 64 limbs 139 us against 325 us with one wave per product and 32-bit
// multiply-adds), for a lone product the latency of its phases (1203 x 901
// limbs 10 us against 24.5 us).  Work grows with the square of the length;
// at the largest products it still beats the NTT (4096 rows of 2000 x 2000
// limbs 277 against 300 us, one row 17 against 27 us).
#include <algorithm>
#include <mutex>
#include <type_traits>
#include <utility>
#include <vector>

#include "common.hpp"

namespace gpupi {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

constexpr uint32_t kTileLimbs = 256;
constexpr uint32_t kMaxTiles = 32;
constexpr uint32_t kPassBias = 1u << 24;
constexpr uint32_t kManyG = 8, kFewG = 5;  // tiles per wave at most: many rows, few rows

// Blocks of 32 digits of an operand (its digits and the recoding's carry).
__host__ __device__ inline uint32_t blocks_of(uint32_t L) { return L / 8u + 1u; }

// How a product runs: W groups of tiles (wave w takes the tiles w, w + W,
// ...), and steps i0 < i0_end in each of which a wave multiplies the blocks
// i0 + 32 W q (q < M) of a with E blocks of columns of b; steps below m_thr
// have M blocks, the others M - 1.
struct MfmaArgs {
    const uint32_t *A, *B;
    uint32_t *C;
    uint32_t LA, LB, sA, sB, sC;
    uint32_t W, M, E, na, nb, i0_end, m_thr;
    uint32_t a_words, b_lead, b_half, lds_words;  // LDS words: a, zeros below b and a half of it, all but the column sums
};

// A ragged launch carries its products in the kernel's arguments: no device
// memory to fill, nothing to wait for, and a captured launch holds its own
// copy.  A product is three words (arg_word), so that as many as possible go
// into the 4 KB that a launch's arguments may take: launches follow each other,
// and with rows of 32 bytes, 96 to a launch, 600 products of 2^9..2^11 limbs
// took 156 us instead of 87.  Above six launches the same rows go into a block
// of device memory, one launch per number of tile groups (600 products of
// 2^9..2^11 limbs 87 us from arguments against 98 from memory, 1500 of them 186
// against 155, 12000 2042 against 879).
constexpr uint32_t kArgRows = 168, kArgRowsMost = 6 * kArgRows;
struct ArgRow {
    uint64_t a, b, c;
};
static_assert(kMulMfmaMaxTotal <= 1u << kArgLengthBits, "a length fits its bits");
struct MfmaRaggedArgs {
    uint32_t W;
    ArgRow rows[kArgRows];
};
static_assert(sizeof(MfmaRaggedArgs) <= 4096, "a launch's arguments");
struct MfmaListArgs {
    uint32_t W;
    const ArgRow *rows;
};

// What of MfmaArgs a ragged launch's W decides: LDS for the longest operands
// of any of its shapes, three blocks of a and five of b.
__host__ __device__ inline MfmaArgs ragged_base(uint32_t W) {
    MfmaArgs s{};
    s.W = W;
    s.a_words = 256u * W * 3u + 20u;
    s.b_lead = 4u * (32u * W - 1u);
    s.b_half = 4u * 32u * W * 5u + s.b_lead;
    s.lds_words = s.a_words + 2 * s.b_half + 2 * kMaxTiles;
    return s;
}
__device__ inline MfmaArgs base_of(const MfmaArgs &a) { return a; }
__device__ inline MfmaArgs base_of(const MfmaRaggedArgs &a) { return ragged_base(a.W); }
__device__ inline MfmaArgs base_of(const MfmaListArgs &a) { return ragged_base(a.W); }

MfmaArgs shape_of(uint32_t LA, uint32_t LB, uint32_t W) {
    MfmaArgs s{};
    s.LA = LA;
    s.LB = LB;
    s.W = W;
    s.na = blocks_of(LA);
    s.nb = blocks_of(LB);
    // blocks i <= na of T reach digits of a
    s.i0_end = std::min(32u * W - 1u, s.na) + 1u;
    s.M = s.na / (32u * W) + 1u;
    s.m_thr = s.na + 1u - 32u * W * (s.M - 1u);
    s.E = (s.nb - 1u + s.i0_end - 1u) / (32u * W) + 1u;
    s.a_words = (8u * (s.i0_end + 32u * W * (s.M - 1u)) + 17u + 3u) & ~3u;
    s.b_lead = 4u * (s.i0_end - 1u);
    s.b_half = 4u * 32u * W * s.E + s.b_lead;
    s.lds_words = s.a_words + 2 * s.b_half + 2 * kMaxTiles;
    return s;
}

// The recoding's carry into limb l0: the nearest lower limb that is not
// 0x7f7f7f7f decides.
__device__ __forceinline__ uint32_t recode_carry_in(const uint32_t *x, uint32_t l0, uint32_t lane) {
    for (int64_t hi = (int64_t)l0 - 1; hi >= 0; hi -= kWave) {
        const int64_t k = hi - (int64_t)lane;
        const uint32_t v = k >= 0 ? x[k] : 0u;
        const uint64_t stop = ballot64(v != 0x7f7f7f7fu);
        if (stop != 0) return (uint32_t)(ballot64(v > 0x7f7f7f7fu) >> __builtin_ctzll(stop)) & 1u;
    }
    return 0u;
}

__device__ __forceinline__ uint32_t lane_bit(uint64_t mask) { return __builtin_amdgcn_inverse_ballot_w64(mask) ? 1u : 0u; }

// Recodes one operand into LDS, wave tw of TW taking its share of 64-limb
// segments: a's limbs in order, b's (REV) as 16-byte groups of reversed
// digits, the even and odd groups in two halves `half` words apart.
template <bool REV>
__device__ __forceinline__ void stage_segment(uint32_t *p, uint32_t v, uint32_t bias, bool in, uint32_t *cin) {
    uint32_t cout;
    const uint64_t cm = resolve_carries(ballot64(v > 0x7f7f7f7fu), ballot64(v == 0x7f7f7f7fu), *cin, &cout);
    *cin = cout;
    const uint32_t y = (v + bias + lane_bit(cm)) ^ bias;
    if (in) *p = REV ? __builtin_bswap32(y) : y;
}
template <bool REV>
__device__ __forceinline__ void stage_operand(uint32_t *s, uint32_t half, const uint32_t *x, uint32_t L, uint32_t blocks,
                                              uint32_t tw, uint32_t TW, uint32_t lane) {
    constexpr int U = 4;
    constexpr uint32_t kSeg = REV ? kWave / 2 : kWave;  // LDS words from one segment to the next (in a half)
    const uint32_t full = L / kWave;                      // segments full..full: the rest and the carry out
    uint32_t sg = 0, s1 = full + 1u, cin = 0;
    if (TW > 1) {
        const uint32_t per = (s1 + TW - 1u) / TW;
        sg = tw * per;
        s1 = min(sg + per, s1);
        if (sg >= s1) return;
        if (sg > 0) cin = recode_carry_in(x, sg * kWave, lane);
    }
    uint32_t *p = s + (REV ? ((lane >> 2) & 1u) * half + (lane >> 3) * 4u + (3u - (lane & 3u)) : lane);
    const uint32_t *xl = x + lane;
    for (; sg + U <= min(s1, full); sg += U) {
        uint32_t v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = xl[(sg + u) * kWave];
#pragma unroll
        for (int u = 0; u < U; ++u) stage_segment<REV>(p + (sg + u) * kSeg, v[u], 0x80808080u, true, &cin);
    }
    for (; sg < min(s1, full); ++sg) stage_segment<REV>(p + sg * kSeg, xl[sg * kWave], 0x80808080u, true, &cin);
    if (sg < s1) {
        // limbs past L are zero but for the carry out at L: no bias there
        const uint32_t l = sg * kWave + lane;
        const bool in = l < L;
        stage_segment<REV>(p + sg * kSeg, in ? xl[sg * kWave] : 0u, in ? 0x80808080u : 0u, l < 8u * blocks, &cin);
    }
}

__device__ __forceinline__ void zero_quads(uint32_t *p, uint32_t quads, uint32_t t, uint32_t step) {
    for (uint32_t x = t; x < quads; x += step) reinterpret_cast<v4u *>(p)[x] = v4u{0u, 0u, 0u, 0u};
}

// LDS written by the product's waves is visible to them.
__device__ __forceinline__ void team_sync(uint32_t TW) {
    if (TW > 1) {
        __syncthreads();
    } else {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        __builtin_amdgcn_wave_barrier();
    }
}

// One step: M blocks of a (32 W apart) against blocks E0..E-1 of columns of b.
template <int M, int E0, int E>
__device__ __forceinline__ void step_mfma(v16i *acc, const uint32_t *pa, const uint32_t *pb, uint32_t W, uint32_t sh) {
    if constexpr (M > 0 && E > E0) {
        v4i b[E];
        uint32_t w[M][5];
#pragma unroll
        for (int q = 0; q < M; ++q) {
            const uint32_t *p = pa + 256u * W * (uint32_t)q;
#pragma unroll
            for (int x = 0; x < 5; ++x) w[q][x] = p[x];
        }
#pragma unroll
        for (int e = E0; e < E; ++e) b[e] = *reinterpret_cast<const v4i *>(pb + 128u * W * (uint32_t)e);
#pragma unroll
        for (int q = 0; q < M; ++q) {
            v4i a;
#pragma unroll
            for (int x = 0; x < 4; ++x) a[x] = (int)__builtin_amdgcn_alignbyte(w[q][x + 1], w[q][x], sh);
#pragma unroll
            for (int e = E0; e < E; ++e) acc[q + e] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b[e], acc[q + e], 0, 0, 0);
        }
    }
}

// The steps [i0, end) of a wave (every S-th): below m_thr M blocks of a, then
// M - 1; from e_thr on all E blocks of b, before that E - 1.
template <int M, int E0, int E, int S>
__device__ __forceinline__ void steps_mfma(v16i *acc, uint32_t &i0, uint32_t end, uint32_t m_thr, uint32_t e_thr,
                                           const uint32_t *a_l, const uint32_t *b_l, uint32_t W, uint32_t sh) {
    m_thr = min(m_thr, end);
    e_thr = min(e_thr, end);
    for (; i0 < min(m_thr, e_thr); i0 += S) step_mfma<M, E0, E - 1>(acc, a_l + 8 * i0, b_l - 4 * (int)i0, W, sh);
    for (; i0 < e_thr; i0 += S) step_mfma<M - 1, E0, E - 1>(acc, a_l + 8 * i0, b_l - 4 * (int)i0, W, sh);
    for (; i0 < m_thr; i0 += S) step_mfma<M, E0, E>(acc, a_l + 8 * i0, b_l - 4 * (int)i0, W, sh);
    for (; i0 < end; i0 += S) step_mfma<M - 1, E0, E>(acc, a_l + 8 * i0, b_l - 4 * (int)i0, W, sh);
}

// A tile's limbs: lane (r, h) = (lane mod 32, lane / 32) holds limbs
// 8 r + 4 h + 0..3 as x and what each of them passes on as y.
struct TileLimbs {
    uint32_t x[4], y[4];
};
__device__ __forceinline__ TileLimbs tile_limbs(const int *d) {
    int k8 = 1 << 8, k16 = 1 << 16, k24 = 1 << 24;
    // opaque factors: three 64-bit multiply-adds instead of 64-bit shifts
    __asm__("" : "+s"(k8), "+s"(k16), "+s"(k24));
    uint32_t lo[4], hi[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        int64_t u = (int64_t)d[4 * m + 1] * k8 + (int64_t)d[4 * m];
        u = (int64_t)d[4 * m + 2] * k16 + u;
        u = (int64_t)d[4 * m + 3] * k24 + u;
        lo[m] = (uint32_t)u;
        hi[m] = (uint32_t)(u >> 32) + kPassBias;
    }
    // the lane's groups are limbs 8 r + 2 m + h
    const auto s0 = __builtin_amdgcn_permlane32_swap(lo[0], lo[2], false, false);
    const auto s1 = __builtin_amdgcn_permlane32_swap(lo[1], lo[3], false, false);
    const auto t0 = __builtin_amdgcn_permlane32_swap(hi[0], hi[2], false, false);
    const auto t1 = __builtin_amdgcn_permlane32_swap(hi[1], hi[3], false, false);
    return TileLimbs{{s0[0], s0[1], s1[0], s1[1]}, {t0[0], t0[1], t1[0], t1[1]}};
}

// The lane's four limbs plus what their lower neighbours pass on, settled
// for a carry-in of zero to the lane; masks over the 32 pairs of lanes
// (r, 0), (r, 1): carry out of the pair for a carry-in of zero, pair passes a
// carry; and the first lane's own two masks.
struct TileCarry {
    uint32_t g0, p0, gen, prop;
};
__device__ __forceinline__ TileCarry tile_settle(TileLimbs &t, uint32_t below_tile, uint32_t lane) {
    const uint32_t r = lane & 31u;
    uint32_t below = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(4u * (lane >= 32u ? r : ((r + 31u) & 31u) + 32u)), (int)t.y[3]);
    if (lane == 0) below = below_tile;
    uint32_t c;
    t.x[0] = __builtin_addc(t.x[0], below, 0u, &c);
    t.x[1] = __builtin_addc(t.x[1], t.y[0], c, &c);
    t.x[2] = __builtin_addc(t.x[2], t.y[1], c, &c);
    t.x[3] = __builtin_addc(t.x[3], t.y[2], c, &c);
    const uint64_t gm = ballot64(c != 0), pm = ballot64((t.x[0] & t.x[1] & t.x[2] & t.x[3]) == 0xffffffffu);
    TileCarry k;
    k.g0 = (uint32_t)gm;
    k.p0 = (uint32_t)pm;
    k.gen = (uint32_t)(gm >> 32) | ((uint32_t)(pm >> 32) & k.g0);
    k.prop = (uint32_t)(pm >> 32) & k.p0;
    return k;
}
__device__ __forceinline__ uint32_t tile_carry_out(const TileCarry &k, uint32_t cin) {
    return (uint32_t)(((uint64_t)(k.gen | k.prop) + k.gen + cin) >> 32);
}
__device__ __forceinline__ void tile_store(uint32_t *c, uint32_t l, uint32_t Lc, const TileLimbs &t, const TileCarry &k,
                                           uint32_t cin) {
    const uint32_t X = k.gen | k.prop;
    const uint32_t cpair = (X + k.gen + cin) ^ X ^ k.gen;  // carry into each pair
    const uint32_t csecond = k.g0 | (k.p0 & cpair);        // and into its second lane
    uint32_t cc = lane_bit((uint64_t)csecond << 32 | cpair);
    Quad q;
#pragma unroll
    for (int i = 0; i < 4; ++i) q.w[i] = __builtin_addc(t.x[i], 0u, cc, &cc);
    if (l + 4 <= Lc) {
        *reinterpret_cast<Quad *>(c + l) = q;
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (l + i < Lc) c[l + i] = q.w[i];
    }
}

// RAGGED (its own ARGS; S > 1, G = 5): block i multiplies row i's operands, of any lengths
// that W takes; M and E are one of three shapes with M + E - 1 = 5 chosen per
// block, and fragments a product does not reach are zero.
// One product per block, W tile groups (WT: W where it is known, else 0).
// S = 1: one wave per group, finishing its own tiles.  S > 1: S waves per
// group, part ks of them taking the steps ks, ks + S, ...; the parts' column
// sums meet in LDS and each wave finishes a tile or two.
constexpr int mfma_waves(int g) { return g <= 1 ? 8 : g <= 2 ? 6 : g <= 5 ? 4 : 2; }
template <int M, int E, int WT, int S, typename ARGS = MfmaArgs>
__global__ void __launch_bounds__(S == 1 ? 256 : 1024) __attribute__((amdgpu_waves_per_eu(mfma_waves(M + E - 1))))
mul_mfma_kernel(ARGS args) {
    constexpr bool RAGGED = !std::is_same_v<ARGS, MfmaArgs>;
    constexpr int G = M + E - 1;
    MfmaArgs a = base_of(args);
    extern __shared__ __align__(16) uint32_t lds[];
    const uint32_t lane = threadIdx.x & (kWave - 1u);
    const uint32_t wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t W = WT > 0 ? (uint32_t)WT : a.W;
    const uint32_t TW = W * S;  // waves per product
    const uint32_t ks = S > 1 ? wid / W : 0u, tw = wid - ks * W;
    const size_t row = RAGGED ? 0 : blockIdx.x;
    if constexpr (RAGGED) {
        const ArgRow rr = args.rows[blockIdx.x];
        a.A = reinterpret_cast<const uint32_t *>(arg_address(rr.a));
        a.B = reinterpret_cast<const uint32_t *>(arg_address(rr.b));
        a.C = reinterpret_cast<uint32_t *>(arg_address(rr.c));
        a.LA = arg_length(rr.a);
        a.LB = arg_length(rr.b);
        a.na = blocks_of(a.LA);
        a.nb = blocks_of(a.LB);
        a.i0_end = min(32u * W - 1u, a.na) + 1u;
        a.m_thr = a.i0_end;
    }
    uint32_t *const a_s = lds + 8;
    const uint32_t b_lead = a.b_lead;
    uint32_t *const b_s = lds + a.a_words + b_lead;
    uint32_t *const h_s = lds + a.a_words + 2 * a.b_half;  // per tile: what it passes on
    uint32_t *const f_s = h_s + kMaxTiles;                 // per tile: carry out for a carry-in of 0, 1
    uint32_t *const d_s = f_s + kMaxTiles;                 // S > 1: column sums

    if (TW == 1) {
        // one wave: its LDS writes stay in order, so everything is cleared first
        zero_quads(a_s - 8, (a.a_words + 2u * a.b_half) / 4u, lane, kWave);
    } else {
        // zeros around the digits, whole 16-byte groups
        const uint32_t t = wid * kWave + lane, step = TW * kWave;
        zero_quads(a_s - 8, 2, t, step);
        zero_quads(a_s + 8 * a.na, (a.a_words - 8u - 8u * a.na) / 4u, t, step);
        zero_quads(b_s - b_lead, b_lead / 4u, t, step);
        zero_quads(b_s - b_lead + a.b_half, b_lead / 4u, t, step);
        const uint32_t above = (a.b_half - b_lead) / 4u - a.nb;
        zero_quads(b_s + 4 * a.nb, above, t, step);
        zero_quads(b_s + a.b_half + 4 * a.nb, above, t, step);
        if (S > 1) zero_quads(d_s, W * G * 256u, t, step);
    }
    stage_operand<false>(a_s, 0, a.A + row * a.sA, a.LA, a.na, wid, TW, lane);
    stage_operand<true>(b_s, a.b_half, a.B + row * a.sB, a.LB, a.nb, wid, TW, lane);
    team_sync(TW);

    // lane (r, h) of T_i: digits 32 i + r - 16 h - 15 + 0..15 (the order of
    // k within 16 is reversed on both sides), from five words shifted by sh
    // bytes; of b's columns: group h of block 32 (tw + W e) - i0 + r
    const uint32_t r = lane & 31u, h = lane >> 5;
    const uint32_t sh = (r + 1u) & 3u;
    const uint32_t *const a_l = a_s + ((int)r - 16 * (int)h - 15 - (int)sh) / 4;
    const uint32_t *const b_l = b_s + h * a.b_half + 4 * (r + 32 * tw);
    v16i acc[G];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int k = 0; k < 16; ++k) acc[g][k] = (k & 3) == 3 && ks == 0 ? -1 : 0;
    uint32_t i0 = ks;
    if constexpr (RAGGED) {
        static_assert(S > 1 && G == (int)kFewG, "every shape has G tiles");
        const uint32_t m_row = a.na / (32u * W) + 1u, e_row = (a.nb - 1u + a.i0_end - 1u) / (32u * W) + 1u;
        const uint32_t first = min(a.i0_end, 32u * (tw + 1u));
        if (m_row <= 1u) {
            steps_mfma<1, 0, 5, S>(acc, i0, first, first, 0u, a_l, b_l, W, sh);
            steps_mfma<1, 1, 5, S>(acc, i0, a.i0_end, a.i0_end, 0u, a_l, b_l, W, sh);
        } else if (e_row > 3u) {
            steps_mfma<2, 0, 4, S>(acc, i0, first, first, 0u, a_l, b_l, W, sh);
            steps_mfma<2, 1, 4, S>(acc, i0, a.i0_end, a.i0_end, 0u, a_l, b_l, W, sh);
        } else {
            steps_mfma<3, 0, 3, S>(acc, i0, first, first, 0u, a_l, b_l, W, sh);
            steps_mfma<3, 1, 3, S>(acc, i0, a.i0_end, a.i0_end, 0u, a_l, b_l, W, sh);
        }
    } else {
    // from e_thr on the last of the E blocks reaches digits of b; from f_thr
    // on the first one lies below them
    const uint32_t e_thr = (uint32_t)max(32 * (int)(tw + W * (E - 1)) - (int)(a.nb - 1u), 0);
    if constexpr (WT == 1) {
        steps_mfma<M, 0, E, S>(acc, i0, a.i0_end, a.m_thr, e_thr, a_l, b_l, W, sh);
    } else {
        steps_mfma<M, 0, E, S>(acc, i0, min(a.i0_end, 32u * (tw + 1u)), a.m_thr, e_thr, a_l, b_l, W, sh);
        steps_mfma<M, 1, E, S>(acc, i0, a.i0_end, a.m_thr, e_thr, a_l, b_l, W, sh);
    }
    }

    uint32_t *const c = a.C + row * a.sC;
    const uint32_t Lc = a.LA + a.LB;
    const uint32_t l0 = 8 * r + 4 * h;
    if constexpr (S > 1) {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int k = 0; k < 16; ++k)
                __hip_atomic_fetch_add(&d_s[((tw + W * g) * 16 + k) * kWave + lane], (uint32_t)acc[g][k],
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __syncthreads();
        // wave w finishes tiles w, w + TW
        constexpr int NT = (G + S - 1) / S;
        TileLimbs x[NT];
        TileCarry k[NT];
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const uint32_t t = wid + n * TW;
            int d[16];
#pragma unroll
            for (int j = 0; j < 16; ++j) d[j] = t < W * G ? (int)d_s[(t * 16 + j) * kWave + lane] : 0;
            x[n] = tile_limbs(d);
            if (lane == 63u) h_s[t] = x[n].y[3];
        }
        __syncthreads();
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const uint32_t t = wid + n * TW;
            k[n] = tile_settle(x[n], t > 0 ? h_s[t - 1] : kPassBias, lane);
            if (lane == 0) f_s[t] = tile_carry_out(k[n], 0u) | tile_carry_out(k[n], 1u) << 1;
        }
        __syncthreads();
        uint32_t seen = 0, cin = 0;
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const uint32_t t = wid + n * TW;
            for (; seen < t; ++seen) cin = (f_s[seen] >> cin) & 1u;
            tile_store(c, kTileLimbs * t + l0, Lc, x[n], k[n], cin);
        }
        return;
    }
    TileLimbs x[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        int d[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) d[k] = acc[g][k];
        x[g] = tile_limbs(d);
    }
    if (TW == 1) {
        uint32_t cin = 0;
        for (int g = 0; g < G; ++g) {
            const uint32_t below = g > 0 ? (uint32_t)__builtin_amdgcn_readlane((int)x[g > 0 ? g - 1 : 0].y[3], 63) : kPassBias;
            const TileCarry k = tile_settle(x[g], below, lane);
            tile_store(c, kTileLimbs * g + l0, Lc, x[g], k, cin);
            cin = tile_carry_out(k, cin);
        }
        return;
    }
#pragma unroll
    for (int g = 0; g < G; ++g)
        if (lane == 63u) h_s[tw + W * g] = x[g].y[3];
    team_sync(TW);
    TileCarry k[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const uint32_t t = tw + W * g;
        k[g] = tile_settle(x[g], t > 0 ? h_s[t - 1] : kPassBias, lane);
        if (lane == 0) f_s[t] = tile_carry_out(k[g], 0u) | tile_carry_out(k[g], 1u) << 1;
    }
    team_sync(TW);
    uint32_t seen = 0, cin = 0;
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const uint32_t t = tw + W * g;
        for (; seen < t; ++seen) cin = (f_s[seen] >> cin) & 1u;
        tile_store(c, kTileLimbs * t + l0, Lc, x[g], k[g], cin);
    }
}

typedef void (*MfmaKernel)(MfmaArgs);
constexpr int kParts = 4;
// Calls f with the kernels <M, E> for M <= E, M + E - 1 <= GMAX in turn until
// it returns true.
template <int M, int E, int WT, int S, uint32_t GMAX, typename F>
bool each_kernel(F &&f) {
    if (f(M, E, mul_mfma_kernel<M, E, WT, S>)) return true;
    if constexpr (M + E <= (int)GMAX) return each_kernel<M, E + 1, WT, S, GMAX>(f);
    else if constexpr (2 * M + 1 <= (int)GMAX) return each_kernel<M + 1, M + 1, WT, S, GMAX>(f);
    else return false;
}

constexpr uint32_t kRaggedMaxW = 4;
template <typename ARGS>
using RaggedKernel = void (*)(ARGS);
const RaggedKernel<MfmaRaggedArgs> kRaggedKernel = mul_mfma_kernel<3, 3, 0, kParts, MfmaRaggedArgs>;
const RaggedKernel<MfmaListArgs> kListKernel = mul_mfma_kernel<3, 3, 0, kParts, MfmaListArgs>;

// The kernels of several parts may take more than 64 KB of LDS; the attribute
// is a property of the current device, set once per device (serving threads
// launch concurrently).
std::mutex g_lds_mu;
uint64_t g_lds_done = 0;  // bit d: set on device d
hipError_t allow_large_lds() {
    int dev = 0;
    GPUPI_RETURN_IF(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_lds_mu);
    const uint64_t bit = dev >= 0 && dev < 64 ? 1ull << dev : 0ull;
    if (bit != 0 && (g_lds_done & bit) != 0) return hipSuccess;
    hipError_t err = hipSuccess;
    each_kernel<1, 1, 0, kParts, kFewG>([&](int, int, MfmaKernel k) {
        err = hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        return err != hipSuccess;
    });
    GPUPI_RETURN_IF(err);
    for (const void *k : {(const void *)kRaggedKernel, (const void *)kListKernel})
        GPUPI_RETURN_IF(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    g_lds_done |= bit;
    return hipSuccess;
}

}  // namespace

// Few rows (at most two per CU) of more than one tile: kParts waves per tile
// group and few tiles per wave, for the latency of a product; otherwise one
// wave per eight tiles, which reads the fewest fragments per MFMA.  512 rows
// of 250 / 500 / 1000 / 2000 limbs: 7 / 9 / 16 / 43 us in parts against
// 7 / 10 / 22 / 52 us; 1024 rows: 9 / 12 / 29 / 84 against 8 / 12 / 25 / 64 us.
constexpr uint32_t kFewRows = 512;

hipError_t launch_mul_mfma(const uint32_t *A, const uint32_t *B, uint32_t *C, uint32_t N, uint32_t LA, uint32_t LB,
                           uint32_t sA, uint32_t sB, uint32_t sC, hipStream_t stream) {
    // the shorter operand gives the Toeplitz matrices (fewer steps)
    if (LA > LB) {
        std::swap(A, B);
        std::swap(LA, LB);
        std::swap(sA, sB);
    }
    if (N == 0 || LA == 0 || (uint64_t)LA + LB > kMulMfmaMaxTotal) return hipErrorInvalidValue;
    const bool few = LA + LB > kTileLimbs && N <= kFewRows;
    uint32_t W = 1;
    MfmaArgs a = shape_of(LA, LB, W);
    while (a.M + a.E - 1 > (few ? kFewG : kManyG)) a = shape_of(LA, LB, ++W);
    a.sA = sA;
    a.sB = sB;
    a.sC = sC;
    const uint32_t tiles = W * (a.M + a.E - 1);
    MfmaKernel k = nullptr;
    const auto match = [&](int m, int e, MfmaKernel f) {
        if ((uint32_t)m != a.M || (uint32_t)e != a.E) return false;
        k = f;
        return true;
    };
    if (few) (void)each_kernel<1, 1, 0, kParts, kFewG>(match);
    else if (W == 1) (void)each_kernel<1, 1, 1, 1, kManyG>(match);
    else (void)each_kernel<1, 1, 0, 1, kManyG>(match);
    const size_t lds = (a.lds_words + (few ? tiles * 1024u : 0u)) * 4u;
    if (k == nullptr || tiles > kMaxTiles || W > 4 || lds > 160 * 1024) return hipErrorInvalidValue;
    if (lds > 65536) GPUPI_RETURN_IF(allow_large_lds());
    // a launch holds fewer than 2^32 threads
    const uint32_t threads = kWave * W * (few ? kParts : 1u), most = 0xffffffffu / threads;
    for (uint32_t r0 = 0; r0 < N; r0 += std::min(most, N - r0)) {
        a.A = A + (size_t)r0 * sA;
        a.B = B + (size_t)r0 * sB;
        a.C = C + (size_t)r0 * sC;
        hipLaunchKernelGGL(k, dim3(std::min(most, N - r0)), dim3(threads), lds, stream, a);
        GPUPI_RETURN_IF(hipGetLastError());
    }
    return hipSuccess;
}

namespace {
// Tile groups that a product of these lengths takes (LA <= LB) in a ragged launch.
uint32_t ragged_groups(uint32_t LA, uint32_t LB) {
    uint32_t W = 1;
    MfmaArgs a = shape_of(LA, LB, W);
    while (a.M + a.E - 1 > kFewG) a = shape_of(LA, LB, ++W);
    return W;
}

template <typename ARGS>
hipError_t launch_ragged(RaggedKernel<ARGS> kernel, const ARGS &args, uint32_t n, hipStream_t stream) {
    const size_t lds = (ragged_base(args.W).lds_words + args.W * kFewG * 1024u) * 4u;
    if (lds > 65536) GPUPI_RETURN_IF(allow_large_lds());
    hipLaunchKernelGGL(kernel, dim3(n), dim3(kWave * args.W * kParts), lds, stream, args);
    return hipGetLastError();
}
}  // namespace

hipError_t launch_mul_mfma_ragged(std::vector<MfmaRow> products, BlockCache &cache, hipStream_t stream) {
    // addresses that no word holds take a launch each
    const auto packs = [](const MfmaRow &r) {
        return arg_packs((uintptr_t)r.A) && arg_packs((uintptr_t)r.B) && arg_packs((uintptr_t)r.C);
    };
    const auto rest = std::stable_partition(products.begin(), products.end(), packs);
    for (auto r = rest; r != products.end(); ++r)
        GPUPI_RETURN_IF(launch_mul_mfma(r->A, r->B, r->C, 1, r->L_a, r->L_b, r->L_a, r->L_b, r->L_a + r->L_b, stream));
    products.erase(rest, products.end());
    const size_t n = products.size();
    // in the order of their tile groups: a launch takes those of its last
    size_t start[kRaggedMaxW + 2] = {};  // start[w]: products of fewer than w groups
    std::vector<uint8_t> groups(n);
    for (size_t i = 0; i < n; ++i) {
        const MfmaRow &r = products[i];
        if (r.L_a == 0 || r.L_b == 0 || (uint64_t)r.L_a + r.L_b > kMulMfmaMaxTotal) return hipErrorInvalidValue;
        const uint32_t w = ragged_groups(std::min(r.L_a, r.L_b), std::max(r.L_a, r.L_b));
        if (w > kRaggedMaxW) return hipErrorInvalidValue;
        groups[i] = (uint8_t)w;
        ++start[w + 1];
    }
    for (uint32_t w = 1; w < kRaggedMaxW + 2; ++w) start[w] += start[w - 1];
    std::vector<ArgRow> rows(n);
    {
        size_t at[kRaggedMaxW + 1];
        std::copy_n(start, kRaggedMaxW + 1, at);
        for (size_t i = 0; i < n; ++i) {
            const MfmaRow &r = products[i];
            uint64_t a = arg_word((uintptr_t)r.A, r.L_a), b = arg_word((uintptr_t)r.B, r.L_b);
            if (r.L_a > r.L_b) std::swap(a, b);
            rows[at[groups[i]]++] = ArgRow{a, b, arg_word((uintptr_t)r.C, 0)};
        }
    }
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (n > kArgRowsMost) GPUPI_RETURN_IF(hipStreamIsCapturing(stream, &capturing));
    if (n > kArgRowsMost && capturing == hipStreamCaptureStatusNone) {
        void *list = nullptr;
        size_t got = 0;
        GPUPI_RETURN_IF(cache.acquire(stream, n * sizeof(ArgRow), &list, &got));
        const ArgRow *const d = static_cast<const ArgRow *>(list);
        hipError_t err = hipMemcpyAsync(list, rows.data(), n * sizeof(ArgRow), hipMemcpyHostToDevice, stream);
        if (err == hipSuccess) err = hipStreamSynchronize(stream);
        for (uint32_t w = 1; w <= kRaggedMaxW && err == hipSuccess; ++w) {
            const size_t m = start[w + 1] - start[w];
            if (m > 0) err = launch_ragged(kListKernel, MfmaListArgs{w, d + start[w]}, (uint32_t)m, stream);
        }
        cache.give_back(list, got, stream);
        return err;
    }
    for (size_t r0 = 0; r0 < n; r0 += kArgRows) {
        const size_t m = std::min<size_t>(kArgRows, n - r0);
        MfmaRaggedArgs a{};
        for (a.W = 1; start[a.W + 1] < r0 + m;) ++a.W;
        std::copy_n(rows.begin() + r0, m, a.rows);
        GPUPI_RETURN_IF(launch_ragged(kRaggedKernel, a, (uint32_t)m, stream));
    }
    return hipSuccess;
}

}  // namespace gpupi
