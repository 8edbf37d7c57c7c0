// Carry-propagating batched ops: add, sub, add_small, sub_small, mul_small,
// shift_add, shift_sub, and the spill-add used to finish NTT products.
//
// Every op is "per-limb digit + one carry/borrow chain": limb j of the result
// is d_j +/- c_j where (d_j, generate_j) come from the inputs and c_j is the
// incoming carry.  The chain is resolved wave-wide with two 64-bit ballots
// (generate and propagate masks) and one 64-bit add (resolve_carries), so a
// wave settles 64 limbs per step instead of the reference's 32-lane
// Kogge-Stone scans (reference batch_mul_addsub_warp.h:5-85).
//
// Layout: rows of at most kThreadRowMax limbs take one thread each; up to 512
// limbs one wave (addsub_chunk_kernel, coalesced 256-byte segments); longer
// rows one wave per chunk of 1024 limbs, four limbs per lane
// (addsub_vec_kernel, spill_add_vec_kernel).  The chunks of a row that one
// block holds (kRowWaves) settle the carries between them in LDS; longer rows
// get a second, tiny kernel: each chunk looks back at its predecessors'
// (generate, all-propagate) flags and, only if its carry-in is 1, ripples it
// through its own limbs.
#include <type_traits>

#include "common.hpp"
#include "ntt_plan.hpp"

namespace gpupi {
namespace {

constexpr uint32_t kThreadRowMax = 16;

struct Digit {
    uint32_t d;
    uint32_t g;
};

struct SpillArgs {
    const uint64_t *spill;
    ntt::RunDivisor run;  // limbs per run
    uint32_t runs_per_row;
};

template <AddSubKind K>
struct OpTraits {
    static constexpr bool kSub = (K == AddSubKind::Sub || K == AddSubKind::SubSmall ||
                                  K == AddSubKind::ShiftSub);
};

__device__ __forceinline__ uint32_t load_or_zero(const uint32_t *p, uint32_t row, uint32_t stride,
                                                 int64_t j, uint32_t len) {
    return (j >= 0 && j < (int64_t)len) ? p[(size_t)row * stride + (size_t)j] : 0u;
}

template <AddSubKind K>
__device__ __forceinline__ Digit digit_at(const AddSubArgs &a, const SpillArgs &sp, uint32_t row,
                                          uint32_t j) {
    uint32_t x, y;
    if constexpr (K == AddSubKind::Add || K == AddSubKind::Sub) {
        x = load_or_zero(a.A, row, a.stride_A, j, a.L_a);
        y = load_or_zero(a.B, row, a.stride_B, j, a.L_b);
    } else if constexpr (K == AddSubKind::AddSmall || K == AddSubKind::SubSmall) {
        x = load_or_zero(a.A, row, a.stride_A, j, a.L_a);
        y = (j == 0) ? a.scalar : 0u;
    } else if constexpr (K == AddSubKind::MulSmall) {
        const uint64_t p = (uint64_t)load_or_zero(a.A, row, a.stride_A, j, a.L_a) * a.scalar;
        const uint64_t q = (uint64_t)load_or_zero(a.A, row, a.stride_A, (int64_t)j - 1, a.L_a) * a.scalar;
        const uint32_t lo = (uint32_t)p;
        const uint32_t d = lo + (uint32_t)(q >> 32);
        return {d, (uint32_t)(d < lo)};
    } else if constexpr (K == AddSubKind::ShiftAdd || K == AddSubKind::ShiftSub) {
        const int64_t i = (int64_t)j - (int64_t)(a.shift >> 5);
        const uint32_t r = a.shift & 31u;
        const uint32_t hi = load_or_zero(a.A, row, a.stride_A, i, a.L_a);
        x = hi;
        if (r != 0) {
            const uint32_t lo = load_or_zero(a.A, row, a.stride_A, i - 1, a.L_a);
            x = (hi << r) | (lo >> (32u - r));
        }
        y = load_or_zero(a.B, row, a.stride_B, j, a.L_b);
    } else {
        // spill-add: C[j] += word of spill[run] at (run + 1) run_len (+1)
        x = load_or_zero(a.A, row, a.stride_A, j, a.L_a);
        y = 0;
        const uint32_t q = sp.run.run_of(j), rem = j - q * sp.run.len;
        if (q >= 1 && rem < 2) {
            const uint64_t s = sp.spill[(size_t)row * sp.runs_per_row + (q - 1)];
            y = rem == 0 ? (uint32_t)s : (uint32_t)(s >> 32);
        }
    }
    if constexpr (OpTraits<K>::kSub) {
        return {x - y, (uint32_t)(x < y)};
    } else {
        const uint32_t d = x + y;
        return {d, (uint32_t)(d < x)};
    }
}

template <AddSubKind K>
__global__ void __launch_bounds__(256) addsub_thread_kernel(AddSubArgs a, SpillArgs sp) {
    const uint32_t row = blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= a.N) return;
    constexpr bool kSub = OpTraits<K>::kSub;
    uint32_t c = 0;
    uint32_t *out = a.C + (size_t)row * a.stride_C;
    for (uint32_t j = 0; j < a.L_c; ++j) {
        const Digit t = digit_at<K>(a, sp, row, j);
        const uint32_t r = kSub ? t.d - c : t.d + c;
        c = t.g | (c & (uint32_t)(kSub ? t.d == 0u : t.d == 0xffffffffu));
        out[j] = r;
    }
}

// One wave per chunk of SEG*64 limbs.  flags[chunk] = carry-out (bit 0) |
// all-propagate (bit 1), both for a carry-in of zero.
template <AddSubKind K, int SEG>
__global__ void __launch_bounds__(256) addsub_chunk_kernel(AddSubArgs a, SpillArgs sp,
                                                           uint32_t chunks_per_row,
                                                           uint64_t total_chunks, uint8_t *flags) {
    constexpr bool kSub = OpTraits<K>::kSub;
    const uint64_t wave = (uint64_t)blockIdx.x * (blockDim.x / kWave) + (threadIdx.x / kWave);
    if (wave >= total_chunks) return;
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t row = (uint32_t)(wave / chunks_per_row);
    const uint32_t chunk = (uint32_t)(wave - (uint64_t)row * chunks_per_row);
    const uint32_t base = chunk * (uint32_t)(SEG * kWave);

    uint32_t d[SEG];
    uint64_t G[SEG], P[SEG];
#pragma unroll
    for (int s = 0; s < SEG; ++s) {
        const uint32_t j = base + s * kWave + lane;
        const bool valid = j < a.L_c;
        Digit t = {0u, 0u};
        if (valid) t = digit_at<K>(a, sp, row, j);
        d[s] = t.d;
        G[s] = ballot64(valid && t.g);
        P[s] = ballot64(valid && (kSub ? t.d == 0u : t.d == 0xffffffffu));
    }
    uint32_t cin = 0;
    bool all_prop = true;
    uint32_t *out = a.C + (size_t)row * a.stride_C;
#pragma unroll
    for (int s = 0; s < SEG; ++s) {
        uint32_t cout;
        const uint64_t cm = resolve_carries(G[s], P[s], cin, &cout);
        const uint32_t bit = (uint32_t)(cm >> lane) & 1u;
        const uint32_t j = base + s * kWave + lane;
        if (j < a.L_c) out[j] = kSub ? d[s] - bit : d[s] + bit;
        all_prop = all_prop && (P[s] == ~0ull);
        cin = cout;
    }
    if (flags != nullptr && lane == 0) flags[wave] = (uint8_t)(cin | (all_prop ? 2u : 0u));
}

// One wave per chunk >= 1 of each row: carry-in by look-back over the
// flags, then an in-chunk ripple if the carry-in is 1.
template <bool kSub>
__global__ void __launch_bounds__(256) carry_fixup_kernel(uint32_t *C, uint32_t stride_C, uint32_t L_c,
                                                          uint32_t chunk_len, uint32_t chunks_per_row,
                                                          uint64_t total, const uint8_t *flags) {
    const uint64_t wave = (uint64_t)blockIdx.x * (blockDim.x / kWave) + (threadIdx.x / kWave);
    if (wave >= total) return;
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t per_row = chunks_per_row - 1;
    const uint32_t row = (uint32_t)(wave / per_row);
    const uint32_t chunk = 1u + (uint32_t)(wave - (uint64_t)row * per_row);
    const uint8_t *rf = flags + (size_t)row * chunks_per_row;

    uint32_t cin = 0;
    for (int64_t hi = (int64_t)chunk - 1; hi >= 0; hi -= kWave) {
        const int64_t k = hi - (int64_t)lane;
        const uint32_t f = (k >= 0) ? rf[k] : 0u;  // k < 0: start of row, carry-in 0
        const uint64_t stop = ballot64((f & 2u) == 0u);
        if (stop != 0) {
            const int first = __builtin_ctzll(stop);
            cin = __shfl(f, first) & 1u;
            break;
        }
    }
    if (cin == 0) return;
    uint32_t *out = C + (size_t)row * stride_C;
    const uint32_t start = chunk * chunk_len;
    const uint32_t end = min(start + chunk_len, L_c);
    for (uint32_t seg = start; seg < end; seg += kWave) {
        const uint32_t j = seg + lane;
        const bool valid = j < end;
        const uint32_t v = valid ? out[j] : 0u;
        const bool prop = valid && (kSub ? v == 0u : v == 0xffffffffu);
        const uint64_t m = ballot64(!prop);
        const uint32_t first = m ? (uint32_t)__builtin_ctzll(m) : 64u;
        if (valid && lane < first) out[j] = kSub ? 0xffffffffu : 0u;
        if (valid && lane == first) out[j] = kSub ? v - 1u : v + 1u;
        if (m != 0) break;
    }
}

// Rows of 2..kRowWaves chunks of 1024 limbs run as one block per row (a wave
// per chunk, ROW): the waves' (carry out, all propagate) flags meet in LDS,
// so no second kernel settles the carries between chunks.  Short launches are
// bound by the time of a launch: one addition of 16000 limbs takes 4.4 us
// instead of 6.8 with carry_fixup_kernel behind it, 64 of them 5.8 instead of
// 6.8, and full chips gain too, by one reading of the flags (8192 rows of 4000
// limbs 73 instead of 78, 1024 additions of 12000 limbs 23.6 instead of 27.0).
// Sixteen waves are the largest block.  Of 13 waves and more two blocks fill a
// CU and wait on memory together, which costs the operations that read most:
// the shifts of more rows than CUs go by chunks there (1024 of 16384 limbs
// 34.6 instead of 42.8 us, 2048 of 14336 66.5 instead of 75; 256 of 14336
// still 8.6 by rows, 10.5 by chunks).
constexpr uint32_t kRowWaves = 16, kRowWavesMany = 12, kManyRows = 256;

// Which chunk a wave works on.
struct ChunkPos {
    uint32_t row, chunk;
    bool valid;
    uint64_t wave;
};
template <bool ROW>
__device__ __forceinline__ ChunkPos chunk_pos(uint32_t chunks_per_row, uint64_t total_chunks) {
    ChunkPos p;
    if constexpr (ROW) {
        p.row = blockIdx.x;
        p.chunk = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
        p.valid = true;
        p.wave = 0;
    } else {
        p.wave = (uint64_t)blockIdx.x * (256 / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
        p.valid = p.wave < total_chunks;
        p.row = (uint32_t)(p.wave / chunks_per_row);
        p.chunk = (uint32_t)(p.wave - (uint64_t)p.row * chunks_per_row);
    }
    return p;
}

// The carry into a wave of a ROW block from the waves below it: G, P are the
// masks of its kSeg groups of 256 limbs (four per lane, settled within it).
constexpr int kSeg = 4;
__device__ __forceinline__ uint32_t carry_into_wave(const uint64_t *G, const uint64_t *P, uint32_t lane) {
    __shared__ uint32_t flags[kRowWaves];
    uint32_t cout = 0;
    bool all_prop = true;
#pragma unroll
    for (int s = 0; s < kSeg; ++s) {
        (void)resolve_carries(G[s], P[s], cout, &cout);
        all_prop = all_prop && P[s] == ~0ull;
    }
    const uint32_t w = threadIdx.x / kWave;
    if (lane == 0) flags[w] = cout | (all_prop ? 2u : 0u);
    __syncthreads();
    uint32_t cin = 0;
    for (uint32_t i = 0; i < w; ++i) cin = (flags[i] & 1u) | ((flags[i] >> 1) & cin);
    return __builtin_amdgcn_readfirstlane(cin);
}

// The spill-add of NTT products of more than 512 limbs with four limbs per
// lane (16-byte loads and stores at any limb): one wave per chunk of 1024
// limbs of one row.  Each lane settles its four limbs for a carry-in of zero,
// the lanes' (generate, propagate) pairs go through one ballot resolution per
// 256 limbs, and the lane adds its carry-in.
template <bool ROW>
__global__ void __launch_bounds__(ROW ? kRowWaves * kWave : 256)
spill_add_vec_kernel(uint32_t *C, uint32_t stride_C, uint32_t L_c, SpillArgs sp, uint32_t chunks_per_row,
                     uint64_t total_chunks, uint8_t *flags) {
    const ChunkPos pos = chunk_pos<ROW>(chunks_per_row, total_chunks);
    if (!pos.valid) return;
    const uint32_t lane = threadIdx.x & (kWave - 1);
    uint32_t *out = C + (size_t)pos.row * stride_C;
    const uint64_t *rsp = sp.spill + (size_t)pos.row * sp.runs_per_row;
    const uint32_t base = pos.chunk * (uint32_t)(kSeg * 4 * kWave) + 4 * lane;
    uint32_t r[kSeg][4];
    uint64_t G[kSeg], P[kSeg];
#pragma unroll
    for (int s = 0; s < kSeg; ++s) {
        const uint32_t j0 = base + (uint32_t)s * (4 * kWave);
        if (j0 + 4 <= L_c) {
            const Quad v = *reinterpret_cast<const Quad *>(out + j0);
#pragma unroll
            for (int t = 0; t < 4; ++t) r[s][t] = v.w[t];
        } else {
#pragma unroll
            for (int t = 0; t < 4; ++t) r[s][t] = j0 + t < L_c ? out[j0 + t] : 0u;
        }
    }
    const auto settle = [&](int s) {
        const uint32_t j0 = base + (uint32_t)s * (4 * kWave);
        // runs are at least 8 limbs, so the four limbs meet at most one run's
        // start: at limb j0 + at (at = -1: its second limb is the first here)
        uint32_t q = sp.run.run_of(j0);
        const uint32_t rem = j0 - q * sp.run.len;
        int at = -(int)rem;
        if (rem > 1) {
            ++q;
            at += (int)sp.run.len;
        }
        uint64_t w = 0;
        if (q >= 1 && at < 4 && (int64_t)j0 + at < (int64_t)L_c) w = rsp[q - 1];
        uint32_t c = 0;
        bool ones = true;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint32_t j = j0 + t;
            const uint32_t y = t == at ? (uint32_t)w : t == at + 1 && j < L_c ? (uint32_t)(w >> 32) : 0u;
            const uint32_t d = r[s][t] + y;
            const uint32_t g = d < y ? 1u : 0u;
            r[s][t] = d + c;
            c = g | (c & (d == 0xffffffffu ? 1u : 0u));
            ones = ones && r[s][t] == 0xffffffffu && j < L_c;
        }
        G[s] = ballot64(j0 < L_c && c != 0);
        P[s] = ballot64(j0 < L_c && ones);
    };
    uint32_t cin = 0;
    if constexpr (ROW) {
#pragma unroll
        for (int s = 0; s < kSeg; ++s) settle(s);
        cin = carry_into_wave(G, P, lane);
    }
    bool all_prop = true;
#pragma unroll
    for (int s = 0; s < kSeg; ++s) {
        if constexpr (!ROW) settle(s);
        const uint32_t j0 = base + (uint32_t)s * (4 * kWave);
        uint32_t cout;
        const uint64_t cm = resolve_carries(G[s], P[s], cin, &cout);
        uint32_t ci = (uint32_t)(cm >> lane) & 1u;
        Quad q;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            q.w[t] = r[s][t] + ci;
            ci = ci & (r[s][t] == 0xffffffffu ? 1u : 0u);
        }
        if (j0 + 4 <= L_c) {
            *reinterpret_cast<Quad *>(out + j0) = q;
        } else {
#pragma unroll
            for (int t = 0; t < 4; ++t)
                if (j0 + t < L_c) out[j0 + t] = q.w[t];
        }
        all_prop = all_prop && (P[s] == ~0ull);
        cin = cout;
    }
    if (flags != nullptr && lane == 0) flags[pos.wave] = (uint8_t)(cin | (all_prop ? 2u : 0u));
}

// The assembly holding launch chunk g (assemblies in chunk order).
__device__ __forceinline__ RaggedAssembly assembly_of(const RaggedAssembly *as, uint32_t n, uint32_t g) {
    uint32_t lo = 0, hi = n;  // the last assembly with chunk0 <= g
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (as[mid].chunk0 <= g) lo = mid;
        else hi = mid;
    }
    return as[lo];
}

// Ragged assembly (RaggedAssembly): one wave per 1024-limb chunk, the
// layout of addsub_vec_kernel (flags per chunk for the fixup).  Limb x of C
// is piece i's staged word x - i s plus, when x - i s < S, piece i - 1's
// word x - i s + s, i = min(x / s, m - 1).  Bound by HBM; four limbs per lane
// and access where they share both pieces (256 ragged pairs with it and the
// copies of whole products: 30.9 -> 29.6 ms; a division and two loads per limb
// took 2.3 ms of them).
__global__ void __launch_bounds__(256) ragged_assemble_kernel(const uint32_t *staging, uint64_t stride,
                                                              const RaggedAssembly *as, uint32_t n,
                                                              uint32_t chunks, uint8_t *flags) {
    constexpr int kSeg = 4;  // 4 x 256 limbs per wave
    const uint32_t g = blockIdx.x * (256 / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    if (g >= chunks) return;
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const RaggedAssembly a = assembly_of(as, n, g);
    const uint32_t chunk = g - a.chunk0;
    uint32_t cin = 0;
    bool all_prop = true;
#pragma unroll
    for (int sg = 0; sg < kSeg; ++sg) {
        const uint32_t j0 = chunk * kAssembleChunk + (uint32_t)sg * (4 * kWave) + 4 * lane;
        uint32_t d[4], gen[4];
        // the lane's four limbs lie in one piece, and all or none of them in
        // the overlap with the piece below, but at the pieces' ends
        uint32_t i0, off0;
        bool below0;
        assembly_source(a, j0, &i0, &off0, &below0);
        if (j0 + 4 <= a.c && (i0 + 1 == a.m || off0 + 4 <= a.s) && (!below0 || off0 + 4 <= a.S)) {
            const Quad u = *reinterpret_cast<const Quad *>(staging + (size_t)(a.row0 + i0) * stride + off0);
            Quad v{};
            if (below0) v = *reinterpret_cast<const Quad *>(staging + (size_t)(a.row0 + i0 - 1) * stride + off0 + a.s);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                d[t] = u.w[t] + v.w[t];
                gen[t] = d[t] < u.w[t] ? 1u : 0u;
            }
        } else {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const uint32_t x = j0 + t;
                d[t] = 0;
                gen[t] = 0;
                if (x < a.c) {
                    uint32_t i, off;
                    bool below;
                    assembly_source(a, x, &i, &off, &below);
                    const uint32_t u = staging[(size_t)(a.row0 + i) * stride + off];
                    const uint32_t v = below ? staging[(size_t)(a.row0 + i - 1) * stride + off + a.s] : 0u;
                    d[t] = u + v;
                    gen[t] = d[t] < u ? 1u : 0u;
                }
            }
        }
        // the lane's four limbs for a carry-in of zero
        uint32_t r[4], c = 0;
        bool prop = true;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            r[t] = d[t] + c;
            c = gen[t] | (c & (d[t] == 0xffffffffu ? 1u : 0u));
            prop = prop && r[t] == 0xffffffffu && j0 + t < a.c;
        }
        const bool valid = j0 < a.c;
        const uint64_t G = ballot64(valid && c != 0), P = ballot64(valid && prop);
        uint32_t cout;
        const uint64_t cm = resolve_carries(G, P, cin, &cout);
        uint32_t ci = (uint32_t)(cm >> lane) & 1u;
        Quad q;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            q.w[t] = r[t] + ci;
            ci = ci & (r[t] == 0xffffffffu ? 1u : 0u);
        }
        if (j0 + 4 <= a.c) {
            *reinterpret_cast<Quad *>(a.C + j0) = q;
        } else {
#pragma unroll
            for (int t = 0; t < 4; ++t)
                if (j0 + t < a.c) a.C[j0 + t] = q.w[t];
        }
        all_prop = all_prop && (P == ~0ull);
        cin = cout;
    }
    if (lane == 0) flags[g] = (uint8_t)(cin | (all_prop ? 2u : 0u));
}

// One wave per chunk >= 1 of each assembly: carry-in by look-back over the
// assembly's flags, then an in-chunk ripple if it is 1 (carry_fixup_kernel
// over ragged rows).
__global__ void __launch_bounds__(256) ragged_assembly_fixup_kernel(const RaggedAssembly *as, uint32_t n,
                                                                    uint32_t chunks, const uint8_t *flags) {
    const uint32_t g = blockIdx.x * (256 / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    if (g >= chunks) return;
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const RaggedAssembly a = assembly_of(as, n, g);
    const uint32_t chunk = g - a.chunk0;
    if (chunk == 0) return;
    const uint8_t *rf = flags + a.chunk0;
    uint32_t cin = 0;
    for (int64_t hi = (int64_t)chunk - 1; hi >= 0; hi -= kWave) {
        const int64_t k = hi - (int64_t)lane;
        const uint32_t f = (k >= 0) ? rf[k] : 0u;  // k < 0: start of the assembly, carry-in 0
        const uint64_t stop = ballot64((f & 2u) == 0u);
        if (stop != 0) {
            cin = __shfl(f, __builtin_ctzll(stop)) & 1u;
            break;
        }
    }
    if (cin == 0) return;
    const uint32_t start = chunk * kAssembleChunk, end = min(start + kAssembleChunk, a.c);
    for (uint32_t seg = start; seg < end; seg += kWave) {
        const uint32_t j = seg + lane;
        const bool valid = j < end;
        const uint32_t v = valid ? a.C[j] : 0u;
        const uint64_t m = ballot64(!(valid && v == 0xffffffffu));
        const uint32_t first = m ? (uint32_t)__builtin_ctzll(m) : 64u;
        if (valid && lane < first) a.C[j] = 0u;
        if (valid && lane == first) a.C[j] = v + 1u;
        if (m != 0) break;
    }
}

// Four limbs x[0..4) of the row r from limb j0 on (zero outside [0, L)).
__device__ __forceinline__ void load4(const uint32_t *r, int64_t j0, uint32_t L, uint32_t *x) {
    if (j0 >= 0 && j0 + 4 <= (int64_t)L) {
        const Quad v = *reinterpret_cast<const Quad *>(r + j0);
#pragma unroll
        for (int t = 0; t < 4; ++t) x[t] = v.w[t];
    } else {
#pragma unroll
        for (int t = 0; t < 4; ++t) x[t] = (j0 + t >= 0 && j0 + t < (int64_t)L) ? r[j0 + t] : 0u;
    }
}

// The ops on rows of more than 512 limbs, four limbs per lane: one wave per
// chunk of 1024 limbs of one row (up to 16 chunks meet in one block,
// carry_fixup_kernel completes longer rows).
// Bound by HBM; the 16-byte accesses start at any limb, so row strides and
// shifts need no alignment (R = (R1 << s) - R2 over 512 rows of 128249 limbs:
// 271 us with a limb per lane, 158 us this way).  The shifted operand's limbs
// lie at any offset from the others': as one limb and four (QUAD) well inside
// the last cache, as five limbs beyond (64 rows of 2^20 limbs in
// 16-byte aligned rows 159 / 150 us, 4096 of 10240 100 / 95; 64 of 128249,
// 98 MB, 19.0 / 20.2; 30000 of 700, 252 MB, 44.0 / 39.0).
constexpr uint64_t kShiftQuadBytes = 160ull << 20;
template <AddSubKind K, bool ROW, bool QUAD>
__global__ void __launch_bounds__(ROW ? kRowWaves * kWave : 256)
addsub_vec_kernel(AddSubArgs a, uint32_t chunks_per_row, uint64_t total_chunks, uint8_t *flags) {
    constexpr bool kSub = OpTraits<K>::kSub;
    constexpr bool kShift = K == AddSubKind::ShiftAdd || K == AddSubKind::ShiftSub;
    const ChunkPos pos = chunk_pos<ROW>(chunks_per_row, total_chunks);
    if (!pos.valid) return;
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t row = pos.row;
    uint32_t *out = a.C + (size_t)row * a.stride_C;
    const uint32_t *ra = a.A + (size_t)row * a.stride_A, *rb = a.B + (size_t)row * a.stride_B;
    const int64_t ws = kShift ? (int64_t)(a.shift >> 5) : 0;
    const uint32_t bs = kShift ? (a.shift & 31u) : 0u;
    const int64_t base = (int64_t)pos.chunk * (kSeg * 4 * kWave);
    uint32_t d[kSeg][4], g[kSeg][4];
#pragma unroll
    for (int s = 0; s < kSeg; ++s) {
        const int64_t j0 = base + s * (4 * kWave) + 4 * (int64_t)lane;
        uint32_t x[4], y[4];
        if constexpr (kShift) {
            // x_t = (A << shift) at limb j0 + t: A[i] << bs | A[i - 1] >> (32 - bs), i = j0 + t - ws
            uint32_t w[5];
            const int64_t i = j0 - ws - 1;
            w[0] = (i >= 0 && i < (int64_t)a.L_a) ? ra[i] : 0u;
            if constexpr (QUAD) {
                load4(ra, i + 1, a.L_a, w + 1);
            } else {
#pragma unroll
                for (int t = 1; t < 5; ++t) w[t] = (i + t >= 0 && i + t < (int64_t)a.L_a) ? ra[i + t] : 0u;
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) x[t] = bs ? (w[t + 1] << bs) | (w[t] >> (32u - bs)) : w[t + 1];
        } else if constexpr (K == AddSubKind::MulSmall) {
            // x: low words of the limb products, y: high words of the ones below
            const uint32_t below = j0 > 0 && j0 <= (int64_t)a.L_a ? ra[j0 - 1] : 0u;
            load4(ra, j0, a.L_a, x);
            y[0] = __umulhi(below, a.scalar);
#pragma unroll
            for (int t = 1; t < 4; ++t) y[t] = __umulhi(x[t - 1], a.scalar);
#pragma unroll
            for (int t = 0; t < 4; ++t) x[t] *= a.scalar;
        } else {
            load4(ra, j0, a.L_a, x);
        }
        if constexpr (K == AddSubKind::AddSmall || K == AddSubKind::SubSmall) {
            y[0] = j0 == 0 ? a.scalar : 0u;
            y[1] = y[2] = y[3] = 0u;
        } else if constexpr (K != AddSubKind::MulSmall) {
            load4(rb, j0, a.L_b, y);
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            d[s][t] = kSub ? x[t] - y[t] : x[t] + y[t];
            g[s][t] = kSub ? (x[t] < y[t] ? 1u : 0u) : (d[s][t] < x[t] ? 1u : 0u);
        }
    }
    constexpr int kHeld = ROW ? kSeg : 1;  // groups settled before the first is stored
    uint32_t r[kHeld][4];
    uint64_t G[kHeld], P[kHeld];
    const auto settle = [&](int s, int h) {
        // the lane's four limbs for a carry-in of zero
        const int64_t j0 = base + s * (4 * kWave) + 4 * (int64_t)lane;
        uint32_t c = 0;
        bool prop = true;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            r[h][t] = kSub ? d[s][t] - c : d[s][t] + c;
            c = g[s][t] | (c & (kSub ? (d[s][t] == 0u ? 1u : 0u) : (d[s][t] == 0xffffffffu ? 1u : 0u)));
            prop = prop && (kSub ? r[h][t] == 0u : r[h][t] == 0xffffffffu) && j0 + t < (int64_t)a.L_c;
        }
        const bool valid = j0 < (int64_t)a.L_c;
        G[h] = ballot64(valid && c != 0);
        P[h] = ballot64(valid && prop);
    };
    uint32_t cin = 0;
    if constexpr (ROW) {
#pragma unroll
        for (int s = 0; s < kSeg; ++s) settle(s, s);
        cin = carry_into_wave(G, P, lane);
    }
    bool all_prop = true;
#pragma unroll
    for (int s = 0; s < kSeg; ++s) {
        const int h = ROW ? s : 0;
        if constexpr (!ROW) settle(s, 0);
        const int64_t j0 = base + s * (4 * kWave) + 4 * (int64_t)lane;
        uint32_t cout;
        const uint64_t cm = resolve_carries(G[h], P[h], cin, &cout);
        uint32_t ci = (uint32_t)(cm >> lane) & 1u;
        Quad q;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            q.w[t] = kSub ? r[h][t] - ci : r[h][t] + ci;
            ci = ci & (kSub ? (r[h][t] == 0u ? 1u : 0u) : (r[h][t] == 0xffffffffu ? 1u : 0u));
        }
        if (j0 + 4 <= (int64_t)a.L_c) {
            *reinterpret_cast<Quad *>(out + j0) = q;
        } else {
#pragma unroll
            for (int t = 0; t < 4; ++t)
                if (j0 + t < (int64_t)a.L_c) out[j0 + t] = q.w[t];
        }
        all_prop = all_prop && (P[h] == ~0ull);
        cin = cout;
    }
    if (flags != nullptr && lane == 0) flags[pos.wave] = (uint8_t)(cin | (all_prop ? 2u : 0u));
}

struct ChunkPlan {
    bool thread_rows;
    int seg;
    uint32_t chunk_len;
    uint32_t chunks_per_row;
};

ChunkPlan plan_for(uint32_t L_c) {
    ChunkPlan p{};
    if (L_c <= kThreadRowMax) {
        p.thread_rows = true;
        p.seg = 0;
        p.chunk_len = L_c;
        p.chunks_per_row = 1;
        return p;
    }
    int seg = 1;
    while (seg < 16 && (uint64_t)seg * kWave < L_c) seg *= 2;
    p.thread_rows = false;
    p.seg = seg;
    p.chunk_len = (uint32_t)seg * kWave;
    p.chunks_per_row = ceil_div(L_c, p.chunk_len);
    return p;
}

template <AddSubKind K>
hipError_t run_addsub(const AddSubArgs &a, const SpillArgs &sp, uint8_t *flags, hipStream_t stream) {
    if (a.N == 0 || a.L_c == 0) return hipSuccess;
    const ChunkPlan p = plan_for(a.L_c);
    if (p.thread_rows) {
        const uint32_t blocks = ceil_div(a.N, 256);
        hipLaunchKernelGGL(addsub_thread_kernel<K>, dim3(blocks), dim3(256), 0, stream, a, sp);
        return hipGetLastError();
    }
    const uint64_t total = (uint64_t)a.N * p.chunks_per_row;
    constexpr bool kShift = K == AddSubKind::ShiftAdd || K == AddSubKind::ShiftSub;
    // one block per row where a row's chunks fit it
    const bool rows =
        p.chunks_per_row > 1 && p.chunks_per_row <= (kShift && a.N > kManyRows ? kRowWavesMany : kRowWaves);
    const bool quad = !kShift || 4ull * a.N * ((uint64_t)a.L_a + a.L_b + a.L_c) <= kShiftQuadBytes;
    const bool need_fix = p.chunks_per_row > 1 && !rows;
    if (p.chunks_per_row > 1 && flags == nullptr) return hipErrorInvalidValue;
    const uint64_t blocks = rows ? a.N : ceil_div64(total, 4);
    if (blocks > 0x7fffffffull) return hipErrorInvalidValue;
    uint8_t *fl = need_fix ? flags : nullptr;
    const dim3 grid((uint32_t)blocks), block(rows ? p.chunks_per_row * kWave : 256u);
    const auto chunks = [&](auto seg) {
        hipLaunchKernelGGL((addsub_chunk_kernel<K, decltype(seg)::value>), grid, block, 0, stream, a, sp,
                           p.chunks_per_row, total, fl);
    };
    switch (p.seg) {
        case 1: chunks(std::integral_constant<int, 1>{}); break;
        case 2: chunks(std::integral_constant<int, 2>{}); break;
        case 4: chunks(std::integral_constant<int, 4>{}); break;
        case 8: chunks(std::integral_constant<int, 8>{}); break;
        default:
            // in place is fine: a lane reads the limbs it writes first
            if constexpr (K == AddSubKind::SpillAdd) {
                const auto k = rows ? spill_add_vec_kernel<true> : spill_add_vec_kernel<false>;
                hipLaunchKernelGGL(k, grid, block, 0, stream, a.C, a.stride_C, a.L_c, sp, p.chunks_per_row, total, fl);
            } else {
                const auto k = !quad ? (rows ? addsub_vec_kernel<K, true, !kShift> : addsub_vec_kernel<K, false, !kShift>)
                                     : (rows ? addsub_vec_kernel<K, true, true> : addsub_vec_kernel<K, false, true>);
                hipLaunchKernelGGL(k, grid, block, 0, stream, a, p.chunks_per_row, total, fl);
            }
    }
    GPUPI_RETURN_IF(hipGetLastError());
    if (need_fix) {
        const uint64_t fix_total = (uint64_t)a.N * (p.chunks_per_row - 1);
        const uint64_t fblocks = ceil_div64(fix_total, 4);
        if (fblocks > 0x7fffffffull) return hipErrorInvalidValue;
        hipLaunchKernelGGL(carry_fixup_kernel<OpTraits<K>::kSub>, dim3((uint32_t)fblocks), dim3(256), 0,
                           stream, a.C, a.stride_C, a.L_c, p.chunk_len, p.chunks_per_row, fix_total,
                           (const uint8_t *)flags);
        GPUPI_RETURN_IF(hipGetLastError());
    }
    return hipSuccess;
}

}  // namespace

size_t carry_flags_bytes(uint32_t N, uint32_t L_c) {
    const ChunkPlan p = plan_for(L_c);
    if (p.chunks_per_row <= 1) return 0;
    return (size_t)N * p.chunks_per_row;
}

hipError_t launch_addsub(const AddSubArgs &a, uint8_t *flags, hipStream_t stream) {
    const SpillArgs sp{};
    switch (a.kind) {
        case AddSubKind::Add: return run_addsub<AddSubKind::Add>(a, sp, flags, stream);
        case AddSubKind::Sub: return run_addsub<AddSubKind::Sub>(a, sp, flags, stream);
        case AddSubKind::AddSmall: return run_addsub<AddSubKind::AddSmall>(a, sp, flags, stream);
        case AddSubKind::SubSmall: return run_addsub<AddSubKind::SubSmall>(a, sp, flags, stream);
        case AddSubKind::MulSmall: return run_addsub<AddSubKind::MulSmall>(a, sp, flags, stream);
        case AddSubKind::ShiftAdd: return run_addsub<AddSubKind::ShiftAdd>(a, sp, flags, stream);
        case AddSubKind::ShiftSub: return run_addsub<AddSubKind::ShiftSub>(a, sp, flags, stream);
        case AddSubKind::SpillAdd: break;  // needs spill words: launch_add_spills
    }
    return hipErrorInvalidValue;
}

hipError_t launch_add_spills(uint32_t *C, const uint64_t *spill, uint32_t N, uint32_t L_c,
                             uint32_t stride_C, uint32_t run_len, uint32_t runs_per_row,
                             uint8_t *flags, hipStream_t stream) {
    AddSubArgs a{};
    a.kind = AddSubKind::SpillAdd;
    a.A = C;
    a.C = C;
    a.N = N;
    a.L_a = L_c;
    a.L_c = L_c;
    a.stride_A = stride_C;
    a.stride_C = stride_C;
    if (run_len < 8 || L_c >= 0x80000000u) return hipErrorInvalidValue;
    const SpillArgs sp{spill, ntt::run_divisor(run_len), runs_per_row};
    return run_addsub<AddSubKind::SpillAdd>(a, sp, flags, stream);
}

hipError_t launch_ragged_assemble(const uint32_t *staging, uint64_t stride, const RaggedAssembly *as, uint32_t n,
                                  uint32_t chunks, uint8_t *flags, hipStream_t stream) {
    if (n == 0 || chunks == 0) return hipSuccess;
    if (staging == nullptr || as == nullptr || flags == nullptr) return hipErrorInvalidValue;
    const uint32_t blocks = (chunks + 3) / 4;
    hipLaunchKernelGGL(ragged_assemble_kernel, dim3(blocks), dim3(256), 0, stream, staging, stride, as, n, chunks, flags);
    GPUPI_RETURN_IF(hipGetLastError());
    hipLaunchKernelGGL(ragged_assembly_fixup_kernel, dim3(blocks), dim3(256), 0, stream, as, n, chunks,
                       (const uint8_t *)flags);
    return hipGetLastError();
}

}  // namespace gpupi

// ---------------------------------------------------------------------------
// C entry points (reference per-op headers); null stream, caller workspace.
// ---------------------------------------------------------------------------
using gpupi::AddSubArgs;
using gpupi::AddSubKind;

static void addsub_entry(AddSubKind kind, const uint32_t *A, const uint32_t *B, uint32_t scalar,
                         uint32_t shift, uint32_t *C, uint32_t *ws, uint32_t N, uint32_t L_a,
                         uint32_t L_b, uint32_t L_c, uint32_t sA, uint32_t sB, uint32_t sC) {
    AddSubArgs a{kind, A, B, C, scalar, shift, N, L_a, L_b, L_c, sA, sB, sC};
    (void)gpupi::launch_addsub(a, (uint8_t *)ws, 0);
}

extern "C" {

void batch_add_simple(uint32_t *A, uint32_t *B, uint32_t *C, uint32_t *workspace, uint32_t N,
                      uint32_t L_a, uint32_t L_b, uint32_t L_c, uint32_t stride_A,
                      uint32_t stride_B, uint32_t stride_C) {
    addsub_entry(AddSubKind::Add, A, B, 0, 0, C, workspace, N, L_a, L_b, L_c, stride_A, stride_B, stride_C);
}
size_t batch_add_simple_workspace_size(uint32_t N, uint32_t, uint32_t, uint32_t L_c) {
    return gpupi::carry_flags_bytes(N, L_c);
}

void batch_sub_simple(uint32_t *A, uint32_t *B, uint32_t *C, uint32_t *workspace, uint32_t N,
                      uint32_t L_a, uint32_t L_b, uint32_t L_c, uint32_t stride_A,
                      uint32_t stride_B, uint32_t stride_C) {
    addsub_entry(AddSubKind::Sub, A, B, 0, 0, C, workspace, N, L_a, L_b, L_c, stride_A, stride_B, stride_C);
}
size_t batch_sub_simple_workspace_size(uint32_t N, uint32_t, uint32_t, uint32_t L_c) {
    return gpupi::carry_flags_bytes(N, L_c);
}

void batch_add_small(const uint32_t *A, uint32_t B, uint32_t *C, uint32_t *workspace, uint32_t N,
                     uint32_t L_a, uint32_t L_c, uint32_t stride_A, uint32_t stride_C) {
    addsub_entry(AddSubKind::AddSmall, A, nullptr, B, 0, C, workspace, N, L_a, 0, L_c, stride_A, 0, stride_C);
}
size_t batch_add_small_workspace_size(uint32_t N, uint32_t, uint32_t L_c) {
    return gpupi::carry_flags_bytes(N, L_c);
}

void batch_sub_small(const uint32_t *A, uint32_t B, uint32_t *C, uint32_t *workspace, uint32_t N,
                     uint32_t L_a, uint32_t L_c, uint32_t stride_A, uint32_t stride_C) {
    addsub_entry(AddSubKind::SubSmall, A, nullptr, B, 0, C, workspace, N, L_a, 0, L_c, stride_A, 0, stride_C);
}
size_t batch_sub_small_workspace_size(uint32_t N, uint32_t, uint32_t L_c) {
    return gpupi::carry_flags_bytes(N, L_c);
}

void batch_mul_small(const uint32_t *A, uint32_t B, uint32_t *C, uint32_t *workspace, uint32_t N,
                     uint32_t L_a, uint32_t L_c, uint32_t stride_A, uint32_t stride_C) {
    addsub_entry(AddSubKind::MulSmall, A, nullptr, B, 0, C, workspace, N, L_a, 0, L_c, stride_A, 0, stride_C);
}
size_t batch_mul_small_workspace_size(uint32_t N, uint32_t, uint32_t L_c) {
    return gpupi::carry_flags_bytes(N, L_c);
}

void batch_shift_add_simple(const uint32_t *A, const uint32_t *B, uint32_t *C, uint32_t *workspace,
                            uint32_t shift, uint32_t N, uint32_t L_a, uint32_t L_b, uint32_t L_c,
                            uint32_t stride_A, uint32_t stride_B, uint32_t stride_C) {
    addsub_entry(AddSubKind::ShiftAdd, A, B, 0, shift, C, workspace, N, L_a, L_b, L_c, stride_A, stride_B, stride_C);
}
size_t batch_shift_add_simple_workspace_size(uint32_t N, uint32_t, uint32_t, uint32_t L_c, uint32_t) {
    return gpupi::carry_flags_bytes(N, L_c);
}

void batch_shift_sub_simple(const uint32_t *A, const uint32_t *B, uint32_t *C, uint32_t *workspace,
                            uint32_t shift, uint32_t N, uint32_t L_a, uint32_t L_b, uint32_t L_c,
                            uint32_t stride_A, uint32_t stride_B, uint32_t stride_C) {
    addsub_entry(AddSubKind::ShiftSub, A, B, 0, shift, C, workspace, N, L_a, L_b, L_c, stride_A, stride_B, stride_C);
}
size_t batch_shift_sub_simple_workspace_size(uint32_t N, uint32_t, uint32_t, uint32_t L_c, uint32_t) {
    return gpupi::carry_flags_bytes(N, L_c);
}

}  // extern "C"
