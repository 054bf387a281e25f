// Prompt-sized products over the canonical int4 operands: y[M,N] = x[M,K] . dequant(W)^T for more activation
// rows than the GEMV launches take (the prompt pass, vrl/models/families/janus_pro/policy.py:640-672, and the
// forward of a training replay, policy.py:419-424, which keeps gate||up itself beside the fused result).
//
// One launch covers up to GEMM_MAX problems (q|k|v of a layer; gate|up with the SiLU epilogue is one problem).
// A workgroup owns BM activation rows x BN weight rows and walks K in chunks of KC.  Both operands reach LDS by
// direct loads (no registers in flight): the activations as bf16, the weights as the packed words, a quarter of
// the bytes.  Every wave reads its own weight rows from LDS, rebuilds the exactly rounded bf16 weights in
// registers (as the GEMV kernels do) and feeds them to v_mfma_f32_16x16x32_bf16 as the A operand, the
// activations as the B operand: a lane then holds four neighbouring output columns of one row.  No bf16 copy of
// the weight is ever written.
//
// Layout in LDS: activation rows are KC bf16 with their 16-byte pieces permuted within the row (piece j of row r
// sits at j ^ f(r)), so that the 16 rows a fragment read touches fall on different banks; the direct loads
// permute the global addresses instead of the LDS side, which they fill in lane order.  Scales and zero-points of
// all of K are laid down once per workgroup as one word each.
#include <atomic>
#include <type_traits>

#include "canonical.hpp"
#include "host_checks.hpp"

namespace {

typedef __attribute__((ext_vector_type(2))) uint32_t u32x2_t;

constexpr int GEMM_MAX = 8;

struct GemmRec {
    const uint16_t *x;
    const uint32_t *qweight;
    const uint16_t *scales;
    const uint32_t *qzeros;
    uint16_t *y;
    uint16_t *product;   // fused records: [M, N] before SiLU, or null
    int32_t M, N;        // N: weight rows (gate||up: both halves)
    int32_t tile_begin;  // first tile of the record in the launch
    int32_t mtiles;
};
struct GemmArgs {
    GemmRec recs[GEMM_MAX];
    int32_t n, K, gshift, tiles;   // every record shares K and the group size 1 << gshift
    int32_t wave_flags;            // there is LDS behind the table for a word per wave
};

// One packed word -> eight exactly rounded bf16 weights in k order, in instructions that can be issued between MFMAs, pair by
// pair: (q - z) s as fma(q', s', c) with an exact product and an exact c, so that the conversion is the one rounding of the
// contract.  Two forms.  Plain, 17 instructions: a nibble under the exponent of 1024 is the half-precision value 1024 + q, or
// 1024 + 16 q where it sits four bits further up, which the mixed fma takes as it is.  Its c, -(1024 + z) s, is finite for
// scales below 2^117; a workgroup that meets a larger one (an infinity, a NaN) takes the wide form for all of its tile:
// the byte converter's float(q) and c = -z s, 23 instructions.  A prompt of 512 rows, four layers: 414 us with the wide form
// everywhere, 399 with the plain one.
struct ScaleZero { float s, c, s16, c16; };
struct Nibbles { uint32_t h[4]; };
struct Masks { uint32_t low, high, bias; };
constexpr uint32_t WIDE_SCALE = 0x7A00u;   // bf16 bits of 2^117

__device__ __forceinline__ float half_of(uint32_t v, int i) {
    typedef __attribute__((ext_vector_type(2))) _Float16 half2_t;
    return (float)__builtin_bit_cast(half2_t, v)[i];
}

template <bool WIDE>
__device__ __forceinline__ ScaleZero scale_zero(uint32_t meta) {   // (scale bits << 16) | half-precision 1024 + zero
    const float s = bf16_bits_to_f32(meta >> 16);
    if constexpr (WIDE) return {s, -s * (float)(meta & 0xFFu), 0.0f, 0.0f};
    const float c = -half_of(meta, 0) * s;
    return {s, c, s * 0.0625f, __builtin_fmaf(960.0f, s, c)};
}

template <bool WIDE>
__device__ __forceinline__ Nibbles nibbles(uint32_t v, const Masks &m) {
    if constexpr (WIDE) {
        Nibbles b{{v & 0x0F0F0F0Fu, (v >> 4) & 0x0F0F0F0Fu, 0u, 0u}};
        asm("" : "+v"(b.h[0]), "+v"(b.h[1]));   // or the compiler takes every nibble out by itself: 28 instructions
        return b;
    }
    const uint32_t w = v >> 8;
    Nibbles b{{(v & m.low) | m.bias, (v & m.high) | m.bias, (w & m.low) | m.bias, (w & m.high) | m.bias}};
    asm("" : "+v"(b.h[0]), "+v"(b.h[1]), "+v"(b.h[2]), "+v"(b.h[3]));   // or half of the and-ors come apart again
    return b;
}

template <bool WIDE>
__device__ __forceinline__ uint32_t dequant_pair(const Nibbles &b, int i, const ScaleZero &c) {
    if constexpr (WIDE)
        return pack_bf16_rne(__builtin_fmaf((float)((b.h[0] >> (8 * i)) & 0xFFu), c.s, c.c),
                             __builtin_fmaf((float)((b.h[1] >> (8 * i)) & 0xFFu), c.s, c.c));
    return pack_bf16_rne(__builtin_fmaf(half_of(b.h[i % 2 * 2], i / 2), c.s, c.c),
                         __builtin_fmaf(half_of(b.h[i % 2 * 2 + 1], i / 2), c.s16, c.c16));
}

// WM x WN x WK waves share a tile: WM and WN split its rows and columns, WK the k of every chunk (their partial
// tiles meet in LDS at the end).  A wave owns MB x NB blocks of 16 x 16.  S chunks of KC k are in LDS at a time.
// AHEAD: a chunk's barrier stands inside the last MFMA step of the chunk before it, whose remaining products cover the
// round trip for the next words and activations and the rebuild of the first weights; otherwise at the chunk's start.
// Tiles of 128 rows and more have the products for that: 1664 rows, K = 2048, gate|up 88.6 -> 82.2 us, q|k|v 54.7 -> 50.3,
// down_proj 51.0 -> 46.0, of which the plain rebuild and precise waits give 5.2, 3.0 and 2.4.  With 64 rows it costs 5 %.
template <int WM_, int WN_, int WK_, int MB_, int NB_, int KC_, int S_, bool AHEAD_>
struct GemmCfg {
    static constexpr int WM = WM_, WN = WN_, WK = WK_, MB = MB_, NB = NB_, KC = KC_, S = S_;
    static constexpr bool AHEAD = AHEAD_;
    static constexpr int WAVES = WM * WN * WK, THREADS = WAVES * WAVE;
    static constexpr int BM = 16 * MB * WM, BN = 16 * NB * WN;
    static constexpr int T = KC / 32 / WK;                // MFMA steps per wave and chunk = packed words a lane reads per row
    static constexpr int XP = KC / 8, WP = KC / 32;       // 16-byte pieces of a staged activation row, of a weight row
    static constexpr int X_BYTES = BM * KC * 2, W_BYTES = BN * KC / 2;
    // direct loads per wave and chunk (where the words are fewer loads than waves, waves repeat each other's)
    static constexpr int W_UNITS = W_BYTES / 1024;
    static constexpr int X_LOADS = X_BYTES / 1024 / WAVES, W_LOADS = W_UNITS < WAVES ? 1 : W_UNITS / WAVES;
    static constexpr int STAGE = X_BYTES + W_BYTES;
    static_assert(X_BYTES % (1024 * WAVES) == 0 && (WAVES % W_UNITS == 0 || W_UNITS % WAVES == 0), "whole direct loads");
    static_assert(T == 2 || T == 4, "a lane's words are one 8- or 16-byte read, inside one group of 32 k");
    static_assert(MB % WK == 0 || WK % MB == 0, "the waves that split K finish a share of the row blocks each, or none");
    static constexpr size_t PARTIAL = WK > 1 ? (size_t)WAVES * MB * NB * 1024 : 0;   // over the stages, once they are done
    static constexpr size_t lds(int groups) {
        const size_t loop = (size_t)S * STAGE + (size_t)BN * groups * 4;
        return loop > PARTIAL ? loop : PARTIAL;
    }
};

// Piece j of staged row r sits at j ^ f(r).  LDS has 64 banks; a 16-byte read goes in four turns of sixteen lanes,
// lanes {0-3, 12-15, 20-27} and {4-11, 16-19, 28-31} of each half of the wave, an 8-byte read in two turns of half
// a wave.  f is chosen per row length (P pieces) and per distance T of two lane quarters' pieces so that a turn's
// lanes cover the banks once: where a turn mixes two quarters, flipping the piece bit that tells them apart must
// not change which of the two sets a row belongs to (its bits 2 and 3).  Half of the LDS cycles were conflicts
// with f(r) = r & 15.
template <int P, int T>
__device__ __forceinline__ int activation_swizzle(int r) {
    if (P == 8) return (r >> 1 & 4) | (r & 2) | (r >> 2 & 1);
    return T == 4 ? (r & 10) | (r & 1) << 2 | (r >> 2 & 1) : r & 15;
}
template <int P>
__device__ __forceinline__ int weight_swizzle(int r) {
    return P == 2 ? r >> 3 & 1 : P == 4 ? -(r >> 2) & 3 : P == 8 ? r >> 1 & 7 : r & 15;
}

// The weight row behind local row r of column tile nt.  Fused records: a wave's first NB/2 blocks of 16 rows are
// gate rows, the others the up rows of the same columns.  Clamped: what lies past the end is never stored.
template <class C, bool FUSED>
__device__ __forceinline__ int weight_row(int r, int nt, int N) {
    if (!FUSED) return min(nt * C::BN + r, N - 1);
    constexpr int HB = C::NB > 1 ? C::NB / 2 : 1;
    const int half = (r / (16 * HB)) & 1;
    const int col = nt * (C::BN / 2) + (r / (32 * HB)) * (16 * HB) + r % (16 * HB);
    return half * (N / 2) + min(col, N / 2 - 1);
}

template <class C, bool FUSED>
__global__ __launch_bounds__(C::THREADS, C::WAVES >= 8 || C::MB * C::NB >= 32 ? 2 : 1) void gemm_int4_kernel(GemmArgs args) {
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lc = lane & 15, kq = lane >> 4;
    const int wn = wave % C::WN, wm = wave / C::WN % C::WM, wk = wave / (C::WN * C::WM);

    // Consecutive workgroups go to the eight XCDs in turn: each XCD gets one contiguous range of tiles, walked in
    // bands of GROUP_M row tiles, so that what its L2 holds is read by several of its workgroups.
    constexpr int XCDS = 8, GROUP_M = 8;
    const int xcd = blockIdx.x % XCDS, per = args.tiles / XCDS, rest = args.tiles % XCDS;
    const int tile = xcd * per + min(xcd, rest) + blockIdx.x / XCDS;
    int ri = 0;
    for (int i = 1; i < args.n; ++i)
        if (tile >= args.recs[i].tile_begin) ri = i;
    const GemmRec p = args.recs[ri];
    const int K = args.K, kwords = K >> 3, groups = K >> args.gshift, zwords = (groups + 7) >> 3;
    const int out_cols = FUSED ? p.N / 2 : p.N;
    constexpr int COLS = FUSED ? C::BN / 2 : C::BN;
    int mt, nt;
    {
        const int local = tile - p.tile_begin, ntiles = (out_cols + COLS - 1) / COLS;
        const int band = local / (GROUP_M * ntiles), rows = min(GROUP_M, p.mtiles - band * GROUP_M);
        const int in = local - band * GROUP_M * ntiles;
        mt = band * GROUP_M + in % rows;
        nt = in / rows;
    }

    uint32_t *table = reinterpret_cast<uint32_t *>(smem + C::S * C::STAGE);

    // this wave's direct loads: byte offsets from the tile's first row and from the weight; a chunk is KC k further on
    const uint8_t *xbase = reinterpret_cast<const uint8_t *>(p.x + (long)mt * C::BM * K);
    const uint8_t *wbase = reinterpret_cast<const uint8_t *>(p.qweight);
    uint32_t xsrc[C::X_LOADS], wsrc[C::W_LOADS];
#pragma unroll
    for (int i = 0; i < C::X_LOADS; ++i) {
        const int at = (wave * C::X_LOADS + i) * 64 + lane;              // 16-byte piece of the staged tile
        const int r = at / C::XP, j = (at % C::XP) ^ activation_swizzle<C::XP, C::T>(r);
        xsrc[i] = (uint32_t)(min(r, p.M - 1 - mt * C::BM) * K + 8 * j) * 2u;
    }
#pragma unroll
    for (int i = 0; i < C::W_LOADS; ++i) {
        const int at = (wave * C::W_LOADS + i) % C::W_UNITS * 64 + lane;
        const int r = at / C::WP, j = (at % C::WP) ^ weight_swizzle<C::WP>(r);
        wsrc[i] = ((uint32_t)weight_row<C, FUSED>(r, nt, p.N) * (uint32_t)kwords + 4 * j) * 4u;   // below 4 GiB
    }
    const int chunks = K / C::KC;
    auto issue = [&](int chunk, int slot) {
        const long c = min(chunk, chunks - 1);   // past the end: a repeat nobody reads, so that every chunk counts alike
        const uint8_t *xc = xbase + c * (C::KC * 2), *wc = wbase + c * (C::KC / 2);
        uint8_t *xl = smem + slot * C::STAGE + wave * (C::X_LOADS * 1024);
        uint8_t *wl = smem + slot * C::STAGE + C::X_BYTES + wave * C::W_LOADS % C::W_UNITS * 1024;
#pragma unroll
        for (int i = 0; i < C::X_LOADS; ++i) dma16(xl + i * 1024, xc, xsrc[i]);
#pragma unroll
        for (int i = 0; i < C::W_LOADS; ++i) dma16(wl + i * 1024, wc, wsrc[i]);
    };

    // scales and zero-points of the tile's rows, (scale bits << 16) | zero, group-major
    bool wide_scales = args.wave_flags == 0;
    for (int idx = tid; idx < C::BN * groups; idx += C::THREADS) {
        const int r = idx / groups, g = idx - r * groups;
        const long row = weight_row<C, FUSED>(r, nt, p.N);
        const uint32_t sb = as_global(p.scales)[row * groups + g];
        const uint32_t z = ((gptr_cu32)(uintptr_t)p.qzeros)[row * zwords + (g >> 3)] >> (4 * (g & 7)) & 0xFu;
        table[g * C::BN + r] = (sb << 16) | (0x6400u + z);
        wide_scales |= (sb & 0x7FFFu) >= WIDE_SCALE;
    }
#pragma unroll
    for (int s = 0; s < C::S - !C::AHEAD; ++s) issue(s, s);
    if (args.wave_flags) {   // (the barrier leaves the direct loads in flight)
        uint32_t *const flags = table + C::BN * groups;
        const bool any = __ballot(wide_scales) != 0;
        if (lane == 0) flags[wave] = any;
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        wide_scales = __ballot(flags[lane % C::WAVES] != 0) != 0;
    }

    f32x4_t acc[C::MB][C::NB];
#pragma unroll
    for (int b = 0; b < C::MB; ++b)
#pragma unroll
        for (int n = 0; n < C::NB; ++n) acc[b][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    const int xrow0 = wm * 16 * C::MB + lc, wrow0 = wn * 16 * C::NB + lc;
    // rows of the other blocks differ by multiples of 16, which no swizzle sees
    const int xswz = activation_swizzle<C::XP, C::T>(lc), xpiece = 4 * C::T * wk + C::T * kq;
    const int wbyte = 16 * C::T * wk + 4 * C::T * kq;
    const int woff = wrow0 * (C::KC / 2) + (((wbyte >> 4) ^ weight_swizzle<C::WP>(lc)) << 4) + (wbyte & 15);
    const int xoff = xrow0 * (C::KC * 2);
    Masks masks{0x000F000Fu, 0x00F000F0u, 0x64006400u};
    asm volatile("" : "+s"(masks.low), "+s"(masks.high));   // one scalar register and no literal per and-or
    asm volatile("" : "+v"(masks.bias));
    auto walk = [&](auto form) {
        constexpr bool WIDE = decltype(form)::value;
        uint32_t w[C::NB][C::T];
        ScaleZero sz[C::NB];
        bf16x8_t xb[C::MB];
        u32x4_t wa[C::NB];
        auto words = [&](int chunk, int slot) {
            const uint8_t *ws = smem + slot * C::STAGE + C::X_BYTES + woff;
            const int g = (min(chunk, chunks - 1) * C::KC + 32 * C::T * wk + 8 * C::T * kq) >> args.gshift;
#pragma unroll
            for (int n = 0; n < C::NB; ++n) {
                typedef __attribute__((ext_vector_type(C::T))) uint32_t words_t;
                const words_t v = *reinterpret_cast<const words_t *>(ws + n * (16 * C::KC / 2));
#pragma unroll
                for (int t = 0; t < C::T; ++t) w[n][t] = v[t];
                sz[n] = scale_zero<WIDE>(table[g * C::BN + wrow0 + 16 * n]);
            }
        };
        auto fetch = [&](int slot, int t, int b) {
            return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t *>(
                smem + slot * C::STAGE + xoff + b * (16 * C::KC * 2) + (((xpiece + t) ^ xswz) << 4)));
        };
        auto first_step = [&](int chunk, int slot) {
            words(chunk, slot);
#pragma unroll
            for (int b = 0; b < C::MB; ++b) xb[b] = fetch(slot, 0, b);
            if (!C::AHEAD) issue(chunk + C::S - 1, slot == 0 ? C::S - 1 : slot - 1);
#pragma unroll
            for (int n = 0; n < C::NB; ++n) {
                const Nibbles q = nibbles<WIDE>(w[n][0], masks);
#pragma unroll
                for (int i = 0; i < 4; ++i) wa[n][i] = dequant_pair<WIDE>(q, i, sz[n]);
            }
        };
        // the next chunk has arrived for every wave, and every wave is done with the slot that is filled next
        auto arrive = [&]() {
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"i"((C::S - 2) * (C::X_LOADS + C::W_LOADS)) : "memory");
        };
        if (C::AHEAD) {
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"i"((C::S - 1) * (C::X_LOADS + C::W_LOADS)) : "memory");
            first_step(0, 0);
        }
        int slot = 0;
        for (int c = 0; c < chunks; ++c) {
            if (!C::AHEAD) {
                arrive();
                first_step(c, slot);
            }
            const int following = slot + 1 == C::S ? 0 : slot + 1;
            // Row block by row block: its MFMAs, the request for its next activations, a share of the next step's
            // weights.  The scheduler is kept to this order: by its own it requests activations right before they are
            // used and rebuilds weights in one piece.
#pragma unroll
            for (int t = 0; t < C::T; ++t) {
                const bool last = t == C::T - 1;
                constexpr int PAIRS = 4 * C::NB;
                constexpr int HOLD = C::MB >= 4 ? C::MB / 4 : 1;             // row blocks ahead of the chunk's barrier
                constexpr int AFTER = C::MB >= 4 ? HOLD + C::MB / 4 : HOLD;  // and ahead of the next words' use
                const int from = last ? AFTER : 0;
                Nibbles q[C::NB];
                u32x4_t next[C::NB];
#pragma unroll
                for (int b = 0; b < C::MB; ++b) {
#pragma unroll
                    for (int n = 0; n < C::NB; ++n)
                        acc[b][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wa[n]), xb[b],
                                                                            acc[b][n], 0, 0, 0);
                    // (the next activations take the registers of those just used)
                    if constexpr (C::MB > 2) __builtin_amdgcn_sched_barrier(2 | 4);   // vector and scalar arithmetic may cross
                    if (!last) {
                        xb[b] = fetch(slot, t + 1, b);
                    } else if (C::AHEAD && b == HOLD - 1) {
                        // All of chunk c is in registers, for every wave, and all of chunk c + 1 has arrived: the rest of
                        // this step's products cover the round trip for its first words and their rebuild.
                        arrive();
                        words(c + 1, following);
                        issue(c + C::S, slot);
#pragma unroll
                        for (int e = 0; e < HOLD; ++e) xb[e] = fetch(following, 0, e);
                    } else if (C::AHEAD && b >= HOLD) {
                        xb[b] = fetch(following, 0, b);
                    }
                    if (!last || C::AHEAD) {
#pragma unroll
                        for (int pair = max(b - from, 0) * PAIRS / (C::MB - from); pair < max(b + 1 - from, 0) * PAIRS / (C::MB - from); ++pair) {
                            const int n = pair / 4, i = pair % 4;
                            if (i == 0) q[n] = nibbles<WIDE>(w[n][last ? 0 : t + 1], masks);
                            next[n][i] = dequant_pair<WIDE>(q[n], i, sz[n]);
                        }
                    }
                    if constexpr (C::MB > 2) __builtin_amdgcn_sched_barrier(0);
                }
                if (!last || C::AHEAD)
#pragma unroll
                    for (int n = 0; n < C::NB; ++n) wa[n] = next[n];
            }
            slot = following;
        }
    };
    if (wide_scales)   // workgroup-uniform
        walk(std::true_type{});
    else
        walk(std::false_type{});
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the repeats must not land in another workgroup's LDS

    int b0 = 0;
    constexpr int OWN = C::MB > C::WK ? C::MB / C::WK : 1;   // row blocks a wave finishes
    if constexpr (C::WK > 1) {
        // partial tiles meet in LDS: wave wk finishes blocks wk * OWN ...
        __syncthreads();
        f32x4_t *red = reinterpret_cast<f32x4_t *>(smem);
        b0 = wk * OWN;
        const int base = (wm * C::WN + wn) * C::MB * C::NB, step = C::WM * C::WN * C::MB * C::NB;
#pragma unroll
        for (int b = 0; b < C::MB; ++b)
#pragma unroll
            for (int n = 0; n < C::NB; ++n) red[(wk * step + base + b * C::NB + n) * WAVE + lane] = acc[b][n];
        __syncthreads();
        if (b0 >= C::MB) return;
#pragma unroll
        for (int b = 0; b < OWN; ++b)
#pragma unroll
            for (int n = 0; n < C::NB; ++n) {
                f32x4_t sum = red[(base + (b0 + b) * C::NB + n) * WAVE + lane];
#pragma unroll
                for (int k = 1; k < C::WK; ++k) sum += red[(k * step + base + (b0 + b) * C::NB + n) * WAVE + lane];
                acc[b][n] = sum;
            }
    }

    // lane: row lc of each row block, columns 4 kq .. 4 kq + 3 of each column block
    constexpr int OB = FUSED ? C::NB / 2 : C::NB;
    const bool wide = (out_cols & 3) == 0;
    auto store = [&](uint16_t *row, int col, const f32x4_t &v) {
        const u32x2_t o = {pack_bf16_rne(v[0], v[1]), pack_bf16_rne(v[2], v[3])};
        uint16_t *at = row + col;
        if (wide) {
            if (col < out_cols) *reinterpret_cast<u32x2_t *>(at) = o;
        } else {
            if (col < out_cols) at[0] = (uint16_t)o[0];
            if (col + 1 < out_cols) at[1] = (uint16_t)(o[0] >> 16);
            if (col + 2 < out_cols) at[2] = (uint16_t)o[1];
            if (col + 3 < out_cols) at[3] = (uint16_t)(o[1] >> 16);
        }
    };
#pragma unroll
    for (int b = 0; b < OWN; ++b) {
        const int m = mt * C::BM + xrow0 + 16 * (b0 + b);
        if (m >= p.M) continue;
#pragma unroll
        for (int n = 0; n < OB; ++n) {
            const int col = nt * COLS + wn * (16 * OB) + 16 * n + 4 * kq;
            f32x4_t v = acc[b][n];
            if constexpr (FUSED) {
                const f32x4_t u = acc[b][n + OB];
                if (p.product) {
                    uint16_t *row = p.product + (long)m * p.N;
                    store(row, col, v);
                    store(row + out_cols, col, u);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = (v[i] / (1.0f + __expf(-v[i]))) * u[i];
            }
            store(p.y + (long)m * out_cols, col, v);
        }
    }
}

constexpr size_t GEMM_LDS_CAP = 160 * 1024;

template <class C, bool FUSED>
long gemm_tiles(GemmArgs &args) {
    constexpr int COLS = FUSED ? C::BN / 2 : C::BN;
    long tiles = 0;
    for (int i = 0; i < args.n; ++i) {
        GemmRec &r = args.recs[i];
        r.mtiles = (r.M + C::BM - 1) / C::BM;
        r.tile_begin = (int)tiles;
        tiles += (long)r.mtiles * (((FUSED ? r.N / 2 : r.N) + COLS - 1) / COLS);
        if (tiles > (1L << 24)) return tiles;
    }
    args.tiles = (int)tiles;
    return tiles;
}

template <class C>
bool gemm_fits(const GemmArgs &args) {
    return args.K % C::KC == 0 && C::lds(args.K >> args.gshift) <= GEMM_LDS_CAP;
}

template <class C, bool FUSED>
int launch_gemm(GemmArgs &args, hipStream_t stream) {
    const long tiles = gemm_tiles<C, FUSED>(args);
    if (tiles > (1L << 24)) return VRL_INT4_ESHAPE;
    if (!gemm_fits<C>(args)) return VRL_INT4_ELIMIT;
    size_t lds = C::lds(args.K >> args.gshift);
    args.wave_flags = lds + C::WAVES * sizeof(uint32_t) <= GEMM_LDS_CAP;
    if (args.wave_flags) lds += C::WAVES * sizeof(uint32_t);
    auto kernel = &gemm_int4_kernel<C, FUSED>;
    if (lds > 64 * 1024) {   // once per build and device, at the largest size a launch may ask for
        static std::atomic<uint64_t> raised{0};
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) dev = 0;
        const uint64_t bit = 1ull << (dev & 63);
        if (!(raised.load(std::memory_order_relaxed) & bit)) {
            hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)GEMM_LDS_CAP);
            if (e != hipSuccess) return (int)e;
            raised.fetch_or(bit, std::memory_order_relaxed);
        }
    }
    return vrl_launch(kernel, dim3((unsigned)tiles), dim3(C::THREADS), lds, stream, args);
}

// Whether the launch takes this tile: all its tiles run at once, one workgroup per CU.
template <class C, bool FUSED>
bool gemm_one_round(GemmArgs &args, long cus) {
    return gemm_fits<C>(args) && gemm_tiles<C, FUSED>(args) <= cus;
}

template <int S> using Gemm32x32 = GemmCfg<1, 2, 8, 2, 1, 512, S, false>;
template <int S> using Gemm32x64 = GemmCfg<1, 2, 8, 2, 2, 512, S, false>;
template <int S> using Gemm32x64Short = GemmCfg<1, 4, 2, 2, 1, 256, S, false>;   // K no multiple of 512
template <int S> using Gemm64x64 = GemmCfg<1, 4, 4, 4, 1, 256, S, false>;
template <int S> using Gemm64x64Fused = GemmCfg<1, 2, 4, 4, 2, 256, S, false>;
using Gemm64x128 = GemmCfg<1, 4, 4, 4, 2, 256, 2, false>;
using Gemm128x128Split = GemmCfg<1, 4, 2, 8, 2, 128, 2, true>;
using Gemm128x128 = GemmCfg<1, 4, 1, 8, 2, 64, 2, true>;
using Gemm256x256 = GemmCfg<1, 8, 1, 16, 2, 64, 2, true>;

// The launch over a tile whose launch is one round, with three chunks in LDS, or two where the table leaves room for no more.
template <template <int> class C, bool FUSED>
bool launch_one_round(GemmArgs &args, long cus, hipStream_t stream, int &rc) {
    if (gemm_one_round<C<3>, FUSED>(args, cus))
        rc = launch_gemm<C<3>, FUSED>(args, stream);
    else if (gemm_one_round<C<2>, FUSED>(args, cus))
        rc = launch_gemm<C<2>, FUSED>(args, stream);
    else
        return false;
    return true;
}

// The smallest tile whose launch is one round of workgroups: until the chip is full a launch takes as long as one
// tile does, and a smaller tile is done sooner (K = 2048, one round: 6.7 / 8.2 / 9.9 / 15.2 / 21.7 us in the order
// below without the short and the fused ones; the waves split K, since a tile alone on its CU is bound by the latency of its own chain).
// The more k a chunk of these has, the fewer trips: down_proj (K = 5632, N = 2048) at 40 rows in chunks of 512 on 32x32
// tiles takes 10.5 us, in chunks of 256 on 32x64 ones 16.0; at 160 rows 32x64 in chunks of 512 takes 14.4 against 17.0.  With
// a third chunk in LDS 64x64 takes 18.8 against 21.9 us (512 rows, K = 5632).  Gate|up of up to 64 rows takes 11.0 us on
// 64x64 tiles of eight waves against 15.1 on 64x128.  Beyond one round tiles whose waves split nothing: 256x256, every
// weight rebuilt once for 256 rows, where its rounds are at least 85 % full (gate|up of 8192 rows by 2048: 339 us),
// 128x128 otherwise.  Not faster: a third chunk for 64x128 or the 128x128 ones, four or five for 32x64, 64x64 tiles with
// their waves two by two (512 rows, K = 5632: 24.9 us), AHEAD for the tiles above 128x128.
//
// The large tile is bound by issuing to the vector and matrix units, the small ones by the latency of a tile's chain.
template <bool FUSED>
int dispatch_gemm(GemmArgs &args, hipStream_t stream) {
    const long cus = device_cu_count();
    int rc;
    if constexpr (!FUSED) {   // a wave of all but the second holds one block of columns, a fused one needs gate and up
        if (launch_one_round<Gemm32x32, false>(args, cus, stream, rc)) return rc;
        if (launch_one_round<Gemm32x64, false>(args, cus, stream, rc)) return rc;
        if (launch_one_round<Gemm32x64Short, false>(args, cus, stream, rc)) return rc;
        if (launch_one_round<Gemm64x64, false>(args, cus, stream, rc)) return rc;
    } else {
        if (launch_one_round<Gemm32x64, true>(args, cus, stream, rc)) return rc;
        if (launch_one_round<Gemm64x64Fused, true>(args, cus, stream, rc)) return rc;
    }
    if (gemm_one_round<Gemm64x128, FUSED>(args, cus)) return launch_gemm<Gemm64x128, FUSED>(args, stream);
    if (gemm_one_round<Gemm128x128Split, FUSED>(args, cus)) return launch_gemm<Gemm128x128Split, FUSED>(args, stream);
    if (gemm_fits<Gemm256x256>(args)) {
        const long tiles = gemm_tiles<Gemm256x256, FUSED>(args), rounds = (tiles + cus - 1) / cus;
        if (tiles * 100 >= rounds * cus * 85) return launch_gemm<Gemm256x256, FUSED>(args, stream);
    }
    return launch_gemm<Gemm128x128, FUSED>(args, stream);
}

}  // namespace

extern "C" int vrl_int4_gemm_bf16(const vrl_int4_problem *problems, int n_problems, void *hip_stream) {
    if (!problems) return VRL_INT4_ENULL;
    if (n_problems < 1 || n_problems > GEMM_MAX) return VRL_INT4_ESHAPE;
    GemmArgs args;
    memset(&args, 0, sizeof args);
    const vrl_int4_problem &q0 = problems[0];
    const bool fused = q0.fused_gate_up != 0;
    for (int i = 0; i < n_problems; ++i) {
        const vrl_int4_problem &q = problems[i];
        const int rc = check_problem(q.x, q.qweight, q.scales, q.qzeros, q.y, q.M, q.N, q.K, q.G);
        if (rc != VRL_INT4_OK) return rc;
        if (q.prepacked || q.K != q0.K || q.G != q0.G || (q.fused_gate_up != 0) != fused || (fused && q.N % 2 != 0))
            return VRL_INT4_ESHAPE;
        if (q.product && !fused) return VRL_INT4_ESHAPE;
        if (!aligned16(q.product)) return VRL_INT4_EALIGN;
        if (q.K % 128 != 0 || q.G % 32 != 0 || !pow2(q.G) || (long)q.N * q.K / 2 >= (1L << 32)) return VRL_INT4_ELIMIT;
        GemmRec &r = args.recs[i];
        r.x = static_cast<const uint16_t *>(q.x);
        r.qweight = static_cast<const uint32_t *>(q.qweight);
        r.scales = static_cast<const uint16_t *>(q.scales);
        r.qzeros = static_cast<const uint32_t *>(q.qzeros);
        r.y = static_cast<uint16_t *>(q.y);
        r.product = static_cast<uint16_t *>(q.product);
        r.M = q.M;
        r.N = q.N;
    }
    args.n = n_problems;
    args.K = q0.K;
    args.gshift = __builtin_ctz((unsigned)q0.G);
    hipStream_t stream = reinterpret_cast<hipStream_t>(hip_stream);
    return fused ? dispatch_gemm<true>(args, stream) : dispatch_gemm<false>(args, stream);
}
