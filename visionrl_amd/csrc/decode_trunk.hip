// One decode step of an int4 Llama trunk in one launch: every layer's norm, q|k|v, rotary + cache append +
// attention, o_proj, norm, gate|up and down_proj for one new token per row (vrl/models/families/janus_pro/
// policy.py:673-678), by one workgroup per compute unit that stays for the whole step.
//
// What bounds it: at few rows a step is a chain of five dependent products per layer over 27 MB of weights (24 layers of
// 2048 / 5632).  As launches of their own each pays the launch boundary (2.4 us between two empty kernels), the first touch
// of what the launch before it wrote, a round trip for its weights and their unpacking.  Here the workgroups hand their
// results to each other through memory in words that carry their own validity, and what does not depend on the result
// waited for is done while waiting: a wave has its 4 KB of the next product's weights loaded and rebuilt in registers, and
// its keys and values requested, before the input arrives.  24 x (2048, 5632), 330 slots: 780 -> 518 us at 2 rows (20 us a
// layer, about half of it the six exchanges); six layers at 4 rows and 400 slots 212 -> 176.  At 8 rows the words alone
// are 180 KB per workgroup and down_proj, and it was slower than the launches (254 against 216), as with rows of 4096
// (four layers, 2 rows: 205 against 197): neither is built.
//
// The exchange.  A word is 8 bytes: 4 bytes of payload (two bf16 values, or a float) and the number of the exchange.  A
// producer stores a word (or two neighbouring ones) at device scope, past its die's L2; a consumer loads words at device
// scope, two at a time, until each carries the number it waits for.  Payload and number travel in one aligned 8-byte
// access, so nothing has to be ordered against anything else: no fence, no counter, no cache write-back.  From one
// workgroup's store to all of 256 having the words in LDS: 1.4 us for 16 KB read by each, 1.6 at 32 KB, 1.8 at 64 KB (a
// counter all arrive at: 6.3; a flag per workgroup and then the data: 3.9).  The numbers run on from launch to launch (the
// workspace holds the last one), so nothing is cleared.
//
// A buffer of words is written again one layer later.  Its last readers are done by then: a workgroup reads an exchange
// only if it has a part in the next one, every part of which is waited for before the one after it begins, and so on
// around the layer.
//
// Who takes part.  The work is laid out for one workgroup per compute unit, all of them there at once, and a workgroup takes
// every register of its compute unit: a single wave of anything else (a collective that waits for a late rank, another
// process, a step from another graph) keeps one of them out, for as long as it likes.  So nothing waits for a workgroup that
// has not started.  The team is fixed once, by one compare-and-swap: by the last to arrive, with everyone, or by one that has
// waited for the others as long as the step would take those that are there (TEAM_TICKS), with those that have taken a ticket
// meanwhile, which is for whoever has waited TEAM_TICKS_LEAST.  Members are running by then and stay, so what one waits for
// comes; a workgroup that starts later finds itself left out and ends.  With everyone
// there each has its own part of every product.  Otherwise the parts are dealt out to the members, product by product:
// the same sums and bits, without the work ahead of its input (24 layers at 2 rows: 518 us with all 256, 834 with 255 or 128
// of them, 6.0 ms with 16; 1.3 ms beside a kernel that keeps one out, the wait included; the launch list takes 780).  The team is looked up behind the first product, before anything is
// handed out, so that the arrivals cost next to nothing.
//
// Waits are bounded all the same: a wave gives up after `budget` unsuccessful looks in total, takes NaN for what did not
// come, hands NaN on and never waits again, so the launch ends and its output says so.  What it left behind in the workspace
// is not to be built on: it marks it, and later launches over it only write NaN, until it is zeroed.
//
// The order of sums is the launch list's, bit for bit: products by super-chunks of 512 k added up in order, norms and
// attention as in stage_x_norm and rope_attn_decode_kernel.  A policy may take either form for the same step (partial
// batches, a recorded generation), and 24 layers amplify a last bit to a percent.
#include <atomic>

#include "prepacked.hpp"

#include "../../include/vrl_decode.h"
#include "host_checks.hpp"

#if defined(__HIP_DEVICE_COMPILE__) && !defined(__gfx950__)
#error "decode_trunk.hip is written for gfx950 (64-wide waves, 160 KB of LDS, v_mfma_f32_16x16x32_bf16)"
#endif

namespace {

constexpr int TT = 1024, TW = TT / WAVE;   // threads and waves of a workgroup
constexpr int HEAD_DIM = 128;
constexpr int STATE = HEAD_DIM + 2;         // words of a softmax state: output, maximum, sum
constexpr uint32_t NOT_COME = 0x7FC07FC0u; // NaN as two bf16 values and as a float
constexpr uint32_t TRUNK_BUDGET = 1u << 22; // looks of about a microsecond each
// How long a workgroup waits for the others to start, in ticks of 10 ns: what a layer takes one workgroup alone (3.9 ms at 2
// rows), divided by those that are there, and never less than the launch itself may need to bring all of them up.
constexpr uint32_t TEAM_TICKS = 400000, TEAM_TICKS_LEAST = 10000;
constexpr uint32_t UNSETTLED = 0x7FFFFFFFu;

// Arrivals are counted in two levels, since those at one address are served one after the other, 27 ns each (24 layers at 2
// rows: a single counter for 256 workgroups 526 us, this way 517; six layers at 4 rows 189 and 181).
constexpr int ARRIVALS = 16;

// The head of the workspace.
struct TrunkState {
    uint64_t team;       // number of a launch's first layer << 32 | workgroups that take part in it
    uint64_t tickets;    // the same number << 32 | workgroups that gave up waiting for everyone
    uint32_t number;     // of the last exchange; the last workgroup to arrive counts it up
    uint32_t complete;   // groups that have arrived; the last workgroup to arrive puts it back
    uint32_t gave_up;    // a wait over this workspace was given up
    uint32_t pad[57];
    struct { uint32_t arrived, pad[63]; } groups[ARRIVALS];   // of workgroups wg % n_groups; the last of a group puts it back
};
static_assert(sizeof(TrunkState) == 256 * (1 + ARRIVALS), "a piece of 256 bytes each");

struct TrunkArgs {
    const vrl_trunk_layer *layers;
    const uint16_t *cur, *cos, *sin, *norm;
    const uint8_t *mask;
    const long long *position;
    uint16_t *normed, *h_out;
    TrunkState *state;
    uint64_t *e_qkv, *e_part, *e_attn, *e_mid, *e_act, *e_out;
    float eps;
    uint32_t budget;
    int32_t grid, most, n_groups;         // workgroups, how many of them may take part, groups (a power of two) they are counted in
    int32_t n_layers, position_stride, M, A, KV, I, heads, kv_heads, L_max;
    int32_t nsc_a, nsc_i;                 // super-chunks of A and I
    int32_t split_from;                   // filled slots from which a pair's slots are divided in ranges
};

constexpr int SC1 = 16;   // cache-policy bit: device scope, past the die's own L2

__device__ __forceinline__ void put_word(uint64_t *at, uint32_t payload, uint32_t number) {
    __hip_atomic_store(at, (uint64_t)number << 32 | payload, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// two neighbouring words in one store
__device__ __forceinline__ void put_pair(uint64_t *base, int words, int at, uint32_t a, uint32_t b, uint32_t number) {
    const rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(base, 0, words * 8, 0x00020000);
    __builtin_amdgcn_raw_buffer_store_b128(u32x4_t{a, number, b, number}, rsrc, at * 8, 0, SC1);
}

// Pairs of words, N of them, as soon as all of a wave's carry `number`: pair i of a lane at words at(i) (the lane's) +
// off(i) (uniform) of the `words` from base on.  One 16-byte load fetches a pair; each half of it is judged by its own
// number, and an aligned 8-byte half is never seen half written (the guard above pins the memory system this rests on).
template <int N, class At, class Off>
__device__ __forceinline__ void await_pairs(uint32_t (&v)[2 * N], uint32_t number, uint32_t &budget, const uint64_t *base,
                                            int words, At at, Off off) {
    const rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint64_t *>(base), 0, words * 8, 0x00020000);
    u32x4_t w[N];
    for (;;) {
#pragma unroll
        for (int i = 0; i < N; ++i) w[i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, at(i) * 8, off(i) * 8, SC1);
        bool all = true;
#pragma unroll
        for (int i = 0; i < N; ++i) all &= w[i][1] == number && w[i][3] == number;
        if (__builtin_amdgcn_ballot_w64(!all) == 0 || budget == 0) break;
        --budget;
        asm volatile("" ::: "memory");   // the next round's loads are not this one's
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
        v[2 * i] = w[i][1] == number ? w[i][0] : NOT_COME;
        v[2 * i + 1] = w[i][3] == number ? w[i][2] : NOT_COME;
    }
}

// A super-chunk (512 k) of a tile of 16 weight rows, as the blob holds it: what a wave works on at a time.
struct Unit {
    u32x4_t slot[4];
    uint32_t meta;
};

// `on` false: the loads are issued all the same (one place in the program fills a unit's registers, whatever the wave
// has to do) through a resource of no bytes, which answers with zeros without touching memory.
__device__ __forceinline__ void load_unit(Unit &u, bool on, int lane, const void *blob, int N, int K, int tile, int sc) {
    const uint32_t tile_bytes = (uint32_t)pp_tile_u4(K, 128) * 16u, meta_bytes = (uint32_t)pp_meta_u4(K, 128) * 16u;
    const rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<void *>(blob), 0, on ? (int)((uint32_t)((N + 15) / 16) * tile_bytes) : 0, 0x00020000);
    const uint32_t base = (uint32_t)tile * tile_bytes;
    u.meta = __builtin_amdgcn_raw_buffer_load_b32(rsrc, lane * 4, (int)(base + (uint32_t)sc * 256u), 0);
#pragma unroll
    for (int d = 0; d < 4; ++d)
        u.slot[d] = __builtin_amdgcn_raw_buffer_load_b128(
            rsrc, lane * 16, (int)(base + meta_bytes + (uint32_t)sc * 4096u + d * 1024u), BUFFER_NT);
}

// eight exactly rounded bf16 weights of the lane's row (the rebuild of stream_rows_pp)
__device__ __forceinline__ u32x4_t rebuild(uint32_t v, const PPGroup &g, uint32_t mask, uint32_t bias) {
    u32x2_t a0, a1;
    a0[0] = (v & mask) | bias;
    a0[1] = ((v >> 4) & mask) | bias;
    a1[0] = ((v >> 8) & mask) | bias;
    a1[1] = ((v >> 12) & mask) | bias;
    const f32x4_t d0 = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(bf16x4_t, a0), g.bdiag, g.cq, 0, 0, 0);
    const f32x4_t d1 = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(bf16x4_t, a1), g.bdiag, g.cq, 0, 0, 0);
    return u32x4_t{pack_bf16_rne(d0[0], d0[1]), pack_bf16_rne(d0[2], d0[3]), pack_bf16_rne(d1[0], d1[1]),
                   pack_bf16_rne(d1[2], d1[3])};
}

// LDS written before it is there for every wave after it.  Not __syncthreads(), which also waits for every load a wave
// has in flight: the weights and cached keys and values requested ahead.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// The same between the lanes of one wave (a wave's LDS accesses are served in order).
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// a and b hold the same value per lane: afterwards a that of the lane in the first, b of the lane in the second half of the
// wave (swap_16: of each half's sixteens), for both.  Register swaps, no trip through the LDS crossbar.
__device__ __forceinline__ void swap_32(float &a, float &b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
    a = __builtin_bit_cast(float, (uint32_t)r[0]), b = __builtin_bit_cast(float, (uint32_t)r[1]);
}
__device__ __forceinline__ void swap_16(float &a, float &b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
    a = __builtin_bit_cast(float, (uint32_t)r[0]), b = __builtin_bit_cast(float, (uint32_t)r[1]);
}

// dot[u] += q . k[u] over a lane's eight values, two products per instruction.  Inline assembly, the four slots' sums in
// turn: this toolchain drops all but the first of several independent __builtin_amdgcn_fdot2_f32_bf16 chains here, and the
// hardware does not interlock a dot result read within three instructions.
__device__ __forceinline__ void dot4(float (&dot)[4], const u32x4_t &q, const u32x4_t *k) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
        asm volatile("v_dot2_f32_bf16 %0, %4, %5, %0\n\t"
                     "v_dot2_f32_bf16 %1, %4, %6, %1\n\t"
                     "v_dot2_f32_bf16 %2, %4, %7, %2\n\t"
                     "v_dot2_f32_bf16 %3, %4, %8, %3\n\t"
                     "s_nop 2"
                     : "+v"(dot[0]), "+v"(dot[1]), "+v"(dot[2]), "+v"(dot[3])
                     : "v"(q[e]), "v"(k[0][e]), "v"(k[1][e]), "v"(k[2][e]), "v"(k[3][e]));
}

__device__ __forceinline__ void opaque(int &v) {   // a uniform value
    v = __builtin_amdgcn_readfirstlane(v);
    asm volatile("" : "+s"(v));
}

__device__ __forceinline__ float low_bf16(uint32_t w) { return bf16_bits_to_f32(w & 0xFFFFu); }
__device__ __forceinline__ float high_bf16(uint32_t w) { return bf16_bits_to_f32(w >> 16); }

typedef const __attribute__((address_space(4))) vrl_trunk_layer *layer_ptr;   // uniform, constant: scalar loads
typedef const __attribute__((address_space(4))) TrunkArgs *arg_ptr;
typedef __attribute__((address_space(1))) uint32_t *gptr_w;

enum Phase { P_QKV, P_O, P_GATE_UP, P_DOWN };

constexpr int H = 2048;                    // hidden
constexpr int NSC = H / PP_SC;             // its super-chunks
constexpr int ROW_WORDS = H / 2;           // words of a row
constexpr int XROW = H / 128 * 136 + 32;   // elements of a staged row: 136 per 128 k, so that the four lane quarters of an
                                           // operand read, 128 k apart, fall on different banks
constexpr int OWN_ROW = 4 * 136;           // the same of one super-chunk
constexpr int STATES = TW;                 // softmax states of a (row, head) at most

// MW: activation rows at most (2 or 4).  P1, P2: waves of the launch list that share a row in the sums of squares of the
// two norms of a layer (norm_parts).  SPLITS: workgroups per (row, head), as the split attention has them.
template <int MW_, int P1_>
struct TrunkCfg {
    static constexpr int MW = MW_, P1 = P1_, P2 = 8 / MW, SPLITS = 16 / MW;
    static constexpr size_t ALL = (size_t)MW * XROW * 2, OWN = (size_t)TW * MW * OWN_ROW * 2;
    static constexpr size_t STAGE_BYTES = ((ALL > OWN ? ALL : OWN) + 15) / 16 * 16;
    static constexpr int PART = TW * MW * 16;   // floats
    static constexpr size_t ATTN_BYTES = (size_t)TW * HEAD_DIM * 4 + 5 * 64 * 4 + 2 * TW * 4;
    static constexpr size_t LDS = STAGE_BYTES + 2 * PART * 4 + ATTN_BYTES + TW * 4 + 16;
};

// A lane's words of a part of a row, and of the norm's weight for its share of them
template <int MW, int P>
struct Rows { uint32_t h[4 * (H / 512 / P)], w[MW]; };

typedef __attribute__((address_space(3))) uint8_t *lds_ptr;
template <class C>
__device__ void share_out(arg_ptr args, lds_ptr smem);

// The step.  SHARED false: every workgroup is there and works on its own part of each product; the kernel.  SHARED true:
// the team is not the whole grid; a function that the kernel calls for the rest of its life, so that neither form's
// registers are the other's (in one function a step of 24 layers took 537 us in place of 511).
template <class C, bool SHARED>
__device__ __forceinline__ void trunk_step(const TrunkArgs &a, arg_ptr args, uint8_t *smem) {
    constexpr int MW = C::MW, splits = C::SPLITS;
    int tid = threadIdx.x, lane, wave, lc, kq;
    int wg = blockIdx.x, G = a.grid;
    int M = a.M, A = a.A, KV = a.KV, I = a.I, heads = a.heads;
    uint16_t *const xs = reinterpret_cast<uint16_t *>(smem);
    float *const parts = reinterpret_cast<float *>(smem + C::STAGE_BYTES);
    float *const pacc = parts + 2 * C::PART;
    uint32_t *const qs = reinterpret_cast<uint32_t *>(pacc + TW * HEAD_DIM), *const ks = qs + 64, *const vs = ks + 64,
             *const turn = vs + 64;
    float *const pm = reinterpret_cast<float *>(turn + 128), *const pl = pm + TW, *const red = pl + TW;
    uint32_t *const joined = reinterpret_cast<uint32_t *>(red + TW);
    uint32_t budget = a.budget;
    uint32_t number = 0;   // exchange e of a layer is number + e; known from the first product on

    // Arguments used once a layer, or once, are read again where they are used.
    auto again = [&]() {
        arg_ptr p = args;
        asm volatile("" : "+s"(p));
        return p;
    };

    uint32_t mask16 = PAIR_MASK, bias16 = PAIR_BIAS;
    asm volatile("" : "+s"(mask16));
    asm volatile("" : "+v"(bias16));

    // What is computed from these stays inside the layer: left alone the compiler keeps every address and unit of a
    // layer in registers from layer to layer and spills hundreds of them.
    auto forget = [&]() {
        asm volatile("" : "+v"(tid));
        lane = tid & (WAVE - 1);
        wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        lc = lane & 15, kq = lane >> 4;
        opaque(wg), opaque(G), opaque(M), opaque(A), opaque(KV), opaque(I), opaque(heads);
    };
    forget();

    // ---- which units of a product are this wave's: unit u counts super-chunks, then gate and up, then tiles
    auto slots_of = [&](int at, int tiles) { return at < tiles ? (tiles - 1 - at) / G + 1 : 0; };
    int slots_qkv, slots_i;
    bool has_h;
    auto place_tiles = [&]() {
        slots_qkv = slots_of(wg, (A + 2 * KV) >> 4), slots_i = slots_of(wg, I >> 4);
        // the tiles of o_proj and down_proj begin at the other end of the grid, where workgroups have fewer of the others
        has_h = G - 1 - wg < H / 16;   // (one at most)
    };
    place_tiles();
    // (a unit: a super-chunk of a tile; never more than sixteen)
    auto units_of = [&](Phase ph) {
        return ph == P_QKV ? slots_qkv * NSC : ph == P_GATE_UP ? slots_i * 2 * NSC : has_h ? (ph == P_O ? a.nsc_a : a.nsc_i) : 0;
    };
    // (the last waves take the units of o_proj and down_proj: the first have the attention to do meanwhile)
    auto unit_of = [&](Phase ph) { return ph == P_O || ph == P_DOWN ? TW - 1 - wave : wave; };
    auto chunk_of = [&](Phase ph, int u) { return ph == P_O || ph == P_DOWN ? u : u % NSC; };
    Unit raw;
    auto load = [&](Phase ph, int layer) {
        const int u = unit_of(ph), sc = chunk_of(ph, u), tile = u / NSC;
        const bool on = layer < a.n_layers && u < units_of(ph);   // wave-uniform
        const layer_ptr L = (layer_ptr)(uintptr_t)a.layers + min(layer, a.n_layers - 1);
        if (ph == P_QKV) {
            const int at = wg + tile * G, kv = at - (A >> 4), v = kv - (KV >> 4);
            load_unit(raw, on, lane, kv < 0 ? L->q : v < 0 ? L->k : L->v, KV + (kv < 0) * (A - KV), H, kv < 0 ? at : v < 0 ? kv : v, sc);
        } else if (ph == P_O) {
            load_unit(raw, on, lane, L->o, H, A, G - 1 - wg, sc);
        } else if (ph == P_GATE_UP) {   // tile: (slot, gate or up)
            load_unit(raw, on, lane, L->gate_up, 2 * I, H, (tile & 1) * (I >> 4) + wg + (tile >> 1) * G, sc);
        } else {
            load_unit(raw, on, lane, L->down, H, I, G - 1 - wg, sc);
        }
    };
    struct Built { u32x4_t w[16]; };
    auto build_ahead = [&](Phase ph, Built &built) {
        // (or a wave without a unit would carry the weights it rebuilt a layer ago)
#pragma unroll
        for (int i = 0; i < 16; ++i) built.w[i] = __builtin_nondeterministic_value(built.w[i]);
        if (unit_of(ph) < units_of(ph)) {
            const PPGroup g = pp_group(raw.meta, lane & 3);
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                built.w[i] = rebuild(raw.slot[i >> 2][i & 3], g, mask16, bias16);
                if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // not all the 4x4x4 products before the first conversion
            }
        }
    };

    // ---- a unit's products; x: the lane's operands
    auto operand_row = [&]() { return min(lc, M - 1); };   // rows past the last repeat it: not looked at
    auto multiply = [&](const uint16_t *x, const Built &built) {
        f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t *>(x + 8 * i)),
                __builtin_bit_cast(bf16x8_t, built.w[i]), acc, 0, 0, 0);
            if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // not all the operands at once
        }
        return acc;
    };
    // the unit's partial tile, rows by 16 columns, into LDS
    auto keep_partial = [&](int parity, int u, const f32x4_t &acc) {
        float *at = parts + parity * C::PART + u * (MW * 16) + lc;   // (rows 0..3 of the product: lanes 0..15)
        if (kq == 0)
#pragma unroll
            for (int i = 0; i < MW; ++i) at[i * 16] = acc[i];
    };
    // the sum of a tile's partial products, in the order of k, for (row, column pair) = lane % (8 MW)
    auto tile_sum = [&](int parity, int unit0, int n) {
        const float *at = parts + parity * C::PART + unit0 * (MW * 16) + 2 * (lane % (8 * MW));
        float2 s = {0.0f, 0.0f};
#pragma unroll 4
        for (int t = 0; t < n; ++t) {
            const float2 v = *reinterpret_cast<const float2 *>(at + t * (MW * 16));
            s.x += v.x;
            s.y += v.y;
        }
        return s;
    };
    auto tile_row = [&]() { return lane % (8 * MW) >> 3; };
    auto stores = [&]() { return lane < 8 * MW && tile_row() < M; };

    // ---- a product over the normalised rows, staged in xs
    auto multiply_staged = [&](Phase ph, const Built &built) {
        const int u = unit_of(ph);
        if (u < units_of(ph)) keep_partial(0, u, multiply(xs + operand_row() * XROW + (chunk_of(ph, u) * 4 + kq) * 136, built));
    };
    // ---- a product over rows a wave stages for itself: only its own super-chunk
    auto own_product = [&](Phase ph, const Built &built, const uint64_t *words, int K, uint32_t number, Phase next, int next_layer) {
        constexpr int PAIRS = 2 * MW;   // pair i of a lane: row i / 2, half i % 2 of the super-chunk
        uint32_t got[2 * PAIRS];
#pragma unroll
        for (int i = 0; i < 2 * PAIRS; ++i) got[i] = __builtin_nondeterministic_value(got[i]);
        const int u = unit_of(ph), k0 = u * PP_SC;
        const bool on = u < units_of(ph);
        if (on)
            await_pairs<PAIRS>(got, number, budget, words, M * K >> 1, [&](int) { return 2 * lane; }, [&](int i) {
                // K % 512 is 0 or 256: where nothing is left a repeat is asked for, and zeros taken
                return (min(i / 2, M - 1) * K + min(k0 + i % 2 * 256, K - 256)) >> 1;
            });
        load(next, next_layer);
        if (on) {
            uint16_t *own = xs + wave * (MW * OWN_ROW);
#pragma unroll
            for (int i = 0; i < PAIRS; ++i) {
                const bool in = k0 + i % 2 * 256 < K;
                *reinterpret_cast<u32x2_t *>(own + i / 2 * OWN_ROW + (i % 2 * 2 + lane / 32) * 136 + lane % 32 * 4) =
                    u32x2_t{in ? got[2 * i] : 0u, in ? got[2 * i + 1] : 0u};
            }
            wave_fence();
            keep_partial(1, u, multiply(own + operand_row() * OWN_ROW + kq * 136, built));
            wave_fence();   // read before the next product's rows are written
        }
    };

    // ---- RMSNorm of every row into xs, the sums of squares in the launch list's order: `n` waves of it share a row, part q
    // has the H / n values from H / n q on, a lane eight neighbouring ones of every 512, one after the other; lanes, then
    // parts.  Here PER = 16 / (MW n) waves take a (row, part) each, all of it for the sum and their share of it to write:
    // GROUPS groups of four values per lane.  (P: n)
    constexpr int GROUPS = MW / 2;
    auto part_of = [&](auto P) { return wave / (TW / MW / P); };   // (row, part)
    auto row_at = [&](auto P) { return part_of(P) % P * (H / P) + lane * 8; };   // the lane's first value in the row
    auto group_of = [&](auto P, int j) { return wave % (TW / MW / P) * GROUPS + j; };   // its share: groups of four
    auto undefined = [](auto &x) {   // not what the registers held a layer ago
#pragma unroll
        for (uint32_t &v : x.h) v = __builtin_nondeterministic_value(v);
#pragma unroll
        for (uint32_t &v : x.w) v = __builtin_nondeterministic_value(v);
    };
    // (`plain`: the rows themselves, in place of words)
    auto take_rows = [&](auto P, Rows<MW, P> &x, const void *weight, const uint64_t *words, uint32_t number, const uint16_t *plain = nullptr) {
        constexpr int EIGHTS = H / 512 / P;
#pragma unroll
        for (int j = 0; j < GROUPS; ++j) {
            const int g = group_of(P, j), at = row_at(P) + g / 2 * 512 + g % 2 * 4;
            const u32x2_t w = ((const __attribute__((address_space(1))) u32x2_t *)(uintptr_t)weight)[at / 4];
            x.w[2 * j] = w[0], x.w[2 * j + 1] = w[1];
        }
        const int row = min(part_of(P) / P, M - 1), at = row_at(P) / 2;
        if (plain) {
#pragma unroll
            for (int i = 0; i < 2 * EIGHTS; ++i) {
                const u32x2_t v = *(const __attribute__((address_space(1))) u32x2_t *)(uintptr_t)(
                    plain + 2 * (row * ROW_WORDS + i / 2 * 256 + i % 2 * 2 + at));
                x.h[2 * i] = v[0], x.h[2 * i + 1] = v[1];
            }
            return;
        }
        await_pairs<2 * EIGHTS>(x.h, number, budget, words, M * ROW_WORDS, [&](int) { return at; },
                                [&](int i) { return row * ROW_WORDS + i / 2 * 256 + i % 2 * 2; });
    };
    auto normalise = [&](auto P, const Rows<MW, P> &x, float eps) {
        constexpr int EIGHTS = H / 512 / P, PER = TW / MW / P;
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < 4 * EIGHTS; ++i) {
            ss = __builtin_fmaf(low_bf16(x.h[i]), low_bf16(x.h[i]), ss);
            ss = __builtin_fmaf(high_bf16(x.h[i]), high_bf16(x.h[i]), ss);
        }
        ss = wave_sum(ss);
        if (lane == 0) red[part_of(P)] = ss;   // (the part's other waves write the same)
        lds_barrier();
        const int row = part_of(P) / P;
        ss = red[row * P];
#pragma unroll
        for (int q = 1; q < P; ++q) ss += red[row * P + q];
        const float r = rsqrtf(__builtin_fmaf(ss, 1.0f / H, eps));
#pragma unroll
        for (int j = 0; j < GROUPS; ++j) {
            const int g = group_of(P, j), k = row_at(P) + g / 2 * 512 + g % 2 * 4;
            uint32_t v[2] = {x.h[2 * j], x.h[2 * j + 1]};
#pragma unroll
            for (int o = 1; o < PER; ++o) {   // (a value each: or the compiler makes an address of the choice, and memory of the registers)
                uint32_t c0 = x.h[2 * (o * GROUPS + j)], c1 = x.h[2 * (o * GROUPS + j) + 1];
                asm("" : "+v"(c0), "+v"(c1));
                v[0] = wave % PER == o ? c0 : v[0], v[1] = wave % PER == o ? c1 : v[1];
            }
            u32x2_t y;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const uint32_t m = pack_bf16_rne(low_bf16(v[e]) * r, high_bf16(v[e]) * r);
                y[e] = pack_bf16_rne(low_bf16(x.w[2 * j + e]) * low_bf16(m), high_bf16(x.w[2 * j + e]) * high_bf16(m));
            }
            *reinterpret_cast<u32x2_t *>(xs + row * XROW + (k >> 7) * 136 + (k & 127)) = y;
        }
        lds_barrier();
    };
    constexpr std::integral_constant<int, C::P1> P1{};
    constexpr std::integral_constant<int, C::P2> P2{};

    // ---- who takes part (lane 0 of wave TW - 1 sees to it): a workgroup counts itself once it knows this launch's number ...
    struct Arrival { uint32_t first, rank; };
    auto arrive = [&](Arrival &mine) {
        TrunkState *const state = again()->state;
        if (lane == 0) {
            mine.first = __hip_atomic_load(&state->number, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            asm volatile("s_waitcnt vmcnt(0)" : "+v"(mine.first)::"memory");   // read before it counts: the last one counts it up
            mine.rank = __hip_atomic_fetch_add(&state->groups[wg & (again()->n_groups - 1)].arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    };
    Arrival arrival{__builtin_nondeterministic_value(0u), __builtin_nondeterministic_value(0u)};
    if (!SHARED && wave == TW - 1) arrive(arrival);

    // ---- this workgroup's share of the attention of one (row, head), the same in every layer; so are the position, the
    // rotation and which slots count.  The order of sums is that of rope_attn_decode_kernel with sixteen waves: groups of
    // sixteen lanes visit the slots of wave w, group g: 64 u + 4 w + g, four at a time; groups, then waves.  The
    // workgroups of a pair take its waves' slots each (`lead`: the first of them), and all waves' states meet through
    // memory; or, from `split_from` filled slots on, a contiguous range of slots as in its split form (`ranges`).
    int pair, split, am, ah, akv, p, j_lo, j_hi, lead, my_waves;
    bool attends, appends, ranges, own_slot;
    auto place_pair = [&]() {
        const arg_ptr t = again();   // (or these arguments are kept in registers from layer to layer)
        const int group = heads / t->kv_heads;
        pair = wg / splits, split = wg % splits;
        attends = pair < M * heads;
        am = attends ? pair / heads : 0, ah = attends ? pair % heads : 0;
        appends = attends && split == 0 && ah % group == 0;
        akv = ah / group;
        p = -1, j_lo = 0, j_hi = 0, lead = 0, my_waves = 0;
        ranges = own_slot = false;
        if (attends) {
            const uint8_t *mrow = t->mask + (long)am * t->L_max;
            const long long p64 = t->position[(long)am * t->position_stride];
            const int at = __builtin_amdgcn_readfirstlane(p64 >= 0 && p64 < t->L_max ? (int)p64 : -1);
            if (at >= 0) {   // else the row is left alone: nothing appended, nothing attended
                p = at;
                ranges = p >= t->split_from;
                const int share = ((p + splits - 1) / splits + 63) / 64 * 64;
                j_lo = ranges ? min(p, split * share) : 0;
                j_hi = ranges ? min(p, j_lo + share) : p;
                if (wave == 0) {   // (read by this wave alone)
                    turn[lane] = ((gptr_cu32)(uintptr_t)(t->cos + (long)p * HEAD_DIM))[lane];
                    turn[64 + lane] = ((gptr_cu32)(uintptr_t)(t->sin + (long)p * HEAD_DIM))[lane];
                }
                own_slot = (split == 0 || !ranges) && mrow[p] != 0;
            }
            my_waves = ranges ? TW : TW / splits;
            lead = ranges ? 0 : split * my_waves;
        }
    };
    place_pair();
    uint32_t live = 0;
    constexpr int BATCH = 4, AT_ONCE = 2 * BATCH;   // slots of a group per step of the running softmax; requested at once
    auto slot_of = [&](int j0, int u) { return j0 + u * (4 * TW) + (lead + wave) * 4 + kq; };   // j0: the first of the trip
    auto counts = [&](int j0) {   // which of the trip's slots count, a bit each
        const uint8_t *mrow = again()->mask + (long)am * a.L_max;
        uint32_t bits = 0;
#pragma unroll
        for (int u = 0; u < AT_ONCE; ++u) {
            const int j = slot_of(j0, u);
            if (j < j_hi && mrow[j] != 0) bits |= 1u << u;
        }
        return bits;
    };
    if (wave < my_waves) live = counts(j_lo);
    struct Slots { u32x4_t k[AT_ONCE], v[AT_ONCE]; };
    auto cache_base = [&]() { return ((long)am * a.kv_heads + akv) * a.L_max * HEAD_DIM; };
    auto request = [&](Slots &kv, layer_ptr L, int j0) {
        const uint16_t *kc = static_cast<const uint16_t *>(L->k_cache) + cache_base();
        const uint16_t *vc = static_cast<const uint16_t *>(L->v_cache) + cache_base();
#pragma unroll
        for (int u = 0; u < AT_ONCE; ++u) {
            kv.k[u] = kv.v[u] = u32x4_t{0u, 0u, 0u, 0u};
            if (slot_of(j0, u) - kq < j_hi) {   // wave-uniform
                const uint32_t at = (uint32_t)min(slot_of(j0, u), j_hi - 1) * (HEAD_DIM * 2) + lc * 16;   // past the end: a repeat
                kv.k[u] = *as_global(reinterpret_cast<const u32x4_t *>(reinterpret_cast<const char *>(kc) + at));
                kv.v[u] = *as_global(reinterpret_cast<const u32x4_t *>(reinterpret_cast<const char *>(vc) + at));
            }
        }
    };

    // The residual stream at (row, column pair) of this workgroup's o_proj and down_proj tiles, kept by the threads that
    // finish them.  The input rows begin it.
    uint32_t stream = 0;
    auto stream_word = [&]() { return tile_row() * ROW_WORDS + (G - 1 - wg) * 8 + (lane & 7); };
    auto begin_stream = [&]() {
        if (has_h && wave == 0 && stores()) stream = ((gptr_cu32)(uintptr_t)again()->cur)[stream_word()];
    };

    // ---- the parts of a layer that both forms of the step go through
    auto publish_qkv = [&]() {
        if (!slots_qkv) return;
        lds_barrier();
        if (wave < slots_qkv) {
            const float2 s = tile_sum(0, wave * NSC, NSC);
            if (stores())
                put_word(a.e_qkv + tile_row() * ((A + 2 * KV) >> 1) + (wg + wave * G) * 8 + (lane & 7),
                         pack_bf16_rne(s.x, s.y), number + 1);
        }
    };
    // wave 0: the new token's query, key (both rotated) and value into LDS, the latter two into the caches
    auto receive_token = [&](layer_ptr L, bool append) __attribute__((always_inline)) {
        // lanes 0..15 the query's dimensions 4 i ... and 64 + 4 i ..., 16..31 the key's, 32..47 the value's (48..63 too)
        const int part = kq, row_words = (A + 2 * KV) >> 1;
        const int at = (part == 0 ? ah * 64 : (part == 1 ? A >> 1 : (A + KV) >> 1) + akv * 64) + 2 * lc;
        uint32_t x[4];
        await_pairs<2>(x, number + 1, budget, a.e_qkv, M * row_words, [&](int) { return at; },
                       [&](int i) { return am * row_words + 32 * i; });
        if (part < 2) {   // bf16(bf16(x cos) + bf16(rotate_half(x) sin))
            auto round = [](float v) { return low_bf16(pack_bf16_rne(v, 0.0f)); };
            const u32x2_t c0 = *reinterpret_cast<const u32x2_t *>(turn + 2 * lc), c1 = *reinterpret_cast<const u32x2_t *>(turn + 32 + 2 * lc);
            const u32x2_t s0 = *reinterpret_cast<const u32x2_t *>(turn + 64 + 2 * lc), s1 = *reinterpret_cast<const u32x2_t *>(turn + 96 + 2 * lc);
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const float a0 = low_bf16(x[e]), a1 = high_bf16(x[e]), b0 = low_bf16(x[2 + e]), b1 = high_bf16(x[2 + e]);
                x[e] = pack_bf16_rne(round(a0 * low_bf16(c0[e])) + round(-b0 * low_bf16(s0[e])),
                                     round(a1 * high_bf16(c0[e])) + round(-b1 * high_bf16(s0[e])));
                x[2 + e] = pack_bf16_rne(round(b0 * low_bf16(c1[e])) + round(a0 * low_bf16(s1[e])),
                                         round(b1 * high_bf16(c1[e])) + round(a1 * high_bf16(s1[e])));
            }
        }
        uint32_t *out = qs + min(part, 2) * 64 + 2 * lc;   // qs, ks, vs
        *reinterpret_cast<u32x2_t *>(out) = u32x2_t{x[0], x[1]};
        *reinterpret_cast<u32x2_t *>(out + 32) = u32x2_t{x[2], x[3]};
        if (append && appends && p >= 0 && part > 0) {
            gptr_w to = (gptr_w)(uintptr_t)(static_cast<uint16_t *>(part == 1 ? L->k_cache : L->v_cache) + cache_base() +
                                            (long)p * HEAD_DIM) + 2 * lc;
            to[0] = x[0], to[1] = x[1], to[32] = x[2], to[33] = x[3];
        }
    };
    // the softmax states of this workgroup's waves over its slots (`kv`: the first of them, requested)
    auto score_slots = [&](layer_ptr L, Slots &kv) __attribute__((always_inline)) {
        const float scaling = L->scaling;
        const u32x4_t q4 = *reinterpret_cast<const u32x4_t *>(qs + lc * 4);
        float mx = -INFINITY, sum = 0.0f, acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        uint32_t now = live;
        for (int j0 = j_lo; j0 + (lead + wave) * 4 < j_hi; j0 += AT_ONCE * 4 * TW) {   // wave-uniform
            if (j0 > j_lo) {
                request(kv, L, j0);
                now = counts(j0);
            }
#pragma unroll
            for (int b = 0; b < AT_ONCE; b += BATCH) {
                if (slot_of(j0, b) - kq >= j_hi) break;   // wave-uniform: nothing in the rest
                float dot[BATCH] = {0.f, 0.f, 0.f, 0.f}, sc[BATCH], m2 = mx;
                dot4(dot, q4, kv.k + b);
#pragma unroll
                for (int u = 0; u < BATCH; ++u) {
                    dot[u] = row16_sum(dot[u]);   // the sixteen lanes that share the slot
                    sc[u] = now >> (b + u) & 1 ? dot[u] * scaling : -INFINITY;
                    m2 = fmaxf(m2, sc[u]);
                }
                const float ref = m2 == -INFINITY ? 0.0f : m2, c0 = __expf(mx - ref);
                mx = m2;
#pragma unroll
                for (int u = 0; u < BATCH; ++u) {
                    const float w = __expf(sc[u] - ref);
                    sum = u ? sum + w : __builtin_fmaf(sum, c0, w);
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float v = e & 1 ? high_bf16(kv.v[b + u][e >> 1]) : low_bf16(kv.v[b + u][e >> 1]);
                        acc[e] = u ? __builtin_fmaf(w, v, acc[e]) : two_products(acc[e], c0, w, v);
                    }
                }
            }
        }
        // the wave's four groups, 0 with 1 and 2 with 3, then both; what group 0 holds then counts
#pragma unroll
        for (int step = 0; step < 2; ++step) {
            float m1 = mx, m2 = mx, l1 = sum, l2 = sum;
            step ? swap_32(m1, m2) : swap_16(m1, m2);
            step ? swap_32(l1, l2) : swap_16(l1, l2);
            mx = fmaxf(m1, m2);
            const float ref = mx == -INFINITY ? 0.0f : mx, c1 = __expf(m1 - ref), c2 = __expf(m2 - ref);
            sum = two_products(l1, c1, l2, c2);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float a1 = acc[e], a2 = acc[e];
                step ? swap_32(a1, a2) : swap_16(a1, a2);
                acc[e] = two_products(a2, c2, a1, c1);
            }
        }
        if (ranges) {
            if (kq == 0) {
                *reinterpret_cast<f32x4_t *>(pacc + wave * HEAD_DIM + lc * 8) = f32x4_t{acc[0], acc[1], acc[2], acc[3]};
                *reinterpret_cast<f32x4_t *>(pacc + wave * HEAD_DIM + lc * 8 + 4) = f32x4_t{acc[4], acc[5], acc[6], acc[7]};
            }
            if (lane == 0) pm[wave] = mx, pl[wave] = sum;
        } else if (kq == 0) {
            uint64_t *state = a.e_part + (long)(pair * STATES + lead + wave) * STATE;
#pragma unroll
            for (int e = 0; e < 8; e += 2)
                put_pair(state, STATE, lc * 8 + e, __builtin_bit_cast(uint32_t, acc[e]), __builtin_bit_cast(uint32_t, acc[e + 1]), number + 2);
            if (lane == 0)
                put_pair(state, STATE, HEAD_DIM, __builtin_bit_cast(uint32_t, mx), __builtin_bit_cast(uint32_t, sum), number + 2);
        }
    };
    // wave 0: the states of this workgroup's waves joined into one and handed on (`ranges` only), and the pair's states
    // joined for this workgroup's share of the columns
    struct Joined { float o0, o1, total, top; };
    auto own_score = [&](layer_ptr L) __attribute__((always_inline)) {
        float own = -INFINITY;   // the new token's own slot, where this workgroup counts it
        if (own_slot) {
            const uint16_t *q = reinterpret_cast<const uint16_t *>(qs), *k = reinterpret_cast<const uint16_t *>(ks);
            const float dot = bf16_bits_to_f32(q[lane]) * bf16_bits_to_f32(k[lane]);
            own = wave_sum(__builtin_fmaf(bf16_bits_to_f32(q[lane + 64]), bf16_bits_to_f32(k[lane + 64]), dot)) * L->scaling;
        }
        return own;
    };
    // n states in LDS (pacc, pm, pl) joined in order for columns col, col + 1, the token's own slot first
    auto join_states = [&](int n, int col, float own) {
        float o0 = 0.0f, o1 = 0.0f, total, top;
            const float m_w = lc < n ? pm[lc] : -INFINITY, l_w = lc < n ? pl[lc] : 0.0f;   // lane w of sixteen: state w
            top = fmaxf(own, row16_max(m_w));
            const float ref = top == -INFINITY ? 0.0f : top, c_w = __expf(m_w - ref), c_own = __expf(own - ref);
            const float v0 = low_bf16(vs[col >> 1]), v1 = high_bf16(vs[col >> 1]);
            total = c_own;
#pragma unroll
            for (int w = 0; w < TW; ++w)
                if (w < n) {   // uniform
                    const float2 v = *reinterpret_cast<const float2 *>(pacc + w * HEAD_DIM + col);
                    const float c = lane_of(c_w, w);
                    o0 = w ? __builtin_fmaf(c, v.x, o0) : two_products(c_own, v0, c, v.x);
                    o1 = w ? __builtin_fmaf(c, v.y, o1) : two_products(c_own, v1, c, v.y);
                    total = __builtin_fmaf(c, lane_of(l_w, w), total);
                }
        return Joined{o0, o1, total, top};
    };
    auto leave_state = [&](float own) __attribute__((always_inline)) {
        const int col = 2 * lane;
        const Joined s = join_states(TW, col, own);
        uint64_t *states = a.e_part + (long)pair * STATES * STATE;
        put_pair(states, STATES * STATE, split * STATE + col, __builtin_bit_cast(uint32_t, s.o0), __builtin_bit_cast(uint32_t, s.o1), number + 2);
        if (lane == 0)
            put_pair(states, STATES * STATE, split * STATE + HEAD_DIM, __builtin_bit_cast(uint32_t, s.top), __builtin_bit_cast(uint32_t, s.total), number + 2);
    };
    auto join_pair = [&](float own) __attribute__((always_inline)) {
        const int n = ranges ? splits : TW;   // states of the pair
        const uint64_t *states = a.e_part + (long)pair * STATES * STATE;
        // this workgroup's share of the columns: lane, load -> (state, column pair); last (maximum, sum)
        constexpr int PAIRS = (HEAD_DIM / 2) / splits, PER_LOAD = WAVE / PAIRS, LOADS = STATES / PER_LOAD;
        const int z = lane / PAIRS, c = lane % PAIRS, col0 = split * (HEAD_DIM / splits);
        uint32_t st[2 * LOADS + 2];
        await_pairs<1 + LOADS>(st, number + 2, budget, states, STATES * STATE, [&](int i) {   // (past n: repeats)
            return i == 0 ? min(lc, n - 1) * STATE + HEAD_DIM : min(z + (i - 1) * PER_LOAD, n - 1) * STATE + col0 + 2 * c;
        }, [](int) { return 0; });
        wave_fence();   // (what was read there before)
        pm[lc] = __builtin_bit_cast(float, st[0]), pl[lc] = __builtin_bit_cast(float, st[1]);
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            *reinterpret_cast<float2 *>(pacc + min(z + i * PER_LOAD, n - 1) * HEAD_DIM + col0 + 2 * c) =
                float2{__builtin_bit_cast(float, st[2 + 2 * i]), __builtin_bit_cast(float, st[3 + 2 * i])};
        wave_fence();
        const int col = col0 + 2 * c;
        Joined s = join_states(n, col, ranges ? -INFINITY : own);
        // every slot masked: zeros (not where they stand for a query that did not come: then 0 / 0)
        if (s.top == -INFINITY && budget) s.o0 = s.o1 = 0.0f, s.total = 1.0f;
        if (lane < (HEAD_DIM / 2) / splits)
            put_word(a.e_attn + am * (A >> 1) + ((ah * HEAD_DIM + col) >> 1), pack_bf16_rne(s.o0 / s.total, s.o1 / s.total), number + 3);
    };
    auto join = [&](int nsc, uint64_t *words, uint32_t n, uint16_t *h_out) {
        lds_barrier();
        if (wave == 0) {
            const float2 s = tile_sum(1, 0, nsc);
            const uint32_t y = pack_bf16_rne(s.x, s.y);
            stream = pack_bf16_rne(low_bf16(stream) + low_bf16(y), high_bf16(stream) + high_bf16(y));
            if (stores()) {
                put_word(words + stream_word(), stream, n);
                if (h_out) ((gptr_w)(uintptr_t)h_out)[stream_word()] = stream;
            }
        }
    };
    auto publish_act = [&]() {
        lds_barrier();
        if (wave < slots_i) {
            const float2 g = tile_sum(0, 2 * wave * NSC, NSC), u = tile_sum(0, (2 * wave + 1) * NSC, NSC);
            const float x = g.x / (1.0f + __expf(-g.x)) * u.x, y = g.y / (1.0f + __expf(-g.y)) * u.y;
            if (stores())
                put_word(a.e_act + tile_row() * (I >> 1) + (wg + wave * G) * 8 + (lane & 7), pack_bf16_rne(x, y), number + 5);
        }
    };
    // the model's norm, a workgroup per row
    const auto last_norm = [&](int row) __attribute__((always_inline)) {
        const arg_ptr t = again();
        // add_rmsnorm_kernel's order of sums: four waves, eight neighbouring values of every 2048 per lane
        uint32_t x[4];
        if (wave < 4) {
            await_pairs<2>(x, number + 6, budget, a.e_out, M * ROW_WORDS,
                                    [&](int) { return 4 * tid; }, [&](int i) { return row * ROW_WORDS + i * 2; });
            float ss = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                ss = __builtin_fmaf(low_bf16(x[i]), low_bf16(x[i]), ss);
                ss = __builtin_fmaf(high_bf16(x[i]), high_bf16(x[i]), ss);
            }
            ss = wave_sum(ss);
            if (lane == 0) red[wave] = ss;
        }
        lds_barrier();
        if (wave < 4) {
            const float r = rsqrtf(__builtin_fmaf(((red[0] + red[1]) + red[2]) + red[3], 1.0f / H, t->eps));
            const u32x4_t w = ((gptr_u4)(uintptr_t)t->norm)[tid];
            u32x4_t y;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t n = pack_bf16_rne(low_bf16(x[e]) * r, high_bf16(x[e]) * r);
                y[e] = pack_bf16_rne(low_bf16(w[e]) * low_bf16(n), high_bf16(w[e]) * high_bf16(n));
            }
            ((__attribute__((address_space(1))) u32x4_t *)(uintptr_t)t->normed)[row * (H / 8) + tid] = y;
        }
    };

    // ---- who takes part, continued: the last of a group counts the group, the last of all finds that every workgroup has read the number: the next
    // launch's, and new counts.  Afterwards `rank` says whether this is the last of all.
    auto count_group = [&](Arrival &mine) {
        if (lane == 0) {
            const arg_ptr t = again();
            TrunkState *const state = t->state;
            const uint32_t n = t->n_groups;
            bool last = (mine.rank + 1) * n == (uint32_t)G;
            if (last) {
                __hip_atomic_store(&state->groups[wg & (n - 1)].arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                last = __hip_atomic_fetch_add(&state->complete, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == n;
            }
            if (last) {
                __hip_atomic_store(&state->number, mine.first + 8u + 8u * t->n_layers, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(&state->complete, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            mine.rank = last;
        }
    };
    // ... and the team: whoever offers first, the last of all with everyone, or one that has waited with those that have taken
    // a ticket by then.  Afterwards all threads know the number; returns the team's size, 0: the workspace is marked (by an
    // earlier launch, so all workgroups find the same), UNSETTLED: nobody has offered in TEAM_TICKS_LEAST, or not all may
    // take part.
    auto settle = [&](const Arrival &mine) {
        if (wave == TW - 1 && lane == 0) {
            const arg_ptr t = again();
            TrunkState *const state = t->state;
            const uint32_t now = mine.first + 8u, all = G;
            const uint32_t gave_up = __hip_atomic_load(&state->gave_up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            uint64_t seen = __hip_atomic_load(&state->team, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if ((uint32_t)t->most == all) {
                const uint64_t since = __builtin_readsteadycounter();
                while (!gave_up && (uint32_t)(seen >> 32) != now && __builtin_readsteadycounter() - since < TEAM_TICKS_LEAST) {
                    const uint64_t everyone = (uint64_t)now << 32 | all;
                    if (!mine.rank)
                        seen = __hip_atomic_load(&state->team, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    else if (__hip_atomic_compare_exchange_strong(&state->team, &seen, everyone, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                                  __HIP_MEMORY_SCOPE_AGENT))
                        seen = everyone;
                }
            }
            // (`joined[1]`: the rank in the team, for those that have no ticket)
            joined[0] = now;
            joined[1] = gave_up || (uint32_t)seen == all ? (uint32_t)wg : all;
            joined[2] = gave_up ? 0u : (uint32_t)(seen >> 32) == now ? (uint32_t)seen : UNSETTLED;
        }
        lds_barrier();
        number = __builtin_amdgcn_readfirstlane(joined[0]);
        return (int)__builtin_amdgcn_readfirstlane(joined[2]);
    };
    // The rest of it, out of the step's way: a ticket, and the offer once the wait is long enough for those that are there.
    auto settle_late = [&]() {
        if (wave == TW - 1 && lane == 0) {
            const arg_ptr t = again();
            TrunkState *const state = t->state;
            const uint32_t now = joined[0], most = t->most;
            const uint64_t since = __builtin_readsteadycounter();
            uint64_t seen = __hip_atomic_load(&state->team, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            uint32_t rank = G;
            if ((uint32_t)(seen >> 32) != now) {
                // The first one begins the count, once; then additions, which need no second try: 255 compare-and-swaps took 500 us.
                uint64_t tickets = __hip_atomic_load(&state->tickets, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if ((uint32_t)(tickets >> 32) != now)
                    (void)__hip_atomic_compare_exchange_strong(&state->tickets, &tickets, (uint64_t)now << 32, __ATOMIC_RELAXED,
                                                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                rank = (uint32_t)__hip_atomic_fetch_add(&state->tickets, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            while ((uint32_t)(seen >> 32) != now) {
                const uint32_t count = (uint32_t)__hip_atomic_load(&state->tickets, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const uint32_t here = min(count, most);
                const uint64_t waited = __builtin_readsteadycounter() - since;
                seen = __hip_atomic_load(&state->team, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if ((rank + 1 == most || waited * here >= (uint64_t)t->n_layers * TEAM_TICKS) && (uint32_t)(seen >> 32) != now) {
                    const uint64_t team = (uint64_t)now << 32 | here;
                    if (__hip_atomic_compare_exchange_strong(&state->team, &seen, team, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                             __HIP_MEMORY_SCOPE_AGENT))
                        seen = team;
                }
            }
            joined[1] = (uint32_t)seen == (uint32_t)G ? (uint32_t)wg : rank;   // everyone after all: each its own parts
            joined[2] = (uint32_t)seen;
        }
        lds_barrier();
    };

    auto mark = [&]() {
        if (budget == 0 && lane == 0)
            __hip_atomic_store(&again()->state->gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };

    // ---- the team is not the whole grid: every product's parts are dealt out to its members, one after the other
    if constexpr (SHARED) {
        number = __builtin_amdgcn_readfirstlane(joined[0]);
        const uint32_t found = __builtin_amdgcn_readfirstlane(joined[2]);
        lds_barrier();   // read by all waves before it is written again
        if (found == UNSETTLED) settle_late();
        const int rank = __builtin_amdgcn_readfirstlane(joined[1]), team = __builtin_amdgcn_readfirstlane(joined[2]);
        static_assert(TT == ROW_WORDS, "a word each");
        if (team == 0 && rank < M) {
            const arg_ptr t = again();
            for (gptr_w out : {(gptr_w)(uintptr_t)t->normed, (gptr_w)(uintptr_t)t->h_out})
                if (out) out[rank * ROW_WORDS + tid] = NOT_COME;
        }
        if (rank >= team) return;   // left out
        auto deal = [&](int parts, auto work) __attribute__((always_inline)) {
            for (int part = rank; part < parts; part += team) {
                forget();
                wg = part;
                work();
                lds_barrier();   // LDS is free for the next part
            }
        };
        const uint64_t *h_words = nullptr;   // the residual stream where the product before left it
        auto take_stream = [&](uint32_t n) {   // wave 0
            if (!h_words) return begin_stream();
            uint64_t w;
            for (;;) {
                w = stores() ? __hip_atomic_load(h_words + stream_word(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : (uint64_t)n << 32;
                if (__builtin_amdgcn_ballot_w64((uint32_t)(w >> 32) != n) == 0 || budget == 0) break;
                --budget;
            }
            stream = (uint32_t)(w >> 32) == n ? (uint32_t)w : NOT_COME;
        };
        for (int l = 0; l < a.n_layers; ++l, number += 8) {
            const layer_ptr L = (layer_ptr)(uintptr_t)a.layers + l;
            deal(G, [&]() {
                place_tiles();
                if (!slots_qkv) return;
                Rows<MW, C::P1> x;
                Built built;
                undefined(x);
                load(P_QKV, l);
                build_ahead(P_QKV, built);
                take_rows(P1, x, L->norm1, a.e_out, number - 2, l == 0 ? again()->cur : nullptr);
                normalise(P1, x, L->eps1);
                multiply_staged(P_QKV, built);
                publish_qkv();
            });
            deal(M * heads * splits, [&]() {
                place_pair();
                Slots kv;
                live = wave < my_waves ? counts(j_lo) : 0u;
                if (wave < my_waves) request(kv, L, j_lo);
                if (wave == 0) receive_token(L, true);
                lds_barrier();
                if (wave < my_waves) score_slots(L, kv);
                if (!ranges) return;
                lds_barrier();
                if (wave == 0) leave_state(own_score(L));
            });
            deal(M * heads * splits, [&]() {
                place_pair();
                if (wave != 0) return;
                wave_fence();
                receive_token(L, false);
                wave_fence();
                join_pair(own_score(L));
            });
            deal(G, [&]() {
                place_tiles();
                Built built;
                load(P_O, l);
                build_ahead(P_O, built);
                own_product(P_O, built, a.e_attn, A, number + 3, P_QKV, a.n_layers);
                if (!has_h) return;
                if (wave == 0) take_stream(number - 2);
                join(a.nsc_a, a.e_mid, number + 4, nullptr);
            });
            h_words = a.e_mid;
            deal(G, [&]() {
                place_tiles();
                if (!slots_i) return;
                Rows<MW, C::P2> x;
                Built built;
                undefined(x);
                load(P_GATE_UP, l);
                build_ahead(P_GATE_UP, built);
                take_rows(P2, x, L->norm2, a.e_mid, number + 4);
                normalise(P2, x, L->eps2);
                multiply_staged(P_GATE_UP, built);
                publish_act();
            });
            deal(G, [&]() {
                place_tiles();
                Built built;
                load(P_DOWN, l);
                build_ahead(P_DOWN, built);
                own_product(P_DOWN, built, a.e_act, I, number + 5, P_QKV, a.n_layers);
                if (!has_h) return;
                if (wave == 0) take_stream(number + 4);
                join(a.nsc_i, a.e_out, number + 6, l + 1 == a.n_layers ? again()->h_out : nullptr);
            });
            h_words = a.e_out;
        }
        number -= 8;
        if (again()->normed) deal(M, [&]() { last_norm(wg); });
        mark();
        return;
    }

    // ---- everyone is there
    begin_stream();
    load(P_QKV, 0);
    for (int l = 0; l < a.n_layers; ++l) {
        const layer_ptr L = (layer_ptr)(uintptr_t)a.layers + l;
        forget();
        opaque(am), opaque(ah), opaque(akv);
        // -------------------------------------------------------------- norm, q|k|v
        {
            Rows<MW, C::P1> x;
            Built built;
            undefined(x);
            build_ahead(P_QKV, built);
            if (l == 0 && wave == TW - 1) count_group(arrival);
            number += 8;
            if (slots_qkv) take_rows(P1, x, L->norm1, a.e_out, number - 2, l == 0 ? again()->cur : nullptr);   // the sixth exchange of the layer before
            load(P_O, l);
            if (slots_qkv) {
                normalise(P1, x, L->eps1);
                multiply_staged(P_QKV, built);
            }
        }
        if (l == 0) {
            const int team = settle(arrival);
            if (__builtin_expect(team != G, 0)) return share_out<C>(args, (lds_ptr)smem);
        }
        // -------------------------------------------------------------- rotary, append, attention
        // Two branches with the same barriers: the waves that attend rebuild o_proj's weights afterwards, the others
        // meanwhile, and neither's registers hold both the weights and the keys and values.
        Built built_o;
        if (wave >= my_waves) {
            publish_qkv();
            build_ahead(P_O, built_o);
            if (attends) lds_barrier();   // (with ranges every wave attends)
        } else {
            Slots kv;
            request(kv, L, j_lo);
            publish_qkv();
            if (wave == 0) receive_token(L, true);
            lds_barrier();
            score_slots(L, kv);
            if (ranges) lds_barrier();
            if (wave == 0) {
                const float own = own_score(L);
                if (ranges) leave_state(own);
                join_pair(own);
            }
            build_ahead(P_O, built_o);
        }
        // -------------------------------------------------------------- o_proj, joined with the residual stream
        own_product(P_O, built_o, a.e_attn, A, number + 3, P_GATE_UP, l);
        if (has_h) join(a.nsc_a, a.e_mid, number + 4, nullptr);
        // -------------------------------------------------------------- norm, gate|up, SiLU
        {
            Rows<MW, C::P2> x;
            Built built;
            undefined(x);
            build_ahead(P_GATE_UP, built);
            if (slots_i) take_rows(P2, x, L->norm2, a.e_mid, number + 4);
            load(P_DOWN, l);
            if (slots_i) {
                normalise(P2, x, L->eps2);
                multiply_staged(P_GATE_UP, built);
            }
        }
        if (slots_i) publish_act();
        // -------------------------------------------------------------- down_proj, joined with the residual stream
        {
            Built built;
            build_ahead(P_DOWN, built);
            own_product(P_DOWN, built, a.e_act, I, number + 5, P_QKV, l + 1);
            if (has_h) join(a.nsc_i, a.e_out, number + 6, l + 1 == a.n_layers ? again()->h_out : nullptr);
        }
    }
    if (again()->normed && wg < M) last_norm(wg);
    mark();
}

template <class C>
__device__ __attribute__((noinline)) void share_out(arg_ptr args, lds_ptr smem) {
    const uint64_t at = (uint64_t)(uintptr_t)args;   // (uniform; not known to be, where it arrives)
    args = (arg_ptr)(uintptr_t)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(at >> 32)) << 32 |
                                (uint32_t)__builtin_amdgcn_readfirstlane((int)at));
    trunk_step<C, true>(*(const TrunkArgs *)args, args, (uint8_t *)smem);
}

template <class C>
__global__ __launch_bounds__(TT) void decode_trunk_kernel(TrunkArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    trunk_step<C, false>(a, (arg_ptr)__builtin_amdgcn_kernarg_segment_ptr(), smem);
}

// ---------------------------------------------------------------- host side
struct TrunkPlan {
    int grid, build;                 // build: index of the kernel, -1: not this launch's
    size_t lds, words[6], bytes;     // words of the six exchanges, workspace bytes
};

constexpr size_t LDS_PER_CU = 160 * 1024;
constexpr size_t ALONE_LDS = 84 * 1024;   // more than half a compute unit's: one workgroup on each

// The kernels: up to 2 rows and up to 4, by the sums of squares of the first norm.
struct TrunkBuild {
    int rows, parts, splits;
    const void *kernel;
    size_t lds;
};
template <class C>
constexpr TrunkBuild trunk_build() {
    return {C::MW, C::P1, C::SPLITS, reinterpret_cast<const void *>(&decode_trunk_kernel<C>), C::LDS};
}
constexpr int TRUNK_N_BUILDS = 4;
const TrunkBuild TRUNK_BUILDS[TRUNK_N_BUILDS] = {trunk_build<TrunkCfg<2, 4>>(), trunk_build<TrunkCfg<2, 2>>(),
                                                 trunk_build<TrunkCfg<4, 2>>(), trunk_build<TrunkCfg<4, 1>>()};

// Waves that share a row in the sums of squares of the normalising launch vrl_int4_gemv_prepacked_norm_bf16 makes of `tiles`
// tiles (stage_x_norm: workgroups of 8 waves for many tiles, of 4 for few).
int norm_parts(int M, long tiles, int cus) {
    const int waves = tiles >= 5L * cus / 4 ? 8 : 4;
    int parts = 1;
    while (2 * parts * M <= waves && 2 * parts <= H / 512) parts *= 2;
    return parts;
}

bool trunk_plan(const vrl_trunk &t, TrunkPlan &plan) {
    plan.build = -1;
    const long A = (long)t.n_heads * HEAD_DIM, KV = (long)t.n_kv_heads * HEAD_DIM;
    if (t.n_layers < 1 || t.n_layers > 4096 || t.M < 1 || t.M > 4 || t.head_dim != HEAD_DIM || t.group_size != 128 ||
        t.n_heads < 1 || t.n_kv_heads < 1 || t.n_heads % t.n_kv_heads || t.L_max < 1 || t.L_max > 8192)
        return false;
    if (t.hidden != H || t.inter < 256 || t.inter % 256 || t.inter > 16384 ||
        A > 8192 || A % 256)
        return false;
    const int G = device_cu_count();
    if (pp_nsc((int)A) > TW || pp_nsc(t.inter) > TW || H / 16 > G) return false;
    auto slots = [&](long tiles) { return (tiles + G - 1) / G; };
    if (slots((A + 2 * KV) / 16) * NSC > TW || slots(t.inter / 16) * 2 * NSC > TW) return false;
    const long pairs = (long)t.M * t.n_heads, splits = pairs <= 32 ? 8 : pairs <= 64 ? 4 : pairs <= 128 ? 2 : 1;
    const int rows = t.M <= 2 ? 2 : 4, parts = norm_parts(t.M, (A + 2 * KV) / 16, G);
    if (pairs * splits > G || norm_parts(t.M, t.inter / 16, G) != 8 / rows) return false;
    for (int i = 0; i < TRUNK_N_BUILDS; ++i) {
        const TrunkBuild &b = TRUNK_BUILDS[i];
        if (b.rows == rows && b.parts == parts && b.splits == splits) plan.build = i;
    }
    if (plan.build < 0) return false;
    plan.grid = G;
    plan.lds = std::max(TRUNK_BUILDS[plan.build].lds, ALONE_LDS);
    const size_t words[6] = {(size_t)t.M * (A + 2 * KV) / 2,
                             (size_t)t.M * t.n_heads * STATES * STATE,
                             (size_t)t.M * A / 2, (size_t)t.M * t.hidden / 2, (size_t)t.M * t.inter / 2,
                             (size_t)t.M * t.hidden / 2};
    plan.bytes = sizeof(TrunkState);
    for (int i = 0; i < 6; ++i) {
        plan.words[i] = words[i];
        plan.bytes += (words[i] * 8 + 255) / 256 * 256;
    }
    return true;
}

// Whether this device runs the build as one cooperative launch; the LDS limit is raised on the way.
int trunk_ready(const TrunkPlan &plan) {
    int dev = 0, coop = 0, per_cu = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev);
    if (e != hipSuccess) return (int)e;
    if (!coop) return VRL_INT4_ELIMIT;
    static std::atomic<uint64_t> ready[TRUNK_N_BUILDS];   // by build, a bit per device
    const uint64_t bit = 1ull << (dev & 63);
    if (dev < 64 && (ready[plan.build].load(std::memory_order_relaxed) & bit)) return VRL_INT4_OK;
    const void *kernel = TRUNK_BUILDS[plan.build].kernel;
    e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_PER_CU);
    if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, TT, LDS_PER_CU);
    if (e != hipSuccess) return (int)e;
    if (per_cu < 1) return VRL_INT4_ELIMIT;
    ready[plan.build].fetch_or(bit, std::memory_order_relaxed);
    return VRL_INT4_OK;
}

}  // namespace

extern "C" size_t vrl_decode_trunk_workspace_bytes(const vrl_trunk *trunk) {
    TrunkPlan plan;
    if (!trunk || !trunk_plan(*trunk, plan) || trunk_ready(plan) != VRL_INT4_OK) return 0;
    return plan.bytes;
}

extern "C" int vrl_decode_trunk_bf16(const vrl_trunk *trunk, void *hip_stream) {
    if (!trunk) return VRL_INT4_ENULL;
    const vrl_trunk &t = *trunk;
    if (!t.layers || !t.x || !t.mask || !t.position || !t.cos || !t.sin || !t.workspace || (t.normed && !t.norm) ||
        (!t.normed && !t.h_out))
        return VRL_INT4_ENULL;
    TrunkPlan plan;
    if (!trunk_plan(t, plan)) return VRL_INT4_ESHAPE;
    const int rc = trunk_ready(plan);
    if (rc != VRL_INT4_OK) return rc;
    if (t.workspace_bytes < plan.bytes) return VRL_INT4_EPLAN;
    auto off = [](const void *p, uintptr_t n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) != 0; };
    if (off(t.layers, 16) || off(t.x, 16) || off(t.cos, 4) || off(t.sin, 4) || off(t.norm, 16) || off(t.normed, 16) ||
        off(t.h_out, 16) || off(t.position, 8) || off(t.workspace, 256))
        return VRL_INT4_EALIGN;
    TrunkArgs a;
    memset(&a, 0, sizeof a);
    a.layers = t.layers;
    a.cur = static_cast<const uint16_t *>(t.x);
    a.cos = static_cast<const uint16_t *>(t.cos);
    a.sin = static_cast<const uint16_t *>(t.sin);
    a.norm = static_cast<const uint16_t *>(t.norm);
    a.mask = static_cast<const uint8_t *>(t.mask);
    a.position = reinterpret_cast<const long long *>(t.position);
    a.position_stride = t.position_per_row ? 1 : 0;
    a.normed = static_cast<uint16_t *>(t.normed);
    a.h_out = static_cast<uint16_t *>(t.h_out);
    a.eps = t.eps;
    a.n_layers = t.n_layers;
    a.M = t.M;
    a.A = t.n_heads * HEAD_DIM;
    a.KV = t.n_kv_heads * HEAD_DIM;
    a.I = t.inter;
    a.heads = t.n_heads;
    a.kv_heads = t.n_kv_heads;
    a.L_max = t.L_max;
    a.budget = t.wait_limit ? t.wait_limit : TRUNK_BUDGET;
    a.grid = plan.grid;
    a.most = t.max_workgroups ? (int)std::min(t.max_workgroups, (uint32_t)plan.grid) : plan.grid;
    a.n_groups = ARRIVALS;
    while (plan.grid % a.n_groups) a.n_groups /= 2;
    a.nsc_a = pp_nsc(a.A);
    a.nsc_i = pp_nsc(a.I);
    a.split_from = t.split_from > 0 ? t.split_from : INT32_MAX;
    uint8_t *ws = static_cast<uint8_t *>(t.workspace);
    a.state = reinterpret_cast<TrunkState *>(ws);
    uint64_t **const at[6] = {&a.e_qkv, &a.e_part, &a.e_attn, &a.e_mid, &a.e_act, &a.e_out};
    size_t offset = sizeof(TrunkState);
    for (int i = 0; i < 6; ++i) {
        *at[i] = reinterpret_cast<uint64_t *>(ws + offset);
        offset += (plan.words[i] * 8 + 255) / 256 * 256;
    }
    void *args[] = {&a};
    const hipError_t e = hipLaunchCooperativeKernel(TRUNK_BUILDS[plan.build].kernel, dim3(plan.grid), dim3(TT), args,
                                                    (unsigned)plan.lds, reinterpret_cast<hipStream_t>(hip_stream));
    if (e != hipSuccess) (void)hipGetLastError();   // a caller may go on with the list: not left for the next check to find
    return (int)e;
}
