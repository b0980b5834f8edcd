// Prompt attention in 32-bit for heads of 32 or 64 over pages of at least 32 keys, on the bfloat16 matrix cores: every number is three bfloat16 ones (number_pieces.h), and a
// product of two numbers six products of pieces, as in gemm_pieces.h. Included by attention.hip behind attention_stream.h, whose way through queries and keys this is: a
// block owns 32 queries of one (request, head), each of its four waves holds all of them and walks every fourth tile of 32 keys with softmax statistics of its own; keys and
// values stream from the pages into LDS that only the wave reads; the waves' results are combined at the end.
//
// What bounds it: what a SIMD can issue. A tile is 48 matrix instructions (1,536 cycles) and some 730 vector instructions, most of which split the tile's keys, its values and
// its weights, the rest is the softmax. So the loop has two halves that each carry both kinds, a few vector instructions behind every two products: the scores of the next tile
// beside this tile's weights and their splitting, and this tile's value products beside the splitting of its values, the loads, and the splitting of the keys of the tile
// after the next. A tile's numbers go from LDS into registers a tile before they are used, so that one place for keys and one for values is enough, and two blocks share
// a compute unit: one's waits run under the other's instructions (blocks of 64 queries, which split a tile's keys and values for twice the products but leave room for one
// block alone, us: two prompts of 1,024 tokens x 12 heads of 64 46 and 42 so, eight of 256 30 and 24, one of 4,096 217 and 204).
// With the 32-bit instruction, a quarter of the pieces' rate, one block a unit and the library's expf -> now, alone in a loop, us: those 58.8 -> 39.6, 32.3 -> 21.9 and 329 -> 194, five
// prompts of 67 to 1,001 70.3 -> 39.8, 512 queries on 7,680 cached keys 192 -> 120, 32 prompts of 70 43.7 -> 25.7, one of 66 9.2 -> 8.5, of 128 9.4 -> 8.6; four of 512 over a window of 128
// with a cap 41.0 -> 24.7. (The blocks' shapes above were compared before the queries' check lost its branches, 0.8 to 1.4 us a block.)
// In a sum of six products the five small ones come first. A score's sum starts at zero, so the large one is rounded once for sixteen numbers (the 32-bit instruction: eight times);
// the values' sum runs over all tiles and takes all six, six roundings for sixteen keys, in which the small ones are lost once it is long (a second sum for them, as gemm_pieces.h
// has it, would take 32 registers that are not there). Against 64 bits, normally distributed numbers: 2.6e-7 -> 1.5e-7 for the first of these, 8.7e-7 -> 7.3e-7 over 8,192 keys.
// (The instruction cuts its sums off downwards: errors lie 2e-8 to 7e-8 of the results' mean magnitude below zero on average, with the 32-bit instruction 1e-8 or less.)
// What pieces cannot hold: a number that is not finite or rounds to infinity has no pieces, and whatever it meets comes out as no number; numbers below 2^-110 lose
// their third piece, below 2^-134 all of them, and weights below 2^-126 are 0. So a weighted sum of values may be off by 2^-126 for each key, times the largest value of its
// column, or by 2^-134 for each, times its weight. Rows with results that are not finite, with weighted sums below 2^-90 or below 2^-90 times the largest value of their column
// (zeros among them, unless every value of the column is zero), or whose queries hold numbers beyond 2^64 or below 2^-90 (which could make up for keys that lost their pieces), are
// taken again one by one in 32-bit (general_row), but for queries that hold what is no number: nothing else can come of them. (General_row ends at the first key whose score is none, so
// that a key which is no number costs the rows behind it a few steps and not a walk: two prompts of 1,024 tokens x 12 heads, of which key 3 is none, 1,484 -> 72 us.)
#pragma once

#include "number_pieces.h"

#include <type_traits>
#include <utility>

namespace prefill_pieces {

using pieces::i32x4;
using prefill_stream::KEYS;
using prefill_stream::Layout;
using prefill_stream::lds_address;
using prefill_stream::most_tiles;
using prefill_stream::tile_of_slot;
using prefill_stream::wait_vmcnt;
using prefill_stream::CAPPED;
using prefill_stream::CAUSAL;
using prefill_stream::KEPT;
using prefill_stream::MASKED;

constexpr int WAVES = 4, QUERIES = 32;

// A wave's LDS: a tile of keys and one of values.
template <int HD>
constexpr int wave_bytes() {
    return 2 * Layout<float, HD, WAVES>::TILE_BYTES;
}

// e^x for x <= 0 (0 for minus infinity and whatever is below 2^-126, x < -87.3: the hardware's 2^x has no subnormal results; no number stays one): 2^t of the rounded
// t = x log2(e), and what the rounding left by the first two terms of its series, x - t ln 2 in two parts. With an exact 2^t within one unit in the last place, 0.33 of it on
// average (the library's expf: 0.64 and 0.25). Six instructions, the library's expf some fourteen.
__device__ __forceinline__ float exp_below(float x) {
    x = __builtin_elementwise_maximum(x, -128.0f);   // (keeps what is no number, and minus infinity from becoming that below)
    const float t = x * 1.44269504f;
    float left = __builtin_fmaf(-t, 0.693147182f, x);   // ln 2 = 0.693147182 - 1.90465421e-9
    left = __builtin_fmaf(t, 1.90465421e-9f, left);
    const float whole = __builtin_amdgcn_exp2f(t);
    return __builtin_fmaf(whole, left, whole);
}

// The LDS reads of a tile as instructions (through the compiler each would wait for all loads into LDS that are under way), a block of them with their wait, so that nothing can
// move a register that is still on its way.
// A lane's eight values of a fragment: keys 0 to 3 and 8 to 11 from `address` on, ROW_BYTES apart; with those of the fragment behind it, keys 16 to 19 and 24 to 27.
template <int ROW_BYTES>
__device__ __forceinline__ void read_values(unsigned address, i32x4 (&low)[2], i32x4 (&high)[2]) {
    int value[16];
    const unsigned behind = address + 16 * ROW_BYTES;
    asm volatile(
        "ds_read_b32 %0, %16 offset:%18\n\t"
        "ds_read_b32 %1, %16 offset:%19\n\t"
        "ds_read_b32 %2, %16 offset:%20\n\t"
        "ds_read_b32 %3, %16 offset:%21\n\t"
        "ds_read_b32 %4, %16 offset:%22\n\t"
        "ds_read_b32 %5, %16 offset:%23\n\t"
        "ds_read_b32 %6, %16 offset:%24\n\t"
        "ds_read_b32 %7, %16 offset:%25\n\t"
        "ds_read_b32 %8, %17 offset:%18\n\t"
        "ds_read_b32 %9, %17 offset:%19\n\t"
        "ds_read_b32 %10, %17 offset:%20\n\t"
        "ds_read_b32 %11, %17 offset:%21\n\t"
        "ds_read_b32 %12, %17 offset:%22\n\t"
        "ds_read_b32 %13, %17 offset:%23\n\t"
        "ds_read_b32 %14, %17 offset:%24\n\t"
        "ds_read_b32 %15, %17 offset:%25\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(value[0]), "=&v"(value[1]), "=&v"(value[2]), "=&v"(value[3]), "=&v"(value[4]), "=&v"(value[5]), "=&v"(value[6]), "=&v"(value[7]), "=&v"(value[8]), "=&v"(value[9]), "=&v"(value[10]), "=&v"(value[11]), "=&v"(value[12]), "=&v"(value[13]), "=&v"(value[14]), "=&v"(value[15])
        : "v"(address), "v"(behind), "n"(0 * ROW_BYTES), "n"(1 * ROW_BYTES), "n"(2 * ROW_BYTES), "n"(3 * ROW_BYTES), "n"(8 * ROW_BYTES), "n"(9 * ROW_BYTES), "n"(10 * ROW_BYTES), "n"(11 * ROW_BYTES)
        : "memory");
#pragma unroll
    for (int e = 0; e < 8; e++) low[e / 4][e % 4] = value[e], high[e / 4][e % 4] = value[8 + e];
}

// Sixteen bytes from each of eight places (or four).
__device__ __forceinline__ void read_keys(const unsigned (&address)[4][2], i32x4 (&out)[4][2]) {
    asm volatile(
        "ds_read_b128 %0, %8\n\t"
        "ds_read_b128 %1, %9\n\t"
        "ds_read_b128 %2, %10\n\t"
        "ds_read_b128 %3, %11\n\t"
        "ds_read_b128 %4, %12\n\t"
        "ds_read_b128 %5, %13\n\t"
        "ds_read_b128 %6, %14\n\t"
        "ds_read_b128 %7, %15\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(out[0][0]), "=&v"(out[0][1]), "=&v"(out[1][0]), "=&v"(out[1][1]), "=&v"(out[2][0]), "=&v"(out[2][1]), "=&v"(out[3][0]), "=&v"(out[3][1])
        : "v"(address[0][0]), "v"(address[0][1]), "v"(address[1][0]), "v"(address[1][1]), "v"(address[2][0]), "v"(address[2][1]), "v"(address[3][0]), "v"(address[3][1])
        : "memory");
}
__device__ __forceinline__ void read_keys(const unsigned (&address)[2][2], i32x4 (&out)[2][2]) {
    asm volatile(
        "ds_read_b128 %0, %4\n\t"
        "ds_read_b128 %1, %5\n\t"
        "ds_read_b128 %2, %6\n\t"
        "ds_read_b128 %3, %7\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(out[0][0]), "=&v"(out[0][1]), "=&v"(out[1][0]), "=&v"(out[1][1])
        : "v"(address[0][0]), "v"(address[0][1]), "v"(address[1][0]), "v"(address[1][1])
        : "memory");
}

// The larger of a lane's number and that of the lane 32 further on or back. (The second copy is hidden from the compiler, which takes the exchange of one register with itself for
// the register itself.)
__device__ __forceinline__ float larger_of_halves(float x) {
    unsigned mine = __builtin_bit_cast(unsigned, x), copy = mine;
    asm volatile("" : "+v"(copy));
    const auto halves = __builtin_amdgcn_permlane32_swap(mine, copy, false, false);
    return fmaxf(__builtin_bit_cast(float, (unsigned)halves[0]), __builtin_bit_cast(float, (unsigned)halves[1]));
}

template <typename F, int... I>
__device__ __forceinline__ void stream_for_each(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void stream_for(F&& f) {   // a loop whose index is a constant in its body
    stream_for_each(static_cast<F&&>(f), std::make_integer_sequence<int, N>{});
}

// FORM: attention_stream.h.
template <int HD, int FORM>
__device__ __forceinline__ void pieces_block(
    int place, const float* __restrict__ q, int q_stride, const float* __restrict__ k_pages, const float* __restrict__ v_pages, float* __restrict__ out, int out_stride,
    const int* __restrict__ q_starts, const int* __restrict__ context_lens, const int* __restrict__ block_tables, int max_blocks, int n_requests, int n_heads,
    int n_kv_heads, int page_shift, int given_window, float scale, ScoreOptions options) {
    typedef Layout<float, HD, WAVES> L;
    const int window = FORM == CAUSAL ? 0 : given_window, chunk = FORM == CAUSAL ? 0 : options.chunk;
    constexpr int KS = HD / 16, DT = HD / 32, WAVE_BYTES = wave_bytes<HD>();
    static_assert(WAVE_BYTES >= QUERIES * HD * 4 && WAVE_BYTES >= MAX_HEAD * 4, "what a wave leaves takes the place of its tiles");
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    __shared__ float stats_lds[WAVES][QUERIES][2];
    __shared__ __attribute__((aligned(16))) float largest_lds[WAVES][HD];
    __shared__ unsigned again;   // bit r: row r of the block is taken once more

    const int tid = threadIdx.x, lane = tid % WAVE;
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int lane32 = lane % 32, half = lane / 32;
    // (places and heads: attention_stream.h)
    const int slot = place / n_heads, at = place % n_heads;
    const int head = at < (n_heads & ~7) ? (at & ~7) | (place & 7) : at;
    int request, q_first, q_len, context, query_tile;
    if (!tile_of_slot<QUERIES>(slot, n_requests, q_starts, context_lens, request, q_first, q_len, context, query_tile)) return;
    const int tile_q0 = query_tile * QUERIES;
    const int kv_head = head / (n_heads / n_kv_heads);
    const int* table = block_tables + (size_t)request * max_blocks;
    const int page_mask = (1 << page_shift) - 1;

    const int block_last_position = context + min(tile_q0 + QUERIES, q_len) - 1;
    const int block_first_key = first_visible_key(context + tile_q0, window, chunk);
    const int first_base = (block_first_key / KEYS) * KEYS;
    // with kept first keys: the tiles that hold them come first, the tiles between them and the window are passed over
    const int kept_tiles = FORM == KEPT ? min((options.keep + KEYS - 1) / KEYS, first_base / KEYS) : 0;
    const int n_tiles = kept_tiles + (block_last_position - first_base) / KEYS + 1;
    const int n_mine = n_tiles > wave ? (n_tiles - wave + WAVES - 1) / WAVES : 0;  // tiles wave, wave + WAVES, ...

    // One half (keys or values) of this wave's i-th tile, into the one place there is for each; beyond the wave's last tile that one again, never used (the count of loads in flight is then the
    // same in every step), and behind the last stored key that key's row again, masked by position.
    unsigned char* const wave_lds = lds + wave * WAVE_BYTES;
    auto tile_base = [&](int i) {
        const int tile = wave + WAVES * min(i, n_mine - 1);
        return FORM == KEPT && tile < kept_tiles ? tile * KEYS : first_base + (tile - kept_tiles) * KEYS;
    };
    struct Half {   // of a tile, about to be asked for
        const unsigned char* base;
        int last_row, place;
    };
    auto half_of = [&](int i, int page, bool is_value) {
        const int k_base = tile_base(i);
        return Half{reinterpret_cast<const unsigned char*>((is_value ? v_pages : k_pages) + ((((size_t)page * n_kv_heads + kv_head) << page_shift) + (k_base & page_mask)) * HD),
                    block_last_position - k_base, is_value ? L::TILE_BYTES : 0};
    };
    const int load_row = lane / L::PPR, load_piece = lane % L::PPR;
    auto issue_load = [&](const Half& half_tile, int l, bool is_value) {
        const int row = l * L::ROWS_PER_LOAD + load_row, piece = load_piece ^ (is_value ? L::v_turn(row) : L::k_turn(row));
        __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(half_tile.base + (unsigned)(min(row, half_tile.last_row) * L::ROW_BYTES + piece * 16)),
                                         (void __attribute__((address_space(3)))*)(wave_lds + half_tile.place + l * 1024), 16, 0, 0);
    };
    auto issue = [&](int i, int page, bool is_value) {
        const Half half_tile = half_of(i, page, is_value);
#pragma unroll
        for (int l = 0; l < L::LOADS; l++) issue_load(half_tile, l, is_value);
    };
    int page_v = 0, page_k = 0;   // of tiles i + 1 and i + 3
    if (n_mine > 0) {
        const int page0 = table[tile_base(0) >> page_shift];
        issue(0, page0, false);
        issue(0, page0, true);
    }

    // The queries' pieces, the second operand of the scores: step s holds columns 16 s + 8 half .. + 8 of this lane's query.
    bf16x8 q_piece[KS][3];
    unsigned largest_q = 0, smallest_q = ~0u;   // bits of the magnitudes, of the smallest one less (0, which has pieces, is then the largest there is)
    const int own_query = tile_q0 + lane32;
    // a lane beyond the portion's end takes the portion's first row and position -1: no key is at or before it, so every score of it is masked
    const int q_position = own_query < q_len ? context + own_query : -1;
    const float* q_row = q + (size_t)(q_first + (own_query < q_len ? own_query : 0)) * q_stride + head * HD;
#pragma unroll
    for (int s = 0; s < KS; s++) {
        i32x4 raw[2];
#pragma unroll
        for (int e = 0; e < 2; e++) raw[e] = *reinterpret_cast<const i32x4*>(q_row + 16 * s + 8 * half + 4 * e);
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const unsigned magnitude = (unsigned)raw[e / 4][e % 4] & 0x7fffffffu;
            largest_q = max(largest_q, magnitude), smallest_q = min(smallest_q, magnitude - 1u);
        }
#pragma unroll
        for (int e = 0; e < 4; e++) pieces::split_pair(raw, e, q_piece[s]);
    }
    auto rows_of = [](bool lanes) {   // the rows of which one of the two lanes
        const unsigned long long which = __ballot(lanes);
        return (unsigned)which | (unsigned)(which >> 32);
    };
    // queries that pieces may not be enough for, and those that hold what is no number: their results are none either, however they are taken
    const unsigned none_rows = rows_of(largest_q > 0x7f800000u);
    const unsigned odd_queries = rows_of((largest_q > __builtin_bit_cast(unsigned, 0x1p64f)) | (smallest_q < __builtin_bit_cast(unsigned, 0x1p-90f) - 1u));

    f32x16 acc_o[DT];
    float running_max = -INFINITY, running_sum = 0.0f;
    float largest[DT];   // magnitude of the values this lane has split, of its column of every 32 (no number if one of them is)
#pragma unroll
    for (int i2 = 0; i2 < DT; i2++) largest[i2] = 0.0f;
    auto split_values = [&](const i32x4 (&raw)[2], int e, bf16x8 (&out)[3], float& so_far) {   // pieces of pair e
        pieces::split_pair(raw, e, out);
        const int first = raw[e / 2][e % 2 * 2], second = raw[e / 2][e % 2 * 2 + 1];
        so_far = __builtin_elementwise_maximum(__builtin_elementwise_maximum(so_far, fabsf(__builtin_bit_cast(float, first))), fabsf(__builtin_bit_cast(float, second)));
    };
#pragma unroll
    for (int i2 = 0; i2 < DT; i2++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc_o[i2][v] = 0.0f;

    // A tile's keys: fragment s (32 keys x 16 columns): lane l holds key l % 32, columns 16 s + 8 (l / 32) .. + 8.
    bf16x8 k_piece[KS][3];
    i32x4 k_raw[KS][2];
    unsigned k_at[KS][2];   // of this lane's pieces in a tile
#pragma unroll
    for (int s = 0; s < KS; s++)
#pragma unroll
        for (int e = 0; e < 2; e++) k_at[s][e] = lds_address(wave_lds + lane32 * L::ROW_BYTES + (((4 * s + 2 * half + e) ^ L::k_turn(lane32)) * 16));
    auto split_keys = [&] {
#pragma unroll
        for (int s = 0; s < KS; s++)
#pragma unroll
            for (int e = 0; e < 4; e++) pieces::split_pair(k_raw[s], e, k_piece[s]);
    };
    // The products of pieces, the smallest first.
    constexpr int FIRST[6] = {2, 0, 1, 1, 0, 0}, SECOND[6] = {0, 2, 1, 0, 1, 0};
    // S^T = K . Q^T: a lane holds one query's scores for sixteen of the tile's keys, 8 (v / 4) + 4 half + v % 4.
    auto scores = [&] {
        f32x16 sums;
#pragma unroll
        for (int v = 0; v < 16; v++) sums[v] = 0.0f;
#pragma unroll
        for (int c = 0; c < 6; c++)
#pragma unroll
            for (int s = 0; s < KS; s++) sums = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k_piece[s][FIRST[c]], q_piece[s][SECOND[c]], sums, 0, 0, 0);
        return sums;
    };

    // Loads, in order: K0 V0 K1 K2, then with tile i: V(i + 1) K(i + 3).
    f32x16 s_acc, s_next;   // this tile's scores and the next one's
    if (n_mine > 0) {
        const int page1 = table[tile_base(1) >> page_shift], page2 = table[tile_base(2) >> page_shift];
        page_v = page1;
        page_k = table[tile_base(3) >> page_shift];
        wait_vmcnt<L::LOADS>();
        read_keys(k_at, k_raw);
        issue(1, page1, false);
        split_keys();
        s_acc = scores();
        wait_vmcnt<0>();
        read_keys(k_at, k_raw);
        issue(2, page2, false);
        split_keys();
    }

    for (int i = 0; i < n_mine; i++) {   // (two tiles a turn, the scores' registers changing places, is no faster: 46.7 and 45.9 us with blocks of 64 queries)
        const int page_next_v = table[tile_base(i + 2) >> page_shift], page_next_k = table[tile_base(i + 4) >> page_shift];
        const int k0 = FORM == KEPT ? tile_base(i) : first_base + (wave + WAVES * i) * KEYS;
        const unsigned char* v_tile = wave_lds + L::TILE_BYTES;

        // ---- cap, mask (only where the tile touches the diagonal, a window or the portion's end) and maximum ----
        const bool interior = window == 0 && chunk == 0 && tile_q0 + 31 < q_len && k0 + KEYS - 1 <= context + tile_q0;
        if ((FORM == CAPPED || FORM == KEPT) && options.softcap > 0.0f) {   // a capped score, left divided by the scale as the plain ones are: cap tanh(scale s / cap) / scale
            const float back = options.softcap / scale, into = scale / options.softcap;
#pragma unroll
            for (int v = 0; v < 16; v++) s_acc[v] = back * tanhf(s_acc[v] * into);
        }
        if (!interior) {
            const int first_allowed = q_position < 0 ? 0 : first_visible_key(q_position, window, chunk);
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int key = k0 + 4 * half + 8 * (v / 4) + (v % 4);
                const bool allowed = (key <= q_position) & ((key >= first_allowed) | (FORM == KEPT && key < options.keep));
                s_acc[v] = allowed ? s_acc[v] : -INFINITY;
            }
        }
        float tile_max = -INFINITY;
#pragma unroll
        for (int v = 0; v < 16; v++) tile_max = fmaxf(tile_max, s_acc[v]);
        tile_max = larger_of_halves(tile_max) * scale;
        const float new_max = fmaxf(running_max, tile_max);
        const float safe_max = new_max == -INFINITY ? 0.0f : new_max;  // a query with no key yet
        if (__any(new_max > running_max)) {  // some query's maximum rose: what has been summed so far shrinks
            const float rescale = exp_below(running_max - safe_max);
            running_sum *= rescale;
#pragma unroll
            for (int i2 = 0; i2 < DT; i2++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc_o[i2][v] *= rescale;
        }
        running_max = new_max;

        // ---- the scores of tile i + 1, and between their products this tile's weights and the weights' pieces: units of one weight or of one pair to split ----
        __builtin_amdgcn_sched_barrier(0);
        bf16x8 p_piece[2][3];   // the second operand of the values: keys 0-15 and 16-31 of the tile
        i32x4 p_raw[2][2];
        constexpr int SCORES = 6 * KS, WEIGHTS = 24, AT_ONCE = 2;   // two products and their units to a group the scheduler may order
        stream_for<SCORES / AT_ONCE>([&](auto group) {
            constexpr int G = decltype(group)::value * AT_ONCE;
            stream_for<AT_ONCE>([&](auto n) {
                constexpr int N = G + decltype(n)::value, c = N / KS, s = N % KS;
                f32x16 start = s_next;
                if constexpr (N == 0) {
#pragma unroll
                    for (int v = 0; v < 16; v++) start[v] = 0.0f;
                }
                s_next = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k_piece[s][FIRST[c]], q_piece[s][SECOND[c]], start, 0, 0, 0);
            });
            constexpr int FROM = G * WEIGHTS / SCORES, TO = (G + AT_ONCE) * WEIGHTS / SCORES;
            stream_for<TO - FROM>([&](auto n) {
                constexpr int U = FROM + decltype(n)::value, slab = U / 12, u = U % 12;
                if constexpr (u < 8) {
                    const float p = exp_below(__builtin_fmaf(s_acc[8 * slab + u], scale, -safe_max));
                    running_sum += p;
                    p_raw[slab][u / 4][u % 4] = __builtin_bit_cast(int, p);
                } else {
                    pieces::split_pair(p_raw[slab], u - 8, p_piece[slab]);
                }
            });
            __builtin_amdgcn_sched_barrier(0);
        });

        // ---- O^T += V^T . P^T, and between the products the pieces of the values behind, the loads, and the pieces of the keys of tile i + 2 ----
        const Half next_v = half_of(i + 1, page_v, true), next_k = half_of(i + 3, page_k, false);
        wait_vmcnt<L::LOADS>();   // V(i) has landed
        i32x4 v_raw[2][DT][2];
#pragma unroll
        for (int i2 = 0; i2 < DT; i2++) {
            // fragment (slab, i2): lane l holds column 32 i2 + l % 32 of keys 16 slab + 4 half .. + 4 and 8 behind them, the keys whose weights its other operand holds
            const unsigned address = lds_address(v_tile + (4 * half) * L::ROW_BYTES + (i2 * 32 + lane32) * 4);
            read_values<L::ROW_BYTES>(address, v_raw[0][i2], v_raw[1][i2]);
        }
        wait_vmcnt<0>();   // K(i + 2) has
        read_keys(k_at, k_raw);
        __builtin_amdgcn_sched_barrier(0);
        constexpr int FRAGMENTS = 2 * DT, EACH = 6, VALUES = FRAGMENTS * EACH, OTHERS = 2 * L::LOADS + 4 * KS;
        bf16x8 v_piece[FRAGMENTS][3];
#pragma unroll
        for (int e = 0; e < 4; e++) split_values(v_raw[0][0], e, v_piece[0], largest[0]);
        stream_for<VALUES / AT_ONCE>([&](auto group) {
            constexpr int G = decltype(group)::value * AT_ONCE, F = G / EACH;
            stream_for<AT_ONCE>([&](auto n) {
                constexpr int N = G + decltype(n)::value, f = N / EACH, c = N % EACH;
                acc_o[f % DT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v_piece[f][FIRST[c]], p_piece[f / DT][SECOND[c]], acc_o[f % DT], 0, 0, 0);
            });
            if constexpr (F + 1 < FRAGMENTS) {
                constexpr int FROM = G % EACH * 4 / EACH, TO = (G % EACH + AT_ONCE) * 4 / EACH;
                stream_for<TO - FROM>([&](auto n) { split_values(v_raw[(F + 1) / DT][(F + 1) % DT], FROM + decltype(n)::value, v_piece[F + 1], largest[(F + 1) % DT]); });
            }
            constexpr int FROM = G * OTHERS / VALUES, TO = (G + AT_ONCE) * OTHERS / VALUES;
            stream_for<TO - FROM>([&](auto n) {
                constexpr int U = FROM + decltype(n)::value;
                if constexpr (U < 2 * L::LOADS) issue_load(U < L::LOADS ? next_v : next_k, U % L::LOADS, U < L::LOADS);
                else pieces::split_pair(k_raw[(U - 2 * L::LOADS) / 4], (U - 2 * L::LOADS) % 4, k_piece[(U - 2 * L::LOADS) / 4]);
            });
            __builtin_amdgcn_sched_barrier(0);
        });
        page_v = page_next_v;
        page_k = page_next_k;
        s_acc = s_next;
    }
    // the loads asked for beyond the last tile land before the tiles' place is written over
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");

    // ---- the waves' partial results, combined: each wave writes its own where its tiles lay, then finishes a share ----
    float* partial = reinterpret_cast<float*>(lds + wave * WAVE_BYTES);
    running_sum += __shfl_xor(running_sum, 32, WAVE);
    if (half == 0) {
        stats_lds[wave][lane32][0] = running_max;
        stats_lds[wave][lane32][1] = running_sum;
    }
#pragma unroll
    for (int i2 = 0; i2 < DT; i2++) {
        const float of_column = larger_of_halves(largest[i2]);
        if (half == 0) largest_lds[wave][i2 * 32 + lane32] = of_column;
    }
#pragma unroll
    for (int i2 = 0; i2 < DT; i2++)
#pragma unroll
        for (int v = 0; v < 16; v++) partial[(i2 * 16 + v) * WAVE + lane] = acc_o[i2][v];
    if (tid == 0) again = 0;
    __syncthreads();
    bool odd = odd_queries >> lane32 & 1;
    f32x4 o[DT];   // of every 32 columns wave w finishes 8 w .. + 8
    if (own_query < q_len) {
        float best = -INFINITY;
#pragma unroll
        for (int w = 0; w < WAVES; w++) best = fmaxf(best, stats_lds[w][lane32][0]);
        float weight[WAVES], total = 0.0f;
#pragma unroll
        for (int w = 0; w < WAVES; w++) {
            weight[w] = expf(stats_lds[w][lane32][0] - best);  // a wave that saw no key: a weight of 0
            total += weight[w] * stats_lds[w][lane32][1];
        }
        if (options.sinks) total += expf(options.sinks[head] - best);   // the sink: once, with no value
        const float inverse = 1.0f / total;
#pragma unroll
        for (int i2 = 0; i2 < DT; i2++) {
            f32x4 most = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int w = 0; w < WAVES; w++) {
                const f32x4 here = *reinterpret_cast<const f32x4*>(&largest_lds[w][i2 * 32 + 8 * wave + 4 * half]);
#pragma unroll
                for (int e = 0; e < 4; e++) most[e] = fmaxf(most[e], here[e]);
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float sum = 0.0f;
#pragma unroll
                for (int w = 0; w < WAVES; w++) sum += weight[w] * reinterpret_cast<const float*>(lds + w * WAVE_BYTES)[(i2 * 16 + 4 * wave + e) * WAVE + lane];
                odd |= (most[e] > 0.0f) & (fabsf(sum) < fmaxf(most[e], 1.0f) * 0x1p-90f);
                o[i2][e] = sum * inverse;
                odd |= !(fabsf(o[i2][e]) < INFINITY);
            }
        }
    }
    const unsigned odd_rows = rows_of(odd & (own_query < q_len)) & ~none_rows;
    if (odd_rows != 0 && lane == 0) atomicOr(&again, odd_rows);
    __syncthreads();
    unsigned rows = __builtin_amdgcn_readfirstlane(again);
    if (own_query < q_len && !(rows >> lane32 & 1)) {   // (not the others: they are read once more below, and the output may lie where they do)
        float* const out_row = out + (size_t)(q_first + own_query) * out_stride + head * HD + 8 * wave + 4 * half;
#pragma unroll
        for (int i2 = 0; i2 < DT; i2++) *reinterpret_cast<f32x4*>(out_row + i2 * 32) = o[i2];
    }
    float* my_q = reinterpret_cast<float*>(lds + wave * WAVE_BYTES);
    for (int n = 0; rows != 0; rows &= rows - 1, n++) {   // by the waves in turn
        if (n % WAVES != wave) continue;
        const int row = tile_q0 + __builtin_ctz(rows);
        general_row<float>(q + (size_t)(q_first + row) * q_stride + head * HD, k_pages, v_pages, out, (size_t)(q_first + row) * out_stride + head * HD, table, context + row, kv_head,
                           head, n_kv_heads, HD, 1 << page_shift, given_window, scale, options, my_q);
    }
}

template <int HD, int FORM>
__global__ __launch_bounds__(64 * WAVES, 2) void attention_prefill_pieces_kernel(
    const float* __restrict__ q, int q_stride, const float* __restrict__ k_pages, const float* __restrict__ v_pages, float* __restrict__ out, int out_stride,
    const int* __restrict__ q_starts, const int* __restrict__ context_lens, const int* __restrict__ block_tables, int max_blocks, int n_requests, int n_heads,
    int n_kv_heads, int page_shift, int given_window, float scale, ScoreOptions options) {
    pieces_block<HD, FORM>(blockIdx.x, q, q_stride, k_pages, v_pages, out, out_stride, q_starts, context_lens, block_tables, max_blocks, n_requests, n_heads, n_kv_heads, page_shift,
                           given_window, scale, options);
}

template <int HD, int FORM>
void launch_with(const float* q, int q_stride, const float* k_pages, const float* v_pages, float* out, int out_stride, const int* q_starts, const int* context_lens,
                 const int* block_tables, int max_blocks, int n_requests, int rows, int max_q_len, int n_heads, int n_kv_heads, int page_shift, int window, float scale,
                 ScoreOptions options, hipStream_t stream) {
    constexpr int LDS_BYTES = WAVES * wave_bytes<HD>();
    static bool raised = false;  // per instantiation: the limit on dynamic LDS is a property of the kernel
    if (!raised && LDS_BYTES > 60 * 1024)  // (if this fails the launch below fails too, and the entry point reports that)
        raised = hipFuncSetAttribute((const void*)attention_prefill_pieces_kernel<HD, FORM>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES) == hipSuccess;
    mllm_count_kernel(MLLM_K_ATTENTION_PREFILL_STREAM);
    attention_prefill_pieces_kernel<HD, FORM><<<n_heads * most_tiles(QUERIES, n_requests, rows, max_q_len), 64 * WAVES, LDS_BYTES, stream>>>(
        q, q_stride, k_pages, v_pages, out, out_stride, q_starts, context_lens, block_tables, max_blocks, n_requests, n_heads, n_kv_heads, page_shift, window, scale, options);
}

template <int HD>
void launch(const float* q, int q_stride, const float* k_pages, const float* v_pages, float* out, int out_stride, const int* q_starts, const int* context_lens,
            const int* block_tables, int max_blocks, int n_requests, int rows, int max_q_len, int n_heads, int n_kv_heads, int page_shift, int window, float scale,
            ScoreOptions options, hipStream_t stream) {
#define MLLM_PIECES_WITH(FORM)                                                                                                                                                \
    launch_with<HD, FORM>(q, q_stride, k_pages, v_pages, out, out_stride, q_starts, context_lens, block_tables, max_blocks, n_requests, rows, max_q_len, n_heads, n_kv_heads, \
                          page_shift, window, scale, options, stream)
    if (options.keep > 0) MLLM_PIECES_WITH(KEPT);
    else if (options.softcap > 0.0f) MLLM_PIECES_WITH(CAPPED);
    else if (window > 0 || options.chunk > 0) MLLM_PIECES_WITH(MASKED);
    else MLLM_PIECES_WITH(CAUSAL);
#undef MLLM_PIECES_WITH
}

}  // namespace prefill_pieces
