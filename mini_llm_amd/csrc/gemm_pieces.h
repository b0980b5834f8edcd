// The 32-bit product for many rows on the bfloat16 matrix cores. Included by gemm.hip.
//
// A 32-bit number (of 2^-110 or more; smaller ones and infinities: at the kernel's end) is the sum of three bfloat16 ones, each what the one before leaves, rounded to the nearest, and a product of two such numbers is the sum of
// nine products of pieces, each exact in 32-bit (the method: Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For
// Higher-Precision Computations", 2019). The three left out are at most 2^-24 of the product and lie on either side of it. (Pieces cut off instead
// of rounded leave out up to 2^-21, always on the product's own side: over 3,072 positive numbers the sums came out 6.5e-6 too small, 7e-8 with rounding.)
// The matrix instruction for bfloat16 does in 32 cycles eight times the work that the 32-bit one does in 64, so six of them are 2.7 times faster. The five
// smaller products have a running sum of their own, added to the large one at the end: in one sum they are lost to its rounding once it is long, and it is
// rounded six times for sixteen numbers of K instead of once (the 32-bit instruction: eight times). Measured against 64-bit sums over rows of 768 and 3,072
// normally distributed numbers: 1.6e-7 and 3.4e-7 of the result's norm, in one sum 4.2e-7 and 8.6e-7, with the 32-bit instruction 5.0e-7 and 9.9e-7; over
// rows of which half are zero, as behind a clamp, 1.2e-7 and 2.7e-7, 4.0e-7 and 8.2e-7, 3.5e-7 and 7.1e-7. It is 64 registers that the 128 x 128 tile
// has left (238 in all, none spilled), and little time: with the loop before the present one 2,048 x 3,072 x 768 60.6 us, 63.2 in one sum, on another machine 64.4 and 63.3.
//
// W's pieces are laid out once, when the matrix is packed (common.h: packed_pieces): the chunks of the packed layout for bfloat16, the three of a k-step
// behind each other. A's rows come as they are, and a wave splits the fragments it has read.
// A block of four waves owns BM x BN outputs and walks K in tiles of 32, two steps of 16: rows of A and chunks of W go from memory straight into LDS
// (global_load_lds_dwordx4), one tile ahead of the products, in two stages, which leave room for two blocks a compute unit (a third stage and one block: 2,048 x 2,304 x 768
// with 128 x 128 58 -> 69 us). What bounds it: the matrix cores, and beside them the chip's power. A SIMD runs a wave's vector instructions under its own matrix instructions
// only where they stand between them: a tile's 48 products behind the splitting of their rows, step by step, take 2,101 cycles, with the splitting of the next step's rows between
// them 1,609, and of two waves a SIMD that split first and multiply then each 1,860. So a step's products carry the splitting of the next step's rows, its fragment reads, and one by one
// the loads of the tile after the next (a compute unit takes a load of 1 KiB every 16 cycles, and a wave that asks for all at once waits).
// With the loads at a tile's start and the splitting in front of its products -> now, alone in a loop, on one machine in turn, us: 2,048 x 2,304 x 768 53.5 -> 44.4 (64 x 64, 128 x 96),
// 2,048 x 3,072 x 768 58.3 -> 51.5 (128 x 64, 128 x 96), 2,670 x 768 x 3,072 in two 79.2 -> 67.6; on one that gives less power 69.8 -> 58.3, 71.1 -> 60.2, 90.1 -> 81.4 and
// 8,192 x 3,072 x 768 217 -> 211; in a prompt step of 2,048 rows the first two take 52 and 63 us.
// Fragment reads are inline assembly with waits of their own: through the compiler each would wait for the loads into LDS that are under way.
#pragma once

#include "number_pieces.h"

namespace pieces {

constexpr int BK = 32;   // numbers of K in a tile

template <int BM, int BN>
constexpr int stage_bytes() {
    return BM * BK * 4 + BN / 16 * 3 * 1024;
}

template <int OFFSET>
__device__ __forceinline__ void ask(i32x4& to, unsigned address) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(to) : "v"(address), "n"(OFFSET));
}
__device__ __forceinline__ void landed(i32x4& first) { asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(first)); }
__device__ __forceinline__ void this_too(i32x4& fragment) { asm volatile("" : "+v"(fragment)); }

// until at most LEFT of the wave's LDS reads, the newest, are under way
template <int LEFT>
__device__ __forceinline__ void landed_but(i32x4& first) { asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(first) : "n"(LEFT)); }
// until at most LEFT of its loads from memory are
template <int LEFT>
__device__ __forceinline__ void wait_but() {
    static_assert(LEFT < 64, "the loads in flight fit the counter");
    __builtin_amdgcn_s_waitcnt((LEFT & 0xF) | ((LEFT >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// The whole product (Group: stream::Whole) or one over rows grouped by expert (stream::ExpertTiles, a one-dimensional grid). W: packed, its pieces behind its
// `matrix_tiles` row tiles. gridDim.z blocks along K take k_per_block of it each (a multiple of 32) and leave partial products.
// W is the first operand of the matrix instruction, so that a lane holds four consecutive columns of a row; the results pass through LDS 32 rows at a time
// and leave in whole rows of a wave's columns. (Stored from where the sums lie, number by number, a block of 128 x 128 took 12 us behind its loop.)
template <int BM, int BN, int WAVES_M, int WAVES_N, typename Group>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N, 2) void gemm_pieces_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                                                                               const float* __restrict__ residual, float* __restrict__ out, int M, int N, int K, int matrix_tiles,
                                                                               int epilogue, CacheScatter scatter, int k_per_block, Group group) {
    constexpr int WAVES = WAVES_M * WAVES_N, STAGE = stage_bytes<BM, BN>(), A_BYTES = BM * BK * 4;
    constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N, TM = WM / 32, TN = WN / 32;
    constexpr int A_LOADS = BM / 8 / WAVES, W_CHUNKS = BN / 16 * 3, W_LOADS = (W_CHUNKS + WAVES - 1) / WAVES;
    static_assert(TM >= 1 && TN >= 1 && BM / 8 % WAVES == 0, "every wave asks for as much");   // (of W's chunks the last may be asked for twice)
    extern __shared__ __attribute__((aligned(16))) unsigned char piece_lds[];
    const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int wave_m = wave / WAVES_N, wave_n = wave % WAVES_N, half = lane / 32, lane32 = lane % 32;
    const int row_tiles = ceil_div(N, 16), k_steps = ceil_div(K, BK);
    int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN, m_end = M, first_tile = 0;
    if constexpr (Group::GROUPED) {
        stream::GroupTile tile;
        if (!stream::group_tile(group, N, BN, tile)) return;  // (the whole block leaves)
        m0 = tile.m0, m_end = tile.m_end, n0 = tile.n0;
        first_tile = tile.expert * row_tiles;
    }
    const int k_begin = blockIdx.z * k_per_block, k_end = min(K, k_begin + k_per_block);
    out += (size_t)blockIdx.z * M * N;
    const unsigned char* w_pieces = reinterpret_cast<const unsigned char*>(W) + packed_pieces_at(matrix_tiles, packed_k_steps<float>(K));
    auto a_row = [&](int r) {   // of the block's tile; beyond the last: that row again, never stored
        const int row = min(m0 + r, m_end - 1);
        if constexpr (Group::GROUPED) return group.a_row ? group.a_row[row] : row;
        else return row;
    };

    // what this lane asks for: eight lanes the 128 bytes a row of A has in a tile, its 16-byte pieces turned by the row (so that the fragment reads of
    // sixteen rows, two of which fill all banks once, meet different ones); a chunk of W as it lies
    unsigned a_from[A_LOADS], w_from[W_LOADS];
#pragma unroll
    for (int l = 0; l < A_LOADS; l++) {
        const int row = (wave + l * WAVES) * 8 + lane / 8;
        a_from[l] = (unsigned)a_row(row) * (unsigned)K * 4u + (unsigned)(((lane % 8) ^ (row / 2 % 8)) * 16);
    }
#pragma unroll
    for (int l = 0; l < W_LOADS; l++) {
        const int chunk = min(wave + l * WAVES, W_CHUNKS - 1), row_tile = first_tile + min(n0 / 16 + chunk / 3, row_tiles - 1);
        w_from[l] = ((unsigned)row_tile * (unsigned)k_steps * 3u + (unsigned)(chunk % 3)) * 1024u + lane * 16u;
    }
    const int tiles = (k_end - k_begin + BK - 1) / BK;
    const unsigned char *a_tile = reinterpret_cast<const unsigned char*>(A + k_begin), *w_tile = w_pieces + (size_t)(k_begin / BK) * 3072;
    constexpr int LOADS = A_LOADS + W_LOADS;
    // load `l` of the tile a_tile and w_tile stand at, into the stage that begins at `stage`
    auto issue_load = [&](int l, unsigned stage) {
        if (l < A_LOADS)
            __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(a_tile + a_from[l]),
                                             (void __attribute__((address_space(3)))*)(piece_lds + stage + (wave + l * WAVES) * 1024), 16, 0, 0);
        else
            __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(w_tile + w_from[l - A_LOADS]),
                                             (void __attribute__((address_space(3)))*)(piece_lds + stage + A_BYTES + min(wave + (l - A_LOADS) * WAVES, W_CHUNKS - 1) * 1024), 16, 0, 0);
    };
    auto next_tile = [&] {
        a_tile += BK * 4;
        w_tile += 3072;
    };

    f32x16 acc[TN][TM], low[TN][TM];   // the sums of the high pieces' products, and of the five others
    const unsigned base = (unsigned)(size_t)(const __attribute__((address_space(3))) unsigned char*)piece_lds;
    unsigned a_at[2][2];   // [step of 16][piece]
#pragma unroll
    for (int kk = 0; kk < 2; kk++)
#pragma unroll
        for (int q = 0; q < 2; q++) a_at[kk][q] = base + (wave_m * WM + lane32) * 128 + (((kk * 4 + half * 2 + q) ^ (lane32 / 2 % 8)) * 16);
    const unsigned w_at = base + A_BYTES + (wave_n * TN * 2 + lane32 / 16) * 3072 + half * 256 + (lane % 16) * 16;

    // of the wave's columns: whether one has a row of W that is tiny throughout, and the largest magnitude in W
    int w_tiny = 0, w_largest = 0;
#pragma unroll
    for (int t = 0; t < WN / 16; t++) {
        const TileRows rows = reinterpret_cast<const TileRows*>(w_pieces + packed_pieces_bytes(matrix_tiles, K))[first_tile + min((n0 + wave_n * WN) / 16 + t, row_tiles - 1)];
        w_tiny |= rows.tiny, w_largest = max(w_largest, rows.largest);
    }
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[j][i][v] = low[j][i][v] = 0.0f;
    if (tiles > 0) {
        i32x4 raw[TM][2], w_high[2][TN], w_low[2][TN];   // the next step's rows; W's first pieces of this step and the next; its second and third pieces
        bf16x8 a[2][TM][3];                              // the pieces of this step's rows, and of the next one's
        using std::integral_constant;
        // reads of a step (kk: the first or second sixteen numbers of K of the tile in the stage)
        auto ask_rows = [&](auto step, unsigned stage) {
            constexpr int kk = decltype(step)::value;
            stream::static_for<TM>([&](auto i) {
                ask<i * 32 * 128>(raw[i][0], a_at[kk][0] + stage);
                ask<i * 32 * 128>(raw[i][1], a_at[kk][1] + stage);
            });
        };
        auto ask_columns = [&](auto step, auto piece, unsigned stage) {
            constexpr int kk = decltype(step)::value, p = decltype(piece)::value;
            stream::static_for<TN>([&](auto j) { ask<j * 2 * 3072 + p * 1024 + kk * 512>(p == 0 ? w_high[kk][j] : w_low[p - 1][j], w_at + stage); });
        };
        auto rows_here = [&] {
#pragma unroll
            for (int i = 0; i < TM; i++) this_too(raw[i][0]), this_too(raw[i][1]);
        };
        auto columns_here = [&](i32x4 (&columns)[TN]) {
#pragma unroll
            for (int j = 0; j < TN; j++) this_too(columns[j]);
        };
        constexpr integral_constant<int, 0> zero;
        constexpr integral_constant<int, 1> one;
        constexpr integral_constant<int, 2> two;

        // The products of two pieces in a step: those of W's third and second piece first, whose registers are then free for the next step's.
        constexpr int OF_A[6] = {0, 1, 0, 2, 1, 0}, OF_W[6] = {2, 1, 1, 0, 0, 0}, EACH = TM * TN, PAIRS = TM * 4;
        auto products = [&](auto step, auto from, auto count, auto&& behind) {   // `count` of them from the one numbered `from`; behind(n): what goes behind product n
            constexpr int kk = decltype(step)::value;
            stream::static_for<decltype(count)::value>([&](auto n) {
                constexpr int at = decltype(from)::value + decltype(n)::value, c = at / EACH, i = at % EACH / TN, j = at % TN, p = OF_W[c];
                const i32x4& columns = p == 0 ? w_high[kk][j] : w_low[p == 0 ? 0 : p - 1][j];
                f32x16& to = c < 5 ? low[j][i] : acc[j][i];
                to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8*>(&columns), a[kk][i][OF_A[c]], to, 0, 0, 0);
                behind(integral_constant<int, at>{});
                __builtin_amdgcn_sched_barrier(0);
            });
        };
        // 64 x 64: few products to put a tile's loads between, and few loads: they go out together, and the blocks that are alone on a unit wait less for them
        constexpr bool AT_ONCE = EACH == 1;
        // One step: its products, and under them the reads of the next step, the splitting of its rows and, in a tile's second step, the loads of a tile further on.
        // LEFT: how many tiles of K are behind this one, 2 for more. Behind the last tile's second step there is no next one: in a block with few tiles of K what
        // it would read and split shows (66 x 1,536 x 768 in five 6.7 -> 6.45 us, 520 x 768 x 768 in six 10.5 -> 10.25).
        auto step = [&](auto which, auto left, unsigned here, unsigned behind) {   // where this tile's stage begins, and the next one's
            constexpr int kk = decltype(which)::value, LEFT = decltype(left)::value;
            constexpr bool loads = kk == 1 && LEFT == 2, last = kk == 1 && LEFT == 0;
            constexpr integral_constant<int, 1 - kk> next;
            const unsigned stage = kk == 0 ? here : behind;   // of the next step
            landed(w_high[kk][0]);
            columns_here(w_high[kk]), columns_here(w_low[0]), columns_here(w_low[1]);
            if constexpr (last) {
                products(which, zero, integral_constant<int, 6 * EACH>{}, [](auto) {});
                return;
            }
            if constexpr (kk == 1) {
                // every read of this tile has landed, and this wave's loads of the next one: behind the barrier everybody's have, and this tile's stage is free
                wait_but<0>();
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
            }
            ask_rows(next, stage);
            ask_columns(next, zero, stage);
            if constexpr (loads && AT_ONCE) stream::static_for<LOADS>([&](auto l) { issue_load(decltype(l)::value, here); });
            __builtin_amdgcn_sched_barrier(0);
            products(which, integral_constant<int, 0>{}, integral_constant<int, EACH>{}, [](auto) {});
            ask_columns(next, two, stage);
            landed_but<2 * TN>(raw[0][0]);
            rows_here();
            __builtin_amdgcn_sched_barrier(0);
            auto under = [&](auto n) {   // the share of product n of the 5 EACH that are left
                constexpr int at = decltype(n)::value - EACH, OF = 5 * EACH;
                stream::static_for<(at + 1) * PAIRS / OF - at * PAIRS / OF>([&](auto p) {
                    constexpr int pair = at * PAIRS / OF + decltype(p)::value, i = pair / 4, e = pair % 4;
                    split_pair(raw[i], e, a[1 - kk][i]);
                });
                if constexpr (loads && !AT_ONCE)
                    stream::static_for<(at + 1) * LOADS / OF - at * LOADS / OF>([&](auto l) { issue_load(at * LOADS / OF + decltype(l)::value, here); });
            };
            products(which, integral_constant<int, EACH>{}, integral_constant<int, 2 * EACH>{}, under);
            ask_columns(next, one, stage);
            __builtin_amdgcn_sched_barrier(0);
            products(which, integral_constant<int, 3 * EACH>{}, integral_constant<int, 3 * EACH>{}, under);
            if constexpr (loads) next_tile();
        };
        auto issue = [&](unsigned stage) {
#pragma unroll
            for (int l = 0; l < LOADS; l++) issue_load(l, stage);
            next_tile();
        };
        issue(0);
        wait_but<0>();
        stream::wait_lgkmcnt<0>();   // (kernel arguments: a scalar load under way would count among the reads below)
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        ask_rows(zero, 0);
        ask_columns(zero, zero, 0);
        ask_columns(zero, one, 0);
        ask_columns(zero, two, 0);
        if (tiles > 1) issue(STAGE);
        landed_but<3 * TN>(raw[0][0]);
        rows_here();
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) split_pair(raw[i], e, a[0][i]);
        __builtin_amdgcn_sched_barrier(0);
        unsigned here = 0;
        auto tile = [&](auto left) {
            step(zero, left, here, STAGE - here);
            step(one, left, here, STAGE - here);
            here = STAGE - here;
        };
        for (int t = 0; t + 2 < tiles; t++) tile(two);
        if (tiles > 1) tile(one);
        tile(zero);
    }

#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
        for (int i = 0; i < TM; i++) acc[j][i] += low[j][i];
    const int row0 = m0 + wave_m * WM, col0 = n0 + wave_n * WN;
    __syncthreads();   // the slabs below lie where the tiles did

    // An infinity has no pieces (its middle is no number), so every sum it belongs to comes out as no number, whatever it should be. And below 2^-110 the
    // last piece of a number falls under the smallest bfloat16 number: what is lost, up to 2^-134, counts where a row has nothing larger. The rows of this
    // wave with a sum that is not finite, and those that are tiny throughout (bit r: row r of the WM), are left out of what is stored below and taken again
    // in 32-bit at the end. What a row holds that is no number itself makes all its sums none, as it should: such a row stays as it is. (Rows that nobody
    // reads may hold anything, and those with an infinity become that behind the next norm.)
    // Whether a row is tiny is not asked while it is split (four instructions for eight numbers: 1.5 % of a pass of ragged prompts) but read again where its
    // sums are no larger than a tiny row's could be.
    static_assert(TM <= 2, "a bit a row");
    const float faint_sum = ldexpf(__builtin_bit_cast(float, w_largest), -94) * (float)(k_end - k_begin);   // (twice as much, for the roundings)
    unsigned long long bad = 0, faint = 0;
#pragma unroll
    for (int i = 0; i < TM; i++) {
        float largest = 0.0f;   // no number if one of them is none (the instruction keeps that: one for two sums)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) largest = __builtin_elementwise_maximum(largest, fabsf(acc[j][i][v]));
        const unsigned long long lanes = __ballot(!(largest < INFINITY));
        bad |= (unsigned long long)((unsigned)lanes | (unsigned)(lanes >> 32)) << (32 * i);
        largest = fmaxf(largest, __shfl_xor(largest, 32, WAVE));
        faint |= (unsigned long long)(unsigned)__ballot(largest > 0.0f && largest <= faint_sum) << (32 * i);
    }
    const int row16 = lane % 16, quad = lane / 16, rows_here = m_end - row0;
    const unsigned long long real = rows_here >= WM ? ~0ull >> (64 - WM) : rows_here > 0 ? (1ull << rows_here) - 1 : 0;   // (beyond the last row: that row again)
    if (w_tiny != 0) bad = ~0ull;
    bad &= real, faint &= real;
    if ((bad | faint) != 0) {
#pragma unroll 1
        for (int g = 0; g < WM / 16; g++) {
            if (((bad | faint) >> (16 * g) & 0xffff) == 0) continue;
            const float* x = A + (size_t)a_row(wave_m * WM + g * 16 + row16) * K + 4 * quad;
            bool none = false;
            uint32_t bits = 0;
            for (int k = k_begin; k < k_end; k += 16) {
                const Vec16 piece = *reinterpret_cast<const Vec16*>(x + k);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    none |= (piece.w[e] & 0x7fffffffu) > 0x7f800000u;
                    bits |= piece.w[e];
                }
            }
            bits |= (uint32_t)__shfl_xor((int)bits, 16, WAVE);
            bits |= (uint32_t)__shfl_xor((int)bits, 32, WAVE);
            const unsigned long long lanes = __ballot(none), tiny_rows = __ballot(tiny(bits)) & 0xffff;
            bad &= ~(((lanes | lanes >> 16 | lanes >> 32 | lanes >> 48) & 0xffff) << (16 * g));
            bad |= faint & tiny_rows << (16 * g);
        }
    }

    // 32 rows of the wave's columns at a time through LDS of its own, 16 bytes of padding a row. GATED: 32 gate and 32 up columns become 32 units.
    constexpr int OUT_COLS = Group::GATED ? WN / 2 : WN, SLAB_ROW = OUT_COLS + 4, LANES_A_ROW = OUT_COLS / 4, ROWS = WAVE / LANES_A_ROW;
    static_assert(!Group::GATED || TN % 2 == 0, "a wave holds gate and up columns of the same units");
    static_assert(WAVES * 32 * SLAB_ROW * 4 <= 2 * STAGE, "the slabs fit the stages");
    float* const slab = reinterpret_cast<float*>(piece_lds) + wave * 32 * SLAB_ROW;
    const int out_cols = Group::GATED ? N / 2 : N, out_col = (Group::GATED ? col0 / 2 : col0) + (lane % LANES_A_ROW) * 4;
    const int width = scatter.enabled ? scatter.q_width : out_cols;
    // where four columns of a q/k/v projection go: they lie in one head (the host sees to it)
    struct Place {
        float* pages;   // null: the output
        int kv_head, d;
    };
    auto place_of = [&](int col) {
        Place place = {nullptr, 0, 0};
        if (!Group::GROUPED && scatter.enabled && col >= scatter.q_width && col < N) {
            int c = col - scatter.q_width;
            place.pages = (float*)(c < scatter.kv_width ? scatter.k_pages : scatter.v_pages);
            if (c >= scatter.kv_width) c -= scatter.kv_width;
            place.kv_head = c / scatter.head_size, place.d = c % scatter.head_size;
        }
        return place;
    };
    auto put = [&](int row, int col, const Place& place, f32x4 value) {
        if (!Group::GROUPED && place.pages) {
            const int slot = scatter.slots[row];
            if (slot < 0) return;
            const int page = slot >> scatter.page_shift, offset = slot & ((1 << scatter.page_shift) - 1);
            *reinterpret_cast<f32x4*>(place.pages + ((((size_t)page * scatter.n_kv_heads + place.kv_head) << scatter.page_shift) + offset) * scatter.head_size + place.d) = value;
            return;
        }
        int to = row;
        if constexpr (Group::GROUPED && !Group::GATED) to = group.out_row ? group.out_row[row] : row;
        const size_t at = (size_t)to * width + col;
        if (!Group::GROUPED && residual) value = *reinterpret_cast<const f32x4*>(residual + at) + value;
        *reinterpret_cast<f32x4*>(out + at) = value;
    };
    const Place place = place_of(out_col);   // a lane's columns are the same in every row
    auto leave = [&](auto kind) {
        constexpr int KIND = decltype(kind)::value;
        constexpr bool UNITS = KIND == MLLM_EPI_GATED_SILU;   // two groups of eight columns become eight
#pragma unroll
        for (int i = 0; i < TM; i++) {
            float in_weight = 1.0f, out_weight = 1.0f;
            if constexpr (Group::GATED) {
                const float weight = group.weight[min(row0 + i * 32 + lane32, m_end - 1)];
                in_weight = group.weigh_input ? weight : 1.0f, out_weight = group.weigh_input ? 1.0f : weight;
            }
#pragma unroll
            for (int j = 0; j < TN; j += Group::GATED ? 2 : 1)
#pragma unroll
                for (int g = 0; g < 4; g += UNITS ? 2 : 1) {
                    f32x4 value;
                    if constexpr (UNITS) {
#pragma unroll
                        for (int e = 0; e < 4; e++) value[e] = gated_silu(acc[j][i][4 * g + e], acc[j][i][4 * g + 4 + e]);
                        *reinterpret_cast<f32x4*>(slab + lane32 * SLAB_ROW + j * 16 + 4 * g + 4 * half) = value;
                        continue;
                    }
                    if constexpr (Group::GATED) {
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            value[e] = gated(acc[j][i][4 * g + e] * in_weight, acc[j + 1][i][4 * g + e] * in_weight, group.unit) * out_weight;
                    } else {
                        const int col = col0 + j * 32 + 8 * g + 4 * half;
                        f32x4 b = {0.0f, 0.0f, 0.0f, 0.0f};
                        if (!Group::GROUPED && bias && col < N) b = *reinterpret_cast<const f32x4*>(bias + col);
#pragma unroll
                        for (int e = 0; e < 4; e++) value[e] = apply_activation<KIND>(acc[j][i][4 * g + e] + b[e]);
                    }
                    *reinterpret_cast<f32x4*>(slab + lane32 * SLAB_ROW + (Group::GATED ? j / 2 : j) * 32 + 8 * g + 4 * half) = value;
                }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
            for (int r = 0; r < 32 / ROWS; r++) {
                const int in_slab = r * ROWS + min(lane / LANES_A_ROW, ROWS - 1), row = row0 + i * 32 + in_slab;
                f32x4 value = *reinterpret_cast<const f32x4*>(slab + in_slab * SLAB_ROW + (lane % LANES_A_ROW) * 4);
                if (lane >= ROWS * LANES_A_ROW || row >= m_end || out_col >= out_cols || ((unsigned)(bad >> (i * 32)) >> in_slab & 1)) continue;
                if constexpr (UNITS) {
                    const int unit = col0 / 2 + (lane % LANES_A_ROW) * 4;
                    if (lane % LANES_A_ROW < LANES_A_ROW / 2 && unit < N / 2) *reinterpret_cast<f32x4*>(out + (size_t)row * (N / 2) + unit) = value;
                    continue;
                }
                put(row, out_col, place, value);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
    };
    using std::integral_constant;
    if constexpr (Group::UNITS) leave(integral_constant<int, MLLM_EPI_GATED_SILU>{});
    else if (Group::GROUPED || epilogue == MLLM_EPI_NONE) leave(integral_constant<int, MLLM_EPI_NONE>{});
    else if (epilogue == MLLM_EPI_GELU_TANH) leave(integral_constant<int, MLLM_EPI_GELU_TANH>{});
    else if (epilogue == MLLM_EPI_GELU_ERF) leave(integral_constant<int, MLLM_EPI_GELU_ERF>{});
    else leave(integral_constant<int, MLLM_EPI_SQUARED_RELU>{});

    // the rows left out, in groups of sixteen that hold one, with the 32-bit instruction and operands straight from memory
    constexpr int TILES = WN / 16;
#pragma unroll 1
    for (int g = 0; g < WM / 16; g++) {
        const unsigned rows = (unsigned)(bad >> (16 * g)) & 0xffff;
        if (rows == 0) continue;
        const float* x = A + (size_t)a_row(wave_m * WM + g * 16 + row16) * K + 4 * quad;
        f32x4 sum[TILES];
#pragma unroll
        for (int t = 0; t < TILES; t++) sum[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
        for (int k = k_begin; k < k_end; k += 16) {
            const f32x4 b = *reinterpret_cast<const f32x4*>(x + k);
            f32x4 a[TILES];
#pragma unroll
            for (int t = 0; t < TILES; t++)
                a[t] = *reinterpret_cast<const f32x4*>(W + packed_offset<float>(first_tile + min(col0 / 16 + t, row_tiles - 1), k / 16, packed_k_steps<float>(K), lane));
#pragma unroll
            for (int t = 0; t < TILES; t++)
#pragma unroll
                for (int e = 0; e < 4; e++) sum[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t][e], b[e], sum[t], 0, 0, 0);
        }
        // sum[t][e] of a lane: row lane % 16, column 16 t + 4 (lane / 16) + e of the wave's
        const int row = row0 + g * 16 + row16;
        if (row >= m_end || !(rows >> row16 & 1)) continue;
        if constexpr (Group::GATED) {
            const float weight = group.weight[row], in_weight = group.weigh_input ? weight : 1.0f, out_weight = group.weigh_input ? 1.0f : weight;
#pragma unroll
            for (int t = 0; t < TILES / 2; t++) {   // 32 gate columns, two tiles of them, and the 32 up columns behind them
                const int col = col0 / 2 + t * 16 + 4 * quad, gate = t / 2 * 4 + t % 2;
                if (col >= out_cols) continue;
                f32x4 value;
#pragma unroll
                for (int e = 0; e < 4; e++) value[e] = gated(sum[gate][e] * in_weight, sum[gate + 2][e] * in_weight, group.unit) * out_weight;
                put(row, col, Place{nullptr, 0, 0}, value);
            }
        } else {
#pragma unroll
            for (int t = 0; t < TILES; t++) {
                const int col = col0 + t * 16 + 4 * quad;
                if constexpr (Group::UNITS) {   // a tile's gate columns in the first 32 lanes, its up columns in the others (of the same rows)
                    f32x4 unit;
#pragma unroll
                    for (int e = 0; e < 4; e++) unit[e] = gated_silu(sum[t][e], __shfl_xor(sum[t][e], 32, WAVE));
                    if (quad < 2 && col < out_cols) *reinterpret_cast<f32x4*>(out + (size_t)row * (N / 2) + col0 / 2 + t * 8 + 4 * quad) = unit;
                    continue;
                }
                if (col >= out_cols) continue;
                f32x4 value = sum[t];
                if (!Group::GROUPED && bias) value += *reinterpret_cast<const f32x4*>(bias + col);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if (!Group::GROUPED && epilogue == MLLM_EPI_GELU_TANH) value[e] = gelu_tanh(value[e]);
                    else if (!Group::GROUPED && epilogue == MLLM_EPI_GELU_ERF) value[e] = gelu_erf(value[e]);
                    else if (!Group::GROUPED && epilogue == MLLM_EPI_SQUARED_RELU) value[e] = squared_relu(value[e]);
                }
                put(row, col, place_of(col), value);
            }
        }
    }
}

// Whether a product takes this kernel: a W that was packed with its pieces (which it is not unless the sizes of W asked for here hold), more rows than the
// kernel for few rows takes, whole tiles of K, whole pieces of 16 bytes in every row and pointer, operands whose bytes a 32-bit offset reaches, and in a
// q/k/v projection four columns never in two heads.
inline bool takes_sizes(int M, int N, int K, int matrix_tiles, int packed) {
    return packed == PACKED_WITH_PIECES && M > 64 && K % BK == 0 && N % 4 == 0 && (long long)M * K * 4 < (1LL << 32) && packed_pieces_bytes(matrix_tiles, K) < (1LL << 32);
}

inline bool takes(const void* a, const void* bias, const void* residual, const void* out, int M, int N, int K, int matrix_tiles, int packed, const CacheScatter& scatter) {
    if (!takes_sizes(M, N, K, matrix_tiles, packed)) return false;
    if (((size_t)a | (size_t)bias | (size_t)residual | (size_t)out) % 16 != 0) return false;
    return !scatter.enabled || (scatter.q_width % 4 == 0 && scatter.kv_width % 4 == 0 && scatter.head_size % 4 == 0 && (((size_t)scatter.k_pages | (size_t)scatter.v_pages) % 16) == 0);
}

template <int BM, int BN, int WAVES_M, int WAVES_N, typename Group>
void launch(const float* a, const float* w, const float* bias, const float* residual, float* o, int M, int N, int K, int matrix_tiles, int epilogue, hipStream_t stream,
            const CacheScatter& scatter, int k_blocks, dim3 grid, const Group& group) {
    constexpr int LDS_BYTES = 2 * stage_bytes<BM, BN>();
    static bool raised = false;  // per instantiation: the limit on dynamic LDS is a property of the kernel
    if (!raised && LDS_BYTES > 60 * 1024)  // (if this fails the launch below fails too, and the entry point reports that)
        raised = hipFuncSetAttribute((const void*)gemm_pieces_kernel<BM, BN, WAVES_M, WAVES_N, Group>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES) == hipSuccess;
    const int k_per_block = ceil_div(ceil_div(K, k_blocks), BK) * BK;
    mllm_count_kernel(MLLM_K_GEMM_TILED);
    gemm_pieces_kernel<BM, BN, WAVES_M, WAVES_N, Group><<<grid, 64 * WAVES_M * WAVES_N, LDS_BYTES, stream>>>(a, w, bias, residual, o, M, N, K, matrix_tiles, epilogue, scatter,
                                                                                                          k_per_block, group);
}

template <int BM, int BN, int WAVES_M, int WAVES_N, typename Group>
void launch_whole(const float* a, const float* w, const float* bias, const float* residual, float* o, int M, int N, int K, int epilogue, hipStream_t stream, const CacheScatter& scatter,
                  int k_blocks) {
    launch<BM, BN, WAVES_M, WAVES_N>(a, w, bias, residual, o, M, N, K, ceil_div(N, 16), epilogue, stream, scatter, k_blocks, dim3(ceil_div(N, BN), ceil_div(M, BM), k_blocks), Group{});
}

// The tiles, and what they cost in microseconds: what lies in front of and behind a block's loop, and a tile of K for each block of a compute unit, alone there or not, and
// more the nearer a round of blocks is to all 256 units (they share the chip's power: products of numbers that are all zero take three quarters of the time).
// Fitted to 900 products of 66 to 6,000 rows, 512 to 4,096 columns, K of 768 to 4,096, whole and cut. A compute unit brings most out of 128 x 128; 128 x 96
// where its blocks are two rounds and 128 x 128's more than one; narrow outputs and few rows fill the chip with smaller ones.
// 128 x 128 / 128 x 64 / 64 x 64 / 128 x 96, us (more sizes: profiles/pieces_tiles_f32.md): 2,048 x 2,304 x 768 53.7 / 49.0 / 49.9 / 44.4, 2,670 x 768 x 3,072 in two 67.6 / 67.6 /
// 79.9 / 82.4, 2,048 x 768 x 3,072 in two 58.6 / 59.0 / 61.6 / 52.9, 130 x 2,304 x 768 28.6 / 18.5 / 14.9 / 22.8.
struct Choice {
    int bm, bn;
    float start, alone, tile, full;
};
constexpr int CHOICES_COUNT = 4;
constexpr Choice CHOICES[CHOICES_COUNT] = {{128, 128, 7.5f, 0.07f, 0.83f, 0.30f}, {128, 64, 5.6f, 0.065f, 0.44f, 0.20f}, {64, 64, 4.9f, 0.09f, 0.29f, 0.09f}, {128, 96, 7.25f, 0.025f, 0.64f, 0.25f}};

// Microseconds of a product cut into k_blocks along K with the best of the tiles (`best`): the rounds of blocks, the start and end of a block, and the sums
// that are written (6 TB/s). Measured at 440 sizes that it was not fitted to: whole products of as many columns as K or more 0.4 % behind the best of the four on average and 15 % at
// most, cut ones of as many at most 1.6 % behind the best tile and count, and 18 % at most (130 and 170 rows: the count is that of 256). Fitted to those instead it came to
// 0.3 and 1.0 % there, and at 559 further sizes was 0.3 % faster on average and up to a quarter slower (550 x 896 x 1,792 19.0 -> 23.8 us): left as it is.
inline float cost(int M, int N, int K, int k_blocks, int& best) {
    float best_cost = 0.0f;
    for (int c = 0; c < CHOICES_COUNT; c++) {
        const Choice& with = CHOICES[c];
        const long long blocks = (long long)ceil_div(M, with.bm) * ceil_div(N, with.bn) * k_blocks;
        const int rounds = (int)((blocks + 255) / 256), tiles = ceil_div(ceil_div(K, k_blocks), BK);
        const float a_tile = rounds * with.tile + (float)blocks / 256.0f * with.full + (rounds == 1 ? with.alone : 0.0f);
        const float us = with.start + tiles * a_tile + (float)M * N * k_blocks * (4.0f / 6e6f);
        if (c == 0 || us < best_cost) best = c, best_cost = us;
    }
    return best_cost;
}

template <typename Group = stream::Whole>
void dispatch(const float* a, const float* w, const float* bias, const float* residual, float* o, int M, int N, int K, int epilogue, hipStream_t stream,
                     const CacheScatter& scatter, int k_blocks) {
    int best = 0;
    cost(M, N, K, k_blocks, best);
    if (best == 0) launch_whole<128, 128, 2, 2, Group>(a, w, bias, residual, o, M, N, K, epilogue, stream, scatter, k_blocks);
    else if (best == 1) launch_whole<128, 64, 4, 1, Group>(a, w, bias, residual, o, M, N, K, epilogue, stream, scatter, k_blocks);
    else if (best == 2) launch_whole<64, 64, 2, 2, Group>(a, w, bias, residual, o, M, N, K, epilogue, stream, scatter, k_blocks);
    else launch_whole<128, 96, 4, 1, Group>(a, w, bias, residual, o, M, N, K, epilogue, stream, scatter, k_blocks);
}

// Into how many partial products a product with sums to be taken by whoever reads them is cut, `most` at most: they are read once more there.
inline int split_blocks(int M, int N, int K, int most) {
    int best = 1, tile = 0;
    float best_cost = 0.0f;
    for (int cuts = 1; cuts <= most && (cuts == 1 || K >= 4 * BK * cuts); cuts++) {
        const float us = cost(M, N, K, cuts, tile) + (float)M * N * cuts * (4.0f / 6e6f);
        if (cuts == 1 || us < best_cost) best = cuts, best_cost = us;
    }
    return best;
}

// The same over rows grouped by expert: a tile of the lists is 128 entries.
template <typename Group>
void launch_grouped(const float* a, const float* w, float* o, int entries, int max_tiles, int N, int K, int matrix_tiles, const Group& group, hipStream_t stream) {
    launch<128, 128, 2, 2>(a, w, nullptr, nullptr, o, entries, N, K, matrix_tiles, MLLM_EPI_NONE, stream, CacheScatter{}, 1, dim3(ceil_div(max_tiles * ceil_div(N, 128), 8) * 8), group);
}

}  // namespace pieces
