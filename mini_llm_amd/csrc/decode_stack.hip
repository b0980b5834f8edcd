// All layers of a pre-norm model for a few rows that bring one token each (decoding), in one kernel.
//
// What bounds a decode step of few rows is not what it reads but how often one part of the chip has to learn what another part has
// computed, five times a layer: stream to norms and q/k/v, these to attention, the heads' outputs to the output product, the stream to norms and up, hidden units to down. A kernel boundary hands on in 3.5 to 4 us
// (the start of a dependent kernel, then its first trip to memory, both for its inputs and for its weights). Inside one kernel whose blocks
// are all on the chip 256 blocks that each store a share and then read everything, and do nothing else, take 2.1 to 3.1 us for 4 to 100 KB. Here, where a block reads what
// it needs and uses first what is there first, a handing-on takes 1.0 to 2.1, and the weights are in registers by then: they do not depend on anything and are asked for a phase earlier.
//
// What is handed on are words of 8 bytes: 4 of numbers and 4 that say of which launch and layer they are (the tag). Who needs the words
// loads them until all tags are the expected ones: no flags, no barriers across the chip, no memory to clear, and what arrives first is
// used first. A word is stored and loaded whole, past the caches that are not shared by the whole chip.
//
// Blocks take one of two parts. Attending blocks own (row, head) pairs: their keys and values are in registers before the query arrives.
// The others own tiles of 16 output columns of each of the four products, all rows at once on the matrix cores, a tile's K divided
// among the block's waves. The owner of a tile of the output product and of the same tile of the down product keeps its part of the residual stream in registers.
//
// Who waits for whom. A wait is only ever for a block that is on the chip. Blocks enter themselves in a count as they start; the set of
// members is closed once, by whoever enters last or by a block that has waited long enough for the rest (another stream's kernels may hold
// the compute units; LOSS_A_LAYER), and blocks that start later leave at once. Work is divided among the members, however many they are. Phases
// follow each other in one order in every block, and a block's waits are for earlier phases only, so the earliest phase that is
// not done can always go on. A wave that has looked for its words very many times takes the device for broken: it goes on without numbers (NaN), so that
// the launch ends, says so in memory that the host reads, and from there on no block keeps keys or values in the cache.
//
// Measured (replayed steps of GPT-2 small in bfloat16 with 512 keys a row; the two layer kernels a layer before): 8 rows 353 -> 206 us a step, 14.4 us a layer, 1 row
// 296 -> 158; in 32-bit (seven kernels a layer before) 8 rows 496 -> 344 (of which the layers 325, and 314 since their sums go on side by side). A layer's 14.4 us are five handings-on from block to block (the stream to normed rows 1.7, q/k/v to the
// attending blocks 1.0, heads' outputs to the output product 1.6, the stream to normed rows 2.1, hidden units to the down product 1.8) and six stretches of a block's own work (q/k/v 1.1,
// scores and values 1.3, their sums 1.2, the stream behind the output product 0.7, hidden units 1.0, the stream behind the down product 0.9). Bound by these trips and by the instructions
// between them (a lone wave's chain, 4 cycles an instruction), not by bytes. Part of that chain are scalars that the compiler brings back from vector lanes: three parts with their regions and
// pointers do not fit 106 scalar registers, 95 of them are spilled where rows have up to 768 columns in bfloat16 (144 for 16 rows), 145 to 236 up to 1,024, 301 to 491 beyond; of vector registers
// 1, and beyond 1,024 columns 32 (119 for 16 rows, which the rule below never sends here); in 32-bit 120 to 292 scalars and 1 to 8 vector registers.
#include "common.h"
#include "key_sweep.h"

#include <type_traits>

namespace {

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;

constexpr int ST_WAVES = 8, ST_THREADS = ST_WAVES * WAVE;
constexpr int ST_HEAD = 64;         // elements of a head
constexpr int ST_MAX_ROWS = 16;     // the other operand's rows on the matrix cores
constexpr int ST_MAX_LAYERS = 64;   // their pointers lie in LDS
constexpr int ST_KEY_LOADS = 16;     // loads of keys, and of values, that a wave keeps in registers: 128 keys in bfloat16, 64 in 32-bit
constexpr int ST_MIN_MEMBERS = 3;   // a block of each part
constexpr int ST_MAX_PAIRS = 4;     // (row, head) pairs of an attending block: its waves are divided among them
// How long (ticks of 10 ns) a launch waits for blocks that have not found a place: CLOSE_AFTER, and what it would lose by going on without them, so that it never
// takes much longer than twice what is best. A step's time goes with one over the members (12 layers of 768 columns, 8 rows in bfloat16, us with
// 16 / 64 / 128 / 192 / 256 blocks: 2,597 / 601 / 344 / 217 / 192), about LOSS_A_LAYER for each time that the missing blocks are as many as the members. Such steps one after the
// other beside another stream's products of 45 us: 200 to 1,080 us each where all that were there after CLOSE_AFTER went on, 220 to 260 now; beside products of
// 177 us 200 to 3,300, and 220 to 590 now.
constexpr int CLOSE_AFTER = 2000, LOSS_A_LAYER = 1000;
// control words, each on a cache line of its own; the last line holds what the host leaves there: PATIENCE, looks at a word, each a trip to memory, before a wave
// takes the device for broken, and GAVE_UP, the address of the word on the host that becomes 1 then (two ints); and for the host TOOK_PART, how many members the last launch had
constexpr int ARRIVED = 0, MEMBERS = 32, LEFT = 64, EPOCH = 96, PATIENCE = 128, GAVE_UP = 130, TOOK_PART = 132, CONTROL_INTS = 160;
constexpr unsigned BROKEN = 0, FIRST_REGION = 128;   // bytes among the words: what is not zero once a wave has given up a wait; where the words to hand on begin

struct StackLayer {
    const float *gain_1, *offset_1;
    const void* w_qkv;
    const float* b_qkv;
    const void* w_out;
    const float* b_out;
    const float *gain_2, *offset_2;
    const void* w_up;
    const float* b_up;
    const void* w_down;
    const float* b_down;
    void *k_pages, *v_pages;
};
constexpr int LAYER_POINTERS = sizeof(StackLayer) / 8;

struct StackArgs {
    const StackLayer* layers;
    const float* rows_in;    // [rows, width]
    float* rows_out;         // [rows, width], the stream behind the last layer; null where that is normed:
    const float *final_gain, *final_offset;
    void* normed_out;        // [rows, width] of the products' type
    const int *token_request, *positions, *slots, *block_tables;
    char* words;             // the regions below, one behind the other
    int* control;
    int n_layers, rows, width, inner, n_heads, max_blocks, page_shift, pairs_a_block, activation;
    float eps_1, eps_2, eps_final, scale;
};

template <typename T>
struct Stacked {
    static constexpr int EPW = 4 / (int)sizeof(T);     // numbers of T in a word
    static constexpr int VEC = 16 / (int)sizeof(T);    // numbers of T in 16 bytes
    static constexpr int KC = 4 * VEC;                 // K columns of a step of the matrix cores' operands: 32 or 16
};

// Stored and loaded past the caches of one compute unit and of one die (the scope of the whole device). The bounds of the
// region are checked by the unit that loads: what would lie outside reads as zero and is not stored.
constexpr int DEVICE_WIDE = 16;
struct Words {
    __amdgpu_buffer_rsrc_t all;
    unsigned first;   // byte of the region among all of them
    // `at`: the lane's own byte, `further`: the same in every lane
    __device__ __forceinline__ u32x4 load(unsigned at, unsigned further) const {
        return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(all, at, first + further, DEVICE_WIDE));
    }
    __device__ __forceinline__ void store(unsigned at, uint32_t a, uint32_t b, uint32_t tag) const {
        __builtin_amdgcn_raw_buffer_store_b128(u32x4{a, tag, b, tag}, all, at, first, DEVICE_WIDE);
    }
};
__device__ __forceinline__ uint32_t bits(float x) { return __builtin_bit_cast(uint32_t, x); }
__device__ __forceinline__ float number(uint32_t x) { return __builtin_bit_cast(float, x); }
__device__ __forceinline__ uint32_t bits_of_pair(float a, float b) {
    bf16x2 p{static_cast<bf16_t>(a), static_cast<bf16_t>(b)};
    return __builtin_bit_cast(uint32_t, p);
}

template <typename V>
__device__ __forceinline__ V load16(const void* uniform_base, unsigned byte_offset) {
    return *reinterpret_cast<const V*>(reinterpret_cast<const char*>(uniform_base) + byte_offset);
}
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Looks that a wave has left, and the block's word for whether any wave of it has given up a wait.
struct Patience {
    int left;
    int* block_gave_up;
    // Whoever reads a word that the block hands on behind this finds BROKEN set.
    __device__ __forceinline__ void give_up(const Words& words) {
        left = 0;
        *static_cast<volatile int*>(block_gave_up) = 1;
        __builtin_amdgcn_raw_buffer_store_b32(1u, words.all, BROKEN, 0, DEVICE_WIDE);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
};

// Loads N pieces of 16 bytes (two words each), piece i `further(i)` bytes behind the lane's `at`, until all of them, in every lane of the wave
// and as far as they count, carry the tag.
template <int N, typename Further, typename Counts>
__device__ __forceinline__ void await_words(u32x4 (&got)[N], const Words& from, uint32_t tag, Patience& patience, unsigned at, Further further, Counts counts) {
    for (;;) {
        asm volatile("" ::: "memory");   // look again, and not at what an earlier look found
#pragma unroll
        for (int i = 0; i < N; i++) got[i] = from.load(at, further(i));
        bool there = true;
#pragma unroll
        for (int i = 0; i < N; i++) there = there && ((got[i][1] == tag && got[i][3] == tag) || !counts(i));
        if (__builtin_amdgcn_ballot_w64(!there) == 0) return;
        if (patience.left-- <= 0) break;
    }
    patience.give_up(from);   // no number at all, here and in all that is computed from it
#pragma unroll
    for (int i = 0; i < N; i++) got[i] = u32x4{~0u, tag, ~0u, tag};
}
template <int N, typename Further>
__device__ __forceinline__ void await_words(u32x4 (&got)[N], const Words& from, uint32_t tag, Patience& patience, unsigned at, Further further) {
    await_words(got, from, tag, patience, at, further, [](int) { return true; });
}
// The same with a place of its own for every piece, in every lane.
template <int N, typename At>
__device__ __forceinline__ void await_words_at(u32x4 (&got)[N], const Words& from, uint32_t tag, Patience& patience, At at) {
    unsigned place[N];
#pragma unroll
    for (int i = 0; i < N; i++) place[i] = at(i);
    for (;;) {
        asm volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < N; i++) got[i] = from.load(place[i], 0);
        bool there = true;
#pragma unroll
        for (int i = 0; i < N; i++) there = there && got[i][1] == tag && got[i][3] == tag;
        if (__builtin_amdgcn_ballot_w64(!there) == 0) return;
        if (patience.left-- <= 0) break;
    }
    patience.give_up(from);
#pragma unroll
    for (int i = 0; i < N; i++) got[i] = u32x4{~0u, tag, ~0u, tag};
}
// A value that is the same in every lane, as if it had just been computed: what follows from it is computed again in every layer (a few scalar
// instructions) and not kept in registers from layer to layer.
template <typename X>
__device__ __forceinline__ void anew(X& x) { asm volatile("" : "+s"(x)); }

// How a region whose rows are operands of a product lies in memory: the pieces of 16 bytes (words 2i and 2i + 1 of the four that a lane holds of a
// step) by step, i, quad (columns quad * VEC .. of the step) and row. Whoever writes should write whole lines of 128 bytes: a line that blocks of
// several dies write pieces of takes them one after the other (the heads' outputs, eight rows: 1 us). So the hidden units, of which a block has 16 columns of all
// rows, have a step's rows side by side, and the heads' outputs, of which a block has 64 columns of one row, a row's steps.
struct Operands {
    unsigned step, row;   // bytes from one to the next
    __device__ __forceinline__ unsigned at(int s, int i, int quad, int r) const { return (unsigned)s * step + (unsigned)i * (step / 2) + (unsigned)quad * (step / 8) + (unsigned)r * row; }
};

// Four (bfloat16) or two (32-bit) neighbouring columns of a row, the first a multiple of as many, as one piece of words.
__device__ __forceinline__ void store_piece(const Words& to, unsigned at, f32x4 v, uint32_t tag) { to.store(at, bits_of_pair(v[0], v[1]), bits_of_pair(v[2], v[3]), tag); }
__device__ __forceinline__ void store_piece(const Words& to, unsigned at, f32x2 v, uint32_t tag) { to.store(at, bits(v[0]), bits(v[1]), tag); }
template <typename T, typename V>
__device__ __forceinline__ void store_operand(const Words& to, const Operands& lie, int row, int column, V v, uint32_t tag) {
    const int step = column / Stacked<T>::KC, within = column % Stacked<T>::KC, quad = within / Stacked<T>::VEC;
    store_piece(to, lie.at(step, within % Stacked<T>::VEC / (Stacked<T>::VEC / 2), quad, row), v, tag);
}

template <typename T>
__device__ __forceinline__ f32x4 multiply(Vec16 w, Vec16 x, f32x4 sum) {
    if constexpr (sizeof(T) == 2) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, x), sum, 0, 0, 0);
    } else {
        const f32x4 a = __builtin_bit_cast(f32x4, w), b = __builtin_bit_cast(f32x4, x);
#pragma unroll
        for (int i = 0; i < 4; i++) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], sum, 0, 0, 0);
        return sum;
    }
}

// A wave's steps of K: wave, wave + 8, ... of a tile of 16 rows of W; zeros beyond K.
template <typename T, int STEPS>
struct Tile {
    Vec16 w[STEPS];
    __device__ __forceinline__ void fetch(const void* matrix, int tile, int n_steps, int wave, int lane) {
        const __amdgpu_buffer_rsrc_t all = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(matrix), 0, -1, 0x00020000);
        const unsigned first = (unsigned)(tile * n_steps + wave) * 1024u;
#pragma unroll
        for (int j = 0; j < STEPS; j++) {
            if (wave + ST_WAVES * j < n_steps) w[j] = __builtin_bit_cast(Vec16, __builtin_amdgcn_raw_buffer_load_b128(all, lane * 16, first + (unsigned)(ST_WAVES * j) * 1024u, 0));
            else w[j] = Vec16{{0u, 0u, 0u, 0u}};
        }
    }
};

// Elements from one normed row in LDS to the next: whole rounds of the 64 banks and a quarter round, so that four rows' pieces of a step (64 bytes each) share no bank.
__host__ __device__ __forceinline__ int normed_stride(int width, int element) { return ((width * element + 255) / 256 * 256 + 64) / element; }

// Sums that a wave's steps of K take in turn, of the products that the rows' blocks and that the norming blocks do. In 32-bit a product's error is that of its sums' roundings in a row: the
// relative error of a step's logits against 64 bits, three layers, with one sum each / two and one / four and two / layer by layer, in 1e-7: 768 columns, 8 rows 5.7 / 5.0 / 4.2 / 5.1,
// 1,024 columns, 2 rows 6.6 / 5.6 / 4.7 / 5.0, 16 rows 6.3 / 5.4 / 4.6 / 5.1. (A step of 12 layers, 8 rows: 768 columns 318 / 312 / 313 us, products of one sum wait for each other; 1,024
// 405 / 403 / 400, of fewer loads at a time.) In bfloat16 the operands' own rounding is all there is to see.
template <typename T>
constexpr int SUMS_OVER_UNITS = sizeof(T) == 4 ? 4 : 1;
template <typename T>
constexpr int SUMS_OVER_WIDTH = sizeof(T) == 4 ? 2 : 1;

constexpr int PART_STRIDE = 20;   // floats a row of a tile's partial sums: 16, and 4 that spread the rows over the LDS banks
typedef float PartRows[ST_WAVES][ST_MAX_ROWS][PART_STRIDE];

// The sum over a wave's four rows of 16 lanes of the numbers of the lanes in the same place, in every lane.
__device__ __forceinline__ float rows_total(float x) {
    auto halves = __builtin_amdgcn_permlane32_swap(bits(x), bits(x), false, false);
    x = number(halves[0]) + number(halves[1]);
    auto rows = __builtin_amdgcn_permlane16_swap(bits(x), bits(x), false, false);
    return number(rows[0]) + number(rows[1]);
}

// STEPS: steps of K a wave has of a product over the width, at most; of one over the hidden units four times that. TILES: tiles of the q/k/v and
// up products whose rows of W a block asks for ahead. ROWS: a power of two, as many rows or more: a load of operands takes in 16 / ROWS steps of K.
template <typename T, int STEPS, int TILES, int ROWS>
__global__ __launch_bounds__(ST_THREADS) void decode_stack_kernel(StackArgs a) {
    typedef Stacked<T> S;
    typedef KeySweep<T, ST_HEAD> Sweep;
    typedef typename Sweep::Raw Raw;
    constexpr int EPW = S::EPW, VEC = S::VEC, KC = S::KC;
    constexpr int NORM_PIECES = (STEPS * ST_WAVES * KC + 127) / 128;   // 16-byte pieces of words a lane has of a row
    constexpr int NORM_ROWS = ROWS > ST_WAVES ? 2 : 1;   // rows a wave norms
    extern __shared__ __attribute__((aligned(16))) char lds[];
    __shared__ StackLayer layer_at[ST_MAX_LAYERS];
    __shared__ int shared_rank, shared_members, shared_epoch, shared_patience, shared_gave_up;

    // each on its own: kept together, as they arrive, sixteen scalar registers are brought back for one
    anew(a.words), anew(a.rows_in), anew(a.rows_out), anew(a.block_tables), anew(a.token_request), anew(a.positions), anew(a.slots), anew(a.layers), anew(a.control);
    anew(a.scale), anew(a.eps_1), anew(a.eps_2), anew(a.rows), anew(a.width), anew(a.inner), anew(a.n_heads), anew(a.page_shift), anew(a.n_layers), anew(a.activation);
    const int tid = threadIdx.x, lane = tid % WAVE;
    int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    int M = a.rows, width = a.width, inner = a.inner;
    if (tid == 0) {
        shared_patience = a.control[PATIENCE], shared_gave_up = 0;
        shared_epoch = __hip_atomic_load(a.control + EPOCH, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int blocks = (int)gridDim.x;
        const int rank = __hip_atomic_fetch_add(a.control + ARRIVED, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        auto close = [&](int count) {
            int open = 0;
            __hip_atomic_compare_exchange_strong(a.control + MEMBERS, &open, count, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        };
        if (rank == blocks - 1) close(blocks);
        const long long since = wall_clock64();
        int members;
        while ((members = __hip_atomic_load(a.control + MEMBERS, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == 0) {
            const long long waited = wall_clock64() - since;
            if (waited > CLOSE_AFTER) {
                const int count = min(__hip_atomic_load(a.control + ARRIVED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), blocks);
                if (count >= ST_MIN_MEMBERS && (waited - CLOSE_AFTER) * count > (long long)LOSS_A_LAYER * a.n_layers * (blocks - count)) close(count);
            }
        }
        shared_members = members;
        shared_rank = members == blocks ? (int)blockIdx.x : rank;   // everyone is there: neighbouring ranks on different dies
    }
    for (int i = tid; i < a.n_layers * LAYER_POINTERS; i += ST_THREADS)
        reinterpret_cast<unsigned long long*>(layer_at)[i] = reinterpret_cast<const unsigned long long*>(a.layers)[i];
    __syncthreads();
    const int members = __builtin_amdgcn_readfirstlane(shared_members), rank = __builtin_amdgcn_readfirstlane(shared_rank);
    const uint32_t first_tag = (uint32_t)__builtin_amdgcn_readfirstlane(shared_epoch) * (uint32_t)(a.n_layers + 1) + 1u;

    // the regions of words: a layer's input rows, the rows behind its attention, q/k/v, the heads' outputs, the hidden units
    const unsigned row_bytes = (unsigned)(M * width) * 8u, mixed_bytes = row_bytes / EPW, unit_bytes = (unsigned)(M * inner) * 8u / EPW;
    const unsigned region_ends = FIRST_REGION + 2 * row_bytes + 4 * mixed_bytes;
    const __amdgpu_buffer_rsrc_t all_words = __builtin_amdgcn_make_buffer_rsrc(a.words, 0, region_ends + unit_bytes, 0x00020000);
    const Words rows_words{all_words, FIRST_REGION}, later_words{all_words, FIRST_REGION + row_bytes}, qkv_words{all_words, FIRST_REGION + 2 * row_bytes};
    const Words mixed_words{all_words, FIRST_REGION + 2 * row_bytes + 3 * mixed_bytes}, unit_words{all_words, region_ends};

    const Operands mixed_lie{128u, (unsigned)(width / KC) * 128u}, unit_lie{(unsigned)M * 128u, 16u};
    // a tile's 16 columns of q, k or v lie together, row behind row
    constexpr unsigned QKV_TILE_ROW = 16 / EPW * 8;
    auto qkv_at = [&](int row, int column) { return (unsigned)(column / 16 * M + row) * QKV_TILE_ROW + (unsigned)(column % 16 / EPW) * 8u; };

    // who does what: attending blocks, blocks that own tiles of the rows (output and down products), blocks that norm (q/k/v and up products)
    const int pairs = M * a.n_heads, per_block = a.pairs_a_block, groups = (pairs + per_block - 1) / per_block;
    const int row_tiles = width / 16;
    const int attending = min(groups, max(members / 2, 1)), summing = min(row_tiles, max((members - attending) / 2, 1));
    const int norming = members - attending - summing;
    Patience patience{__builtin_amdgcn_readfirstlane(shared_patience), &shared_gave_up};
    auto pointer = [&](auto StackLayer::*which, int layer) {   // a pointer of a layer, in scalar registers
        const unsigned long long held = (unsigned long long)(layer_at[layer].*which);
        const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)held), hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(held >> 32));
        return reinterpret_cast<typename std::remove_reference<decltype(layer_at[layer].*which)>::type>((unsigned long long)hi << 32 | lo);
    };

    // What adds up a tile's eight partial sums, one a wave. A thread's columns of a row are what it stores as one piece of 16 bytes (a line
    // that arrives in one store is there at once, in two it is not): four where they go on in bfloat16, two in 32-bit.
    const int row16 = lane % 16, quad = lane / 16, own_row = min(row16, M - 1);
    auto leave_part = [&](PartRows& part, f32x4 sum) { *reinterpret_cast<f32x4*>(&part[wave][row16][4 * quad]) = sum; };
    auto whole_sum = [&](const PartRows& part, int row, int column, auto columns) {
        typedef typename decltype(columns)::type V;
        V sum = *reinterpret_cast<const V*>(&part[0][row][column]);
#pragma unroll
        for (int w = 1; w < ST_WAVES; w++) sum += *reinterpret_cast<const V*>(&part[w][row][column]);
        return sum;
    };
    struct Two { typedef f32x2 type; };
    struct Four { typedef f32x4 type; };
    typedef typename std::conditional<sizeof(T) == 2, Four, Two>::type Own;   // of a product whose numbers go on in T
    typedef typename Own::type OwnColumns;
    constexpr int OWN = 4 / (sizeof(T) / 2), TILE_THREADS = ST_MAX_ROWS * 16 / OWN;
    // Partial sums alternate between two places in LDS: a wave may be at the next product's while the last one's are still being added up, and meets
    // the others in between.
    int turn = 0;

    if (rank < attending) {
        // ---- attending: the block's waves are divided among its pairs, and a pair's waves share its keys, the token's own (the newest) among them
        constexpr int LPR = Sweep::LPR, RPI = Sweep::RPI;   // lanes that share a key, keys a load of the wave covers
        float (*merged)[ST_HEAD + 4] = reinterpret_cast<float (*)[ST_HEAD + 4]>(lds);   // [waves]: output, maximum, sum
        Vec16 (*own_rows)[2][LPR] = reinterpret_cast<Vec16 (*)[2][LPR]>(lds + sizeof(float) * ST_WAVES * (ST_HEAD + 4));   // [waves]: the token's own key and value
        const int pair_waves = ST_WAVES / per_block, wave_in_pair = wave % pair_waves;
        const int sub = lane % LPR, group_in_wave = lane / LPR, page_mask = (1 << a.page_shift) - 1;
        int token, head, slot, far, begin, end, own;   // the wave's keys: far .. begin-1 from memory, begin .. end-1 in registers; the own key's place among these (or none: < 0)
        bool live;
        const int* table;
        unsigned key_at[ST_KEY_LOADS];   // where the lane's pieces of the keys lie in a layer's pages, in bytes
        Raw keys[ST_KEY_LOADS], values[ST_KEY_LOADS];
        Sweep sweep;
        auto take_up = [&](int group) {
            const int pair = group * per_block + wave / pair_waves;
            live = pair < pairs;
            token = live ? pair / a.n_heads : 0, head = live ? pair % a.n_heads : 0;
            const int request = __builtin_amdgcn_readfirstlane(a.token_request[token]);
            const int position = request < 0 || !live ? 0 : __builtin_amdgcn_readfirstlane(a.positions[token]);
            slot = request < 0 || !live ? -1 : __builtin_amdgcn_readfirstlane(a.slots[token]);
            // a padding row has its own key alone; what its wave loads meanwhile is a row of the first page
            table = a.block_tables + (size_t)max(request, 0) * a.max_blocks;
            const int share = ((position + pair_waves) / pair_waves + RPI - 1) / RPI * RPI;
            far = min(wave_in_pair * share, position + 1);
            end = min(far + share, position + 1);
            begin = max(far, end - ST_KEY_LOADS * RPI);
            own = end == position + 1 && begin < end ? position - begin : -1;
#pragma unroll
            for (int u = 0; u < ST_KEY_LOADS; u++) {
                const int key = max(min(begin + u * RPI + group_in_wave, end - 1), 0);   // lanes past the last key take it again; they do not count
                const unsigned page = (unsigned)max(table[key >> a.page_shift], 0);
                key_at[u] = ((((page * (unsigned)a.n_heads + (unsigned)head) << a.page_shift) + (unsigned)(key & page_mask)) * ST_HEAD + (unsigned)(sub * VEC)) * (unsigned)sizeof(T);
            }
        };
        int taken_up = -1;
#pragma unroll 1
        for (int layer = 0; layer < a.n_layers; layer++) {
            const uint32_t tag = first_tag + (uint32_t)layer;
#pragma unroll 1
            for (int group = rank; group < groups; group += attending) {   // one, as a rule
                if (group != taken_up) take_up(group);
                taken_up = group;
                {   // asked for long before there is a query, which takes the other blocks the rest of the layer before
                    const void *k_pages = pointer(&StackLayer::k_pages, layer), *v_pages = pointer(&StackLayer::v_pages, layer);
#pragma unroll
                    for (int u = 0; u < ST_KEY_LOADS; u++)
                        if (u * RPI < end - begin) keys[u] = load16<Raw>(k_pages, key_at[u]);
#pragma unroll
                    for (int u = 0; u < ST_KEY_LOADS; u++)
                        if (u * RPI < end - begin) values[u] = load16<Raw>(v_pages, key_at[u]);
                }
                // the query; the wave that has the token's own key and value also takes these
                const unsigned q_at = qkv_at(token, head * ST_HEAD + sub * VEC), step = (unsigned)(width / 16 * M) * QKV_TILE_ROW;
                u32x4 q_words[2];
                if (own >= 0) {
                    u32x4 six[6];
                    await_words(six, qkv_words, tag, patience, q_at, [&](int i) { return (unsigned)(i / 2) * step + (unsigned)(i % 2) * 16u; });
                    q_words[0] = six[0], q_words[1] = six[1];
                    const Vec16 key{{six[2][0], six[2][2], six[3][0], six[3][2]}}, value{{six[4][0], six[4][2], six[5][0], six[5][2]}};
                    if (lane < LPR) own_rows[wave][0][sub] = key, own_rows[wave][1][sub] = value;
#pragma unroll
                    for (int u = 0; u < ST_KEY_LOADS; u++)
                        if (u == own / RPI && group_in_wave >= own % RPI) keys[u] = __builtin_bit_cast(Raw, key), values[u] = __builtin_bit_cast(Raw, value);
                } else {
                    await_words(q_words, qkv_words, tag, patience, q_at, [&](int i) { return (unsigned)i * 16u; });
                }
                const Vec16 query{{q_words[0][0], q_words[0][2], q_words[1][0], q_words[1][2]}};
                sweep.init();
                float scaled[VEC];
#pragma unroll
                for (int i = 0; i < VEC; i++) scaled[i] = to_float(reinterpret_cast<const T*>(&query)[i]) * a.scale;
                if (far < begin) {   // more keys than the wave's registers hold
                    const T *k_pages = reinterpret_cast<const T*>(pointer(&StackLayer::k_pages, layer)), *v_pages = reinterpret_cast<const T*>(pointer(&StackLayer::v_pages, layer));
                    if constexpr (sizeof(T) == 2) sweep.keys(__builtin_bit_cast(bf16x8, query), a.scale, k_pages, v_pages, table, head, a.n_heads, a.page_shift, far, begin, lane);
                    else sweep.keys(scaled, k_pages, v_pages, table, head, a.n_heads, a.page_shift, far, begin, lane);
                }
                // all scores of the keys in registers, then one maximum, then their weights and the weighted values
                float score[ST_KEY_LOADS], most = -INFINITY;
#pragma unroll
                for (int u = 0; u < ST_KEY_LOADS; u++) {
                    score[u] = -INFINITY;
                    if (u * RPI < end - begin) {
                        float dot = 0.0f;
                        if constexpr (sizeof(T) == 2) {
                            const bf16x2 *q = reinterpret_cast<const bf16x2*>(&query), *k = reinterpret_cast<const bf16x2*>(&keys[u]);
#pragma unroll
                            for (int i = 0; i < VEC / 2; i++) dot = __builtin_amdgcn_fdot2_f32_bf16(q[i], k[i], dot, false);
                            dot *= a.scale;
                        } else {
#pragma unroll
                            for (int i = 0; i < VEC; i++) dot += scaled[i] * keys[u][i];
                        }
                        dot = lanes_sum<LPR>(dot);
                        score[u] = begin + u * RPI + group_in_wave < end ? dot : -INFINITY;
                        most = fmaxf(most, score[u]);
                    }
                }
                most = fmaxf(sweep.running_max, wave_max_total(most));
                const float reference = most == -INFINITY ? 0.0f : most;   // a wave without keys
                const float rescale = sweep_exp<T>(sweep.running_max - reference);
                sweep.running_sum *= rescale;
#pragma unroll
                for (int i = 0; i < VEC; i++) sweep.o[i] *= rescale;
#pragma unroll
                for (int u = 0; u < ST_KEY_LOADS; u++)
                    if (u * RPI < end - begin) {
                        const float p = sweep_exp<T>(score[u] - reference);
                        sweep.running_sum += p;
#pragma unroll
                        for (int i = 0; i < VEC; i++) sweep.o[i] += p * Chunk<T>::get(values[u], i);
                    }
                sweep.merge_inside_rows();   // the wave's four rows of lanes have one maximum: their sums are added as they are
                sweep.running_sum = rows_total(sweep.running_sum);
#pragma unroll
                for (int i = 0; i < VEC; i++) sweep.o[i] = rows_total(sweep.o[i]);
                if (lane < LPR) {
#pragma unroll
                    for (int i = 0; i < VEC; i += 4) *reinterpret_cast<f32x4*>(&merged[wave][sub * VEC + i]) = f32x4{sweep.o[i], sweep.o[i + 1], sweep.o[i + 2], sweep.o[i + 3]};
                }
                if (lane == 0) *reinterpret_cast<f32x2*>(&merged[wave][ST_HEAD]) = f32x2{most, sweep.running_sum};
                lds_barrier();   // every wave's (output, maximum, sum) is in LDS
                if (wave_in_pair == 0) {   // a lane an element; the weights of the pair's waves in the first lanes
                    float part[ST_WAVES];
#pragma unroll
                    for (int w = 0; w < ST_WAVES; w++) part[w] = merged[wave + min(w, pair_waves - 1)][lane];
                    const f32x2 state = *reinterpret_cast<const f32x2*>(&merged[wave + min(lane, pair_waves - 1)][ST_HEAD]);
                    const float wave_most = lane < pair_waves ? state[0] : -INFINITY;
                    const float weight = sweep_exp<T>(wave_most - wave_max_total(wave_most));   // a maximum there is: the token's own key counts
                    const float sum = wave_total(lane < pair_waves ? weight * state[1] : 0.0f);
                    float out = 0.0f;
#pragma unroll
                    for (int w = 0; w < ST_WAVES; w++) out += number((uint32_t)__builtin_amdgcn_readlane((int)bits(weight), w)) * part[w];   // (zero beyond the pair's waves)
                    out = slot < 0 ? 0.0f : out / sum;
                    OwnColumns piece;   // of each four or two lanes
                    if constexpr (sizeof(T) == 2) piece = f32x4{out, dpp_moved<0x55>(out), dpp_moved<0xAA>(out), dpp_moved<0xFF>(out)};
                    else piece = f32x2{out, dpp_moved<0xB1>(out)};
                    if (lane % OWN == 0 && live) store_operand<T>(mixed_words, mixed_lie, token, head * ST_HEAD + lane, piece, tag);
                }
                lds_barrier();   // what this layer has to say is on its way before the next keys are asked for: a unit's memory pipeline is one queue
                // Into the cache, for later steps, once all else is done that others wait for: behind a look at whether these are numbers.
                if (own >= 0 && slot >= 0 && __builtin_amdgcn_raw_buffer_load_b32(all_words, BROKEN, 0, DEVICE_WIDE) == 0u && lane < LPR) {
                    const size_t row = ((((size_t)(slot >> a.page_shift) * a.n_heads + head) << a.page_shift) + (slot & page_mask)) * ST_HEAD + sub * VEC;
                    *reinterpret_cast<Vec16*>(reinterpret_cast<T*>(pointer(&StackLayer::k_pages, layer)) + row) = own_rows[wave][0][sub];
                    *reinterpret_cast<Vec16*>(reinterpret_cast<T*>(pointer(&StackLayer::v_pages, layer)) + row) = own_rows[wave][1][sub];
                }
            }
        }
    } else if (rank < attending + summing) {
        // ---- tiles of the rows: output product and down product, and the residual stream at their columns
        PartRows* parts = reinterpret_cast<PartRows*>(lds);   // [2]
        const int g = rank - attending;
        int width_steps = width / KC, unit_steps = inner / KC;
        // The wave's steps of a tile, their rows straight into its registers. The matrix cores' operand has 16 rows: where there are fewer, one
        // load takes in several of the wave's steps, a step's rows behind the last one's, and a step's turn comes by turning the lanes' rows
        // (what the rows beyond hold meanwhile goes into sums that nobody takes).
        constexpr int FOLD = ST_MAX_ROWS / ROWS;
        auto operand_sum = [&](const auto& w, const Words& from, const Operands& lie, int n_steps, uint32_t tag) {
            constexpr int ALL = (int)(sizeof(w.w) / sizeof(Vec16)), LOADS = (ALL + FOLD - 1) / FOLD;
            constexpr int CHUNK = LOADS <= 12 ? LOADS : LOADS == 16 && sizeof(T) == 4 ? 4 : LOADS % 8 == 0 ? 8 : 7;   // (1,024 columns, 8 rows in 32-bit: eight at a time spill 39 registers, 424 us a step for 399)
            static_assert(LOADS % CHUNK == 0, "whole chunks");
            const int folded = row16 / ROWS, folded_row = min(row16 % ROWS, M - 1);
            constexpr int SUMS = SUMS_OVER_UNITS<T>;
            f32x4 sum[SUMS];
#pragma unroll
            for (int i = 0; i < SUMS; i++) sum[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            auto turned = [&](auto amount, u32x4 a, u32x4 b) {
                constexpr int N = decltype(amount)::value;
                Vec16 x{{a[0], a[2], b[0], b[2]}};
                if constexpr (N > 0) {
#pragma unroll
                    for (int i = 0; i < 4; i++) x.w[i] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x.w[i], 0x120 + (16 - N), 0xf, 0xf, false);   // lane r of 16 takes lane (r + N) % 16
                }
                return x;
            };
#pragma unroll
            for (int c = 0; c < LOADS; c += CHUNK) {
                u32x4 got[2 * CHUNK];
                // steps past the wave's last take its first ones again; their rows of W are zeros
                const int left = n_steps - wave;   // > 0 where the wave has a step
                auto lane_step = [&](int load) { return (load * FOLD + folded) * ST_WAVES; };
                if constexpr (FOLD == 1) {
                    await_words(got, from, tag, patience, lie.at(0, 0, quad, folded_row),
                                [&](int i) { return lie.at(min(wave + ST_WAVES * (c + i / 2), n_steps - 1), i % 2, 0, 0); });
                } else {
                    // the lane's own step differs within the wave: clamped per lane where the last load is not full
                    u32x4 (&all)[2 * CHUNK] = got;
                    await_words_at(all, from, tag, patience, [&](int i) {
                        const int past = lane_step(c + i / 2);
                        return lie.at(past < left ? wave + past : min(wave, n_steps - 1), i % 2, quad, folded_row);
                    });
                }
#pragma unroll
                for (int j = 0; j < CHUNK; j++) {
                    auto step = [&](auto fold) {
                        constexpr int F = decltype(fold)::value;
                        if constexpr (F < FOLD) {
                            if ((c + j) * FOLD + F < ALL) {
                                f32x4& into = sum[((c + j) * FOLD + F) % SUMS];
                                into = multiply<T>(w.w[(c + j) * FOLD + F < ALL ? (c + j) * FOLD + F : 0], turned(std::integral_constant<int, F * ROWS % 16>{}, got[2 * j], got[2 * j + 1]), into);
                            }
                        }
                    };
                    step(std::integral_constant<int, 0>{}), step(std::integral_constant<int, 1>{}), step(std::integral_constant<int, 2>{}), step(std::integral_constant<int, 3>{});
                    step(std::integral_constant<int, 4>{}), step(std::integral_constant<int, 5>{}), step(std::integral_constant<int, 6>{}), step(std::integral_constant<int, 7>{});
                    step(std::integral_constant<int, 8>{}), step(std::integral_constant<int, 9>{}), step(std::integral_constant<int, 10>{}), step(std::integral_constant<int, 11>{});
                    step(std::integral_constant<int, 12>{}), step(std::integral_constant<int, 13>{}), step(std::integral_constant<int, 14>{}), step(std::integral_constant<int, 15>{});
                }
            }
#pragma unroll
            for (int apart = 1; apart < SUMS; apart *= 2)
#pragma unroll
                for (int i = 0; i + apart < SUMS; i += 2 * apart) sum[i] += sum[i + apart];
            return sum[0];
        };
        const int sum_row = tid / 8, sum_column = tid % 8 * 2;   // two columns of a row to a thread: the stream goes on in 32-bit
        const bool sums = sum_row < M;
        f32x2 stream = f32x2{0.0f, 0.0f};   // the residual stream there (at the block's first tile)
        if (sums) stream = *reinterpret_cast<const f32x2*>(a.rows_in + (size_t)sum_row * width + g * 16 + sum_column);
        // what the stream is at another of the block's tiles
        auto stream_at = [&](const Words& words, bool plain, uint32_t tag, int tile) {
            const int column = tile * 16 + sum_column, row = min(sum_row, M - 1);
            if (plain) return *reinterpret_cast<const f32x2*>(a.rows_in + (size_t)row * width + column);
            u32x4 got[1];
            await_words(got, words, tag, patience, (unsigned)(row * width + column) * 8u, [&](int) { return 0u; });
            return f32x2{number(got[0][0]), number(got[0][2])};
        };
        auto store_stream = [&](const Words& to, int tile, f32x2 v, uint32_t tag) { store_piece(to, (unsigned)(sum_row * width + tile * 16 + sum_column) * 8u, v, tag); };
        // One product and its sum with the stream: `keep(tile, rows)` in the threads that add up.
        auto summed_product = [&](auto& w, const void* matrix, const float* bias, const Words& from, const Operands& lie, int n_steps, uint32_t tag, auto before, auto keep) {
#pragma unroll 1
            for (int tile = g; tile < row_tiles; tile += summing) {
                if (tile != g) w.fetch(matrix, tile, n_steps, wave, lane);
                f32x2 add = f32x2{0.0f, 0.0f};
                if (sums) add = *reinterpret_cast<const f32x2*>(bias + tile * 16 + sum_column);
                PartRows& part = parts[turn];
                turn ^= 1;
                const f32x4 sum = operand_sum(w, from, lie, n_steps, tag);
                leave_part(part, sum);
                lds_barrier();
                if (tid < ST_MAX_ROWS * 8) {
                    const f32x2 here = tile == g ? stream : before(tile);
                    if (sums) {
                        const f32x2 v = here + (whole_sum(part, sum_row, sum_column, Two{}) + add);
                        if (tile == g) stream = v;
                        keep(tile, v);
                    }
                }
            }
        };
        Tile<T, STEPS> out_w;
        out_w.fetch(pointer(&StackLayer::w_out, 0), g, width_steps, wave, lane);
#pragma unroll 1
        for (int layer = 0; layer < a.n_layers; layer++) {
            anew(wave), anew(M), anew(width), anew(width_steps), anew(unit_steps);
            const uint32_t tag = first_tag + (uint32_t)layer;
            const bool first_layer = layer == 0, last_layer = layer + 1 == a.n_layers;
            summed_product(out_w, pointer(&StackLayer::w_out, layer), pointer(&StackLayer::b_out, layer), mixed_words, mixed_lie, width_steps, tag,
                           [&](int tile) { return stream_at(rows_words, first_layer, tag, tile); },
                           [&](int tile, f32x2 v) { store_stream(later_words, tile, v, tag); });
            Tile<T, 4 * STEPS> down_w;
            lds_barrier();
            down_w.fetch(pointer(&StackLayer::w_down, layer), g, unit_steps, wave, lane);
            summed_product(down_w, pointer(&StackLayer::w_down, layer), pointer(&StackLayer::b_down, layer), unit_words, unit_lie, unit_steps, tag,
                           [&](int tile) { return stream_at(later_words, false, tag, tile); },
                           [&](int tile, f32x2 v) {
                               if (last_layer && a.rows_out) *reinterpret_cast<f32x2*>(a.rows_out + (size_t)sum_row * width + tile * 16 + sum_column) = v;
                               else store_stream(rows_words, tile, v, tag + 1u);
                           });
            lds_barrier();
            out_w.fetch(pointer(&StackLayer::w_out, min(layer + 1, a.n_layers - 1)), g, width_steps, wave, lane);
        }
    } else if (rank < members) {
        // ---- norm and the products that widen: q/k/v, up
        const int g = rank - attending - summing;
        int stride = normed_stride(width, (int)sizeof(T));   // of a normed row in LDS
        T* normed = reinterpret_cast<T*>(lds);                                                                                     // [rows][stride]
        PartRows* parts = reinterpret_cast<PartRows*>(lds + (((size_t)M * stride * sizeof(T) + 15) & ~(size_t)15));   // [2][TILES]
        int width_steps = width / KC;
        const int qkv_tiles = 3 * width / 16, up_tiles = inner / 16;

        const int sum_tile = tid / TILE_THREADS, sum_row = tid % TILE_THREADS / (16 / OWN), sum_column = tid % (16 / OWN) * OWN;

        Tile<T, STEPS> w[TILES];
        auto fetch_tiles = [&](const void* matrix, int tiles, int first) {
#pragma unroll
            for (int t = 0; t < TILES; t++)
                if (t == 0 || first + t * norming < tiles) w[t].fetch(matrix, min(first + t * norming, tiles - 1), width_steps, wave, lane);
        };
        f32x2 gain[NORM_PIECES], offset[NORM_PIECES];
        auto ask_norm = [&](const float* gains, const float* offsets) {
#pragma unroll
            for (int i = 0; i < NORM_PIECES; i++) {
                gain[i] = offset[i] = f32x2{0.0f, 0.0f};
                if (128 * i + 2 * lane < width) {
                    gain[i] = load16<f32x2>(gains + 128 * i, lane * 8);
                    offset[i] = load16<f32x2>(offsets + 128 * i, lane * 8);
                }
            }
        };
        // rows -> norm -> LDS
        auto norm_rows = [&](const Words& from, bool plain, uint32_t tag, float eps) {
            if (wave >= M) return;
            u32x4 got[NORM_ROWS * NORM_PIECES];
            auto row_of = [&](int r) { return min(wave + r * ST_WAVES, M - 1); };
            auto inside = [&](int i) { return 128 * (i % NORM_PIECES) + 2 * lane < width; };
            if (plain) {
#pragma unroll
                for (int i = 0; i < NORM_ROWS * NORM_PIECES; i++) {
                    got[i] = u32x4{0u, 0u, 0u, 0u};
                    if (inside(i)) {
                        const f32x2 two = load16<f32x2>(a.rows_in + (size_t)row_of(i / NORM_PIECES) * width + 128 * (i % NORM_PIECES), lane * 8);
                        got[i] = u32x4{bits(two[0]), 0u, bits(two[1]), 0u};
                    }
                }
            } else {
                await_words(got, from, tag, patience, (unsigned)lane * 16u,
                            [&](int i) { return (unsigned)(row_of(i / NORM_PIECES) * width + 128 * (i % NORM_PIECES)) * 8u; }, inside);
            }
            auto norm = [&](auto whole_constant) {
                constexpr bool WHOLE = decltype(whole_constant)::value;   // the row fills the lanes' pieces
#pragma unroll
                for (int r = 0; r < NORM_ROWS; r++) {
                    if (wave + r * ST_WAVES >= M) break;
                    const u32x4* row = got + r * NORM_PIECES;
                    auto counts = [&](int i) { return WHOLE || 128 * i + 2 * lane < width; };
                    float sum = 0.0f;
#pragma unroll
                    for (int i = 0; i < NORM_PIECES; i++) sum += counts(i) ? number(row[i][0]) + number(row[i][2]) : 0.0f;
                    const float mean = wave_total(sum) / (float)width;
                    float squares = 0.0f;
#pragma unroll
                    for (int i = 0; i < NORM_PIECES; i++) {
                        const float d = number(row[i][0]) - mean, e = number(row[i][2]) - mean;
                        squares += counts(i) ? d * d + e * e : 0.0f;
                    }
                    const float variance = wave_total(squares) / (float)width + eps;
                    float inverse_stddev;
                    if constexpr (sizeof(T) == 2) inverse_stddev = __builtin_amdgcn_rsqf(variance);   // one unit in the last of 24 bits, of which eight are kept
                    else inverse_stddev = 1.0f / sqrtf(variance);
                    T* to = normed + (wave + r * ST_WAVES) * stride + 2 * lane;
#pragma unroll
                    for (int i = 0; i < NORM_PIECES; i++) {
                        if (counts(i)) {
                            const float y = (number(row[i][0]) - mean) * inverse_stddev * gain[i][0] + offset[i][0];
                            const float z = (number(row[i][2]) - mean) * inverse_stddev * gain[i][1] + offset[i][1];
                            if constexpr (sizeof(T) == 2) *reinterpret_cast<uint32_t*>(to + 128 * i) = bits_of_pair(y, z);
                            else *reinterpret_cast<f32x2*>(to + 128 * i) = f32x2{y, z};
                        }
                    }
                }
            };
            if (width == 128 * NORM_PIECES) norm(std::true_type{});
            else norm(std::false_type{});
        };
        // Tiles g, g + norming, ... of a product over the normed rows: `finish(tile, sums of four columns)` in the threads that add up.
        auto normed_product = [&](const Words& from, bool plain, uint32_t tag, float eps, const float* gains, const float* offsets, const void* matrix, const float* bias,
                                  int tiles, auto finish) {
            if (g >= tiles) return;
            ask_norm(gains, offsets);
            auto bias_of = [&](int first) {
                const int tile = first + sum_tile * norming;
                OwnColumns out = {};
                if (sum_tile < TILES && tile < tiles) out = *reinterpret_cast<const OwnColumns*>(bias + tile * 16 + sum_column);
                return out;
            };
            OwnColumns add = bias_of(g);
            norm_rows(from, plain, tag, eps);
            lds_barrier();
#pragma unroll 1
            for (int first = g; first < tiles; first += TILES * norming) {
                if (first != g) {
                    add = bias_of(first);
                    fetch_tiles(matrix, tiles, first);
                }
                PartRows* part = parts + turn * TILES;
                turn ^= 1;
                constexpr int SUMS = SUMS_OVER_WIDTH<T>;
                f32x4 sum[TILES][SUMS];
#pragma unroll
                for (int t = 0; t < TILES; t++)
#pragma unroll
                    for (int i = 0; i < SUMS; i++) sum[t][i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int j = 0; j < STEPS; j++) {
                    const int step = min(wave + ST_WAVES * j, width_steps - 1);
                    const Vec16 x = *reinterpret_cast<const Vec16*>(normed + own_row * stride + step * KC + quad * VEC);
#pragma unroll
                    for (int t = 0; t < TILES; t++)
                        if (t == 0 || first + t * norming < tiles) sum[t][j % SUMS] = multiply<T>(w[t].w[j], x, sum[t][j % SUMS]);
                }
#pragma unroll
                for (int t = 0; t < TILES; t++)
                    if (t == 0 || first + t * norming < tiles) {
#pragma unroll
                        for (int i = 1; i < SUMS; i++) sum[t][0] += sum[t][i];
                        leave_part(part[t], sum[t][0]);
                    }
                lds_barrier();
                const int tile = first + sum_tile * norming;
                if (sum_tile < TILES && tile < tiles && sum_row < M) finish(tile, whole_sum(part[sum_tile], sum_row, sum_column, Own{}) + add);
            }
        };

        fetch_tiles(pointer(&StackLayer::w_qkv, 0), qkv_tiles, g);
#pragma unroll 1
        for (int layer = 0; layer < a.n_layers; layer++) {
            anew(wave), anew(M), anew(width), anew(width_steps), anew(stride);
            const uint32_t tag = first_tag + (uint32_t)layer;
            normed_product(rows_words, layer == 0, tag, a.eps_1, pointer(&StackLayer::gain_1, layer), pointer(&StackLayer::offset_1, layer),
                           pointer(&StackLayer::w_qkv, layer), pointer(&StackLayer::b_qkv, layer), qkv_tiles, [&](int tile, OwnColumns v) {
                               store_piece(qkv_words, qkv_at(sum_row, tile * 16 + sum_column), v, tag);
                           });
            lds_barrier();
            fetch_tiles(pointer(&StackLayer::w_up, layer), up_tiles, g);
            normed_product(later_words, false, tag, a.eps_2, pointer(&StackLayer::gain_2, layer), pointer(&StackLayer::offset_2, layer),
                           pointer(&StackLayer::w_up, layer), pointer(&StackLayer::b_up, layer), up_tiles, [&](int tile, OwnColumns v) {
#pragma unroll
                               for (int i = 0; i < OWN; i++) {
                                   if constexpr (sizeof(T) == 2) v[i] = a.activation == MLLM_EPI_GELU_TANH ? gelu_tanh_for_bf16(v[i]) : gelu_erf_for_bf16(v[i]);
                                   else v[i] = a.activation == MLLM_EPI_GELU_TANH ? gelu_tanh(v[i]) : gelu_erf(v[i]);
                               }
                               store_operand<T>(unit_words, unit_lie, sum_row, tile * 16 + sum_column, v, tag);
                           });
            lds_barrier();
            fetch_tiles(pointer(&StackLayer::w_qkv, min(layer + 1, a.n_layers - 1)), qkv_tiles, g);
        }
        // The norm behind the last layer, a block a row: one handing-on more (some 2 us) for a kernel less. Passes of GPT-2
        // small, against the start in turn, ms: eight sequences and 48 tokens each in bfloat16 13.31 -> 13.15, in 32-bit and 32 tokens 18.09 -> 18.01, one and 16 3.27 -> 3.26.
        if (a.normed_out && g < M) {
            ask_norm(a.final_gain, a.final_offset);
            norm_rows(rows_words, false, first_tag + (uint32_t)a.n_layers, a.eps_final);
            lds_barrier();
#pragma unroll 1
            for (int row = g; row < M; row += norming)
                for (int piece = tid; piece < width / VEC; piece += ST_THREADS)
                    reinterpret_cast<Vec16*>(reinterpret_cast<T*>(a.normed_out) + (size_t)row * width)[piece] = reinterpret_cast<const Vec16*>(normed + row * stride)[piece];
        }
    }
    // the block that leaves last makes the control words ready for the next launch, which begins behind this one's end
    __syncthreads();
    if (tid == 0) {
        if (shared_gave_up) __hip_atomic_store(*reinterpret_cast<int* const*>(a.control + GAVE_UP), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        const int left = __hip_atomic_fetch_add(a.control + LEFT, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (left == (int)gridDim.x - 1) {
            __hip_atomic_store(a.control + ARRIVED, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            a.control[TOOK_PART] = members;
            __hip_atomic_store(a.control + MEMBERS, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(a.control + LEFT, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(a.control + EPOCH, shared_epoch + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

}  // namespace

// How many steps of K a wave has of a product over the width (0: no kernel for these sizes).
static int stack_steps(int rows, int width, int inner, int n_heads, int element_size) {
    const int kc = 64 / element_size;
    if (rows < 1 || rows > ST_MAX_ROWS || width < 64 || width % 64 || n_heads * ST_HEAD != width || inner < 32 || inner % 32) return 0;
    const int steps = ceil_div(width / kc, ST_WAVES), long_steps = ceil_div(inner / kc, ST_WAVES);
    for (int built : {3, 4, 6, 7, 8}) {
        if ((element_size == 2) == (built == 6 || built == 8)) continue;   // (those two in 32-bit)
        if (steps <= built && long_steps <= 4 * built) return built;
    }
    return 0;
}

// Whether one kernel runs all layers of such a model for so many rows.
MLLM_API int mllm_decode_stack_supported(int rows, int n_layers, int width, int inner, int n_heads, int head_size, int page_size, int dtype) {
    if (n_layers < 1 || n_layers > ST_MAX_LAYERS || head_size != ST_HEAD || page_size < 1 || (page_size & (page_size - 1))) return 0;
    if (dtype != MLLM_F32 && dtype != MLLM_BF16) return 0;
    return stack_steps(rows, width, inner, n_heads, dtype == MLLM_BF16 ? 2 : 4) > 0;
}

// Whether a step of so many rows, none of whose sequences is longer than `reach`, is faster as one kernel than layer by layer, of models with many layers and hidden units four times
// the columns. Measured on whole steps of random GPT-2 models (layer by layer / one kernel, us; 24 layers at 1,024 columns in bfloat16, 12 else):
//   bfloat16,   768 columns: 1 row 297 / 168 at 500 keys, 327 / 185 at 1,000, 363 / 340 at 1,900; 8 rows 328 / 208, 398 / 281, 476 / 416; 16 rows 365 / 289, 429 / 430, 551 / 696
//   bfloat16, 1,024 columns: 1 row 752 / 359, 810 / 517, 816 / 766; 8 rows 761 / 447, 872 / 547, 989 / 823; 16 rows 843 / 614, 1,018 / 916, 1,260 / 1,432
//   bfloat16, 1,600 columns: 1 row 492 / 279, 520 / 289, 528 / 419; 2 rows 486 / 296, 515 / 309, 587 / 442; 4 rows 487 / 436, 521 / 455, 595 / 595; 8 rows 516 / 507, 580 / 652
//   32-bit,     768 columns: 1 row 442 / 267, 491 / 335, 490 / 462; 8 rows 483 / 318, 559 / 400, 635 / 544; 16 rows 545 / 452, 632 / 619, 821 / 874
//   32-bit,   1,024 columns: 1 row 475 / 329, 523 / 404, 532 / 540; 8 rows 531 / 411, 691 / 574, 739 / 654; 16 rows 621 / 598, 922 / 782, 1,017 / 1,032
// Many keys are what one block takes long for, and rows of 1,600 columns fill the blocks that norm with more tiles than they ask for ahead.
MLLM_API int mllm_decode_stack_pays(int rows, int reach, int width) {
    if (width <= 1024) return rows <= 8 ? reach <= 1792 : rows <= 16 && reach <= 1024;
    return rows <= 2 ? reach <= 1792 : rows <= 4 && reach <= 1024;
}

// The same for any model. Measured as above with 1, 2, 4 and 12 layers of 64 to 1,792 columns and inner / columns of 1.9 to 16, at 60, 1,000 and 1,780 keys, 1 to 16 rows; where nothing
// else is said at least as fast as one kernel (us, layer by layer / one kernel):
//   one layer: 768 columns 38 / 33 (1 row, 60 keys), 44 / 46 (8 rows, 1,000), 48 / 58 (16 rows, 1,000), 40 / 43 (1 row, 1,780): its start costs what a layer gains. Two: 62 / 44, 71 / 62, 71 / 70
//   more than 8 rows: few layers (16 rows, 1,000 keys in bfloat16: 128 columns, 2 layers 55 / 62, 4 layers 99 / 102, 12 of 64 columns 258 / 240; 768 columns, 2 layers 79 / 86, 4 142 / 153, 12
//     429 / 430) and many hidden units (60 keys: 512 columns and 7,168 units 372 / 454, 1,024 and 5,632 404 / 520; in 32-bit 256 and 4,096 345 / 387). What is
//     left is behind at the last of its keys alone (640 columns 289 / 247 at 60 keys, 404 / 425 at 1,000)
//   more than 2 rows of more than 1,024 columns: 1,600, 4 rows of 60 and of 1,000 keys, 2 layers 87 / 90 and 94 / 96, 4 layers 154 / 153 and 185 / 171
//   32-bit beyond 1,024 keys (1,780): few layers (1,024 columns, 1 row, 2 layers 89 / 93, 4 174 / 184, 12 518 / 512), few columns (192, 8 rows 416 / 447; 384, 4 rows 426 / 451; 512, 2 rows
//     430 / 435; 640, 2 rows 488 / 452) and many hidden units (512 and 4,096, 1 row 443 / 485; 768 and 4,096 502 / 503)
MLLM_API int mllm_decode_stack_pays_for(int rows, int reach, int n_layers, int width, int inner, int dtype) {
    if (!mllm_decode_stack_pays(rows, reach, width) || n_layers < 2) return 0;
    if (rows > 8 && (n_layers < 8 || inner > 4 * width)) return 0;
    if (rows > 2 && width > 1024 && n_layers < 4) return 0;
    return dtype != MLLM_F32 || reach <= 1024 || (n_layers >= 8 && width >= 640 && inner <= 4 * width);
}

MLLM_API long long mllm_decode_stack_word_bytes(int rows, int width, int inner, int dtype) {
    const long long row = (long long)rows * width * 8, per = dtype == MLLM_BF16 ? 2 : 1;
    return FIRST_REGION + 2 * row + 4 * row / per + (long long)rows * inner * 8 / per;
}
MLLM_API int mllm_decode_stack_control_ints() { return CONTROL_INTS; }
MLLM_API int mllm_decode_stack_patience_at() { return PATIENCE; }   // where among the control words the host leaves the patience, two ints on the address of the word that says of a wait given up, and again two on finds how many blocks took part
MLLM_API int mllm_decode_stack_layer_pointers() { return LAYER_POINTERS; }

MLLM_API int mllm_decode_stack(const void* layers, int n_layers, const float* rows_in, float* rows_out, const int* token_request, const int* positions,
                               const float* final_gain, const float* final_offset, float eps_final, void* normed_out,
                               const int* slots, const int* block_tables, int max_blocks, void* words, int* control, int rows, int width, int inner,
                               int n_heads, int page_size, float eps_1, float eps_2, float scale, int activation, int dtype, int blocks, hipStream_t stream) {
    MLLM_REQUIRE(mllm_decode_stack_supported(rows, n_layers, width, inner, n_heads, ST_HEAD, page_size, dtype), "decode_stack: no kernel for %d rows of %d, %d hidden units, %d heads",
                 rows, width, inner, n_heads);
    MLLM_REQUIRE(activation == MLLM_EPI_GELU_TANH || activation == MLLM_EPI_GELU_ERF, "decode_stack: unknown activation %d", activation);
    MLLM_REQUIRE((rows_out != nullptr) != (normed_out != nullptr) && (!normed_out || (final_gain && final_offset)), "decode_stack: rows go out as they are or normed");
    MLLM_REQUIRE(max_blocks > 0 && blocks >= ST_MIN_MEMBERS, "decode_stack: bad table or grid");
    int page_shift = 0;
    while ((1 << page_shift) < page_size) page_shift++;
    // as few pairs a block as leave half of the blocks to the products
    int pairs_a_block = 1;
    while (pairs_a_block < ST_MAX_PAIRS && ceil_div(rows * n_heads, pairs_a_block) > blocks / 2) pairs_a_block *= 2;
    StackArgs a{(const StackLayer*)layers, rows_in, rows_out, final_gain, final_offset, normed_out, token_request, positions, slots, block_tables, (char*)words, control,
                n_layers, rows, width, inner, n_heads, max_blocks, page_shift, pairs_a_block, activation, eps_1, eps_2, eps_final, scale};
    const int element = dtype == MLLM_BF16 ? 2 : 4, steps = stack_steps(rows, width, inner, n_heads, element);
    const size_t normed = (size_t)rows * normed_stride(width, element) * element, attend = ST_WAVES * ((ST_HEAD + 4) * 4 + 2 * ST_HEAD * element);
#define MLLM_STACK_LAUNCH(T, STEPS, TILES, ROWS)                                                                                     \
    case ROWS: {                                                                                                                     \
        auto kernel = decode_stack_kernel<T, STEPS, TILES, ROWS>;                                                                    \
        size_t lds = (normed + 15) / 16 * 16 + 2 * TILES * sizeof(PartRows);                                                         \
        if (lds < attend) lds = attend;                                                                                              \
        if (lds < 84 * 1024) lds = 84 * 1024; /* a compute unit takes one block: all of them find a place at once */                 \
        hipError_t status = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);          \
        MLLM_REQUIRE(status == hipSuccess, "decode_stack: %s", hipGetErrorString(status));                                           \
        kernel<<<blocks, ST_THREADS, lds, stream>>>(a);                                                                              \
        break;                                                                                                                       \
    }
#define MLLM_STACK_ROWS(T, STEPS, TILES)                                                                                             \
    switch (padded) {                                                                                                                \
        MLLM_STACK_LAUNCH(T, STEPS, TILES, 1)                                                                                        \
        MLLM_STACK_LAUNCH(T, STEPS, TILES, 2)                                                                                        \
        MLLM_STACK_LAUNCH(T, STEPS, TILES, 4)                                                                                        \
        MLLM_STACK_LAUNCH(T, STEPS, TILES, 8)                                                                                        \
        MLLM_STACK_LAUNCH(T, STEPS, TILES, 16)                                                                                       \
    }
    int padded = 1;
    while (padded < rows) padded *= 2;
    mllm_count_kernel(MLLM_K_DECODE_STACK);
    if (steps == 3) { MLLM_STACK_ROWS(bf16_t, 3, 2) }
    else if (steps == 4) { MLLM_STACK_ROWS(bf16_t, 4, 4) }
    else if (steps == 7) { MLLM_STACK_ROWS(bf16_t, 7, 4) }
    else if (steps == 6) { MLLM_STACK_ROWS(float, 6, 2) }
    else { MLLM_STACK_ROWS(float, 8, 3) }
#undef MLLM_STACK_ROWS
#undef MLLM_STACK_LAUNCH
    return mllm_check_launch("decode_stack");
}

