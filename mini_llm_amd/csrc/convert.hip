// Load-time work on weights: element type conversion with an optional transpose (GPT-2 stores its
// matrices [in, out]; the matrix kernels read [out, in]). The reference converts its fp16 weight
// copy with a kernel of this kind (engine/src/matvec.cu:190-195) and transposes the head on the
// host (engine/src/gpt2_gpu.cu:30-48).
#include "common.h"

namespace {

template <typename S, typename D>
__global__ void convert_kernel(const S* __restrict__ src, D* __restrict__ dst, int rows, int cols, int transpose) {
    // 32x32 tiles through LDS so that both the read and the write run along rows
    __shared__ float tile[32][33];
    int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
    for (int i = threadIdx.y; i < 32; i += blockDim.y) {
        int r = r0 + i, c = c0 + threadIdx.x;
        if (r < rows && c < cols) tile[i][threadIdx.x] = to_float(src[(size_t)r * cols + c]);
    }
    __syncthreads();
    if (!transpose) {
        for (int i = threadIdx.y; i < 32; i += blockDim.y) {
            int r = r0 + i, c = c0 + threadIdx.x;
            if (r < rows && c < cols) dst[(size_t)r * cols + c] = from_float<D>(tile[i][threadIdx.x]);
        }
    } else {
        for (int i = threadIdx.y; i < 32; i += blockDim.y) {
            int c = c0 + i, r = r0 + threadIdx.x;  // dst is [cols, rows]
            if (r < rows && c < cols) dst[(size_t)c * rows + r] = from_float<D>(tile[threadIdx.x][i]);
        }
    }
}

// dst: the matrix W [rows, cols] (src row-major, or stored [cols, rows] with `transpose`) in the
// packed layout of the matrix kernels (common.h, packed_offset): chunks of 16 rows x 64 bytes, a
// chunk's 64 pieces of 16 bytes in the order the lanes of a wave take them as MFMA operands. One
// wave a chunk; zeros beyond the matrix.
template <typename S, typename D>
__global__ __launch_bounds__(256) void pack_kernel(const S* __restrict__ src, D* __restrict__ dst, int rows, int cols, int transpose) {
    constexpr int VEC = 16 / sizeof(D);
    const int k_steps = ceil_div(cols, 4 * VEC);
    const size_t chunk = (size_t)blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
    if (chunk >= (size_t)ceil_div(rows, 16) * k_steps) return;
    const int lane = threadIdx.x % WAVE;
    const int row = (int)(chunk / k_steps) * 16 + lane % 16;
    const int col = (int)(chunk % k_steps) * 4 * VEC + (lane / 16) * VEC;
    D* at = dst + (chunk * WAVE + lane) * VEC;
#pragma unroll
    for (int i = 0; i < VEC; i++) {
        float value = 0.0f;
        if (row < rows && col + i < cols)
            value = to_float(transpose ? src[(size_t)(col + i) * rows + row] : src[(size_t)row * cols + col + i]);
        at[i] = from_float<D>(value);
    }
}

// The pieces of the packed 32-bit matrix in front of them (gemm_pieces.h): a wave 16 rows x 32 columns.
__global__ __launch_bounds__(256) void pack_pieces_kernel(const float* __restrict__ packed, unsigned char* __restrict__ pieces, int row_tiles, int cols) {
    const int k_steps = ceil_div(cols, 32);
    const size_t step = (size_t)blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
    if (step >= (size_t)row_tiles * k_steps) return;
    const int lane = threadIdx.x % WAVE, row_tile = (int)(step / k_steps), k_step = (int)(step % k_steps);
    bf16x8 out[3];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const int col = k_step * 32 + (lane / 16) * 8 + e;   // the bfloat16 chunk's place: row lane % 16, columns 8 (lane / 16) ..
        float rest = col < cols ? packed[packed_element<float>(row_tile * 16 + lane % 16, col, cols)] : 0.0f;
#pragma unroll
        for (int p = 0; p < 3; p++) {
            bf16_t piece = from_float<bf16_t>(rest);
            if (fabsf(to_float(piece)) == INFINITY && fabsf(rest) < INFINITY) {   // rounded beyond the largest: cut off instead
                const uint16_t upper = (uint16_t)(__builtin_bit_cast(uint32_t, rest) >> 16);
                piece = __builtin_bit_cast(bf16_t, upper);
            }
            out[p][e] = piece;
            rest -= to_float(piece);
        }
    }
#pragma unroll
    for (int p = 0; p < 3; p++) *reinterpret_cast<bf16x8*>(pieces + (step * 3 + p) * 1024 + lane * 16) = out[p];
}

// What the product in pieces asks of every sixteen rows of the packed 32-bit matrix: a wave each.
__global__ __launch_bounds__(64) void tile_rows_kernel(const float* __restrict__ packed, TileRows* __restrict__ out, int cols) {
    const int lane = threadIdx.x, k_steps = packed_k_steps<float>(cols);
    uint32_t bits = 0, largest = 0;   // of row lane % 16
    for (int step = 0; step < k_steps; step++) {
        const Vec16 piece = *reinterpret_cast<const Vec16*>(packed + packed_offset<float>(blockIdx.x, step, k_steps, lane));
#pragma unroll
        for (int e = 0; e < 4; e++) bits |= piece.w[e], largest = max(largest, piece.w[e] & 0x7fffffffu);
    }
    bits |= (uint32_t)__shfl_xor((int)bits, 16, WAVE);
    bits |= (uint32_t)__shfl_xor((int)bits, 32, WAVE);
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) largest = max(largest, (uint32_t)__shfl_xor((int)largest, offset, WAVE));
    const unsigned long long lanes = __ballot(tiny(bits));
    if (lane == 0) out[blockIdx.x] = TileRows{(int)(lanes & 0xffff), (int)largest};
}

template <typename S, typename D>
void launch_pack(const void* src, void* dst, int rows, int cols, int transpose, hipStream_t stream) {
    const size_t chunks = (size_t)ceil_div(rows, 16) * ceil_div(cols, 4 * (16 / (int)sizeof(D)));
    mllm_count_kernel(MLLM_K_PACK);
    pack_kernel<S, D><<<(unsigned)((chunks + 3) / 4), 256, 0, stream>>>((const S*)src, (D*)dst, rows, cols, transpose);
}

template <typename S, typename D>
void launch_convert(const void* src, void* dst, int rows, int cols, int transpose, hipStream_t stream) {
    dim3 grid(ceil_div(cols, 32), ceil_div(rows, 32)), block(32, 8);
    mllm_count_kernel(MLLM_K_CONVERT);
    convert_kernel<S, D><<<grid, block, 0, stream>>>((const S*)src, (D*)dst, rows, cols, transpose);
}

}  // namespace

// dst = src (rows x cols, row-major) in another element type; with transpose, dst is cols x rows.
MLLM_API int mllm_convert(const void* src, void* dst, int rows, int cols, int src_dtype, int dst_dtype,
                          int transpose, hipStream_t stream) {
    MLLM_REQUIRE(rows >= 0 && cols >= 0, "convert: negative size");
    MLLM_REQUIRE(ceil_div(rows, 32) <= 65535, "convert: too many rows for one launch");
    if (rows == 0 || cols == 0) return 0;
    if (src_dtype == MLLM_F32 && dst_dtype == MLLM_F32) launch_convert<float, float>(src, dst, rows, cols, transpose, stream);
    else if (src_dtype == MLLM_F32 && dst_dtype == MLLM_BF16) launch_convert<float, bf16_t>(src, dst, rows, cols, transpose, stream);
    else if (src_dtype == MLLM_BF16 && dst_dtype == MLLM_F32) launch_convert<bf16_t, float>(src, dst, rows, cols, transpose, stream);
    else if (src_dtype == MLLM_BF16 && dst_dtype == MLLM_BF16) launch_convert<bf16_t, bf16_t>(src, dst, rows, cols, transpose, stream);
    else MLLM_REQUIRE(false, "convert: unknown element types %d -> %d", src_dtype, dst_dtype);
    return mllm_check_launch("convert");
}

// Elements the packed form of a rows x cols matrix takes (rows padded to 16, cols to 64 bytes).
MLLM_API long long mllm_packed_elements(int rows, int cols, int dtype) {
    const int vec = dtype == MLLM_F32 ? 4 : 8;
    return (long long)ceil_div(rows, 16) * ceil_div(cols, 4 * vec) * 64 * vec;
}

// dst = the matrix [rows, cols] in the packed layout; src is row-major [rows, cols], or with
// `transpose` the stored [cols, rows].
MLLM_API int mllm_pack_matrix(const void* src, void* dst, int rows, int cols, int src_dtype, int dst_dtype,
                              int transpose, hipStream_t stream) {
    MLLM_REQUIRE(rows > 0 && cols > 0, "pack_matrix: bad size %d x %d", rows, cols);
    if (src_dtype == MLLM_F32 && dst_dtype == MLLM_F32) launch_pack<float, float>(src, dst, rows, cols, transpose, stream);
    else if (src_dtype == MLLM_F32 && dst_dtype == MLLM_BF16) launch_pack<float, bf16_t>(src, dst, rows, cols, transpose, stream);
    else if (src_dtype == MLLM_BF16 && dst_dtype == MLLM_F32) launch_pack<bf16_t, float>(src, dst, rows, cols, transpose, stream);
    else if (src_dtype == MLLM_BF16 && dst_dtype == MLLM_BF16) launch_pack<bf16_t, bf16_t>(src, dst, rows, cols, transpose, stream);
    else MLLM_REQUIRE(false, "pack_matrix: unknown element types %d -> %d", src_dtype, dst_dtype);
    return mllm_check_launch("pack_matrix");
}

// Bytes the pieces of a packed 32-bit matrix take behind it, with what is known of its rows; 0: no product would take them (pieces::takes_sizes).
MLLM_API long long mllm_pieces_bytes(int rows, int cols) {
    const int row_tiles = ceil_div(rows, 16);
    const long long bytes = packed_pieces_bytes(row_tiles, cols);
    return cols % 32 != 0 || rows % 4 != 0 || bytes >= (1LL << 32) ? 0 : bytes + (long long)sizeof(TileRows) * row_tiles;
}

// Lays the pieces of a packed 32-bit matrix [rows, cols] behind it, at packed + mllm_packed_elements.
MLLM_API int mllm_pack_pieces(float* packed, int rows, int cols, hipStream_t stream) {
    MLLM_REQUIRE(rows > 0 && cols > 0 && packed != nullptr, "pack_pieces: bad size %d x %d", rows, cols);
    MLLM_REQUIRE(mllm_pieces_bytes(rows, cols) > 0, "pack_pieces: no product takes pieces of a %d x %d matrix", rows, cols);
    const int row_tiles = ceil_div(rows, 16);
    unsigned char* pieces = reinterpret_cast<unsigned char*>(packed) + packed_pieces_at(row_tiles, packed_k_steps<float>(cols));
    const size_t steps = (size_t)row_tiles * ceil_div(cols, 32);
    mllm_count_kernel(MLLM_K_PACK);
    pack_pieces_kernel<<<(unsigned)((steps + 3) / 4), 256, 0, stream>>>(packed, pieces, row_tiles, cols);
    mllm_count_kernel(MLLM_K_PACK);
    tile_rows_kernel<<<row_tiles, 64, 0, stream>>>(packed, reinterpret_cast<TileRows*>(pieces + packed_pieces_bytes(row_tiles, cols)), cols);
    return mllm_check_launch("pack_pieces");
}
