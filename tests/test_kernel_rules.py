"""Rules by which host code chooses among kernels and launch shapes."""

import pytest


@pytest.mark.parametrize("rows,heads,keys,key_bytes,best", [
    # measured best within 2 % (bfloat16 heads of 64: 128 bytes a key; 32-bit: 256)
    (8, 12, 64, 128, {1}), (1, 12, 65, 128, {2}), (1, 12, 128, 128, {2}), (8, 12, 128, 128, {2}), (64, 12, 128, 128, {2}), (8, 12, 200, 128, {4, 8}),
    (8, 12, 300, 128, {8}), (8, 12, 500, 128, {8}), (1, 16, 500, 128, {8}), (16, 25, 500, 128, {4, 8}), (8, 12, 900, 128, {8}), (8, 12, 1500, 128, {8}), (8, 12, 3000, 128, {8, 16}),
    (8, 12, 900, 256, {16}), (8, 12, 500, 256, {8, 16}), (64, 12, 900, 256, {4, 8}), (8, 12, 4096, 32, {8, 16}),
    # a launch holds 4,096 waves at the most, except where single waves are more
    (400, 12, 3000, 128, {1}), (64, 25, 3000, 128, {2}), (1, 1, 1, 64, {1})])
def test_waves_of_the_decode_attention(rows, heads, keys, key_bytes, best):
    from mini_llm_amd.ops import kernels as K

    assert K.decode_waves(rows * heads, keys, key_bytes) in best


@pytest.mark.parametrize("runs,keys,key_bytes,best", [(2, 512, 128, {4, 8}), (8, 512, 128, {4}), (2, 750, 128, {8}), (4, 750, 128, {8}), (2, 512, 256, {8})])
def test_waves_of_the_decode_attention_of_one_row_in_runs(runs, keys, key_bytes, best):
    from mini_llm_amd.ops import kernels as K

    assert K.decode_waves(12 * runs, keys, key_bytes, cut=True) in best


@pytest.mark.parametrize("rows,width,partials,block", [
    # measured: which is faster, a block or a wave a row
    (8, 64, 5, 0), (256, 60, 1, 0), (64, 256, 1, 0), (64, 256, 0, 1), (257, 256, 0, 0), (8, 64, 0, 0), (8, 768, 0, 1), (64, 320, 1, 1), (256, 384, 9, 1), (512, 512, 4, 1), (768, 512, 9, 0), (2048, 512, 1, 0), (8192, 512, 8, 0),
    (2048, 576, 4, 1), (8, 768, 1, 1), (8192, 768, 16, 1), (32768, 768, 5, 0), (8192, 1024, 5, 1), (8192, 1024, 8, 0), (2048, 1024, 9, 1), (2048, 1024, 16, 0),
    (8192, 1600, 16, 1), (8192, 2048, 8, 1),
    # what the kernel does not take
    (8, 770, 1, 0), (8, 2052, 1, 0)])
def test_rms_norm_with_a_block_or_a_wave_a_row(rows, width, partials, block):
    from mini_llm_amd.ops.library import library

    assert library().mllm_rms_norm_block_a_row(rows, width, partials) == block


def test_every_tile_of_the_streaming_product_has_a_shape_in_its_test():
    from mini_llm_amd.ops.library import library
    from test_stream_tiles_gpu import SHAPES

    tile = library().mllm_gemm_stream_tile
    for m, n, k, tile_f32, tile_bf16, tile_cut in SHAPES:
        assert (tile(m, n, k, 1, 0), tile(m, n, k, 1, 1), tile(m, n, k, 3, 0)) == (tile_f32, tile_bf16, tile_cut)
    assert {shape[3] for shape in SHAPES} == {1281920, 1921280, 2561280, 1281280, 1280640, 1280641, 1280642}
    assert {shape[4] for shape in SHAPES} == {1281920, 1921280, 2561280, 1281280, 1280640, 1280641, 1280642, 2562560}
    assert tile(64, 768, 768, 1, 0) == tile(65, 770, 768, 1, 0) == tile(65, 768, 736, 1, 0) == 0   # other kernels'


@pytest.mark.parametrize("m,n,k,out,tile", [
    # a long K in one round of narrow tiles: shared where measured faster (see the kernel's rule)
    (65, 1024, 4096, 0, 1280641), (1500, 1024, 4096, 0, 1280641), (300, 2048, 8192, 1, 1280641), (2048, 1024, 4096, 0, 1280640), (65, 1600, 6400, 1, 1280641), (128, 1600, 6400, 0, 1280640),
    (2048, 768, 3072, 0, 1280640), (300, 768, 2048, 0, 1280640), (65, 768, 2048, 0, 1280640),
    # many rounds
    (16384, 1600, 6400, 0, 2561280), (65536, 64, 768, 0, 1280642)])
def test_tiles_of_the_streaming_product_by_measurement(m, n, k, out, tile):
    from mini_llm_amd.ops.library import library

    assert library().mllm_gemm_stream_tile(m, n, k, 1, out) == tile


@pytest.mark.parametrize("m,n,k,packed,row_major", [
    # counts within 3 % of the best measured, with the layer norm behind the product
    (100, 768, 3072, {6, 7, 8}, {6, 7, 8}), (400, 1024, 1024, {2, 3}, {2}), (400, 1280, 1280, {2}, {2, 3}), (528, 1280, 1280, {1, 2}, None), (528, 1280, 5120, {2}, None),
    (400, 1600, 1600, {2}, {2}), (528, 1600, 1600, {1, 2}, {2}), (400, 2048, 2048, {2}, {2}), (200, 1600, 1600, {3, 4}, None), (1200, 256, 1024, {2, 3}, None),
    (1000, 1600, 6400, None, {1, 2}), (257, 1280, 1280, None, {2}), (2048, 768, 3072, {1}, {1}), (2048, 1600, 1600, {1}, {1})])
def test_cuts_along_k_of_bfloat16_products_of_many_rows(m, n, k, packed, row_major):
    from mini_llm_amd.ops.library import library

    lib = library()
    assert packed is None or lib.mllm_gemm_split_blocks_anywhere(m, n, k, 1) in packed
    assert row_major is None or lib.mllm_gemm_split_blocks_row_major(m, n, k, 1) in row_major
    # the same for all counts of rows that need the same number of 128-row tiles, and never an answer of 0 or beyond 8
    for rows in (-(-m // 128) * 128, (m - 1) // 128 * 128 + 1):
        assert rows <= 64 or lib.mllm_gemm_split_blocks_anywhere(rows, n, k, 1) == lib.mllm_gemm_split_blocks_anywhere(m, n, k, 1)
        assert rows <= 64 or lib.mllm_gemm_split_blocks_row_major(rows, n, k, 1) == lib.mllm_gemm_split_blocks_row_major(m, n, k, 1)


@pytest.mark.parametrize("rows,heads,requests,max_q_len,longest,by_matrix", [
    (255, 12, 1, 255, 255, False), (256, 12, 1, 256, 256, True), (1024, 12, 1, 1024, 1024, True), (2000, 12, 100, 20, 20, False), (256, 12, 256, 1, 60, False),
    (256, 12, 256, 1, 100, True), (512, 12, 64, 8, 100, True), (2100, 12, 101, 100, 100, False), (1154, 12, 30, 70, 70, False), (2600, 12, 101, 600, 600, True),
    (324, 12, 77, 20, 600, True), (960, 12, 16, 128, 128, True)])
def test_32_bit_latent_attention_by_matrix_instructions(rows, heads, requests, max_q_len, longest, by_matrix):
    from mini_llm_amd.ops import kernels as K

    assert K.latent_f32_by_matrix(rows, heads, requests, max_q_len, longest) == by_matrix


@pytest.mark.parametrize("m,n,k,cuts,tile", [
    # the best tile as measured, or within 3 % of it; and what another kernel takes
    (2048, 2304, 768, 1, 128096), (2670, 2304, 768, 1, 128096), (2048, 768, 3072, 2, 128096), (2670, 768, 3072, 2, 128128), (2048, 4096, 768, 1, 128128), (130, 768, 768, 6, 64064),
    (300, 768, 3072, 8, 64064), (1024, 768, 3072, 2, 128064), (64, 768, 768, 1, 0), (65, 768, 760, 1, 0), (65, 770, 768, 1, 0)])
def test_tiles_of_the_product_in_pieces_by_measurement(m, n, k, cuts, tile):
    from mini_llm_amd.ops.library import library

    assert library().mllm_gemm_pieces_tile(m, n, k, cuts) == tile


def test_every_tile_of_the_product_in_pieces_has_a_shape_in_its_test():
    from test_pieces_tiles_gpu import SHAPES

    assert {shape[3] for shape in SHAPES} == {64064, 128064, 128096, 128128}


def test_every_tile_of_the_product_in_pieces_is_compared_with_the_32_bit_instruction():
    from mini_llm_amd.ops.library import library
    from test_kernels_gpu import NEARER_SHAPES

    assert {library().mllm_gemm_pieces_tile(*shape, 1) for shape in NEARER_SHAPES} == {64064, 128064, 128096, 128128}
