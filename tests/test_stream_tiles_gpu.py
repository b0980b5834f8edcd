"""bfloat16 products of many rows at the edges of the tiles that their sizes choose, and of the places their blocks take."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# (rows, columns, K; the tile of the whole product with 32-bit and with bfloat16 out, and of one cut in three: 10,000 x rows + 10 x columns, and of 128 x 64 its
# kernel: 0, 1 two waves that share a tile along K, 2 two blocks a compute unit). Every tile, a row or a piece of columns short of whole ones or beyond them, with an odd
# count of tiles along K among them; eight shares of the tiles with a remainder, one tile alone, strips of which the last is lower, shares of several rounds.
SHAPES = [(65, 8, 64, 1280640, 1280640, 1280640), (129, 72, 64, 1280640, 1280640, 1280640), (300, 3080, 768, 1280640, 1280640, 1281280),
          (2047, 776, 768, 1280640, 1280640, 1921280), (3000, 776, 1600, 1281280, 1281280, 2561280), (528, 4088, 256, 1281280, 1281280, 1281280),
          (1500, 2296, 768, 1281280, 1281280, 1921280), (4000, 3064, 128, 2561280, 2562560, 2561280), (2049, 3072, 192, 2561280, 2561280, 2561280),
          (1489, 3064, 768, 1921280, 1921280, 2561280), (2111, 2312, 128, 2561280, 2561280, 2561280), (2040, 4088, 256, 2561280, 2561280, 2561280),
          (2040, 6392, 128, 2561280, 2562560, 2561280), (2048, 3072, 768, 1281920, 1281920, 2561280), (1925, 3064, 768, 1281920, 1281920, 2561280),
          (65, 136, 3136, 1280641, 1280641, 1280640), (96, 72, 3072, 1280641, 1280641, 1280640), (97, 72, 3072, 1280640, 1280640, 1280640),
          (300, 72, 4096, 1280641, 1280641, 1280640), (150, 72, 12288, 1280641, 1280641, 1280641), (65500, 40, 256, 1280642, 1280642, 2561280),
          (9000, 2312, 128, 2561280, 2561280, 2561280)]


@pytest.mark.parametrize("m,n,k,tile_f32,tile_bf16,tile_cut", SHAPES)
@pytest.mark.parametrize("cuts", [1, 3])
def test_tiles_of_the_streaming_product(m, n, k, tile_f32, tile_bf16, tile_cut, cuts):
    from mini_llm_amd.ops import kernels as K
    from mini_llm_amd.ops.library import library

    tile = library().mllm_gemm_stream_tile
    assert (tile(m, n, k, 1, 0), tile(m, n, k, 1, 1), tile(m, n, k, 3, 0)) == (tile_f32, tile_bf16, tile_cut)   # else the shape no longer tests what it is here for
    generator = torch.Generator(device="cuda").manual_seed(m + n)
    x, w = (torch.randn(rows, k, generator=generator, device="cuda").bfloat16() for rows in (m, n))
    bias, residual = torch.randn(n, generator=generator, device="cuda"), torch.randn(m, n, generator=generator, device="cuda")
    want = x.double() @ w.double().T
    size = (x.double().abs() @ w.double().abs().T).max()   # of a sum's terms: each of k / 16 roundings is 2^-24 of a partial sum, which is less
    bound = float(size) * 2.0 ** -24 * (k / 16 + cuts + 2)
    packed = K.pack_matrix(w)
    if cuts > 1:
        parts = K.linear_split(x, packed, cuts)
        assert parts.shape[0] == cuts and (parts.double().sum(0) - want).abs().max() <= bound
        return
    assert (K.linear(x, packed, out_dtype=torch.float32).double() - want).abs().max() <= bound
    assert (K.linear(x, packed, bias, residual=residual).double() - (want + bias + residual)).abs().max() <= bound + 2.0 ** -22 * 8
    rounded = K.linear(x, packed, bias).double()
    assert ((rounded - (want + bias)).abs() <= (want + bias).abs() * 2.0 ** -8 + bound).all()
