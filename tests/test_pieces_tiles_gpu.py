"""32-bit products of many rows in bfloat16 pieces, at the edges of the tiles that their sizes choose."""

import pytest
import torch

pytestmark = pytest.mark.gpu

# (rows, columns, K, the tile: 1,000 x its rows and its columns): a row or four columns beyond whole tiles or short of them, even and odd counts of tiles along K
SHAPES = [(129, 100, 160, 64064), (66, 68, 256, 64064), (1281, 772, 384, 128064), (4100, 196, 416, 128064), (897, 2180, 384, 128096), (1400, 2180, 256, 128096),
          (641, 3076, 416, 128096), (3000, 2052, 256, 128128), (2690, 2308, 288, 128128)]


@pytest.mark.parametrize("m,n,k,tile", SHAPES)
def test_tiles_of_the_product_in_pieces(m, n, k, tile):
    from mini_llm_amd.ops import kernels as K
    from mini_llm_amd.ops.library import library

    assert library().mllm_gemm_pieces_tile(m, n, k, 1) == tile   # else the shape no longer tests what it is here for
    generator = torch.Generator(device="cuda").manual_seed(m + n)
    x, w, b, r = (torch.randn(*size, generator=generator, device="cuda") for size in ((m, k), (n, k), (n,), (m, n)))
    packed = K.pack_matrix(w)
    # a matrix instruction may leave a sum a unit in its last place off, six for sixteen numbers of K, and the pieces' products that are left out are 2^-24 of a product
    bound = 2**-23 * (6 * k / 16 + 4) * (x.abs().double() @ w.abs().double().T + b.abs().double() + r.abs().double())
    ref = x.double() @ w.double().T
    assert bool(((K.linear(x, packed, b, residual=r).double() - (ref + b.double() + r.double())).abs() <= bound).all())
    for cuts in (2, k // 32, k // 32 + 1):   # several, one and (behind the last part) no tiles of K a block
        assert bool(((K.linear_split(x, packed, cuts).double().sum(0) - ref).abs() <= bound).all())
    # a row with an infinity is taken again with the 32-bit instruction, in every tile of columns; the others know nothing of it
    for row in (0, m // 2, m - 1):
        x[row, (7 * row) % k] = torch.inf
    got, ref = K.linear(x, packed), (x.double() @ w.double().T)
    infinite = ~ref.isfinite()
    assert bool((got.double()[infinite] == ref[infinite]).all()) and int(infinite.sum()) == 3 * n
    assert bool(((got.double() - ref).abs() <= bound)[~infinite].all())
