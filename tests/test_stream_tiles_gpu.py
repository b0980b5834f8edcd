"""bfloat16 products of many rows at the edges of the tiles that their sizes choose, and of the places their blocks take."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# 128 x 64 in one round of blocks and in several, 128 x 128, 128 x 192, 192 x 128, 256 x 128 and 256 x 256, each a row or a piece of columns short of whole tiles or
# beyond them; eight shares of the tiles with a remainder, one tile alone, strips of which the last is lower
@pytest.mark.parametrize("m,n,k", [(65, 8, 64), (129, 72, 64), (300, 3080, 768), (2047, 776, 768), (3000, 776, 1600), (528, 4088, 256), (1500, 2296, 768), (4000, 3064, 128),
                                   (2049, 3072, 192), (1489, 3064, 768), (2111, 2312, 128), (2040, 4088, 256), (2040, 6392, 128)])
@pytest.mark.parametrize("cuts", [1, 3])
def test_tiles_of_the_streaming_product(m, n, k, cuts):
    from mini_llm_amd.ops import kernels as K

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
