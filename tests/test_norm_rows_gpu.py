"""Norms with a block a row: widths at the edges of their threads, partial products beyond those asked for at once, every option."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,width", [(1, 4), (3, 60), (9, 132), (64, 256), (257, 512), (5, 1024), (300, 1028), (2, 2048), (9, 2052), (7, 770)])
@pytest.mark.parametrize("partials", [0, 1, 2, 4, 5, 9])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_norm_of_a_row_by_a_block(rows, width, partials, out_dtype):
    from mini_llm_amd.ops import kernels as K

    generator = torch.Generator(device="cuda").manual_seed(rows * width + partials)
    draw = lambda *shape: torch.randn(*shape, generator=generator, device="cuda")
    x, weight, residual, following = draw(rows, width), draw(width), draw(rows, width), draw(width)
    addend = draw(partials, rows, width) if partials else None
    if partials == 1:
        addend = addend[0].to(out_dtype)
    eps, alpha = 1e-5, 0.7
    h = x.double() * alpha + (0 if addend is None else addend.double().reshape(-1, rows, width).sum(0))
    norm = lambda v, g: v / (v.pow(2).mean(1, keepdim=True) + eps).sqrt() * (1.0 + g.double())
    want = residual.double() + norm(h, weight)
    # 32-bit sums of up to 11 addends and of 2,052 squares, a square root and a division: some 2^-23 times twenty of numbers around 10
    close = lambda got, ref: (got.double() - ref).abs().max() <= 2e-5 + (ref.abs().max() * 2.0 ** -8 if got.dtype == torch.bfloat16 else 0)
    assert close(K.rms_norm(x, weight, eps, addend=addend, alpha=alpha, one_plus=True, residual=residual), want)
    stream, normed = K.rms_norm(x, weight, eps, addend=addend, alpha=alpha, one_plus=True, residual=residual, with_stream=True, out_dtype=out_dtype)
    assert close(stream, want) and close(normed, want)
    if width <= 2048:
        stream, twice = K.rms_norm(x, weight, eps, addend=addend, alpha=alpha, one_plus=True, residual=residual, with_stream=True, out_dtype=out_dtype, next_weight=following)
        assert close(stream, want) and close(twice, norm(want, following))
    index = torch.randint(rows, (rows + 2,), generator=generator, device="cuda").int()
    assert close(K.rms_norm(x, weight, eps, one_plus=True, row_index=index, out_dtype=out_dtype), norm(x.double(), weight)[index.long()])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,n,k,cut", [(1, 768, 1535, (False, False)), (8, 768, 1536, (True, False)), (16, 1024, 2048, (True, True)), (3, 1040, 2048, (True, False)), (5, 1040, 3072, (True, True))])
def test_branch_products_of_few_rows_are_cut_from_a_long_k_on(dtype, rows, n, k, cut):
    from mini_llm_amd.ops import kernels as K
    from mini_llm_amd.parts.linear import BranchProduct

    generator = torch.Generator(device="cuda").manual_seed(rows + k)
    k = k // 8 * 8   # (whole 16-byte pieces)
    x, w = torch.randn(rows, k, generator=generator, device="cuda").to(dtype), (torch.randn(n, k, generator=generator, device="cuda") / k ** 0.5).to(dtype)
    weight, residual = torch.randn(n, generator=generator, device="cuda"), torch.randn(rows, n, generator=generator, device="cuda")
    branch = BranchProduct()(x, K.pack_matrix(w))
    assert (branch.dim() == 3) == cut[dtype == torch.bfloat16]
    h = x.double() @ w.double().T
    want = residual.double() + h / (h.pow(2).mean(1, keepdim=True) + 1e-5).sqrt() * weight.double()
    first, rest = (branch[0], branch[1:]) if branch.dim() == 3 else (branch, None)
    # sums of k products of numbers around 1 / sqrt(k), each rounding 2^-24 of a partial sum of at most some 5, sixteen terms at a time
    assert (K.rms_norm(first, weight, 1e-5, addend=rest, residual=residual).double() - want).abs().max() <= 5 * 4 * 2.0 ** -24 * (k / 16) ** 0.5 * 4


# waves without a column, rows of 4,096 (a piece of four columns a thread of the largest block) and of more (several), groups of threads that share a row's sums
@pytest.mark.parametrize("rows,width,partials", [(3, 4, 1), (2, 4, 16), (300, 60, 9), (64, 64, 17), (9, 260, 20), (2, 1024, 16), (65, 1024, 16), (300, 1028, 8), (3, 2052, 5), (3, 4096, 9), (3, 4100, 9),
                                                 (2, 8200, 17), (5, 4100, 0)])
@pytest.mark.parametrize("with_bias", [False, True])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_layer_norm_of_pending_rows_at_the_borders_of_its_threads(rows, width, partials, with_bias, out_dtype):
    from mini_llm_amd.ops import kernels as K

    generator = torch.Generator(device="cuda").manual_seed(rows * width + partials)
    draw = lambda *shape: torch.randn(*shape, generator=generator, device="cuda")
    base, parts, bias, gain, offset = draw(rows, width), draw(partials, rows, width), draw(width), draw(width), draw(width)
    pending = K.PendingRows(base, parts if partials else None, bias if with_bias else None)
    total = base.double() + parts.double().sum(0) + (bias.double() if with_bias else 0)
    want = torch.nn.functional.layer_norm(total, (width,), gain.double(), offset.double(), 1e-5)
    # 32-bit sums of up to 19 addends and of 8,200 numbers, a square root and a division: some 2^-23 times twenty of numbers around 10
    close = lambda got, ref: (got.double() - ref).abs().max() <= 2e-5 + (ref.abs().max() * 2.0 ** -8 if got.dtype == torch.bfloat16 else 0)
    normed, summed = K.layernorm(pending, gain, offset, 1e-5, out_dtype=out_dtype, with_sums=True)
    assert close(normed, want) and close(summed, total)
    index = torch.randint(rows, (rows + 2,), generator=generator, device="cuda").int()
    assert close(K.layernorm(pending, gain, offset, 1e-5, out_dtype=out_dtype, row_index=index), want[index.long()])
