"""The bounds of the 32-bit kernels in bfloat16 pieces tell the six products of pieces from fewer of them, and their second way (numbers that have no pieces) from
none: on what the pieces alone give, in 64 bits."""

import plain_pieces as P
import pytest
import torch


def _prompt(rows, head_size, seed):
    generator = torch.Generator().manual_seed(seed)
    return *(torch.randn(rows, head_size, generator=generator) for _ in range(3)), torch.ones(rows, rows).tril().bool()


def _exact(q, keys, values, seen, scale):
    return (q.double() @ keys.double().T * scale).masked_fill(~seen, -torch.inf).softmax(1) @ values.double()


def _norm(got, ref):
    return float((got - ref).norm() / ref.norm())


@pytest.mark.parametrize("without", [None, *P.PAIRS])
@pytest.mark.parametrize("k", [160, 416, 3072])
def test_bound_of_products(without, k):
    generator = torch.Generator().manual_seed(k)
    x, w = torch.randn(70, k, generator=generator), torch.randn(90, k, generator=generator)
    error = _norm(P.product(x, w, [p for p in P.PAIRS if p != without]), x.double() @ w.double().T)
    assert error < P.NORM_BOUND / 5 if without is None else error > 2 * P.NORM_BOUND


@pytest.mark.parametrize("without", [None, *P.PAIRS])
@pytest.mark.parametrize("where", ["scores", "values"])
@pytest.mark.parametrize("head_size", [32, 64])
@pytest.mark.parametrize("rows", [65, 300, 1000])
def test_bound_of_attention(without, where, head_size, rows):
    q, keys, values, seen = _prompt(rows, head_size, rows)
    fewer = [p for p in P.PAIRS if p != without]
    pairs = dict(score_pairs=fewer) if where == "scores" else dict(value_pairs=fewer)
    error = _norm(P.attention(q, keys, values, seen, head_size**-0.5, **pairs), _exact(q, keys, values, seen, head_size**-0.5))
    assert error < P.NORM_BOUND / 2 if without is None else error > 2 * P.NORM_BOUND


@pytest.mark.parametrize("head_size", [32, 64])
@pytest.mark.parametrize("what", ["tiny values", "tiny queries", "large queries"])
def test_numbers_without_pieces_are_wrong_by_more_than_is_allowed(what, head_size):
    q, keys, values, seen = _prompt(140, head_size, 5)
    scaled = dict(q=1.0, keys=1.0, values=1.0) | P.ODD[what]
    q, keys, values = q * scaled["q"], keys * scaled["keys"], values * scaled["values"]
    error = _norm(P.attention(q, keys, values, seen, head_size**-0.5) / scaled["values"], _exact(q, keys, values, seen, head_size**-0.5) / scaled["values"])
    assert error > 4 * P.ODD_BOUND
