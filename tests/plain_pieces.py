"""What 32-bit products come out as when every number is a sum of bfloat16 pieces, in 64 bits: all six products of pieces, or some left out (what the bounds of the
kernels' tests must not let pass)."""

import torch

# the products of pieces that count (the first operand's, the second's): what is left out of them is at most 2^-24 of a product
PAIRS = [(2, 0), (0, 2), (1, 1), (1, 0), (0, 1), (0, 0)]

# The error against 64 bits that the kernels' tests allow, in the norm, of sums of up to a thousand normally distributed numbers: the pieces' own is below 1e-7, rounded sums
# in 32-bit come to 1e-7 to 2.5e-7; with any of the six products left out it is 1.2e-6 or more.
NORM_BOUND = 5e-7

# Operands of attention whose pieces are lost (below 2^-110 the third, and so on), each with what makes up for it; and what the tests allow there, in the norm: 32-bit
# products and sums of up to 140 of them, one after another.
ODD = {"tiny values": dict(values=2.0**-124), "tiny queries": dict(q=2.0**-120, keys=2.0**120), "large queries": dict(q=2.0**120, keys=2.0**-120)}
ODD_BOUND = 2e-6


def pieces(x):
    """float32 -> three float64 tensors, each what the ones before leave, rounded to bfloat16."""
    rest, out = x.float(), []
    for _ in range(3):
        out.append(rest.bfloat16().float())
        rest = rest - out[-1]
    return [p.double() for p in out]


def product(x, w, pairs=PAIRS):
    """x @ w.T from the products of pieces named in ``pairs``."""
    xs, ws = pieces(x), pieces(w)
    return sum(xs[a] @ ws[b].T for a, b in pairs)


def attention(q, keys, values, seen, scale, score_pairs=PAIRS, value_pairs=PAIRS):
    """One head: float32 [rows, d], [keys, d], [keys, d], bool [rows, keys] -> float64 [rows, d]; scores and weights are rounded to 32-bit, weights below 2^-126 are 0."""
    scores = (product(q, keys, [(b, a) for a, b in score_pairs]) * scale).float().double().masked_fill(~seen, -torch.inf)
    weights = torch.exp(scores - scores.amax(1, keepdim=True)).float()
    weights = torch.where(weights < 2.0**-126, 0.0, weights)
    return product(weights, values.T.contiguous(), [(b, a) for a, b in value_pairs]) / weights.double().sum(1, keepdim=True)
