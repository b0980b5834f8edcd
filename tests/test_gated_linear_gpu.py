"""The product over gate and up rows in turn with its unit inside, silu(x gate^T) * (x up^T), against 64 bits: the kernels that have such an end at the edges of
their tiles, and what is left to the product and a kernel of its own."""

import numpy as np
import pytest
import torch

DEV = "cuda:0"
B, F = torch.bfloat16, torch.float32


def _sides(rng, rows, inner, width, dtype):
    stored = lambda a: torch.as_tensor(a, dtype=torch.float32).to(dtype)
    x, gate, up = (stored(rng.standard_normal(shape) * scale) for shape, scale in (((rows, width), 1.0), ((inner, width), 2.0 * width ** -0.5), ((inner, width), width ** -0.5)))
    return x, gate, up


def _exact(x, gate, up):
    x, gate, up = (t.double().numpy() for t in (x, gate, up))
    g, u = x @ gate.T, x @ up.T
    return g / (1.0 + np.exp(-g)) * u


@pytest.mark.parametrize("rows,inner,width,dtype,inside", [
    (1536, 14336, 4096, B, False), (4096, 4096, 8192, B, False), (16384, 11008, 4096, B, False),   # the plain product's tile of 256 x 256, over a long K
    (4096, 9472, 3584, B, True), (2048, 5632, 2048, B, True),                                     # over a shorter one
    (1024, 5632, 4096, B, True), (2048, 2048, 8192, B, True), (64, 2048, 8192, B, True),          # another tile, the kernel for few rows
    (1536, 14336, 4096, F, True)])
def test_where_the_unit_is_inside(rows, inner, width, dtype, inside):
    from mini_llm_amd.ops import kernels as K
    from mini_llm_amd.ops.library import library

    code, address, packed = (1, 256, 1) if dtype == B else (0, 256, K.PACKED_WITH_PIECES)
    assert bool(library().mllm_gemm_gated_takes(address, address, rows, 2 * inner, width, packed, code)) == inside


@pytest.mark.gpu
@pytest.mark.parametrize("rows,inner,width,inside", [
    (1, 8, 64, True), (1, 2048, 768, True), (8, 2048, 768, True), (16, 40, 96, True), (17, 1000, 64, True), (33, 2048, 768, True), (64, 2760, 320, True),
    (64, 4096, 64, False),                                                              # as many columns as a head has: the tiled kernel
    (65, 8, 64, True), (65, 56, 64, True), (130, 1000, 128, True), (300, 2048, 768, True), (528, 344, 1024, True), (2048, 2048, 768, True), (2100, 3200, 192, True),
    (1100, 72, 3136, True), (20000, 24, 64, True),
    (70, 64, 72, False),                                                                # rows that are no whole tiles of K
])
@pytest.mark.parametrize("dtype", [B, F])
def test_gate_and_up_rows_in_turn(rows, inner, width, inside, dtype):
    from mini_llm_amd.ops import kernels as K

    x, gate, up = _sides(np.random.default_rng(rows + inner), rows, inner, width, dtype)
    weight = K.pack_matrix(K.gate_up_rows(gate, up).contiguous().to(DEV))
    want = _exact(x, gate, up)
    before = K.launch_counts()
    out = K.gated_linear(x.to(DEV), weight)
    assert ("silu_mul" not in K.launches_since(before)) == inside
    # In 32-bit sums of up to 3,136 products, a product of two sums of order one; in bfloat16 one rounding (2^-9 of the value), or three where the unit is a kernel of its own.
    tolerance = dict(rtol=2e-5, atol=2e-5) if dtype == F else dict(rtol=2.0 ** -8 if inside else 2.0 ** -6, atol=1e-3 if inside else 2e-2)
    np.testing.assert_allclose(out.float().cpu().numpy(), want, **tolerance)
    assert torch.equal(K.gated_linear(x.to(DEV), weight), out)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [8, 150])
def test_rows_that_have_no_pieces(rows):
    # an infinity makes its own row's units infinite or no numbers, as in 64 bits, and no other row's (in 32-bit many rows take their sums again without pieces)
    from mini_llm_amd.ops import kernels as K

    x, gate, up = _sides(np.random.default_rng(3), rows, 200, 96, F)
    x[5, 17], x[rows - 1, 3] = float("inf"), 3e38
    with np.errstate(all="ignore"):
        want = _exact(x, gate, up)
    out = K.gated_linear(x.to(DEV), K.pack_matrix(K.gate_up_rows(gate, up).contiguous().to(DEV))).cpu().numpy().astype(np.float64)
    plain = [r for r in range(rows) if r not in (5, rows - 1)]
    np.testing.assert_allclose(out[plain], want[plain], rtol=2e-5, atol=2e-5)
    # of sums that are infinite: an infinite gate of minus sign gives no number, else the product is infinite (or, of a gate that vanishes, what 32 bits make of it)
    assert np.array_equal(np.isnan(out[5]), np.isnan(want[5])) and np.array_equal(out[5][~np.isnan(out[5])], want[5][~np.isnan(want[5])])
    assert not np.isfinite(out[rows - 1]).all()   # the products of 3e38 leave 32 bits


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [B, F])
@pytest.mark.parametrize("inner,turn", [(40, 8), (36, 4), (21, 7), (24, 24)])
def test_silu_mul_of_columns_in_turn(dtype, inner, turn):
    from mini_llm_amd.ops import kernels as K

    both = torch.randn((5, 2 * inner), generator=torch.Generator().manual_seed(inner)).to(dtype)
    parts = both.reshape(5, -1, 2, turn).double()
    want = (torch.nn.functional.silu(parts[:, :, 0]) * parts[:, :, 1]).reshape(5, inner)
    got = K.silu_mul(both.to(DEV), turn=turn).cpu().double()
    torch.testing.assert_close(got, want, rtol=2.0 ** -8 if dtype == B else 1e-6, atol=1e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [B, F])
def test_rows_in_the_packed_layout(dtype):
    from mini_llm_amd.ops import kernels as K

    _, gate, up = _sides(np.random.default_rng(9), 1, 200, 96, dtype)
    weight = K.pack_matrix(K.gate_up_rows(gate, up).contiguous().to(DEV))
    stream, gain, offset = (torch.randn(shape, generator=torch.Generator().manual_seed(i)).to(DEV) for i, shape in enumerate(((20, 96), (96,), (96,))))
    plain, packed = (K.layernorm(stream, gain, offset, 1e-5, out_dtype=dtype, packed_out=packed) for packed in (False, True))
    assert isinstance(packed, K.PackedRows)
    out = K.gated_linear(packed, weight).float().cpu().numpy()
    tolerance = dict(rtol=2e-5, atol=2e-5) if dtype == F else dict(rtol=2.0 ** -6, atol=2e-2)   # (as above, the unit in a kernel of its own)
    np.testing.assert_allclose(out, _exact(plain.cpu(), gate, up), **tolerance)
