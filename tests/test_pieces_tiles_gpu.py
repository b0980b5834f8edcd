"""32-bit products of many rows and 32-bit prompt attention in bfloat16 pieces: at the edges of their tiles, in each of their forms, and with numbers that have no pieces.
That the bounds here tell the six products of pieces from fewer: test_pieces_bounds.py."""

import plain_pieces
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
    assert _norm(K.linear(x, packed), ref) < plain_pieces.NORM_BOUND
    for cuts in (2, k // 32, k // 32 + 1):   # several, one and (behind the last part) no tiles of K a block
        parts = K.linear_split(x, packed, cuts).double().sum(0)
        assert bool(((parts - ref).abs() <= bound).all()) and _norm(parts, ref) < plain_pieces.NORM_BOUND
    # a row with an infinity is taken again with the 32-bit instruction, in every tile of columns; the others know nothing of it
    for row in (0, m // 2, m - 1):
        x[row, (7 * row) % k] = torch.inf
    got, ref = K.linear(x, packed), (x.double() @ w.double().T)
    infinite = ~ref.isfinite()
    assert bool((got.double()[infinite] == ref[infinite]).all()) and int(infinite.sum()) == 3 * n
    assert bool(((got.double() - ref).abs() <= bound)[~infinite].all())


def _norm(got, ref):
    return float((got.double() - ref).norm() / ref.norm())


@pytest.mark.parametrize("m,n,k,tile", [(897, 2304, 384, 128096), (2690, 2304, 288, 128128), (1400, 768, 384, 128064)])
def test_what_tiles_of_128_rows_leave(m, n, k, tile):
    """Activations; q/k/v columns into pages (with 96 columns a wave, sixteen of its lanes store nothing) with rows that have no place there; rows of x and of W that are tiny throughout."""
    from mini_llm_amd.ops import kernels as K
    from mini_llm_amd.ops.library import library

    assert library().mllm_gemm_pieces_tile(m, n, k, 1) == tile
    generator = torch.Generator(device="cuda").manual_seed(m)
    x, w, b = (torch.randn(*size, generator=generator, device="cuda") for size in ((m, k), (n, k), (n,)))
    w *= k**-0.5
    packed, ref = K.pack_matrix(w), x.double() @ w.double().T + b.double()
    # (an activation's own error: some 2^-22 of numbers up to about 20)
    gelu_new = lambda y: 0.5 * y * (1 + torch.tanh(0.7978845608028654 * (y + 0.044715 * y**3)))
    for activation, of in (("gelu_new", gelu_new), ("gelu", lambda y: 0.5 * y * (1 + torch.erf(y * 0.5**0.5))), ("squared_relu", lambda y: y.clamp(min=0) ** 2)):
        got, want = K.linear(x, packed, b, activation), of(ref)
        assert _norm(got, want) < 1e-6 and float((got.double() - want).abs().max()) < 2e-5
    heads, size, page = n // 192, 64, 32
    slots = torch.randperm((m // page + 2) * page, generator=generator, device="cuda")[:m].int()
    slots[1::50] = -1
    k_pages, v_pages = (torch.full((m // page + 2, heads, page, size), 7.0, device="cuda") for _ in range(2))
    q = K.linear_qkv_cache(x, packed, b, k_pages, v_pages, slots, heads, heads, size)
    stored = slots >= 0
    for got, want in ((q, ref[:, : n // 3]), *((pages[slots.long() // page, :, slots.long() % page].reshape(m, -1)[stored], ref[stored, at : at + n // 3])
                                               for pages, at in ((k_pages, n // 3), (v_pages, n * 2 // 3)))):
        assert _norm(got, want) < plain_pieces.NORM_BOUND
    for pages in (k_pages, v_pages):   # places that no row has are as they were
        free = torch.ones(pages.shape[0] * page, dtype=torch.bool, device="cuda")
        free[slots[stored].long()] = False
        assert bool((pages.transpose(1, 2).reshape(-1, heads * size)[free] == 7.0).all())
    x[::7] *= 2.0**-124
    w[5::16] *= 2.0**-122
    packed, ref = K.pack_matrix(w), x.double() @ w.double().T
    got = K.linear(x, packed).double()
    bound = 2**-23 * (6 * k / 16 + 4) * (x.abs().double() @ w.abs().double().T) + k * 2.0**-149
    assert bool(((got - ref).abs() <= bound).all())
    tiny = torch.arange(m, device="cuda") % 7 == 0
    plain = torch.arange(n, device="cuda") % 16 != 5
    assert _norm(got[tiny][:, plain] * 2.0**124, ref[tiny][:, plain] * 2.0**124) < 1e-6 and _norm(got[~tiny][:, ~plain] * 2.0**122, ref[~tiny][:, ~plain] * 2.0**122) < 1e-6


def _prompt(lengths, contexts, heads, head_size, kv_heads=None, page_size=32):
    """Queries, pages and the batch's arrays of prompts on cached keys: (q, k_pages, v_pages, requests, positions, tables, starts, contexts), float32."""
    generator = torch.Generator(device="cuda").manual_seed(sum(lengths) + head_size)
    pages = [-(-(n + c) // page_size) for n, c in zip(lengths, contexts)]
    tables = torch.zeros(len(lengths), max(pages), dtype=torch.int32)
    for r, count in enumerate(pages):
        tables[r, :count] = torch.arange(sum(pages[:r]), sum(pages[:r]) + count).flip(0)
    k_pages, v_pages = (torch.randn(sum(pages), kv_heads or heads, page_size, head_size, generator=generator, device="cuda") for _ in range(2))
    q = torch.randn(sum(lengths), heads * head_size, generator=generator, device="cuda")
    requests = torch.cat([torch.full((n,), r) for r, n in enumerate(lengths)]).int().cuda()
    positions = torch.cat([torch.arange(c, c + n) for n, c in zip(lengths, contexts)]).int().cuda()
    starts = torch.tensor([0, *lengths]).cumsum(0).int().cuda()
    return q, k_pages, v_pages, requests, positions, tables.cuda(), starts, torch.tensor(contexts).int().cuda()


def _attention(q, k_pages, v_pages, requests, positions, tables, starts, contexts, lengths, heads, head_size, **options):
    from mini_llm_amd.ops import kernels as K

    before = K.launch_counts()
    out = K.paged_attention(q, k_pages, v_pages, requests, positions, tables, heads, k_pages.shape[1], head_size, head_size**-0.5, max_q_len=max(lengths),
                            max_len=int(positions.max()) + 1, q_starts=starts, context_lens=contexts, **options)
    assert list(K.launches_since(before)) == ["attention_prefill_stream"]   # (in 32-bit: the kernel in pieces, there is no other of that name)
    return out


def _exact(q, k_pages, v_pages, tables, starts, contexts, heads, head_size, window=0, keep_first=0, chunk=0, softcap=0.0, sinks=None, one_by_one=False):
    """The same in 64 bits."""
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    for r in range(len(contexts)):
        lo, hi, context = int(starts[r]), int(starts[r + 1]), int(contexts[r])
        keys, values = (pages[tables[r].long()].permute(1, 0, 2, 3).reshape(pages.shape[1], -1, head_size)[:, : context + hi - lo].double().repeat_interleave(heads // pages.shape[1], 0)
                        for pages in (k_pages, v_pages))
        scores = torch.matmul(q[lo:hi].view(-1, heads, head_size).permute(1, 0, 2).double(), keys.transpose(1, 2).contiguous()) * head_size**-0.5
        if softcap:
            scores = softcap * torch.tanh(scores / softcap)
        at, key = torch.arange(context, context + hi - lo, device="cuda")[:, None], torch.arange(context + hi - lo, device="cuda")[None]
        seen = (key <= at) & ((key > at - window) | (key < keep_first) if window else key >= 0) & (key // chunk == at // chunk if chunk else key >= 0)
        scores = scores.masked_fill(~seen, -torch.inf)
        if sinks is not None:   # a score without a key
            scores = torch.cat([scores, sinks.double()[:, None, None].expand(-1, hi - lo, 1)], 2)
        weights = scores.softmax(-1)[:, :, : context + hi - lo]
        # (a key that a row does not see adds nothing to it, whatever its value)
        mixed = torch.where(seen[None, :, :, None], weights[..., None] * values[:, None], 0.0).sum(2) if one_by_one else torch.matmul(weights, values)
        out[lo:hi] = mixed.permute(1, 0, 2).reshape(hi - lo, -1)
    return out


def _with_sinks(options, heads):
    return options | (dict(sinks=torch.linspace(-1.0, 2.0, heads, device="cuda")) if options.get("sinks") else {})


# heads, heads of keys, keys a page, and what bounds or bends the scores: every form of the kernel
FORMS = [(3, 3, 32, {}), (4, 2, 64, {}), (3, 1, 32, dict(sinks=True)), (2, 2, 32, dict(window=28)), (4, 2, 32, dict(window=33, sinks=True)), (2, 2, 64, dict(chunk=50)),
         (2, 1, 32, dict(softcap=2.0)), (2, 2, 64, dict(softcap=2.0, window=40, sinks=True)), (2, 2, 32, dict(softcap=2.0, chunk=64)), (3, 3, 32, dict(window=40, keep_first=5)),
         (4, 2, 64, dict(window=33, keep_first=70, softcap=2.0, sinks=True))]


@pytest.mark.parametrize("head_size", [32, 64])
@pytest.mark.parametrize("heads,kv_heads,page_size,options", FORMS)
# tiles of 32 queries and keys, a row more or less; waves without a tile, with one and with many; with windows, rows whose only keys of a tile are its last four
@pytest.mark.parametrize("lengths,contexts", [([65], [0]), ([66, 129, 97], [0, 31, 32]), ([128, 300], [700, 0]), ([200, 90], [0, 100])])
def test_prompt_attention_in_pieces(head_size, heads, kv_heads, page_size, options, lengths, contexts):
    arrays, options = _prompt(lengths, contexts, heads, head_size, kv_heads, page_size), _with_sinks(options, heads)
    out = _attention(*arrays, lengths, heads, head_size, **options)
    ref = _exact(*(arrays[n] for n in (0, 1, 2, 5, 6, 7)), heads, head_size, **options)
    assert _norm(out, ref) < plain_pieces.NORM_BOUND
    # scores of head_size products, each 2^-24 off at the most, with as many roundings as there are instructions; the weights' and the values' sums alike, over up to 1,000 keys whose
    # values are of order one: some 2^-24 (head_size + 60) of the largest value
    assert float((out.double() - ref).abs().max()) < 2**-24 * (head_size + 60) * 4


@pytest.mark.parametrize("what", ["infinite key", "infinite value", "largest value", "no number", "tiny values", "tiny queries", "large queries"])
@pytest.mark.parametrize("head_size,heads,kv_heads,options", [
    (64, 2, 2, {}), (32, 4, 2, dict(sinks=True)), (32, 2, 2, dict(window=40)), (64, 2, 2, dict(chunk=48)), (64, 4, 2, dict(softcap=3.0)), (32, 2, 1, dict(window=40, keep_first=35, sinks=True))])
def test_prompt_attention_of_numbers_that_have_no_pieces(what, head_size, heads, kv_heads, options):
    lengths, contexts = [100, 70], [0, 40]
    arrays, options = _prompt(lengths, contexts, heads, head_size, kv_heads), _with_sinks(options, heads)
    q, k_pages, v_pages, tables = arrays[0], arrays[1], arrays[2], arrays[5]
    page = int(tables[0, 1])   # keys 32 to 63 of the first request
    if what == "infinite key":      # a score of minus infinity for queries on its other side, no number for those on its own
        k_pages[page, 0, 3, 5] = torch.inf
    elif what == "infinite value":
        v_pages[page, -1, 4, 7] = -torch.inf
    elif what == "largest value":   # rounds to infinity as a bfloat16 number
        v_pages[page, -1, 4, 7] = torch.finfo(torch.float32).max
    elif what == "no number":
        v_pages[page, 0, 9, 0] = torch.nan
    else:
        scaled = dict(q=1.0, keys=1.0, values=1.0) | plain_pieces.ODD[what]
        q *= scaled["q"]
        k_pages *= scaled["keys"]
        v_pages[:, -1] *= scaled["values"]
    out = _attention(*arrays, lengths, heads, head_size, **options)
    ref = _exact(*(arrays[n] for n in (0, 1, 2, 5, 6, 7)), heads, head_size, one_by_one=True, **options)
    # a product with an infinity in 64 bits is that in 32: what is no number there is none here, infinities are the same, and so is the rest
    assert bool((out.isnan() == ref.isnan()).all())
    plain = ref.isfinite() & out.isfinite()
    assert bool((out.double() == ref)[~plain & ~ref.isnan() & ref.isinf()].all())
    # errors beside a head's common size: 2^-24 of it (or of a number below the smallest normal one) for each of some hundred roundings
    tiny_heads = torch.arange(heads, device="cuda") // (heads // kv_heads) == kv_heads - 1
    size = torch.where(tiny_heads, plain_pieces.ODD["tiny values"]["values"] if what == "tiny values" else 1.0, 1.0).double().repeat_interleave(head_size)
    error = ((out.double() - ref).abs() / torch.maximum(ref.abs(), size))[plain]
    assert float(error.max()) < 2**-24 * 300
    if what in plain_pieces.ODD:
        assert _norm(out.double()[:, tiny_heads.repeat_interleave(head_size)] / scaled["values"], ref[:, tiny_heads.repeat_interleave(head_size)] / scaled["values"]) < plain_pieces.ODD_BOUND


@pytest.mark.parametrize("head_size", [32, 64])
@pytest.mark.parametrize("what", ["a large value at a small weight", "a column of tiny values"])
def test_prompt_attention_whose_pieces_are_lost(head_size, what):
    """Finite results of ordinary size (or exact zeros) to which numbers belong that leave no pieces: they are taken again in 32-bit."""
    heads, lengths, contexts = 2, [100, 70], [0, 40]
    arrays = _prompt(lengths, contexts, heads, head_size)
    q, k_pages, v_pages, tables = arrays[0], arrays[1], arrays[2], arrays[5]
    page = int(tables[0, 1])   # keys 32 to 63 of the first request
    if what == "a column of tiny values":
        v_pages[:, 1, :, 9] = 2.0**-136 * (1 + torch.rand(v_pages.shape[0], v_pages.shape[2], device="cuda"))
    else:   # all scores 0, but -88 for key 35, whose weight is e^-88 = 6e-39 and whose value is 1.3e38
        k_pages.zero_(), q.zero_()
        k_pages[page, 0, 3, 0], q[:, 0] = -1.0, 88.0 * head_size**0.5
        v_pages[page, 0, 3, 7] = 1.5 * 2.0**126
    out = _attention(*arrays, lengths, heads, head_size)
    ref = _exact(*(arrays[n] for n in (0, 1, 2, 5, 6, 7)), heads, head_size)
    if what == "a column of tiny values":   # subnormal sums of at most 110 products over a total of at least 1, each a part of 2^-149 off: the weights add up to the total
        at = head_size + 9
        assert float((out[:, at].double() - ref[:, at]).abs().max()) <= 2**-149 * 4
    else:   # the weight is subnormal, 2^-22 off itself, and so is its share of 0.8 / n; the rest as ever
        assert float((out[:100, 7].double() - ref[:100, 7]).abs().max()) < 2**-20
        assert float((ref[40:100, 7] - _exact(q, k_pages, v_pages.clamp(max=1e30), *(arrays[n] for n in (5, 6, 7)), heads, head_size)[40:100, 7]).abs().min()) > 1e-3   # (it counts)


@pytest.mark.parametrize("what", ["a tiny number", "a large number", "no number"])
def test_a_query_taken_again_leaves_the_others_alone(what):
    """Rows of a query tile that need no second way keep their results, bit for bit, beside one that does (and what is no number needs none)."""
    heads, head_size, lengths, contexts = 2, 64, [100, 70], [0, 40]
    arrays = _prompt(lengths, contexts, heads, head_size)
    q, row = arrays[0], 40
    plain = _attention(*arrays, lengths, heads, head_size)
    q[row, 5] = {"a tiny number": 2.0**-100, "a large number": 2.0**70, "no number": torch.nan}[what]
    out = _attention(*arrays, lengths, heads, head_size)
    others = torch.arange(q.shape[0], device="cuda") != row
    assert bool((out[others] == plain[others]).all()) and bool((out[row, head_size:] == plain[row, head_size:]).all())
    assert bool(out[row, :head_size].isnan().all()) == (what == "no number")


def test_prompt_attention_over_its_own_queries():
    """Results may take the queries' place: what is taken again reads them before anything is stored over them."""
    heads, head_size, lengths, contexts = 2, 64, [100, 70], [0, 40]
    arrays = _prompt(lengths, contexts, heads, head_size)
    arrays[2][int(arrays[5][0, 1]), 1, 4, 7] = -torch.inf
    arrays[0][50, 3] = 2.0**-100
    want = _attention(*arrays, lengths, heads, head_size)
    got = _attention(*arrays, lengths, heads, head_size, out=arrays[0])
    assert got.data_ptr() == arrays[0].data_ptr() and bool(got.isfinite().any())
    torch.testing.assert_close(got, want, rtol=0, atol=0, equal_nan=True)
