"""32-bit latent attention on the matrix cores against sums in 64 bits."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def attend(q, rows, positions, rank, scale, sinks):
    """q [n, heads, size] and the sequence's cached rows, in 64 bits."""
    scores = torch.einsum("nhd,kd->nhk", q, rows) * scale
    scores = scores.masked_fill(torch.arange(rows.shape[0])[None, None, :] > positions[:, None, None], -math.inf)
    if sinks is not None:
        scores = torch.cat([scores, sinks[None, :, None].expand(q.shape[0], -1, 1)], dim=2)
    weights = torch.softmax(scores, dim=2)[:, :, : rows.shape[0]]
    # a key that a row does not see has no part in it, whatever it holds
    seen = torch.arange(rows.shape[0])[None, :] <= positions[:, None]
    return torch.stack([weights[i][:, seen[i]] @ rows[seen[i], :rank] for i in range(q.shape[0])])


@pytest.mark.parametrize("heads,rank,rot,page_size,runs", [(12, 256, 32, 64, False), (5, 129, 30, 16, True), (7, 100, 20, 32, False), (3, 64, 32, 16, True), (1, 61, 3, 8, False), (2, 21, 7, 4, True)])
@pytest.mark.parametrize("sink", [True, False])
def test_32_bit_latent_attention_on_the_matrix_cores(monkeypatch, heads, rank, rot, page_size, runs, sink):
    # portions whose ends lie beside the borders of the tiles of 32 keys and of the eight waves' 256, single tokens, rows of no request
    from mini_llm_amd.ops import kernels as k

    monkeypatch.setattr(k, "LATENT_F32_PAIRS", 1)
    if not runs:
        monkeypatch.setattr(k, "LATENT_TARGET_BLOCKS", 0)
    contexts, portions, pad = [0, 255, 31, 600, 0, 256], [67, 3, 1, 33, 1, 1], 3
    size = k.latent_row_size(rank + rot)
    generator = torch.Generator().manual_seed(rank)
    lengths = [c + p for c, p in zip(contexts, portions)]
    blocks = [-(-n // page_size) for n in lengths]
    pages = torch.zeros(sum(blocks) + 1, 1, page_size, size)
    tables = torch.full((len(lengths) + 1, max(blocks) + 1), -1, dtype=torch.int32)
    order, at, cached = torch.randperm(sum(blocks) + 1, generator=generator), 0, []
    for r, n in enumerate(lengths):
        rows = torch.randn(n, size, generator=generator)
        rows[:, rank + rot :] = 0
        cached.append(rows)
        for b in range(blocks[r]):
            tables[r, b] = order[at]
            chunk = rows[b * page_size : (b + 1) * page_size]
            pages[order[at], 0, : len(chunk)] = chunk
            at += 1
    owner = torch.cat([torch.full((p,), i) for i, p in enumerate(portions)] + [torch.full((pad,), -1)])
    positions = torch.cat([torch.arange(c, c + p) for c, p in zip(contexts, portions)] + [torch.zeros(pad, dtype=torch.long)])
    starts = torch.tensor([0] + [sum(portions[: i + 1]) for i in range(len(portions))] + [sum(portions) + pad])
    q = torch.randn(sum(portions) + pad, heads, size, generator=generator)
    q[:, :, rank + rot :] = 0
    sinks = torch.randn(heads, generator=generator)
    ints = lambda t: t.int().cuda()
    scale = 0.15

    def run(pages, longest):
        return k.latent_attention(q.cuda(), pages.cuda(), sinks.cuda() if sink else None, ints(owner), ints(positions), ints(tables), rank, scale, max_len=longest,
                                  q_starts=ints(starts), context_lens=ints(torch.tensor(contexts + [-1])), max_q_len=max(portions)).cpu().double()

    for longest in (max(lengths), 4 * max(lengths)):
        got = run(pages, longest)
        assert (got[sum(portions) :] == 0).all()
        for r, rows in enumerate(cached):
            mine = slice(int(starts[r]), int(starts[r + 1]))
            want = attend(q[mine].double(), rows.double(), positions[mine], rank, scale, sinks.double() if sink else None)
            # a score is a sum of up to 288 products of numbers around 1 (each rounded to 2^-24 of the running sum, some 2^5 here) and is off by about 2^-24 * 2^5
            # * 0.15 * 17 roundings (square root of 288) < 5e-6; its exponential by as much of itself, and the sums by a little more
            assert (got[mine] - want).norm() / want.norm() < 1e-5

    # an infinity in a row's latent: those before it do not see it, those from it on do
    hurt = pages.clone()
    place = 40
    hurt[int(tables[0, place // page_size]), 0, place % page_size, 5] = math.inf
    got = run(hurt, max(lengths))
    first = int(starts[0])
    assert got[first : first + place].isfinite().all()
    assert not got[first + place : first + portions[0], :, 5].isfinite().any()
    assert got[first + portions[0] : sum(portions)].isfinite().all()


# one request, an even and an odd number of them, eight (the most of which a request's tiles lie side by side) and more, a padding one at the end and rows of no request; portions of one tile beside ones of several
@pytest.mark.parametrize("contexts,portions", [([0], [70]), ([5], [1]), ([300, 0], [1, 40]), ([0, 90, 300], [33, 1, 2]), ([40, 0, 200, 7, 0, 150, 31, 9], [1, 30, 1, 1, 12, 1, 1, 1]),
                                               ([130] * 10 + [0], [1] * 10 + [60])])
@pytest.mark.parametrize("padding", [0, 1])
def test_32_bit_latent_attention_finds_every_tile_of_every_request(monkeypatch, contexts, portions, padding):
    from mini_llm_amd.ops import kernels as k

    monkeypatch.setattr(k, "LATENT_F32_PAIRS", 1)
    monkeypatch.setattr(k, "LATENT_F32_KEYS", 1)
    heads, rank, size, page_size, scale = 6, 160, 192, 16, 0.1
    generator = torch.Generator().manual_seed(len(contexts))
    blocks = [-(-(c + p) // page_size) for c, p in zip(contexts, portions)]
    pages = torch.randn(sum(blocks) + 1, 1, page_size, size, generator=generator)
    order = torch.randperm(sum(blocks) + 1, generator=generator)
    tables = torch.full((len(contexts) + padding, max(blocks)), -1, dtype=torch.int32)
    for r, n in enumerate(blocks):
        tables[r, :n] = order[sum(blocks[:r]) : sum(blocks[: r + 1])]
    rows, spare = sum(portions), 5 * padding
    owner = torch.cat([torch.full((p,), i) for i, p in enumerate(portions)] + [torch.full((spare,), -1)])
    positions = torch.cat([torch.arange(c, c + p) for c, p in zip(contexts, portions)] + [torch.zeros(spare, dtype=torch.long)])
    starts = torch.tensor([0] + [sum(portions[: i + 1]) for i in range(len(portions))] + [rows + spare] * padding)
    q = torch.randn(rows + spare, heads, size, generator=generator)
    ints = lambda t: t.int().cuda()
    got = k.latent_attention(q.cuda(), pages.cuda(), None, ints(owner), ints(positions), ints(tables), rank, scale, max_len=max(c + p for c, p in zip(contexts, portions)),
                             q_starts=ints(starts), context_lens=ints(torch.tensor(contexts + [-1] * padding)), max_q_len=max(portions)).cpu().double()
    assert (got[rows:] == 0).all()
    for r in range(len(contexts)):
        mine = slice(int(starts[r]), int(starts[r + 1]))
        cached = pages[tables[r, : blocks[r]].long()].reshape(-1, size)[: contexts[r] + portions[r]].double()
        want = attend(q[mine].double(), cached, positions[mine], rank, scale, None)
        assert (got[mine] - want).norm() / want.norm() < 1e-5   # (the bound above, for shorter rows)
