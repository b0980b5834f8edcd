"""Decoding rows and prompt portions in one launch, against the two launches that take each kind by itself (which the tests of the kernels hold against
the plain implementation)."""

import numpy as np
import pytest
import torch

DEV = "cuda:0"
B, F = torch.bfloat16, torch.float32


@pytest.mark.parametrize("short_rows,heads,reach,longest,takes", [
    (112, 8, 2048, 65, True), (113, 8, 2048, 65, False), (896, 1, 64, 512, True), (32, 28, 2048, 512, True), (64, 16, 2048, 512, False), (65535, 65535, 64, 512, False),
    (16, 16, 2049, 512, False), (16, 16, 2048, 64, False)])
@pytest.mark.parametrize("dtype", [B, F])
def test_where_both_kinds_take_one_launch(dtype, short_rows, heads, reach, longest, takes):
    from mini_llm_amd.ops.library import library

    stride = min(heads, 1024) * 64
    assert bool(library().mllm_attention_mixed_takes(256, stride, 256, stride, short_rows, heads, 64, 64, longest, reach, 0.125, 1 if dtype == B else 0)) == takes


def _step(seed, dtype, heads, kv_heads, page_size, max_blocks, stored, portions):
    """Queries, pages and tables of a step: rows that decode over ``stored`` keys each (-1: a padding row), then prompt portions (keys stored, new tokens)."""
    rng = torch.Generator(device=DEV).manual_seed(seed)
    contexts, news = stored + [c for c, _ in portions], [1] * len(stored) + [n for _, n in portions]
    needs = [-(-(c + n) // page_size) if c >= 0 else 0 for c, n in zip(contexts, news)]
    pages = torch.randperm(sum(needs) + 1, generator=torch.Generator().manual_seed(1)).tolist()
    tables = np.full((len(contexts), max_blocks), -1, dtype=np.int32)
    for r, need in enumerate(needs):
        tables[r, :need] = [pages.pop() for _ in range(need)]
    rand = lambda *shape: torch.randn(shape, generator=rng, device=DEV).to(dtype)
    k_pages, v_pages = (rand(sum(needs) + 1, kv_heads, page_size, 64) for _ in range(2))
    q = rand(sum(news), heads * 64)
    request = np.concatenate([np.full(n, r if c >= 0 else -1) for r, (c, n) in enumerate(zip(contexts, news))])
    position = np.concatenate([max(c, 0) + np.arange(n) for c, n in zip(contexts, news)])
    ints = lambda a: torch.as_tensor(np.asarray(a, dtype=np.int32), device=DEV)
    request, position, starts, lens, tables = ints(request), ints(position), ints(np.cumsum([0] + news)), ints(contexts), ints(tables)
    shared = dict(n_heads=heads, n_kv_heads=kv_heads, head_size=64, scale=0.125)
    return q, (k_pages, v_pages), (request, position, tables), (starts, lens), news, shared


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [B, F])
@pytest.mark.parametrize("heads,kv_heads,page_size,max_blocks,stored,portions,one_launch", [
    (1, 1, 64, 4, [0], [(0, 65)], True),                                                  # the smallest: one row of one key
    (12, 12, 64, 16, [511, -1, 5, 1000], [(0, 96), (200, 70)], True),                     # a padding row
    (5, 5, 32, 64, [63, 64, 65], [(0, 64), (31, 130), (1900, 148)], True),                # heads and rows that are no multiple of eight; the reach's edge
    (25, 25, 64, 8, [17] * 9 + [-1] * 7, [(0, 33), (64, 100), (0, 8 + 1)], True),         # a portion just longer than a short one
    (16, 4, 64, 16, [700] * 32, [(0, 512), (100, 400), (0, 300)], True),                  # blocks of 64 queries in bfloat16; grouped heads
    (4, 4, 64, 33, [2000], [(0, 80)], False),                                             # a block table that reaches further
    (4, 4, 16, 16, [20], [(0, 80)], False),                                               # pages shorter than a tile
])
def test_both_kinds_in_one_launch(dtype, heads, kv_heads, page_size, max_blocks, stored, portions, one_launch):
    from mini_llm_amd.ops import kernels as K

    q, (k_pages, v_pages), (request, position, tables), (starts, lens), news, shared = _step(heads * max_blocks, dtype, heads, kv_heads, page_size, max_blocks, stored, portions)
    few, longest = len(stored), max(news)
    before = K.launch_counts()
    got = K.paged_attention(q, k_pages, v_pages, request, position, tables, max_q_len=longest, q_starts=starts, context_lens=lens, short_rows=few, short_requests=few, **shared)
    assert K.launches_since(before).get("attention_mixed", 0) == int(one_launch)
    rows = K.paged_attention(q[:few], k_pages, v_pages, request, position, tables, max_q_len=1, **shared)
    prompts = K.paged_attention(q, k_pages, v_pages, request, position, tables[few:], max_q_len=longest, q_starts=starts[few:], context_lens=lens[few:], **shared)
    # Sums in 32-bit in another order, and in bfloat16 the one rounding of the result (2^-8) and those of the prompts' weights, each taken at another maximum (2^-9 of
    # a mean of values around 1, the weights sum to 1).
    bound = 2e-5 if dtype == F else 2.0 ** -7
    for here, there in ((got[:few], rows), (got[few:], prompts[few:])):
        torch.testing.assert_close(here.float(), there.float(), rtol=bound, atol=bound)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,keys", [(8, 700), (16, 2000)])
def test_32_bit_rows_beside_a_prompt_are_no_further_off_than_alone(rows, keys):
    # The relative error (2-norm) against 64 bits over a few steps: four waves a row here, sixteen or several blocks in a launch of their own.
    from mini_llm_amd.ops import kernels as K

    errors = {True: [], False: []}
    for seed in range(3):
        q, (k_pages, v_pages), (request, position, tables), (starts, lens), news, shared = _step(seed, F, 12, 12, 64, 32, [keys] * rows, [(0, 480)])
        want = torch.empty((rows, 12 * 64), dtype=torch.float64, device=DEV)
        for r in range(rows):
            pages = tables[r][tables[r] >= 0].long()
            k, v = (p[pages].double().transpose(0, 1).reshape(12, -1, 64)[:, : keys + 1] for p in (k_pages, v_pages))
            weights = torch.softmax((q[r].double().view(12, 1, 64) * k).sum(-1) * 0.125, -1)
            want[r] = (weights[..., None] * v).sum(1).reshape(-1)
        beside = K.paged_attention(q, k_pages, v_pages, request, position, tables, max_q_len=max(news), q_starts=starts, context_lens=lens, short_rows=rows, short_requests=rows, **shared)
        alone = K.paged_attention(q[:rows], k_pages, v_pages, request, position, tables, max_q_len=1, **shared)
        for here, out in ((True, beside[:rows]), (False, alone)):
            errors[here].append(((out.double() - want).norm() / want.norm()).item())
    assert np.mean(errors[True]) <= np.mean(errors[False]), errors
