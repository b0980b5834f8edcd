"""The kernel that decodes all layers of a pre-norm model at once, against the same layers one by one in float64 with numbers kept in the kernel's
precision where it keeps them: sizes at the edges of its tiles, steps and key rounds, few and many blocks, padding rows."""

import math

import numpy as np
import pytest
import torch

import plain_gpt2 as P

DEV = "cuda:0"


@pytest.mark.parametrize("rows,reach,width,pays", [(1, 1024, 768, True), (8, 1792, 768, True), (8, 1793, 768, False), (9, 1024, 768, True), (16, 1025, 768, False),
                                                   (17, 64, 768, False), (2, 1792, 1600, True), (4, 1024, 1600, True), (4, 1792, 1600, False), (5, 64, 1600, False)])
def test_where_one_kernel_for_all_layers_pays(rows, reach, width, pays):
    from mini_llm_amd.ops.library import library

    assert bool(library().mllm_decode_stack_pays(rows, reach, width)) == pays


@pytest.mark.parametrize("rows,reach,layers,width,inner,dtype,pays", [
    (8, 1792, 12, 768, 3072, torch.bfloat16, True), (16, 1024, 12, 768, 3072, torch.bfloat16, True), (8, 1793, 12, 768, 3072, torch.bfloat16, False),
    (1, 64, 1, 768, 3072, torch.bfloat16, False), (1, 64, 2, 768, 3072, torch.bfloat16, True), (1, 64, 1, 768, 3072, torch.float32, False),          # one layer
    (16, 64, 7, 768, 3072, torch.bfloat16, False), (16, 64, 8, 768, 3072, torch.bfloat16, True), (8, 64, 2, 768, 3072, torch.bfloat16, True),       # more than 8 rows: few layers,
    (16, 64, 12, 768, 3104, torch.bfloat16, False), (8, 64, 12, 768, 3104, torch.bfloat16, True), (16, 64, 12, 1024, 5632, torch.bfloat16, False),   # many hidden units
    (4, 64, 3, 1600, 6400, torch.bfloat16, False), (4, 64, 4, 1600, 6400, torch.bfloat16, True), (2, 64, 2, 1600, 6400, torch.bfloat16, True),
    (1, 1025, 7, 768, 3072, torch.float32, False), (1, 1025, 8, 768, 3072, torch.float32, True), (1, 1024, 2, 768, 3072, torch.float32, True),       # 32-bit and many keys
    (1, 1025, 12, 576, 2304, torch.float32, False), (1, 1025, 12, 640, 2560, torch.float32, True), (1, 1025, 12, 640, 2592, torch.float32, False),
    (1, 1025, 2, 128, 4096, torch.bfloat16, True)])
def test_for_which_models_one_kernel_for_all_layers_pays(rows, reach, layers, width, inner, dtype, pays):
    from mini_llm_amd.ops import kernels as K

    assert K.decode_stack_pays(rows, reach, layers, width, inner, width // 64, 64, 64, dtype) == pays


@pytest.mark.parametrize("rows,layers,width,inner,heads,head,page,dtype,supported", [
    (1, 12, 768, 3072, 12, 64, 64, torch.bfloat16, True), (16, 64, 768, 3072, 12, 64, 1, torch.float32, True), (16, 48, 1600, 6400, 25, 64, 64, torch.bfloat16, True),
    (17, 12, 768, 3072, 12, 64, 64, torch.bfloat16, False), (1, 65, 768, 3072, 12, 64, 64, torch.bfloat16, False), (1, 12, 768, 3072, 24, 32, 64, torch.bfloat16, False),
    (1, 12, 768, 3088, 12, 64, 64, torch.bfloat16, False), (1, 12, 768, 3104, 12, 64, 64, torch.bfloat16, True), (1, 12, 1600, 6400, 25, 64, 64, torch.float32, False),
    (1, 12, 768, 3072, 12, 64, 48, torch.bfloat16, False), (1, 12, 768, 3072, 11, 64, 64, torch.bfloat16, False), (1, 12, 1856, 1024, 29, 64, 64, torch.bfloat16, False)])
def test_what_one_kernel_for_all_layers_takes(rows, layers, width, inner, heads, head, page, dtype, supported):
    from mini_llm_amd.ops import kernels as K

    assert K.decode_stack_supported(rows, layers, width, inner, heads, head, page, dtype) == supported


def _plain_block(width=128, heads=2, kv_heads=None, window=None, inner=256, eps=(1e-5, 1e-5), dtype=torch.bfloat16):
    """A pre-norm layer as a GPT-2 has it, every matrix packed (their numbers do not matter here)."""
    from mini_llm_amd.ops import kernels as K
    from mini_llm_amd.parts.attention import CausalSelfAttention
    from mini_llm_amd.parts.block import PreNormBlock
    from mini_llm_amd.parts.feedforward import DenseMLP
    from mini_llm_amd.parts.norms import LayerNorm

    block = PreNormBlock(LayerNorm(width, eps[0]), CausalSelfAttention(width, heads, kv_heads, window=window), LayerNorm(width, eps[1]), DenseMLP(width, inner, "gelu_new"), dtype)
    for norm in (block.norm_1, block.norm_2):
        norm.weight, norm.bias = torch.ones(width), torch.zeros(width)
    for product in (block.mixer.qkv, block.mixer.out, block.feed_forward.up, block.feed_forward.down):
        product.weight = K.PackedMatrix(torch.zeros(product.out_features * product.in_features, dtype=dtype), product.out_features, product.in_features)
        product.bias = torch.zeros(product.out_features)
    return block


def _context(width=128, dtype=torch.bfloat16, write_cache=True, page_size=16):
    from types import SimpleNamespace

    pages = torch.zeros((3, width // 64, page_size, 64), dtype=dtype)
    return SimpleNamespace(k_pages=pages, v_pages=pages, write_cache=write_cache)


def test_the_layers_that_one_kernel_takes():
    from mini_llm_amd.ops import kernels as K
    from mini_llm_amd.parts.feedforward import PlainMLP
    from mini_llm_amd.parts.norms import LayerNorm, RMSNorm

    layer, shared = _plain_block().stack_layer(_context())
    assert isinstance(layer, K.StackLayer) and shared == (128, 256, 2, 64, 16, 1e-5, 1e-5, 0.125, "gelu_new")

    def refused(change=lambda block: None, context=None, **how):
        block = _plain_block(**how)
        change(block)
        return block.stack_layer(context or _context()) is None

    row_major = lambda product: setattr(product, "weight", torch.zeros((product.out_features, product.in_features), dtype=torch.bfloat16))
    assert not refused()
    assert refused(window=32)
    assert refused(heads=2, kv_heads=1)
    assert refused(lambda b: setattr(b, "norm_1", RMSNorm(128, 1e-5))) and refused(lambda b: setattr(b, "norm_2", type("Other", (LayerNorm,), {})(128, 1e-5)))
    assert refused(lambda b: setattr(b, "feed_forward", PlainMLP(128, 256, "gelu_new")))
    for product in (lambda b: b.mixer.qkv, lambda b: b.mixer.out, lambda b: b.feed_forward.up, lambda b: b.feed_forward.down):
        assert refused(lambda b: row_major(product(b)))
        assert refused(lambda b: setattr(product(b), "bias", None))
    assert refused(context=_context(dtype=torch.float32))             # pages of another type than the matrices
    assert refused(context=_context(write_cache=False))               # a layer that reads what another has stored
    no_pages = _context()
    no_pages.k_pages = None
    assert refused(context=no_pages)


def test_the_models_and_steps_that_one_kernel_takes(monkeypatch):
    from types import SimpleNamespace

    from mini_llm_amd.models.base import LayerCall, Model
    from mini_llm_amd.ops import kernels as K
    from mini_llm_amd.parts.norms import LayerNorm, RMSNorm

    monkeypatch.setattr(K, "DecodeStack", lambda layers, rows, n_heads, eps_1, eps_2, scale, activation, final: (len(layers), rows, n_heads, eps_1, eps_2, scale, activation, final))

    def made(blocks=None, schedule=None, rows=4, reach=512, wanted=None, groups=1, vectors=None, norm=LayerNorm, page_size=16):
        blocks = [_plain_block(), _plain_block()] if blocks is None else blocks
        model = SimpleNamespace(blocks=blocks, schedule=[LayerCall(i, i) for i in range(len(blocks))] if schedule is None else schedule, step_vectors=vectors, final_norm=norm(128, 3e-5))
        model.final_norm.weight = model.final_norm.bias = torch.ones(128)
        batch = SimpleNamespace(n_tokens=rows, n_logit_rows=rows if wanted is None else wanted, max_total_len=reach)
        cache = SimpleNamespace(groups=[None] * groups, layer_context=lambda batch, call: _context(page_size=page_size))
        return Model.decode_stack(model, batch, cache)

    *sizes, final = made()
    assert sizes == [2, 4, 2, 1e-5, 1e-5, 0.125, "gelu_new"] and final[2] == 3e-5
    assert made(norm=RMSNorm)[-1] is None and made(wanted=3)[-1] is None   # the norm in front of the head stays a kernel of its own
    assert made(blocks=[_plain_block(), _plain_block(eps=(1e-5, 1e-6))]) is None and made(blocks=[_plain_block(), _plain_block(inner=512)]) is None
    assert made(blocks=[_plain_block(), _plain_block(window=16)]) is None and made(blocks=[]) is None
    assert made(schedule=[LayerCall(0, 0), LayerCall(0, 1)]) is None      # a block that runs twice
    assert made(groups=2) is None and made(vectors=object()) is None
    assert made(reach=1793) is None and made(rows=17) is None and made(blocks=[_plain_block()]) is None and made(page_size=24) is None


def _stack(rng, layers, width, inner, contexts, page_size, dtype, activation, blocks):
    """A DecodeStack over random layers and a cache that holds ``contexts`` keys a row (-1: a padding row), what it is run on, and what the layers give in float64."""
    from test_kernels_gpu import as_weight, bf16_round, dev, plain_paged_attention

    from mini_llm_amd.ops import kernels as K

    kept = bf16_round if dtype == torch.bfloat16 else (lambda a: np.asarray(a, dtype=np.float32).astype(np.float64))
    heads, rows, eps = width // 64, len(contexts), 2e-5
    blocks_of = [(c + 1 + page_size - 1) // page_size if c >= 0 else 0 for c in contexts]
    num_pages, max_blocks = sum(blocks_of) + 2, max(blocks_of)
    order = rng.permutation(num_pages).tolist()
    tables, slots = np.full((rows, max_blocks), -1, dtype=np.int32), np.full(rows, -1, dtype=np.int32)
    for r, n in enumerate(blocks_of):
        tables[r, :n] = [order.pop() for _ in range(n)]
        if n:
            slots[r] = tables[r, contexts[r] // page_size] * page_size + contexts[r] % page_size
    stream = rng.standard_normal((rows, width)).astype(np.float32)
    x, made, expected_rows = stream.astype(np.float64), [], []
    for _ in range(layers):
        vector = lambda n, mean=0.0: (mean + 0.1 * rng.standard_normal(n)).astype(np.float32)
        matrix = lambda n, k, scale: kept(rng.standard_normal((n, k)) * (scale / math.sqrt(k)))
        g1, o1, g2, o2 = vector(width, 1.0), vector(width), vector(width, 1.0), vector(width)
        w_qkv, w_out, w_up, w_down = matrix(3 * width, width, 2.0), matrix(width, width, 0.5), matrix(inner, width, 1.0), matrix(width, inner, 0.5)
        b_qkv, b_out, b_up, b_down = vector(3 * width), vector(width), vector(inner), vector(width)
        k_pages = torch.full((num_pages, heads, page_size, 64), float("nan"), device=DEV, dtype=dtype)
        v_pages = torch.full_like(k_pages, float("nan"))
        qkv = kept(kept(P.layernorm(x, g1, o1, eps)) @ w_qkv.T + b_qkv)
        mixed, here = np.zeros((rows, width)), []
        for r, context in enumerate(contexts):
            if context < 0:
                continue
            keys, values = kept(rng.standard_normal((context + 1, width))), kept(rng.standard_normal((context + 1, width)))
            if context:
                at = np.array([tables[r, p // page_size] * page_size + p % page_size for p in range(context)], dtype=np.int32)
                K.cache_write(dev(keys[:context], dtype), dev(values[:context], dtype), k_pages, v_pages, dev(at, torch.int32), heads, 64)
            keys[context], values[context] = qkv[r, width : 2 * width], qkv[r, 2 * width :]
            here.append((int(slots[r]), keys[context], values[context]))
            mixed[r] = kept(plain_paged_attention(qkv[r : r + 1, :width], keys, values, heads, heads, None))[0]
        x = x + mixed @ w_out.T + b_out
        up = kept(P.layernorm(x, g2, o2, eps)) @ w_up.T + b_up
        gelu = 0.5 * up * (1.0 + np.tanh(0.7978845608 * (up + 0.044715 * up**3))) if activation == "gelu_new" else \
            0.5 * up * (1.0 + torch.erf(torch.as_tensor(up / math.sqrt(2.0))).numpy())
        x = x + kept(gelu) @ w_down.T + b_down
        weight = lambda w: as_weight(K, w, dtype, True)
        made.append(K.StackLayer(dev(g1), dev(o1), weight(w_qkv), dev(b_qkv), weight(w_out), dev(b_out), dev(g2), dev(o2), weight(w_up), dev(b_up), weight(w_down), dev(b_down),
                                 k_pages, v_pages))
        expected_rows.append(here)
    request = np.array([r if c >= 0 else -1 for r, c in enumerate(contexts)], dtype=np.int32)
    stack = K.DecodeStack(made, rows, heads, eps, eps, 0.125, activation, blocks=blocks)
    given = (dev(stream), dev(request, torch.int32), dev(np.maximum(contexts, 0), torch.int32), dev(slots, torch.int32), dev(tables, torch.int32))
    return stack, given, x, expected_rows


B, F = torch.bfloat16, torch.float32


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,layers,width,inner,contexts,page_size,activation,blocks", [
    (B, 1, 64, 32, [0], 64, "gelu_new", None),                              # the smallest: one head, one step of K for a wave or none
    (B, 2, 128, 512, [5, 0, 64], 16, "gelu", None),
    (B, 3, 768, 3072, [0, 1, 7, 8, 9, 63, 512, 700], 64, "gelu_new", None),  # key shares of a wave at the edges of a load of eight keys
    (B, 2, 768, 3072, [1023, 1024, -1, 1030], 64, "gelu_new", None),         # 128 keys a wave in registers, and more; a padding row
    (B, 2, 768, 3104, [100] * 5, 1, "gelu_new", None),                       # pages of one key; hidden units beyond whole rounds of steps
    (B, 2, 832, 1056, [33, 600], 32, "gelu", None),                          # 26 steps of K for eight waves
    (B, 2, 1024, 4096, [40] * 16, 64, "gelu_new", None),                     # two pairs a block
    (B, 2, 1600, 6400, [20, 129], 64, "gelu_new", None),                     # norm pieces that end inside a row of lanes
    (B, 1, 1600, 6400, [70, -1, 300] + [9] * 13, 64, "gelu_new", None),      # four pairs a block, tiles not asked for ahead
    (F, 2, 64, 32, [3, 0], 64, "gelu_new", None),
    (F, 2, 768, 3072, [0, 3, 4, 5, 511, 512, 600, -1], 64, "gelu_new", None),
    (F, 1, 768, 3072, [77] * 16, 16, "gelu", None),
    (F, 2, 1024, 4096, [1, 200, 30], 64, "gelu_new", None),
    (F, 2, 832, 1056, [33], 64, "gelu", None),
    # work divided among fewer blocks: several groups of pairs a block, several tiles of the rows, rounds of tiles
    (B, 2, 192, 768, [10, 3, 100], 16, "gelu_new", 3), (B, 2, 768, 3072, [10, 65], 64, "gelu_new", 7), (F, 2, 192, 768, [10, 3, 100], 16, "gelu_new", 4),
    (B, 2, 768, 3072, [300] * 8, 64, "gelu_new", 40),
    (B, 2, 768, 3072, [30] * 8, 64, "gelu_new", 300),                        # more blocks than find a compute unit at once: the late ones are not members
])
def test_all_layers_in_one_kernel(dtype, layers, width, inner, contexts, page_size, activation, blocks):
    from test_kernels_gpu import host

    rng = np.random.default_rng(width + inner + len(contexts))
    stack, given, expected, new_rows = _stack(rng, layers, width, inner, contexts, page_size, dtype, activation, blocks)
    before = [(layer.k_pages.clone(), layer.v_pages.clone()) for layer in stack.layers]
    live = [r for r, c in enumerate(contexts) if c >= 0]
    # The bounds of the kernels for half a layer (5e-3: what roundings to bfloat16 that fall the other way come to) for each half; in 32-bit
    # sums of up to 4,096 products of numbers around 1 in another order, 2^-24 sqrt(4,096) each, a few times over a layer.
    bound = 1e-2 * layers if dtype == B else 2e-5 * layers
    out = stack.run(*given)
    np.testing.assert_allclose(host(out)[live], expected[live], rtol=bound, atol=bound)
    assert torch.isfinite(out).all()   # the padding row too
    for layer, (k_before, v_before), here in zip(stack.layers, before, new_rows):
        for pages, was, which in ((layer.k_pages, k_before, 1), (layer.v_pages, v_before, 2)):
            flat, flat_was = (t.permute(0, 2, 1, 3).reshape(-1, width) for t in (pages, was))
            for row in here:
                np.testing.assert_allclose(host(flat[row[0]]), row[which], rtol=bound, atol=bound)
                flat_was[row[0]] = flat[row[0]]
            raw = torch.int16 if dtype == B else torch.int32
            assert torch.equal(flat.view(raw), flat_was.view(raw))   # nothing else was written
    # launch after launch the same bits (the words of the last launch lie where this one's will), and the control words ready for the next
    for _ in range(3):
        assert torch.equal(stack.run(*given), out)
    control = stack.control.cpu()
    assert control[96] == 4 and int(control.count_nonzero()) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,width,contexts,blocks", [(B, 64, [3], None), (B, 768, [5] * 8, None), (B, 832, [9] * 16, None), (F, 768, [4, -1, 70], None), (F, 192, [10, 3, 8, 2], 4)])
def test_the_norm_behind_the_last_layer(dtype, width, contexts, blocks):
    # one block that norms and several rows; more rows than waves; a padding row
    from mini_llm_amd.ops import kernels as K

    rng = np.random.default_rng(width)
    stack, given, _, _ = _stack(rng, 2, width, 2 * width, contexts, 64, dtype, "gelu_new", blocks)
    stream = stack.run(*given)
    gain, offset = (torch.as_tensor(rng.standard_normal(width).astype(np.float32), device=DEV) for _ in range(2))
    normed = K.DecodeStack(stack.layers, len(contexts), width // 64, 2e-5, 2e-5, 0.125, "gelu_new", blocks=blocks, final=(gain, offset, 3e-5))
    out = normed.run(*given)
    # the norm's sums in another order: a few 2^-24 of numbers around 1; in bfloat16 a rounding that falls the other way, 2^-8 of them
    bound = 2.0 ** -7 if dtype == B else 1e-5
    torch.testing.assert_close(out.float(), K.layernorm(stream, gain, offset, 3e-5, out_dtype=dtype).float(), rtol=bound, atol=bound)
    for _ in range(3):
        assert out.dtype == dtype and torch.equal(normed.run(*given), out)


@pytest.mark.gpu
def test_all_layers_in_one_kernel_replayed_and_beside_another_stream():
    # a captured launch replayed with other work between the replays, and two stacks at once on two streams: each takes the units it finds
    rng = np.random.default_rng(5)
    first, given, expected, _ = _stack(rng, 2, 768, 3072, [50] * 8, 64, B, "gelu_new", None)
    second, given_2, expected_2, _ = _stack(rng, 2, 768, 3072, [80] * 4, 64, B, "gelu_new", None)
    out, out_2 = first.run(*given), second.run(*given_2)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        replayed = first.run(*given)
    for _ in range(4):
        replayed.zero_()
        graph.replay()
        assert torch.equal(replayed, out)
        assert torch.equal(first.run(*given), out)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = [[], []]
    torch.cuda.synchronize()
    for _ in range(20):
        for stream, stack, args, into in ((streams[0], first, given, outs[0]), (streams[1], second, given_2, outs[1])):
            with torch.cuda.stream(stream):
                into.append(stack.run(*args))
    torch.cuda.synchronize()
    # with fewer members a block has more tiles and pairs, each summed in the same order: the same bits
    assert all(torch.equal(o, out) for o in outs[0]) and all(torch.equal(o, out_2) for o in outs[1])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,with_norm", [(B, False), (B, True), (F, False), (F, True)])
def test_a_wait_that_is_given_up(dtype, with_norm):
    # Without patience the first look at words that are not there yet is the last one: the launch ends, says so, and neither rows nor cache hold numbers
    # that were not computed.
    from mini_llm_amd.ops import kernels as K

    rng = np.random.default_rng(11)
    contexts = [70, 5, -1]
    stack, given, _, _ = _stack(rng, 3, 768, 3072, contexts, 64, dtype, "gelu_new", None)
    good = stack.run(*given).clone()
    torch.cuda.synchronize()
    stack.check()
    kept = [(layer.k_pages.clone(), layer.v_pages.clone()) for layer in stack.layers]
    vector = lambda: torch.as_tensor(rng.standard_normal(768).astype(np.float32), device=DEV)
    hasty = K.DecodeStack(stack.layers, len(contexts), 12, 2e-5, 2e-5, 0.125, "gelu_new", final=(vector(), vector(), 2e-5) if with_norm else None, patience=0)
    out = hasty.run(*given)
    torch.cuda.synchronize()
    assert torch.isnan(out).any()
    with pytest.raises(RuntimeError, match="given up"):
        hasty.check()
    for layer, pages in zip(stack.layers, kept):   # (the keys and values of this token, where its launch came so far, are those of the launch before)
        for here, was in zip((layer.k_pages, layer.v_pages), pages):
            raw = torch.int16 if dtype == B else torch.int32
            assert torch.equal(here.view(raw), was.view(raw))
    control = hasty.control.cpu()
    assert control[96] == 1 and int(control.count_nonzero()) == 1   # ready for the next launch
    assert torch.equal(stack.run(*given), good)                     # and others are as they were
    stack.check()


@pytest.mark.gpu
def test_an_engine_reports_a_step_that_was_given_up(monkeypatch):
    from mini_llm_amd.config import config_from_dict
    from mini_llm_amd.engine import StepEntry
    from mini_llm_amd.engine.engine import Engine, EngineOptions
    from mini_llm_amd.ops import kernels as K

    monkeypatch.setattr(K.DecodeStack, "PATIENCE", 0)
    raw = {"architectures": ["GPT2LMHeadModel"], "n_layer": 2, "n_embd": 128, "n_head": 2, "n_inner": 512, "vocab_size": 300, "n_positions": 128,
           "layer_norm_epsilon": 1e-5, "activation_function": "gelu_new"}
    engine = Engine.from_random(config_from_dict(raw), 3, EngineOptions(dtype="bfloat16", max_sessions=4))
    handle = engine.try_take_cache()
    token = engine.prefill_greedy(handle, [1, 2, 3])
    with pytest.raises(RuntimeError, match="given up"):
        engine.decode_batch([handle], [token])                       # chosen tokens: as they are read
    length = engine.cache.length(handle)
    with pytest.raises(RuntimeError, match="given up"):
        engine.runner.step([StepEntry(handle, [4], [0])], choose=True)   # the next step of the kind: before it is launched
    assert engine.cache.length(handle) == length
    with engine.open_session() as session:
        session.prefill([5, 6, 7])
        with pytest.raises(RuntimeError, match="given up"):
            session.decode(8)                                        # logits: as they are read
    engine.close()


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 8])
def test_a_launch_waits_for_compute_units_that_come_free_soon(rows):
    # Beside one product of another stream that holds the compute units for some 45 us: a launch of 12 layers would wait 140 us before it went on with half of its
    # blocks, and gives the same bits with however many.
    from mini_llm_amd.ops import kernels as K

    rng = np.random.default_rng(rows)
    stack, given, _, _ = _stack(rng, 2, 768, 3072, [40] * rows, 64, B, "gelu_new", None)
    stack = K.DecodeStack(stack.layers * 6, rows, 12, 2e-5, 2e-5, 0.125, "gelu_new")
    out = stack.run(*given)
    assert stack.blocks_of_last() == stack.blocks
    x = torch.randn((2048, 1600), device=DEV).to(B)
    w = K.pack_matrix((0.02 * torch.randn((6400, 1600), device=DEV)).to(B))
    K.linear(x, w)
    streams, members = [torch.cuda.Stream(), torch.cuda.Stream()], []
    for _ in range(20):
        torch.cuda.synchronize()
        with torch.cuda.stream(streams[0]):
            K.linear(x, w)
        with torch.cuda.stream(streams[1]):
            here = stack.run(*given)
        torch.cuda.synchronize()
        members.append(stack.blocks_of_last())
        assert torch.equal(here, out)
    assert min(members) >= stack.blocks // 2, members


@pytest.mark.gpu
def test_rows_that_do_not_match_their_tables_are_refused():
    stack, given, _, _ = _stack(np.random.default_rng(2), 1, 64, 64, [3, 4], 64, B, "gelu_new", None)
    hidden, request, positions, slots, tables = given
    for wrong in ((hidden[:1], request, positions, slots, tables), (hidden, request[:1], positions, slots, tables), (hidden, request, positions[:1], slots, tables),
                  (hidden, request, positions, slots[:1], tables), (hidden, request, positions, slots, tables[:1])):
        with pytest.raises(ValueError):
            stack.run(*wrong)


@pytest.mark.gpu
@pytest.mark.parametrize("width,rows", [(768, 8), (1024, 2), (1024, 16), (512, 4), (192, 16)])
def test_32_bit_sums_are_no_further_off_than_layer_by_layer(tmp_path, monkeypatch, width, rows):
    # The relative error (2-norm) of a decode step's logits against 64 bits, over all rows of a few models: one kernel's sums run over as many products as the
    # separate kernels', in an order of their own, so that neither should be the further off.
    from mini_llm_amd.config import config_from_dict
    from mini_llm_amd.engine import StepEntry
    from mini_llm_amd.engine.engine import Engine, EngineOptions
    from mini_llm_amd.ops import kernels as K
    from mini_llm_amd.weights import write_model_dir

    raw = {"architectures": ["GPT2LMHeadModel"], "n_layer": 3, "n_embd": width, "n_head": width // 64, "n_inner": 4 * width, "vocab_size": 600, "n_positions": 64,
           "layer_norm_epsilon": 1e-5, "activation_function": "gelu_new"}
    errors = {True: [], False: []}
    for seed in range(3):
        folder = tmp_path / str(seed)
        write_model_dir(config_from_dict(raw), seed, folder)
        config, weights = P.load_model_dir(folder)
        rng = np.random.default_rng(seed)
        sequences = [rng.integers(0, 600, 24).tolist() for _ in range(rows)]
        want = np.stack([P.forward(config, weights, tokens)[-1] for tokens in sequences]).astype(np.float64)
        for one_kernel in (True, False):
            with monkeypatch.context() as patch:
                patch.setattr(K, "decode_stack_pays", lambda *sizes: one_kernel)
                engine = Engine(folder, EngineOptions(dtype="float32", max_sessions=rows))
                handles = [engine.try_take_cache() for _ in sequences]
                engine.runner.step([StepEntry(h, tokens[:-1], []) for h, tokens in zip(handles, sequences)])
                before = K.launch_counts()
                got = engine.runner.step([StepEntry(h, tokens[-1:], [0]) for h, tokens in zip(handles, sequences)]).double().cpu().numpy()
                assert ("decode_stack" in K.launches_since(before)) == one_kernel
                engine.close()
            errors[one_kernel].append(np.linalg.norm(got - want) / np.linalg.norm(want))
    assert np.mean(errors[True]) <= np.mean(errors[False]), errors
    assert np.mean(errors[True]) > 0.0
