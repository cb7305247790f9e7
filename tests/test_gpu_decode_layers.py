"""GPU parity: all layers of a decode step in one launch (l3_decode_layers) against float32 arithmetic on the same bf16
weights, for every number of rows and at positions around the edges of its attention tiles (32 tokens, 256 per round of
a row's wavefronts), and the way back to the operators when a launch has reported a wait that ran out."""

import pytest
import torch

from helpers import randn_bf16

pytestmark = pytest.mark.gpu

C, H, QH, KVH, HD, EPS = 2048, 8192, 32, 8, 64, 1e-5


def _layers(gpu, n, batch, length):
    def w(seed, *shape):
        return randn_bf16(shape, seed, scale=0.02).to(gpu)

    return [dict(ln_1=(1 + w(i, C)), ln_2=(1 + w(i + 1, C)), c_attn=w(i + 2, (QH + 2 * KVH) * HD, C), c_proj=w(i + 3, C, C),
                 c_fc2=w(i + 4, H, C), c_fc=w(i + 5, H, C), mlp_proj=w(i + 6, C, H),
                 cache_k=randn_bf16((batch, length, KVH, HD), i + 7).to(gpu),
                 cache_v=randn_bf16((batch, length, KVH, HD), i + 8).to(gpu)) for i in range(0, 10 * n, 10)]


def _rotate(t, table):
    a, b = t[..., 0::2], t[..., 1::2]
    cos, sin = table[0::2], table[1::2]
    return torch.stack((a * cos - b * sin, a * sin + b * cos), -1).flatten(-2)


def _float32_step(x, layers, table, pos):
    """Hidden state behind the layers and the appended (key, value) rows, without any intermediate rounding."""
    x = x[:, 0].float()
    B, rows = x.shape[0], []
    for L in layers:
        def norm(t, w):
            return t * torch.rsqrt((t * t).mean(-1, keepdim=True) + EPS) * w.float()

        q, k, v = (norm(x, L["ln_1"]) @ L["c_attn"].float().t()).split([QH * HD, KVH * HD, KVH * HD], -1)
        q, k, v = _rotate(q.view(B, QH, HD), table[pos]), _rotate(k.view(B, KVH, HD), table[pos]), v.view(B, KVH, HD)
        rows.append((k, v))
        keys = torch.cat((L["cache_k"][:B, :pos].float(), k[:, None]), 1)
        values = torch.cat((L["cache_v"][:B, :pos].float(), v[:, None]), 1)
        score = (q.view(B, 1, KVH, QH // KVH, HD) * keys[:, :, :, None]).sum(-1) / HD ** 0.5
        y = (torch.softmax(score, 1)[..., None] * values[:, :, :, None]).sum(1).reshape(B, C)
        x = x + y @ L["c_proj"].float().t()
        h = norm(x, L["ln_2"])
        x = x + (torch.nn.functional.silu(h @ L["c_fc2"].float().t()) * (h @ L["c_fc"].float().t())) @ L["mlp_proj"].float().t()
    return x, rows


@pytest.mark.parametrize("B", [1, 2, 3, 4])
def test_decode_layers_against_float32(gpu, B):
    from custom_kernels import custom_kernels_extension as ops
    from llama_arch import precompute_freqs_cis

    layers = _layers(gpu, 2, B, 600)
    one_launch = ops.DecodeLayers(layers, B)
    table = precompute_freqs_cis(HD, 640, 500000.0, True, scale_factor=32.0, device=gpu)
    for pos in (0, 31, 32, 127, 256, 599):
        print(f"decode_layers B={B} pos={pos}", flush=True)
        x = randn_bf16((B, 1, C), 900 + pos).to(gpu)
        before = [(L["cache_k"].clone(), L["cache_v"].clone()) for L in layers]
        want, rows = _float32_step(x, layers, table, pos)
        y = one_launch(x, table, torch.tensor([pos], dtype=torch.int32, device=gpu), EPS)
        assert not one_launch.failed()
        # Per layer ten roundings to bf16 lie on the way (input norm, qkv, rotated q, attention weights and output, the two
        # products with their additions, second norm, gate, silu and up with their product), each off by at most
        # 2^-9 of its value and 2^-9 / sqrt(3) in the mean: sqrt(20) of those in two layers, 5.1e-3 of the result.
        tol = 3 * 20 ** 0.5 * 2.0 ** -9 / 3 ** 0.5
        assert (y[:, 0].float() - want).norm() <= tol * want.norm()
        for L, (k0, v0), (k, v) in zip(layers, before, rows):
            for cache, old, new in ((L["cache_k"], k0, k), (L["cache_v"], v0, v)):
                assert (cache[:, pos].float() - new).norm() <= tol * new.norm()
                cache[:, pos] = old[:, pos]
                assert torch.equal(cache, old)      # nothing but the appended row has changed
        # the same from an embedding whose rows tokens with a stride pick, the first and the last row among them
        rows = 27 - 9 * torch.arange(B, device=gpu)
        embedding = randn_bf16((28, C), 901).to(gpu)
        embedding[rows] = x[:, 0]
        tokens = torch.full((B, 5), 10 ** 9, device=gpu)
        tokens[:, 2] = rows
        assert torch.equal(one_launch.from_tokens(tokens[:, 2:3], embedding, table, torch.tensor([pos], dtype=torch.int32, device=gpu),
                                                  EPS), y)


# (rows, position): around the tiles of 32 tokens and the rounds of a row's wavefronts, and the last position of the longest
# cache for which the decode step is used (rows x length = 4096)
@pytest.mark.parametrize("B,pos", [(1, 31), (1, 32), (1, 255), (1, 256), (1, 4095), (2, 130), (2, 2047), (3, 96), (3, 1364), (4, 65), (4, 1023)])
def test_every_edge_token_counts(gpu, B, pos):
    """Attention of the one launch with a handful of tokens, at every kind of edge, that share nearly all of the weight and
    carry large values of their own: attending to one of them less (checked in the float32 reference) moves the result by far
    more than the bound.  The appended token is one of them."""
    from custom_kernels import custom_kernels_extension as ops
    from llama_arch import LlamaDecoder, precompute_freqs_cis

    assert B * (pos + 1) <= LlamaDecoder.ONE_LAUNCH_MAX_POSITIONS
    L = _layers(gpu, 1, B, pos + 1)[0]
    table = precompute_freqs_cis(HD, pos + 1, 500000.0, True, scale_factor=32.0, device=gpu)
    x = randn_bf16((B, 1, C), 950 + pos).to(gpu)
    # a key head's weights are those of its query heads together, so that the appended key points where the queries point
    rep = QH // KVH
    w_q = L["c_attn"][:QH * HD].float().view(KVH, rep, HD, C)
    L["c_attn"][QH * HD:(QH + KVH) * HD] = w_q.sum(1).reshape(KVH * HD, C).to(torch.bfloat16)
    h = x[:, 0].float()
    h = h * torch.rsqrt((h * h).mean(-1, keepdim=True) + EPS) * L["ln_1"].float()
    key = _rotate((h @ L["c_attn"][QH * HD:(QH + KVH) * HD].float().t()).view(B, KVH, HD), table[pos])
    edges = sorted({t for t in (0, 31, 32, 127, 128, 255, 256, pos // 2, pos - 1) if 0 <= t < pos})
    L["cache_k"][:, edges] = (key[:, None] + 0.05 * randn_bf16((B, len(edges), KVH, HD), 951).to(gpu)).to(torch.bfloat16)
    L["cache_v"][:, edges] = randn_bf16((B, len(edges), KVH, HD), 952, scale=6.0).to(gpu)
    # The appended value joins them: its weights are larger too.
    L["c_attn"][(QH + KVH) * HD:] *= 6
    # all keys larger, so that those few tokens have the weight of thousands
    gain = 2.0
    L["c_attn"][QH * HD:(QH + KVH) * HD] *= gain
    L["cache_k"][:, edges] *= gain
    want, _ = _float32_step(x, [L], table, pos)

    # Ten roundings lie on the way in a layer (as above), each off by 2^-9 / sqrt(3) in the mean.  A score is the sum of HD
    # products of a query and a key that have been rounded twice each, four such roundings of its terms, whose root sum of
    # squares is `spread`; the weights of the few tokens are off by as much, and attention's part of the result with them.
    # All of it independent, and rows differ: twice the mean.
    q = _rotate((h @ L["c_attn"][:QH * HD].float().t()).view(B, KVH, rep, HD), table[pos])
    spread2 = (q * (gain * key)[:, :, None]).pow(2).sum(-1).mean().item() / HD
    tol = 2 * 2.0 ** -9 / 3 ** 0.5 * (10 + 4 * spread2) ** 0.5
    scale = want.norm(dim=-1)

    def without(t, head):
        """The reference with no weight on token t for the query heads of one key head: what one XCD could get wrong."""
        kept = dict(L)
        if t == pos:
            rows = slice((QH + head) * HD, (QH + head + 1) * HD)
            kept["c_attn"] = L["c_attn"].clone()
            kept["c_attn"][rows] *= -1
        else:
            kept["cache_k"] = L["cache_k"].clone()
            kept["cache_k"][:, t, head] *= -1
        return _float32_step(x, [kept], table, pos)[0]

    print(f"decode_layers edges B={B} pos={pos} tol={tol:.4f}", flush=True)
    for t in edges + [pos]:
        assert ((without(t, t % KVH) - want).norm(dim=-1) > 1.5 * tol * scale).all(), t
    one_launch = ops.DecodeLayers([L], B)
    y = one_launch(x, table, torch.tensor([pos], dtype=torch.int32, device=gpu), EPS)
    assert not one_launch.failed()
    off = ((y[:, 0].float() - want).norm(dim=-1) / scale).max().item()
    print(f"  off by {off:.4f}", flush=True)
    assert off <= tol


def test_one_launch_up_to_its_last_position_and_no_further(gpu):
    from custom_kernels import custom_kernels_extension as ops
    from llama_arch import LlamaConfig, LlamaDecoder

    m = LlamaDecoder(LlamaConfig(n_layer=1, vocab_size=512, max_model_len=4200, max_gen_batch_size=5), ops, gpu)
    for rows, most in ((1, 4096), (2, 2048), (3, 1365), (4, 1024)):
        assert m._one_launch(rows, most) is not None and m._one_launch(rows, most + 1) is None
    assert m._one_launch(5, 8) is None


def _handed_over(one_launch, rows, n_layer):
    """The words that the workgroups of an XCD have handed each other, (layer, XCD, word), from the workspace: residual rows
    (written from the second layer on), rows behind c_proj, q | k | v, hidden units."""
    words = one_launch.workspace.view(torch.int32)[8192 // 4 + 2 * 8 * rows * C * 2:].cpu()
    return words.view(n_layer, 8, rows * (2 * C + (QH // KVH + 2) * HD + H // 8))


@pytest.mark.parametrize("B", [1, 4])
def test_handed_over_words_name_their_launch_and_the_xcd_that_wrote_them(gpu, B):
    """... so that what a workgroup behind another L2 wrote is never taken (its K/V row among it, whose arrival only these words
    tell); also where the launch number leaves its bits of the tag."""
    from custom_kernels import custom_kernels_extension as ops
    from llama_arch import precompute_freqs_cis

    layers = _layers(gpu, 2, B, 64)
    one_launch = ops.DecodeLayers(layers, B)
    table = precompute_freqs_cis(HD, 64, 500000.0, True, scale_factor=32.0, device=gpu)
    x, pos = randn_bf16((B, 1, C), 910).to(gpu), torch.tensor([40], dtype=torch.int32, device=gpu)
    first = one_launch(x, table, pos, EPS)
    for before in (1, 4094, 4095, 4096, 65534, 65535, 65536):
        one_launch.workspace.view(torch.int32)[64] = before              # launches so far
        print(f"decode_layers B={B} launch {before + 1}", flush=True)
        assert torch.equal(one_launch(x, table, pos, EPS), first) and not one_launch.failed()
        tags = _handed_over(one_launch, B, 2) & 0xffff
        assert torch.equal(tags[1], tags[1, :, :1].expand_as(tags[1])) and torch.equal(tags[0, :, B * C:], tags[1, :, B * C:])
        assert (tags[1] >> 4 == (before + 1) % 4096).all()
        assert sorted((tags[1, :, 0] & 15).tolist()) == list(range(8))


@pytest.mark.parametrize("B", [1, 2, 4])
def test_generation_by_the_one_launch_and_by_the_operators(gpu, B):
    """The same tokens, and keys and values as near as two orders of the sums leave them.  The embedding is wide, so that the
    pick does not hang on the last bit of a logit."""
    from custom_kernels import custom_kernels_extension as ops
    from llama_arch import LlamaConfig, LlamaDecoder, random_prompts

    m = LlamaDecoder(LlamaConfig(n_layer=4, vocab_size=4096, max_model_len=48, max_gen_batch_size=B), ops, gpu)
    m.wte = randn_bf16((4096, C), 77).to(gpu)
    prompts = random_prompts(B, 16, 4096, 5)
    if B > 1:
        prompts[1] = prompts[1][:9]       # (prompt tokens through the decode step)
    for generate in (m.generate, m.generate_graphed):
        results = []
        for m._layers_in_one_launch in (True, False):
            m._graphs.clear()
            tokens = generate(prompts, 16, ignore_eos=True)
            results.append((tokens, [L[n][:, :31].float() for L in m.layers for n in ("cache_k", "cache_v")]))
        (tokens, one), (tokens_op, by_operators) = results
        assert tokens == tokens_op and B in m._layer_launches and not m._layer_launches[B].failed()
        # ten roundings per layer on either side, up to the layer in question
        for i, (a, b) in enumerate(zip(one, by_operators)):
            tol = 3 * (2 * 10 * (i // 2 + 1)) ** 0.5 * 2.0 ** -9 / 3 ** 0.5
            assert ((a - b).norm(dim=(-1, -2)) <= tol * b.norm(dim=(-1, -2))).all(), (i, tol)


def test_generation_without_the_one_launch_after_a_wait_ran_out(gpu):
    from custom_kernels import custom_kernels_extension as ops
    from llama_arch import LlamaConfig, LlamaDecoder, random_prompts

    m = LlamaDecoder(LlamaConfig(n_layer=2, vocab_size=4096, max_model_len=48, max_gen_batch_size=2), ops, gpu)
    prompts = random_prompts(2, 16, 4096, 5)
    for generate in (m.generate, m.generate_graphed):
        m._layers_in_one_launch = True
        first = generate(prompts, 16, ignore_eos=True)
        assert m._layers_in_one_launch and not m._layer_launches[2].failed()
        with torch.inference_mode():
            m._layer_launches[2].workspace[0] = 1       # what a launch leaves when a wait has run out
        again = generate(prompts, 16, ignore_eos=True)
        assert not m._layers_in_one_launch
        assert again == generate(prompts, 16, ignore_eos=True)
        assert len(first[0]) == len(again[0]) == 16


@pytest.mark.parametrize("name", ["c_attn", "c_proj", "c_fc", "mlp_proj", "wte", "cache_k"])
def test_weights_that_only_the_operators_take_are_left_to_them(gpu, name):
    """Rows with a padded stride (in one layer, in the embedding, in the cache): the operators take them, so generation does."""
    from custom_kernels import custom_kernels_extension as ops
    from llama_arch import LlamaConfig, LlamaDecoder, random_prompts

    m = LlamaDecoder(LlamaConfig(n_layer=2, vocab_size=4096, max_model_len=48, max_gen_batch_size=2), ops, gpu)
    prompts = random_prompts(2, 16, 4096, 5)
    assert m._one_launch(2, 32) is not None
    m._layers_in_one_launch = False
    want = m.generate(prompts, 16, ignore_eos=True)
    m._layers_in_one_launch = True

    def padded(t):
        wide = torch.zeros(t.shape[:-1] + (t.shape[-1] + 64,), dtype=t.dtype, device=t.device)[..., :t.shape[-1]]
        return wide.copy_(t)

    if name == "wte":
        m.wte = padded(m.wte)
    elif name == "cache_k":
        for n in ("cache_k", "cache_v"):
            m.layers[1][n] = torch.zeros((2, 96) + m.layers[1][n].shape[2:], dtype=torch.bfloat16, device=gpu)[:, :48]
    elif name == "c_fc":
        for n in ("c_fc", "c_fc2"):     # (a pair has one stride)
            m.layers[1][n] = padded(m.layers[1][n])
    else:
        m.layers[1][name] = padded(m.layers[1][name])
    print(f"operators for a strided {name}", flush=True)
    assert m._one_launch(2, 32) is None
    assert m.generate(prompts, 16, ignore_eos=True) == want
    graphed = m.generate_graphed(prompts, 16, ignore_eos=True)
    # (the loops plan the attention splits differently, a near tie may fork a stream)
    assert all(a[:8] == b[:8] for a, b in zip(graphed, want))


def test_a_token_outside_the_vocabulary_is_refused(gpu):
    """In a prompt that reaches past the common prefix the decode step looks it up, not the prompt pass."""
    from custom_kernels import custom_kernels_extension as ops
    from llama_arch import LlamaConfig, LlamaDecoder, random_prompts

    m = LlamaDecoder(LlamaConfig(n_layer=2, vocab_size=4096, max_model_len=48, max_gen_batch_size=2), ops, gpu)
    good = random_prompts(2, 16, 4096, 5)
    assert m._one_launch(2, 33) is not None
    for generate in (m.generate, m.generate_graphed):
        for bad in (4096, -1):
            with pytest.raises(IndexError):
                generate([good[0], good[1] + [bad]], 16, ignore_eos=True)
        assert len(generate([good[0], good[1] + [4095]], 16, ignore_eos=True)[1]) == 16      # (padded with 128004)


def test_the_one_launch_comes_back_after_a_wait_ran_out(gpu):
    """A failure is told, costs the generation after it the launch, and each further one in a row twice as many."""
    from custom_kernels import custom_kernels_extension as ops
    from llama_arch import LlamaConfig, LlamaDecoder, random_prompts

    m = LlamaDecoder(LlamaConfig(n_layer=2, vocab_size=4096, max_model_len=48, max_gen_batch_size=2), ops, gpu)
    prompts = random_prompts(2, 16, 4096, 5)

    def failing(generate):
        launch = m._one_launch(2, 32)
        with torch.inference_mode():
            launch.workspace[0] = 1
        with pytest.warns(RuntimeWarning, match="one by one"):
            return generate(prompts, 16, ignore_eos=True)

    for generate in (m.generate, m.generate_graphed):
        first = generate(prompts, 16, ignore_eos=True)
        assert 2 in m._layer_launches
        for rests in (1, 2, 4):
            by_operators = failing(generate)
            for _ in range(rests):
                assert m._one_launch(2, 32) is None
                assert generate(prompts, 16, ignore_eos=True) == by_operators
            assert m._one_launch(2, 32) is not None
        assert generate(prompts, 16, ignore_eos=True) == first and 2 in m._layer_launches
        assert m._one_launch_failures == 0
    assert "l3_decode_layers" in m.decode_route(2, 32) and "given up 6 times" in m.decode_route(2, 32)
    assert "l3_decode_layers" not in m.decode_route(2, 2049)
    key, loop = next(iter(m._graphs.items()))
    assert key == (2, 32) and loop.layers is m._layer_launches[2]
