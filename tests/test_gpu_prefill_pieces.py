"""Causal prefill of a few queries behind many cached tokens: the launch is cut into pieces of rows x tokens, and a
second launch adds them up (l3_attn_prefill_ws)."""

import numpy as np
import pytest
import torch

from helpers import assert_attn_close, randn_bf16, t2bits, t2f32


def cut_bytes(B, QH, KVH, T, S, HD):
    from custom_kernels import _l3lib

    return _l3lib.load().l3_attn_prefill_workspace_bytes(B, QH, KVH, T, S, HD, 0)


def make(B, QH, KVH, T, S, HD, gain=1.0, head_major=False):
    q = randn_bf16((B, T, QH, HD), 301, scale=gain)
    k, v = randn_bf16((B, S + 5, KVH, HD), 302), randn_bf16((B, S + 5, KVH, HD), 303)

    def view(t, dev):
        t = t.to(dev)[:, :S].transpose(1, 2)
        return t.contiguous() if head_major else t

    return lambda dev: (q.to(dev).transpose(1, 2), view(k, dev), view(v, dev))


# 12 tiles are the fewest that are cut; lengths either side of a tile's edge; queries either side of a block's edge, for every
# head ratio; blocks of one and of two column blocks; pieces that begin where some of a wavefront's columns see nothing
SHAPES = [(1, 8, 1, 1, 705, 64), (1, 32, 8, 8, 768, 64), (2, 32, 8, 16, 1023, 64), (1, 24, 8, 21, 1025, 64), (1, 8, 8, 65, 1000, 64),
          (1, 16, 8, 63, 2049, 64), (3, 16, 2, 40, 1500, 64), (1, 32, 8, 200, 1216, 64), (8, 32, 8, 64, 2600, 64),
          (1, 4, 2, 3, 5000, 64)]


def test_which_calls_are_cut():
    for B, QH, KVH, T, S, HD in SHAPES:
        assert cut_bytes(B, QH, KVH, T, S, HD) > 0
        assert cut_bytes(B, QH, KVH, T, S, 128) > 0
    for B, QH, KVH, T, S, HD in [(1, 32, 8, 8, 704, 64), (1, 32, 8, 512, 1000, 64), (2, 32, 8, 1531, 1531, 64), (64, 32, 8, 128, 128, 64),
                                 (16, 32, 8, 512, 1100, 128), (1, 32, 8, 8, 4096, 96), (1, 32, 8, 8, 7, 64)]:
        assert cut_bytes(B, QH, KVH, T, S, HD) == 0
    # a range (of one token, read over and over through a zero stride, it fits) whose tiles x pieces overflow 32 bits
    assert cut_bytes(1, 8, 1, 8, 1 << 30, 64) > 0 and 127 * ((1 << 30) // 64) < 2 ** 31
    for S in ((1 << 30) + 1, 1_200_000_000, 2 ** 31 - 1):
        assert cut_bytes(1, 8, 1, 8, S, 64) == 0
    from custom_kernels import _l3lib

    for flag in (_l3lib.L3_ATTN_FLAG_PREFILL_WAVE, _l3lib.L3_ATTN_FLAG_PREFILL_TILED):      # a forced form is never cut
        assert _l3lib.load().l3_attn_prefill_workspace_bytes(1, 32, 8, 8, 4096, 64, flag) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("HD", [64, 128])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s[:5])))
def test_against_oracle(gpu, shape, HD):
    from custom_kernels import custom_kernels_extension as cke
    from oracle import attention_prefill_ref

    B, QH, KVH, T, S, _ = shape
    print(f"prefill pieces B={B} QH={QH} KVH={KVH} T={T} S={S} HD={HD}", flush=True)
    inputs = make(B, QH, KVH, T, S, HD)
    out = cke.flash_attention_prefill(*inputs(gpu))
    torch.cuda.synchronize()
    assert_attn_close(out, attention_prefill_ref(*(t2f32(t) for t in inputs("cpu"))), what=f"pieces {shape} HD={HD}")
    again = cke.flash_attention_prefill(*inputs(gpu))
    np.testing.assert_array_equal(t2bits(out), t2bits(again))
    dense = cke.flash_attention_prefill(*make(B, QH, KVH, T, S, HD, head_major=True)(gpu))      # other strides
    np.testing.assert_array_equal(t2bits(out), t2bits(dense))


@pytest.mark.gpu
@pytest.mark.parametrize("B,T,S,HD", [(1, 512, 7012, 64), (1, 512, 7012, 128), (1, 1400, 8000, 128), (1, 1500, 6600, 64), (16, 64, 6564, 64)])
def test_against_the_uncut_kernel(gpu, B, T, S, HD):
    """The largest shapes that are cut, with scores spread over many powers of two: both against the same float64 rows."""
    from custom_kernels import custom_kernels_extension as cke
    from oracle import attention_prefill_ref

    assert cut_bytes(B, 32, 8, T, S, HD) > 0
    print(f"prefill pieces against the uncut kernel B={B} T={T} S={S} HD={HD}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(5)
    q = torch.empty(B, T, 32, HD, dtype=torch.bfloat16, device=gpu).normal_(0, 3, generator=g).transpose(1, 2)
    k, v = (torch.empty(B, S, 8, HD, dtype=torch.bfloat16, device=gpu).normal_(0, 1, generator=g).transpose(1, 2) for _ in range(2))
    out = cke.flash_attention_prefill(q, k, v)
    with cke.attention_flags(prefill="tiled"):
        uncut = cke.flash_attention_prefill(q, k, v)
    torch.cuda.synchronize()
    for i in (0, 31, 32, 33, T // 2, T - 1):
        n = S - T + i + 1
        ref = attention_prefill_ref(t2f32(q[-1:, :, i:i + 1].cpu()), t2f32(k[-1:, :, :n].cpu()), t2f32(v[-1:, :, :n].cpu()))
        for o, name in ((out, "cut"), (uncut, "uncut")):
            assert_attn_close(o[-1:, :, i:i + 1], ref, what=f"{name} row {i}", regression=False)
    # two bf16 roundings of results that differ by float32 sums in another order and bf16 weights against another reference
    # (2^-9 of the result each): two units in the last place of the largest value
    assert float((out.float() - uncut.float()).abs().max()) <= 2.0 ** -6 * float(uncut.float().abs().max())


@pytest.mark.gpu
def test_recorded_and_on_streams(gpu):
    """The bits are the eager call's, on every replay, every stream and the first call that allocates there."""
    from custom_kernels import custom_kernels_extension as cke

    q, k, v = make(1, 32, 8, 40, 3000, 64)(gpu)
    ref = t2bits(cke.flash_attention_prefill(q, k, v))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = cke.flash_attention_prefill(q, k, v)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(t2bits(out), ref)
        np.testing.assert_array_equal(t2bits(cke.flash_attention_prefill(q, k, v)), ref)
    streams = [torch.cuda.Stream() for _ in range(3)]
    outs = []
    for _ in range(4):
        for s in streams:
            s.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(s):
                outs.append(cke.flash_attention_prefill(q, k, v))
    torch.cuda.synchronize()
    for o in outs:
        np.testing.assert_array_equal(t2bits(o), ref)


@pytest.mark.gpu
def test_a_nan_key(gpu):
    """It reaches the rows that see it and no other."""
    from custom_kernels import custom_kernels_extension as cke

    q, k, v = make(1, 8, 2, 24, 2000, 64)(gpu)
    clean = cke.flash_attention_prefill(q, k, v)
    k = k.clone()
    k[0, 0, 1990] = float("nan")
    out = cke.flash_attention_prefill(q, k, v)
    torch.cuda.synchronize()
    assert torch.equal(out[:, 4:], clean[:, 4:])                    # the other kv head's
    first = 1990 - (2000 - 24)                                      # the first query that sees it
    # (columns of a wavefront follow a new maximum together, so a neighbour's may move the last bit)
    assert float((out[:, :4, :first].float() - clean[:, :4, :first].float()).abs().max()) <= 2.0 ** -7 * float(clean.float().abs().max())
    assert bool(out[:, :4, first:].isnan().all())


@pytest.mark.gpu
@pytest.mark.parametrize("at", [1, 700, 1990])
@pytest.mark.parametrize("HD", [64, 128])
def test_an_infinite_key(gpu, HD, at):
    """Scores of +inf make their rows NaN, as without pieces; those of -inf weigh nothing, also against the pieces' own reference."""
    from custom_kernels import custom_kernels_extension as cke
    from oracle import attention_prefill_ref

    q, k, v = make(1, 8, 2, 24, 2000, HD)(gpu)
    assert cut_bytes(1, 8, 2, 24, 2000, HD) > 0
    k = k.clone()
    k[0, 0, at, 3] = float("inf")
    out = cke.flash_attention_prefill(q, k, v)
    with cke.attention_flags(prefill="tiled"):
        uncut = cke.flash_attention_prefill(q, k, v)
    sees = torch.arange(24, device=gpu) + 2000 - 24 >= at
    plus = (q[0, :4, :, 3] > 0) & sees                               # of the kv head's four query heads
    assert torch.equal(out[0, :4].isnan().all(-1), plus) and torch.equal(out[0, :4].isnan().any(-1), plus)
    assert torch.equal(uncut.isnan(), out.isnan()) and bool(plus.any()) and not bool(plus.all())
    k[0, 0, at] = 0.0
    k[0, 0, at, 3] = -3.0e38                                         # finite, and as good as -inf for the rows that are left
    q[0, :4, :, 3] = q[0, :4, :, 3].abs()
    ref = attention_prefill_ref(*(t2f32(t.cpu()) for t in (q, k, v)))
    low = cke.flash_attention_prefill(q, k, v)
    assert_attn_close(low, ref, what=f"a key of no weight at {at} HD={HD}", min_kv_len=1976)


@pytest.mark.gpu
@pytest.mark.parametrize("B,QH,KVH,T,S,HD", [(1, 32, 8, 8, 4096, 64), (1, 24, 8, 21, 1025, 64), (1, 8, 8, 65, 1000, 128), (1, 32, 8, 512, 7012, 64),
                                             (1, 16, 4, 2016, 4032, 128), (1, 32, 8, 1400, 8000, 128)])
def test_pieces_stay_in_the_workspace(gpu, B, QH, KVH, T, S, HD):
    """Through the C ABI on exactly the bytes that it asks for: nothing is written before or behind them, and the bits are the
    operator's.  Blocks of one and of two column blocks, some blocks cut and others not (2016 of 4032), up to five pieces per
    compute unit (1400 of 8000)."""
    from custom_kernels import _l3lib, custom_kernels_extension as cke

    print(f"prefill workspace B={B} QH={QH} KVH={KVH} T={T} S={S} HD={HD}", flush=True)
    lib, g = _l3lib.load(), torch.Generator(device=gpu).manual_seed(6)
    q = torch.empty(B, T, QH, HD, dtype=torch.bfloat16, device=gpu).normal_(0, 1, generator=g).transpose(1, 2)
    k, v = (torch.empty(B, S, KVH, HD, dtype=torch.bfloat16, device=gpu).normal_(0, 1, generator=g).transpose(1, 2) for _ in range(2))
    want = cke.flash_attention_prefill(q, k, v)
    n, guard = cut_bytes(B, QH, KVH, T, S, HD), 1 << 20
    assert n > 0
    ws = torch.full((guard + n + guard,), 0xa5, dtype=torch.uint8, device=gpu)
    out = torch.full_like(want, float("nan"))
    strides = lambda t: _l3lib.i64_array(t.stride()[:3])  # noqa: E731
    rc = lib.l3_attn_prefill_ws(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), ws.data_ptr() + guard, n, B, QH, KVH, T, S, HD,
                                strides(q), strides(k), strides(v), strides(out), 1.0 / HD ** 0.5, 0,
                                torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    torch.cuda.synchronize()
    assert bool((ws[:guard] == 0xa5).all()) and bool((ws[guard + n:] == 0xa5).all())
    np.testing.assert_array_equal(t2bits(out), t2bits(want))


@pytest.mark.gpu
def test_without_memory_for_the_pieces(gpu):
    """A call that was served without a buffer is still served when there is none to be had: it is not cut."""
    from custom_kernels import custom_kernels_extension as cke

    q, k, v = make(1, 32, 8, 512, 7000, 64)(gpu)
    cut = cke.flash_attention_prefill(q, k, v)
    with cke.attention_flags(prefill="tiled"):
        want = cke.flash_attention_prefill(q, k, v)
    torch.cuda.synchronize()
    room = torch.empty_like(want)
    torch.cuda.empty_cache()
    print("prefill with the allocator at its limit", flush=True)
    held = []
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (64 << 20)) / torch.cuda.get_device_properties(0).total_memory)
    try:
        try:
            while True:
                held.append(torch.empty(8 << 20, dtype=torch.uint8, device=gpu))
        except torch.OutOfMemoryError:
            pass
        assert cut_bytes(1, 32, 8, 512, 7000, 64) > 8 << 20
        del room                                       # of the result, and of nothing larger
        out = cke.flash_attention_prefill(q, k, v)
        torch.cuda.synchronize()
        with pytest.raises(torch.OutOfMemoryError):
            torch.empty(cut_bytes(1, 32, 8, 512, 7000, 64), dtype=torch.uint8, device=gpu)
    finally:
        held.clear()
        torch.cuda.set_per_process_memory_fraction(1.0)
    np.testing.assert_array_equal(t2bits(out), t2bits(want))
    np.testing.assert_array_equal(t2bits(cke.flash_attention_prefill(q, k, v)), t2bits(cut))
    assert not torch.equal(cut, want)                  # (the two forms differ in their last bits, so the test sees which ran)
