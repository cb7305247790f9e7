"""Decode attention with more (batch, kv head) pairs than compute units: workgroups of four wavefronts, one per pair."""

import numpy as np
import pytest
import torch

from helpers import assert_attn_close, make_qkv, t2bits, t2f32

CUS = 256


def splits(B, KVH, S, HD):
    from custom_kernels import custom_kernels_extension as cke

    return cke.attention_num_splits(B, KVH, S, HD, CUS)


def test_lengths_that_take_one_workgroup_per_head():
    """One split up to each line, splits again beyond it (where the streaming form has several)."""
    for units, last in ((320, {64: 512, 128: 416}), (448, {64: 832, 128: 1024}), (512, {64: 1024, 128: 1024}), (576, {64: 512, 128: 480}),
                        (768, {64: 1024, 128: 1024}),
                        (896, {64: 448, 128: 416})):
        for HD in (64, 128):
            assert splits(units // 8, 8, last[HD], HD) == 1
            assert splits(units // 8, 8, last[HD] + 1, HD) > 1, (units, HD)
    # kv heads that do not fill whole rows stream in more splits: not where their partials would not fit the static scratch
    for KVH in (3, 5):
        for HD in (64, 128):
            assert splits(-(-513 // KVH), KVH, 1024, HD) == splits(575 // KVH, KVH, 1024, HD) == 1
    # a quarter of the device is not left alone with a long stream
    assert splits(64, 8, 1300, 64) == 3 and splits(112, 8, 1300, 64) == 2 and splits(128, 8, 1300, 64) == 1


# pairs either side of one, 5/4, 2, 3 and 4 per compute unit; lengths of one tile and less, of one and of more rounds of the four
# wavefronts with a ragged end, and the longest each takes; every head ratio
CASES = [(257, 1, 1), (33, 8, 16), (33, 8, 129), (33, 8, 384), (40, 8, 512), (41, 8, 257), (64, 8, 63), (64, 8, 255), (64, 8, 1000),
         (65, 8, 33), (65, 8, 300), (96, 8, 70), (96, 8, 1024), (97, 8, 65), (97, 8, 97), (128, 8, 380), (128, 8, 448), (140, 2, 700), (129, 8, 40),
         (65, 8, 384), (65, 8, 385)]


@pytest.mark.gpu
@pytest.mark.parametrize("HD", [64, 128])
@pytest.mark.parametrize("B,KVH,S", CASES)
def test_against_oracle(gpu, B, KVH, S, HD):
    from custom_kernels import custom_kernels_extension as cke
    from oracle import attention_decode_ref

    R = (1, 2, 3, 4, 8)[(B + S) % 5]
    print(f"many heads B={B} KVH={KVH} R={R} S={S} HD={HD} splits={splits(B, KVH, S, HD)}", flush=True)
    q, k, v = make_qkv(B, R * KVH, KVH, S, HD, seed=91, cache_len=S + 9)
    qg, kg, vg = make_qkv(B, R * KVH, KVH, S, HD, seed=91, cache_len=S + 9, device=gpu)
    out = cke.flash_attention_decode(qg, kg, vg)
    torch.cuda.synchronize()
    some = [0, 1, B // 2, B - 1]
    assert_attn_close(out[some], attention_decode_ref(t2f32(q[some]), t2f32(k[some]), t2f32(v[some])), what=f"B={B} S={S} HD={HD}")
    # every other sequence against the streaming form (partials of three splits and a combine)
    other = cke.flash_attention_decode(qg, kg, vg, 3)
    assert_attn_close(out, t2f32(other).astype(np.float64), what=f"against the streaming form B={B} S={S} HD={HD}", regression=False)


@pytest.mark.gpu
@pytest.mark.parametrize("HD", [64, 128])
@pytest.mark.parametrize("length", [1, 31, 64, 200, 256])
def test_length_on_the_device(gpu, length, HD):
    """The length of a recorded step: planned for the whole cache, whose other rows are not numbers."""
    from custom_kernels import custom_kernels_extension as cke
    from oracle import attention_decode_ref

    B, QH, KVH, S = 64, 32, 8, 256
    print(f"many heads, device length {length} HD={HD}", flush=True)
    q, k, v = make_qkv(B, QH, KVH, S, HD, seed=92, cache_len=S)
    ref = attention_decode_ref(t2f32(q[:2]), t2f32(k[:2, :, :length]), t2f32(v[:2, :, :length]))
    k[:, :, length:], v[:, :, length:] = float("nan"), float("nan")
    n = torch.tensor([length], dtype=torch.int32, device=gpu)
    out = cke.flash_attention_decode_devlen(q.to(gpu), k.to(gpu), v.to(gpu), n)
    torch.cuda.synchronize()
    assert_attn_close(out[:2], ref, what=f"device length {length}", regression=False)
    assert bool(torch.isfinite(out.float()).all())
    np.testing.assert_array_equal(t2bits(out), t2bits(cke.flash_attention_decode_devlen(q.to(gpu), k.to(gpu), v.to(gpu), n)))


@pytest.mark.gpu
@pytest.mark.parametrize("HD", [64, 128])
@pytest.mark.parametrize("B,S", [(33, 16), (33, 129), (40, 200), (48, 257), (64, 1), (64, 31), (64, 33), (64, 100), (64, 225), (64, 256),
                                 (64, 300), (64, 384), (64, 512)])
def test_bits_do_not_hang_on_the_batch(gpu, B, S, HD):
    """The sequences of a batch with more (batch, kv head) pairs than compute units have the bits that they have in batches
    with fewer, whose workgroups have eight wavefronts: a batch generates what its halves generate."""
    from custom_kernels import custom_kernels_extension as cke

    KVH = 8
    print(f"many heads, bits B={B} S={S} HD={HD}", flush=True)
    q, k, v = make_qkv(B, 4 * KVH, KVH, S, HD, seed=93, cache_len=S + 7, device=gpu)
    out = cke.flash_attention_decode(q, k, v)
    half = (B + 1) // 2
    parts = [cke.flash_attention_decode(q[i:i + half], k[i:i + half], v[i:i + half]) for i in range(0, B, half)]
    assert splits(B, KVH, S, HD) == splits(half, KVH, S, HD) == 1 and B * KVH > CUS >= half * KVH > CUS // 2
    np.testing.assert_array_equal(t2bits(out), np.concatenate([t2bits(p) for p in parts]))


@pytest.mark.gpu
@pytest.mark.parametrize("HD,cap", [(64, 256), (64, 512), (128, 256), (128, 512)])
def test_recorded_steps_have_the_bits_of_the_eager_ones(gpu, HD, cap):
    """A step that is planned for the whole cache and reads its length on the device, and one that is planned for its length."""
    from custom_kernels import custom_kernels_extension as cke

    q, k, v = make_qkv(64, 32, 8, cap, HD, seed=94, cache_len=cap, device=gpu)
    for S in (1, 40, 130, 200, cap - 1, cap):
        print(f"many heads, eager and recorded length {S} of {cap} HD={HD}", flush=True)
        n = torch.tensor([S], dtype=torch.int32, device=gpu)
        out = cke.flash_attention_decode_devlen(q, k, v, n)
        np.testing.assert_array_equal(t2bits(out), t2bits(cke.flash_attention_decode(q, k[:, :, :S], v[:, :, :S])))
