"""GPU parity: the linear whose workgroups share the activations through LDS (l3_linear_wide), against the
float64 oracle at the edges of its tiles: every count of 16-row activation blocks and one row either side, weight
rows that end inside a workgroup (64, or 128 where the matrix fills the device), k ranges shorter than the ring
of stages, one stage longer, and long ones."""

import pytest
import torch

from helpers import randn_bf16, t2f32
from oracle import linear_ref, swiglu_linear_ref
from test_gpu_linear import assert_linear_close

pytestmark = pytest.mark.gpu

# (rows, N, K); from 32768 weight rows on the tile is turned in LDS and stored in whole lines
SHAPES = [(1, 8, 128), (15, 72, 256), (16, 64, 384), (17, 136, 512), (32, 56, 640), (33, 200, 128), (48, 264, 1152),
          (49, 64, 256), (64, 1000, 4096), (5, 16392, 256), (64, 16392, 384), (1, 32768, 128), (16, 32776, 256),
          (31, 32840, 384), (64, 33000, 256)]


def _wide(x, w, up, res):
    from custom_kernels import _l3lib

    M, K, N = x.shape[0], x.shape[1], w.shape[0]
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=x.device)
    rc = _l3lib.load().l3_linear_wide(x.data_ptr(), w.data_ptr(), up.data_ptr() if up is not None else None,
                                      res.data_ptr() if res is not None else None, y.data_ptr(), M, N, K, x.stride(0),
                                      w.stride(0), N, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, rc
    torch.cuda.synchronize()
    return y


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_linear_wide_against_oracle(gpu, M, N, K):
    print(f"linear_wide M={M} N={N} K={K}", flush=True)
    x = randn_bf16((M, K), 201).to(gpu)
    w = randn_bf16((N, K + 8), 202, scale=0.05).to(gpu)[:, :K]         # rows with a padded stride
    y = _wide(x, w, None, None)
    assert_linear_close(y, linear_ref(t2f32(x), t2f32(w)), f"wide {M}x{N}x{K}")
    res = randn_bf16((M, N), 203, scale=3.0).to(gpu)
    assert torch.equal(_wide(x, w, None, res), res + y)                # torch's bf16 add: float sum, one rounding


@pytest.mark.parametrize("M,N,K", [(1, 4, 128), (16, 36, 384), (17, 60, 256), (33, 100, 512), (64, 1684, 1024), (64, 8200, 256)])
def test_linear_wide_swiglu_against_oracle(gpu, M, N, K):
    print(f"linear_wide swiglu M={M} N={N} K={K}", flush=True)
    x = randn_bf16((M, K), 211).to(gpu)
    wg = randn_bf16((N, K), 212, scale=0.05).to(gpu)
    wu = randn_bf16((N, K), 213, scale=0.05).to(gpu)
    y = _wide(x, wg, wu, None)
    # The oracle rounds gate, silu and up where the kernel does.  A factor whose float32 sum straddles a bf16 boundary may
    # round the other way: one ulp (2^-7 at most) of the product for each of gate, silu and up, and half an ulp of its own.
    ref = torch.from_numpy(swiglu_linear_ref(t2f32(x), t2f32(wg), t2f32(wu)))
    err = (y.double().cpu() - ref).abs()
    assert (err <= 3.5 * 2.0 ** -7 * ref.abs() + 2.0 ** -18 * ref.abs().max()).all(), err.max().item()
    res = randn_bf16((M, N), 214, scale=3.0).to(gpu)
    assert torch.equal(_wide(x, wg, wu, res), res + y)


@pytest.mark.parametrize("B,NH,KVH,HD,K", [(1, 4, 1, 8, 128), (16, 32, 8, 64, 2048), (17, 6, 2, 72, 1152), (33, 8, 2, 128, 640),
                                           (48, 4, 4, 64, 384), (49, 32, 8, 64, 1024), (64, 32, 8, 64, 2048)])
def test_linear_qkv_rope_append_rows_against_oracle(gpu, B, NH, KVH, HD, K):
    from custom_kernels import custom_kernels_extension as cke
    from custom_kernels import precompute_freqs_cis

    print(f"linear_qkv_rope_append_rows B={B} NH={NH} KVH={KVH} HD={HD} K={K}", flush=True)
    L, at = 40, 17
    x = randn_bf16((B, K), 221).to(gpu)
    w = randn_bf16(((NH + 2 * KVH) * HD, K + 8), 222, scale=0.05).to(gpu)[:, :K]
    table = precompute_freqs_cis(HD, 64, 500000.0, True, scale_factor=32.0, device=gpu)
    before_k, before_v = randn_bf16((B + 1, L, KVH, HD), 223).to(gpu), randn_bf16((B + 1, L, KVH, HD), 224).to(gpu)
    k, v = before_k.clone(), before_v.clone()
    q = cke.linear_qkv_rope_append_rows(x.view(B, 1, K), w, table, k, v, torch.tensor([at], dtype=torch.int32, device=gpu), NH)
    assert q.shape == (B, 1, NH, HD)
    ref = linear_ref(t2f32(x), t2f32(w)).reshape(B, NH + 2 * KVH, HD)
    assert_linear_close(v[:B, at].reshape(B, -1), ref[:, NH + KVH:].reshape(B, -1), "values")
    # A sum that straddles a bf16 boundary may round the other way, one ulp (2^-7 at most) of each of the two values that a
    # rotation adds up, and the result is rounded once (2^-8); sums that cancel as in assert_linear_close.
    c, s = (table[at, i::2].double().cpu().numpy() for i in (0, 1))
    r = ref[:, :NH + KVH].astype("float64")
    a, b = r[..., 0::2], r[..., 1::2]
    got = torch.cat((q[:, 0], k[:B, at]), 1).double().cpu().numpy()
    slack = 2.0 ** -17 * abs(ref).max()
    for y, want, size in ((got[..., 0::2], a * c - b * s, abs(a * c) + abs(b * s)), (got[..., 1::2], a * s + b * c, abs(a * s) + abs(b * c))):
        assert (abs(y - want) <= (2.0 ** -7 + 2.0 ** -8) * size + slack).all()
    # nothing else is written, and nothing at all at a position outside the cache
    k[:B, at], v[:B, at] = before_k[:B, at], before_v[:B, at]
    cke.linear_qkv_rope_append_rows(x.view(B, 1, K), w, table, k, v, torch.tensor([L], dtype=torch.int32, device=gpu), NH)
    assert torch.equal(k, before_k) and torch.equal(v, before_v)


@pytest.mark.parametrize("M,N,K,ksplit", [(1, 8, 128, 1), (3, 24, 1152, 3), (17, 8, 640, 2), (2, 8, 1280, 8)])
@pytest.mark.parametrize("far", ["x", "w", "both"])
def test_linear_splitk_of_rows_far_apart(gpu, M, N, K, ksplit, far):
    """Rows more than 2^28 elements apart (activations picked out of a long context, say): the library's entry point takes
    them, with splits that get no k among them, and so do the operators."""
    from custom_kernels import _l3lib
    from custom_kernels import custom_kernels_extension as cke

    print(f"linear_splitk far={far} M={M} N={N} K={K} ksplit={ksplit}", flush=True)

    def rows(values, apart):
        t = torch.empty((values.shape[0] - 1) * apart + K, dtype=torch.bfloat16, device=gpu)
        return t.as_strided(values.shape, (apart, 1)).copy_(values)

    xv, wv = randn_bf16((M, K), 231), randn_bf16((N, K), 232, scale=0.05)
    x = rows(xv, (1 << 28) + 8) if far != "w" else xv.to(gpu)
    w = rows(wv, (1 << 28) + 8) if far != "x" else wv.to(gpu)
    part = torch.full((ksplit, M, N), float("nan"), device=gpu)
    rc = _l3lib.load().l3_linear_splitk(x.data_ptr(), w.data_ptr(), part.data_ptr(), part.numel() * 4, M, N, K, (1 << 28) + 8 if far != "w" else K,
                                        w.stride(0), ksplit, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, rc
    per = -(-(K // 128) // ksplit) * 128
    for s in range(ksplit):
        want = xv[:, s * per:(s + 1) * per].double() @ wv[:, s * per:(s + 1) * per].double().t()
        # 32-bit sums of at most 1280 products of these sizes
        assert ((part[s].cpu().double() - want).abs() <= 2.0 ** -20 * (xv.double().abs() @ wv.double().abs().t())).all()
    if ksplit == 1 or M == 17:      # (the operator chooses its own splits)
        assert_linear_close(cke.linear_splitk_finish(cke.linear_splitk(x, w)), linear_ref(t2f32(xv), t2f32(wv)), "far rows")


# one shape per route: wide, split from 5 rows on, split from 1 row on, pair
ROUTES = [(4, 16384, 2048, False), (5, 2048, 8192, False), (1, 4096, 8192, False), (4, 8192, 2048, True)]


@pytest.mark.parametrize("M,N,K,pair", ROUTES)
def test_a_residual_aligned_to_eight_bytes_is_taken_whatever_the_route(gpu, M, N, K, pair):
    from custom_kernels import custom_kernels_extension as cke

    print(f"linear_decode_fused residual M={M} N={N} K={K} pair={pair}", flush=True)
    x = randn_bf16((M, 1, K), 241).to(gpu)
    w, up = randn_bf16((N, K), 242, scale=0.05).to(gpu), randn_bf16((N, K), 243, scale=0.05).to(gpu) if pair else None
    product = cke.linear_decode_fused(x, w, w_up=up)
    res = randn_bf16((M * N + 4,), 244, scale=3.0).to(gpu)
    shifted = res[4:].view(M, 1, N)
    assert shifted.data_ptr() % 16 == 8
    y = cke.linear_decode_fused(x, w, w_up=up, residual=shifted)
    if pair:
        assert torch.equal(y, shifted + product)
    else:
        # another kernel's sum may round the other way, one ulp of the product, and the addition rounds once more
        assert ((y - (shifted + product)).float().abs() <= 2.0 ** -7 * (product.float().abs() + y.float().abs())
                + 2.0 ** -17 * product.float().abs().max()).all()
    aligned = shifted.clone()
    assert torch.equal(cke.linear_decode_fused(x, w, w_up=up, residual=aligned), aligned + product)


@pytest.mark.parametrize("M,N,K,pair", ROUTES)
def test_activations_that_the_skinny_kernel_refuses_are_refused_whatever_the_route(gpu, M, N, K, pair):
    """Rows on top of each other and rows off 16 bytes, also where a norm in front would make a dense copy of them."""
    from custom_kernels import custom_kernels_extension as cke

    w = randn_bf16((N, K), 242, scale=0.05).to(gpu)
    up = w if pair else None
    rows = min(M, cke.linear_decode_fused_max_rows(K))
    norm = torch.ones(K, dtype=torch.bfloat16, device=gpu)
    off = randn_bf16((rows * K + 1,), 245).to(gpu)[1:].view(rows, K)
    one = randn_bf16((1, K), 246).to(gpu).as_strided((rows, K), (0, 1))
    for x in (off, one):
        for kw in (dict(), dict(norm_weight=norm)):
            with pytest.raises(RuntimeError):
                cke.linear_decode_fused(x, w, w_up=up, **kw)


@pytest.mark.parametrize("M", [4, 7, 11])
def test_a_norm_in_front_of_a_linear_that_fills_the_device(gpu, M):
    """More than three rows of a vocabulary projection: the norm is a launch of its own and rounds where it would inside."""
    from custom_kernels import custom_kernels_extension as cke

    N, K, eps = 12288, 2048, 1e-5
    print(f"norm and wide linear M={M}", flush=True)
    x, norm = randn_bf16((M, 1, K), 251).to(gpu), randn_bf16((K,), 252, scale=0.02, mean=1.0).to(gpu)
    w = randn_bf16((N, K), 253, scale=0.05).to(gpu)
    y = cke.linear_decode_fused(x, w, norm_weight=norm, eps=eps)
    h = cke.rms_norm(x, norm, eps)
    assert_linear_close(y.view(M, N), linear_ref(t2f32(h.view(M, K)), t2f32(w)), f"norm and wide {M}")
    assert torch.equal(y, cke.linear_decode(h, w))
