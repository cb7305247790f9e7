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
