"""Operands on two GPUs are refused before anything is launched.  Fake tensors stand for the second GPU (and the first)."""

import pytest
import torch
from torch._subclasses import FakeTensorMode

from custom_kernels import _l3lib
from custom_kernels import custom_kernels_extension as cke

B, NH, KVH, HD, K, L = 2, 4, 2, 64, 256, 16


def _fake(device, *shape, dtype=torch.bfloat16):
    with FakeTensorMode():
        return torch.empty(shape, dtype=dtype, device=device)


def _cache_arguments(elsewhere):
    shapes = dict(table=((64, HD), torch.float32), k=((B, L, KVH, HD), torch.bfloat16), v=((B, L, KVH, HD), torch.bfloat16),
                  pos=((1,), torch.int32))
    return [_fake("cuda:1" if name in elsewhere else "cuda:0", *shape, dtype=dtype) for name, (shape, dtype) in shapes.items()]


@pytest.mark.parametrize("elsewhere", [("table",), ("pos",), ("v",), ("k", "v")])
def test_operators_that_append_to_the_cache_refuse_a_second_gpu(elsewhere):
    native = _l3lib.native()
    N = (NH + 2 * KVH) * HD
    x, w = _fake("cuda:0", B, 1, K), _fake("cuda:0", N, K)
    part = _fake("cuda:0", 3, B, N, dtype=torch.float32)
    args = _cache_arguments(elsewhere)
    for call in (lambda: native.linear_qkv_rope_append_rows(x, w, *args, NH), lambda: native.linear_qkv_rope_append(x, w, *args, NH, None, 1e-5),
                 lambda: native.rot_embed_append_partials(part, *args, NH)):
        with pytest.raises(RuntimeError, match="same device"):
            call()


@pytest.mark.parametrize("elsewhere", ["table", "pos"])
def test_the_one_launch_step_refuses_a_second_gpu(elsewhere):
    launch = object.__new__(cke.DecodeLayers)
    launch.rows, launch.n_layer, launch.C, launch.HD = B, 1, K, HD
    launch.table = _fake("cuda:0", 1, 9, dtype=torch.int64)
    table = _fake("cuda:1" if elsewhere == "table" else "cuda:0", 64, HD, dtype=torch.float32)
    pos = _fake("cuda:1" if elsewhere == "pos" else "cuda:0", 1, dtype=torch.int32)
    with pytest.raises(RuntimeError, match="on the GPU of the layers"):
        launch._launch("l3_decode_layers", (0,), table, pos, 1e-5)
