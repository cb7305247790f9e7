"""The operators under several Python threads and streams: the interpreter lock is free while an operator works, calls of
several threads on one stream keep their scratch apart, and so do more streams than workspaces are kept for."""

import os
import re
import subprocess
import threading
import time

import pytest
import torch

from helpers import assert_attn_close, make_qkv, t2f32
from oracle import attention_decode_ref

pytestmark = pytest.mark.gpu


def test_other_threads_run_while_an_operator_works(gpu, tmp_path):
    """A stand-in for the library whose silu_mul takes 0.3 s of host time."""
    import build as l3_build
    from custom_kernels import _l3lib

    names = sorted(set(re.findall(r"X\((l3_\w+)\)", open(os.path.join(l3_build.CSRC, "torch_ops.cpp")).read())))
    assert "l3_silu_mul" in names
    source, stub = tmp_path / "stub.cpp", tmp_path / "libstub.so"
    source.write_text("#include <unistd.h>\n" + "".join(
        f'extern "C" int {n}() {{ {"usleep(300000);" if n == "l3_silu_mul" else ""} return 0; }}\n' for n in names))
    subprocess.run(["g++", "-shared", "-fPIC", str(source), "-o", str(stub)], check=True)
    native = _l3lib.native()
    x = torch.ones(64, dtype=torch.bfloat16, device=gpu)
    ticks, done = [], threading.Event()

    def tick():
        while not done.is_set():
            ticks.append(time.perf_counter())
            time.sleep(0.001)

    thread = threading.Thread(target=tick)
    native.bind(str(stub))
    try:
        thread.start()
        start = time.perf_counter()
        native.silu_mul(x, x)
        end = time.perf_counter()
    finally:
        done.set()
        native.bind(_l3lib.library_path())
        thread.join()
    assert end - start >= 0.3
    assert any(start + 0.1 < t < start + 0.2 for t in ticks)


def _in_threads(n, work):
    failures = []

    def guarded(i):
        try:
            work(i)
        except BaseException as e:
            failures.append((i, e))

    threads = [threading.Thread(target=guarded, args=(i,)) for i in range(n)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures[0]


@pytest.mark.parametrize("launches", ["auto", "two"])
def test_threads_that_share_a_stream(gpu, launches):
    """Eight threads, one stream, decode attention with splits: the launches of a call stay together, whose partials are."""
    from custom_kernels import custom_kernels_extension as cke

    S = 3000
    print(f"threads on one stream: launches={launches}", flush=True)
    inputs = [make_qkv(1, 8, 2, S, 64, seed=300 + 3 * i, device=gpu) for i in range(8)]
    with cke.attention_flags(launches=launches):
        want = [cke.flash_attention_decode(*qkv) for qkv in inputs]
    got = [None] * 8

    def work(i):
        with cke.attention_flags(launches=launches):
            got[i] = [cke.flash_attention_decode(*inputs[i]) for _ in range(100)]

    _in_threads(8, work)
    torch.cuda.synchronize()
    for outs, w in zip(got, want):
        assert all(torch.equal(o, w) for o in outs)
    assert_attn_close(want[0], attention_decode_ref(*(t2f32(t) for t in inputs[0])), "threads", min_kv_len=S)


def test_more_streams_than_workspaces_are_kept(gpu):
    from custom_kernels import custom_kernels_extension as cke

    qkv = make_qkv(2, 8, 2, 3000, 64, seed=320, device=gpu)
    want = cke.flash_attention_decode(*qkv)
    torch.cuda.synchronize()
    handles = [torch.cuda.ExternalStream(_new_stream()) for _ in range(80)]
    print("80 streams in turn", flush=True)
    outs = []
    for _ in range(3):
        for s in handles:
            with torch.cuda.stream(s):
                outs.append(cke.flash_attention_decode(*qkv))
    torch.cuda.synchronize()
    assert all(torch.equal(o, want) for o in outs)


def _new_stream():
    """A stream of its own (torch hands out 32 in turn)."""
    import ctypes

    with open("/proc/self/maps") as maps:       # the runtime that torch has loaded
        loaded = [line.split()[-1] for line in maps if "libamdhip64.so" in line]
    hip = ctypes.CDLL(next(p for p in loaded if "torch" in p))
    handle = ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(handle), 1) == 0
    return handle.value
