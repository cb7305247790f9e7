"""The three operators the reference binds in custom_kernels/main.cpp:5-9, same names and
positional signatures, backed by the gfx950 kernels of libl3kernels.so.

    flash_attention_decode(query, keys, values) -> Tensor    custom_kernels.cu:233-338
    rms_norm(input, weight, eps) -> Tensor                   custom_kernels.cu:369-389
    rot_embed(input, freq) -> Tensor                         custom_kernels.cu:418-442

Outputs are fresh tensors with the reference's shapes, dtypes and strides
(``empty_like(query)``, ``empty_like(input)``, and a contiguous (B, T, NH, HD) tensor for
rot_embed).  Unsupported arguments raise RuntimeError like the reference's TORCH_CHECKs.
Kernels are enqueued on torch's current stream of the input's device and the call does
not synchronise.  There is no fallback path: a missing library or a non-GPU tensor raises.
"""

import contextlib
import contextvars
import math

import torch

from . import _l3lib

__all__ = ["flash_attention_decode", "rms_norm", "rot_embed", "attention_num_splits", "attention_flags",
           "flash_attention_decode_static",
           "flash_attention_split", "flash_attention_combine", "flash_attention_decode_devlen",
           "rot_embed_append", "add_rms_norm", "silu_mul", "argmax", "flash_attention_prefill"]

_workspaces = {}  # (device index, stream handle) -> uint8 tensor


def _fail(code: int, detail: str = ""):
    msg = _l3lib.strerror(code)
    raise RuntimeError(f"{msg}{': ' + detail if detail else ''} (l3 error {code})")


def _require_gpu_bf16(name: str, t: torch.Tensor):
    if not isinstance(t, torch.Tensor):
        raise TypeError(f"{name} must be a torch.Tensor")
    if not t.is_cuda:
        raise RuntimeError(f"{name} must be on the GPU (got {t.device}); there is no CPU path")
    if t.dtype != torch.bfloat16:
        # the reference's data_ptr<at::BFloat16>() raises the same way (custom_kernels.cu:274)
        raise RuntimeError(f"expected scalar type BFloat16 for {name} but found {t.dtype}")


# The raw handle of torch's current stream without building a Stream object (2 us per call saved);
# the public accessor is the fallback where this build of torch does not have the direct one.
_raw_current_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_NO_GUARD = contextlib.nullcontext()


def _stream_ptr(device) -> int:
    if _raw_current_stream is not None:
        idx = device.index
        return _raw_current_stream(idx if idx is not None else torch.cuda.current_device())
    return torch.cuda.current_stream(device).cuda_stream


def _on_device(device):
    """Context in which `device` is the current one: nothing to do (and nothing to pay) when it
    already is, which is every call of a single-GPU process."""
    idx = device.index
    if idx is None or idx == torch.cuda.current_device():
        return _NO_GUARD
    return torch.cuda.device(idx)


def _workspace(device, stream_ptr: int, nbytes: int):
    """Scratch for the argmax partials, kept per (device, stream) and grown on demand so that a decode
    step does not allocate.  Calls on one stream are ordered and can share it; another stream gets its
    own.  While a stream is being captured into a HIP graph the buffer comes from the graph's own memory pool instead (a plain
    allocation that lives and dies with the graph) and is not cached."""
    if torch.cuda.is_current_stream_capturing():
        return torch.empty(max(nbytes, 256), dtype=torch.uint8, device=device)
    key = (device.index if device.index is not None else torch.cuda.current_device(), stream_ptr)
    ws = _workspaces.get(key)
    if ws is None or ws.numel() < nbytes:
        ws = torch.empty(max(nbytes, 1 << 20), dtype=torch.uint8, device=device)
        _workspaces[key] = ws
    return ws


# Flags the attention operators pass to the library when the caller gives none: a context-local
# value (per thread / per asyncio task), never a process-wide switch.  The library itself keeps no
# option between calls.
_attn_flags = contextvars.ContextVar("l3_attn_flags", default=0)

_KERNEL_BITS = {"mfma": 0, "fma": _l3lib.L3_ATTN_FLAG_KERNEL_FMA}
_PREFILL_BITS = {"auto": 0, "wave": _l3lib.L3_ATTN_FLAG_PREFILL_WAVE, "tiled": _l3lib.L3_ATTN_FLAG_PREFILL_TILED,
                 "tiled-no-max": _l3lib.L3_ATTN_FLAG_PREFILL_TILED_NO_MAX}
_LAUNCH_BITS = {"auto": 0, "two": _l3lib.L3_ATTN_FLAG_TWO_LAUNCHES}


@contextlib.contextmanager
def attention_flags(kernel=None, prefill=None, launches=None):
    """Within the block, attention calls of this thread that pass no ``flags`` use the named
    split-KV kernel ("mfma" / "fma"), prefill form ("auto" / "wave" / "tiled" / "tiled-no-max") and launch scheme
    ("auto" / "two": always split kernel + combine kernel).  An argument that is not given keeps what
    an enclosing block chose, so blocks nest.  For measurements and tests; the defaults are the
    library's own choices."""
    bits = _attn_flags.get()
    for name, table, mask in ((kernel, _KERNEL_BITS, _l3lib.L3_ATTN_FLAG_KERNEL_FMA),
                              (prefill, _PREFILL_BITS, _l3lib.L3_ATTN_FLAG_PREFILL_MASK),
                              (launches, _LAUNCH_BITS, _l3lib.L3_ATTN_FLAG_TWO_LAUNCHES)):
        if name is not None:
            bits = (bits & ~mask) | table[name]
    token = _attn_flags.set(bits)
    try:
        yield
    finally:
        _attn_flags.reset(token)


def _flags(flags):
    return _attn_flags.get() if flags is None else int(flags)


def attention_num_splits(B: int, KVH: int, S: int, HD: int, num_cus: int = 256, flags=None) -> int:
    """Split count the kernel picks for this problem (pure host logic, runs without a GPU)."""
    n = _l3lib.load().l3_attn_choose_splits(B, KVH, S, HD, num_cus, _flags(flags))
    if n < 0:
        _fail(n)
    return n


def _check_out(out, like, what: str):
    """A caller-supplied output is written through its raw pointer with `like`'s shape: it must be
    a bf16 tensor of that shape on the same device whose rows the kernels can address."""
    if not isinstance(out, torch.Tensor) or out.dtype != torch.bfloat16 or out.device != like.device \
            or tuple(out.shape) != tuple(like.shape):
        raise RuntimeError(f"{what}: out must be a bf16 tensor of shape {tuple(like.shape)} on {like.device}")
    if out.stride(-1) != 1 or any(st % 8 for st, n in zip(out.stride()[:-1], out.shape[:-1]) if n > 1):
        raise RuntimeError(f"{what}: out needs a contiguous last dimension and 16-byte aligned rows")


def flash_attention_decode(query, keys, values, num_splits: int = 0, flags=None):
    """query (B, QH, 1, HD); keys/values (B, KVH, S, HD) views of the KV cache (model.py:107-118).

    ``num_splits`` (0 = automatic) and ``flags`` (L3_ATTN_FLAG_* bits, None = attention_flags()'s
    context, normally 0) are extensions for tests and sweeps; the reference signature is the three
    tensors.
    """
    return _l3lib.native().flash_attention_decode(query, keys, values, num_splits, _flags(flags))


def flash_attention_decode_static(query, keys, values, out, num_splits: int = 0, flags=None):
    """flash_attention_decode into the caller's ``out`` with the partials in the library's static
    device scratch: the call allocates nothing (l3_attn_decode_static).  Raises when the problem
    needs more scratch than the static array holds.  Calls that overlap on one GPU race."""
    lib = _l3lib.load()
    flags = _flags(flags)
    B, QH, KVH, S, HD = _check_qkv(query, keys, values)
    if keys.device != query.device or values.device != query.device:
        raise RuntimeError("query, keys and values must be on the same device")
    _check_out(out, query, "flash_attention_decode_static")
    with _on_device(query.device):
        rc = lib.l3_attn_decode_static(
            query.data_ptr(), keys.data_ptr(), values.data_ptr(), out.data_ptr(), B, QH, KVH, S, HD,
            _l3lib.i64_array((query.stride(0), query.stride(1))),
            _l3lib.i64_array((keys.stride(0), keys.stride(1), keys.stride(2))),
            _l3lib.i64_array((values.stride(0), values.stride(1), values.stride(2))),
            _l3lib.i64_array((out.stride(0), out.stride(1))),
            1.0 / math.sqrt(HD), num_splits, flags, _stream_ptr(query.device))
    if rc != 0:
        _fail(rc, f"B={B} QH={QH} KVH={KVH} S={S} HD={HD}")
    return out


def _check_qkv(query, keys, values):
    _require_gpu_bf16("query", query)
    _require_gpu_bf16("keys", keys)
    _require_gpu_bf16("values", values)
    if query.dim() != 4 or keys.dim() != 4 or values.dim() != 4:
        raise RuntimeError("expected 4-D query, keys and values")
    B, KVH, S, HD = keys.shape
    QH = query.size(1)
    if query.size(0) != B or query.size(2) != 1 or query.size(3) != HD or tuple(values.shape) != tuple(keys.shape):
        raise RuntimeError(
            f"shape mismatch: query {tuple(query.shape)}, keys {tuple(keys.shape)}, values {tuple(values.shape)}")
    if query.stride(3) != 1 or keys.stride(3) != 1 or values.stride(3) != 1:
        raise RuntimeError("the head dimension of query, keys and values must be contiguous")
    return B, QH, KVH, S, HD


def flash_attention_prefill(query, keys, values, flags=None):
    """Causal GQA attention for T > 1 query tokens: query (B, QH, T, HD), keys / values
    (B, KVH, S, HD) cache views with S >= T; query i attends to tokens 0 .. S - T + i.  Returns a
    (B, QH, T, HD) view of a contiguous (B, T, QH, HD) tensor, so the model's
    ``y.transpose(1, 2).contiguous()`` (model.py:120) is free.  For S == T it computes what the
    reference asks of torch for this case (model.py:114-116).  An extension of the operator set."""
    return _l3lib.native().flash_attention_prefill(query, keys, values, _flags(flags))


def flash_attention_split(query, keys, values, num_splits: int = 0, flags=None):
    """First stage of flash_attention_decode on its own (an extension; the reference runs its two
    kernels only together, custom_kernels.cu:274-275).  Returns float32 partials
    ``(part_o (B, QH, n, HD), part_ml (B, QH, n, 2))``: unnormalised outputs and (max, sum) per
    split, scores in log2 units.  Partials of several token ranges of one sequence can be
    concatenated along dim 2 and finished by flash_attention_combine."""
    lib = _l3lib.load()
    flags = _flags(flags)
    B, QH, KVH, S, HD = _check_qkv(query, keys, values)
    with _on_device(query.device):
        n_req = num_splits if num_splits > 0 else lib.l3_attn_choose_splits(B, KVH, S, HD, 0, flags)
        if n_req < 0:
            _fail(n_req)
        part_o = torch.empty((B, QH, n_req, HD), dtype=torch.float32, device=query.device)
        part_ml = torch.empty((B, QH, n_req, 2), dtype=torch.float32, device=query.device)
        n = lib.l3_attn_split(
            query.data_ptr(), keys.data_ptr(), values.data_ptr(), part_o.data_ptr(), part_ml.data_ptr(),
            B, QH, KVH, S, HD,
            _l3lib.i64_array((query.stride(0), query.stride(1))),
            _l3lib.i64_array((keys.stride(0), keys.stride(1), keys.stride(2))),
            _l3lib.i64_array((values.stride(0), values.stride(1), values.stride(2))),
            1.0 / math.sqrt(HD), num_splits, flags, _stream_ptr(query.device))
    if n < 0:
        _fail(n, f"B={B} QH={QH} KVH={KVH} S={S} HD={HD}")
    if n != n_req:  # the kernel laid its rows out for n splits: re-view the front of the buffers
        part_o = part_o.flatten()[: B * QH * n * HD].view(B, QH, n, HD)
        part_ml = part_ml.flatten()[: B * QH * n * 2].view(B, QH, n, 2)
    return part_o, part_ml


def flash_attention_combine(part_o, part_ml, dtype=torch.bfloat16):
    """Second stage on its own: log-sum-exp merge of (B, QH, n, HD) / (B, QH, n, 2) float32
    partials into a (B, QH, 1, HD) bf16 tensor laid out like empty_like of the model's query view."""
    lib = _l3lib.load()
    if not part_o.is_cuda or part_o.dtype != torch.float32 or part_ml.dtype != torch.float32:
        raise RuntimeError("partials must be float32 GPU tensors")
    B, QH, n, HD = part_o.shape
    if tuple(part_ml.shape) != (B, QH, n, 2):
        raise RuntimeError(f"part_ml is {tuple(part_ml.shape)}, expected {(B, QH, n, 2)}")
    po = part_o if part_o.is_contiguous() else part_o.contiguous()
    pm = part_ml if part_ml.is_contiguous() else part_ml.contiguous()
    out = torch.empty((B, 1, QH, HD), dtype=dtype, device=part_o.device).transpose(1, 2)
    with _on_device(part_o.device):
        rc = lib.l3_attn_combine(po.data_ptr(), pm.data_ptr(), out.data_ptr(), B, QH, HD, n,
                                 _l3lib.i64_array((out.stride(0), out.stride(1))), _stream_ptr(part_o.device))
    if rc != 0:
        _fail(rc, f"B={B} QH={QH} HD={HD} n={n}")
    return out


def flash_attention_decode_devlen(query, keys, values, kv_len, num_splits: int = 0, out=None, flags=None):
    """flash_attention_decode whose KV length is the int32 GPU scalar ``kv_len`` instead of the
    tensor shape: ``keys`` / ``values`` are (B, KVH, L, HD) views of the whole cache and only the
    first ``kv_len`` tokens are attended.  The launch does not depend on the length, so it can be
    captured once in a HIP graph and replayed while the cache grows (an extension; the reference
    takes the length from keys.size(2), custom_kernels.cu:246).  ``out`` may be supplied to keep
    the call allocation-free under capture."""
    if out is not None:
        _check_out(out, query, "flash_attention_decode_devlen")
    return _l3lib.native().flash_attention_decode_devlen(query, keys, values, kv_len, num_splits, out, _flags(flags))


def rot_embed_append(qkv, freq_table, cache_k, cache_v, pos, n_head: int, out=None):
    """Decode-step fusion of model.py:100-106 for one new token per sequence: rotates the query
    and key heads of ``qkv`` (B, 1, (n_head + 2*KVH)*HD, the fused projection in q|k|v order) with
    row ``pos`` of ``freq_table`` ((rows, HD) float32), writes the rotated keys and the values
    into ``cache_k`` / ``cache_v`` ((maxB, L, KVH, HD)) at token ``pos`` and returns the rotated
    queries (B, 1, n_head, HD).  ``pos`` is a one-element int32 GPU tensor read by the kernel, so
    the launch can be replayed from a HIP graph.  An extension of the reference's operator set."""
    lib = _l3lib.load()
    _require_gpu_bf16("qkv", qkv)
    _require_gpu_bf16("cache_k", cache_k)
    _require_gpu_bf16("cache_v", cache_v)
    if qkv.dim() != 3 or qkv.size(1) != 1 or qkv.stride(2) != 1:
        raise RuntimeError("qkv must be (B, 1, (n_head + 2*KVH)*HD) with a contiguous last dimension")
    if cache_k.dim() != 4 or cache_k.shape != cache_v.shape or cache_k.stride() != cache_v.stride():
        raise RuntimeError("cache_k and cache_v must be (maxB, L, KVH, HD) tensors of the same layout")
    maxB, L, KVH, HD = cache_k.shape
    B = qkv.size(0)
    if qkv.size(2) != (n_head + 2 * KVH) * HD or B > maxB:
        raise RuntimeError(f"qkv {tuple(qkv.shape)} does not match n_head={n_head}, cache {tuple(cache_k.shape)}")
    if cache_k.stride(3) != 1 or cache_k.stride(2) != HD:
        raise RuntimeError("the (KVH, HD) dimensions of the cache must be contiguous")
    if not freq_table.is_cuda or freq_table.dtype != torch.float32 or freq_table.dim() != 2 \
            or freq_table.size(1) != HD or not freq_table.is_contiguous():
        raise RuntimeError("freq_table must be a contiguous (rows, HD) float32 GPU tensor")
    if not pos.is_cuda or pos.dtype != torch.int32 or pos.numel() != 1 or pos.device != qkv.device:
        raise RuntimeError("pos must be a one-element int32 tensor on qkv's GPU")
    if cache_k.device != qkv.device or cache_v.device != qkv.device or freq_table.device != qkv.device:
        raise RuntimeError("qkv, freq_table and the caches must be on the same device")
    if out is None:
        out = torch.empty((B, 1, n_head, HD), dtype=qkv.dtype, device=qkv.device)
    elif not isinstance(out, torch.Tensor) or out.dtype != torch.bfloat16 or out.device != qkv.device \
            or tuple(out.shape) != (B, 1, n_head, HD) or not out.is_contiguous():
        raise RuntimeError(f"rot_embed_append: out must be a contiguous bf16 tensor of shape {(B, 1, n_head, HD)} "
                           f"on {qkv.device}")
    with _on_device(qkv.device):
        rc = lib.l3_rot_embed_append(qkv.data_ptr(), freq_table.data_ptr(), out.data_ptr(), cache_k.data_ptr(),
                                     cache_v.data_ptr(), pos.data_ptr(), B, n_head, KVH, HD, qkv.stride(0),
                                     _l3lib.i64_array((cache_k.stride(0), cache_k.stride(1))), L,
                                     freq_table.size(0), _stream_ptr(qkv.device))
    if rc != 0:
        _fail(rc, f"B={B} NH={n_head} KVH={KVH} HD={HD}")
    return out


def linear_qkv_rope_append(x, w_qkv, freq_table, cache_k, cache_v, pos, n_head: int, norm_weight=None,
                           eps: float = 1e-5):
    """linear_decode_fused(x, w_qkv, norm_weight) followed by rot_embed_append in one launch: the
    whole of model.py:95-106 for one new token per sequence.  x (B, 1, K); returns the rotated
    queries (B, 1, n_head, HD); keys and values are written into the caches at ``pos``."""
    return _l3lib.native().linear_qkv_rope_append(x, w_qkv, freq_table, cache_k, cache_v, pos, n_head, norm_weight, eps)


def linear_qkv_rope_append_rows(x, w_qkv, freq_table, cache_k, cache_v, pos, n_head: int):
    """linear_qkv_rope_append without a norm for up to 64 sequences: x (B, 1, K), K a multiple of 128.  An extension."""
    return _l3lib.native().linear_qkv_rope_append_rows(x, w_qkv, freq_table, cache_k, cache_v, pos, n_head)


def rms_norm(input, weight, eps):
    """input (B, T, C) bf16, weight (C,) bf16 -> (B, T, C) bf16 (model.py:70-72)."""
    return _l3lib.native().rms_norm(input, weight, eps)


def add_rms_norm(input, residual, weight, eps):
    """(input + residual, rms_norm(input + residual, weight, eps)) in one launch: the residual
    addition of model.py:147-148 fused with the norm that follows it.  Both outputs carry the same
    bits as ``s = input + residual`` (bf16) followed by ``rms_norm(s, weight, eps)``.  An extension
    of the reference's operator set."""
    return _l3lib.native().add_rms_norm(input, residual, weight, eps)


def silu_mul(a, b):
    """F.silu(a) * b for two bf16 tensors of the same shape in one launch (model.py:134), with the
    two roundings of the two torch kernels, so the bits are the same.  An extension."""
    return _l3lib.native().silu_mul(a, b)


def linear_decode(x, weight):
    """F.linear(x, weight) for at most 64 activation rows (model.py:95,121,134,225 when T == 1):
    one pass over the weight matrix at HBM speed instead of a GEMM.  x (..., K), weight (N, K)
    -> (..., N).  17..64 rows need N % 8 == 0 and K % 128 == 0.  One launch up to 16 rows and, whatever the rows, where those of
    the matrix fill the device (a vocabulary projection); otherwise linear_splitk and linear_splitk_finish, two launches, from 17
    rows on and for large matrices before (16 M elements from 5 rows on, 32 M from one).  An extension."""
    return _l3lib.native().linear_decode(x, weight)


def linear_swiglu_decode(x, w_gate, w_up):
    """F.silu(F.linear(x, w_gate)) * F.linear(x, w_up) for at most 64 activation rows in one
    launch (model.py:134 with w_gate = c_fc2, w_up = c_fc), same rounding points; from 17 rows on
    K % 128 == 0.  An extension."""
    return _l3lib.native().linear_swiglu_decode(x, w_gate, w_up)


def linear_decode_fused_max_rows(K: int) -> int:
    """Most activation rows of width K for which linear_decode_fused accepts a norm_weight."""
    return min(16, _l3lib.L3_LINEAR_STAGE_ELEMS // (K + 8)) if K % 512 == 0 else 0


def linear_decode_fused(x, weight, norm_weight=None, eps: float = 1e-5, w_up=None, residual=None):
    """linear_decode with the operators around it folded in, each optional (in the same launches; a norm in front of what is not
    the one-launch form for up to 16 rows is one of its own): rms_norm(x, norm_weight, eps) in front (model.py:70-72), the SwiGLU product with a second
    matrix w_up (weight is then the gate, model.py:134), and `residual + result` behind
    (model.py:147-148) -- all with the rounding points of the separate operators.  An extension."""
    return _l3lib.native().linear_decode_fused(x, weight, norm_weight, eps, w_up, residual)


def linear_splitk(x, weight, ksplit: int = 0):
    """x (..., K) with up to 64 rows times weight (N, K)^T as float32 partial products
    (ksplit, rows, N) -- NOT added up: hand them to add_rms_norm_partials or
    rot_embed_append_partials, which sum the splits on their way (or sum them yourself).
    ksplit 0 lets the library choose.  Stands for nn.Linear at batch sizes where the activations no
    longer fit one matrix-instruction column block (model.py:95,121,134).  An extension."""
    return _l3lib.native().linear_splitk(x, weight, ksplit)


def linear_splitk_finish(part, residual=None):
    """bf16(part.sum(0)) for linear_splitk's partial products (ksplit, rows, N), summed in split
    order and rounded once -- what the unsplit linear would have returned -- plus ``residual``
    (rows x N, bf16) with the rounding of a separate addition if given.  Returns (rows, N)."""
    return _l3lib.native().linear_splitk_finish(part, residual)


def add_rms_norm_partials(input, part, weight, eps):
    """add_rms_norm(input, r, weight, eps) with r = bf16(part.sum(0)) formed inside the kernel:
    ``part`` is linear_splitk's output for the linear whose result is the residual branch
    (model.py:147-148).  Returns (input + r, rms_norm(input + r))."""
    return _l3lib.native().add_rms_norm_partials(input, part, weight, eps)


def rot_embed_append_partials(part, freq_table, cache_k, cache_v, pos, n_head: int):
    """rot_embed_append on a fused qkv projection that is still in linear_splitk's partial
    products (ksplit, B, (n_head + 2*KVH)*HD): summed, rounded to bf16, rotated, appended."""
    return _l3lib.native().rot_embed_append_partials(part, freq_table, cache_k, cache_v, pos, n_head)


class DecodeLayers:
    """All transformer layers of one decode step in one launch (l3_decode_layers), for up to four sequences of the
    1B architecture.  ``layers``: dicts with ln_1, c_attn, c_proj, ln_2, c_fc2 (gate), c_fc (up), mlp_proj, cache_k and
    cache_v.  The workgroups of a launch wait for each other, with bounds; ``failed()`` (it synchronises) says
    whether a wait has run out: every result since then is void and the object of no more use, the operators one by
    one do the same work.  One launch of an object at a time.  An extension."""

    NAMES = ("ln_1", "c_attn", "c_proj", "ln_2", "c_fc2", "c_fc", "mlp_proj", "cache_k", "cache_v")

    def __init__(self, layers, rows: int):
        if (why := self.unserved(layers, rows)) is not None:
            raise RuntimeError(f"DecodeLayers: {why}")
        self.rows, self.n_layer = rows, len(layers)
        self.tensors = [[L[n] for n in self.NAMES] for L in layers]     # kept alive
        self.pointers = [[t.data_ptr() for t in row] for row in self.tensors]
        cache = layers[0]["cache_k"]
        _, self.cache_len, _, HD = cache.shape
        C = layers[0]["c_fc"].shape[1]
        with _on_device(cache.device):
            nbytes = _l3lib.load().l3_decode_layers_workspace_bytes(rows, self.n_layer)
        self.table = torch.tensor(self.pointers, dtype=torch.int64, device=cache.device)
        self.workspace = torch.zeros(nbytes, dtype=torch.uint8, device=cache.device)
        self.strides, self.C, self.HD = (cache.stride(0), cache.stride(1)), C, HD

    @staticmethod
    def unserved(layers, rows: int):
        """Why the launch does not take these layers (rows with a padded stride, another architecture ...), or None where it does.
        The operators one by one take more."""
        first = layers[0]
        cache = first["cache_k"]
        for L in layers:
            for name in DecodeLayers.NAMES:
                t = L[name]
                _require_gpu_bf16(name, t)
                if not t.is_contiguous() or t.data_ptr() % 16 or t.shape != first[name].shape or t.device != cache.device:
                    return f"{name} must be contiguous and alike in all layers"
        if cache.dim() != 4 or first["c_fc"].dim() != 2:
            return f"cache {tuple(cache.shape)}, c_fc {tuple(first['c_fc'].shape)}"
        maxB, _, KVH, HD = cache.shape
        H, C = first["c_fc"].shape
        QH = first["c_attn"].shape[0] // HD - 2 * KVH
        want = dict(ln_1=(C,), ln_2=(C,), c_attn=((QH + 2 * KVH) * HD, C), c_proj=(C, QH * HD), c_fc=(H, C), c_fc2=(H, C),
                    mlp_proj=(C, H), cache_v=tuple(cache.shape))
        wrong = [n for n, shape in want.items() if tuple(first[n].shape) != shape]
        with _on_device(cache.device):
            if rows > maxB or wrong or not DecodeLayers.supported(rows, C, H, QH, KVH, HD):
                return f"rows={rows} C={C} H={H} QH={QH} KVH={KVH} HD={HD} is not served {wrong}"
        return None

    def holds(self, layers) -> bool:
        """Whether ``layers`` are still the tensors, in the memory, that this object was made for."""
        return len(layers) == self.n_layer and all(L[n] is t and t.data_ptr() == at
                                                   for L, row, ptrs in zip(layers, self.tensors, self.pointers)
                                                   for n, t, at in zip(self.NAMES, row, ptrs))

    @staticmethod
    def supported(rows: int, C: int, H: int, QH: int, KVH: int, HD: int) -> bool:
        return bool(_l3lib.load().l3_decode_layers_supported(rows, C, H, QH, KVH, HD))

    def __call__(self, x, freq_table, pos, eps: float):
        """x (rows, 1, C) -> the hidden state behind the last layer, (rows, 1, C); keys and values are appended to the
        caches at the device-side position ``pos``."""
        _require_gpu_bf16("x", x)
        if tuple(x.shape) != (self.rows, 1, self.C) or not x.is_contiguous() or x.device != self.table.device:
            raise RuntimeError(f"DecodeLayers: x {tuple(x.shape)} does not fit ({self.rows}, 1, {self.C})")
        return self._launch("l3_decode_layers", (x.data_ptr(),), freq_table, pos, eps)

    def from_tokens(self, tokens, embedding, freq_table, pos, eps: float):
        """The same with x = embedding[tokens]: tokens (rows, 1) int64 with any row stride, embedding (vocab, C)."""
        _require_gpu_bf16("embedding", embedding)
        if embedding.dim() != 2 or embedding.size(1) != self.C or not embedding.is_contiguous() or embedding.device != self.table.device:
            raise RuntimeError(f"DecodeLayers: embedding {tuple(embedding.shape)} does not fit (vocab, {self.C})")
        if tuple(tokens.shape) != (self.rows, 1) or tokens.dtype != torch.int64 or tokens.device != self.table.device:
            raise RuntimeError(f"DecodeLayers: tokens must be ({self.rows}, 1) int64 on the GPU of the layers")
        return self._launch("l3_decode_layers_tokens", (tokens.data_ptr(), tokens.stride(0), embedding.data_ptr(), embedding.size(0)),
                            freq_table, pos, eps)

    def _launch(self, function, source, freq_table, pos, eps):
        if not freq_table.is_cuda or freq_table.dtype != torch.float32 or freq_table.dim() != 2 \
                or freq_table.size(1) != self.HD or not freq_table.is_contiguous():
            raise RuntimeError("freq_table must be a contiguous (rows, HD) float32 GPU tensor")
        if not pos.is_cuda or pos.dtype != torch.int32 or pos.numel() != 1:
            raise RuntimeError("pos must be a one-element int32 GPU tensor")
        device = self.table.device
        if freq_table.device != device or pos.device != device:
            raise RuntimeError("DecodeLayers: freq_table and pos must be on the GPU of the layers")
        out = torch.empty((self.rows, 1, self.C), dtype=torch.bfloat16, device=device)
        with _on_device(device):
            rc = getattr(_l3lib.load(), function)(self.table.data_ptr(), self.n_layer, *source, out.data_ptr(), self.rows,
                                                  freq_table.data_ptr(), freq_table.size(0), pos.data_ptr(),
                                                  _l3lib.i64_array(self.strides), self.cache_len, float(eps),
                                                  self.workspace.data_ptr(), self.workspace.numel(), _stream_ptr(device))
        if rc != 0:
            _fail(rc, f"rows={self.rows} n_layer={self.n_layer}")
        return out

    def failed(self) -> bool:
        return bool(self.workspace[:4].any().item())


def argmax(logits):
    """Index of the first maximum along the last dimension of a 2-D bf16 tensor (rows, V), as
    int64 -- torch.argmax(logits.float(), dim=-1) for the greedy pick of model.py:371 (the float
    conversion of model.py:225 is monotone, so it is skipped).  An extension."""
    lib = _l3lib.load()
    _require_gpu_bf16("logits", logits)
    if logits.dim() != 2 or logits.stride(1) != 1:
        raise RuntimeError("argmax expects a 2-D (rows, V) tensor with a contiguous last dimension")
    rows, V = logits.shape
    out = torch.empty(rows, dtype=torch.int64, device=logits.device)
    if rows == 0:
        return out
    with _on_device(logits.device):
        ws_bytes = lib.l3_argmax_workspace_bytes(rows, V)
        stream_ptr = _stream_ptr(logits.device)
        ws = _workspace(logits.device, stream_ptr, ws_bytes)
        rc = lib.l3_argmax(logits.data_ptr(), logits.stride(0), rows, V, ws.data_ptr(), ws_bytes, out.data_ptr(),
                           stream_ptr)
    if rc != 0:
        _fail(rc, f"rows={rows} V={V}")
    return out


def greedy_step(logits, tokens, text_mask, tok, pos, kv_len, eos, stop_tokens):
    """The tail of one greedy decoding step, in place and on the device (model.py:371-378): pick
    argmax(logits[b]) unless position pos + 1 still belongs to the prompt (text_mask), store the
    token into tokens[:, pos + 1] and tok, mark rows that produced a stop token in eos, and
    advance pos and kv_len by one.  logits (rows, V) bf16; tokens (rows, L) int64; text_mask
    (rows, L) bool; tok (rows, 1) or (rows,) int64; pos, kv_len int32 scalars; eos (rows) bool;
    stop_tokens int64.  An extension."""
    lib = _l3lib.load()
    _require_gpu_bf16("logits", logits)
    if logits.dim() != 2 or logits.stride(1) != 1:
        raise RuntimeError("greedy_step expects (rows, V) logits with a contiguous last dimension")
    rows, V = logits.shape
    L = tokens.shape[1]
    ok = (tokens.dtype == torch.int64 and tokens.is_contiguous() and tokens.shape[0] == rows
          and text_mask.dtype == torch.bool and text_mask.is_contiguous() and tuple(text_mask.shape) == (rows, L)
          and tok.dtype == torch.int64 and tok.is_contiguous() and tok.numel() == rows
          and pos.dtype == torch.int32 and pos.numel() == 1 and kv_len.dtype == torch.int32 and kv_len.numel() == 1
          and eos.dtype == torch.bool and eos.is_contiguous() and eos.numel() == rows
          and stop_tokens.dtype == torch.int64 and stop_tokens.is_contiguous())
    if not ok or any(t.device != logits.device for t in (tokens, text_mask, tok, pos, kv_len, eos, stop_tokens)):
        raise RuntimeError("greedy_step: state tensors have the wrong dtype, shape, layout or device")
    with _on_device(logits.device):
        ws_bytes = lib.l3_argmax_workspace_bytes(rows, V)
        stream_ptr = _stream_ptr(logits.device)
        ws = _workspace(logits.device, stream_ptr, ws_bytes)
        rc = lib.l3_greedy_step(logits.data_ptr(), logits.stride(0), rows, V, ws.data_ptr(), ws_bytes,
                                tokens.data_ptr(), text_mask.data_ptr(), L, tok.data_ptr(), pos.data_ptr(),
                                kv_len.data_ptr(), eos.data_ptr(), stop_tokens.data_ptr(), stop_tokens.numel(),
                                stream_ptr)
    if rc != 0:
        _fail(rc, f"rows={rows} V={V}")


def rot_embed(input, freq):
    """input (B, T, NH, HD) bf16 (any strides on the first three dims), freq (T, HD) float32
    interleaved cos/sin -> contiguous (B, T, NH, HD) bf16 (model.py:100-101)."""
    return _l3lib.native().rot_embed(input, freq)
