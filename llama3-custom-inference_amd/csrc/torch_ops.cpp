// The operators on torch tensors: argument checks, output allocation, workspaces and the call into
// libl3kernels.so, as a CPython extension module (custom_kernels/_l3torch.so).  It takes the place of
// the pybind table of main.cpp:5-9 and of the tensor handling at the head of the host launchers
// (custom_kernels.cu:233-338, 369-389, 418-442).
//
// Why it is native: a decode step calls small operators one after the other, and the calls, not the
// kernels, set the pace.  The HIP runtime takes 2.4 us to enqueue a kernel; the same checks in Python with a
// ctypes call took 6.5 us for rms_norm of one row, 7.9 us for rot_embed, 11.9 us for
// flash_attention_decode over 256 tokens and 19.5 us for a split-K linear with its finishing pass.  Here
// they take 3.9, 3.8, 4.5 and 13.5 us (the last is the kernels' own time).
// Hence METH_FASTCALL functions with positional arguments, tensors unpacked in place, and outputs
// taken from torch's caching allocator without a trip through the dispatcher.
//
// libl3kernels.so itself stays free of torch: its C functions are looked up by name (bind) in the
// library that the Python side has loaded.
#include <Python.h>
#include <dlfcn.h>

#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/ops/empty_like.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cmath>
#include <memory>
#include <mutex>
#include <utility>
#include <vector>

#include "../../include/l3_kernels.h"

namespace {

using at::Tensor;
using at::TensorBase;

#define L3_FUNCTIONS(X)                                                                                          \
    X(l3_strerror) X(l3_attn_decode) X(l3_attn_decode_devlen) X(l3_attn_decode_workspace_bytes)                  \
    X(l3_attn_workspace_init) X(l3_attn_prefill_ws) X(l3_attn_prefill_workspace_bytes) X(l3_rms_norm) X(l3_add_rms_norm) X(l3_add_rms_norm_partials)   \
    X(l3_rot_embed) X(l3_rot_embed_append_partials) X(l3_silu_mul) X(l3_silu_mul_rows)       \
    X(l3_linear_decode_fused) X(l3_linear_qkv_rope_append) X(l3_linear_splitk_rows_plan)   \
    X(l3_linear_splitk) X(l3_linear_splitk_finish) X(l3_linear_wide) X(l3_linear_qkv_rope_append_rows)

struct Library {
#define X(name) decltype(&::name) name = nullptr;
    L3_FUNCTIONS(X)
#undef X
} lib;

// ------------------------------------------------------------------------------------------ arguments

const Tensor& tensor(PyObject* o, const char* name) {
    TORCH_CHECK_TYPE(THPVariable_Check(o), name, " must be a torch.Tensor");
    return THPVariable_Unpack(o);
}

void require_gpu_bf16(const Tensor& t, const char* name) {
    TORCH_CHECK(t.is_cuda(), name, " must be on the GPU (got ", t.device(), "); there is no CPU path");
    // the reference's data_ptr<at::BFloat16>() raises the same way (custom_kernels.cu:274)
    TORCH_CHECK(t.scalar_type() == at::kBFloat16, "expected scalar type BFloat16 for ", name, " but found ", t.scalar_type());
}

const Tensor& gpu_bf16(PyObject* o, const char* name) {
    const Tensor& t = tensor(o, name);
    require_gpu_bf16(t, name);
    return t;
}

int integer(PyObject* o) {
    const long v = PyLong_AsLong(o);
    if (v == -1 && PyErr_Occurred()) throw python_error();
    return int(v);
}

double number(PyObject* o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw python_error();
    return v;
}

const Tensor* optional_tensor(PyObject* o, const char* name) { return o == Py_None ? nullptr : &gpu_bf16(o, name); }

// Raises for an error code of the library.
template <typename... Detail>
void check(int64_t rc, const Detail&... detail) {
    TORCH_CHECK(rc >= 0, lib.l3_strerror(int(rc)), ": ", detail..., " (l3 error ", rc, ")");
}

int64_t size_at(const Tensor& t, int i) { return t.sizes()[i]; }
int64_t stride_at(const Tensor& t, int i) { return t.strides()[i]; }
void* ptr(const TensorBase& t) { return t.data_ptr(); }

// A contiguous tensor with t's values; t itself (kept alive by the caller's arguments) where it is one.
const Tensor& contiguous(const Tensor& t, Tensor& copy) {
    if (t.is_contiguous()) return t;
    copy = t.contiguous();
    return copy;
}

Tensor new_empty(at::IntArrayRef sizes, const Tensor& like, at::ScalarType type = at::kBFloat16) {
    return Tensor(at::detail::empty_cuda(sizes, type, like.device(), std::nullopt));
}

// torch.empty_like for a dense tensor: the same sizes and strides.
Tensor empty_like_dense(const Tensor& t) {
    return Tensor(at::detail::empty_strided_cuda(t.sizes(), t.strides(), t.scalar_type(), t.device()));
}

// The work of a call with the interpreter lock released, so that other Python threads go on meanwhile (a launch waits while
// the queue is full, an allocation may go to the driver, the first decode attention on a device synchronises).  Arguments are
// unpacked before and results wrapped after it.
template <typename F>
auto unlocked(F&& work) {
    struct Release {
        PyThreadState* const state = PyEval_SaveThread();
        ~Release() { PyEval_RestoreThread(state); }
    } released;
    return work();
}

PyObject* wrap(Tensor&& t) { return THPVariable_Wrap(std::move(t)); }

PyObject* wrap(std::pair<Tensor, Tensor>&& t) {
    PyObject* pair = PyTuple_New(2);
    if (!pair) throw python_error();
    PyTuple_SET_ITEM(pair, 0, wrap(std::move(t.first)));
    PyTuple_SET_ITEM(pair, 1, wrap(std::move(t.second)));
    return pair;
}

// The tensor's device made current for the length of a call (nothing to do in a single-GPU process),
// and torch's current stream there.
struct OnDevice {
    c10::DeviceIndex before = -1;
    c10::DeviceIndex index;
    hipStream_t stream;
    explicit OnDevice(const Tensor& t) : index(t.device().index()) {
        const c10::DeviceIndex now = c10::hip::current_device();
        if (now != index) {
            c10::hip::set_device(index);
            before = now;
        }
        stream = c10::hip::getCurrentHIPStream(index).stream();
    }
    ~OnDevice() {
        if (before >= 0) c10::hip::set_device(before);
    }
    OnDevice(const OnDevice&) = delete;
    OnDevice& operator=(const OnDevice&) = delete;
};

// ------------------------------------------------------------------------------------- decode attention

// Workspaces of decode attention: one per (device, stream), grown on demand, whose head holds the arrival
// counters of the single-launch form.  Calls on one stream are ordered and can share one; another stream
// gets its own.  `in_use` keeps the launches of a call together where several threads call on one stream (the interpreter lock
// is released by then).  The list is bounded: beyond kMaxWorkspaces streams the
// one unused longest goes back to torch's allocator, which hands its memory only to later work of the
// stream it was allocated on.
struct Workspace {
    c10::DeviceIndex device;
    hipStream_t stream;
    std::mutex in_use;
    TensorBase memory;   // guarded by in_use
    Workspace(c10::DeviceIndex d, hipStream_t s) : device(d), stream(s) {}
};
constexpr size_t kMaxWorkspaces = 64;

std::shared_ptr<Workspace> attention_workspace(const OnDevice& on) {
    static auto& all = *new std::vector<std::shared_ptr<Workspace>>();   // outlives the allocator's own teardown
    static auto& all_mutex = *new std::mutex();
    const std::lock_guard<std::mutex> lock(all_mutex);
    size_t i = 0;
    while (i < all.size() && !(all[i]->stream == on.stream && all[i]->device == on.index)) ++i;
    if (i == all.size()) {
        if (all.size() >= kMaxWorkspaces) all.pop_back();
        i = all.size();
        all.push_back(std::make_shared<Workspace>(on.index, on.stream));
    }
    if (i > 0) std::rotate(all.begin(), all.begin() + i, all.begin() + i + 1);   // most recently used first
    return all[0];
}

// At least nbytes, prepared.  (With in_use held.)
void* grown(Workspace& w, const Tensor& like, size_t nbytes) {
    if (!w.memory.defined() || size_t(w.memory.numel()) < nbytes) {
        TensorBase memory = at::detail::empty_cuda({int64_t(std::max(nbytes, size_t(4) << 20))}, at::kByte, like.device(),
                                                   std::nullopt);
        check(lib.l3_attn_workspace_init(ptr(memory), size_t(memory.numel()), w.stream), "l3_attn_workspace_init");
        w.memory = std::move(memory);
    }
    return ptr(w.memory);
}

struct DecodeShape {
    int B, QH, KVH, S, HD;
};

DecodeShape check_qkv(const Tensor& q, const Tensor& k, const Tensor& v) {
    TORCH_CHECK(q.dim() == 4 && k.dim() == 4 && v.dim() == 4, "expected 4-D query, keys and values");
    const auto qs = q.sizes(), ks = k.sizes();
    TORCH_CHECK(qs[0] == ks[0] && qs[2] == 1 && qs[3] == ks[3] && ks == v.sizes(), "shape mismatch: query ", qs, ", keys ",
                ks, ", values ", v.sizes());
    TORCH_CHECK(stride_at(q, 3) == 1 && stride_at(k, 3) == 1 && stride_at(v, 3) == 1,
                "the head dimension of query, keys and values must be contiguous");
    TORCH_CHECK(k.device() == q.device() && v.device() == q.device(), "query, keys and values must be on the same device");
    return {int(ks[0]), int(qs[1]), int(ks[1]), int(ks[2]), int(ks[3])};
}

void check_heads(int QH, int KVH, int HD) {
    if (HD != 64 && HD != 128) check(L3_ERR_HEAD_SIZE, HD);
    const int R = KVH > 0 && QH % KVH == 0 ? QH / KVH : 0;
    if (R != 1 && R != 2 && R != 3 && R != 4 && R != 8) check(L3_ERR_HEAD_RATIO, QH, "/", KVH);
}

// With kv_len the KV length is read from device memory and S only bounds it.
void decode(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out, const DecodeShape& s, int num_splits,
            int flags, const int32_t* kv_len) {
    const OnDevice on(q);
    // Outside stream capture the workspace is the one kept for the stream.  Preparing a new one synchronises,
    // which a capture does not allow, so a call under capture takes a plain buffer from the graph's memory pool
    // and runs split kernel + combine.
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    TORCH_CHECK(hipStreamIsCapturing(on.stream, &capture) == hipSuccess, "hipStreamIsCapturing failed");
    const bool capturing = capture != hipStreamCaptureStatusNone;
    flags = capturing ? flags & ~L3_ATTN_FLAG_WS_COUNTERS : flags | L3_ATTN_FLAG_WS_COUNTERS;
    const size_t nbytes = lib.l3_attn_decode_workspace_bytes(s.B, s.QH, s.KVH, s.S, s.HD, num_splits, flags);
    TensorBase own;
    void* ws = nullptr;
    std::shared_ptr<Workspace> kept;
    std::unique_lock<std::mutex> in_use;
    if (nbytes > 0 && capturing) {
        own = at::detail::empty_cuda({int64_t(std::max(nbytes, size_t(256)))}, at::kByte, q.device(), std::nullopt);
        ws = ptr(own);
    } else if (nbytes > 0) {
        kept = attention_workspace(on);
        in_use = std::unique_lock<std::mutex>(kept->in_use);
        ws = grown(*kept, q, nbytes);
    }
    const float scale = float(1.0 / std::sqrt(double(s.HD)));
    const int64_t* qs = q.strides().data();
    const int64_t* ks = k.strides().data();
    const int64_t* vs = v.strides().data();
    const int64_t* os = out.strides().data();
    const int rc = kv_len ? lib.l3_attn_decode_devlen(ptr(q), ptr(k), ptr(v), ptr(out), ws, nbytes, s.B, s.QH, s.KVH, s.S,
                                                      s.HD, qs, ks, vs, os, scale, num_splits, flags, kv_len, on.stream)
                          : lib.l3_attn_decode(ptr(q), ptr(k), ptr(v), ptr(out), ws, nbytes, s.B, s.QH, s.KVH, s.S, s.HD,
                                               qs, ks, vs, os, scale, num_splits, flags, on.stream);
    check(rc, "B=", s.B, " QH=", s.QH, " KVH=", s.KVH, " S=", s.S, " HD=", s.HD);
}

Tensor empty_like_query(const Tensor& q) {
    if (q.is_non_overlapping_and_dense()) return empty_like_dense(q);
    Tensor out = at::empty_like(q);
    return stride_at(out, 3) == 1 ? out : new_empty(q.sizes(), q);
}

// (query, keys, values, num_splits, flags)
PyObject* flash_attention_decode(PyObject* const* a) {
    const Tensor& q = gpu_bf16(a[0], "query");
    const Tensor& k = gpu_bf16(a[1], "keys");
    const Tensor& v = gpu_bf16(a[2], "values");
    const DecodeShape s = check_qkv(q, k, v);
    check_heads(s.QH, s.KVH, s.HD);
    TORCH_CHECK(s.B > 0 && s.S > 0, "flash_attention_decode needs at least one sequence and one cached token");
    const int num_splits = integer(a[3]), flags = integer(a[4]);
    return wrap(unlocked([&] {
        Tensor out = empty_like_query(q);
        decode(q, k, v, out, s, num_splits, flags, nullptr);
        return out;
    }));
}

// (query, keys, values, kv_len, num_splits, out or None, flags)
PyObject* flash_attention_decode_devlen(PyObject* const* a) {
    const Tensor& q = gpu_bf16(a[0], "query");
    const Tensor& k = gpu_bf16(a[1], "keys");
    const Tensor& v = gpu_bf16(a[2], "values");
    const DecodeShape s = check_qkv(q, k, v);
    const Tensor& len = tensor(a[3], "kv_len");
    TORCH_CHECK(len.is_cuda() && len.scalar_type() == at::kInt && len.numel() == 1 && len.device() == q.device(),
                "kv_len must be a one-element int32 tensor on the query's GPU");
    const int num_splits = integer(a[4]), flags = integer(a[6]);
    Tensor given = a[5] == Py_None ? Tensor() : tensor(a[5], "out");
    return wrap(unlocked([&] {
        Tensor out = given.defined() ? std::move(given) : empty_like_query(q);
        decode(q, k, v, out, s, num_splits, flags, static_cast<const int32_t*>(ptr(len)));
        return out;
    }));
}

// (query, keys, values, flags)
PyObject* flash_attention_prefill(PyObject* const* a) {
    const Tensor& q = gpu_bf16(a[0], "query");
    const Tensor& k = gpu_bf16(a[1], "keys");
    const Tensor& v = gpu_bf16(a[2], "values");
    TORCH_CHECK(q.dim() == 4 && k.dim() == 4 && k.sizes() == v.sizes(),
                "flash_attention_prefill expects 4-D query, keys and values (keys and values alike)");
    const auto qs = q.sizes(), ks = k.sizes();
    const int64_t B = qs[0], QH = qs[1], T = qs[2], HD = qs[3], KVH = ks[1], S = ks[2];
    TORCH_CHECK(ks[0] == B && ks[3] == HD && T <= S, "shape mismatch: query ", qs, ", keys ", ks);
    TORCH_CHECK(stride_at(q, 3) == 1 && stride_at(k, 3) == 1 && stride_at(v, 3) == 1,
                "the head dimension of query, keys and values must be contiguous");
    check_heads(int(QH), int(KVH), int(HD));
    const int flags = integer(a[3]);
    return wrap(unlocked([&] {
        // a (B, QH, T, HD) view of a contiguous (B, T, QH, HD) tensor
        const int64_t sizes[4] = {B, QH, T, HD}, strides[4] = {T * QH * HD, HD, QH * HD, 1};
        Tensor out(at::detail::empty_strided_cuda(sizes, strides, at::kBFloat16, q.device()));
        if (out.numel() > 0) {
            const OnDevice on(q);
            // partial results live for the call; where there is no memory for them the call is not cut
            size_t nbytes = lib.l3_attn_prefill_workspace_bytes(int(B), int(QH), int(KVH), int(T), int(S), int(HD), flags);
            TensorBase part;
            try {
                if (nbytes > 0) part = at::detail::empty_cuda({int64_t(nbytes)}, at::kByte, q.device(), std::nullopt);
            } catch (const c10::OutOfMemoryError&) {
                nbytes = 0;
            }
            const int rc = lib.l3_attn_prefill_ws(ptr(q), ptr(k), ptr(v), ptr(out), nbytes > 0 ? ptr(part) : nullptr, nbytes,
                                                  int(B), int(QH), int(KVH), int(T), int(S), int(HD), q.strides().data(),
                                                  k.strides().data(), v.strides().data(), strides,
                                                  float(1.0 / std::sqrt(double(HD))), flags, on.stream);
            check(rc, "B=", B, " QH=", QH, " KVH=", KVH, " T=", T, " S=", S, " HD=", HD);
        }
        return out;
    }));
}

// ------------------------------------------------------------------------------------ row-wise operators

// (input, weight, eps)
PyObject* rms_norm(PyObject* const* a) {
    const Tensor& input = gpu_bf16(a[0], "input");
    const Tensor& weight = gpu_bf16(a[1], "weight");
    TORCH_CHECK(input.dim() == 3, "rms_norm expects a 3-D (B, T, C) input");
    const int64_t C = size_at(input, 2);
    TORCH_CHECK(weight.numel() == C, "weight has ", weight.numel(), " elements, expected ", C);
    const float eps = float(number(a[2]));
    return wrap(unlocked([&] {
        Tensor xc, wc;
        const Tensor& x = contiguous(input, xc);
        const Tensor& w = contiguous(weight, wc);
        Tensor out = empty_like_dense(x);
        const int64_t rows = size_at(x, 0) * size_at(x, 1);
        if (rows > 0) {
            const OnDevice on(x);
            check(lib.l3_rms_norm(ptr(x), ptr(w), ptr(out), rows, int(C), eps, on.stream), "rows=", rows, " C=", C);
        }
        return out;
    }));
}

// (input, residual, weight, eps)
PyObject* add_rms_norm(PyObject* const* a) {
    const Tensor& input = gpu_bf16(a[0], "input");
    const Tensor& residual = gpu_bf16(a[1], "residual");
    const Tensor& weight = gpu_bf16(a[2], "weight");
    TORCH_CHECK(input.dim() == 3 && residual.sizes() == input.sizes(),
                "add_rms_norm expects two (B, T, C) tensors of the same shape");
    const int64_t C = size_at(input, 2);
    TORCH_CHECK(weight.numel() == C, "weight has ", weight.numel(), " elements, expected ", C);
    const float eps = float(number(a[3]));
    return wrap(unlocked([&] {
        Tensor xc, rc_, wc;
        const Tensor& x = contiguous(input, xc);
        const Tensor& r = contiguous(residual, rc_);
        const Tensor& w = contiguous(weight, wc);
        Tensor s = new_empty(x.sizes(), x), y = new_empty(x.sizes(), x);
        const int64_t rows = size_at(x, 0) * size_at(x, 1);
        if (rows > 0) {
            const OnDevice on(x);
            check(lib.l3_add_rms_norm(ptr(x), ptr(r), ptr(w), ptr(s), ptr(y), rows, int(C), eps, on.stream), "rows=", rows, " C=", C);
        }
        return std::pair(std::move(s), std::move(y));
    }));
}

const Tensor& partials(PyObject* o, const char* what) {
    const Tensor& part = tensor(o, "part");
    TORCH_CHECK(part.is_cuda() && part.scalar_type() == at::kFloat && part.dim() == 3 && part.is_contiguous(), what,
                ": expected contiguous float32 (ksplit, rows, N) partials");
    return part;
}

// (input, part, weight, eps)
PyObject* add_rms_norm_partials(PyObject* const* a) {
    const Tensor& input = gpu_bf16(a[0], "input");
    const Tensor& weight = gpu_bf16(a[2], "weight");
    const Tensor& part = partials(a[1], "add_rms_norm_partials");
    const int64_t C = input.dim() > 0 ? input.sizes().back() : 0;
    const int64_t rows = C > 0 ? input.numel() / C : 0;
    TORCH_CHECK(size_at(part, 1) == rows && size_at(part, 2) == C, "add_rms_norm_partials: partials ", part.sizes(),
                " do not fit input ", input.sizes());
    TORCH_CHECK(weight.numel() == C && weight.is_contiguous(), "weight has ", weight.numel(), " elements, expected ", C);
    const float eps = float(number(a[3]));
    return wrap(unlocked([&] {
        Tensor xc;
        const Tensor& x = contiguous(input, xc);
        Tensor s = new_empty(x.sizes(), x), y = new_empty(x.sizes(), x);
        const OnDevice on(x);
        check(lib.l3_add_rms_norm_partials(ptr(x), ptr(part), int(size_at(part, 0)), ptr(weight), ptr(s), ptr(y), int(rows), int(C),
                                           eps, on.stream),
              "rows=", rows, " C=", C, " ksplit=", size_at(part, 0));
        return std::pair(std::move(s), std::move(y));
    }));
}

Tensor silu_mul_of(const Tensor& a, const Tensor& b) {
    Tensor y = new_empty(a.sizes(), a);
    if (a.numel() == 0) return y;
    const OnDevice on(a);
    if (a.is_contiguous() && b.is_contiguous()) {
        check(lib.l3_silu_mul(ptr(a), ptr(b), ptr(y), y.numel(), on.stream), "n=", y.numel());
        return y;
    }
    const int64_t C = a.sizes().back(), rows = a.numel() / C;
    if (C % 8 == 0 && a.strides().back() == 1 && b.strides().back() == 1) {
        // rows with a stride (the two halves of a fused gate|up projection): no copies where the leading
        // dimensions fold into one
        const Tensor a2 = a.reshape({rows, C}), b2 = b.reshape({rows, C});
        const auto row_ok = [](const Tensor& t2, const Tensor& t) {
            return stride_at(t2, 1) == 1 && reinterpret_cast<uintptr_t>(ptr(t2)) % 16 == 0 && stride_at(t2, 0) % 8 == 0 &&
                   ptr(t2) == ptr(t);
        };
        if (row_ok(a2, a) && row_ok(b2, b)) {
            check(lib.l3_silu_mul_rows(ptr(a2), ptr(b2), ptr(y), rows, C, std::max(stride_at(a2, 0), C),
                                       std::max(stride_at(b2, 0), C), on.stream),
                  "rows=", rows, " cols=", C);
            return y;
        }
    }
    const Tensor ac = a.contiguous(), bc = b.contiguous();
    check(lib.l3_silu_mul(ptr(ac), ptr(bc), ptr(y), y.numel(), on.stream), "n=", y.numel());
    return y;
}

// (a, b)
PyObject* silu_mul(PyObject* const* args) {
    const Tensor& a = gpu_bf16(args[0], "a");
    const Tensor& b = gpu_bf16(args[1], "b");
    TORCH_CHECK(a.sizes() == b.sizes(), "silu_mul: shapes differ: ", a.sizes(), " vs ", b.sizes());
    return wrap(unlocked([&] { return silu_mul_of(a, b); }));
}

// (input, freq)
PyObject* rot_embed(PyObject* const* a) {
    const Tensor& x = gpu_bf16(a[0], "input");
    const Tensor& freq = tensor(a[1], "freq");
    TORCH_CHECK(freq.is_cuda() && freq.scalar_type() == at::kFloat, "expected a GPU float32 freq table but found ",
                freq.scalar_type(), " on ", freq.device());
    TORCH_CHECK(x.dim() == 4 && freq.dim() == 2, "rot_embed expects a 4-D (B, T, NH, HD) input and a 2-D (T, HD) freq table");
    const auto xs = x.sizes();
    TORCH_CHECK(size_at(freq, 0) == xs[1] && size_at(freq, 1) == xs[3], "freq is ", freq.sizes(), ", expected (", xs[1], ", ",
                xs[3], ")");
    TORCH_CHECK(stride_at(x, 3) == 1, "the head dimension of input must be contiguous");
    return wrap(unlocked([&] {
        Tensor fc;
        const Tensor& f = contiguous(freq, fc);
        Tensor out = new_empty(xs, x);
        if (out.numel() > 0) {
            const OnDevice on(x);
            check(lib.l3_rot_embed(ptr(x), static_cast<const float*>(ptr(f)), ptr(out), int(xs[0]), int(xs[1]), int(xs[2]),
                                   int(xs[3]), x.strides().data(), on.stream),
                  "B=", xs[0], " T=", xs[1], " NH=", xs[2], " HD=", xs[3], " strides=", x.strides());
        }
        return out;
    }));
}

// ---------------------------------------------------------------------------------------------- linears

// The activations of a linear as rows with a stride, and what is common to its argument checks.
struct Rows {
    const void* x;
    int64_t stride, K, rows;
    Tensor copy;   // keeps a rearranged copy alive
};

void check_rows(int64_t rows, int max_rows, const Tensor& x) {
    TORCH_CHECK(rows >= 1 && rows <= max_rows, "linear_decode: 1..", max_rows, " activation rows expected, got ", x.sizes());
}

// `near_each_other`: for the kernels that share activations through LDS, which address a few rows with 32 bits.
Rows linear_rows(const Tensor& x, int max_rows, bool near_each_other) {
    Rows r;
    r.K = x.dim() > 0 ? x.sizes().back() : 0;
    r.rows = r.K > 0 ? x.numel() / r.K : 0;
    check_rows(r.rows, max_rows, x);
    if (x.dim() == 2 && stride_at(x, 1) == 1) {
        r.x = ptr(x);   // rows as they are (any row stride)
        r.stride = stride_at(x, 0);
    } else if (x.is_contiguous()) {
        r.x = ptr(x);
        r.stride = r.K;
    } else {
        r.copy = x.reshape({r.rows, r.K});
        if (stride_at(r.copy, 1) != 1) r.copy = r.copy.contiguous();
        r.x = ptr(r.copy);
        r.stride = stride_at(r.copy, 0);
    }
    if (near_each_other && r.stride > L3_LINEAR_WIDE_MAX_STRIDE) {
        if (r.rows > 1) {
            r.copy = x.contiguous();
            r.x = ptr(r.copy);
        }
        r.stride = r.K;
    }
    return r;
}

void check_weight(const Tensor& w, const Tensor& like, const Tensor& x, int64_t K) {
    TORCH_CHECK(w.dim() == 2 && size_at(w, 1) == K && stride_at(w, 1) == 1 && size_at(w, 0) == size_at(like, 0) &&
                    stride_at(w, 0) == stride_at(like, 0),
                "linear_decode: weight ", w.sizes(), " does not fit x ", x.sizes());
}

// A contiguous output of x's leading shape with N columns.
Tensor rows_out(const Tensor& x, int64_t N) {
    c10::SmallVector<int64_t, 5> sizes(x.sizes().begin(), x.sizes().end());
    sizes.back() = N;
    return new_empty(sizes, x);
}

// Which kernels a linear takes.  kSkinny streams weights past operands held in registers: up to 16 rows, anything
// folded in, one launch.  kWide and kSplit share the activations through LDS (K % 128 == 0, N % 8 == 0): one launch
// where the rows of the matrix fill the device, partial products plus a finishing pass where they do not.
enum class Route { kSkinny, kWide, kSplit };

// From here on the rows of a matrix alone fill the device (64 to a workgroup; 32 of each of the SwiGLU pair).
constexpr int64_t kWideRows = 12288, kWidePairRows = 6144;

// Graph-timed over rotating weights, skinny against wide or split plus finish (us; + 2 with a norm in front, which
// is then a launch of its own): vocabulary projection 128256 x 2048, 2 rows 81 / 86, 3 rows 88 / 86, 4 rows 96 / 85, 16
// rows 139 / 87; gate|up pair 8192 x 2048, 3 rows 14.0 / 13.2, 4 rows 14.7 / 13.3, 16 rows 21.0 / 12.8; pair 14336 x
// 4096 (235 MB), 1 row 47.9 / 39.2; 2048 x 8192, 4 rows 10.2 / 10.6, 5 rows 15.4 / 10.7; 4096 x 4096, 5 rows 10.1 / 10.4, 16
// rows 12.3 / 10.6; 6144 x 4096, 2 rows 11.3 / 12.8, 5 rows 16.2 / 12.9; 4096 x 14336, 1 row 23.2 / 22.9; 2048 x 2048 and
// 3072 x 2048, 12 rows 6.7 / 6.6 and 6.9 / 7.1.  With the norm in front (inside the skinny kernel): gate|up pair 8192 x
// 2048, 4 rows 13.8 / 15.0, 5 rows 22.6 / 15.2; pair 14336 x 4096, 1 row 44.8 / 41.9.
//
// Up to 16 rows the skinny kernel says what is taken and what is refused: operands that it takes and the others do not stay
// with it, and so do those that it refuses.
Route route_of(const Rows& r, const Tensor& w, bool norm, bool pair, const Tensor* residual) {
    const int64_t K = r.K, N = size_at(w, 0);
    const bool near_rows = stride_at(w, 0) <= L3_LINEAR_WIDE_MAX_STRIDE;
    if (r.rows > L3_LINEAR_MAX_ROWS) {
        if (pair) return residual ? Route::kSkinny : Route::kWide;
        return N >= kWideRows && near_rows ? Route::kWide : Route::kSplit;
    }
    const auto misaligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 != 0; };
    if (K % 128 != 0 || N % 8 != 0 || !near_rows || misaligned(r.x) || r.stride < K || r.stride % 8 != 0) return Route::kSkinny;
    if (pair) {
        const bool large = N * K >= int64_t(32) << 20;   // each of the two
        return N >= kWidePairRows && (r.rows >= (norm ? 5 : 4) || large) ? Route::kWide : Route::kSkinny;
    }
    if (residual && residual->is_contiguous() && misaligned(ptr(*residual))) return Route::kSkinny;
    if (N >= kWideRows) return r.rows >= 4 ? Route::kWide : Route::kSkinny;
    return N * K >= int64_t(r.rows >= 5 ? 16 : 32) << 20 ? Route::kSplit : Route::kSkinny;
}

// Float32 partial products (ksplit, rows, N); ksplit 0 = the library's choice.
Tensor splitk(const Tensor& x, const Tensor& w, int ksplit) {
    const Rows r = linear_rows(x, L3_LINEAR_SPLITK_MAX_ROWS, true);
    check_weight(w, w, x, r.K);
    const int64_t N = size_at(w, 0);
    const OnDevice on(x);
    if (ksplit <= 0) {
        ksplit = lib.l3_linear_splitk_rows_plan(int(r.rows), int(N), int(r.K), 0);
        check(ksplit, "N=", N, " K=", r.K);
    }
    Tensor part = new_empty({ksplit, r.rows, N}, x, at::kFloat);
    check(lib.l3_linear_splitk(r.x, ptr(w), ptr(part), size_t(part.numel()) * 4, int(r.rows), int(N), int(r.K), r.stride,
                               stride_at(w, 0), ksplit, on.stream),
          "M=", r.rows, " N=", N, " K=", r.K, " ksplit=", ksplit);
    return part;
}

const void* residual_rows(const Tensor* residual, int64_t rows, int64_t N, Tensor& copy, const char* what) {
    if (!residual) return nullptr;
    TORCH_CHECK(residual->numel() == rows * N && residual->dim() > 0 && residual->sizes().back() == N, what, ": residual ",
                residual->sizes(), " does not fit (", rows, ", ", N, ")");
    return ptr(contiguous(*residual, copy));
}

// bf16(sum of the partials) (+ residual) into y, contiguous with rows x N elements.
void splitk_finish(const Tensor& part, const Tensor* residual, const Tensor& y) {
    const int64_t rows = size_at(part, 1), N = size_at(part, 2);
    Tensor copy;
    const void* r = residual_rows(residual, rows, N, copy, "linear_splitk_finish");
    const OnDevice on(part);
    check(lib.l3_linear_splitk_finish(ptr(part), int(size_at(part, 0)), r, ptr(y), int(rows), int(N), N, on.stream), "rows=", rows,
          " N=", N, " ksplit=", size_at(part, 0));
}

// The whole product (or, with up, the SwiGLU product of two) of up to 64 rows in one launch.
Tensor wide(const Tensor& x, const Tensor& w, const Tensor* up, const Tensor* residual) {
    const Rows r = linear_rows(x, L3_LINEAR_SPLITK_MAX_ROWS, true);
    check_weight(w, w, x, r.K);
    if (up) check_weight(*up, w, x, r.K);
    const int64_t N = size_at(w, 0);
    Tensor copy;
    const void* res = residual_rows(residual, r.rows, N, copy, "linear_decode_fused");
    Tensor y = rows_out(x, N);
    const OnDevice on(x);
    check(lib.l3_linear_wide(r.x, ptr(w), up ? ptr(*up) : nullptr, res, ptr(y), int(r.rows), int(N), int(r.K), r.stride,
                             stride_at(w, 0), N, on.stream),
          "M=", r.rows, " N=", N, " K=", r.K);
    return y;
}

// (How many rows of that width the skinny kernel's norm takes; the same limit whatever the route.)
void check_norm_weight(const Tensor& norm, int64_t rows, int64_t K, const char* what) {
    TORCH_CHECK(norm.dim() == 1 && norm.numel() == K && norm.is_contiguous(), what, ": norm_weight ", norm.sizes(),
                " does not fit K=", K);
    const int64_t most = K % 512 == 0 ? std::min<int64_t>(16, L3_LINEAR_NORM_STAGE_ELEMENTS / (K + 8)) : 0;
    TORCH_CHECK(rows <= most, what, ": the input norm takes at most ", most, " rows of width ", K, ", got ", rows);
}

// x (.. , K) normalised into a tensor of its own.
Tensor normalised(const Tensor& x, const Tensor& norm, double eps) {
    Tensor copy;
    const Tensor& xc = contiguous(x, copy);
    Tensor h = new_empty(x.sizes(), x);
    const int64_t K = x.sizes().back(), rows = x.numel() / K;
    const OnDevice on(x);
    check(lib.l3_rms_norm(ptr(xc), ptr(norm), ptr(h), rows, int(K), float(eps), on.stream), "rows=", rows, " C=", K);
    return h;
}

// The linear with what is folded into it.
Tensor linear(const Tensor& x, const Tensor& w, const Tensor* norm, double eps, const Tensor* up, const Tensor* residual) {
    const Rows r = linear_rows(x, L3_LINEAR_SPLITK_MAX_ROWS, false);
    check_weight(w, w, x, r.K);
    if (up) check_weight(*up, w, x, r.K);
    const Route route = route_of(r, w, norm != nullptr, up != nullptr, residual);
    if (route == Route::kSkinny) check_rows(r.rows, L3_LINEAR_MAX_ROWS, x);
    if (norm) check_norm_weight(*norm, r.rows, r.K, "linear_decode_fused");
    if (route != Route::kSkinny) {
        const Tensor h = norm ? normalised(x, *norm, eps) : x;
        if (route == Route::kWide) return wide(h, w, up, residual);
        const Tensor part = splitk(h, w, 0);
        Tensor y = rows_out(x, size_at(w, 0));
        splitk_finish(part, residual, y);   // the residual joins when the splits are added up
        return y;
    }
    const int64_t N = size_at(w, 0);
    Tensor copy;
    const void* res = residual_rows(residual, r.rows, N, copy, "linear_decode_fused");
    Tensor y = rows_out(x, N);
    const OnDevice on(x);
    check(lib.l3_linear_decode_fused(r.x, norm ? ptr(*norm) : nullptr, float(eps), ptr(w), up ? ptr(*up) : nullptr, res, ptr(y),
                                     int(r.rows), int(N), int(r.K), r.stride, stride_at(w, 0), N, on.stream),
          "M=", r.rows, " N=", N, " K=", r.K);
    return y;
}

// (x, weight)
PyObject* linear_decode(PyObject* const* a) {
    const Tensor &x = gpu_bf16(a[0], "x"), &w = gpu_bf16(a[1], "weight");
    return wrap(unlocked([&] { return linear(x, w, nullptr, 0.0, nullptr, nullptr); }));
}

// (x, w_gate, w_up)
PyObject* linear_swiglu_decode(PyObject* const* a) {
    const Tensor &x = gpu_bf16(a[0], "x"), &w = gpu_bf16(a[1], "weight"), &up = gpu_bf16(a[2], "weight");
    return wrap(unlocked([&] { return linear(x, w, nullptr, 0.0, &up, nullptr); }));
}

// (x, weight, norm_weight or None, eps, w_up or None, residual or None)
PyObject* linear_decode_fused(PyObject* const* a) {
    const Tensor &x = gpu_bf16(a[0], "x"), &w = gpu_bf16(a[1], "weight");
    const Tensor *norm = optional_tensor(a[2], "norm_weight"), *up = optional_tensor(a[4], "weight");
    const Tensor* residual = optional_tensor(a[5], "residual");
    const double eps = number(a[3]);
    return wrap(unlocked([&] { return linear(x, w, norm, eps, up, residual); }));
}

// (x, weight, ksplit)
PyObject* linear_splitk(PyObject* const* a) {
    const Tensor &x = gpu_bf16(a[0], "x"), &w = gpu_bf16(a[1], "weight");
    const int ksplit = integer(a[2]);
    return wrap(unlocked([&] { return splitk(x, w, ksplit); }));
}

// (part, residual or None)
PyObject* linear_splitk_finish(PyObject* const* a) {
    const Tensor& part = partials(a[0], "linear_splitk_finish");
    const Tensor* residual = optional_tensor(a[1], "residual");
    return wrap(unlocked([&] {
        Tensor y = new_empty({size_at(part, 1), size_at(part, 2)}, part);
        splitk_finish(part, residual, y);
        return y;
    }));
}

// Rotary table, position and cache of the operators that append to the KV cache.
struct Cache {
    const Tensor *k, *v, *table, *pos;
    int64_t maxB, L, KVH, HD;
};

// `like`: the activations, whose GPU all of it has to be on.
Cache cache_args(const Tensor& like, PyObject* table, PyObject* cache_k, PyObject* cache_v, PyObject* pos) {
    Cache c{&gpu_bf16(cache_k, "cache_k"), &gpu_bf16(cache_v, "cache_v"), &tensor(table, "freq_table"), &tensor(pos, "pos"),
            0, 0, 0, 0};
    TORCH_CHECK(c.k->dim() == 4 && c.k->sizes() == c.v->sizes() && c.k->strides() == c.v->strides(),
                "cache_k and cache_v must be (maxB, L, KVH, HD) tensors of the same layout");
    const auto s = c.k->sizes();
    c.maxB = s[0], c.L = s[1], c.KVH = s[2], c.HD = s[3];
    TORCH_CHECK(stride_at(*c.k, 3) == 1 && stride_at(*c.k, 2) == c.HD, "the (KVH, HD) dimensions of the cache must be contiguous");
    TORCH_CHECK(c.table->is_cuda() && c.table->scalar_type() == at::kFloat && c.table->dim() == 2 &&
                    size_at(*c.table, 1) == c.HD && c.table->is_contiguous(),
                "freq_table must be a contiguous (rows, HD) float32 GPU tensor");
    TORCH_CHECK(c.pos->is_cuda() && c.pos->scalar_type() == at::kInt && c.pos->numel() == 1,
                "pos must be a one-element int32 GPU tensor");
    for (const Tensor* t : {c.k, c.v, c.table, c.pos}) {
        TORCH_CHECK(t->device() == like.device(), "activations, freq_table, pos and the caches must be on the same device");
    }
    return c;
}

// (x, w_qkv, freq_table, cache_k, cache_v, pos, n_head, norm_weight or None, eps)
PyObject* linear_qkv_rope_append(PyObject* const* a) {
    const Tensor& x = gpu_bf16(a[0], "x");
    const Tensor& w = gpu_bf16(a[1], "weight");
    const Cache c = cache_args(x, a[2], a[3], a[4], a[5]);
    const int64_t NH = integer(a[6]);
    const Tensor* norm = optional_tensor(a[7], "norm_weight");
    const float eps = float(number(a[8]));
    return wrap(unlocked([&] {
        const Rows r = linear_rows(x, L3_LINEAR_MAX_ROWS, false);
        check_weight(w, w, x, r.K);
        TORCH_CHECK(size_at(w, 0) == (NH + 2 * c.KVH) * c.HD && r.rows <= c.maxB, "w_qkv ", w.sizes(), " does not match n_head=",
                    NH, ", cache ", c.k->sizes());
        if (norm) check_norm_weight(*norm, r.rows, r.K, "linear_qkv_rope_append");
        Tensor out = new_empty({r.rows, 1, NH, c.HD}, x);
        const OnDevice on(x);
        check(lib.l3_linear_qkv_rope_append(r.x, norm ? ptr(*norm) : nullptr, eps, ptr(w),
                                            static_cast<const float*>(ptr(*c.table)), ptr(out), ptr(*c.k), ptr(*c.v),
                                            static_cast<const int32_t*>(ptr(*c.pos)), int(r.rows), int(NH), int(c.KVH),
                                            int(c.HD), int(r.K), r.stride, stride_at(w, 0), c.k->strides().data(), int(c.L),
                                            int(size_at(*c.table, 0)), on.stream),
              "B=", r.rows, " NH=", NH, " KVH=", c.KVH, " HD=", c.HD, " K=", r.K);
        return out;
    }));
}

// (x, w_qkv, freq_table, cache_k, cache_v, pos, n_head)
PyObject* linear_qkv_rope_append_rows(PyObject* const* a) {
    const Tensor& x = gpu_bf16(a[0], "x");
    const Tensor& w = gpu_bf16(a[1], "weight");
    const Cache c = cache_args(x, a[2], a[3], a[4], a[5]);
    const int64_t NH = integer(a[6]);
    return wrap(unlocked([&] {
        const Rows r = linear_rows(x, L3_LINEAR_SPLITK_MAX_ROWS, true);
        check_weight(w, w, x, r.K);
        TORCH_CHECK(size_at(w, 0) == (NH + 2 * c.KVH) * c.HD && r.rows <= c.maxB, "w_qkv ", w.sizes(), " does not match n_head=",
                    NH, ", cache ", c.k->sizes());
        Tensor out = new_empty({r.rows, 1, NH, c.HD}, x);
        const OnDevice on(x);
        check(lib.l3_linear_qkv_rope_append_rows(r.x, ptr(w), static_cast<const float*>(ptr(*c.table)), ptr(out), ptr(*c.k),
                                                 ptr(*c.v), static_cast<const int32_t*>(ptr(*c.pos)), int(r.rows), int(NH),
                                                 int(c.KVH), int(c.HD), int(r.K), r.stride, stride_at(w, 0),
                                                 c.k->strides().data(), int(c.L), int(size_at(*c.table, 0)), on.stream),
              "B=", r.rows, " NH=", NH, " KVH=", c.KVH, " HD=", c.HD, " K=", r.K);
        return out;
    }));
}

// (part, freq_table, cache_k, cache_v, pos, n_head)
PyObject* rot_embed_append_partials(PyObject* const* a) {
    const Tensor& part = partials(a[0], "rot_embed_append_partials");
    const Cache c = cache_args(part, a[1], a[2], a[3], a[4]);
    const int64_t NH = integer(a[5]), ksplit = size_at(part, 0), B = size_at(part, 1);
    TORCH_CHECK(size_at(part, 2) == (NH + 2 * c.KVH) * c.HD && B <= c.maxB, "partials ", part.sizes(), " do not match n_head=", NH,
                ", cache ", c.k->sizes());
    return wrap(unlocked([&] {
        Tensor out = new_empty({B, 1, NH, c.HD}, part);
        const OnDevice on(part);
        check(lib.l3_rot_embed_append_partials(static_cast<const float*>(ptr(part)), int(ksplit),
                                               static_cast<const float*>(ptr(*c.table)), ptr(out), ptr(*c.k), ptr(*c.v),
                                               static_cast<const int32_t*>(ptr(*c.pos)), int(B), int(NH), int(c.KVH), int(c.HD),
                                               c.k->strides().data(), int(c.L), int(size_at(*c.table, 0)), on.stream),
              "B=", B, " NH=", NH, " KVH=", c.KVH, " HD=", c.HD, " ksplit=", ksplit);
        return out;
    }));
}

// --------------------------------------------------------------------------------------------- the module

template <PyObject* (*F)(PyObject* const*), int N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != N) {
        PyErr_Format(PyExc_TypeError, "%d arguments expected, got %zd", N, n);
        return nullptr;
    }
    if (!lib.l3_strerror) {
        PyErr_SetString(PyExc_RuntimeError, "bind() has not been called");
        return nullptr;
    }
    try {
        return F(args);
    } catch (python_error& e) {
        e.restore();
    } catch (...) {
        torch::translate_exception_to_python(std::current_exception());
    }
    return nullptr;
}

// bind(path): looks the library's functions up; the Python side has loaded it from the same path.
PyObject* bind(PyObject*, PyObject* arg) {
    const char* path = PyUnicode_AsUTF8(arg);
    if (!path) return nullptr;
    void* handle = dlopen(path, RTLD_NOW | RTLD_LOCAL);
    if (!handle) {
        PyErr_Format(PyExc_ImportError, "%s: %s", path, dlerror());
        return nullptr;
    }
    Library found;
#define X(name)                                                                       \
    if (!(found.name = reinterpret_cast<decltype(found.name)>(dlsym(handle, #name)))) { \
        PyErr_Format(PyExc_ImportError, "%s has no " #name, path);                    \
        return nullptr;                                                               \
    }
    L3_FUNCTIONS(X)
#undef X
    lib = found;
    Py_RETURN_NONE;
}

#define ENTRY(name, n) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<name, n>)), METH_FASTCALL, nullptr}

PyMethodDef methods[] = {
    {"bind", bind, METH_O, nullptr},
    ENTRY(flash_attention_decode, 5),
    ENTRY(flash_attention_decode_devlen, 7),
    ENTRY(flash_attention_prefill, 4),
    ENTRY(rms_norm, 3),
    ENTRY(add_rms_norm, 4),
    ENTRY(add_rms_norm_partials, 4),
    ENTRY(silu_mul, 2),
    ENTRY(rot_embed, 2),
    ENTRY(linear_decode, 2),
    ENTRY(linear_swiglu_decode, 3),
    ENTRY(linear_decode_fused, 6),
    ENTRY(linear_splitk, 3),
    ENTRY(linear_splitk_finish, 2),
    ENTRY(linear_qkv_rope_append, 9),
    ENTRY(linear_qkv_rope_append_rows, 7),
    ENTRY(rot_embed_append_partials, 6),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef definition = {PyModuleDef_HEAD_INIT, "_l3torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__l3torch() { return PyModule_Create(&definition); }
