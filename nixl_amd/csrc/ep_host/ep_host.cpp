// The allocations and launches of nixl_amd.ep.Buffer's calls, as one native call each.
//
// A small call is bound by its host: torch.empty from Python takes 1.7 us and a launch through ctypes 1.5 us
// more than the launch itself, and a low-latency dispatch allocates seven tensors, a normal-mode dispatch nine.
// From here the same allocations go through the same dispatcher (and its caching allocator and modes) at a
// third of that.  Passes of dispatch and combine, us: 8 ranks x 2 tokens x 7168 27.9 -> 18.2, 16 x 61 x 2560 from
// logits 31.3 -> 22.4, normal mode 4 x 333 x 4096 58.2 -> 37.3; passes that the GPU bounds stay as they are.
// Arguments are checked in ep.py; what comes here is tensors, None, and plain integers.
#define PY_SSIZE_T_CLEAN
#include <torch/csrc/python_headers.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/slice.h>
#include <ATen/ops/transpose.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <chrono>
#include <cstdint>
#include <initializer_list>
#include <string>

#include "nixl_amd_ep.h"

namespace {

// The interpreter goes on with other threads while this one allocates, launches and waits.
class NoGil {
public:
    NoGil() : state_(PyEval_SaveThread()) {}
    ~NoGil() { PyEval_RestoreThread(state_); }
    NoGil(const NoGil &) = delete;
    NoGil &operator=(const NoGil &) = delete;

    // Signal handlers that are due, as between two lines of Python.
    void
    look_at_signals() {
        PyEval_RestoreThread(state_);
        python_error raised;
        const bool any = PyErr_CheckSignals() != 0;
        if (any) raised.persist();
        state_ = PyEval_SaveThread();
        if (any) throw raised;
    }

private:
    PyThreadState *state_;
};

// The arguments of a call, taken in order.
class Args {
public:
    Args(const char *what, PyObject *const *args, Py_ssize_t n, Py_ssize_t expected) : what_(what), next_(args) {
        if (n != expected) throw py_type(std::to_string(expected) + " arguments");
    }

    // None: a tensor that is not defined.
    at::Tensor
    tensor() {
        PyObject *const o = *next_++;
        if (o == Py_None) return {};
        if (!THPVariable_Check(o)) throw py_type("a tensor or None");
        return THPVariable_Unpack(o);
    }

    // Whatever stands for an integer in Python: NumPy's integers and tensors of one too.
    int64_t
    integer() {
        PyObject *const o = *next_++;
        if (!PyIndex_Check(o)) throw py_type("an integer");
        PyObject *const number = PyNumber_Index(o);
        if (!number) throw python_error();
        const int64_t v = PyLong_AsLongLong(number);
        Py_DECREF(number);
        if (v == -1 && PyErr_Occurred()) throw python_error();
        return v;
    }

    // What the entry points of the kernels take.
    int
    small() {
        const int64_t v = integer();
        if (v != static_cast<int>(v)) throw py_type("an integer of 32 bits");
        return static_cast<int>(v);
    }

    void *
    pointer() {
        PyObject *const o = *next_++;
        if (o == Py_None) return nullptr;
        void *const p = PyLong_AsVoidPtr(o);
        if (!p && PyErr_Occurred()) throw python_error();
        return p;
    }

    double
    real() {
        const double v = PyFloat_AsDouble(*next_++);
        if (v == -1.0 && PyErr_Occurred()) throw python_error();
        return v;
    }

private:
    torch::TypeError
    py_type(const std::string &expected) const {
        return torch::TypeError(std::string(what_) + ": " + expected + " expected");
    }

    const char *const what_;
    PyObject *const *next_;
};

template<typename T = void>
T *
ptr(const at::Tensor &t) {
    return t.defined() ? static_cast<T *>(t.data_ptr()) : nullptr;
}

at::Tensor
empty(std::initializer_list<int64_t> shape, at::ScalarType type, at::Device device) {
    return at::empty(at::IntArrayRef(shape.begin(), shape.size()), at::TensorOptions().dtype(type).device(device));
}

// Tensors (None where not defined) with `rc` behind them.
PyObject *
pack(int rc, std::initializer_list<at::Tensor> tensors) {
    PyObject *const out = PyTuple_New(static_cast<Py_ssize_t>(tensors.size()) + 1);
    if (!out) throw python_error();
    Py_ssize_t i = 0;
    for (const at::Tensor &t : tensors) {
        PyObject *const o = THPVariable_Wrap(t); // None for one that is not defined
        if (!o) {
            Py_DECREF(out);
            throw python_error();
        }
        PyTuple_SET_ITEM(out, i++, o);
    }
    PyObject *const status = PyLong_FromLong(rc);
    if (!status) {
        Py_DECREF(out);
        throw python_error();
    }
    PyTuple_SET_ITEM(out, i, status);
    return out;
}

// (x, topk_idx | None, logits | None, workspace | None, stats | None, tokens per rank | None, mask address | None,
//  local experts, rows of an expert, K, max tokens, experts, fp8, round_scale, ue8m0, launch, stream) ->
// (rows, scales | None, src_info, layout_range, count, row_map, topk_idx, topk_weights | None, workspace, rc); the
// scales as a view with the expert's rows in front of the groups of channels.
// Without `launch` the tensors are made and nothing is queued.
PyObject *
ll_dispatch(PyObject *, PyObject *const *argv, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Args a("ll_dispatch", argv, n, 17);
    const at::Tensor x = a.tensor();
    at::Tensor topk_idx = a.tensor();
    const at::Tensor logits = a.tensor();
    at::Tensor workspace = a.tensor();
    const at::Tensor stats = a.tensor(), tokens_per_rank = a.tensor();
    void *const mask = a.pointer();
    const int64_t El = a.integer(), N = a.integer();
    const int K = a.small(), max_tokens = a.small(), experts = a.small();
    const bool fp8 = a.small(), round_scale = a.small(), ue8m0 = a.small(), launch = a.small();
    void *const stream = a.pointer();
    const int64_t R = x.size(0), T = x.size(1), H = x.size(2);
    at::Tensor rows, scales, src_info, layout, count, row_map, weights;
    int rc = 0;
    {
        NoGil no_gil;
        const at::Device dev = x.device();
        rows = empty({R, El, N, H}, fp8 ? at::kFloat8_e4m3fn : at::kBFloat16, dev);
        src_info = empty({R, El, N}, at::kInt, dev);
        layout = empty({R, El, R}, at::kLong, dev);
        count = empty({R, El}, at::kInt, dev);
        if (fp8) scales = ue8m0 ? empty({R, El, H / 512, N}, at::kInt, dev) : empty({R, El, H / 128, N}, at::kFloat, dev);
        row_map = empty({R, T, K}, at::kInt, dev);
        const int r = static_cast<int>(R), t = static_cast<int>(T), h = static_cast<int>(H);
        const size_t need = nixl_amd_ep_ll_workspace_bytes(r, experts, t, K, h);
        if (!workspace.defined() || static_cast<size_t>(workspace.numel()) < need)
            workspace = empty({std::max<int64_t>(static_cast<int64_t>(need), 1)}, at::kByte, x.device());
        if (logits.defined()) {
            topk_idx = empty({R, T, K}, at::kInt, dev);
            weights = empty({R, T, K}, at::kFloat, dev);
        }
        const size_t bytes = static_cast<size_t>(workspace.numel());
        if (launch && logits.defined())
            rc = nixl_amd_ep_ll_route_dispatch(ptr(rows), ptr(scales), ptr<int>(src_info), ptr<int64_t>(layout), ptr<int>(count),
                                               static_cast<const int *>(mask), ptr<int>(stats), ptr(x), ptr<float>(logits),
                                               ptr<int32_t>(topk_idx), ptr<float>(weights), ptr<int>(tokens_per_rank), t, h,
                                               max_tokens, K, r, experts, fp8, round_scale, ue8m0, ptr<int>(row_map),
                                               ptr(workspace), bytes, stream);
        else if (launch)
            rc = nixl_amd_ep_ll_dispatch(ptr(rows), ptr(scales), ptr<int>(src_info), ptr<int64_t>(layout), ptr<int>(count),
                                         static_cast<const int *>(mask), ptr<int>(stats), ptr(x), ptr<int32_t>(topk_idx),
                                         ptr<int>(tokens_per_rank), t, h, max_tokens, K, r, experts, fp8, round_scale, ue8m0,
                                         ptr<int>(row_map), ptr(workspace), bytes, stream);
        if (fp8) scales = scales.transpose(2, 3);
    }
    return pack(rc, {rows, scales, src_info, layout, count, row_map, topk_idx, weights, workspace});
    END_HANDLE_TH_ERRORS
}

// (out | None, x, topk_idx, topk_weights, src_info, layout_range, tokens per rank | None, row_map | None,
//  mask address | None, hidden, max tokens, logfmt, stream) -> (combined, rc).
PyObject *
ll_combine(PyObject *, PyObject *const *argv, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Args a("ll_combine", argv, n, 13);
    at::Tensor combined = a.tensor();
    const at::Tensor x = a.tensor(), topk_idx = a.tensor(), weights = a.tensor(), src_info = a.tensor(), layout = a.tensor();
    const at::Tensor tokens_per_rank = a.tensor(), row_map = a.tensor();
    void *const mask = a.pointer();
    const int hidden = a.small(), max_tokens = a.small();
    const bool logfmt = a.small();
    void *const stream = a.pointer();
    const int64_t R = topk_idx.size(0), T = topk_idx.size(1), K = topk_idx.size(2);
    int rc = 0;
    {
        NoGil no_gil;
        if (!combined.defined()) combined = empty({R, T, hidden}, at::kBFloat16, x.device());
        rc = nixl_amd_ep_ll_combine(ptr(combined), ptr(x), ptr<int32_t>(topk_idx), ptr<float>(weights), ptr<int>(src_info),
                                    ptr<int64_t>(layout), static_cast<const int *>(mask), ptr<int>(tokens_per_rank),
                                    ptr<int>(row_map), static_cast<int>(T), hidden, max_tokens, static_cast<int>(K),
                                    static_cast<int>(R), static_cast<int>(x.size(1) * R), logfmt, stream);
    }
    return pack(rc, {combined});
    END_HANDLE_TH_ERRORS
}

// (topk_idx, experts, stream) -> (per_rank, per_expert, in_rank, rc).
PyObject *
layout(PyObject *, PyObject *const *argv, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Args a("layout", argv, n, 3);
    const at::Tensor topk_idx = a.tensor();
    const int experts = a.small();
    void *const stream = a.pointer();
    const int64_t R = topk_idx.size(0), T = topk_idx.size(1), K = topk_idx.size(2);
    at::Tensor per_rank, per_expert, in_rank;
    int rc = 0;
    {
        NoGil no_gil;
        const at::Device dev = topk_idx.device();
        per_rank = empty({R, R}, at::kInt, dev);
        per_expert = empty({R, experts}, at::kInt, dev);
        in_rank = empty({R, T, R}, at::kBool, dev);
        rc = nixl_amd_ep_get_dispatch_layout(ptr<int32_t>(topk_idx), ptr<int>(per_rank), ptr<int>(per_expert),
                                             ptr<uint8_t>(in_rank), static_cast<int>(T), static_cast<int>(K),
                                             static_cast<int>(R), experts, stream);
    }
    return pack(rc, {per_rank, per_expert, in_rank});
    END_HANDLE_TH_ERRORS
}

struct Received {
    at::Tensor x, scales, idx, weights, meta;
};

int
dispatch_rows(const Received &to, const at::Tensor &x, const at::Tensor &scales, const at::Tensor &idx, const at::Tensor &weights,
              const at::Tensor &in_rank, const at::Tensor &prefix, const at::Tensor &send_head, const at::Tensor &row_offset,
              int K, int experts, void *stream) {
    const bool scaled = scales.defined();
    return nixl_amd_ep_ht_dispatch_scaled(
        ptr(to.x), ptr(to.scales), ptr<int32_t>(to.idx), ptr<float>(to.weights), ptr<int32_t>(to.meta), ptr(x), ptr(scales),
        ptr<int32_t>(idx), ptr<float>(weights), ptr<uint8_t>(in_rank), ptr<int>(prefix), ptr<int>(send_head),
        ptr<int64_t>(row_offset), static_cast<int>(x.size(1)), static_cast<int>(x.size(2)), static_cast<int>(x.element_size()),
        scaled ? static_cast<int>(scales.size(2)) : 0, scaled ? scales.stride(0) : 0, scaled ? scales.stride(1) : 0,
        scaled ? scales.stride(2) : 0, K, static_cast<int>(x.size(0)), experts, stream);
}

Received
empty_rows(int64_t rows, const at::Tensor &x, const at::Tensor &scales, int64_t K, bool meta) {
    const at::Device dev = x.device();
    Received r;
    r.x = empty({rows, x.size(2)}, x.scalar_type(), dev);
    if (scales.defined()) r.scales = empty({rows, scales.size(2)}, scales.scalar_type(), dev);
    if (K) {
        r.idx = empty({rows, K}, at::kInt, dev);
        r.weights = empty({rows, K}, at::kFloat, dev);
    }
    if (meta) r.meta = empty({rows, 2}, at::kInt, dev);
    return r;
}

// (x, scales | None, in_rank, prefix, send_head, row_offset, rows, stream) -> (recv_x, recv_scales | None, rc).
PyObject *
ht_dispatch_cached(PyObject *, PyObject *const *argv, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Args a("ht_dispatch_cached", argv, n, 8);
    const at::Tensor x = a.tensor(), scales = a.tensor(), in_rank = a.tensor(), prefix = a.tensor(), send_head = a.tensor();
    const at::Tensor row_offset = a.tensor();
    const int64_t rows = a.integer();
    void *const stream = a.pointer();
    Received to;
    int rc = 0;
    {
        NoGil no_gil;
        to = empty_rows(rows, x, scales, 0, false);
        rc = dispatch_rows(to, x, scales, {}, {}, in_rank, prefix, send_head, row_offset, 0, static_cast<int>(x.size(0)), stream);
    }
    return pack(rc, {to.x, to.scales});
    END_HANDLE_TH_ERRORS
}

// Until the GPU has written every count.  Looks at Python's signals now and then, as a loop in Python would.
bool
wait_counts(const int32_t *counts, int64_t n, double seconds, NoGil &no_gil) {
    using Clock = std::chrono::steady_clock;
    const auto begin = Clock::now();
    int64_t seen = 0;
    for (uint32_t looks = 1;; ++looks) {
        while (seen < n && __atomic_load_n(counts + seen, __ATOMIC_ACQUIRE) >= 0)
            ++seen;
        if (seen == n) return true;
        __builtin_ia32_pause();
        if (looks % 65536) continue;
        if (std::chrono::duration<double>(Clock::now() - begin).count() > seconds) return false;
        no_gil.look_at_signals();
    }
}

// What the second half of ht_dispatch's status says.
constexpr int kNotify = 1; // the first half is the counts' launch's
constexpr int kLate = 2; // the counts did not arrive in time

// (x, scales | None, in_rank, per_expert, topk_idx | None, topk_weights | None, host counts, local experts, channels,
//  alignment, worst-case rows, seconds, stream) ->
// (recv_x, recv_scales | None, recv_idx | None, recv_weights | None, recv_meta, prefix, chan, send_head, row_offset,
//  (rc, stage)): `host counts` is a pinned int32 tensor of R + R * local experts words, where the counts are
// left; with `worst-case rows` the rows are queued behind the counts into tensors that hold any number of them.
PyObject *
ht_dispatch(PyObject *, PyObject *const *argv, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Args a("ht_dispatch", argv, n, 13);
    const at::Tensor x = a.tensor(), scales = a.tensor(), in_rank = a.tensor(), per_expert = a.tensor();
    const at::Tensor idx = a.tensor(), weights = a.tensor(), mapped = a.tensor();
    const int64_t El = a.integer();
    const int channels = a.small(), alignment = a.small();
    const bool ahead = a.small();
    const double seconds = a.real();
    void *const stream = a.pointer();
    const int64_t R = x.size(0), T = x.size(1), K = idx.defined() ? idx.size(2) : 0, E = per_expert.size(1);
    at::Tensor prefix, chan, send_head, row_offset;
    Received to;
    int rc = 0, stage = 0;
    {
        NoGil no_gil;
        const at::Device dev = x.device();
        prefix = empty({R, R}, at::kInt, dev);
        chan = empty({R, R, channels}, at::kInt, dev);
        send_head = empty({R, T, R}, at::kInt, dev);
        row_offset = empty({R + 1}, at::kLong, dev);
        int32_t *const counts = ptr<int32_t>(mapped);
        const int64_t n_counts = R + R * El;
        std::fill_n(counts, n_counts, -1);
        rc = nixl_amd_ep_ht_notify_dispatch(ptr<uint8_t>(in_rank), ptr<int>(per_expert), ptr<int>(prefix), counts + R,
                                            ptr<int>(chan), ptr<int>(send_head), ptr<int64_t>(row_offset), counts,
                                            static_cast<int>(T), static_cast<int>(R), static_cast<int>(E), channels, alignment,
                                            stream);
        if (rc != 0) stage = kNotify;
        const auto total = [&] {
            int64_t sum = 0;
            for (int64_t r = 0; r < R; ++r)
                sum += counts[r];
            return sum;
        };
        if (rc == 0 && !ahead && !wait_counts(counts, n_counts, seconds, no_gil)) stage = kLate;
        if (stage == 0) {
            to = empty_rows(ahead ? R * T * R : total(), x, scales, K, true);
            rc = dispatch_rows(to, x, scales, idx, weights, in_rank, prefix, send_head, row_offset, static_cast<int>(K),
                               static_cast<int>(E), stream);
        }
        if (rc == 0 && stage == 0 && ahead) {
            if (!wait_counts(counts, n_counts, seconds, no_gil)) {
                stage = kLate;
            } else {
                const int64_t rows = total();
                for (at::Tensor *t : {&to.x, &to.scales, &to.idx, &to.weights, &to.meta})
                    if (t->defined()) *t = t->slice(0, 0, rows);
            }
        }
    }
    PyObject *const out = pack(rc, {to.x, to.scales, to.idx, to.weights, to.meta, prefix, chan, send_head, row_offset});
    PyObject *const status = Py_BuildValue("(ii)", rc, stage);
    if (!status) {
        Py_DECREF(out);
        throw python_error();
    }
    PyTuple_SetItem(out, PyTuple_GET_SIZE(out) - 1, status);
    return out;
    END_HANDLE_TH_ERRORS
}

// (x, topk_weights | None, bias | None, bias | None, in_rank, prefix, send_head, row_offset, stream) ->
// (combined, combined weights | None, rc).
PyObject *
ht_combine(PyObject *, PyObject *const *argv, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Args a("ht_combine", argv, n, 9);
    const at::Tensor x = a.tensor(), weights = a.tensor(), bias_0 = a.tensor(), bias_1 = a.tensor(), in_rank = a.tensor();
    const at::Tensor prefix = a.tensor(), send_head = a.tensor(), row_offset = a.tensor();
    void *const stream = a.pointer();
    const int64_t R = in_rank.size(0), T = in_rank.size(1), H = x.size(1), K = weights.defined() ? weights.size(1) : 0;
    at::Tensor combined, combined_w;
    int rc = 0;
    {
        NoGil no_gil;
        combined = empty({R, T, H}, at::kBFloat16, x.device());
        if (K) combined_w = empty({R, T, K}, at::kFloat, x.device());
        rc = nixl_amd_ep_ht_combine_rows(ptr(combined), ptr<float>(combined_w), ptr(x), ptr<float>(weights), ptr(bias_0),
                                         ptr(bias_1), ptr<uint8_t>(in_rank), ptr<int>(prefix), ptr<int>(send_head),
                                         ptr<int64_t>(row_offset), x.size(0), static_cast<int>(T), static_cast<int>(H),
                                         static_cast<int>(std::max<int64_t>(K, 1)), static_cast<int>(R), stream);
    }
    return pack(rc, {combined, combined_w});
    END_HANDLE_TH_ERRORS
}

template<PyObject *(*F)(PyObject *, PyObject *const *, Py_ssize_t)>
constexpr PyMethodDef
method(const char *name) {
    return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(F)), METH_FASTCALL, nullptr};
}

PyMethodDef methods[] = {
    method<ll_dispatch>("ll_dispatch"),
    method<ll_combine>("ll_combine"),
    method<layout>("layout"),
    method<ht_dispatch_cached>("ht_dispatch_cached"),
    method<ht_dispatch>("ht_dispatch"),
    method<ht_combine>("ht_combine"),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ep_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC
PyInit__ep_host() {
    return PyModule_Create(&module);
}
