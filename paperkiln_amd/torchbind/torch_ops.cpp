// The attention operators of paperkiln_amd.ops on torch tensors, as native code: argument checks, output allocation, the
// C ABI call and the autograd node. Python keeps the signatures (ops.py) and hands its arguments over in one call.
//
// What bounds it: nothing but host instructions. A small attention call is 10-60 us of GPU work, and in Python the same
// path (ctypes structures, torch.empty and tensor properties one by one, a Python autograd.Function whose backward takes
// the interpreter lock on the engine's thread) cost 34 us for a forward + backward pair and 165-195 us under autograd.
// All arithmetic still runs in libpaperkiln_amd.so.
#include <Python.h>
#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/utils/python_numbers.h>

#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "paperkiln_amd.h"

namespace {

using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

PyObject* g_error = nullptr;  // paperkiln_amd._lib.PkError

// A refused C ABI call as the package's own exception, on any thread (the autograd engine's included).
void check(int rc) {
    if (rc == PK_OK) return;
    const std::string msg = pk_last_error();
    pybind11::gil_scoped_acquire gil;
    if (PyObject* e = PyObject_CallFunction(g_error, "is", rc, msg.c_str())) {
        PyErr_SetObject(g_error, e);
        Py_DECREF(e);
    }
    throw python_error();
}

int dtype_code(at::ScalarType t) {
    if (t == at::kFloat) return PK_F32;
    if (t == at::kBFloat16) return PK_BF16;
    throw std::runtime_error("dtype must be float32 or bfloat16");
}

struct Mask {
    double scale;
    bool causal;
    int window, sinks;
    // > 0: the tensors are one head's [rows, dk] matrices of stacked sequences of this many tokens, as the reference's
    // operators take them (paperkiln src/ops.cpp:869-879); 0: [B, T, H, dk]
    int64_t seq_len = 0;
};

pk_tensor4 view4(const Tensor& x, const Mask& m) {
    if (m.seq_len > 0 && x.dim() == 2 && x.stride(1) == 1)
        return pk_tensor4{x.data_ptr(), m.seq_len * x.stride(0), x.stride(0), x.size(1)};
    if (m.seq_len > 0 || x.dim() != 4 || x.stride(3) != 1)
        throw std::runtime_error("expected a [B,T,H,dk] tensor with contiguous head_dim");
    return pk_tensor4{x.data_ptr(), x.stride(0), x.stride(1), x.stride(2)};
}

pk_attn_shape shape_of(const Tensor& q, const Tensor& k, const Mask& m, at::ScalarType grad) {
    const bool head = m.seq_len > 0;
    if (q.dim() != (head ? 2 : 4) || k.dim() != q.dim()) throw std::runtime_error("fused_attention: shape mismatch");
    pk_attn_shape s;
    s.B = static_cast<int32_t>(head ? q.size(0) / m.seq_len : q.size(0)), s.T = static_cast<int32_t>(head ? m.seq_len : q.size(1));
    s.Hq = head ? 1 : static_cast<int32_t>(q.size(2)), s.Hkv = head ? 1 : static_cast<int32_t>(k.size(2));
    s.dk = static_cast<int32_t>(q.size(-1));
    s.causal = m.causal, s.window = m.window, s.sinks = m.sinks;
    s.scale = static_cast<float>(m.scale);
    s.dtype = dtype_code(q.scalar_type()), s.grad_dtype = dtype_code(grad);
    return s;
}

void* stream() { return at::hip::getCurrentHIPStream().stream(); }

Tensor empty_of(at::IntArrayRef sizes, at::ScalarType t, const Tensor& like) {
    return at::empty(sizes, like.options().dtype(t).memory_format(c10::nullopt));
}

std::pair<Tensor, Tensor> forward(const Tensor& q, const Tensor& k, const Tensor& v, const Mask& m) {
    if (!q.is_cuda()) throw std::runtime_error("paperkiln_amd has no CPU path: tensors must live on the GPU");
    const pk_attn_shape s = shape_of(q, k, m, q.scalar_type());
    if (k.sizes() != v.sizes() || k.size(0) != q.size(0) || k.size(-1) != q.size(-1) || (m.seq_len == 0 && k.size(1) != q.size(1)))
        throw std::runtime_error("fused_attention: shape mismatch");
    if (k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type())
        throw std::runtime_error("fused_attention: dtype mismatch");
    at::AutoDispatchBelowAutograd below;
    Tensor o = empty_of(q.sizes(), q.scalar_type(), q);
    Tensor lse = empty_of({s.B, s.Hq, s.T}, at::kFloat, q);
    const pk_tensor4 q4 = view4(q, m), k4 = view4(k, m), v4 = view4(v, m), o4 = view4(o, m);
    check(pk_attn_fwd(&s, &q4, &k4, &v4, &o4, static_cast<float*>(lse.data_ptr()), stream()));
    return {std::move(o), std::move(lse)};
}

struct Grads {
    Tensor dq, dk, dv;
};

// `out`: dq, dk, dv and the workspace, or nullptr for new ones
Grads backward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& lse, const Tensor& d_o,
               const Mask& m, at::ScalarType grad, const Tensor* out, int stages) {
    const pk_attn_shape s = shape_of(q, k, m, grad);
    at::AutoDispatchBelowAutograd below;
    Grads g;
    Tensor ws;
    if (out) {
        g = Grads{out[0], out[1], out[2]};
        ws = out[3];
    } else {
        g = Grads{empty_of(q.sizes(), grad, q), empty_of(k.sizes(), grad, q), empty_of(v.sizes(), grad, q)};
        const int64_t bytes = static_cast<int64_t>(pk_attn_bwd_workspace_bytes(&s));
        ws = empty_of({bytes > 16 ? bytes : 16}, at::kByte, q);
    }
    const pk_tensor4 q4 = view4(q, m), k4 = view4(k, m), v4 = view4(v, m), o4 = view4(o, m), g4 = view4(d_o, m),
                     dq4 = view4(g.dq, m), dk4 = view4(g.dk, m), dv4 = view4(g.dv, m);
    check(pk_attn_bwd_stages(&s, &q4, &k4, &v4, &o4, static_cast<const float*>(lse.data_ptr()), &g4, &dq4, &dk4, &dv4,
                             ws.data_ptr(), static_cast<size_t>(ws.numel()), stages, stream()));
    return g;
}

// Tape node that keeps O and LSE only (plus its parents Q, K, V), in place of the reference closure's captured [T,T]
// matrix A (paperkiln src/ops.cpp:902).
struct AttentionBackward : public Node {
    SavedVariable q, k, v, o, lse;
    Mask mask{};

    explicit AttentionBackward(torch::autograd::edge_list&& next) : Node(std::move(next)) {}
    std::string name() const override { return "AttentionBackward"; }
    // Backward passes of two threads may share this node, and one that does not keep the graph releases it: under the node's
    // lock, like every node that holds tensors.
    void release_variables() override {
        const std::lock_guard<std::mutex> lock(mutex_);
        q.reset_data(), k.reset_data(), v.reset_data(), o.reset_data(), lse.reset_data();
    }
    variable_list apply(variable_list&& in) override {
        const auto self = getptr();
        Tensor tq, tk, tv, to, tl;
        {
            const std::lock_guard<std::mutex> lock(mutex_);
            tq = q.unpack(), tk = k.unpack(), tv = v.unpack(), to = o.unpack(self), tl = lse.unpack();
        }
        Tensor d_o = in[0].defined() ? in[0] : at::zeros_like(to);
        if (d_o.stride(-1) != 1) d_o = d_o.contiguous();
        Grads g = backward(tq, tk, tv, to, tl, d_o, mask, tq.scalar_type(), nullptr, PK_BWD_ALL);
        return {std::move(g.dq), std::move(g.dk), std::move(g.dv)};
    }
};

Tensor attention(const Tensor& q, const Tensor& k, const Tensor& v, const Mask& m) {
    for (const Tensor* x : {&q, &k, &v})  // a tangent would be dropped without a word
        if (x->_fw_grad(0).defined()) throw std::runtime_error("attention: forward-mode differentiation is not implemented");
    auto [o, lse] = forward(q, k, v, m);
    if (at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad())) {
        auto node = std::shared_ptr<AttentionBackward>(new AttentionBackward(torch::autograd::collect_next_edges(q, k, v)),
                                                       torch::autograd::deleteNode);
        torch::autograd::set_history(o, node);
        node->q = SavedVariable(q, false), node->k = SavedVariable(k, false), node->v = SavedVariable(v, false);
        node->o = SavedVariable(o, true), node->lse = SavedVariable(lse, false);
        node->mask = m;
    }
    return o;
}

// ---- Python side: positional arguments in the order ops.py passes them ----

const Tensor& tensor_arg(PyObject* o, const char* what) {
    if (!THPVariable_Check(o)) throw torch::TypeError(std::string(what) + " must be a tensor, not " + Py_TYPE(o)->tp_name);
    return THPVariable_Unpack(o);
}
int int_arg(PyObject* o) {  // what Python's int() takes, inside 32 bits
    PyObject* i = PyNumber_Long(o);
    if (!i) throw python_error();
    const long x = PyLong_AsLong(i);
    Py_DECREF(i);
    if (x == -1 && PyErr_Occurred()) throw python_error();
    return static_cast<int>(x);
}
double float_arg(PyObject* o) {
    const double x = PyFloat_AsDouble(o);
    if (x == -1.0 && PyErr_Occurred()) throw python_error();
    return x;
}
bool bool_arg(PyObject* o) {
    const int x = PyObject_IsTrue(o);
    if (x < 0) throw python_error();
    return x != 0;
}
Mask mask_args(PyObject* const* a) { return Mask{float_arg(a[0]), bool_arg(a[1]), int_arg(a[2]), int_arg(a[3]), 0}; }
void expect(Py_ssize_t n, Py_ssize_t want) {
    if (n != want) throw torch::TypeError("expected " + std::to_string(want) + " arguments, got " + std::to_string(n));
}

// (q, k, v, scale, causal, window, sinks) -> (o, lse)
PyObject* py_fwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    expect(n, 7);
    const Tensor &q = tensor_arg(a[0], "q"), &k = tensor_arg(a[1], "k"), &v = tensor_arg(a[2], "v");
    const Mask m = mask_args(a + 3);
    std::pair<Tensor, Tensor> r;
    {
        pybind11::gil_scoped_release no_gil;
        r = forward(q, k, v, m);
    }
    PyObject* o = THPVariable_Wrap(std::move(r.first));
    PyObject* l = THPVariable_Wrap(std::move(r.second));
    PyObject* t = PyTuple_Pack(2, o, l);
    Py_DECREF(o);
    Py_DECREF(l);
    return t;
    END_HANDLE_TH_ERRORS
}

// (q, k, v, o, lse, d_o, scale, causal, window, sinks, grad_like, out or None, stages) -> (dq, dk, dv)
PyObject* py_bwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    expect(n, 13);
    const Tensor &q = tensor_arg(a[0], "q"), &k = tensor_arg(a[1], "k"), &v = tensor_arg(a[2], "v"), &o = tensor_arg(a[3], "o"),
                 &lse = tensor_arg(a[4], "lse"), &d_o = tensor_arg(a[5], "d_o");
    const Mask m = mask_args(a + 6);
    at::ScalarType grad = q.scalar_type();
    if (a[10] != Py_None) {
        if (!THPDtype_Check(a[10])) throw torch::TypeError("grad_dtype must be a torch dtype");
        grad = reinterpret_cast<THPDtype*>(a[10])->scalar_type;
    }
    const int stages = int_arg(a[12]);
    std::vector<Tensor> out;
    if (a[11] != Py_None) {
        PyObject* seq = PySequence_Fast(a[11], "out must be (dq, dk, dv, workspace)");
        if (!seq) throw python_error();
        const Py_ssize_t m4 = PySequence_Fast_GET_SIZE(seq);
        for (Py_ssize_t i = 0; i < m4 && m4 == 4; ++i) {
            PyObject* item = PySequence_Fast_GET_ITEM(seq, i);
            if (THPVariable_Check(item)) out.push_back(THPVariable_Unpack(item));
        }
        Py_DECREF(seq);
        if (out.size() != 4) TORCH_CHECK_VALUE(false, "out must be the four tensors (dq, dk, dv, workspace)");
    }
    Grads g;
    {
        pybind11::gil_scoped_release no_gil;
        g = backward(q, k, v, o, lse, d_o, m, grad, out.empty() ? nullptr : out.data(), stages);
    }
    PyObject *x = THPVariable_Wrap(std::move(g.dq)), *y = THPVariable_Wrap(std::move(g.dk)), *z = THPVariable_Wrap(std::move(g.dv));
    PyObject* t = PyTuple_Pack(3, x, y, z);
    Py_DECREF(x);
    Py_DECREF(y);
    Py_DECREF(z);
    return t;
    END_HANDLE_TH_ERRORS
}

// (q, k, v, scale, causal, window, sinks) -> o, on the tape
PyObject* py_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    expect(n, 7);
    const Tensor &q = tensor_arg(a[0], "q"), &k = tensor_arg(a[1], "k"), &v = tensor_arg(a[2], "v");
    const Mask m = mask_args(a + 3);
    Tensor o;
    {
        pybind11::gil_scoped_release no_gil;
        o = attention(q, k, v, m);
    }
    return THPVariable_Wrap(std::move(o));
    END_HANDLE_TH_ERRORS
}

// (q, k, v, scale, causal, window, sinks, seq_len, name) -> o for one head's [rows, dk] matrices, on the tape
PyObject* py_head(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    expect(n, 9);
    const Tensor &q = tensor_arg(a[0], "q"), &k = tensor_arg(a[1], "k"), &v = tensor_arg(a[2], "v");
    Mask m = mask_args(a + 3);
    const char* who = PyUnicode_AsUTF8(a[8]);
    if (!who) throw python_error();
    if (q.dim() != 2 || k.sizes() != q.sizes() || v.sizes() != q.sizes()) throw std::runtime_error(std::string(who) + ": shape mismatch");
    const int64_t rows = q.size(0), sl = int_arg(a[7]);
    m.seq_len = sl == 0 ? rows : sl;
    if (m.seq_len <= 0 || rows % m.seq_len != 0) throw std::runtime_error(std::string(who) + ": rows not a multiple of seq_len");
    Tensor o;
    {
        pybind11::gil_scoped_release no_gil;
        o = attention(q, k, v, m);
    }
    return THPVariable_Wrap(std::move(o));
    END_HANDLE_TH_ERRORS
}

PyMethodDef g_methods[] = {
    {"attn_fwd", reinterpret_cast<PyCFunction>(py_fwd), METH_FASTCALL, "forward: (o, lse)"},
    {"attn_bwd", reinterpret_cast<PyCFunction>(py_bwd), METH_FASTCALL, "recompute backward: (dq, dk, dv)"},
    {"attention", reinterpret_cast<PyCFunction>(py_attention), METH_FASTCALL, "all heads at once, differentiable"},
    {"attention_head", reinterpret_cast<PyCFunction>(py_head), METH_FASTCALL, "one head on [rows, dk] matrices, differentiable"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_torch_ops", "native side of paperkiln_amd.ops", -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_ops() {
    PyObject* lib = PyImport_ImportModule("paperkiln_amd._lib");
    if (!lib) return nullptr;
    g_error = PyObject_GetAttrString(lib, "PkError");
    Py_DECREF(lib);
    return g_error ? PyModule_Create(&g_module) : nullptr;
}
