// The per-call part of the Python binding in C++: takes the tensors apart, allocates outputs and workspaces from
// torch's caching allocator, and calls the C ABI of libtfq.so on torch's current stream.  Host code only (g++).
//
// Why: a decode-sized product runs 3 to 15 us on the GPU, and the same steps through ctypes and the tensors' Python
// attributes took longer, so the host, not the kernel, set the rate of a loop of such calls.  Host time per call, ctypes
// and here: gemv 10.7 and 4.2 us (1024 x 4096, one bf16 row), with a workspace 12.3 and 5.1, one fused product 9.0 and
// 3.2, router and routed mixture (two calls, five launches) 40 and 25; the launch itself is about 2 us of each.
//
// The C calls run without the GIL, as they do under ctypes.  Nothing is kept between calls.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <vector>

#include "../../include/tfq.h"

namespace {

PyObject* g_error = nullptr;  // TfqError
PyObject* g_handle_name = nullptr;

struct PyFail {};  // a Python exception is set

[[noreturn]] void raise(PyObject* type, const char* msg) {
    PyErr_SetString(type, msg);
    throw PyFail{};
}
void check(int rc) {
    if (rc == TFQ_OK) return;
    PyErr_Format(g_error, "tfq error %d: %s", rc, tfq_last_error());
    throw PyFail{};
}
template <class F>
void call(F&& f) {
    int rc;
    {
        PyThreadState* ts = PyEval_SaveThread();
        rc = f();
        PyEval_RestoreThread(ts);
    }
    check(rc);
}
const at::Tensor& tensor(PyObject* o) {
    if (!THPVariable_Check(o)) raise(PyExc_TypeError, "expected a torch.Tensor");
    return THPVariable_Unpack(o);
}
void require(bool ok, const char* msg) {
    if (!ok) raise(PyExc_AssertionError, msg);
}
int dtype_code(const at::Tensor& t) {
    if (t.scalar_type() == at::kFloat) return TFQ_F32;
    if (t.scalar_type() == at::kBFloat16) return TFQ_BF16;
    PyErr_Format(g_error, "unsupported dtype %s", c10::toString(t.scalar_type()));
    throw PyFail{};
}
at::ScalarType dtype_or(PyObject* o, at::ScalarType fallback) {
    if (o == Py_None) return fallback;
    if (!THPDtype_Check(o)) raise(PyExc_TypeError, "expected a torch.dtype");
    return reinterpret_cast<THPDtype*>(o)->scalar_type;
}
int64_t integer(PyObject* o) {
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw PyFail{};
    return v;
}
void* address(PyObject* o) {
    void* p = PyLong_AsVoidPtr(o);
    if (!p && PyErr_Occurred()) throw PyFail{};
    return p;
}
double number(PyObject* o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw PyFail{};
    return v;
}
bool truth(PyObject* o) {
    const int v = PyObject_IsTrue(o);
    if (v < 0) throw PyFail{};
    return v != 0;
}
const tfq_weight_t* weight_of(PyObject* w) {
    PyObject* h = PyObject_GetAttr(w, g_handle_name);
    if (!h) throw PyFail{};
    void* p = PyLong_AsVoidPtr(h);
    Py_DECREF(h);
    if (!p && PyErr_Occurred()) throw PyFail{};
    return static_cast<const tfq_weight_t*>(p);
}
std::vector<const tfq_weight_t*> weights_of(PyObject* seq) {
    PyObject* f = PySequence_Fast(seq, "expected a sequence of Weight");
    if (!f) throw PyFail{};
    std::vector<const tfq_weight_t*> v((size_t)PySequence_Fast_GET_SIZE(f));
    try {
        for (size_t i = 0; i < v.size(); ++i) v[i] = weight_of(PySequence_Fast_GET_ITEM(f, (Py_ssize_t)i));
    } catch (...) {
        Py_DECREF(f);
        throw;
    }
    Py_DECREF(f);
    return v;
}
tfq_stream_t stream() { return reinterpret_cast<tfq_stream_t>(c10::hip::getCurrentHIPStream().stream()); }
at::Tensor empty(c10::IntArrayRef size, at::ScalarType t, const at::Tensor& like) {
    return at::empty(size, at::TensorOptions().dtype(t).device(like.device()));
}
at::Tensor bytes(size_t n, const at::Tensor& like) { return empty({(int64_t)n}, at::kByte, like); }
// Parameter counts are fixed: the Python wrappers pass every argument by position.
void count(Py_ssize_t n, Py_ssize_t want) {
    if (n != want) raise(PyExc_TypeError, "wrong number of arguments");
}

// handle, N, K, x, out_dtype, out, workspace
PyObject* gemv(PyObject* const* a, Py_ssize_t n) {
    count(n, 7);
    const auto* w = static_cast<const tfq_weight_t*>(address(a[0]));
    const int64_t N = integer(a[1]), K = integer(a[2]);
    const at::Tensor x = tensor(a[3]).contiguous();
    require(x.is_cuda() && x.dim() > 0 && x.size(-1) == K, "x must be a device tensor [.., K]");
    const int B = (int)(x.numel() / K), xd = dtype_code(x);
    at::Tensor out = a[5] == Py_None ? empty({B, N}, dtype_or(a[4], at::kFloat), x) : tensor(a[5]);
    const int od = dtype_code(out);
    const size_t need = tfq_gemv_workspace_bytes(w, xd, B);
    if (need == 0) {
        const tfq_stream_t s = stream();
        call([&] { return tfq_gemv(w, x.data_ptr(), xd, B, out.data_ptr(), od, s); });
    } else {
        const at::Tensor ws = a[6] == Py_None ? bytes(need, x) : tensor(a[6]);
        require((size_t)ws.numel() >= need && reinterpret_cast<uintptr_t>(ws.data_ptr()) % 256 == 0, "workspace too small or not 256-byte aligned");
        const tfq_stream_t s = stream();
        call([&] { return tfq_gemv_ws(w, x.data_ptr(), xd, B, out.data_ptr(), od, ws.data_ptr(), (size_t)ws.numel(), s); });
    }
    if (a[5] != Py_None) {
        Py_INCREF(a[5]);
        return a[5];
    }
    return THPVariable_Wrap(std::move(out));
}

// handle, N, K, x, out_dtype, use_workspace
PyObject* gemm(PyObject* const* a, Py_ssize_t n) {
    count(n, 6);
    const auto* w = static_cast<const tfq_weight_t*>(address(a[0]));
    const int64_t N = integer(a[1]), K = integer(a[2]);
    const at::Tensor x = tensor(a[3]).contiguous();
    require(x.is_cuda() && x.dim() > 0 && x.size(-1) == K, "x must be a device tensor [.., K]");
    const int M = (int)(x.numel() / K), xd = dtype_code(x);
    at::Tensor y = empty({M, N}, dtype_or(a[4], at::kFloat), x);
    const int yd = dtype_code(y);
    const size_t need = truth(a[5]) ? tfq_gemm_workspace_bytes(w, xd, M) : 0;
    if (need == 0) {
        const tfq_stream_t s = stream();
        call([&] { return tfq_gemm(w, x.data_ptr(), xd, M, y.data_ptr(), yd, s); });
    } else {
        const at::Tensor ws = bytes(need, x);
        const tfq_stream_t s = stream();
        call([&] { return tfq_gemm_ws(w, x.data_ptr(), xd, M, y.data_ptr(), yd, ws.data_ptr(), need, s); });
    }
    return THPVariable_Wrap(std::move(y));
}

struct Outs {
    std::vector<void*> p;  // one per matrix; null where there are fewer outputs
    int dtype = 0;
};
// What the matrices' count allows is the C call's to say (TfqError), as is a missing output; outputs without a matrix
// are an IndexError, as for a fixed-size array.
Outs outs_of(PyObject* seq, size_t matrices, bool repeat_single = false) {
    PyObject* f = PySequence_Fast(seq, "expected a sequence of tensors");
    if (!f) throw PyFail{};
    Outs o;
    try {
        const Py_ssize_t n = PySequence_Fast_GET_SIZE(f);
        o.p.reserve(4);
        for (Py_ssize_t i = 0; i < n; ++i) o.p.push_back(tensor(PySequence_Fast_GET_ITEM(f, i)).data_ptr());
        if (repeat_single && n == 1) o.p.push_back(o.p[0]);
        if (o.p.empty() || o.p.size() > matrices) raise(PyExc_IndexError, "no matrices or outputs, or more outputs than matrices");
        o.p.resize(matrices, nullptr);
        o.dtype = dtype_code(THPVariable_Unpack(PySequence_Fast_GET_ITEM(f, 0)));
    } catch (...) {
        Py_DECREF(f);
        throw;
    }
    Py_DECREF(f);
    return o;
}

// weights, x, outs
PyObject* gemv_multi(PyObject* const* a, Py_ssize_t n) {
    count(n, 3);
    const auto ws = weights_of(a[0]);
    const at::Tensor& x = tensor(a[1]);
    const Outs o = outs_of(a[2], ws.size());
    int64_t K = 0;
    tfq_weight_info(ws[0], nullptr, nullptr, &K, nullptr);
    const int B = K ? (int)(x.numel() / K) : 0, xd = dtype_code(x);
    const tfq_stream_t s = stream();
    call([&] { return tfq_gemv_multi(ws.data(), (int)ws.size(), x.data_ptr(), xd, B, o.p.data(), o.dtype, s); });
    Py_INCREF(a[2]);
    return a[2];
}

// weights, x, outs, rmsnorm, swiglu_up, eps, gamma_plus_one, mid_dtype, accumulate, pair_swiglu
PyObject* gemv_multi_fused(PyObject* const* a, Py_ssize_t n) {
    count(n, 10);
    const auto ws = weights_of(a[0]);
    const at::Tensor& x = tensor(a[1]);
    require(x.is_contiguous() && x.dim() > 0, "x must be contiguous");
    tfq_prologue_t pro{};
    pro.accumulate = truth(a[8]);
    pro.pair_swiglu = truth(a[9]);
    // (the second output of a pair is not written; the C call still wants two pointers)
    const Outs o = outs_of(a[2], ws.size(), pro.pair_swiglu);
    if (a[3] != Py_None) {
        const at::Tensor& g = tensor(a[3]);
        require(g.scalar_type() == at::kFloat, "rmsnorm must be float32");
        pro.op = TFQ_PRO_RMSNORM;
        pro.gamma = static_cast<const float*>(g.data_ptr());
        pro.eps = (float)number(a[5]);
        pro.gamma_plus_one = truth(a[6]);
    } else if (a[4] != Py_None) {
        const at::Tensor& up = tensor(a[4]);
        require(up.scalar_type() == at::kFloat && up.sizes() == x.sizes() && up.is_contiguous(), "swiglu_up must be a contiguous float32 tensor of x's shape");
        pro.op = TFQ_PRO_SWIGLU;
        pro.up = static_cast<const float*>(up.data_ptr());
        pro.mid_dtype = dtype_or(a[7], at::kFloat) == at::kBFloat16 ? TFQ_BF16 : TFQ_F32;
    }
    const int B = (int)x.size(0), xd = dtype_code(x);
    const tfq_stream_t s = stream();
    call([&] { return tfq_gemv_multi_fused(ws.data(), (int)ws.size(), x.data_ptr(), xd, B, o.p.data(), o.dtype, &pro, s); });
    Py_INCREF(a[2]);
    return a[2];
}

// gate, up, down, x, out_dtype, mid_dtype
PyObject* mlp_step(PyObject* const* a, Py_ssize_t n) {
    count(n, 6);
    const tfq_weight_t *g = weight_of(a[0]), *u = weight_of(a[1]), *d = weight_of(a[2]);
    int64_t F = 0, D = 1, O = 0;
    tfq_weight_info(g, nullptr, &F, &D, nullptr);
    tfq_weight_info(d, nullptr, &O, nullptr, nullptr);
    const at::Tensor x = tensor(a[3]).contiguous();
    const int B = (int)(x.numel() / D), xd = dtype_code(x);
    at::Tensor y = empty({B, O}, dtype_or(a[4], at::kFloat), x);
    const int yd = dtype_code(y), mid = dtype_or(a[5], x.scalar_type()) == at::kBFloat16 ? TFQ_BF16 : TFQ_F32;
    const size_t need = tfq_mlp_workspace_bytes(B, F);
    const at::Tensor ws = bytes(need, x);
    const tfq_stream_t s = stream();
    call([&] { return tfq_mlp_step(g, u, d, x.data_ptr(), xd, B, y.data_ptr(), yd, mid, ws.data_ptr(), need, s); });
    return THPVariable_Wrap(std::move(y));
}

// x, router_w, k, bias
PyObject* moe_router(PyObject* const* a, Py_ssize_t n) {
    count(n, 4);
    const at::Tensor &x = tensor(a[0]), &r = tensor(a[1]);
    require(x.dim() == 2 && r.dim() == 2 && r.scalar_type() == at::kFloat && r.is_contiguous() && x.is_contiguous(),
            "x [T][D] and a float32 router [E][D], both contiguous");
    const int64_t T = x.size(0), D = x.size(1), E = r.size(0), k = integer(a[2]);
    const int64_t kk = std::max<int64_t>(1, std::min(k, E));
    at::Tensor logits = empty({T, E}, at::kFloat, x), probs = empty({T, E}, at::kFloat, x);
    at::Tensor idx = empty({T, kk}, at::kInt, x), w = empty({T, kk}, at::kFloat, x);
    const float* bias = a[3] == Py_None ? nullptr : static_cast<const float*>(tensor(a[3]).data_ptr());
    const int xd = dtype_code(x);
    const tfq_stream_t s = stream();
    call([&] {
        return tfq_moe_router(x.data_ptr(), xd, static_cast<const float*>(r.data_ptr()), bias, (int)T, (int)D, (int)E, (int)k,
                              static_cast<float*>(logits.data_ptr()), static_cast<float*>(probs.data_ptr()),
                              static_cast<int32_t*>(idx.data_ptr()), static_cast<float*>(w.data_ptr()), s);
    });
    PyObject* t = PyTuple_New(4);
    if (!t) throw PyFail{};
    PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(std::move(logits)));
    PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(std::move(probs)));
    PyTuple_SET_ITEM(t, 2, THPVariable_Wrap(std::move(idx)));
    PyTuple_SET_ITEM(t, 3, THPVariable_Wrap(std::move(w)));
    return t;
}

struct Buffer {  // a C-contiguous host array
    Py_buffer b{};
    explicit Buffer(PyObject* o) {
        if (PyObject_GetBuffer(o, &b, PyBUF_C_CONTIGUOUS) != 0) throw PyFail{};
    }
    ~Buffer() { PyBuffer_Release(&b); }
};

// gate, up, down, idx (int64 array [T][k]), weights (float32 array [T][k]), T, k, x, out_dtype, mid_dtype
PyObject* moe_ffn(PyObject* const* a, Py_ssize_t n) {
    count(n, 10);
    const auto g = weights_of(a[0]);
    auto u = weights_of(a[1]), d = weights_of(a[2]);
    if (g.empty() || u.size() > g.size() || d.size() > g.size()) raise(PyExc_IndexError, "no experts, or more up or down matrices than gate matrices");
    u.resize(g.size(), nullptr);  // a missing one is the C call's to refuse
    d.resize(g.size(), nullptr);
    const int T = (int)integer(a[5]), k = (int)integer(a[6]);
    const Buffer idx(a[3]), wts(a[4]);
    require(idx.b.len >= (Py_ssize_t)T * k * 8 && wts.b.len >= (Py_ssize_t)T * k * 4, "routing arrays of int64 and float32 [T][k]");
    int64_t F = 0, D = 0;
    tfq_weight_info(g[0], nullptr, &F, &D, nullptr);
    const at::Tensor x = tensor(a[7]).contiguous();
    at::Tensor y = empty({T, D}, dtype_or(a[8], at::kFloat), x);
    const int xd = dtype_code(x), yd = dtype_code(y), mid = dtype_or(a[9], x.scalar_type()) == at::kBFloat16 ? TFQ_BF16 : TFQ_F32;
    const size_t need = tfq_moe_workspace_bytes(T, k, D, F);
    const at::Tensor ws = bytes(need, x);
    const tfq_stream_t s = stream();
    call([&] {
        return tfq_moe_ffn(g.data(), u.data(), d.data(), (int)g.size(), static_cast<const int64_t*>(idx.b.buf), static_cast<const float*>(wts.b.buf),
                           T, k, x.data_ptr(), xd, y.data_ptr(), yd, mid, ws.data_ptr(), need, s);
    });
    return THPVariable_Wrap(std::move(y));
}

// addresses of the handle arrays gate, up, down; E, table, idx, wts, T, k, x, y, workspace
PyObject* moe_ffn_routed(PyObject* const* a, Py_ssize_t n) {
    count(n, 12);
    auto* g = static_cast<const tfq_weight_t* const*>(address(a[0]));
    auto* u = static_cast<const tfq_weight_t* const*>(address(a[1]));
    auto* d = static_cast<const tfq_weight_t* const*>(address(a[2]));
    const int E = (int)integer(a[3]), T = (int)integer(a[7]), k = (int)integer(a[8]);
    const at::Tensor &table = tensor(a[4]), &idx = tensor(a[5]), &wts = tensor(a[6]), &x = tensor(a[9]), &y = tensor(a[10]), &ws = tensor(a[11]);
    require(idx.is_cuda() && wts.is_cuda() && idx.element_size() == 4 && x.is_contiguous() && y.is_contiguous(),
            "idx (int32) and weights on the device, x and y contiguous");
    const int xd = dtype_code(x), yd = dtype_code(y);
    const tfq_stream_t s = stream();
    call([&] {
        return tfq_moe_ffn_routed(g, u, d, E, table.data_ptr(), static_cast<const int32_t*>(idx.data_ptr()), static_cast<const float*>(wts.data_ptr()),
                                  T, k, x.data_ptr(), xd, y.data_ptr(), yd, TFQ_BF16, ws.data_ptr(), (size_t)ws.numel(), s);
    });
    Py_INCREF(a[10]);
    return a[10];
}

// wire id, w
PyObject* encode(PyObject* const* a, Py_ssize_t n) {
    count(n, 2);
    const int64_t fmt = integer(a[0]);
    const at::Tensor w = tensor(a[1]).contiguous();
    require(w.is_cuda() && w.scalar_type() == at::kFloat, "a float32 device tensor");
    const int64_t count_w = w.numel();
    size_t full = 0, tail = 0;
    check(tfq_block_bytes((uint8_t)fmt, 256, &full));
    if (count_w % 256) check(tfq_block_bytes((uint8_t)fmt, (uint32_t)(count_w % 256), &tail));
    const size_t need = (size_t)(count_w / 256) * full + tail;
    at::Tensor out = bytes(need, w);
    const tfq_stream_t s = stream();
    call([&] { return tfq_encode_blocks((uint8_t)fmt, static_cast<const float*>(w.data_ptr()), count_w, static_cast<uint8_t*>(out.data_ptr()), need, s); });
    return THPVariable_Wrap(std::move(out));
}

// wire id, payload, n
PyObject* decode(PyObject* const* a, Py_ssize_t n) {
    count(n, 3);
    const int64_t fmt = integer(a[0]), count_w = integer(a[2]);
    const at::Tensor& p = tensor(a[1]);
    require(p.is_cuda() && p.scalar_type() == at::kByte, "a uint8 device tensor");
    at::Tensor out = empty({count_w}, at::kFloat, p);
    const tfq_stream_t s = stream();
    call([&] {
        return tfq_decode_blocks((uint8_t)fmt, static_cast<const uint8_t*>(p.data_ptr()), (size_t)p.numel(), count_w, static_cast<float*>(out.data_ptr()), s);
    });
    return THPVariable_Wrap(std::move(out));
}

template <PyObject* (*F)(PyObject* const*, Py_ssize_t)>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    try {
        return F(args, n);
    } catch (const PyFail&) {
        return nullptr;
    }
    END_HANDLE_TH_ERRORS
}

PyObject* set_error(PyObject*, PyObject* type) {
    Py_INCREF(type);
    Py_XDECREF(g_error);
    g_error = type;
    Py_RETURN_NONE;
}

#define TFQ_ENTRY(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(entry<name>)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {TFQ_ENTRY(gemv), TFQ_ENTRY(gemm), TFQ_ENTRY(gemv_multi), TFQ_ENTRY(gemv_multi_fused), TFQ_ENTRY(mlp_step),
                          TFQ_ENTRY(moe_router), TFQ_ENTRY(moe_ffn), TFQ_ENTRY(moe_ffn_routed), TFQ_ENTRY(encode), TFQ_ENTRY(decode),
                          {"set_error", set_error, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_tfq_torch", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__tfq_torch(void) {
    g_handle_name = PyUnicode_InternFromString("_h");
    g_error = PyExc_RuntimeError;
    Py_INCREF(g_error);
    return PyModule_Create(&kModule);
}
