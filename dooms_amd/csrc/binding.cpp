// The torch front end's common path as a CPython extension (dooms_amd._native): each function takes the arguments of
// its namesake in attention.py in order, checks the tensors, allocates what the caller left out, and calls the C ABI.
//
// What bounds it: a decode step of a short context is 5 to 7 us of kernel, and through ctypes a call took 12 to 15 us of
// host time (about 2 of it the launch itself), so a Python decoder was bound by the front end.
//
// Only the plain case is handled: exact torch.Tensor arguments of the right device, type, shape and strides, plain ints
// and floats, a caller-owned workspace. For anything else (and for every error but a code returned by the library) a
// function returns None, having done nothing, and attention.py takes its general path, which raises what it always
// raised. A code other than 0 is returned as an int. The library's functions are handed over as addresses (bind), so
// this extension links neither the library nor a GPU runtime beyond torch's.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <climits>
#include <cmath>
#include <vector>

#include "mx_attn.h"
#include "mx_linear.h"

namespace {

struct Api {
    decltype(&mx_attn_prefill_ws) prefill_ws = nullptr;
    decltype(&mx_attn_decode) decode = nullptr;
    decltype(&mx_attn_decode_f32) decode_f32 = nullptr;
    decltype(&mx_attn_decode_rope) decode_rope = nullptr;
    decltype(&mx_attn_prefill_rope_ws) prefill_rope_ws = nullptr;
    decltype(&mx_linear_call_workspace_bytes) linear_workspace_bytes = nullptr;
    decltype(&mx_linear) linear = nullptr;
    decltype(&mx_self_attention_workspace_bytes) self_attention_workspace_bytes = nullptr;
    decltype(&mx_self_attention) self_attention = nullptr;
};
Api api;

// Thrown where the general path has to take over.
struct General {};

void need(bool ok) {
    if (!ok) throw General{};
}

const at::Tensor & tensor(PyObject * o) {
    need(THPVariable_CheckExact(o));
    return THPVariable_Unpack(o);
}

int64_t integer(PyObject * o) {
    need(PyLong_CheckExact(o));
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        throw General{};
    }
    return v;
}

int32_t int32(PyObject * o) {
    const int64_t v = integer(o);
    need(v >= INT32_MIN && v <= INT32_MAX);
    return (int32_t)v;
}

double real(PyObject * o) {
    if (PyFloat_CheckExact(o)) return PyFloat_AS_DOUBLE(o);
    return (double)int32(o);
}

int truth(PyObject * o) {
    const int t = PyObject_IsTrue(o);
    if (t < 0) {
        PyErr_Clear();
        throw General{};
    }
    return t;
}

// A device tensor [rows][features] with unit feature stride.
const at::Tensor & rows(PyObject * o, at::ScalarType dtype) {
    const at::Tensor & t = tensor(o);
    need(t.is_cuda() && t.scalar_type() == dtype && t.dim() == 2 && t.stride(1) == 1);
    return t;
}

template <typename T>
T * data(const at::Tensor & t) {
    return static_cast<T *>(t.data_ptr());
}

// out (checked) or a new [n][width] tensor of its type on like's device
at::Tensor rows_or_new(PyObject * o, int64_t n, int64_t width, at::ScalarType dtype, const at::Tensor & like) {
    if (o != Py_None) return rows(o, dtype);
    return at::empty({n, width}, like.options().dtype(dtype));
}

// A prefill's workspace: the address and the bytes of the caller's tensor, or neither (the flash kernel).
struct Workspace {
    void * p = nullptr;
    size_t n = 0;
    explicit Workspace(PyObject * o) {
        if (o == Py_None) return;
        const at::Tensor & t = tensor(o);
        p = t.data_ptr();
        n = (size_t)t.numel();
    }
};

// The caller's lse as it is, or a new one, or none.
at::Tensor lse_or_new(PyObject * o, PyObject * want, int64_t n, int64_t heads, const at::Tensor & like) {
    if (o != Py_None) return tensor(o);
    if (!truth(want)) return {};
    return at::empty({n, heads}, like.options().dtype(at::kFloat));
}

PyObject * pair(const at::Tensor & out, PyObject * out_arg, const at::Tensor & lse, PyObject * lse_arg) {
    PyObject * a = out_arg != Py_None ? Py_NewRef(out_arg) : THPVariable_Wrap(out);
    PyObject * b = lse_arg != Py_None ? Py_NewRef(lse_arg) : lse.defined() ? THPVariable_Wrap(lse) : Py_NewRef(Py_None);
    if (!a || !b) {
        Py_XDECREF(a);
        Py_XDECREF(b);
        return nullptr;
    }
    PyObject * r = PyTuple_Pack(2, a, b);
    Py_DECREF(a);
    Py_DECREF(b);
    return r;
}

void * stream() { return c10::hip::getCurrentHIPStream().stream(); }

struct Unlocked {  // other Python threads run while the library does
    PyThreadState * s = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(s); }
};

// The entries of a list or tuple, held only for the duration of a call that keeps the container alive.
std::vector<PyObject *> items(PyObject * o) {
    need(PyList_CheckExact(o) || PyTuple_CheckExact(o));
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(o);
    PyObject ** p = PySequence_Fast_ITEMS(o);
    return std::vector<PyObject *>(p, p + n);
}

mx_attn_desc desc(PyObject * const * heads, int32_t n_q, int64_t q_stride, int64_t kv_stride, int64_t out_stride,
                  PyObject * scale) {
    mx_attn_desc d{};
    d.n_head = int32(heads[0]);
    d.n_head_kv = int32(heads[1]);
    d.head_dim = int32(heads[2]);
    need(d.head_dim > 0);
    d.n_q = n_q;
    d.q_stride = q_stride;
    d.kv_stride = kv_stride;
    d.out_stride = out_stride;
    d.scale = scale == Py_None ? (float)(1.0 / std::sqrt((double)d.head_dim)) : (float)real(scale);
    return d;
}

struct Caches {
    std::vector<uint16_t *> k, v;
    std::vector<int32_t> len;
    int64_t stride;
    Caches(PyObject * ks, PyObject * vs, PyObject * lens) {
        const auto ki = items(ks), vi = items(vs), li = items(lens);
        need(!ki.empty() && ki.size() == li.size() && vi.size() == li.size());
        stride = rows(ki[0], at::kHalf).stride(0);
        for (size_t i = 0; i < li.size(); i++) {
            const at::Tensor & a = rows(ki[i], at::kHalf), & b = rows(vi[i], at::kHalf);
            need(a.stride(0) == stride && b.stride(0) == stride);
            k.push_back(data<uint16_t>(a));
            v.push_back(data<uint16_t>(b));
            len.push_back(int32(li[i]));
        }
    }
};

PyObject * code(int32_t rc) { return PyLong_FromLong(rc); }

// q, k_caches, v_caches, kv_len, n_head, n_head_kv, head_dim, n_q, causal, scale, out, lse, want_lse, workspace
PyObject * decode(PyObject * const * a) {
    const at::Tensor & q0 = tensor(a[0]);
    const at::ScalarType t = q0.scalar_type() == at::kFloat ? at::kFloat : at::kHalf;
    const at::Tensor & q = rows(a[0], t);
    const Caches c(a[1], a[2], a[3]);
    const int32_t n_head = int32(a[4]), head_dim = int32(a[6]);
    const at::Tensor & ws = tensor(a[13]);
    const at::Tensor out = rows_or_new(a[10], q.size(0), (int64_t)n_head * head_dim, t, q);
    const at::Tensor lse = lse_or_new(a[11], a[12], q.size(0), n_head, q);
    mx_attn_desc d = desc(a + 4, int32(a[7]), q.stride(0), c.stride, out.stride(0), a[9]);
    d.causal = truth(a[8]);
    float * l = lse.defined() ? data<float>(lse) : nullptr;
    const int32_t n = (int32_t)c.len.size();
    int32_t rc;
    {
        Unlocked u;
        rc = t == at::kFloat ? api.decode_f32(&d, n, c.len.data(), data<float>(q), c.k.data(), c.v.data(), data<float>(out), l,
                                              ws.data_ptr(), (size_t)ws.numel(), stream())
                             : api.decode(&d, n, c.len.data(), data<uint16_t>(q), c.k.data(), c.v.data(),
                                          data<uint16_t>(out), l, ws.data_ptr(), (size_t)ws.numel(), stream());
    }
    return rc ? code(rc) : pair(out, a[10], lse, a[11]);
}

// qkv, k_caches, v_caches, kv_len, n_head, n_head_kv, head_dim, rope_mode, rope_base, scale, out, lse, want_lse, workspace
PyObject * decode_rope(PyObject * const * a) {
    const at::Tensor & q = rows(a[0], at::kFloat);
    const Caches c(a[1], a[2], a[3]);
    const int32_t n_head = int32(a[4]), head_dim = int32(a[6]), n = (int32_t)c.len.size();
    const mx_attn_rope rope{int32(a[7]), (float)real(a[8])};
    const at::Tensor & ws = tensor(a[13]);
    const at::Tensor out = rows_or_new(a[10], n, (int64_t)n_head * head_dim, at::kFloat, q);
    const at::Tensor lse = lse_or_new(a[11], a[12], n, n_head, q);
    const mx_attn_desc d = desc(a + 4, 1, q.stride(0), c.stride, out.stride(0), a[9]);
    int32_t rc;
    {
        Unlocked u;
        rc = api.decode_rope(&d, &rope, n, c.len.data(), data<float>(q), c.k.data(), c.v.data(), data<float>(out),
                             lse.defined() ? data<float>(lse) : nullptr, ws.data_ptr(), (size_t)ws.numel(), stream());
    }
    return rc ? code(rc) : pair(out, a[10], lse, a[11]);
}

// The chunk's descriptor: n_head, n_head_kv, head_dim at heads; p0, causal, n_kv, scale.
mx_attn_desc chunk(PyObject * const * heads, const at::Tensor & q, const at::Tensor & k, const at::Tensor & out, PyObject * p0,
                   PyObject * causal, PyObject * n_kv, PyObject * scale) {
    need(q.size(0) <= INT32_MAX);
    mx_attn_desc d = desc(heads, (int32_t)q.size(0), q.stride(0), k.stride(0), out.stride(0), scale);
    d.p0 = int32(p0);
    d.causal = truth(causal);
    d.n_kv = n_kv == Py_None ? 0 : int32(n_kv);
    return d;
}

// q, k_cache, v_cache, n_head, n_head_kv, head_dim, p0, causal, n_kv, scale, out, lse, want_lse, workspace
PyObject * prefill(PyObject * const * a) {
    const at::Tensor & q = rows(a[0], at::kHalf), & k = rows(a[1], at::kHalf), & v = rows(a[2], at::kHalf);
    need(k.stride(0) == v.stride(0));
    const int32_t n_head = int32(a[3]), head_dim = int32(a[5]);
    const Workspace ws(a[13]);
    const at::Tensor out = rows_or_new(a[10], q.size(0), (int64_t)n_head * head_dim, at::kHalf, q);
    const at::Tensor lse = lse_or_new(a[11], a[12], q.size(0), n_head, q);
    const mx_attn_desc d = chunk(a + 3, q, k, out, a[6], a[7], a[8], a[9]);
    int32_t rc;
    {
        Unlocked u;
        rc = api.prefill_ws(&d, data<uint16_t>(q), data<uint16_t>(k), data<uint16_t>(v), data<uint16_t>(out),
                            lse.defined() ? data<float>(lse) : nullptr, ws.p, ws.n, stream());
    }
    return rc ? code(rc) : pair(out, a[10], lse, a[11]);
}

// qkv, k_cache, v_cache, n_head, n_head_kv, head_dim, rope_mode, rope_base, p0, causal, n_kv, scale, out, lse, want_lse,
// workspace
PyObject * prefill_rope(PyObject * const * a) {
    const at::Tensor & q = rows(a[0], at::kFloat), & k = rows(a[1], at::kHalf), & v = rows(a[2], at::kHalf);
    need(k.stride(0) == v.stride(0));
    const int32_t n_head = int32(a[3]), head_dim = int32(a[5]);
    const mx_attn_rope rope{int32(a[6]), (float)real(a[7])};
    const Workspace ws(a[15]);
    const at::Tensor out = rows_or_new(a[12], q.size(0), (int64_t)n_head * head_dim, at::kFloat, q);
    const at::Tensor lse = lse_or_new(a[13], a[14], q.size(0), n_head, q);
    const mx_attn_desc d = chunk(a + 3, q, k, out, a[8], a[9], a[10], a[11]);
    int32_t rc;
    {
        Unlocked u;
        rc = api.prefill_rope_ws(&d, &rope, data<float>(q), data<uint16_t>(k), data<uint16_t>(v), data<float>(out),
                                 lse.defined() ? data<float>(lse) : nullptr, ws.p, ws.n, stream());
    }
    return rc ? code(rc) : pair(out, a[12], lse, a[13]);
}

// x, weights (one tensor, or a list), out (None, a tensor or a list, as weights), gamma, bias, eps, accumulate, out_f16
PyObject * linear(PyObject * const * a) {
    const at::Tensor & x = rows(a[0], at::kFloat);
    const bool single = THPVariable_CheckExact(a[1]), f16 = truth(a[7]);
    const std::vector<PyObject *> ws = single ? std::vector<PyObject *>{a[1]} : items(a[1]);
    const size_t n = ws.size();
    need(n > 0);
    const at::ScalarType odt = f16 ? at::kHalf : at::kFloat;
    std::vector<const uint16_t *> w;
    int64_t N = 0, K = 0;
    for (PyObject * o : ws) {
        const at::Tensor & t = rows(o, at::kHalf);
        if (w.empty()) N = t.size(0), K = t.size(1);
        need(t.size(0) == N && t.size(1) == K && t.stride(0) == K);
        w.push_back(data<uint16_t>(t));
    }
    need(N <= INT32_MAX && K <= INT32_MAX && x.size(0) <= INT32_MAX && n <= INT32_MAX);
    std::vector<at::Tensor> outs;
    if (a[2] == Py_None) {
        for (size_t i = 0; i < n; i++) outs.push_back(at::empty({x.size(0), N}, x.options().dtype(odt)));
    } else if (single) {
        outs.push_back(rows(a[2], odt));
    } else {
        for (PyObject * o : items(a[2])) outs.push_back(rows(o, odt));
        need(outs.size() == n);
    }
    std::vector<void *> y;
    for (const at::Tensor & t : outs) {
        need(t.stride(0) == outs[0].stride(0));
        y.push_back(t.data_ptr());
    }
    const float * gamma = a[3] == Py_None ? nullptr : data<const float>(tensor(a[3]));
    std::vector<const float *> bias;
    if (a[4] != Py_None) {
        if (THPVariable_CheckExact(a[4])) {
            bias.push_back(data<const float>(tensor(a[4])));
        } else {
            for (PyObject * o : items(a[4])) bias.push_back(o == Py_None ? nullptr : data<const float>(tensor(o)));
        }
        need(bias.size() == n);
    }
    mx_linear_desc d{};
    d.M = (int32_t)x.size(0);
    d.N = (int32_t)N;
    d.K = (int32_t)K;
    d.flags = (a[3] != Py_None ? MX_LINEAR_RMS_NORM : 0) | (truth(a[6]) ? MX_LINEAR_ACCUMULATE : 0) |
              (a[4] != Py_None ? MX_LINEAR_BIAS : 0) | (f16 ? MX_LINEAR_OUT_F16 : 0);
    d.x_stride = x.stride(0);
    d.y_stride = outs[0].stride(0);
    d.eps = (float)real(a[5]);
    const size_t bytes = api.linear_workspace_bytes(&d, (int32_t)n);
    const int64_t room = (int64_t)std::max<size_t>(bytes, 256);
    const at::Tensor work = bytes ? at::empty({room}, x.options().dtype(at::kByte)) : at::Tensor();
    int32_t rc;
    {
        Unlocked u;
        rc = api.linear(&d, (int32_t)n, w.data(), data<float>(x), y.data(), gamma, bias.empty() ? nullptr : bias.data(),
                        bytes ? work.data_ptr() : nullptr, bytes ? (size_t)work.numel() : 0, stream());
    }
    if (rc) return code(rc);
    if (a[2] != Py_None) return single ? Py_NewRef(a[2]) : PySequence_List(a[2]);
    if (single) return THPVariable_Wrap(outs[0]);
    PyObject * r = PyList_New((Py_ssize_t)n);
    for (size_t i = 0; r && i < n; i++) {
        PyObject * o = THPVariable_Wrap(outs[i]);
        if (!o) Py_CLEAR(r);
        else PyList_SET_ITEM(r, (Py_ssize_t)i, o);
    }
    return r;
}

// qkv, heads, scale, out
PyObject * self_attention(PyObject * const * a) {
    const at::Tensor & x = tensor(a[0]);
    const at::ScalarType t = x.scalar_type();
    need(x.is_cuda() && x.dim() == 3 && x.is_contiguous() && (t == at::kFloat || t == at::kHalf || t == at::kBFloat16));
    const int64_t B = x.size(0), N = x.size(1), E = x.size(2) / 3;
    const int32_t heads = int32(a[1]);
    need(x.size(2) % 3 == 0 && heads >= 1 && E % heads == 0 && E / heads >= 1);
    need(B <= INT32_MAX && N <= INT32_MAX && E <= INT32_MAX);
    mx_self_attn_desc d{};
    d.batch = (int32_t)B;
    d.n_tok = (int32_t)N;
    d.heads = heads;
    d.embed = (int32_t)E;
    d.dtype = t == at::kFloat ? MX_ATTN_F32 : t == at::kHalf ? MX_ATTN_F16 : MX_ATTN_BF16;
    d.scale = (float)(a[2] == Py_None ? std::pow((double)(E / heads), -0.5) : real(a[2]));
    const at::Tensor out = a[3] != Py_None ? tensor(a[3]) : at::empty({B, N, E}, x.options());
    const size_t bytes = api.self_attention_workspace_bytes(&d);
    const at::Tensor work = bytes ? at::empty({(int64_t)bytes}, x.options().dtype(at::kByte)) : at::Tensor();
    int32_t rc;
    {
        Unlocked u;
        rc = api.self_attention(&d, x.data_ptr(), out.data_ptr(), bytes ? work.data_ptr() : nullptr, bytes, stream());
    }
    if (rc) return code(rc);
    return a[3] != Py_None ? Py_NewRef(a[3]) : THPVariable_Wrap(out);
}

template <PyObject * (*F)(PyObject * const *), Py_ssize_t N>
PyObject * entry(PyObject *, PyObject * const * args, Py_ssize_t n) {
    if (n != N) {
        PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", N, n);
        return nullptr;
    }
    try {
        return F(args);
    } catch (...) {  // the general path meets the same condition and says what it is
        PyErr_Clear();
        Py_RETURN_NONE;
    }
}

// bind(abi version, (sizes of mx_attn_desc, mx_attn_rope, mx_linear_desc, mx_self_attn_desc), addresses): the library's
// functions in the order of Api. A library of another version, or descriptors of another layout than this extension was
// compiled with, are refused.
PyObject * bind(PyObject *, PyObject * args) {
    int version;
    Py_ssize_t size[4];
    unsigned long long p[9];
    if (!PyArg_ParseTuple(args, "i(nnnn)KKKKKKKKK", &version, size, size + 1, size + 2, size + 3, p, p + 1, p + 2, p + 3, p + 4,
                          p + 5, p + 6, p + 7, p + 8))
        return nullptr;
    const size_t own[4] = {sizeof(mx_attn_desc), sizeof(mx_attn_rope), sizeof(mx_linear_desc), sizeof(mx_self_attn_desc)};
    bool same = version == MX_ATTN_ABI_VERSION;
    for (int i = 0; i < 4; i++) same = same && (size_t)size[i] == own[i];
    if (!same) {
        PyErr_Format(PyExc_ImportError,
                     "dooms_amd._native was built for version %d of the library, which is %d, or for other descriptors: build "
                     "both with `python -m dooms_amd.build`",
                     (int)MX_ATTN_ABI_VERSION, version);
        return nullptr;
    }
    auto set = [](auto & f, unsigned long long v) {
        f = reinterpret_cast<std::remove_reference_t<decltype(f)>>((uintptr_t)v);
    };
    set(api.prefill_ws, p[0]);
    set(api.decode, p[1]);
    set(api.decode_f32, p[2]);
    set(api.decode_rope, p[3]);
    set(api.prefill_rope_ws, p[4]);
    set(api.linear_workspace_bytes, p[5]);
    set(api.linear, p[6]);
    set(api.self_attention_workspace_bytes, p[7]);
    set(api.self_attention, p[8]);
    Py_RETURN_NONE;
}

#define MX_ENTRY(name, n) \
    {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(entry<name, n>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    MX_ENTRY(decode, 14), MX_ENTRY(decode_rope, 14), MX_ENTRY(prefill, 14), MX_ENTRY(prefill_rope, 16), MX_ENTRY(linear, 8),
    MX_ENTRY(self_attention, 4), {"bind", bind, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module); }
