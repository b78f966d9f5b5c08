// Host side of the most frequent calls, without an interpreter between the tensors and the C ABI.
//
// A call of a few microseconds on the device is bound by the host: the ctypes wrapper of
// attention_kernels.py spends about 16 us on describing eight tensors, allocating the results and converting
// nineteen arguments.  These functions do the same from C++ in about 3.  Each returns None where anything
// about its arguments is not the plain case (another device or type, shapes that do not match, a status other
// than OK); the Python wrapper then takes its own path, which raises what has to be raised.  C++ exceptions (no
// memory for a result, a tensor without storage) become Python's in every entry.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <cstdint>

#include "../../include/artab_attention.h"

namespace {

// Entry points of the library that is in use (the package may route its calls through the benchmark build):
// addresses given by bind().
struct Entries {
    decltype(&artab_workspace_bytes) workspace_bytes;
    decltype(&artab_context_attention) context_attention;
    decltype(&artab_decode_attention) decode_attention;
} lib{};
PyObject *workspace_of = nullptr;  // Python: workspace(device_index, nbytes) -> tensor

struct Call {
    int device = -1, dtype = -1;
    at::ScalarType type;
    bool ok;
    // the first tensor names the call's HIP device and element type
    explicit Call(const at::Tensor &t) : type(t.scalar_type()) {
        dtype = type == at::kBFloat16 ? ARTAB_BF16 : type == at::kHalf ? ARTAB_F16 : type == at::kFloat ? ARTAB_F32 : -1;
        device = t.is_cuda() ? t.get_device() : -1;
        ok = device >= 0 && dtype >= 0;
    }
    // another tensor of the call: once `ok` is false it stays so
    void join(const at::Tensor &t) { ok = ok && t.is_cuda() && t.get_device() == device && t.scalar_type() == type; }
    void *stream() const { return c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(device)).stream(); }
};

artab_view view(const at::Tensor &t) {  // [B, H, N, Dh], or [H, N, Dh] shared by the batch
    if (t.dim() == 3) return {t.data_ptr(), 0, t.stride(0), t.stride(1)};
    return {t.data_ptr(), t.stride(0), t.stride(1), t.stride(2)};
}
bool rows_contiguous(const at::Tensor &t) { return t.size(-1) <= 1 || t.stride(-1) == 1; }

// [B, H, Lq, Dh] over [B, Lq, H, Dh] storage
at::Tensor heads_out(const at::Tensor &q) {
    const int64_t B = q.size(0), H = q.size(1), L = q.size(2), D = q.size(3);
    return at::empty_strided({B, H, L, D}, {L * H * D, D, H * D, 1}, q.options().requires_grad(false));
}

// Scratch memory for `bytes` (null for none): the device's scratch tensor, or for float32 calls memory of the
// call's own, which `own` keeps until the launch; false: the Python side failed
bool workspace(const Call &c, const at::Tensor &q, size_t bytes, at::Tensor &own, void **ptr, size_t *have) {
    *ptr = nullptr;
    *have = 0;
    if (bytes == 0) return true;
    if (c.type == at::kFloat) {
        own = at::empty({static_cast<int64_t>(bytes)}, q.options().dtype(at::kByte).requires_grad(false));
        *ptr = own.data_ptr();
        *have = bytes;
        return true;
    }
    PyObject *t = PyObject_CallFunction(workspace_of, "in", c.device, static_cast<Py_ssize_t>(bytes));
    if (!t) return false;
    if (THPVariable_Check(t)) {
        const at::Tensor &w = THPVariable_Unpack(t);
        *ptr = w.data_ptr();
        *have = w.nbytes();
    }
    Py_DECREF(t);  // (kept alive by the package, as for the calls made from Python)
    return true;
}

PyObject *none() { Py_RETURN_NONE; }

// A number that does not convert: left to the Python path
PyObject *not_plain() {
    PyErr_Clear();
    return none();
}

// context_attention(q, k_ctx, v_ctx, scale, impl) -> (out, lse) or None
PyObject *context_attention(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 5 || !lib.context_attention) return none();
    for (int i = 0; i < 3; ++i)
        if (!THPVariable_Check(args[i])) return none();
    const at::Tensor &q = THPVariable_Unpack(args[0]), &k = THPVariable_Unpack(args[1]), &v = THPVariable_Unpack(args[2]);
    Call c(q);
    c.join(k);
    c.join(v);
    if (!c.ok || q.dim() != 4 || (k.dim() != 3 && k.dim() != 4) || k.sizes() != v.sizes() || !rows_contiguous(q) || !rows_contiguous(k) || !rows_contiguous(v))
        return none();
    const int64_t B = q.size(0), H = q.size(1), Lq = q.size(2), Dh = q.size(3), Nc = k.size(-2);
    if (k.size(-3) != H || k.size(-1) != Dh || (k.dim() == 4 && k.size(0) != B) || Nc < 1) return none();
    double scale = 0.;
    if (args[3] != Py_None) {
        scale = PyFloat_AsDouble(args[3]);
        if (PyErr_Occurred()) return not_plain();
    }
    const int impl = static_cast<int>(PyLong_AsLong(args[4]));
    if (PyErr_Occurred()) return not_plain();
    at::AutoDispatchBelowAutograd guard;
    at::Tensor own;
    void *ws;
    size_t have;
    if (!workspace(c, q, lib.workspace_bytes(B, H, Lq, Nc, Dh, c.dtype), own, &ws, &have)) return nullptr;
    at::Tensor out = heads_out(q), lse = at::empty({B, H, Lq}, q.options().dtype(at::kFloat).requires_grad(false));
    const artab_view qv = view(q), kv = view(k), vv = view(v), ov = view(out);
    if (lib.context_attention(&qv, &kv, &vv, &ov, lse.data_ptr<float>(), B, H, Lq, Nc, Dh, static_cast<float>(scale), c.dtype, ws, have, impl,
                              c.stream()) != ARTAB_OK)
        return none();
    PyObject *r = PyTuple_New(2);
    if (!r) return nullptr;
    PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(std::move(out)));
    PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(std::move(lse)));
    return r;
    END_HANDLE_TH_ERRORS
}

// decode_attention(q, k_ctx, v_ctx, k_buf, v_buf, n_buf, k_new, v_new, impl) -> out or None
PyObject *decode_attention(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 9 || !lib.decode_attention) return none();
    const int tensors[] = {0, 1, 2, 3, 4, 6, 7};
    if (!THPVariable_Check(args[0])) return none();
    Call c(THPVariable_Unpack(args[0]));
    for (int i : tensors) {
        if (!THPVariable_Check(args[i])) {
            if (i >= 6 && args[i] == Py_None) continue;
            return none();
        }
        const at::Tensor &t = THPVariable_Unpack(args[i]);
        c.join(t);
        if (!c.ok || !rows_contiguous(t) || (t.dim() != 4 && !((i == 1 || i == 2) && t.dim() == 3))) return none();
    }
    const at::Tensor &q = THPVariable_Unpack(args[0]), &kc = THPVariable_Unpack(args[1]), &vc = THPVariable_Unpack(args[2]),
                     &kb = THPVariable_Unpack(args[3]), &vb = THPVariable_Unpack(args[4]);
    const int64_t B = q.size(0), H = q.size(1), Lq = q.size(2), Dh = q.size(3), Nc = kc.size(-2), cap = kb.size(2);
    const bool has_new = args[6] != Py_None;
    if ((Lq != 1 && Lq != 2) || kc.size(-3) != H || kc.size(-1) != Dh || kc.sizes() != vc.sizes() || (kc.dim() == 4 && kc.size(0) != B) || Nc < 1 ||
        kb.sizes() != vb.sizes() || kb.size(0) != B || kb.size(1) != H || kb.size(3) != Dh || has_new != (args[7] != Py_None) || !PyLong_Check(args[5]))
        return none();
    const long n_buf = PyLong_AsLong(args[5]);
    const int impl = static_cast<int>(PyLong_AsLong(args[8]));
    if (PyErr_Occurred()) return not_plain();
    if (n_buf < 0 || n_buf > cap) return none();
    artab_view knv{}, vnv{};
    if (has_new) {
        const at::Tensor &kn = THPVariable_Unpack(args[6]), &vn = THPVariable_Unpack(args[7]);
        if (kn.sizes() != vn.sizes() || kn.size(0) != B || kn.size(1) != H || kn.size(2) != 1 || kn.size(3) != Dh) return none();
        knv = view(kn);
        vnv = view(vn);
    }
    at::AutoDispatchBelowAutograd guard;
    at::Tensor own;
    void *ws;
    size_t have;
    if (!workspace(c, q, lib.workspace_bytes(B, H, Lq, Nc, Dh, c.dtype), own, &ws, &have)) return nullptr;
    at::Tensor out = heads_out(q);
    const artab_view qv = view(q), kv = view(kc), vv = view(vc), kbv = view(kb), vbv = view(vb), ov = view(out);
    if (lib.decode_attention(&qv, &kv, &vv, &kbv, &vbv, has_new ? &knv : nullptr, has_new ? &vnv : nullptr, &ov, B, H, Lq, Nc,
                             static_cast<int>(n_buf), nullptr, cap, Dh, 0.f, c.dtype, ws, have, impl, c.stream()) != ARTAB_OK)
        return none();
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// bind(addresses: dict, workspace: callable)
PyObject *bind(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 2 || !PyDict_Check(args[0]) || !PyCallable_Check(args[1])) {
        PyErr_SetString(PyExc_TypeError, "bind(addresses, workspace)");
        return nullptr;
    }
    auto at = [&](const char *name) -> void * {
        PyObject *v = PyDict_GetItemString(args[0], name);  // borrowed
        return v ? PyLong_AsVoidPtr(v) : nullptr;
    };
    lib.workspace_bytes = reinterpret_cast<decltype(lib.workspace_bytes)>(at("artab_workspace_bytes"));
    lib.context_attention = reinterpret_cast<decltype(lib.context_attention)>(at("artab_context_attention"));
    lib.decode_attention = reinterpret_cast<decltype(lib.decode_attention)>(at("artab_decode_attention"));
    if (PyErr_Occurred()) return nullptr;
    Py_INCREF(args[1]);
    Py_XSETREF(workspace_of, args[1]);
    Py_RETURN_NONE;
}

#define ARTAB_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {ARTAB_METHOD(bind), ARTAB_METHOD(context_attention), ARTAB_METHOD(decode_attention), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() {
    PyObject *m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) < 0) Py_CLEAR(m);
    return m;
}
