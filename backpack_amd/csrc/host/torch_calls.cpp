// torch_calls.cpp — the per-call part of backpack_amd/kquant.py in native code: checks, output allocation, the current stream and
// the call through the C ABI.
//
// A decode projection's kernel takes 4 us and its call from Python took 9: 2.6 for the stream object, 1.4 for the output, 1.1 for
// ctypes' conversions, 0.9 for attributes and checks, the rest the launch.  Here the call takes 4.5 of the host's time (one 4096 x
// 4096 Q4_K matvec, one MI355X: 9.2 -> 4.7 us a call in a row of them; an embedding lookup of 512 rows 8.3 -> 4.7, a mixture layer of
// one token with its router, two calls, 25.4 -> 21.7).
//
// Every function takes plain tensors and whole numbers in their range and returns NotImplemented for anything else (a subclass, a
// weight that the library owns, a layout that the checks refuse) before it has done anything: kquant.py then takes the general
// path, which accepts or refuses the call.  Exceptions of the C++ side become Python's; a status of the library goes to the
// checker that bind() was given.  The interpreter's lock is released around the allocation of outputs and the library's call, as torch.empty
// and ctypes do: an allocation may free cached memory and wait for the device, where a host callback may want the lock.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../../include/bpk_kquant.h"

namespace {

// the library's functions, in the order of bind()'s addresses
decltype(&bpk_kq_matmul) f_matmul;
decltype(&bpk_kq_matmul_bf16) f_matmul_bf16;
decltype(&bpk_kq_matmul_fused) f_matmul_fused;
decltype(&bpk_kq_matmul_fused_workspace_bytes) f_workspace_bytes;
decltype(&bpk_kq_matmul_argmax) f_matmul_argmax;
decltype(&bpk_prefill_rows_bf16) f_prefill_rows;
decltype(&bpk_kq_dequant_rows) f_dequant_rows;
decltype(&bpk_moe_route) f_route;
decltype(&bpk_kq_moe_ffn) f_ffn;
decltype(&bpk_kq_moe_ffn_scratch_bytes) f_ffn_bytes;
PyObject* g_check;   // callable: raises for a status
PyObject *s_data, *s_type, *s_N, *s_K, *s_n_blocks, *s_stride;

PyObject* not_implemented()
{
    Py_INCREF(Py_NotImplemented);
    return Py_NotImplemented;
}

bool whole(PyObject* o, uint32_t& out)
{
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
    if (overflow || v < 0 || v > 0xFFFFFFFFll) return false;
    out = (uint32_t)v;
    return true;
}
bool attribute(PyObject* o, PyObject* name, uint32_t& out)
{
    PyObject* v = PyObject_GetAttr(o, name);
    if (!v) { PyErr_Clear(); return false; }
    const bool ok = whole(v, out);
    Py_DECREF(v);
    return ok;
}
bool real(PyObject* o, float& out)
{
    if (!PyFloat_CheckExact(o)) return false;
    out = (float)PyFloat_AS_DOUBLE(o);
    return true;
}
const at::Tensor* tensor(PyObject* o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }
// a tensor's memory, or none
bool memory(PyObject* o, void*& out)
{
    out = nullptr;
    if (o == Py_None) return true;
    const at::Tensor* t = tensor(o);
    if (t) out = t->data_ptr();
    return t != nullptr;
}
const at::Tensor* rows_of(PyObject* o, at::ScalarType dtype)
{
    const at::Tensor* t = tensor(o);
    return t && t->is_cuda() && t->scalar_type() == dtype && t->dim() > 0 && t->is_contiguous() ? t : nullptr;
}

struct Weight {
    void* data;
    uint32_t type, N, K, n_blocks, row_stride_words;
    at::Device device{at::kCPU};
    bool from(PyObject* w)
    {
        PyObject* d = PyObject_GetAttr(w, s_data);
        if (!d) { PyErr_Clear(); return false; }
        const at::Tensor* t = tensor(d);
        if (t) { data = t->data_ptr(); device = t->device(); }
        Py_DECREF(d);   // (the weight keeps it)
        return t && attribute(w, s_type, type) && attribute(w, s_N, N) && attribute(w, s_K, K) && K != 0 &&
               attribute(w, s_n_blocks, n_blocks) && attribute(w, s_stride, row_stride_words);
    }
};

at::Tensor make(at::IntArrayRef size, at::ScalarType dtype, at::Device device)
{
    return at::empty(size, at::TensorOptions().dtype(dtype).device(device));
}
void* stream() { return (void*)c10::hip::getCurrentHIPStream().stream(); }

struct Unlocked {   // of the interpreter's lock, also where something throws
    PyThreadState* state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};

// Runs c without the interpreter's lock; false with Python's exception set
template <class CALL> bool call(CALL&& c)
{
    int rc;
    {
        const Unlocked unlocked;
        rc = c();
    }
    if (rc == 0) return true;
    PyObject* r = PyObject_CallFunction(g_check, "i", rc);
    if (r) {
        Py_DECREF(r);
        PyErr_Format(PyExc_RuntimeError, "status %d of the library was not raised", rc);
    }
    return false;
}
#define TAKES(n) if (nargs != (n)) return not_implemented()

// matmul(x, w, bias, out, y_offset)
PyObject* matmul(PyObject*, PyObject* const* a, Py_ssize_t nargs)
{
    HANDLE_TH_ERRORS
    TAKES(5);
    const at::Tensor* x = rows_of(a[0], at::kFloat);
    const bool bf16 = !x;
    if (bf16) x = rows_of(a[0], at::kBFloat16);
    Weight w;
    uint32_t y_offset;
    void* bias;
    if (!x || !w.from(a[1]) || x->size(-1) != (int64_t)w.K || !memory(a[2], bias) || !whole(a[4], y_offset)) return not_implemented();
    const int64_t M = x->numel() / w.K;
    if (M > 0xFFFFFFFFll || (y_offset && (bf16 || a[3] == Py_None))) return not_implemented();
    at::Tensor y;
    if (a[3] != Py_None) {
        const at::Tensor* out = tensor(a[3]);
        if (!out || !out->is_contiguous() || out->scalar_type() != at::kFloat) return not_implemented();
        y = *out;
    }
    void* px = x->data_ptr();
    const at::Device device = x->device();
    if (!call([&] {
            if (!y.defined()) y = make({M, (int64_t)w.N}, at::kFloat, device);
            void *py = y.data_ptr(), *s = stream();
            return bf16 ? f_matmul_bf16(w.type, (const uint16_t*)px, w.data, (const float*)bias, (float*)py, (uint32_t)M, w.N, w.K, w.n_blocks,
                                        w.row_stride_words, s)
                        : f_matmul(w.type, (const float*)px, w.data, (const float*)bias, (float*)py, (uint32_t)M, w.N, w.K, w.n_blocks,
                                   w.row_stride_words, y_offset, s);
        }))
        return nullptr;
    if (a[3] != Py_None) {
        Py_INCREF(a[3]);
        return a[3];
    }
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// matmul_fused(x, w, prologue, norm_w, eps, residual, bias, out, workspace, allow_workspace, epilogue)
PyObject* matmul_fused(PyObject*, PyObject* const* a, Py_ssize_t nargs)
{
    HANDLE_TH_ERRORS
    TAKES(11);
    const at::Tensor* x = rows_of(a[0], at::kFloat);
    Weight w;
    uint32_t pro, epi;
    float eps;
    void *norm_w, *residual, *bias;
    if (!x || !w.from(a[1]) || !whole(a[2], pro) || !whole(a[10], epi) || !real(a[4], eps) || !memory(a[3], norm_w) ||
        !memory(a[5], residual) || !memory(a[6], bias) || !PyBool_Check(a[9]) || pro > 3u || epi > 3u)
        return not_implemented();
    const int64_t row = (int64_t)w.K * (pro >= BPK_PRO_SILU_MUL ? 2 : 1);
    if (x->size(-1) != row) return not_implemented();
    const int64_t M = x->numel() / row, n_out = epi ? w.N / 2u : w.N;
    if (M > 0xFFFFFFFFll) return not_implemented();
    at::Tensor y, ws;
    void* pws = nullptr;
    size_t ws_bytes = 0;
    const at::Tensor *out = a[7] == Py_None ? nullptr : tensor(a[7]), *given = a[8] == Py_None ? nullptr : tensor(a[8]);
    if ((a[7] != Py_None && !out) || (a[8] != Py_None && !given)) return not_implemented();
    if (out) y = *out;
    if (given) {
        ws_bytes = (size_t)given->numel() * given->element_size();
        pws = given->data_ptr();
    }
    const bool own_workspace = !given && a[9] == Py_True;
    const bpk_kq_fusion f{(int)pro, (const float*)norm_w, eps, (const float*)residual, (int)epi};
    void* px = x->data_ptr();
    const at::Device device = x->device();
    if (!call([&] {
            if (!out) y = make({M, n_out}, at::kFloat, device);
            if (own_workspace) {
                ws_bytes = f_workspace_bytes((uint32_t)M, (uint32_t)n_out, w.K);
                ws = make({(int64_t)ws_bytes}, at::kByte, device);
                pws = ws.data_ptr();
            }
            void *py = y.data_ptr(), *s = stream();
            return f_matmul_fused(w.type, (const float*)px, w.data, (const float*)bias, (float*)py, (uint32_t)M, (uint32_t)n_out, w.K, w.n_blocks,
                                  w.row_stride_words, 0, &f, pws, ws_bytes, s);
        }))
        return nullptr;
    if (out) {
        Py_INCREF(a[7]);
        return a[7];
    }
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// matmul_argmax(x, w, bias) -> (logits, index, value)
PyObject* matmul_argmax(PyObject*, PyObject* const* a, Py_ssize_t nargs)
{
    HANDLE_TH_ERRORS
    TAKES(3);
    const at::Tensor* x = rows_of(a[0], at::kFloat);
    Weight w;
    void* bias;
    if (!x || !w.from(a[1]) || x->size(-1) != (int64_t)w.K || !memory(a[2], bias)) return not_implemented();
    const int64_t M = x->numel() / w.K;
    if (M > 0xFFFFFFFFll) return not_implemented();
    at::Tensor y, index, value;
    void* px = x->data_ptr();
    const at::Device device = x->device();
    if (!call([&] {
            y = make({M, (int64_t)w.N}, at::kFloat, device);
            index = make({M}, at::kInt, device);
            value = make({M}, at::kFloat, device);
            void *py = y.data_ptr(), *pi = index.data_ptr(), *pv = value.data_ptr(), *s = stream();
            return f_matmul_argmax(w.type, (const float*)px, w.data, (const float*)bias, (float*)py, (uint32_t)M, w.N, w.K, w.n_blocks,
                                   w.row_stride_words, (int32_t*)pi, (float*)pv, s);
        }))
        return nullptr;
    return Py_BuildValue("(NNN)", THPVariable_Wrap(std::move(y)), THPVariable_Wrap(std::move(index)), THPVariable_Wrap(std::move(value)));
    END_HANDLE_TH_ERRORS
}

// prefill_rows_bf16(x, K, prologue, norm_w, eps)
PyObject* prefill_rows_bf16(PyObject*, PyObject* const* a, Py_ssize_t nargs)
{
    HANDLE_TH_ERRORS
    TAKES(5);
    const at::Tensor* x = rows_of(a[0], at::kFloat);
    uint32_t K, pro;
    void* norm_w;
    float eps;
    if (!x || !whole(a[1], K) || K == 0 || !whole(a[2], pro) || pro > 3u || !memory(a[3], norm_w) || !real(a[4], eps)) return not_implemented();
    const int64_t row = (int64_t)K * (pro >= BPK_PRO_SILU_MUL ? 2 : 1);
    if (x->size(-1) != row) return not_implemented();
    const int64_t M = x->numel() / row;
    if (M > 0xFFFFFFFFll) return not_implemented();
    at::Tensor y;
    void* px = x->data_ptr();
    const at::Device device = x->device();
    if (!call([&] {
            y = make({M, (int64_t)K}, at::kBFloat16, device);
            void *py = y.data_ptr(), *s = stream();
            return f_prefill_rows((int)pro, (const float*)px, (const float*)norm_w, eps, (uint32_t)M, K, (uint16_t*)py, s);
        }))
        return nullptr;
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// dequant_rows(w, rows)
PyObject* dequant_rows(PyObject*, PyObject* const* a, Py_ssize_t nargs)
{
    HANDLE_TH_ERRORS
    TAKES(2);
    Weight w;
    const at::Tensor* rows = tensor(a[1]);
    if (!rows || !rows->is_cuda() || rows->scalar_type() != at::kInt || !w.from(a[0])) return not_implemented();
    const int64_t M = rows->numel();
    if (M > 0xFFFFFFFFll) return not_implemented();
    at::Tensor y;
    void* pr = rows->data_ptr();
    if (!call([&] {
            y = make({M, (int64_t)w.K}, at::kFloat, w.device);
            void *py = y.data_ptr(), *s = stream();
            return f_dequant_rows(w.type, w.data, w.row_stride_words, (const int32_t*)pr, (uint32_t)M, w.K, (float*)py, s);
        }))
        return nullptr;
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// moe_route(x, router_w, k, normalize) -> (index, weight)
PyObject* moe_route(PyObject*, PyObject* const* a, Py_ssize_t nargs)
{
    HANDLE_TH_ERRORS
    TAKES(4);
    const at::Tensor *x = tensor(a[0]), *r = tensor(a[1]);
    uint32_t k;
    if (!x || !r || x->scalar_type() != at::kFloat || r->scalar_type() != at::kFloat || x->dim() != 2 || r->dim() < 1 || !x->is_contiguous() ||
        !r->is_contiguous() || !whole(a[2], k) || !PyBool_Check(a[3]))
        return not_implemented();
    const int64_t T = x->size(0), H = x->size(1), E = r->size(0);
    if ((T | H | E) > 0xFFFFFFFFll) return not_implemented();
    at::Tensor index, weight;
    void *px = x->data_ptr(), *pr = r->data_ptr();
    const at::Device device = x->device();
    const int normalize = a[3] == Py_True;
    if (!call([&] {
            index = make({T, (int64_t)k}, at::kInt, device);
            weight = make({T, (int64_t)k}, at::kFloat, device);
            void *pi = index.data_ptr(), *pw = weight.data_ptr(), *s = stream();
            return f_route((const float*)px, (const float*)pr, (uint32_t)T, (uint32_t)H, (uint32_t)E, k, normalize, nullptr, (uint32_t*)pi, (float*)pw, s);
        }))
        return nullptr;
    return Py_BuildValue("(NN)", THPVariable_Wrap(std::move(index)), THPVariable_Wrap(std::move(weight)));
    END_HANDLE_TH_ERRORS
}

// moe_ffn(x, gate, up, down, expert_idx, expert_wt, n_experts)
PyObject* moe_ffn(PyObject*, PyObject* const* a, Py_ssize_t nargs)
{
    HANDLE_TH_ERRORS
    TAKES(7);
    const at::Tensor *x = tensor(a[0]), *idx = tensor(a[4]), *wt = tensor(a[5]);
    Weight gate, up, down;
    uint32_t E;
    if (!x || !idx || !wt || idx->dim() != 2 || !gate.from(a[1]) || !up.from(a[2]) || !down.from(a[3]) || !whole(a[6], E)) return not_implemented();
    const int64_t T = idx->size(0), k = idx->size(1);
    if ((T | k) > 0xFFFFFFFFll) return not_implemented();
    at::Tensor scratch, y;
    void *px = x->data_ptr(), *pi = idx->data_ptr(), *pw = wt->data_ptr();
    const at::Device device = x->device();
    if (!call([&] {
            const size_t bytes = f_ffn_bytes((uint32_t)T, (uint32_t)k, gate.K, down.K);
            scratch = make({(int64_t)bytes}, at::kByte, device);
            y = make({T, (int64_t)gate.K}, at::kFloat, device);
            void *py = y.data_ptr(), *ps = scratch.data_ptr(), *s = stream();
            return f_ffn(gate.type, down.type, (const float*)px, gate.data, up.data, down.data, (const uint32_t*)pi, (const float*)pw, (float*)py,
                         (uint32_t)T, (uint32_t)k, E, gate.K, down.K, ps, bytes, s);
        }))
        return nullptr;
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// stream() -> the current device's current stream
PyObject* current_stream(PyObject*, PyObject*)
{
    HANDLE_TH_ERRORS
    return PyLong_FromVoidPtr(stream());
    END_HANDLE_TH_ERRORS
}

// bind(addresses, check): the functions of a loaded library, by address
PyObject* bind(PyObject*, PyObject* args)
{
    PyObject *list, *check;
    if (!PyArg_ParseTuple(args, "O!O", &PyList_Type, &list, &check)) return nullptr;
    void* p[10];
    if (PyList_GET_SIZE(list) != 10) {
        PyErr_SetString(PyExc_ValueError, "ten addresses expected");
        return nullptr;
    }
    for (int i = 0; i < 10; ++i) {
        p[i] = PyLong_AsVoidPtr(PyList_GET_ITEM(list, i));
        if (!p[i]) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "an address is null");
            return nullptr;
        }
    }
    f_matmul = (decltype(f_matmul))p[0];
    f_matmul_bf16 = (decltype(f_matmul_bf16))p[1];
    f_matmul_fused = (decltype(f_matmul_fused))p[2];
    f_workspace_bytes = (decltype(f_workspace_bytes))p[3];
    f_matmul_argmax = (decltype(f_matmul_argmax))p[4];
    f_prefill_rows = (decltype(f_prefill_rows))p[5];
    f_dequant_rows = (decltype(f_dequant_rows))p[6];
    f_route = (decltype(f_route))p[7];
    f_ffn = (decltype(f_ffn))p[8];
    f_ffn_bytes = (decltype(f_ffn_bytes))p[9];
    Py_INCREF(check);
    Py_XSETREF(g_check, check);
    Py_RETURN_NONE;
}

#define FAST(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST(matmul), FAST(matmul_fused), FAST(matmul_argmax), FAST(prefill_rows_bf16), FAST(dequant_rows), FAST(moe_route),
                         FAST(moe_ffn), {"stream", current_stream, METH_NOARGS, nullptr}, {"bind", bind, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_torch_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_calls(void)
{
    s_data = PyUnicode_InternFromString("data");
    s_type = PyUnicode_InternFromString("type");
    s_N = PyUnicode_InternFromString("N");
    s_K = PyUnicode_InternFromString("K");
    s_n_blocks = PyUnicode_InternFromString("n_blocks");
    s_stride = PyUnicode_InternFromString("row_stride_words");
    return PyModule_Create(&module_def);
}
