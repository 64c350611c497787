// torch_calls.cpp - the Python binding's call path for torch tensors: Backend.matmul / matmul_ex / matmul_norm / matmul_static.
//
// A small linear is bound by the host: the launch itself takes 2.9 us of host time, the kernel behind it less.  Looking
// the tensors over in Python (shape, device, contiguity, type, address: a dozen attribute calls) and going through
// ctypes added 2.5 us to that; here both cost 0.5 us (one row, 4096 -> 1024, call to call: 5.8 -> 3.7 us).  Nothing is decided here: a call whose
// arguments are not exactly what the checks in backend.py accept is handed back (kSlow), and the Python code answers it, errors
// included.  That goes for tensors that cannot be looked over from here too: subclasses, which may answer in Python, and
// tensors of a transform (torch.vmap, torch.func.grad), which have no address - asking them throws, and nothing that is thrown
// leaves an entry.
#include <Python.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include "../../include/cybq.h"

namespace {

constexpr int kSlow = 1;             // (statuses are zero or negative)

struct Args {
    cybq_ctx* ctx;
    const cybq_weight* w;
    int device;
    int64_t N = 0, K = 0, M = 0;
    void* stream = nullptr;
};

// number of elements `t` has to hold -> its address, or nullptr where the Python checks have to look at it
void* address(PyObject* o, int device, int64_t elems, int* dtype)
{
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.is_cuda() || t.get_device() != device || !t.is_contiguous() || t.numel() < elems) return nullptr;
    if (dtype) {
        switch (t.scalar_type()) {
            case at::kFloat: *dtype = CYBQ_F32; break;
            case at::kHalf: *dtype = CYBQ_F16; break;
            case at::kBFloat16: *dtype = CYBQ_BF16; break;
            default: return nullptr;
        }
    }
    return t.data_ptr();
}

bool as_int(PyObject* o, int64_t* v)
{
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    *v = PyLong_AsLongLongAndOverflow(o, &overflow);
    return overflow == 0;
}

// ctx, device, weight address; M (or None: the rows of x), stream
bool common(PyObject* const* a, PyObject* x, PyObject* m, PyObject* stream, Args* r)
{
    int64_t ctx, device, w, st;
    if (!as_int(a[0], &ctx) || !as_int(a[1], &device) || !as_int(a[2], &w) || !as_int(stream, &st)) return false;
    if (!ctx || !w) return false;
    r->ctx = reinterpret_cast<cybq_ctx*>(static_cast<uintptr_t>(ctx));
    r->w = reinterpret_cast<const cybq_weight*>(static_cast<uintptr_t>(w));
    r->device = (int)device;
    r->stream = reinterpret_cast<void*>(static_cast<uintptr_t>(st));
    if (m == Py_None) {
        if (!THPVariable_CheckExact(x)) return false;
        const at::Tensor& t = THPVariable_Unpack(x);
        r->M = t.dim() == 2 ? t.size(0) : 1;
    } else if (!as_int(m, &r->M)) {
        return false;
    }
    return r->M >= 1 && r->M <= (int64_t)1 << 24 && cybq_weight_info(r->w, nullptr, &r->N, &r->K, nullptr) == CYBQ_OK;
}

PyObject* answer(int rc) { return PyLong_FromLong(rc); }

// the library runs without the interpreter's lock, as under ctypes
struct Unlocked {
    PyThreadState* state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};

using Call = PyObject*(PyObject* const*, Py_ssize_t);

template <Call* F>
PyObject* entry(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    try {
        return F(a, n);
    } catch (...) {
        PyErr_Clear();                  // (a subclass's own exception; the Python checks meet it again)
        return answer(kSlow);
    }
}

// matmul(ctx, device, w, x, y, M, xdt, ydt, stream)
PyObject* matmul(PyObject* const* a, Py_ssize_t n)
{
    Args r;
    if (n != 9 || !common(a, a[3], a[5], a[8], &r)) return answer(kSlow);
    int xdt = 0, ydt = 0;
    int64_t code;
    void* x = address(a[3], r.device, r.M * r.K, a[6] == Py_None ? &xdt : nullptr);
    void* y = address(a[4], r.device, r.M * r.N, a[7] == Py_None ? &ydt : nullptr);
    if (!x || !y) return answer(kSlow);
    if (a[6] != Py_None) {
        if (!as_int(a[6], &code)) return answer(kSlow);
        xdt = (int)code;
    }
    if (a[7] != Py_None) {
        if (!as_int(a[7], &code)) return answer(kSlow);
        ydt = (int)code;
    }
    int rc;
    {
        Unlocked u;
        rc = cybq_matmul(r.ctx, r.w, x, (cybq_dtype)xdt, r.M, y, (cybq_dtype)ydt, r.stream);
    }
    return answer(rc);
}

// matmul_static(ctx, device, w, x, y, M, stream)
PyObject* matmul_static(PyObject* const* a, Py_ssize_t n)
{
    Args r;
    if (n != 7 || !common(a, a[3], a[5], a[6], &r)) return answer(kSlow);
    int xdt = 0, ydt = 0;
    void* x = address(a[3], r.device, r.M * r.K, &xdt);
    void* y = address(a[4], r.device, r.M * r.N, &ydt);
    if (!x || !y) return answer(kSlow);
    int rc;
    {
        Unlocked u;
        rc = cybq_matmul_static(r.ctx, r.w, x, (cybq_dtype)xdt, r.M, y, (cybq_dtype)ydt, r.stream);
    }
    return answer(rc);
}

// matmul_fused(ctx, device, w, x, gamma or None, eps, y, epilogue, residual or None, M, stream)
PyObject* matmul_fused(PyObject* const* a, Py_ssize_t n)
{
    Args r;
    int64_t epi;
    if (n != 11 || !common(a, a[3], a[9], a[10], &r) || !as_int(a[7], &epi)) return answer(kSlow);
    const int64_t cols = epi == CYBQ_EPI_SWIGLU ? r.N / 2 : r.N;
    int xdt = 0, ydt = 0, gdt = 0;
    void* x = address(a[3], r.device, r.M * r.K, &xdt);
    void* y = address(a[6], r.device, r.M * cols, &ydt);
    if (!x || !y) return answer(kSlow);
    void *gamma = nullptr, *residual = nullptr;
    if (a[4] != Py_None && !(gamma = address(a[4], r.device, r.K, &gdt))) return answer(kSlow);
    if (a[8] != Py_None && !(residual = address(a[8], r.device, r.M * cols, nullptr))) return answer(kSlow);
    double eps = 0.0;
    if (gamma) {
        if (!PyFloat_CheckExact(a[5])) return answer(kSlow);
        eps = PyFloat_AS_DOUBLE(a[5]);
    }
    int rc;
    {
        Unlocked u;
        if (gamma)
            rc = cybq_matmul_norm(r.ctx, r.w, x, (cybq_dtype)xdt, r.M, gamma, (cybq_dtype)gdt, (float)eps, y, (cybq_dtype)ydt,
                                  (cybq_epilogue)epi, residual, r.stream);
        else
            rc = cybq_matmul_ex(r.ctx, r.w, x, (cybq_dtype)xdt, r.M, y, (cybq_dtype)ydt, (cybq_epilogue)epi, residual, r.stream);
    }
    return answer(rc);
}

PyMethodDef kMethods[] = {
    {"matmul", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(entry<matmul>)), METH_FASTCALL, nullptr},
    {"matmul_static", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(entry<matmul_static>)), METH_FASTCALL, nullptr},
    {"matmul_fused", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(entry<matmul_fused>)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_torch_calls", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_calls(void)
{
    PyObject* m = PyModule_Create(&kModule);
    if (m && PyModule_AddStringConstant(m, "TORCH_VERSION", TORCH_VERSION) != 0) Py_CLEAR(m);
    return m;
}
