// tuna_amd/_native.so: the ops' path from torch tensors to the C ABI, as a CPython extension.
//
// A small launch (4096 x 4096, one token: 5 us on the device) was bounded by the host: argument checks, the device
// guard, the current stream and the ctypes conversion took 11 us a call in Python.  Here the same checks read the
// tensors' C++ objects: 3.5 us a call, 2.8 of them the HIP launch (a pass of that launch among others 10.9 -> 4.1 us,
// 6144 x 4096 at 16 tokens 11.1 -> 6.6).  A call whose arguments do not pass - or whose tensors are not on the current device - returns
// None without having done anything, and the Python op then goes its own way, which raises what it always raised or
// runs the call; so there is one place that words the errors.  Otherwise the status of the C ABI call is returned.
//
// The entry points are those of the library that _lib.py has active (product or diagnostic build): bind() takes them.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <vector>

#include "../../include/tuna_amd.h"

namespace {

struct EntryPoints {
    decltype(&tuna_matmul) matmul;
    decltype(&tuna_matmul_fused) matmul_fused;
    decltype(&tuna_matmul_multi) matmul_multi;
    decltype(&tuna_matmul_grouped) matmul_grouped;
    decltype(&tuna_matmul_blockwise) matmul_blockwise;
    decltype(&tuna_dequant) dequant;
    decltype(&tuna_dequant_blockwise) dequant_blockwise;
    decltype(&tuna_quantize_blockwise) quantize_blockwise;
};
EntryPoints g_fn;  // written and read under the GIL only: a call takes its pointer before it lets go of the GIL
constexpr int kEntryPoints = sizeof(EntryPoints) / sizeof(void *);

// The arguments of one call.  The first tensor names the device; `ok` turns false at the first argument that the
// Python op would refuse or convert.
struct Args {
    bool ok = true;
    int device = -1;

    void *tensor(PyObject *o, at::ScalarType type, int64_t numel)
    {
        if (!ok || !THPVariable_Check(o)) return refuse();
        const at::Tensor &t = THPVariable_Unpack(o);
        if (!t.is_cuda() || t.scalar_type() != type || !t.is_contiguous() || t.numel() != numel) return refuse();
        const int dev = t.get_device();
        if (device < 0) {
            device = dev;
            if (c10::hip::current_device() != dev) return refuse();
        } else if (dev != device) {
            return refuse();
        }
        return t.data_ptr();
    }
    int integer(PyObject *o)
    {
        if (!ok) return 0;
        if (!PyLong_CheckExact(o)) return refuse(), 0;
        int overflow = 0;
        const long v = PyLong_AsLongAndOverflow(o, &overflow);
        if (overflow || v < 0 || v > 0x7fffffff) return refuse(), 0;
        return (int)v;
    }
    // m, n, k of a GEMM, in the order of the ops' arguments
    void shape(PyObject *const *a, int &m, int &n, int &k)
    {
        m = integer(a[0]), n = integer(a[1]), k = integer(a[2]);
        if (m <= 0 || n <= 0 || k <= 0 || m % 8 || k % 8) ok = false;
    }
    void *stream() const { return c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }

private:
    void *refuse()
    {
        ok = false;
        return nullptr;
    }
};

constexpr at::ScalarType kHalf = at::kHalf, kByte = at::kByte, kFloat = at::kFloat;

// The ABI call runs without the GIL, as it did through ctypes.  (`call` holds its entry point by value.)
template <class F>
PyObject *status_of(F &&call)
{
    int rc;
    Py_BEGIN_ALLOW_THREADS rc = call();
    Py_END_ALLOW_THREADS return PyLong_FromLong(rc);
}

// data_ptr() of a tensor without storage throws: such a call is the Python op's to refuse.
#define NATIVE_OP(name, nargs)                                                   \
    PyObject *name##_checked(PyObject *const *a);                                \
    PyObject *name(PyObject *, PyObject *const *a, Py_ssize_t n)                 \
    {                                                                            \
        if (n != nargs || !g_fn.matmul) Py_RETURN_NONE;                          \
        try {                                                                    \
            return name##_checked(a);                                            \
        } catch (const std::exception &) {                                       \
            Py_RETURN_NONE;                                                      \
        }                                                                        \
    }                                                                            \
    PyObject *name##_checked(PyObject *const *a)

NATIVE_OP(matmul, 8)  // x, q, s, c, o, m, n, k
{
    Args g;
    int m, n, k;
    g.shape(a + 5, m, n, k);
    void *x = g.tensor(a[0], kHalf, (int64_t)n * k), *q = g.tensor(a[1], kByte, (int64_t)m * k / 2);
    void *s = g.tensor(a[2], kFloat, m), *c = g.tensor(a[3], kFloat, 16), *o = g.tensor(a[4], kHalf, (int64_t)n * m);
    if (!g.ok) Py_RETURN_NONE;
    void *st = g.stream();
    return status_of([&, fn = g_fn.matmul] { return fn(q, x, c, s, o, m, n, k, st); });
}

NATIVE_OP(matmul_fused, 10)  // x, q, s, c, o, m, n, k, epilogue, residual or None
{
    Args g;
    int m, n, k;
    g.shape(a + 5, m, n, k);
    const int ep = g.integer(a[8]);
    void *x = g.tensor(a[0], kHalf, (int64_t)n * k), *q = g.tensor(a[1], kByte, (int64_t)m * k / 2);
    void *s = g.tensor(a[2], kFloat, m), *c = g.tensor(a[3], kFloat, 16);
    void *o = g.tensor(a[4], kHalf, (int64_t)n * (ep == TUNA_EPILOGUE_SILU_MUL ? m / 2 : m));
    void *r = ep == TUNA_EPILOGUE_RESIDUAL ? g.tensor(a[9], kHalf, (int64_t)n * m) : nullptr;
    if (!g.ok) Py_RETURN_NONE;
    void *st = g.stream();
    return status_of([&, fn = g_fn.matmul_fused] { return fn(q, x, c, s, o, m, n, k, nullptr, TUNA_DECODE_GEMM, ep, r, st); });
}

NATIVE_OP(matmul_blockwise, 9)  // x, q, s, c, o, m, n, k, block_size
{
    Args g;
    int m, n, k;
    g.shape(a + 5, m, n, k);
    const int bs = g.integer(a[8]);
    if (!g.ok || bs <= 0 || k % bs) Py_RETURN_NONE;
    void *x = g.tensor(a[0], kHalf, (int64_t)n * k), *q = g.tensor(a[1], kByte, (int64_t)m * k / 2);
    void *s = g.tensor(a[2], kFloat, (int64_t)m * (k / bs)), *c = g.tensor(a[3], kFloat, 16);
    void *o = g.tensor(a[4], kHalf, (int64_t)n * m);
    if (!g.ok) Py_RETURN_NONE;
    void *st = g.stream();
    return status_of([&, fn = g_fn.matmul_blockwise] { return fn(q, x, c, s, o, m, n, k, bs, st); });
}

NATIVE_OP(matmul_multi, 1)  // list or tuple of (x, q, s, c, o, m, n, k) tuples
{
    if (!PyList_CheckExact(a[0]) && !PyTuple_CheckExact(a[0])) Py_RETURN_NONE;
    const Py_ssize_t count = PySequence_Fast_GET_SIZE(a[0]);
    PyObject **items = PySequence_Fast_ITEMS(a[0]);
    Args g;
    std::vector<tuna_gemm_problem> p((size_t)count);
    for (Py_ssize_t i = 0; i < count && g.ok; ++i) {
        if (!PyTuple_CheckExact(items[i]) || PyTuple_GET_SIZE(items[i]) != 8) Py_RETURN_NONE;
        PyObject **t = PySequence_Fast_ITEMS(items[i]);
        int m, n, k;
        g.shape(t + 5, m, n, k);
        p[i].x = g.tensor(t[0], kHalf, (int64_t)n * k);
        p[i].q = g.tensor(t[1], kByte, (int64_t)m * k / 2);
        p[i].absmax = g.tensor(t[2], kFloat, m);
        p[i].code = g.tensor(t[3], kFloat, 16);
        p[i].out = g.tensor(t[4], kHalf, (int64_t)n * m);
        p[i].m = m, p[i].n = n, p[i].k = k;
    }
    if (!g.ok || !count) Py_RETURN_NONE;
    void *st = g.stream();
    return status_of([&, fn = g_fn.matmul_multi] { return fn(p.data(), (int)count, st); });
}

NATIVE_OP(matmul_grouped, 9)  // x, q, s, c, o, m_group, n_groups, k, token_offsets (list or tuple)
{
    Args g;
    const int m = g.integer(a[5]), groups = g.integer(a[6]), k = g.integer(a[7]);
    if (!g.ok || m <= 0 || groups <= 0 || k <= 0 || (!PyList_CheckExact(a[8]) && !PyTuple_CheckExact(a[8])) ||
        PySequence_Fast_GET_SIZE(a[8]) != (Py_ssize_t)groups + 1)
        Py_RETURN_NONE;
    std::vector<int> offs((size_t)groups + 1);
    for (int i = 0; i <= groups; ++i) offs[i] = g.integer(PySequence_Fast_ITEMS(a[8])[i]);
    const int64_t n = offs[groups], rows = (int64_t)m * groups;
    void *x = g.tensor(a[0], kHalf, n * k), *q = g.tensor(a[1], kByte, rows * k / 2), *s = g.tensor(a[2], kFloat, rows);
    void *c = g.tensor(a[3], kFloat, 16), *o = g.tensor(a[4], kHalf, n * m);
    if (!g.ok) Py_RETURN_NONE;
    void *st = g.stream();
    return status_of([&, fn = g_fn.matmul_grouped] { return fn(q, x, c, s, o, m, groups, k, offs.data(), nullptr, TUNA_DECODE_GEMM, st); });
}

NATIVE_OP(dequant, 7)  // q, absmax, codebook, o, m, k, block_size or None
{
    Args g;
    const int m = g.integer(a[4]), k = g.integer(a[5]);
    const int bs = a[6] == Py_None ? k : g.integer(a[6]);
    if (!g.ok || m <= 0 || k <= 0 || m % 8 || k % 8 || bs <= 0 || k % bs) Py_RETURN_NONE;
    void *q = g.tensor(a[0], kByte, (int64_t)m * k / 2), *s = g.tensor(a[1], kFloat, (int64_t)m * (k / bs));
    void *c = g.tensor(a[2], kFloat, 16), *o = g.tensor(a[3], kHalf, (int64_t)m * k);
    if (!g.ok) Py_RETURN_NONE;
    void *st = g.stream();
    return status_of([&, per_row = g_fn.dequant, blockwise = g_fn.dequant_blockwise] {
        return bs == k ? per_row(q, s, c, o, m, k, st) : blockwise(q, s, c, o, m, k, bs, TUNA_DECODE_DEQUANT, st);
    });
}

NATIVE_OP(quantize, 3)  // w, codebook, block_size or None -> (status, q, absmax)
{
    if (!THPVariable_Check(a[0])) Py_RETURN_NONE;
    const at::Tensor &wt = THPVariable_Unpack(a[0]);
    if (wt.dim() != 2 || wt.size(0) > 0x7fffffff || wt.size(1) > 0x7fffffff) Py_RETURN_NONE;
    const int m = (int)wt.size(0), k = (int)wt.size(1);
    Args g;
    const int bs = a[2] == Py_None ? k : g.integer(a[2]);
    if (!g.ok || m <= 0 || k <= 0 || m % 8 || k % 8 || bs <= 0 || k % bs) Py_RETURN_NONE;
    void *w = g.tensor(a[0], kHalf, (int64_t)m * k), *c = g.tensor(a[1], kFloat, 16);
    if (!g.ok) Py_RETURN_NONE;
    at::Tensor q = at::empty({m / 8, k / 8, 32}, wt.options().dtype(kByte));
    at::Tensor absmax = a[2] == Py_None ? at::empty({m}, wt.options().dtype(kFloat)) : at::empty({m, k / bs}, wt.options().dtype(kFloat));
    void *st = g.stream(), *qp = q.data_ptr(), *ap = absmax.data_ptr();
    const auto fn = g_fn.quantize_blockwise;
    int rc;
    Py_BEGIN_ALLOW_THREADS rc = fn(w, c, qp, ap, m, k, bs, st);
    Py_END_ALLOW_THREADS
    return Py_BuildValue("iNN", rc, THPVariable_Wrap(std::move(q)), THPVariable_Wrap(std::move(absmax)));
}

PyObject *bind(PyObject *, PyObject *addresses)
{
    if (!PyTuple_CheckExact(addresses) || PyTuple_GET_SIZE(addresses) != kEntryPoints)
        return PyErr_Format(PyExc_ValueError, "bind takes a tuple of %d addresses", kEntryPoints);
    void *p[kEntryPoints];
    for (int i = 0; i < kEntryPoints; ++i)
        if (!(p[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(addresses, i))))
            return PyErr_Occurred() ? nullptr : PyErr_Format(PyExc_ValueError, "address %d is null", i);
    memcpy(&g_fn, p, sizeof g_fn);
    Py_RETURN_NONE;
}

#define OP(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {OP(matmul),         OP(matmul_fused), OP(matmul_blockwise), OP(matmul_multi),
                          OP(matmul_grouped), OP(dequant),      OP(quantize),         {"bind", bind, METH_O, nullptr},
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, kMethods};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&kModule); }
