// Python extension `aiter_amd._bridge`: calls an entry point of libaiter_fp8bs.so with torch tensors, without the detour
// over ctypes.  A decode step is bound by the host: of the 8.8 us that a GEMM call took, 5 were tensor descriptors and
// argument conversion in Python; here they are 0.5.
//
//   bind(name, address)     the entry points' addresses, once
//   call(name, *args)       the entry point's status; None where an argument is not of the plain kind handled here (a tensor
//                           subclass, a wrapped or symbolic tensor, a type that does not fit the parameter): nothing has
//                           been called then, and the caller takes the ctypes route, whose errors are the interface's
//
// Nothing is kept from one call to the next: descriptors live on the stack of the call.
#include <Python.h>

#include <array>
#include <cstring>
#include <tuple>
#include <utility>

#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/aiter_fp8bs.h"

namespace {

int dtype_id(c10::ScalarType t) // ids as in aiter_amd/dtypes.py
{
    switch(t)
    {
    case c10::ScalarType::Float8_e4m3fn: return 0;
    case c10::ScalarType::Float8_e8m0fnu: return 1;
    case c10::ScalarType::Half: return 2;
    case c10::ScalarType::BFloat16: return 3;
    case c10::ScalarType::Float: return 4;
    case c10::ScalarType::UInt32: return 7;
    case c10::ScalarType::Int: return 8;
    case c10::ScalarType::Short: return 9;
    case c10::ScalarType::Char: return 10;
    case c10::ScalarType::Byte: return 11;
    case c10::ScalarType::Long: return 12;
    case c10::ScalarType::UInt64: return 13;
    default: return -1;
    }
}

struct Context
{
    int  device = -1; // of the first GPU tensor
    bool ok     = true;
};

// one argument into one parameter; `d` is the parameter's own descriptor, used where it is a tensor
void convert(PyObject* a, aiter_tensor_t& d, aiter_tensor_t*& out, Context& c)
{
    out = nullptr;
    if(a == Py_None)
        return;
    if(!THPVariable_CheckExact(a))
    {
        c.ok = false;
        return;
    }
    const at::Tensor& t  = THPVariable_Unpack(a);
    const int         id = dtype_id(t.scalar_type());
    const auto        sizes = t.sizes(), strides = t.strides();
    if(id < 0 || sizes.size() > 8)
    {
        c.ok = false;
        return;
    }
    std::memset(&d, 0, sizeof d);
    d.ptr    = t.data_ptr();
    d.numel_ = (size_t)t.numel();
    d.ndim   = (int)sizes.size();
    for(size_t i = 0; i < sizes.size(); ++i)
    {
        d.shape[i]   = sizes[i];
        d.strides[i] = strides[i];
    }
    d.dtype_            = (decltype(d.dtype_))id;
    const c10::Device v = t.device();
    d.device_id         = v.is_cpu() ? -1 : (int)v.index();
    if(c.device < 0 && v.is_cuda())
        c.device = v.index();
    out = &d;
}

template <class I>
void convert_integer(PyObject* a, I& out, Context& c)
{
    out = 0;
    if(!PyLong_Check(a)) // (a bool is one)
    {
        c.ok = false;
        return;
    }
    int             over = 0;
    const long long v    = PyLong_AsLongLongAndOverflow(a, &over);
    c.ok                 = c.ok && over == 0 && (long long)(I)v == v;
    out                  = (I)v;
}
void convert(PyObject* a, aiter_tensor_t&, int& out, Context& c) { convert_integer(a, out, c); }
void convert(PyObject* a, aiter_tensor_t&, int64_t& out, Context& c) { convert_integer(a, out, c); }

void convert(PyObject* a, aiter_tensor_t&, float& out, Context& c)
{
    out = 0.f;
    if(PyFloat_Check(a))
        out = (float)PyFloat_AS_DOUBLE(a);
    else
        c.ok = false;
}

void convert(PyObject* a, aiter_tensor_t&, const char*& out, Context& c)
{
    out = nullptr;
    if(a == Py_None)
        return;
    out = PyUnicode_Check(a) ? PyUnicode_AsUTF8(a) : nullptr;
    if(!out)
    {
        PyErr_Clear();
        c.ok = false;
    }
}

template <class F>
struct Invoke;
template <class... P>
struct Invoke<int (*)(P...)>
{
    static constexpr size_t kArgs = sizeof...(P) - 1; // the last parameter is the stream

    // false: not called
    static bool run(void* address, PyObject* const* a, Py_ssize_t n, int& status)
    {
        return n == (Py_ssize_t)kArgs && go(address, a, status, std::make_index_sequence<kArgs>());
    }
    template <size_t... I>
    static bool go(void* address, PyObject* const* a, int& status, std::index_sequence<I...>)
    {
        std::array<aiter_tensor_t, kArgs> d;
        std::tuple<P...>                  v;
        Context                           c;
        (convert(a[I], d[I], std::get<I>(v), c), ...);
        if(!c.ok)
            return false;
        std::get<kArgs>(v) = c.device < 0 ? nullptr : c10::hip::getCurrentHIPStream((c10::DeviceIndex)c.device).stream();
        Py_BEGIN_ALLOW_THREADS
        status = std::apply((int (*)(P...))address, v);
        Py_END_ALLOW_THREADS
        return true;
    }
};

struct Entry
{
    const char* name;
    bool (*run)(void*, PyObject* const*, Py_ssize_t, int&);
    void* address;
};
#define ENTRY(f) {#f, &Invoke<decltype(&f)>::run, nullptr}
Entry entries[] = {
    ENTRY(gemm_a8w8_blockscale),
    ENTRY(gemm_a8w8_blockscale_bpreshuffle),
    ENTRY(dynamic_per_token_scaled_quant),
    ENTRY(rmsnorm_quant),
    ENTRY(add_rmsnorm_quant),
    ENTRY(rmsnorm),
    ENTRY(add_rmsnorm),
    ENTRY(topk_softmax),
    ENTRY(moe_sorting_fwd),
    ENTRY(fmoe_fp8_blockscale_g1u1),
    ENTRY(weight_per_128x128_quant),
    ENTRY(gemm_a8w8_blockscale_noalloc),
    ENTRY(gemm_a8w8_blockscale_bpreshuffle_asm),
};

Entry* find(PyObject* name)
{
    const char* s = PyUnicode_Check(name) ? PyUnicode_AsUTF8(name) : nullptr;
    if(s)
        for(Entry& e : entries)
            if(std::strcmp(e.name, s) == 0)
                return &e;
    PyErr_Clear();
    return nullptr;
}

PyObject* bridge_bind(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    Entry* e = n == 2 ? find(a[0]) : nullptr;
    if(e)
        e->address = PyLong_AsVoidPtr(a[1]);
    if(PyErr_Occurred())
        return nullptr;
    Py_RETURN_NONE;
}

PyObject* bridge_call(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    Entry* e = n >= 1 ? find(a[0]) : nullptr;
    if(!e || !e->address)
        Py_RETURN_NONE;
    int status = 0;
    try
    {
        if(!e->run(e->address, a + 1, n - 1, status))
            Py_RETURN_NONE;
    }
    catch(...) // a tensor without a plain address or with symbolic sizes
    {
        Py_RETURN_NONE;
    }
    return PyLong_FromLong(status);
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void (*)())bridge_bind, METH_FASTCALL, nullptr},
    {"call", (PyCFunction)(void (*)())bridge_call, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_bridge", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__bridge() { return PyModule_Create(&module); }
