// Host path of the linears: one native call per forward for the calls a model
// makes (contiguous GPU activations, operands as the layers keep them).  It
// checks the operands, allocates the output and the intermediates and calls the
// library; anything else returns None and takes the Python path, which handles
// every form and raises the errors.
//
// The intermediates come from torch's caching allocator on the current stream
// and go back to it when the call returns, which orders their reuse on that
// stream; nothing is kept between calls.  Shapes whose GEMM splits k over
// workgroups need a workspace with cleared counters and are left to Python,
// which keeps one per stream.
//
// Measured on MI355X (M = 1, 256 x 256, back to back): 17.3 us per W4A4
// call through Python and ctypes, 7.1 here; 21.9 and 9.5 with a LoRA; W8A8 27.2
// (16.0 as one library call) and 6.8.

#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <pybind11/pybind11.h>

#include "../../include/convrot_mi355x.h"

namespace {

// f32 0, bf16 1, f16 2 (the library's dtype codes), -1: none of them
int dtype_code(const at::Tensor& t) {
    switch (t.scalar_type()) {
        case at::kFloat: return 0;
        case at::kBFloat16: return 1;
        case at::kHalf: return 2;
        default: return -1;
    }
}

constexpr int kEpiF16 = 5;

// A plain strided GPU tensor on `dev`, contiguous, its data 16-byte aligned.
bool plain(const at::Tensor& t, c10::Device dev) {
    return t.defined() && t.layout() == at::kStrided && t.device() == dev && !t.is_neg() && t.has_storage() &&
           t.is_contiguous() && reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0;
}

// None, or a tensor of exactly torch.Tensor / Parameter type; false for other objects
bool optional_tensor(PyObject* o, at::Tensor* t) {
    if (o == Py_None) return true;
    if (!THPVariable_CheckExact(o)) return false;
    *t = THPVariable_Unpack(o);
    return true;
}

struct Linear {
    at::Tensor x, w, scales, bias;
    int64_t M, N, K;
    int xdt, bdt, odt, epi;
};

// The operands common to the linears; K and N from the caller.  False: not a call for this path.
bool common(Linear& l, PyObject* ox, PyObject* os, PyObject* ob) {
    if (!THPVariable_CheckExact(ox) || !THPVariable_CheckExact(os)) return false;
    if (c10::impl::TorchDispatchModeTLS::any_modes_set()) return false;   // modes see the Python path's operations
    l.x = THPVariable_Unpack(ox);
    l.scales = THPVariable_Unpack(os);
    if (!l.x.is_cuda() || l.x.dim() < 1 || !optional_tensor(ob, &l.bias)) return false;
    const c10::Device dev = l.x.device();
    if (dev.index() != c10::hip::current_device() || !plain(l.x, dev) || !plain(l.scales, dev)) return false;
    l.xdt = dtype_code(l.x);
    l.K = l.x.size(-1);
    if (l.xdt < 0 || l.K <= 0 || l.x.numel() == 0 || l.scales.scalar_type() != at::kFloat) return false;
    const int64_t M = l.x.numel() / l.K;
    if (M > INT32_MAX) return false;
    l.M = M;
    l.bdt = 0;
    if (l.bias.defined()) {
        l.bdt = dtype_code(l.bias);
        if (l.bdt < 0 || !plain(l.bias, dev)) return false;
    }
    return true;
}

at::Tensor empty_out(const Linear& l) {
    std::vector<int64_t> sizes(l.x.sizes().begin(), l.x.sizes().end());
    sizes.back() = l.N;
    return at::empty(sizes, l.x.options().requires_grad(false));
}

int group_of(PyObject* o) {
    if (!PyLong_CheckExact(o)) return -1;
    const long g = PyLong_AsLong(o);
    if (g == -1 && PyErr_Occurred()) { PyErr_Clear(); return -1; }
    return g == 16 || g == 64 || g == 256 ? (int)g : -1;
}

const void* ptr(const at::Tensor& t) { return t.defined() ? t.const_data_ptr() : nullptr; }

PyObject* finish(int rc, const char* what, at::Tensor out) {
    if (rc != 0) {
        PyErr_Format(PyExc_RuntimeError, "%s failed, hipError=%d", what, rc);
        return nullptr;
    }
    return THPVariable_Wrap(std::move(out));
}

// w4a4(x, qweight, wscales, bias, groupsize, eager, lora, qweight_bf6)
PyObject* w4a4(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Linear l;
    if (n != 8 || !common(l, a[0], a[2], a[3]) || !THPVariable_CheckExact(a[1])) Py_RETURN_NONE;
    const c10::Device dev = l.x.device();
    const at::Tensor& qw = THPVariable_Unpack(a[1]);
    const int G = group_of(a[4]);
    if (G < 0 || l.K % G != 0 || qw.dim() != 2 || qw.size(1) * 2 != l.K || qw.size(0) < 1) Py_RETURN_NONE;
    l.N = qw.size(0);
    if (l.N > INT32_MAX || l.scales.numel() != l.N || (l.bias.defined() && l.bias.numel() != l.N)) Py_RETURN_NONE;
    const bool bf6 = l.K % 128 == 0 && l.K <= cr_max_quant_bf6_k();
    if (bf6) {
        if (!THPVariable_CheckExact(a[7])) Py_RETURN_NONE;
        l.w = THPVariable_Unpack(a[7]);
        if (!plain(l.w, dev) || l.w.scalar_type() != at::kByte || l.w.dim() != 2 || l.w.size(1) != l.K / 4 * 3 ||
            l.w.size(0) != (l.N + 255) / 256 * 256)
            Py_RETURN_NONE;
    } else {
        l.w = qw;
        if (l.K % 64 != 0 || l.K > cr_max_quant_k() || !plain(l.w, dev) || l.w.scalar_type() != at::kChar) Py_RETURN_NONE;
    }
    at::Tensor down, up;
    int R = 0;
    if (a[6] != Py_None) {
        if (!PyTuple_CheckExact(a[6]) || PyTuple_GET_SIZE(a[6]) != 2) Py_RETURN_NONE;
        PyObject *od = PyTuple_GET_ITEM(a[6], 0), *ou = PyTuple_GET_ITEM(a[6], 1);
        if (l.xdt == 0 || !THPVariable_CheckExact(od) || !THPVariable_CheckExact(ou)) Py_RETURN_NONE;
        down = THPVariable_Unpack(od);
        up = THPVariable_Unpack(ou);
        if (!plain(down, dev) || !plain(up, dev) || down.scalar_type() != at::kBFloat16 ||
            up.scalar_type() != at::kBFloat16 || down.dim() != 2 || up.dim() != 2 || down.size(1) != l.K ||
            up.size(0) != l.N || up.size(1) != down.size(0) || down.size(0) > 128 || down.size(0) < 32 ||
            down.size(0) % 32 != 0)
            Py_RETURN_NONE;
        R = (int)down.size(0);
    }
    const int M = (int)l.M, N = (int)l.N, K = (int)l.K;
    if (bf6 && cr_convrot_w4a4_linear_bf6_split(M, N, K)) Py_RETURN_NONE;
    const size_t ws_bytes = bf6 ? cr_convrot_w4a4_linear_bf6_min_workspace(M, N, K, R)
                                : cr_convrot_w4a4_linear_packed_workspace(M, N, K, R);
    const int epi = l.xdt == 1 ? (a[5] == Py_True ? 2 : 1) : 0;
    int rc;
    at::Tensor out;
    {
        pybind11::gil_scoped_release no_gil;
        out = empty_out(l);
        const at::Tensor ws = at::empty({(int64_t)ws_bytes}, l.x.options().dtype(at::kByte).requires_grad(false));
        void* st = c10::hip::getCurrentHIPStream(dev.index()).stream();
        if (bf6 && l.xdt == 2)
            rc = cr_convrot_w4a4_linear_bf6_f16(l.x.const_data_ptr(), l.xdt, l.w.const_data_ptr(), l.scales.const_data_ptr(),
                                                ptr(l.bias), l.bdt, ptr(down), ptr(up), R, 1.0f, out.mutable_data_ptr(), M, N,
                                                K, G, ws.mutable_data_ptr(), ws_bytes, st);
        else if (bf6)
            rc = cr_convrot_w4a4_linear_bf6(l.x.const_data_ptr(), l.xdt, l.w.const_data_ptr(), l.scales.const_data_ptr(),
                                            ptr(l.bias), l.bdt, ptr(down), ptr(up), R, 1.0f, out.mutable_data_ptr(), epi, M,
                                            N, K, G, ws.mutable_data_ptr(), ws_bytes, st);
        else
            rc = cr_convrot_w4a4_linear_packed(l.x.const_data_ptr(), l.xdt, l.w.const_data_ptr(), l.scales.const_data_ptr(),
                                               ptr(l.bias), l.bdt, ptr(down), ptr(up), R, 1.0f, out.mutable_data_ptr(),
                                               l.xdt == 2 ? kEpiF16 : epi, M, N, K, G, ws.mutable_data_ptr(), ws_bytes, st);
    }
    return finish(rc, "the W4A4 linear", std::move(out));
    END_HANDLE_TH_ERRORS
}

// w8a8(x, qweight, wscales, bias, groupsize, qweight_i8t)
PyObject* w8a8(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Linear l;
    if (n != 6 || !common(l, a[0], a[2], a[3]) || !THPVariable_CheckExact(a[1]) || !THPVariable_CheckExact(a[5]))
        Py_RETURN_NONE;
    const c10::Device dev = l.x.device();
    const at::Tensor& qw = THPVariable_Unpack(a[1]);
    l.w = THPVariable_Unpack(a[5]);
    const int G = group_of(a[4]);
    if (G < 0 || l.K % G != 0 || l.K % 64 != 0 || l.K > cr_max_quant_bf6_k() || qw.dim() != 2 || qw.size(1) != l.K ||
        qw.size(0) < 1)
        Py_RETURN_NONE;
    l.N = qw.size(0);
    if (l.N > INT32_MAX || l.scales.numel() != l.N || (l.bias.defined() && l.bias.numel() != l.N) || !plain(l.w, dev) ||
        l.w.scalar_type() != at::kChar || l.w.dim() != 2 || l.w.size(1) != l.K || l.w.size(0) != (l.N + 255) / 256 * 256)
        Py_RETURN_NONE;
    const int M = (int)l.M, N = (int)l.N, K = (int)l.K;
    if (cr_convrot_w8a8_linear_i8t_split(M, N, K)) Py_RETURN_NONE;
    const size_t ws_bytes = cr_convrot_w8a8_linear_i8t_workspace(M, N, K);
    int rc;
    at::Tensor out;
    {
        pybind11::gil_scoped_release no_gil;
        out = empty_out(l);
        const at::Tensor ws = at::empty({(int64_t)ws_bytes}, l.x.options().dtype(at::kByte).requires_grad(false));
        void* st = c10::hip::getCurrentHIPStream(dev.index()).stream();
        rc = cr_convrot_w8a8_linear_i8t(l.x.const_data_ptr(), l.xdt, l.w.const_data_ptr(),
                                        l.scales.const_data_ptr(), ptr(l.bias), l.bdt, out.mutable_data_ptr(),
                                        l.xdt == 2 ? kEpiF16 : l.xdt, M, N, K, G, ws.mutable_data_ptr(), ws_bytes, st);
    }
    return finish(rc, "the W8A8 linear", std::move(out));
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"w4a4", (PyCFunction)(void (*)(void))w4a4, METH_FASTCALL, nullptr},
    {"w8a8", (PyCFunction)(void (*)(void))w8a8, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// ABI_VERSION: of the library's signatures this module was compiled with.
PyMODINIT_FUNC PyInit__host(void) {
    PyObject* m = PyModule_Create(&module);
    if (m != nullptr && PyModule_AddIntConstant(m, "ABI_VERSION", CR_ABI_VERSION) != 0) Py_CLEAR(m);
    return m;
}
