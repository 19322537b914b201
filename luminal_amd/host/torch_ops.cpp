// The host path of QuantizedMatmul and QuantizedMatmulBf16 (luminal_amd/quantized.py) in one native call: the output's allocation, the
// workspace's where the shape wants one, and the launch through the C ABI.
//
// Replaces what the reference's process() does in Rust around its launch (crates/luminal_cuda/src/quantized.rs:116-168).  A call of
// the operators from Python is bound by the host where the kernel takes a few microseconds: of 7.3 us for one row through a
// 1024 x 4096 weight the kernel takes 2.5 and hipLaunchKernel 2.7; the rest was torch.empty's and ctypes' argument handling and
// the interpreter's work between them.  With this 7.4 -> 4.5 us a call among others, 27 -> 19 us for a first call that is waited for.
//
// The plain case only: plain contiguous tensors on the current device whose shapes agree.  Everything else, errors included, gives
// None, and the caller's Python path takes it as it always did.
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Exceptions.h>
#include <ATen/ops/empty.h>

#include "../../include/luminal_hip.h"

namespace {

// quantized_matmul(x, planar, n, k, bf16, device, stream) -> y or None; x is bf16, or f32 or f16.  The workspace rules are quantized.py's rows_workspace_nbytes and
// bf16_workspace_nbytes.
PyObject *quantized_matmul(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 7 || !THPVariable_CheckExact(args[0]) || !THPVariable_CheckExact(args[1])) Py_RETURN_NONE;
    const at::Tensor &x = THPVariable_Unpack(args[0]);
    const at::Tensor &planar = THPVariable_Unpack(args[1]);
    const int64_t n = PyLong_AsLongLong(args[2]), k = PyLong_AsLongLong(args[3]), device = PyLong_AsLongLong(args[5]);
    const bool bf16 = args[4] == Py_True;
    void *stream = PyLong_AsVoidPtr(args[6]);
    if (PyErr_Occurred()) return nullptr;
    const auto dtype = x.scalar_type();
    const bool f16 = dtype == at::kHalf;
    if (!(bf16 ? dtype == at::kBFloat16 : f16 || dtype == at::kFloat) || !x.is_cuda() || x.device().index() != device || planar.device() != x.device() ||
        !x.has_storage() || !planar.has_storage() || x.layout() != at::kStrided || x.dim() < 1 || x.dim() > 8 || n <= 0 || k <= 0 ||
        x.size(-1) != k || x.numel() == 0 || !x.is_contiguous())
        Py_RETURN_NONE;
    const int64_t m = x.numel() / k;
    at::Tensor y, space;
    lhip_status st;
    {
        pybind11::gil_scoped_release no_gil;
        c10::SmallVector<int64_t, 8> sizes(x.sizes().begin(), x.sizes().end());
        sizes.back() = n;
        y = at::empty(sizes, x.options());
        size_t need = 0;
        if (bf16 ? m > 128 || k % 512 != 0 : m > 64 || (m > 1 && (k % 512 != 0 || n % 4 != 0)))
            need = bf16 ? lhip_q8_0_matmul_bf16_workspace_nbytes(m, n, k, LHIP_GEMM_OUT_BF16) : lhip_q8_0_matmul_workspace_nbytes(m, n, k);
        if (need) space = at::empty({static_cast<int64_t>(need)}, x.options().dtype(at::kByte));
        const void *w = planar.const_data_ptr(), *in = x.const_data_ptr();
        void *out = y.mutable_data_ptr(), *ws = need ? space.mutable_data_ptr() : nullptr;
        if (bf16)
            st = need ? lhip_q8_0_matmul_bf16_ws(w, in, out, m, n, k, LHIP_GEMM_OUT_BF16, ws, need, stream)
                      : lhip_q8_0_matmul_bf16(w, in, out, m, n, k, stream);
        else if (f16)
            st = need ? lhip_q8_0_matmul_f16_ws(w, in, out, m, n, k, ws, need, stream) : lhip_q8_0_matmul_f16(w, in, out, m, n, k, stream);
        else
            st = need ? lhip_q8_0_matmul_f32_ws(w, static_cast<const float *>(in), static_cast<float *>(out), m, n, k, ws, need, stream)
                      : lhip_q8_0_matmul_f32(w, static_cast<const float *>(in), static_cast<float *>(out), m, n, k, stream);
    }
    if (st != LHIP_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"quantized_matmul", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(quantized_matmul)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_torch_ops", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// What it was built for, which quantized.py compares with what runs: at::Tensor's layout goes with the one, the C ABI's signatures with
// the other.  (The file's name goes with the Python.)
PyMODINIT_FUNC PyInit__torch_ops() {
    PyObject *module = PyModule_Create(&module_def);
    if (module && (PyModule_AddStringConstant(module, "torch_version", LHIP_TORCH_VERSION) || PyModule_AddStringConstant(module, "c_header", LHIP_C_HEADER))) {
        Py_DECREF(module);
        return nullptr;
    }
    return module;
}
