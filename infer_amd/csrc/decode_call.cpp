// The call of decode attention on torch tensors, as a Python extension module (infer_amd/_decode_call.so).
//
// A decode call of a few short sequences takes the GPU 8 us, and Python 9 to look at the tensors in front of two launches: decode(...) looks at them
// here.  It takes what is plain and complete and returns the result; for everything else, whatever the reason, it returns None and has done
// nothing, and the caller takes the general way, which raises what there is to raise.
//
// The workspace is the one that infer_amd.ops shares among the calls of a shape; ops says here which one and on which stream it was used
// last (claim), and a call on another stream is left to ops, which checks that the last one has ended.  All entries hold the interpreter's lock.
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include <array>
#include <map>

#include "infer_kv.h"

namespace {

struct Claim {
    void* workspace;
    size_t bytes;
    void* stream;
};
std::map<std::array<int64_t, 3>, Claim>& claims() {       // (device, query heads, KV heads); head_dim is 128 throughout
    static auto* all = new std::map<std::array<int64_t, 3>, Claim>();
    return *all;
}

// claim(device, query heads, KV heads, address, bytes, stream)
PyObject* claim(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 6) return PyErr_Format(PyExc_TypeError, "claim takes 6 numbers");
    unsigned long long v[6];
    for (int i = 0; i < 6; ++i) {
        v[i] = PyLong_AsUnsignedLongLong(args[i]);
        if (PyErr_Occurred()) return nullptr;
    }
    claims()[{(int64_t)v[0], (int64_t)v[1], (int64_t)v[2]}] = Claim{(void*)v[3], (size_t)v[4], (void*)v[5]};
    Py_RETURN_NONE;
}

// A tensor that is its memory and nothing else, on a GPU
const at::Tensor* plain(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    const auto keys = t.key_set();
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.is_nested() || t.is_neg() || t.is_conj() || keys.has(c10::DispatchKey::Python) ||
        keys.has(c10::DispatchKey::FuncTorchBatched) || keys.has(c10::DispatchKey::FuncTorchGradWrapper) || keys.has(c10::DispatchKey::Functionalize) ||
        !t.has_storage())
        return nullptr;
    return &t;
}

// decode(q [B, 1, Hq, D], k_cache, v_cache [blocks, block, Hkv, D], lengths [B], block_table [B, columns], scale) -> [B, 1, Hq, D] or None
PyObject* decode(PyObject*, PyObject* const* args, Py_ssize_t n) try {
    if (n != 6) return PyErr_Format(PyExc_TypeError, "decode takes 6 arguments");
    const at::Tensor *q = plain(args[0]), *k = plain(args[1]), *v = plain(args[2]), *lens = plain(args[3]), *table = plain(args[4]);
    if (!q || !k || !v || !lens || !table || !(PyFloat_CheckExact(args[5]) || args[5] == Py_None)) Py_RETURN_NONE;
    if (at::impl::torch_function_mode_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set() || torch::jit::tracer::isTracing()) Py_RETURN_NONE;
    if (q->scalar_type() != at::kBFloat16 || k->scalar_type() != at::kBFloat16 || v->scalar_type() != at::kBFloat16 || lens->scalar_type() != at::kInt ||
        table->scalar_type() != at::kInt)
        Py_RETURN_NONE;
    if (q->dim() != 4 || k->dim() != 4 || k->sizes() != v->sizes() || k->strides() != v->strides() || table->dim() != 2) Py_RETURN_NONE;
    const int64_t b = q->size(0), hq = q->size(2), d = q->size(3), hkv = k->size(2);
    if (q->size(1) != 1 || d != 128 || q->stride(3) != 1 || q->stride(2) != d || k->size(3) != d || k->stride(3) != 1 || k->stride(2) != d) Py_RETURN_NONE;
    if (lens->numel() != b || !lens->is_contiguous() || table->size(0) != b || table->size(1) < 1 || table->stride(1) != 1) Py_RETURN_NONE;
    const auto device = q->get_device();
    if (k->get_device() != device || v->get_device() != device || lens->get_device() != device || table->get_device() != device) Py_RETURN_NONE;
    const auto found = claims().find({device, hq, hkv});
    if (found == claims().end()) Py_RETURN_NONE;
    if (c10::hip::current_device() != device) Py_RETURN_NONE;
    void* stream = c10::hip::getCurrentHIPStream(device).stream();
    if (stream != found->second.stream) Py_RETURN_NONE;
    const double scale = args[5] == Py_None ? 1.0 / std::sqrt((double)d) : PyFloat_AS_DOUBLE(args[5]);
    at::Tensor out = at::empty({b, 1, hq, d}, q->options().requires_grad(false));
    if (!out.is_cuda() || out.scalar_type() != at::kBFloat16) Py_RETURN_NONE;
    const int rc = infer_paged_decode_bf16(q->data_ptr(), q->stride(0), k->data_ptr(), v->data_ptr(), k->stride(0), k->stride(1), out.data_ptr(), hq * d,
                                           (const int32_t*)table->data_ptr(), table->stride(0), table->size(1), (const int32_t*)lens->data_ptr(), b, hq,
                                           hkv, d, k->size(1), k->size(0), (float)scale, 0, found->second.workspace, found->second.bytes, stream);
    if (rc != 0) Py_RETURN_NONE;
    return THPVariable_Wrap(out);
} catch (...) {
    Py_RETURN_NONE;      // the general way meets the same and says it
}

PyMethodDef methods[] = {
    {"claim", (PyCFunction)(void (*)(void))claim, METH_FASTCALL, "the workspace of a shape and the stream that used it last"},
    {"decode", (PyCFunction)(void (*)(void))decode, METH_FASTCALL, "decode attention of plain tensors, or None"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_decode_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__decode_call(void) { return PyModule_Create(&module); }
