// What the native host side's two parts share: checks, the stream, views of rows.  Host code only.
#pragma once
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/SavedTensorHooks.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/variable.h>

#include "../../include/bgemm_mi355x.h"

namespace bgemm_native {

using at::Tensor;

// The module's functions as _lib.py knows them (NATIVE_VERSION there): another number when one is added or called another way.
constexpr long NATIVE_VERSION = 2;

// Turns a negative status into the exception _lib.check() raises.
inline void check(const int rc)
{
    if (rc == BGEMM_OK) return;
    const std::string msg = bgemm_last_error();
    if (rc == BGEMM_EINVAL || rc == BGEMM_ENULL || rc == BGEMM_EALIGN || rc == BGEMM_EWORKSPACE) TORCH_CHECK_VALUE(false, msg);
    TORCH_CHECK(false, msg);
}

inline void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
inline bool is_param_type(const at::ScalarType t) { return t == at::kFloat || t == at::kHalf; }
inline int src_type(const Tensor& t) { return t.scalar_type() == at::kFloat ? BGEMM_SRC_F32 : BGEMM_SRC_F16; }
inline void* data_or_null(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
inline const Tensor& tensor_at(PyObject* o) { return THPVariable_Unpack(o); }
inline Tensor tensor_or_none(PyObject* o) { return o == Py_None ? Tensor() : THPVariable_Unpack(o); }

// Whether a tensor is memory on the GPU and nothing else: no transform's wrapper, no subclass with a dispatch of its own (fake tensors
// among them), no view that is negated or conjugated when read, no sparse or quantised layout.
inline bool is_memory(const Tensor& t)
{
    using c10::DispatchKey;
    static const uint64_t usual = c10::DispatchKeySet({DispatchKey::Dense, DispatchKey::AutogradFunctionality, DispatchKey::ADInplaceOrView,
                                                       DispatchKey::AutocastCUDA}).raw_repr() | c10::full_backend_mask;
    return (t.key_set().raw_repr() & ~usual) == 0;
}

// Whether something else has to see each torch operation: a mode, a trace, a function transform.
inline bool is_watched()
{
    using c10::DispatchKey;
    static const uint64_t usual = c10::DispatchKeySet({DispatchKey::BackendSelect, DispatchKey::ADInplaceOrView, DispatchKey::AutocastCUDA,
                                                       DispatchKey::AutocastCPU}).raw_repr() | c10::full_backend_mask;
    return (c10::impl::tls_local_dispatch_key_set().included_.raw_repr() & ~usual) != 0 || at::impl::torch_function_mode_enabled();
}

// Forward-mode derivatives are torch's business: the kernels know none.
inline bool has_tangent(const Tensor& t) { return t.defined() && t._fw_grad(/*level=*/0).defined(); }

// Kernels are enqueued and memory is allocated without the interpreter's lock.
struct WithoutGil {
    PyThreadState* state = PyEval_SaveThread();
    ~WithoutGil() { PyEval_RestoreThread(state); }
};

// [..., C] as rows [R, C] whose elements are dense, and their stride (C or more: a single row's own stride means nothing and may be
// anything, also after contiguous()).
struct Rows { Tensor t; int64_t ld; };

inline Rows rows_2d(const Tensor& t)
{
    const int64_t C = t.size(-1);
    Tensor r = t.dim() == 2 ? t : t.reshape({t.numel() / C, C});
    if (r.size(0) == 1) return {r.stride(1) == 1 || C == 1 ? r : r.contiguous(), C};
    if (r.stride(1) != 1 || r.stride(0) < C) r = r.contiguous();
    return {r, r.stride(0)};
}

// x [.., N, K] @ right [.., K, M] of binarised operands, one launch over the batch -> fp16 [.., N, M]; undefined: a form it does not take.
Tensor batched_product_of(const Tensor& x, const Tensor& right, int mode);
// The gradients of such a product by their one-launch kernel (bgemm_linear._one_launch_grads and, above `narrow` columns, fewer than `most`
// multiplications a product: _scores_grad_ahead); false: a form it does not take.
bool attention_grads(bool context, const Tensor& m, const Tensor& a, const Tensor& b, bool need0, bool need1, int64_t longest, int64_t narrow, int64_t most,
                     Tensor& g0, Tensor& g1);

// Functions of the inference and attention part, for the module's table.
extern PyMethodDef infer_methods[];
extern const int infer_method_count;

}  // namespace bgemm_native
