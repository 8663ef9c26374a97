// Autograd of the dense evaluation in C++: gm.evaluate / gm.evaluate_inversed on plain device tensors, forward and backward
// without a line of Python between the caller and the launches (the backward pass runs on torch's engine thread without the
// interpreter lock).  Replaces nothing of the Python classes EvaluateInversed / EvaluateCovariance in
// gmc/cpp/extensions/evaluate_inversed/evaluate_inversed.py: what is not plain (see `plain`), and every input that
// `check_input` of gmc/_native.py would refuse, is left to them; `evaluate` returns None then.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/InferenceMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/autograd.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/version.h>

#include "gmc_hip.h"

namespace {

using at::Tensor;
using c10::DispatchKey;
using c10::DispatchKeySet;

void check(int code) { TORCH_CHECK(code == GMC_OK, "gmc_hip: ", gmc_error_string(code)); }

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.get_device()).stream(); }

// address of a tensor, null for an empty one
const void* address(const Tensor& t) { return t.numel() > 0 ? t.const_data_ptr() : nullptr; }
void* address_to_write(Tensor& t) { return t.numel() > 0 ? t.mutable_data_ptr() : nullptr; }

gmc_shape shape_of(const Tensor& mixture, const Tensor& xes) {
    return gmc_shape{int(mixture.size(0)), int(mixture.size(1)), int(mixture.size(2)), int(xes.size(2)), int(xes.size(3)),
                     int(xes.size(0)), int(xes.size(1)), mixture.scalar_type() == at::kFloat ? GMC_F32 : GMC_F64};
}

// Rules and messages of check_input and eval_bwd in gmc/_native.py, for the backward pass: a hook on saved tensors may hand
// back anything in their place.
void check_saved(const Tensor& mixture, const Tensor& xes, const Tensor& grad_out) {
    TORCH_CHECK(mixture.dim() == 4, "mixture must have 4 dimensions");
    TORCH_CHECK(mixture.size(3) == 7 || mixture.size(3) == 13, "mixture must have 7 or 13 elements in the last dimension");
    TORCH_CHECK(mixture.is_contiguous(), "mixture must be contiguous");
    TORCH_CHECK(xes.is_contiguous(), "xes must be contiguous");
    TORCH_CHECK(xes.dim() == 4, "xes must have 4 dimensions");
    TORCH_CHECK(xes.scalar_type() == mixture.scalar_type(), "mixture and xes must have the same dtype");
    TORCH_CHECK(xes.device() == mixture.device(), "mixture and xes must have the same device");
    TORCH_CHECK(mixture.scalar_type() == at::kFloat || mixture.scalar_type() == at::kDouble,
                "unsupported datatype: evaluate_inversed is implemented for float32 and float64");
    TORCH_CHECK(xes.size(0) == 1 || xes.size(0) == mixture.size(0), "xes must have a batch dimension equal to one or the mixture");
    TORCH_CHECK(xes.size(1) == 1 || xes.size(1) == mixture.size(1), "xes must have a layer dimension equal to one or the mixture");
    TORCH_CHECK(xes.size(3) == (mixture.size(3) == 7 ? 2 : 3),
                "xes must have the last dimension equal to the number of dimensions of the mixture");
    TORCH_CHECK(mixture.is_cuda(), "gmc_hip evaluates on an AMD GPU only: mixture and xes must be HIP ('cuda') tensors; "
                                   "this build has no CPU implementation");
    for (int i = 0; i < 3; ++i)
        TORCH_CHECK(mixture.size(i) <= INT_MAX && xes.size(i) <= INT_MAX, "gmc_hip: ", gmc_error_string(GMC_E_SHAPE));
    TORCH_CHECK(grad_out.dim() == 3, "grad_output has wrong number of dimensions");
    TORCH_CHECK(grad_out.size(0) == mixture.size(0), "grad_output has wrong batch dimension");
    TORCH_CHECK(grad_out.size(1) == mixture.size(1), "grad_output has wrong layer dimension");
    TORCH_CHECK(grad_out.size(2) == xes.size(2), "grad_output has wrong xes dimension");
    TORCH_CHECK(grad_out.scalar_type() == mixture.scalar_type(), "grad_output dtype does not match with mixture dtype");
    TORCH_CHECK(grad_out.device() == mixture.device(), "grad_output must live on the device of the mixture");
}

Tensor forward(const Tensor& mixture, const Tensor& xes, bool covariance_form) {
    const gmc_shape s = shape_of(mixture, xes);
    const c10::DeviceGuard guard(mixture.device());
    Tensor out = at::empty({s.B, s.L, s.N}, mixture.options().requires_grad(false));
    check((covariance_form ? gmc_eval_cov_fwd : gmc_eval_fwd)(address(mixture), address(xes), address_to_write(out), &s, stream_of(mixture)));
    return out;
}

template <bool COVARIANCE>
struct Evaluate : public torch::autograd::Function<Evaluate<COVARIANCE>> {
    static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& mixture, const Tensor& xes) {
        const Tensor m = mixture.contiguous(), x = xes.contiguous();
        ctx->save_for_backward({m, x});
        return ::forward(m, x, COVARIANCE);
    }

    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const bool want_mixture = ctx->needs_input_grad(0), want_xes = ctx->needs_input_grad(1);
        torch::autograd::variable_list result(2);
        {
            const at::AutoGradMode off(false);
            const Tensor mixture = saved[0].detach(), xes = saved[1].detach(), grad_out = grads[0].detach().contiguous();
            check_saved(mixture, xes, grad_out);
            const gmc_shape s = shape_of(mixture, xes);
            const c10::DeviceGuard guard(mixture.device());
            if (want_mixture) result[0] = at::empty_like(mixture);
            if (want_xes) result[1] = at::empty_like(xes);
            const size_t bytes = want_mixture ? gmc_eval_bwd_workspace_bytes(&s) : 0;
            Tensor workspace;
            if (bytes > 0) workspace = at::empty({int64_t((bytes + 7) / 8)}, mixture.options().dtype(at::kDouble));
            if (want_mixture || want_xes)
                check((COVARIANCE ? gmc_eval_cov_bwd : gmc_eval_bwd)(
                    address(grad_out), address(mixture), address(xes), want_mixture ? address_to_write(result[0]) : nullptr,
                    want_xes ? address_to_write(result[1]) : nullptr, bytes > 0 ? workspace.mutable_data_ptr() : nullptr, bytes,
                    &s, want_mixture, want_xes, stream_of(mixture)));
        }
        // no second derivatives: what torch.autograd.function.once_differentiable does
        if (at::GradMode::is_enabled() && grads[0].requires_grad()) {
            torch::autograd::variable_list outputs;
            for (auto& r : result) outputs.push_back(r.defined() ? r.detach().requires_grad_(true) : r);
            const auto error = std::make_shared<torch::autograd::DelayedError>(
                "trying to differentiate twice a function that was marked with @once_differentiable", outputs.size());
            return (*error)(std::move(outputs));
        }
        return result;
    }
};

// Ordinary device tensors: no subclass, wrapper of a transformation (vmap, grad, functionalisation), lazy view or tangent of
// forward-mode differentiation.
bool plain(PyObject* object) {
    if (!THPVariable_CheckExact(object)) return false;
    const Tensor& t = THPVariable_Unpack(object);
    const DispatchKeySet ordinary =
        DispatchKeySet({DispatchKey::CUDA, DispatchKey::AutogradCUDA, DispatchKey::ADInplaceOrView}) | c10::autocast_dispatch_keyset;
    return t.defined() && (t.key_set() | ordinary) == ordinary && !t._fw_grad(0).defined();
}

// No mode, transformation or tracer wants to see the call.
bool undisturbed() {
    const auto keys = c10::impl::tls_local_dispatch_key_set();
    const DispatchKeySet usual = c10::default_included_set | c10::autocast_dispatch_keyset;
    return (keys.included_ | usual) == usual && !at::impl::torch_function_mode_enabled() && !torch::jit::tracer::isTracing() &&
           !c10::InferenceMode::is_enabled();
}

bool accepted(const Tensor& mixture, const Tensor& xes) {
    if (mixture.dim() != 4 || xes.dim() != 4 || mixture.device() != xes.device() || mixture.scalar_type() != xes.scalar_type()) return false;
    if (mixture.scalar_type() != at::kFloat && mixture.scalar_type() != at::kDouble) return false;
    const int64_t d = mixture.size(3) == 7 ? 2 : mixture.size(3) == 13 ? 3 : 0;
    for (int i = 0; i < 4; ++i)
        if (mixture.size(i) > INT_MAX || xes.size(i) > INT_MAX) return false;
    return d != 0 && xes.size(3) == d && (xes.size(0) == 1 || xes.size(0) == mixture.size(0)) &&
           (xes.size(1) == 1 || xes.size(1) == mixture.size(1));
}

// evaluate(mixture, xes, covariance_form) -> values, or None where the Python classes have to do it
PyObject* evaluate(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 3 || !plain(args[0]) || !plain(args[1]) || !undisturbed()) Py_RETURN_NONE;
    const Tensor& mixture = THPVariable_Unpack(args[0]);
    const Tensor& xes = THPVariable_Unpack(args[1]);
    if (!accepted(mixture, xes)) Py_RETURN_NONE;
    const bool covariance_form = args[2] == Py_True;
    Tensor out;
    {
        pybind11::gil_scoped_release released;
        if (at::GradMode::is_enabled() && (mixture.requires_grad() || xes.requires_grad()))
            out = covariance_form ? Evaluate<true>::apply(mixture, xes) : Evaluate<false>::apply(mixture, xes);
        else
            out = forward(mixture.contiguous(), xes.contiguous(), covariance_form);
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// versions() -> ABI version of the header this file was built from, of the library it is linked to, version of torch's headers
PyObject* versions(PyObject*, PyObject*) { return Py_BuildValue("iis", GMC_ABI_VERSION, gmc_abi_version(), TORCH_VERSION); }

PyMethodDef methods[] = {
    {"evaluate", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(evaluate)), METH_FASTCALL,
     "evaluate(mixture, xes, covariance_form) -> values, or None for what is not a plain device tensor or not accepted"},
    {"versions", versions, METH_NOARGS, "versions() -> (ABI version of the header, of the library, version of torch's headers)"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_gmc_autograd", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__gmc_autograd() { return PyModule_Create(&module); }
