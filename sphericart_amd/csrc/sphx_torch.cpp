// The torch operators' device implementations in C++: libsphericart_amd_torch.so, loaded with
// torch.ops.load_library. Host code only (no kernel): it defines the schemas of the `sphericart_amd` namespace and
// implements them for tensors on the GPU by calling the C entry points of libsphericart_amd.so on the tensor's
// current stream, as the reference's extension does with its calculators
// (sphericart-torch/src/torch.cpp:237-294 _compute_raw_cuda, :367-385 TORCH_LIBRARY). Autograd of GPU tensors is here
// too; its rules in Python (sphericart_amd/torch/ops.py, the reference's register.py:82-185) serve the operators
// implemented in Python and tensors without a device, as do the fake-tensor and vmap rules. A call through these costs
// the host the dispatcher, the allocation of its outputs and one C call; the same operators implemented in Python over
// ctypes, which ops.py registers when this library has not been built, cost about twice that.
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/library.h>

#include <ATen/core/LegacyTypeDispatch.h>
#include <ATen/core/dispatch/Dispatcher.h>

#include <memory>
#include <optional>
#include <string>
#include <tuple>

#include "../../include/sphx_launch.h"

namespace {

using at::Tensor;

void check(int status) {
    TORCH_CHECK(status == SPHX_OK, sphx_last_error());
}

bool is_double(const Tensor& tensor, const char* what) {
    TORCH_CHECK_TYPE(tensor.scalar_type() == at::kFloat || tensor.scalar_type() == at::kDouble, what,
                     " are implemented for float32 and float64, not ", tensor.scalar_type());
    return tensor.scalar_type() == at::kDouble;
}

// an empty tensor's pointer may be anything: the library takes null for "no array"
template <typename T> T* pointer(const Tensor& tensor) {
    return tensor.defined() && tensor.numel() > 0 ? tensor.data_ptr<T>() : nullptr;
}

void* stream_of(const Tensor& tensor) {
    return c10::hip::getCurrentHIPStream(tensor.device().index()).stream();
}

// compute_raw / _compute_raw_cuda (sphericart-torch/src/torch.cpp:126-146, 238-294)
std::tuple<Tensor, Tensor, Tensor> forward(const Tensor& xyz_in, int64_t l_max, bool normalized, int mode) {
    TORCH_CHECK_VALUE(xyz_in.dim() == 2 && xyz_in.size(1) == 3,
                      "xyz tensor must be a 2D array with shape `n_samples x 3`");
    TORCH_CHECK_VALUE(l_max >= 0, "l_max must be non-negative");
    const bool f64 = is_double(xyz_in, "spherical harmonics");
    const Tensor xyz = xyz_in.detach().contiguous();
    const int64_t n = xyz.size(0), ny = (l_max + 1) * (l_max + 1);
    const auto options = xyz.options();
    Tensor sph = at::empty({n, ny}, options), dsph, ddsph;
    if (mode >= 1) dsph = at::empty({n, 3, ny}, options);
    if (mode >= 2) ddsph = at::empty({n, 3, 3, ny}, options);
    const c10::DeviceGuard guard(xyz.device());
    if (f64) {
        check(sphx_forward_f64(pointer<double>(xyz), static_cast<size_t>(n), static_cast<int>(l_max), normalized, mode,
                               pointer<double>(sph), pointer<double>(dsph), pointer<double>(ddsph), stream_of(xyz)));
    } else {
        check(sphx_forward_f32(pointer<float>(xyz), static_cast<size_t>(n), static_cast<int>(l_max), normalized, mode,
                               pointer<float>(sph), pointer<float>(dsph), pointer<float>(ddsph), stream_of(xyz)));
    }
    return {sph, dsph, ddsph};
}

template <bool NORMALIZED> Tensor values(const Tensor& xyz, int64_t l_max) {
    return std::get<0>(forward(xyz, l_max, NORMALIZED, SPHX_VALUES));
}
template <bool NORMALIZED> std::tuple<Tensor, Tensor> with_gradients(const Tensor& xyz, int64_t l_max) {
    auto all = forward(xyz, l_max, NORMALIZED, SPHX_GRADIENTS);
    return {std::get<0>(all), std::get<1>(all)};
}
template <bool NORMALIZED> std::tuple<Tensor, Tensor, Tensor> with_hessians(const Tensor& xyz, int64_t l_max) {
    return forward(xyz, l_max, NORMALIZED, 2);
}

// What the operators below share: points [n, 3], and weights of a given shape and the points' dtype on their device.
void check_points(const Tensor& xyz, int64_t l_max) {
    TORCH_CHECK_VALUE(xyz.dim() == 2 && xyz.size(1) == 3, "xyz tensor must be a 2D array with shape `n_samples x 3`");
    TORCH_CHECK_VALUE(l_max >= 0, "l_max must be non-negative");
}
void check_weights(const Tensor& xyz, const Tensor& weights, at::IntArrayRef shape, const char* what) {
    TORCH_CHECK_VALUE(weights.scalar_type() == xyz.scalar_type() && weights.device() == xyz.device(), "xyz and ", what,
                      " must share dtype and device");
    TORCH_CHECK_VALUE(weights.sizes() == shape, what, " must have shape ", shape);
}

// the product of the gradients with sph_grad without the gradient array (sphx_vjp_*)
template <bool NORMALIZED> Tensor vjp(const Tensor& xyz_in, const Tensor& sph_grad_in, int64_t l_max) {
    const bool f64 = is_double(xyz_in, "spherical harmonics");
    check_points(xyz_in, l_max);
    check_weights(xyz_in, sph_grad_in, {xyz_in.size(0), (l_max + 1) * (l_max + 1)}, "sph_grad");
    const Tensor xyz = xyz_in.detach().contiguous(), sph_grad = sph_grad_in.detach().contiguous();
    Tensor out = at::empty_like(xyz);
    const c10::DeviceGuard guard(xyz.device());
    if (f64) {
        check(sphx_vjp_f64(pointer<double>(xyz), pointer<double>(sph_grad), static_cast<size_t>(xyz.size(0)),
                           static_cast<int>(l_max), NORMALIZED, pointer<double>(out), 0, stream_of(xyz)));
    } else {
        check(sphx_vjp_f32(pointer<float>(xyz), pointer<float>(sph_grad), static_cast<size_t>(xyz.size(0)),
                           static_cast<int>(l_max), NORMALIZED, pointer<float>(out), 0, stream_of(xyz)));
    }
    return out;
}

// xyz_grad = sum_k derivatives * upstream over the last axis (and, one order up, over the axis before the
// last but one as well): sphx_backward_* / sphx_backward_second_*
template <bool SECOND> Tensor contract(const Tensor& derivatives_in, const Tensor& upstream_in) {
    const bool f64 = is_double(derivatives_in, "contractions");
    TORCH_CHECK_VALUE(upstream_in.scalar_type() == derivatives_in.scalar_type() &&
                          upstream_in.device() == derivatives_in.device(),
                      "the two tensors of a contraction must share dtype and device");
    // dsph [n, 3, k] with sph_grad [n, k]; ddsph [n, 3, 3, k] with dsph_grad [n, 3, k]
    bool fit = derivatives_in.dim() == (SECOND ? 4 : 3) && upstream_in.dim() == derivatives_in.dim() - 1 &&
               derivatives_in.size(1) == 3;
    for (int64_t axis = 0; fit && axis < upstream_in.dim(); ++axis) {
        fit = upstream_in.size(axis) == derivatives_in.size(axis == 0 ? 0 : axis + 1);
    }
    TORCH_CHECK_VALUE(fit, "shapes ", derivatives_in.sizes(), " and ", upstream_in.sizes(), " do not contract");
    const Tensor derivatives = derivatives_in.detach().contiguous(), upstream = upstream_in.detach().contiguous();
    const int64_t n = derivatives.size(0), n_total = derivatives.size(-1);
    Tensor out = at::empty({n, 3}, derivatives.options());
    const c10::DeviceGuard guard(derivatives.device());
    void* stream = stream_of(derivatives);
    int status;
    if (f64) {
        auto* entry = SECOND ? sphx_backward_second_f64 : sphx_backward_f64;
        status = entry(pointer<double>(derivatives), pointer<double>(upstream), static_cast<size_t>(n),
                       static_cast<int>(n_total), pointer<double>(out), 0, stream);
    } else {
        auto* entry = SECOND ? sphx_backward_second_f32 : sphx_backward_f32;
        status = entry(pointer<float>(derivatives), pointer<float>(upstream), static_cast<size_t>(n),
                       static_cast<int>(n_total), pointer<float>(out), 0, stream);
    }
    check(status);
    return out;
}

// The derivatives of vjp with the upstream gradient `grad` [n, 3]: with respect to xyz and to sph_grad
// (sphx_vjp_backward_*; from the derivative arrays where that does not reach).
template <bool NORMALIZED>
std::tuple<Tensor, Tensor> vjp_backward(const Tensor& xyz_in, const Tensor& sph_grad_in, const Tensor& grad_in, int64_t l_max) {
    const bool f64 = is_double(xyz_in, "spherical harmonics");
    check_points(xyz_in, l_max);
    const int64_t n = xyz_in.size(0), ny = (l_max + 1) * (l_max + 1);
    check_weights(xyz_in, sph_grad_in, {n, ny}, "sph_grad");
    check_weights(xyz_in, grad_in, {n, 3}, "grad");
    const Tensor xyz = xyz_in.detach().contiguous(), sph_grad = sph_grad_in.detach().contiguous(), grad = grad_in.detach().contiguous();
    Tensor xyz_grad = at::empty_like(xyz), sph_grad_grad = at::empty_like(sph_grad);
    const c10::DeviceGuard guard(xyz.device());
    const size_t count = static_cast<size_t>(n);
    const int order = static_cast<int>(l_max);
    const int status =
        f64 ? sphx_vjp_backward_f64(pointer<double>(xyz), pointer<double>(sph_grad), pointer<double>(grad), count, order, NORMALIZED,
                                    pointer<double>(xyz_grad), pointer<double>(sph_grad_grad), stream_of(xyz))
            : sphx_vjp_backward_f32(pointer<float>(xyz), pointer<float>(sph_grad), pointer<float>(grad), count, order, NORMALIZED,
                                    pointer<float>(xyz_grad), pointer<float>(sph_grad_grad), stream_of(xyz));
    if (status == SPHX_ERR_UNSUPPORTED) {
        const auto all = forward(xyz, l_max, NORMALIZED, 2);
        return {contract<true>(std::get<2>(all), grad.unsqueeze(2) * sph_grad.unsqueeze(1)),
                (grad.unsqueeze(2) * std::get<1>(all)).sum(1)};
    }
    check(status);
    return {xyz_grad, sph_grad_grad};
}

// The backward pass of values and gradients (sphx_gradients_backward_*; from the derivative arrays where that does
// not reach). sph_grad may be missing.
template <bool NORMALIZED>
Tensor gradients_backward(const Tensor& xyz_in, const std::optional<Tensor>& sph_grad_in, const Tensor& dsph_grad_in, int64_t l_max) {
    const bool f64 = is_double(xyz_in, "spherical harmonics");
    check_points(xyz_in, l_max);
    const int64_t n = xyz_in.size(0), ny = (l_max + 1) * (l_max + 1);
    check_weights(xyz_in, dsph_grad_in, {n, 3, ny}, "dsph_grad");
    if (sph_grad_in.has_value()) check_weights(xyz_in, *sph_grad_in, {n, ny}, "sph_grad");
    const Tensor xyz = xyz_in.detach().contiguous(), dsph_grad = dsph_grad_in.detach().contiguous();
    Tensor sph_grad;
    if (sph_grad_in.has_value()) sph_grad = sph_grad_in->detach().contiguous();
    Tensor xyz_grad = at::empty_like(xyz);
    const c10::DeviceGuard guard(xyz.device());
    const size_t count = static_cast<size_t>(n);
    const int order = static_cast<int>(l_max);
    const int status =
        f64 ? sphx_gradients_backward_f64(pointer<double>(xyz), pointer<double>(sph_grad), pointer<double>(dsph_grad), count, order,
                                          NORMALIZED, pointer<double>(xyz_grad), stream_of(xyz))
            : sphx_gradients_backward_f32(pointer<float>(xyz), pointer<float>(sph_grad), pointer<float>(dsph_grad), count, order,
                                          NORMALIZED, pointer<float>(xyz_grad), stream_of(xyz));
    if (status == SPHX_ERR_UNSUPPORTED) {
        const auto all = forward(xyz, l_max, NORMALIZED, 2);
        Tensor sum = contract<true>(std::get<2>(all), dsph_grad);
        return sph_grad.defined() ? sum + contract<false>(std::get<1>(all), sph_grad) : sum;
    }
    check(status);
    return xyz_grad;
}

[[noreturn]] void no_cpu() {
    TORCH_CHECK(false, "sphericart_amd evaluates on AMD GPUs only: move the tensor to the device "
                       "(there is no CPU implementation behind these operators)");
}
Tensor cpu_values(const Tensor&, int64_t) { no_cpu(); }
std::tuple<Tensor, Tensor> cpu_with_gradients(const Tensor&, int64_t) { no_cpu(); }
std::tuple<Tensor, Tensor, Tensor> cpu_with_hessians(const Tensor&, int64_t) { no_cpu(); }
Tensor cpu_vjp(const Tensor&, const Tensor&, int64_t) { no_cpu(); }
Tensor cpu_contract(const Tensor&, const Tensor&) { no_cpu(); }
std::tuple<Tensor, Tensor> cpu_vjp_backward(const Tensor&, const Tensor&, const Tensor&, int64_t) { no_cpu(); }
Tensor cpu_gradients_backward(const Tensor&, const std::optional<Tensor>&, const Tensor&, int64_t) { no_cpu(); }

} // namespace

// the reference's six schemas (torch.cpp:367-374) and, without counterpart there, the fused products
TORCH_LIBRARY(sphericart_amd, m) {
    for (const char* prefix : {"spherical_harmonics", "solid_harmonics"}) {
        const std::string name(prefix);
        m.def((name + "(Tensor xyz, int l_max) -> Tensor").c_str());
        m.def((name + "_with_gradients(Tensor xyz, int l_max) -> (Tensor, Tensor)").c_str());
        m.def((name + "_with_hessians(Tensor xyz, int l_max) -> (Tensor, Tensor, Tensor)").c_str());
        m.def((name + "_vjp(Tensor xyz, Tensor sph_grad, int l_max) -> Tensor").c_str());
        m.def((name + "_vjp_backward(Tensor xyz, Tensor sph_grad, Tensor grad, int l_max) -> (Tensor, Tensor)").c_str());
        m.def((name + "_gradients_backward(Tensor xyz, Tensor? sph_grad, Tensor dsph_grad, int l_max) -> Tensor").c_str());
    }
    m.def("contract_gradients(Tensor dsph, Tensor sph_grad) -> Tensor");
    m.def("contract_hessians(Tensor ddsph, Tensor dsph_grad) -> Tensor");
    m.def("owns_reference_namespace() -> bool");
}

// (the key of GPU tensors in a ROCm build of torch is CUDA)
TORCH_LIBRARY_IMPL(sphericart_amd, CUDA, m) {
    m.impl("spherical_harmonics", &values<true>);
    m.impl("spherical_harmonics_with_gradients", &with_gradients<true>);
    m.impl("spherical_harmonics_with_hessians", &with_hessians<true>);
    m.impl("spherical_harmonics_vjp", &vjp<true>);
    m.impl("spherical_harmonics_vjp_backward", &vjp_backward<true>);
    m.impl("spherical_harmonics_gradients_backward", &gradients_backward<true>);
    m.impl("solid_harmonics", &values<false>);
    m.impl("solid_harmonics_with_gradients", &with_gradients<false>);
    m.impl("solid_harmonics_with_hessians", &with_hessians<false>);
    m.impl("solid_harmonics_vjp", &vjp<false>);
    m.impl("solid_harmonics_vjp_backward", &vjp_backward<false>);
    m.impl("solid_harmonics_gradients_backward", &gradients_backward<false>);
    m.impl("contract_gradients", &contract<false>);
    m.impl("contract_hessians", &contract<true>);
}

TORCH_LIBRARY_IMPL(sphericart_amd, CPU, m) {
    for (const char* prefix : {"spherical_harmonics", "solid_harmonics"}) {
        const std::string name(prefix);
        m.impl(name.c_str(), &cpu_values);
        m.impl((name + "_with_gradients").c_str(), &cpu_with_gradients);
        m.impl((name + "_with_hessians").c_str(), &cpu_with_hessians);
        m.impl((name + "_vjp").c_str(), &cpu_vjp);
        m.impl((name + "_vjp_backward").c_str(), &cpu_vjp_backward);
        m.impl((name + "_gradients_backward").c_str(), &cpu_gradients_backward);
    }
    m.impl("contract_gradients", &cpu_contract);
    m.impl("contract_hessians", &cpu_contract);
}

// ---- autograd of GPU tensors --------------------------------------------------------------------------------
//
// The reference's backward formulas (sphericart-torch/python/sphericart/torch/register.py:82-175), with the products in
// place of the derivative arrays wherever the pass is not differentiated again (grad mode is off inside it then); a pass
// that is takes operators that are differentiable themselves. Registered for the Autograd key of the GPU, in front of
// the Python rules of the same operators: a training step on a small structure is bound by the host, and a rule in
// Python costs it 10 to 20 us per operator and direction (1 500 points at l_max = 6, values and their product: 79 us per
// step with the rules in Python, 46 with these, 32 for a step of torch's own sine).
namespace {

using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

template <typename Signature> c10::TypedOperatorHandle<Signature> twin(const std::string& name) {
    return c10::Dispatcher::singleton().findSchemaOrThrow(("sphericart_amd::" + name).c_str(), "").typed<Signature>();
}

template <bool NORMALIZED> const char* prefix_of() {
    return NORMALIZED ? "spherical_harmonics" : "solid_harmonics";
}

using ValuesSignature = Tensor(const Tensor&, int64_t);
using GradientsSignature = std::tuple<Tensor, Tensor>(const Tensor&, int64_t);
using HessiansSignature = std::tuple<Tensor, Tensor, Tensor>(const Tensor&, int64_t);
using VjpSignature = Tensor(const Tensor&, const Tensor&, int64_t);
using VjpBackwardSignature = std::tuple<Tensor, Tensor>(const Tensor&, const Tensor&, const Tensor&, int64_t);
using GradientsBackwardSignature = Tensor(const Tensor&, const std::optional<Tensor>&, const Tensor&, int64_t);
using ContractSignature = Tensor(const Tensor&, const Tensor&);

template <bool NORMALIZED> struct Operators {
    static std::string name(const char* suffix) { return std::string(prefix_of<NORMALIZED>()) + suffix; }
    static const auto& values() {
        static const auto op = twin<ValuesSignature>(name(""));
        return op;
    }
    static const auto& gradients() {
        static const auto op = twin<GradientsSignature>(name("_with_gradients"));
        return op;
    }
    static const auto& hessians() {
        static const auto op = twin<HessiansSignature>(name("_with_hessians"));
        return op;
    }
    static const auto& vjp() {
        static const auto op = twin<VjpSignature>(name("_vjp"));
        return op;
    }
    static const auto& vjp_backward() {
        static const auto op = twin<VjpBackwardSignature>(name("_vjp_backward"));
        return op;
    }
    static const auto& gradients_backward() {
        static const auto op = twin<GradientsBackwardSignature>(name("_gradients_backward"));
        return op;
    }
};
Tensor contract_gradients(const Tensor& dsph, const Tensor& sph_grad) {
    static const auto op = twin<ContractSignature>("contract_gradients");
    return op.call(dsph, sph_grad);
}
Tensor contract_hessians(const Tensor& ddsph, const Tensor& dsph_grad) {
    static const auto op = twin<ContractSignature>("contract_hessians");
    return op.call(ddsph, dsph_grad);
}

// Whether a backward pass that is not differentiated again takes the product without the arrays; beyond its l_max the pass
// contracts what it has saved, and forms no more than is asked for. (No size is looked at: they may be symbolic here.)
bool without_arrays(const Tensor& xyz, int64_t l_max, bool rows) {
    return !at::GradMode::is_enabled() &&
           sphx_second_order_supported(rows, static_cast<int>(l_max), xyz.scalar_type() == at::kDouble) != 0;
}

std::optional<Tensor> maybe(const Tensor& tensor) {
    return tensor.defined() ? std::optional<Tensor>(tensor) : std::nullopt;
}

template <bool NORMALIZED> struct ValuesFunction : Function<ValuesFunction<NORMALIZED>> {
    static constexpr bool is_traceable = true;
    static Tensor forward(AutogradContext* ctx, const Tensor& xyz, int64_t l_max) {
        ctx->set_materialize_grads(false);
        ctx->saved_data["l_max"] = l_max;
        ctx->save_for_backward({xyz});
        const at::AutoDispatchBelowAutograd guard;
        return Operators<NORMALIZED>::values().call(xyz, l_max);
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        if (!grads[0].defined() || !ctx->needs_input_grad(0)) return {Tensor(), Tensor()};
        const auto saved = ctx->get_saved_variables();
        return {Operators<NORMALIZED>::vjp().call(saved[0], grads[0], ctx->saved_data["l_max"].toInt()), Tensor()};
    }
};

// the derivatives of the fused product xyz_grad[i, a] = sum_k dsph[i, a, k] w[i, k]
template <bool NORMALIZED> struct VjpFunction : Function<VjpFunction<NORMALIZED>> {
    static constexpr bool is_traceable = true;
    static Tensor forward(AutogradContext* ctx, const Tensor& xyz, const Tensor& sph_grad, int64_t l_max) {
        ctx->saved_data["l_max"] = l_max;
        ctx->save_for_backward({xyz, sph_grad});
        const at::AutoDispatchBelowAutograd guard;
        return Operators<NORMALIZED>::vjp().call(xyz, sph_grad, l_max);
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        const auto saved = ctx->get_saved_variables();
        const Tensor &xyz = saved[0], &sph_grad = saved[1], &grad = grads[0];
        const int64_t l_max = ctx->saved_data["l_max"].toInt();
        if (without_arrays(xyz, l_max, false)) {
            auto both = Operators<NORMALIZED>::vjp_backward().call(xyz, sph_grad, grad, l_max);
            return {std::get<0>(both), std::get<1>(both), Tensor()};
        }
        const auto all = Operators<NORMALIZED>::hessians().call(xyz, l_max);
        Tensor d_xyz, d_sph_grad;
        if (ctx->needs_input_grad(0)) {
            // d/d xyz[i, b]: sum_{a, k} grad[i, a] w[i, k] ddsph[i, a, b, k]
            d_xyz = contract_hessians(std::get<2>(all), grad.unsqueeze(2) * sph_grad.unsqueeze(1));
        }
        if (ctx->needs_input_grad(1)) d_sph_grad = (grad.unsqueeze(2) * std::get<1>(all)).sum(1);
        return {d_xyz, d_sph_grad, Tensor()};
    }
};

// Backward from the gradients of values and gradients, either of which may be missing, by the arrays.
template <typename Dsph, typename Ddsph>
Tensor backward_from(const Tensor& grad_sph, const Tensor& grad_dsph, Dsph dsph, Ddsph ddsph) {
    Tensor sum;
    if (grad_sph.defined()) sum = contract_gradients(dsph(), grad_sph);
    if (grad_dsph.defined()) {
        const Tensor extra = contract_hessians(ddsph(), grad_dsph);
        sum = sum.defined() ? sum + extra : extra;
    }
    return sum;
}

template <bool NORMALIZED> struct GradientsFunction : Function<GradientsFunction<NORMALIZED>> {
    static constexpr bool is_traceable = true;
    static variable_list forward(AutogradContext* ctx, const Tensor& xyz, int64_t l_max) {
        const at::AutoDispatchBelowAutograd guard;
        const auto both = Operators<NORMALIZED>::gradients().call(xyz, l_max);
        ctx->set_materialize_grads(false); // outputs that were not used arrive undefined
        ctx->saved_data["l_max"] = l_max;
        ctx->save_for_backward({xyz, std::get<1>(both)});
        return {std::get<0>(both), std::get<1>(both)};
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        if (!ctx->needs_input_grad(0)) return {Tensor(), Tensor()};
        const auto saved = ctx->get_saved_variables();
        const Tensor &xyz = saved[0], &dsph = saved[1];
        const int64_t l_max = ctx->saved_data["l_max"].toInt();
        if (grads[1].defined() && without_arrays(xyz, l_max, true)) {
            return {Operators<NORMALIZED>::gradients_backward().call(xyz, maybe(grads[0]), grads[1], l_max), Tensor()};
        }
        return {backward_from(grads[0], grads[1], [&] { return dsph; },
                              [&] { return std::get<2>(Operators<NORMALIZED>::hessians().call(xyz, l_max)); }),
                Tensor()};
    }
};

// (xyz is not saved: both arrays are there, and a program may have moved its points meanwhile)
template <bool NORMALIZED> struct HessiansFunction : Function<HessiansFunction<NORMALIZED>> {
    static constexpr bool is_traceable = true;
    static variable_list forward(AutogradContext* ctx, const Tensor& xyz, int64_t l_max) {
        const at::AutoDispatchBelowAutograd guard;
        const auto all = Operators<NORMALIZED>::hessians().call(xyz, l_max);
        ctx->set_materialize_grads(false);
        ctx->save_for_backward({std::get<1>(all), std::get<2>(all)});
        return {std::get<0>(all), std::get<1>(all), std::get<2>(all)};
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        TORCH_CHECK(!grads[2].defined(), "Third derivatives of the spherical harmonics with respect to the Cartesian coordinates "
                                         "are not supported.");
        const auto saved = ctx->get_saved_variables();
        return {backward_from(grads[0], grads[1], [&] { return saved[0]; }, [&] { return saved[1]; }), Tensor()};
    }
};

// The kernels of the Autograd key: straight on where nothing asks for a gradient.
bool records(const Tensor& a) { return at::GradMode::is_enabled() && a.requires_grad(); }

template <bool NORMALIZED> Tensor autograd_values(c10::DispatchKeySet keys, const Tensor& xyz, int64_t l_max) {
    if (records(xyz)) return ValuesFunction<NORMALIZED>::apply(xyz, l_max);
    return Operators<NORMALIZED>::values().redispatch(keys & c10::after_autograd_keyset, xyz, l_max);
}
template <bool NORMALIZED>
std::tuple<Tensor, Tensor> autograd_with_gradients(c10::DispatchKeySet keys, const Tensor& xyz, int64_t l_max) {
    if (!records(xyz)) return Operators<NORMALIZED>::gradients().redispatch(keys & c10::after_autograd_keyset, xyz, l_max);
    const auto both = GradientsFunction<NORMALIZED>::apply(xyz, l_max);
    return {both[0], both[1]};
}
template <bool NORMALIZED>
std::tuple<Tensor, Tensor, Tensor> autograd_with_hessians(c10::DispatchKeySet keys, const Tensor& xyz, int64_t l_max) {
    if (!records(xyz)) return Operators<NORMALIZED>::hessians().redispatch(keys & c10::after_autograd_keyset, xyz, l_max);
    const auto all = HessiansFunction<NORMALIZED>::apply(xyz, l_max);
    return {all[0], all[1], all[2]};
}
template <bool NORMALIZED>
Tensor autograd_vjp(c10::DispatchKeySet keys, const Tensor& xyz, const Tensor& sph_grad, int64_t l_max) {
    if (records(xyz) || records(sph_grad)) return VjpFunction<NORMALIZED>::apply(xyz, sph_grad, l_max);
    return Operators<NORMALIZED>::vjp().redispatch(keys & c10::after_autograd_keyset, xyz, sph_grad, l_max);
}

} // namespace

TORCH_LIBRARY_IMPL(sphericart_amd, AutogradCUDA, m) {
    m.impl("spherical_harmonics", TORCH_FN(autograd_values<true>));
    m.impl("spherical_harmonics_with_gradients", TORCH_FN(autograd_with_gradients<true>));
    m.impl("spherical_harmonics_with_hessians", TORCH_FN(autograd_with_hessians<true>));
    m.impl("spherical_harmonics_vjp", TORCH_FN(autograd_vjp<true>));
    m.impl("solid_harmonics", TORCH_FN(autograd_values<false>));
    m.impl("solid_harmonics_with_gradients", TORCH_FN(autograd_with_gradients<false>));
    m.impl("solid_harmonics_with_hessians", TORCH_FN(autograd_with_hessians<false>));
    m.impl("solid_harmonics_vjp", TORCH_FN(autograd_vjp<false>));
}

// ---- the reference's namespace (sphericart-torch/src/torch.cpp:367-385) -------------------------------------
//
// `sphericart_torch` with the reference's eight schemas, so that code written against torch.ops.sphericart_torch.*,
// saved TorchScript modules included, resolves against this library alone. Every operator forwards to its twin
// above through the dispatcher (a composite implementation: whatever autograd, fake-tensor and vmap rules the twin
// has apply unchanged); the two *_omp_num_threads operators report 1, there being no host evaluator and no OpenMP
// team behind these operators. Defined when this library is loaded unless the namespace is taken already (the
// reference's own extension is loaded): then nothing is defined and owns_reference_namespace() says so.
namespace {

template <bool NORMALIZED> Tensor reference_values(const Tensor& xyz, int64_t l_max) {
    static const auto op = twin<Tensor(const Tensor&, int64_t)>(prefix_of<NORMALIZED>());
    return op.call(xyz, l_max);
}
template <bool NORMALIZED> std::tuple<Tensor, Tensor> reference_with_gradients(const Tensor& xyz, int64_t l_max) {
    static const auto op =
        twin<std::tuple<Tensor, Tensor>(const Tensor&, int64_t)>(std::string(prefix_of<NORMALIZED>()) + "_with_gradients");
    return op.call(xyz, l_max);
}
template <bool NORMALIZED>
std::tuple<Tensor, Tensor, Tensor> reference_with_hessians(const Tensor& xyz, int64_t l_max) {
    static const auto op = twin<std::tuple<Tensor, Tensor, Tensor>(const Tensor&, int64_t)>(
        std::string(prefix_of<NORMALIZED>()) + "_with_hessians");
    return op.call(xyz, l_max);
}
int64_t one_thread(int64_t) { return 1; }

std::unique_ptr<torch::Library> define_reference_namespace() {
    try {
        auto m = std::make_unique<torch::Library>(torch::Library::DEF, "sphericart_torch", c10::nullopt, __FILE__,
                                                  __LINE__);
        for (const char* prefix : {"spherical_harmonics", "solid_harmonics"}) {
            const std::string name(prefix);
            m->def((name + "(Tensor xyz, int l_max) -> Tensor").c_str());
            m->def((name + "_with_gradients(Tensor xyz, int l_max) -> (Tensor, Tensor)").c_str());
            m->def((name + "_with_hessians(Tensor xyz, int l_max) -> (Tensor, Tensor, Tensor)").c_str());
            m->def((name + "_omp_num_threads(int l_max) -> int").c_str());
            m->impl((name + "_omp_num_threads").c_str(), c10::DispatchKey::CompositeExplicitAutograd, &one_thread);
        }
        const auto composite = c10::DispatchKey::CompositeImplicitAutograd;
        m->impl("spherical_harmonics", composite, &reference_values<true>);
        m->impl("spherical_harmonics_with_gradients", composite, &reference_with_gradients<true>);
        m->impl("spherical_harmonics_with_hessians", composite, &reference_with_hessians<true>);
        m->impl("solid_harmonics", composite, &reference_values<false>);
        m->impl("solid_harmonics_with_gradients", composite, &reference_with_gradients<false>);
        m->impl("solid_harmonics_with_hessians", composite, &reference_with_hessians<false>);
        return m;
    } catch (const c10::Error&) {
        return nullptr; // another library owns the namespace
    }
}

const std::unique_ptr<torch::Library> reference_namespace = define_reference_namespace();

bool owns_reference_namespace() { return reference_namespace != nullptr; }

} // namespace

TORCH_LIBRARY_IMPL(sphericart_amd, CompositeExplicitAutograd, m) {
    m.impl("owns_reference_namespace", &owns_reference_namespace);
}
