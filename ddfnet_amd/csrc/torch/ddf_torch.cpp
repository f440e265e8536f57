// PyTorch front end of libddf_hip.so as a C++ extension: the `ddf` operator as a
// C++ autograd function.  Host-side mirror of DDFFunction / ddf of the reference
// (ddf/ddf.py:27-122): same arguments, same assertion messages.  This file holds
// no device code; every kernel is behind the C ABI of include/ddf_hip.h, and
// torch is used for tensors, the caching allocator and the current stream.
//
// What it saves over the Python autograd.Function in functional.py is host time
// per call: argument checks, dtype promotion, output allocation and the two
// library calls happen without the interpreter.
#include <torch/extension.h>

#include <ATen/FuncTorchTLS.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/autograd/VariableTypeUtils.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <sstream>
#include <string>

#include "ddf_hip.h"

namespace ddf_torch {

namespace py = pybind11;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// `assert cond, msg` of the Python front end.
// (Also reached from the autograd engine's threads, which do not hold the GIL.)
[[noreturn]] inline void assertion_error(const std::string &msg) {
    py::gil_scoped_acquire gil;
    PyErr_SetString(PyExc_AssertionError, msg.c_str());
    throw py::error_already_set();
}

// A failed library call, raised as ddfnet_amd._lib.DDFHipError.
inline void check_status(int status) {
    if (status == DDF_OK) return;
    const std::string msg = std::string(ddf_hip_status_string(status)) + ": " + ddf_hip_last_error();
    py::gil_scoped_acquire gil;
    py::object cls = py::module_::import("ddfnet_amd._lib").attr("DDFHipError");
    PyErr_SetString(cls.ptr(), msg.c_str());
    throw py::error_already_set();
}

inline int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kHalf: return DDF_F16;
        case at::kFloat: return DDF_F32;
        case at::kDouble: return DDF_F64;
        default: return -1;
    }
}

inline int combine_code(const std::string &kernel_combine) {
    if (kernel_combine == "mul") return DDF_MUL;
    if (kernel_combine == "add") return DDF_ADD;
    assertion_error("only support mul or add combination, instead of " + kernel_combine);
}

std::string size_string(const at::Tensor &t) {
    // as torch.Size prints: torch.Size([2, 3, 4, 5])
    std::ostringstream os;
    os << "torch.Size([";
    for (int64_t i = 0; i < t.dim(); ++i) os << (i ? ", " : "") << t.size(i);
    os << "])";
    return os.str();
}

inline hipStream_t current_stream(const at::Tensor &t) {
    return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

// A new device tensor, without the dispatcher (every kernel of the library writes every
// element, so nothing has to be filled in either).
inline at::Tensor new_tensor(c10::IntArrayRef sizes, at::ScalarType type, const at::Device &device) {
    return at::Tensor(at::detail::empty_cuda(sizes, type, device, c10::nullopt));
}

inline bool has_tangent(const at::Tensor &t) { return torch::autograd::isFwGradDefined(t); }
// No derivative is lost in silence: forward mode (whether or not gradients are recorded) and
// torch.func's transforms are refused, as a torch::autograd::Function does.
inline void refuse_transforms() {
    if (const auto &tls = at::functorch::functorchTLSAccessor()) tls->checkSupportsCppAutogradFunction();
}

// Somebody takes part in what the dispatcher would see of this call and a launch does not show:
// a tensor of a subclass with a dispatch of its own, a dispatch mode, torch.func, a tracer.
inline bool dispatch_watched(const at::Tensor &t) {
    return t.unsafeGetTensorImpl()->is_python_dispatch() || c10::impl::TorchDispatchModeTLS::any_modes_set() ||
           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
           torch::jit::tracer::isTracing();
}

// The operator's gradient as a node of the autograd graph.  (A torch::autograd::Function
// does the same through a generic context - argument lists, a dictionary of boxed values,
// lists of optional results - at a few microseconds per call and direction.)
struct DDFNode : public torch::autograd::Node {
    torch::autograd::SavedVariable features_, channel_filter_, spatial_filter_;
    int k, d, s, combine, variant;

    std::string name() const override { return "DDFBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        features_.reset_data();
        channel_filter_.reset_data();
        spatial_filter_.reset_data();
    }
    variable_list apply(variable_list &&grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        variable_list result(3);
        if (!grads[0].defined()) return result;
        const at::Tensor features = features_.unpack(), channel_filter = channel_filter_.unpack(),
                         spatial_filter = spatial_filter_.unpack();
        const at::ScalarType type = features.scalar_type();
        const at::Device device = features.device();
        at::Tensor go = std::move(grads[0]);
        if (!go.is_cuda()) assertion_error("");
        if (go.scalar_type() != type) go = go.to(type);
        if (!go.is_contiguous()) go = go.contiguous();

        // only the gradients autograd asks for are computed
        unsigned need = 0;
        if (task_should_compute_output(0)) { need |= DDF_NEED_DX; result[0] = new_tensor(features.sizes(), type, device); }
        if (task_should_compute_output(1)) { need |= DDF_NEED_DCF; result[1] = new_tensor(channel_filter.sizes(), type, device); }
        if (task_should_compute_output(2)) { need |= DDF_NEED_DSF; result[2] = new_tensor(spatial_filter.sizes(), type, device); }
        if (!need) return result;
        const int64_t b = features.size(0), c = features.size(1), h = features.size(2), w = features.size(3);
        const int dt = dtype_code(type);
        c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(device);
        const size_t bytes = ddf_hip_backward_workspace_bytes(b, c, h, w, k, d, s, combine, dt, need, variant);
        at::Tensor ws;
        if (bytes) ws = new_tensor({(int64_t)bytes}, at::kByte, device);
        auto ptr = [](const at::Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; };
        check_status(ddf_hip_backward(go.data_ptr(), features.data_ptr(), channel_filter.data_ptr(),
                                      spatial_filter.data_ptr(), ptr(result[0]), ptr(result[1]), ptr(result[2]),
                                      ptr(ws), bytes, b, c, h, w, k, d, s, combine, dt, need, variant,
                                      current_stream(features)));
        return result;
    }
};

// ddf(features, channel_filter, spatial_filter, kernel_size=3, dilation=1, stride=1,
//     kernel_combine='mul', version=''): checks in the order and with the messages of
// DDFFunction.forward in functional.py (ddf/ddf.py:29-62 of the reference).
at::Tensor ddf(at::Tensor features, at::Tensor channel_filter, at::Tensor spatial_filter,
               int64_t kernel_size, int64_t dilation, int64_t stride,
               const std::string &kernel_combine, const std::string &version) {
    if (!features.is_cuda()) assertion_error("input feature must be a CUDA tensor.");
    if (!channel_filter.is_cuda()) assertion_error("channel_filter must be a CUDA tensor.");
    if (!spatial_filter.is_cuda()) assertion_error("spatial_filter must be a CUDA tensor.");

    // One working dtype for the three operands.  Under autocast to fp16 that is
    // fp16 (the kernels accumulate in fp32); bf16 is not a storage type of the
    // library, so autocast to bf16 leaves the operands as they are.
    at::ScalarType dtype = at::promote_types(
        at::promote_types(features.scalar_type(), channel_filter.scalar_type()),
        spatial_filter.scalar_type());
    if (at::autocast::is_autocast_enabled(at::kCUDA) &&
        at::autocast::get_autocast_dtype(at::kCUDA) == at::kHalf && dtype == at::kFloat)
        dtype = at::kHalf;
    if (dtype_code(dtype) < 0) {
        std::ostringstream os;
        os << "unsupported dtype " << dtype;
        assertion_error(os.str());
    }
    if (features.dim() != 4 || channel_filter.dim() != 4 || spatial_filter.dim() != 4)
        assertion_error("features, channel_filter and spatial_filter must be 4-dimensional");
    if (stride < 1) assertion_error("");
    for (at::Tensor *t : {&features, &channel_filter, &spatial_filter}) {
        if (t->scalar_type() != dtype) *t = t->to(dtype);
        if (!t->is_contiguous()) *t = t->contiguous();
    }

    const int64_t b = features.size(0), c = features.size(1), h = features.size(2), w = features.size(3);
    const int64_t out_h = h / stride, out_w = w / stride;
    if (channel_filter.size(0) != b || channel_filter.size(1) != c)
        assertion_error("channel_filter size " + size_string(channel_filter) +
                        " does not match feature size " + size_string(features));
    if (channel_filter.size(2) != kernel_size || channel_filter.size(3) != kernel_size)
        assertion_error("channel_filter size " + size_string(channel_filter) +
                        " does not match kernel size " + std::to_string(kernel_size));
    if (spatial_filter.size(0) != b || spatial_filter.size(2) != out_h || spatial_filter.size(3) != out_w)
        assertion_error("spatial_filter size " + size_string(spatial_filter) +
                        " does not match feature size " + size_string(features) + " with stride " +
                        std::to_string(stride));
    if (spatial_filter.size(1) != kernel_size * kernel_size)
        assertion_error("spatial_filter size " + size_string(spatial_filter) +
                        " does not match kernel size " + std::to_string(kernel_size));
    if ((kernel_size - 1) % 2 != 0 || kernel_size < 1 || dilation < 1) assertion_error("");
    const int combine = combine_code(kernel_combine);
    int variant;
    if (version.empty()) variant = DDF_VARIANT_AUTO;
    else if (version == "o") variant = DDF_VARIANT_GENERIC;
    else if (version == "f") variant = DDF_VARIANT_TILED;
    else assertion_error("version must be '', 'o' or 'f', instead of " + version);

    refuse_transforms();
    if (has_tangent(features) || has_tangent(channel_filter) || has_tangent(spatial_filter))
        throw std::runtime_error("ddf has no forward-mode derivative");

    at::Tensor out = new_tensor({b, c, out_h, out_w}, dtype, features.device());
    {
        c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(features.device());
        check_status(ddf_hip_forward(features.data_ptr(), channel_filter.data_ptr(), spatial_filter.data_ptr(),
                                     out.data_ptr(), b, c, h, w, (int)kernel_size, (int)dilation, (int)stride, combine,
                                     dtype_code(dtype), variant, current_stream(features)));
    }
    if (at::GradMode::is_enabled() &&
        (features.requires_grad() || channel_filter.requires_grad() || spatial_filter.requires_grad())) {
        auto node = std::shared_ptr<DDFNode>(new DDFNode(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(features, channel_filter, spatial_filter));
        node->k = (int)kernel_size;
        node->d = (int)dilation;
        node->s = (int)stride;
        node->combine = combine;
        // 'f' forces the tiled kernels in the forward pass only (the reference's
        // faster modules export no backward)
        node->variant = variant == DDF_VARIANT_GENERIC ? DDF_VARIANT_GENERIC : DDF_VARIANT_AUTO;
        node->features_ = torch::autograd::SavedVariable(features, false);
        node->channel_filter_ = torch::autograd::SavedVariable(channel_filter, false);
        node->spatial_filter_ = torch::autograd::SavedVariable(spatial_filter, false);
        torch::autograd::set_history(out, node);
    }
    return out;
}

// Direct entry for the ordinary call - tensors, numbers and texts by position - without
// pybind11's argument casters; anything else goes to the function above through them.
PyObject *ddf_fast(PyObject *self, PyObject *const *args, Py_ssize_t nargs, PyObject *kwnames);

// Up-sampling DDF (DDFUpPack.forward, ddf/ddf.py:264-272 of the reference: one
// ddf call per sub-pixel branch, torch.stack, F.pixel_shuffle) as one operator:
// one library call forward, one backward.  `filters` holds the scale*scale
// channel filters followed by the scale*scale spatial filters.
class DDFUpAutograd : public torch::autograd::Function<DDFUpAutograd> {
public:
    // (filters as a TensorList: that is the list type whose elements autograd tracks)
    static at::Tensor forward(AutogradContext *ctx, const at::Tensor &features, at::TensorList filters,
                              int64_t k, int64_t d, int64_t scale, int64_t combine) {
        const int64_t branches = scale * scale;
        const int64_t b = features.size(0), c = features.size(1), h = features.size(2),
                      w = features.size(3);
        const void *cf[DDF_UP_MAX_BRANCHES], *sf[DDF_UP_MAX_BRANCHES];
        for (int64_t i = 0; i < branches; ++i) {
            cf[i] = filters[i].data_ptr();
            sf[i] = filters[branches + i].data_ptr();
        }
        at::Tensor out = at::empty({b, c, h * scale, w * scale}, features.options());
        {
            c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(features.device());
            check_status(ddf_hip_up_forward(features.data_ptr(), cf, sf, out.data_ptr(), b, c, h, w,
                                            (int)k, (int)d, (int)scale, (int)combine,
                                            dtype_code(features.scalar_type()),
                                            current_stream(features)));
        }
        bool any = features.requires_grad();
        for (const auto &t : filters) any = any || t.requires_grad();
        if (any) {
            variable_list saved;
            saved.reserve(1 + filters.size());
            saved.push_back(features);
            for (const auto &t : filters) saved.push_back(t);
            ctx->save_for_backward(saved);
        }
        ctx->saved_data["k"] = k;
        ctx->saved_data["d"] = d;
        ctx->saved_data["scale"] = scale;
        ctx->saved_data["combine"] = combine;
        return out;
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const at::Tensor &features = saved[0];
        const int k = (int)ctx->saved_data["k"].toInt(), d = (int)ctx->saved_data["d"].toInt(),
                  scale = (int)ctx->saved_data["scale"].toInt(),
                  combine = (int)ctx->saved_data["combine"].toInt();
        const int branches = scale * scale;
        const at::Tensor go = grads[0].to(features.scalar_type()).contiguous();
        variable_list result(1 + 2 * branches + 4);
        unsigned need = 0;
        const void *cf[DDF_UP_MAX_BRANCHES], *sf[DDF_UP_MAX_BRANCHES];
        void *dcf[DDF_UP_MAX_BRANCHES], *dsf[DDF_UP_MAX_BRANCHES];
        if (ctx->needs_input_grad(0)) {
            need |= DDF_NEED_DX;
            result[0] = at::empty_like(features);
        }
        for (int i = 0; i < branches; ++i) {
            cf[i] = saved[1 + i].data_ptr();
            sf[i] = saved[1 + branches + i].data_ptr();
            dcf[i] = dsf[i] = nullptr;
            if (ctx->needs_input_grad(1 + i)) {
                need |= DDF_NEED_DCF;
                result[1 + i] = at::empty_like(saved[1 + i]);
                dcf[i] = result[1 + i].data_ptr();
            }
            if (ctx->needs_input_grad(1 + branches + i)) {
                need |= DDF_NEED_DSF;
                result[1 + branches + i] = at::empty_like(saved[1 + branches + i]);
                dsf[i] = result[1 + branches + i].data_ptr();
            }
        }
        if (need) {
            const int64_t b = features.size(0), c = features.size(1), h = features.size(2),
                          w = features.size(3);
            const int dt = dtype_code(features.scalar_type());
            c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(features.device());
            const size_t bytes = ddf_hip_up_backward_workspace_bytes(b, c, h, w, k, d, scale, combine,
                                                                     dt, need);
            at::Tensor ws = at::empty({(int64_t)std::max<size_t>(bytes, 1)},
                                      features.options().dtype(at::kByte));
            check_status(ddf_hip_up_backward(
                go.data_ptr(), features.data_ptr(), cf, sf,
                result[0].defined() ? result[0].data_ptr() : nullptr, dcf, dsf, ws.data_ptr(), bytes,
                b, c, h, w, k, d, scale, combine, dt, need, current_stream(features)));
        }
        return result;
    }
};

// ddf_up(features, channel_filters, spatial_filters, kernel_size, dilation, scale_factor,
// kernel_combine): the checks of DDFUpFunction.forward in functional.py.  The caller has
// asked ddf_hip_up_forward's coverage (functional.ddf_up falls back to the composition).
at::Tensor ddf_up(at::Tensor features, std::vector<at::Tensor> channel_filters,
                  std::vector<at::Tensor> spatial_filters, int64_t kernel_size, int64_t dilation,
                  int64_t scale, const std::string &kernel_combine) {
    const int64_t branches = scale * scale;
    if (scale < 2 || branches > DDF_UP_MAX_BRANCHES ||
        (int64_t)channel_filters.size() != branches || (int64_t)spatial_filters.size() != branches)
        assertion_error("expected " + std::to_string(branches) + " channel filters followed by " +
                        std::to_string(branches) + " spatial filters");
    if (!features.is_cuda()) assertion_error("input feature must be a CUDA tensor.");
    const int combine = combine_code(kernel_combine);
    if ((kernel_size - 1) % 2 != 0 || kernel_size < 1 || dilation < 1) assertion_error("");
    at::ScalarType dtype = features.scalar_type();
    for (const auto *list : {&channel_filters, &spatial_filters})
        for (const auto &t : *list) {
            if (!t.is_cuda()) assertion_error("filters must be CUDA tensors.");
            dtype = at::promote_types(dtype, t.scalar_type());
        }
    if (at::autocast::is_autocast_enabled(at::kCUDA) &&
        at::autocast::get_autocast_dtype(at::kCUDA) == at::kHalf && dtype == at::kFloat)
        dtype = at::kHalf;
    if (dtype_code(dtype) < 0) {
        std::ostringstream os;
        os << "unsupported dtype " << dtype;
        assertion_error(os.str());
    }
    if (features.dim() != 4) assertion_error("features must be 4-dimensional");
    auto as_operand = [dtype](at::Tensor &t) {
        if (t.scalar_type() != dtype) t = t.to(dtype);
        if (!t.is_contiguous()) t = t.contiguous();
    };
    as_operand(features);
    const int64_t b = features.size(0), c = features.size(1), h = features.size(2), w = features.size(3);
    variable_list filters;
    filters.reserve(2 * branches);
    for (auto &t : channel_filters) {
        as_operand(t);
        if (t.dim() != 4 || t.size(0) != b || t.size(1) != c || t.size(2) != kernel_size ||
            t.size(3) != kernel_size)
            assertion_error("channel_filter size " + size_string(t) + " does not match feature size " +
                            size_string(features));
        filters.push_back(t);
    }
    for (auto &t : spatial_filters) {
        as_operand(t);
        if (t.dim() != 4 || t.size(0) != b || t.size(1) != kernel_size * kernel_size ||
            t.size(2) != h || t.size(3) != w)
            assertion_error("spatial_filter size " + size_string(t) + " does not match feature size " +
                            size_string(features));
        filters.push_back(t);
    }
    return DDFUpAutograd::apply(features, at::TensorList(filters), kernel_size, dilation, scale,
                                (int64_t)combine);
}

namespace {
py::object *g_ddf_casting = nullptr;    // ddf bound through pybind11 (kept for the process)

bool int_argument(PyObject *o, int64_t *v) {
    if (!PyLong_CheckExact(o)) return false;
    *v = PyLong_AsLongLong(o);
    if (*v == -1 && PyErr_Occurred()) { PyErr_Clear(); return false; }
    return true;
}
}  // namespace

PyObject *ddf_fast(PyObject *, PyObject *const *args, Py_ssize_t nargs, PyObject *kwnames) {
    int64_t number[3] = {3, 1, 1};
    std::string text[2] = {"mul", ""};
    bool plain = nargs >= 3 && nargs <= 8 && (kwnames == nullptr || PyTuple_GET_SIZE(kwnames) == 0);
    for (Py_ssize_t i = 0; plain && i < 3; ++i) plain = THPVariable_CheckExact(args[i]);
    for (Py_ssize_t i = 3; plain && i < nargs && i < 6; ++i) plain = int_argument(args[i], &number[i - 3]);
    for (Py_ssize_t i = 6; plain && i < nargs; ++i) {
        Py_ssize_t len = 0;
        const char *c = PyUnicode_CheckExact(args[i]) ? PyUnicode_AsUTF8AndSize(args[i], &len) : nullptr;
        if (c) text[i - 6].assign(c, (size_t)len);
        else { PyErr_Clear(); plain = false; }
    }
    if (!plain) return PyObject_Vectorcall(g_ddf_casting->ptr(), args, (size_t)nargs, kwnames);
    HANDLE_TH_ERRORS
    return THPVariable_Wrap(ddf(THPVariable_Unpack(args[0]), THPVariable_Unpack(args[1]), THPVariable_Unpack(args[2]),
                                number[0], number[1], number[2], text[0], text[1]));
    END_HANDLE_TH_ERRORS
}

namespace {
PyMethodDef g_ddf_method = {"ddf", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&ddf_fast)),
                            METH_FASTCALL | METH_KEYWORDS, "ddf(features, channel_filter, spatial_filter, ...)"};
}  // namespace

}  // namespace ddf_torch

#include "ddf_pack.h"

#include "ddf_net.h"

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    using namespace ddf_torch;
    m.doc() = "ddf operator of libddf_hip.so as a C++ autograd function";
    m.def("_ddf_casting", &ddf, py::arg("features"), py::arg("channel_filter"), py::arg("spatial_filter"),
          py::arg("kernel_size") = 3, py::arg("dilation") = 1, py::arg("stride") = 1,
          py::arg("kernel_combine") = "mul", py::arg("version") = "");
    g_ddf_casting = new py::object(m.attr("_ddf_casting"));
    m.attr("ddf") = py::reinterpret_steal<py::object>(PyCFunction_NewEx(&g_ddf_method, nullptr, nullptr));
    m.def("ddf_up", &ddf_up, py::arg("features"), py::arg("channel_filters"),
          py::arg("spatial_filters"), py::arg("kernel_size") = 3, py::arg("dilation") = 1,
          py::arg("scale_factor") = 2, py::arg("kernel_combine") = "mul");
    py::class_<ModuleGuard::Rules>(m, "GuardRules")
        .def(py::init([](py::dict classes, py::dict own, py::tuple operators, py::tuple silent) {
            return ModuleGuard::Rules{classes, own, operators, silent};
        }));
    py::class_<ModuleGuard>(m, "ModuleGuard", py::custom_type_setup(collectable<ModuleGuard>))
        .def("holds", &ModuleGuard::holds)
        .def("covers", &ModuleGuard::covers);
    m.def("guard_of", &ModuleGuard::make, "a guard of modules (the first is the owner), or None");
    py::class_<ModuleSnapshot>(m, "ModuleSnapshot", py::custom_type_setup(collectable<ModuleSnapshot>))
        .def(py::init<const ModuleGuard::Rules &, py::list>())
        .def("holds", &ModuleSnapshot::holds);
    py::class_<PackPlan>(m, "PackPlan", py::custom_type_setup(collectable<PackPlan>))
        .def(py::init<py::object, py::list, double, double, int64_t, int, int, int, int, const std::string &, bool,
                      bool>())
        .def("valid", &PackPlan::holds)
        .def("misfit", &PackPlan::misfit, "why the branch kernels cannot run these features, or None");
    m.def("pack_forward", &pack_forward, "DDFPack.forward through a plan, or None");
    m.def("pack_infer", &pack_infer,
          "DDFPack.forward without gradients, refusing with an error what the kernels do not take");
    py::class_<NetPlan>(m, "NetPlan", py::custom_type_setup(collectable<NetPlan>))
        .def(py::init<py::object>())
        .def("set_ends", &NetPlan::set_ends)
        .def("add_block", &NetPlan::add_block)
        .def("valid", &NetPlan::holds)
        .def("misfit", &NetPlan::misfit, "why the native inference cannot run this input, or None");
    m.def("net_forward", &net_forward, "DDFResNet.forward through a plan, or None");
    m.def("library_version", []() { return ddf_hip_version(); });
}
