// Direct calls of torch.ops.npu.* from Python.
//
// torch.ops.<namespace>.<op>(...) is a Python-level call of an overload packet, which matches the arguments against the
// schema, boxes them on an IValue stack and unboxes the results: about as long as the rest of the host side of a decode-sized
// launch.  install() gives the packets of this library's operators a type whose call slot converts the arguments straight to
// the C++ types of the operator and calls the dispatcher's typed entry, so that everything the dispatcher provides (fake
// tensors, dispatch modes, profiler, autograd keys) stays in place.  Anything this converter does not take - a
// __torch_function__ override or mode, tracing, an argument of another type, a missing or unknown argument - goes to the packet's
// own call, with its results and its error messages.
#include <Python.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/ATen.h>
#include <ATen/core/LegacyTypeDispatch.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <array>
#include <string>
#include <tuple>
#include <utility>
#include <vector>

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using OptType = std::optional<at::ScalarType>;

// What one argument becomes: held by value (tensors by reference), `load` says whether the Python object fits.
template <class T>
struct Arg;
// torch.Tensor and torch.nn.Parameter themselves; any other subclass may override the call
PyTypeObject *parameter_type = nullptr;
bool plain_tensor(PyObject *o) { return THPVariable_CheckExact(o) || Py_TYPE(o) == parameter_type; }
template <>
struct Arg<const Tensor &> {
    const Tensor *v = nullptr;
    bool load(PyObject *o)
    {
        if (!plain_tensor(o)) return false;
        v = &THPVariable_Unpack(o);
        return true;
    }
    bool load_default(const c10::IValue &) { return false; }
    const Tensor &get() const { return *v; }
};
template <>
struct Arg<const OptTensor &> {
    OptTensor v;
    bool load(PyObject *o)
    {
        if (o == Py_None) return true;
        if (!plain_tensor(o)) return false;
        v = THPVariable_Unpack(o);
        return true;
    }
    bool load_default(const c10::IValue &d) { return d.isNone(); }
    const OptTensor &get() const { return v; }
};
template <>
struct Arg<int64_t> {
    int64_t v = 0;
    bool load(PyObject *o)
    {
        if (!PyLong_CheckExact(o)) return false;
        int overflow = 0;
        v = PyLong_AsLongLongAndOverflow(o, &overflow);
        return overflow == 0;
    }
    bool load_default(const c10::IValue &d) { return d.isInt() ? (v = d.toInt(), true) : false; }
    int64_t get() const { return v; }
};
template <>
struct Arg<bool> {
    bool v = false;
    bool load(PyObject *o)
    {
        v = o == Py_True;
        return v || o == Py_False;
    }
    bool load_default(const c10::IValue &d) { return d.isBool() ? (v = d.toBool(), true) : false; }
    bool get() const { return v; }
};
template <>
struct Arg<at::ScalarType> {
    at::ScalarType v = at::ScalarType::Undefined;
    bool load(PyObject *o)
    {
        if (!THPDtype_Check(o)) return false;
        v = reinterpret_cast<THPDtype *>(o)->scalar_type;
        return true;
    }
    bool load_default(const c10::IValue &) { return false; }
    at::ScalarType get() const { return v; }
};
template <>
struct Arg<OptType> {
    OptType v;
    bool load(PyObject *o)
    {
        if (o == Py_None) return true;
        if (!THPDtype_Check(o)) return false;
        v = reinterpret_cast<THPDtype *>(o)->scalar_type;
        return true;
    }
    bool load_default(const c10::IValue &d) { return d.isNone(); }
    OptType get() const { return v; }
};

PyObject *to_python(Tensor &&t) { return THPVariable_Wrap(std::move(t)); }
template <class... T>
PyObject *to_python(std::tuple<T...> &&r)
{
    PyObject *out = PyTuple_New(sizeof...(T));
    if (!out) return nullptr;
    Py_ssize_t i = 0;
    bool ok = true;
    std::apply(
        [&](auto &...t) {
            (([&] {
                 PyObject *o = ok ? THPVariable_Wrap(std::move(t)) : nullptr;
                 ok = ok && o;
                 PyTuple_SET_ITEM(out, i++, o);
             }()),
             ...);
        },
        r);
    if (ok) return out;
    Py_DECREF(out);
    return nullptr;
}

struct NoGil {
    PyThreadState *state = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(state); }
};

template <class F>
struct Op;
template <class R, class... A>
struct Op<R(A...)> {
    static constexpr int kArgs = sizeof...(A);
    c10::TypedOperatorHandle<R(A...)> handle;
    std::array<PyObject *, kArgs> names{};                 // interned
    std::vector<c10::IValue> defaults;
    int positional = 0;
    PyObject *packet_call = nullptr;                       // the packet type's own __call__

    explicit Op(const char *name) : handle(c10::Dispatcher::singleton().findSchemaOrThrow(name, "").template typed<R(A...)>())
    {
        const auto &args = handle.schema().arguments();
        TORCH_CHECK((int)args.size() == kArgs, name, ": the schema and the typed call differ");
        for (int i = 0; i < kArgs; i++) {
            names[i] = PyUnicode_InternFromString(args[i].name().c_str());
            defaults.push_back(args[i].default_value().value_or(c10::IValue(std::string("none"))));
            if (!args[i].kwarg_only()) positional = i + 1;
        }
    }

    template <size_t... I>
    bool load(std::tuple<Arg<A>...> &v, const std::array<PyObject *, kArgs> &slot, std::index_sequence<I...>) const
    {
        return ((slot[I] ? std::get<I>(v).load(slot[I]) : std::get<I>(v).load_default(defaults[I])) && ...);
    }
    template <size_t... I>
    R invoke(const std::tuple<Arg<A>...> &v, std::index_sequence<I...>) const
    {
        return handle.call(std::get<I>(v).get()...);
    }

    PyObject *fall_back(PyObject *self, PyObject *args, PyObject *kwargs) const
    {
        const Py_ssize_t n = PyTuple_GET_SIZE(args);
        PyObject *with_self = PyTuple_New(n + 1);
        if (!with_self) return nullptr;
        Py_INCREF(self);
        PyTuple_SET_ITEM(with_self, 0, self);
        for (Py_ssize_t i = 0; i < n; i++) {
            PyObject *a = PyTuple_GET_ITEM(args, i);
            Py_INCREF(a);
            PyTuple_SET_ITEM(with_self, i + 1, a);
        }
        PyObject *r = PyObject_Call(packet_call, with_self, kwargs);
        Py_DECREF(with_self);
        return r;
    }

    PyObject *call(PyObject *self, PyObject *args, PyObject *kwargs) const
    {
        HANDLE_TH_ERRORS
        std::array<PyObject *, kArgs> slot{};
        const Py_ssize_t n = PyTuple_GET_SIZE(args);
        bool fits = n <= positional && !at::impl::torch_function_mode_enabled() && !torch::jit::tracer::isTracing();
        for (Py_ssize_t i = 0; fits && i < n; i++) slot[i] = PyTuple_GET_ITEM(args, i);
        if (fits && kwargs) {
            PyObject *key, *value;
            Py_ssize_t pos = 0;
            while (fits && PyDict_Next(kwargs, &pos, &key, &value)) {
                int at = -1;
                for (int i = (int)n; i < kArgs; i++)
                    if (names[i] == key) at = i;           // keyword names in code are interned
                fits = at >= 0;
                if (fits) slot[at] = value;
            }
        }
        std::tuple<Arg<A>...> v;
        constexpr auto each = std::index_sequence_for<A...>{};
        if (!fits || !load(v, slot, each)) return fall_back(self, args, kwargs);
        std::optional<R> r;
        {
            NoGil no_gil;
            r.emplace(invoke(v, each));
        }
        return to_python(std::move(*r));
        END_HANDLE_TH_ERRORS
    }
};

// One operator = one Python type (a subclass of the packet's type that adds nothing but the call slot).
template <class Tag, class F>
PyObject *slot_call(PyObject *self, PyObject *args, PyObject *kwargs);
template <class Tag, class F>
Op<F> *&op_of()
{
    static Op<F> *op = nullptr;
    return op;
}
template <class Tag, class F>
PyObject *slot_call(PyObject *self, PyObject *args, PyObject *kwargs)
{
    return op_of<Tag, F>()->call(self, args, kwargs);
}

template <class Tag, class F>
bool install_one(PyObject *namespace_, const char *name)
{
    PyObject *packet = PyObject_GetAttrString(namespace_, name);
    if (!packet) return false;
    bool ok = false;
    PyTypeObject *base = Py_TYPE(packet);
    if (!op_of<Tag, F>()) {
        Op<F> *op = new Op<F>((std::string("npu::") + name).c_str());
        op->packet_call = PyObject_GetAttrString(reinterpret_cast<PyObject *>(base), "__call__");
        if (!op->packet_call) return false;
        op_of<Tag, F>() = op;
        PyType_Slot slots[] = {{Py_tp_call, reinterpret_cast<void *>(&slot_call<Tag, F>)}, {0, nullptr}};
        PyType_Spec spec = {"torch._ops.OpOverloadPacket", 0, 0, Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE, slots};
        PyObject *bases = PyTuple_Pack(1, reinterpret_cast<PyObject *>(base));
        PyObject *type = bases ? PyType_FromSpecWithBases(&spec, bases) : nullptr;
        Py_XDECREF(bases);
        ok = type && PyObject_SetAttrString(packet, "__class__", type) == 0;
        Py_XDECREF(type);
    } else {
        ok = true;
    }
    Py_DECREF(packet);
    return ok;
}

using DynQuant = std::tuple<Tensor, Tensor>(const Tensor &, const OptTensor &, const OptTensor &, OptType);
using DynQuantAsym = std::tuple<Tensor, Tensor, Tensor>(const Tensor &, const OptTensor &, const OptTensor &, OptType);
using QuantMatmul = Tensor(const Tensor &, const Tensor &, const Tensor &, const OptTensor &, const OptTensor &, const OptTensor &, OptType);
using WeightQuant = Tensor(const Tensor &, const Tensor &, const Tensor &, const OptTensor &, const OptTensor &, const OptTensor &,
                           const OptTensor &, int64_t, int64_t, OptType);
using Swiglu = Tensor(const Tensor &, int64_t);
using SwigluQuant = std::tuple<Tensor, Tensor>(const Tensor &, const OptTensor &, const OptTensor &, const OptTensor &, bool, int64_t, int64_t,
                                               OptType);
using AntiQuant = Tensor(const Tensor &, const Tensor &, const OptTensor &, OptType, OptType);
using TransParam = Tensor(const Tensor &, const OptTensor &);
using Quantize = Tensor(const Tensor &, const Tensor &, const OptTensor &, at::ScalarType, int64_t, bool);

// ---- forward passes of the contrib modules.  A module stores [out_features, in_features] weights and [N, G] parameters and the
// operator takes their transposed views; forming three views and looking up every parameter in Python takes longer than the
// launch.  These calls, for weights on the GPU, form the views here; they return NotImplemented for what the module's Python code has to
// handle.

bool usable(const Tensor &t) { return !t.requires_grad(); }
bool usable(const OptTensor &t) { return !t || !t->requires_grad(); }
// (the views never leave the call, so no autograd view tracking is needed)
Tensor transposed(const Tensor &t) { return t.transpose(-2, -1); }
Tensor group_major(const Tensor &t) { return t.dim() == 2 ? t.transpose(-2, -1) : t; }
bool plain_call(Py_ssize_t nargs, Py_ssize_t want) { return nargs == want && !at::impl::torch_function_mode_enabled() && !torch::jit::tracer::isTracing(); }
PyObject *not_implemented() { Py_RETURN_NOTIMPLEMENTED; }

// linear_quant(x, weight [N, K], scale, offset, pertoken_scale, bias, output_dtype)
PyObject *linear_quant(PyObject *, PyObject *const *args, Py_ssize_t nargs)
{
    HANDLE_TH_ERRORS
    static const Op<QuantMatmul> op("npu::npu_quant_matmul");
    Arg<const Tensor &> x, w, scale;
    Arg<const OptTensor &> offset, ps, bias;
    Arg<OptType> dt;
    if (!plain_call(nargs, 7) || !x.load(args[0]) || !w.load(args[1]) || !scale.load(args[2]) || !offset.load(args[3]) || !ps.load(args[4]) ||
        !bias.load(args[5]) || !dt.load(args[6]) || w.get().dim() < 2 || !w.get().is_cuda() || !usable(w.get()))
        return not_implemented();
    Tensor r;
    {
        NoGil no_gil;
        Tensor wt;
        {
            at::AutoDispatchBelowADInplaceOrView below;
            wt = transposed(w.get());
        }
        r = op.handle.call(x.get(), wt, scale.get(), offset.get(), ps.get(), bias.get(), dt.get());
    }
    return to_python(std::move(r));
    END_HANDLE_TH_ERRORS
}

// linear_weight_quant(x, weight [N, K] or [N, K / 8], scale, offset, quant_scale, quant_offset, bias, group_size, inner_precise)
PyObject *linear_weight_quant(PyObject *, PyObject *const *args, Py_ssize_t nargs)
{
    HANDLE_TH_ERRORS
    static const Op<WeightQuant> op("npu::npu_weight_quant_batchmatmul");
    Arg<const Tensor &> x, w, scale;
    Arg<const OptTensor &> offset, qs, qo, bias;
    Arg<int64_t> group, inner;
    if (!plain_call(nargs, 9) || !x.load(args[0]) || !w.load(args[1]) || !scale.load(args[2]) || !offset.load(args[3]) || !qs.load(args[4]) ||
        !qo.load(args[5]) || !bias.load(args[6]) || !group.load(args[7]) || !inner.load(args[8]) || w.get().dim() < 2 || !w.get().is_cuda() ||
        !usable(w.get()) || !usable(scale.get()) || !usable(offset.get()))
        return not_implemented();
    Tensor r;
    {
        NoGil no_gil;
        Tensor wt, st;
        OptTensor ot;
        {
            at::AutoDispatchBelowADInplaceOrView below;
            wt = transposed(w.get());
            st = group_major(scale.get());
            if (offset.get()) ot = group_major(*offset.get());
        }
        r = op.handle.call(x.get(), wt, st, ot, qs.get(), qo.get(), bias.get(), group.get(), inner.get(), std::nullopt);
    }
    return to_python(std::move(r));
    END_HANDLE_TH_ERRORS
}

PyObject *install(PyObject *, PyObject *args)
{
    HANDLE_TH_ERRORS
    PyObject *namespace_;
    if (!PyArg_ParseTuple(args, "OO!", &namespace_, &PyType_Type, &parameter_type)) return nullptr;
    Py_INCREF(parameter_type);
    const bool ok = install_one<struct T0, DynQuant>(namespace_, "npu_dynamic_quant") &&
                    install_one<struct T1, DynQuantAsym>(namespace_, "npu_dynamic_quant_asymmetric") &&
                    install_one<struct T2, QuantMatmul>(namespace_, "npu_quant_matmul") &&
                    install_one<struct T3, WeightQuant>(namespace_, "npu_weight_quant_batchmatmul") &&
                    install_one<struct T4, Swiglu>(namespace_, "npu_swiglu") &&
                    install_one<struct T5, SwigluQuant>(namespace_, "npu_swiglu_quant") &&
                    install_one<struct T6, AntiQuant>(namespace_, "npu_anti_quant") &&
                    install_one<struct T7, TransParam>(namespace_, "npu_trans_quant_param") &&
                    install_one<struct T8, Quantize>(namespace_, "npu_quantize");
    if (!ok) return nullptr;
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {{"install", install, METH_VARARGS, "install(torch.ops.npu, torch.nn.Parameter): direct calls for the operators' packets"},
                         {"linear_quant", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(&linear_quant)), METH_FASTCALL, "forward of LinearQuant"},
                         {"linear_weight_quant", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(&linear_weight_quant)), METH_FASTCALL,
                          "forward of LinearWeightQuant"},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_op_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__op_call() { return PyModule_Create(&module_def); }
