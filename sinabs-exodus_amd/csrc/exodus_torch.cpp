// The host side of the kernel calls in native code: what a call checks, allocates and hands to the C ABI of
// libexodus_hip.so, between the Python wrappers of _hip.py and the library.  No device code and no state: the library's
// entry points are bound once at import (bind), the current stream and device are asked for in every call.
//
// Why it exists: a training step of a small layer is host time, and the autograd engine runs the backward pass on a thread
// of its own, where the 55 us of Python and ctypes that a backward pass was took up to 165 (caches and a core of its own).
// Python and ctypes / the calls in native code / the layers' nodes as well (LifLayer, LeakyLayer below), us per step through the layer,
// forward and backward: IAF (8, 100, 256) 238 / 149 / 96, LIF (32, 100, 512) with a trained time constant 271 / 173 / 113, a streamed
// chunk (1, 10, 1024) without gradients, which has no node, 47 / 24 / 21.
#include <ATen/Functions.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <pybind11/pybind11.h>
#include <pybind11/stl.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <cstring>
#include <optional>
#include <stdexcept>
#include <string>
#include <tuple>
#include <vector>

#include "exodus_hip.h"

namespace py = pybind11;

namespace {

using at::Tensor;
using Maybe = std::optional<Tensor>;
using Shape = std::vector<int64_t>;
// results of a call, None in Python where undefined
using Two = std::tuple<Tensor, Tensor>;
using Three = std::tuple<Tensor, Tensor, Tensor>;
using Five = std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor>;
using Eight = std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor>;

// ---------------------------------------------------------------------------------------------
// the library
// ---------------------------------------------------------------------------------------------
#define EXODUS_ENTRIES(X)                                                                                               \
    X(exodus_hip_abi_version)                                                                                           \
    X(exodus_lif_forward) X(exodus_lif_backward_fused) X(exodus_leaky_forward) X(exodus_leaky_backward_fused)           \
    X(exodus_layer_sum_slots) X(exodus_layer_checkpoint_interval) X(exodus_layer_lif_forward_decays)                    \
    X(exodus_layer_lif_backward) X(exodus_layer_lif_backward_from_input) X(exodus_layer_leaky_forward_decays)            \
    X(exodus_layer_leaky_backward) X(exodus_decay_expand) X(exodus_decay_work) X(exodus_decay_grad)
struct Library {
#define EXODUS_MEMBER(name) decltype(&::name) name = nullptr;
    EXODUS_ENTRIES(EXODUS_MEMBER)
#undef EXODUS_MEMBER
};
Library lib;
int64_t interval = 0;                                          // steps between checkpoints
PyObject *raise_status = nullptr;                              // (status, what): raises for a status other than 0
PyObject *place_of = nullptr;                                  // (like): what allocates large results (see `large`), or None

// on_place: what `place_of` is, for the layers' nodes; None keeps what an earlier call gave
void bind(const py::dict &addresses, const py::object &on_status, const py::object &on_place)
{
    Library given;
#define EXODUS_BIND(name) \
    given.name = reinterpret_cast<decltype(given.name)>(py::cast<uintptr_t>(addresses[#name]));
    EXODUS_ENTRIES(EXODUS_BIND)
#undef EXODUS_BIND
    const int version = given.exodus_hip_abi_version();        // the signatures above are those of one version of the header
    if (version != EXODUS_HIP_ABI_VERSION)
        throw py::import_error("the library has ABI version " + std::to_string(version) + ", _exodus_torch was built for " +
                               std::to_string(EXODUS_HIP_ABI_VERSION));
    lib = given;
    interval = lib.exodus_layer_checkpoint_interval();
    Py_XDECREF(raise_status);
    raise_status = py::object(on_status).release().ptr();
    if (on_place.is_none()) return;
    Py_XDECREF(place_of);
    place_of = py::object(on_place).release().ptr();
}

// call a function of the library on the tensor's device and stream
template <class F>
void launch(const Tensor &like, const char *what, F &&call)
{
    int status;
    {
        const c10::DeviceGuard guard(like.device());
        status = call(static_cast<void *>(c10::hip::getCurrentHIPStream(like.device().index()).stream()));
    }
    if (status != 0) {
        py::gil_scoped_acquire locked;
        py::reinterpret_borrow<py::object>(raise_status)(status, what);
    }
}

// ---------------------------------------------------------------------------------------------
// checks
// ---------------------------------------------------------------------------------------------
std::string text(c10::IntArrayRef sizes)
{
    std::string s = "(";
    for (size_t i = 0; i < sizes.size(); ++i) s += (i ? ", " : "") + std::to_string(sizes[i]);
    return s + (sizes.size() == 1 ? ",)" : ")");
}

[[noreturn]] void refuse(const std::string &why) { throw std::runtime_error(why); }

const Tensor &dev(const Tensor &x, const char *name, const Tensor *like = nullptr)
{
    if (!x.is_cuda())
        refuse(std::string(name) + " must be a tensor on a HIP device (got " + x.device().str() + "); there is no CPU path");
    if (x.scalar_type() != at::kFloat) {
        py::gil_scoped_acquire locked;
        refuse(std::string(name) + " must be float32 (got " + std::string(py::str(py::cast(x).attr("dtype"))) + ")");
    }
    if (!x.is_contiguous()) refuse(std::string(name) + " must be contiguous");
    if (like && x.device() != like->device()) refuse(std::string(name) + " and the first tensor must be on the same device");
    return x;
}

const float *rows(const Tensor &x, const char *name, const Tensor &like, int64_t n)
{
    dev(x, name, &like);
    if (x.dim() != 1 || x.size(0) != n)
        refuse(std::string(name) + " must have shape (" + std::to_string(n) + ",), got " + text(x.sizes()));
    return x.const_data_ptr<float>();
}

const Tensor &present(const Maybe &x, const char *name)
{
    if (!x || !x->defined()) throw py::type_error(std::string(name) + " must be a tensor");
    return *x;
}

const float *rows(const Maybe &x, const char *name, const Tensor &like, int64_t n)
{
    return rows(present(x, name), name, like, n);
}

const float *same(const Tensor &x, const char *name, const Tensor &like, const char *as)
{
    dev(x, name, &like);
    if (x.sizes() != like.sizes()) refuse(std::string(name) + " must have the shape of " + as);
    return x.const_data_ptr<float>();
}

const float *matrix(const Tensor &x, const char *name, const Tensor &like, int64_t n, int64_t t)
{
    dev(x, name, &like);
    if (x.dim() != 2 || x.size(0) != n || x.size(1) != t)
        refuse(std::string(name) + " must have shape (" + std::to_string(n) + ", " + std::to_string(t) + "), got " +
               text(x.sizes()));
    return x.const_data_ptr<float>();
}

const Tensor &three(const Tensor &x, const char *name, const Tensor *like = nullptr)
{
    dev(x, name, like);
    if (x.dim() != 3) refuse(std::string(name) + " must be 3-D (batch, time, neurons)");
    return x;
}

const Tensor &two(const Tensor &x, const char *name)
{
    dev(x, name);
    if (x.dim() != 2) refuse(std::string(name) + " must be 2-D (rows, time)");
    return x;
}

bool has(const Maybe &x) { return x && x->defined(); }
float *out(const Tensor &x) { return x.defined() ? x.mutable_data_ptr<float>() : nullptr; }
double *out64(const Tensor &x) { return x.defined() ? x.mutable_data_ptr<double>() : nullptr; }

// ---------------------------------------------------------------------------------------------
// memory
// ---------------------------------------------------------------------------------------------
Tensor fresh(c10::IntArrayRef shape, const Tensor &like, at::ScalarType type = at::kFloat)
{
    return at::empty(shape, at::TensorOptions().device(like.device()).dtype(type));
}

// the (batch, time, neurons) and (rows, time) results: `place`, if given, allocates them (shape, like)
Tensor large(c10::IntArrayRef shape, const Tensor &like, const py::handle place)
{
    if (place.is_none()) return fresh(shape, like);
    py::gil_scoped_acquire locked;
    return py::cast<Tensor>(place(py::cast(Shape(shape.begin(), shape.end())), like));
}

int64_t elements(const Shape &shape)
{
    int64_t n = 1;
    for (int64_t s : shape) n *= s;
    return n;
}

// a float64 scalar for the sum of a forward call's outputs and the memory the kernels add it up in; both are written by the
// call (which launches nothing, and leaves the total as it is, when there is nothing to walk)
void total_and_work(const Tensor &input, Tensor &total, Tensor &work)
{
    if (input.numel() == 0) {
        total = at::zeros({}, at::TensorOptions().device(input.device()).dtype(at::kDouble));
        return;
    }
    total = fresh({}, input, at::kDouble);
    work = fresh({lib.exodus_layer_sum_slots(input.size(0), input.size(2))}, input, at::kDouble);
}

Shape state_shape_of(const std::optional<Shape> &asked, int64_t n)
{
    if (!asked) return {n};
    if (elements(*asked) != n)
        refuse("stateShape " + text(*asked) + " does not hold " + std::to_string(n) + " neurons");
    return *asked;
}

// ---------------------------------------------------------------------------------------------
// layers on (batch, time, neurons)
// ---------------------------------------------------------------------------------------------
// time constants whose decay factors the forward kernel works out (`decays`) into alpha_mem / alpha_syn
Eight layer_lif_forward_decays(const exodus_layer_decays *decays, const Tensor &input, const Tensor &v_init, const Maybe &i_init,
                            const Tensor &alpha_mem,
                            const Maybe &alpha_syn, const Tensor &subtract, const Tensor &theta, const Maybe &theta_low,
                            bool apply_low, int64_t max_spikes, bool decay_early, bool norm_input, bool want_checkpoints,
                            bool want_records, bool want_pre_reset, bool want_sum, const Maybe &out_spikes,
                            const std::optional<Shape> &state_shape, const py::handle place)
{
    if (want_records && want_pre_reset) refuse("wantRecords and wantPreReset exclude each other");
    three(input, "input");
    const int64_t b = input.size(0), t = input.size(1), m = input.size(2), n = b * m;
    const bool syn = has(alpha_syn);
    const float *v0 = rows(v_init, "vmemPostInitial", input, n), *am = rows(alpha_mem, "alphaMem", input, n);
    const float *c = rows(subtract, "membrSubtract", input, n), *th = rows(theta, "theta", input, n);
    const float *i0 = syn ? rows(i_init, "isynInitial", input, n) : nullptr;
    const float *as = syn ? rows(alpha_syn, "alphaSyn", input, n) : nullptr;
    const float *lo = apply_low ? rows(theta_low, "thetaLow", input, n) : nullptr;
    const Shape shape{b, t, m}, states = state_shape_of(state_shape, n), kept{b, (t + interval - 1) / interval, m};
    Tensor spikes = has(out_spikes) ? *out_spikes : large(shape, input, place);
    if (spikes.sizes() != input.sizes()) refuse("outSpikes must have the shape of input");
    dev(spikes, "outSpikes", &input);
    const Tensor v_last = fresh(states, input), i_last = syn ? fresh(states, input) : Tensor();
    const Tensor ckpt_v = want_checkpoints ? large(kept, input, place) : Tensor();
    const Tensor ckpt_i = want_checkpoints && syn ? large(kept, input, place) : Tensor();
    const Tensor v_rec = want_records || want_pre_reset ? large(shape, input, place) : Tensor();
    const Tensor i_rec = want_records && syn ? large(shape, input, place) : Tensor();
    Tensor total, work;
    if (want_sum) total_and_work(input, total, work);
    if (t == 0) {                                              // nothing to integrate: the final states are the initial ones
        v_last.copy_(v_init.reshape(states));
        if (syn) i_last.copy_(i_init->reshape(states));
    }
    const bool worked_out = decays && (decays->tau_mem || decays->tau_syn);
    launch(input, worked_out ? "exodus_layer_lif_forward_decays" : "exodus_layer_lif_forward_total", [&](void *stream) {
        return lib.exodus_layer_lif_forward_decays(
            out(spikes), out(v_rec), out(i_rec), out(ckpt_v), out(ckpt_i), out(v_last), out(i_last), out64(total), out64(work),
            decays, input.const_data_ptr<float>(), v0, i0, am, as, c, th, lo, apply_low, static_cast<int>(max_spikes), decay_early,
            norm_input, want_pre_reset, b, t, m, stream);
    });
    return {spikes, v_last, i_last, ckpt_v, ckpt_i, v_rec, i_rec, total};
}

Eight layer_lif_forward(const Tensor &input, const Tensor &v_init, const Maybe &i_init, const Tensor &alpha_mem,
                        const Maybe &alpha_syn, const Tensor &subtract, const Tensor &theta, const Maybe &theta_low, bool apply_low,
                        int64_t max_spikes, bool decay_early, bool norm_input, bool want_checkpoints, bool want_records,
                        bool want_pre_reset, bool want_sum, const Maybe &out_spikes, const std::optional<Shape> &state_shape,
                        const py::handle place)
{
    return layer_lif_forward_decays(nullptr, input, v_init, i_init, alpha_mem, alpha_syn, subtract, theta, theta_low, apply_low,
                                    max_spikes, decay_early, norm_input, want_checkpoints, want_records, want_pre_reset, want_sum,
                                    out_spikes, state_shape, place);
}

// -> (grad_input, alpha_mem, alpha_syn, v_init, i_init)
Five layer_lif_backward(const Tensor &grad_spikes, const Maybe &grad_v_last, const Maybe &grad_i_last, const Tensor &input,
                             const Maybe &ckpt_v, const Maybe &ckpt_i, const Maybe &v_init, const Maybe &i_init,
                             const Tensor &alpha_mem, const Maybe &alpha_syn, const Tensor &subtract, const Tensor &theta,
                             const Maybe &theta_low, bool apply_low, int64_t max_spikes, bool decay_early, bool norm_input,
                             int kind, double p0, double p1, const Maybe &grad_input_given, const Maybe &surr_given,
                             Maybe grad_v_rec, Maybe grad_i_rec, bool want_alpha_mem, bool want_alpha_syn, bool want_v_init,
                             bool want_i_init, bool uniform, const py::handle place)
{
    three(input, "input");
    const int64_t b = input.size(0), t = input.size(1), m = input.size(2), n = b * m;
    const bool syn = has(alpha_syn);
    if (uniform) {
        if (dev(grad_spikes, "gradSpikes", &input).numel() != 1)
            refuse("gradSpikes must hold one value when gradUniform is set");
        if (kind == EXODUS_SURR_TENSOR || has(grad_v_rec) || has(grad_i_rec))
            refuse("gradUniform needs an in-kernel surrogate and no gradients on the state records");
    } else {
        same(three(grad_spikes, "gradSpikes", &input), "gradSpikes", input, "input");
    }
    const bool from_input = !has(ckpt_v);
    const Shape shape{b, t, m}, kept{b, (t + interval - 1) / interval, m};
    const auto checkpoint = [&](const Maybe &x, const char *name) {
        if (three(present(x, name), name, &input).sizes() != c10::IntArrayRef(kept))
            refuse(std::string(name) + " must have shape " + text(kept));
        return x->const_data_ptr<float>();
    };
    const float *cv = from_input ? nullptr : checkpoint(ckpt_v, "ckptV");
    const float *ci = from_input || !syn ? nullptr : checkpoint(ckpt_i, "ckptI");
    const float *v0 = rows(v_init, "vmemPostInitial", input, n), *am = rows(alpha_mem, "alphaMem", input, n);
    const float *c = rows(subtract, "membrSubtract", input, n), *th = rows(theta, "theta", input, n);
    const float *i0 = syn ? rows(i_init, "isynInitial", input, n) : nullptr;
    const float *as = syn ? rows(alpha_syn, "alphaSyn", input, n) : nullptr;
    const auto last = [&](const Maybe &x, const char *name) -> const float * {
        if (!has(x)) return nullptr;
        if (dev(*x, name, &input).numel() != n) refuse(std::string(name) + " must hold " + std::to_string(n) + " values");
        return x->const_data_ptr<float>();
    };
    const float *gvl = last(grad_v_last, "gradVLast"), *gil = syn ? last(grad_i_last, "gradILast") : nullptr;
    const float *lo = apply_low ? rows(theta_low, "thetaLow", input, n) : nullptr;
    if (has(grad_input_given)) same(three(*grad_input_given, "gradInput", &input), "gradInput", input, "input");
    const Tensor grad_input = has(grad_input_given) ? *grad_input_given : large(shape, input, place);
    const float *surr = nullptr;
    if (kind == EXODUS_SURR_TENSOR) {
        if (!has(surr_given)) refuse("surr must be given with the shape of input");
        if (three(*surr_given, "surr", &input).sizes() != input.sizes()) refuse("surr must be given with the shape of input");
        surr = surr_given->const_data_ptr<float>();
    }
    if (!syn) grad_i_rec.reset();
    const float *gvr = nullptr, *gir = nullptr;
    if (has(grad_v_rec) || has(grad_i_rec)) {                  // one that is missing while the other is given counts as zero
        if (!has(grad_v_rec)) grad_v_rec = at::zeros_like(input);
        if (syn && !has(grad_i_rec)) grad_i_rec = at::zeros_like(input);
        gvr = same(three(*grad_v_rec, "gradVRec", &input), "gradVRec", input, "input");
        if (syn) gir = same(three(*grad_i_rec, "gradIRec", &input), "gradIRec", input, "input");
    }
    // the kernel writes every neuron's entry of each vector it is given -- unless there is no step to walk: then nothing is
    // launched, the decay factors have no influence and a gradient on a final state is the gradient of the initial state it
    // equals (the wanted vectors are rows of one allocation)
    const bool wanted[4] = {want_alpha_mem, want_v_init, syn && want_alpha_syn, syn && want_i_init};
    const int64_t many = wanted[0] + wanted[1] + wanted[2] + wanted[3];
    Tensor block, vectors[4];
    if (many) {
        block = t == 0 ? at::zeros({many, n}, input.options()) : fresh({many, n}, input);
        for (int64_t k = 0, at = 0; k < 4; ++k)
            if (wanted[k]) vectors[k] = block.select(0, at++);
    }
    const Tensor &am_g = vectors[0], &v0_g = vectors[1], &as_g = vectors[2], &i0_g = vectors[3];
    if (t == 0) {
        if (v0_g.defined() && gvl) v0_g.copy_(grad_v_last->reshape({-1}));
        if (i0_g.defined() && gil) i0_g.copy_(grad_i_last->reshape({-1}));
    }
    const float *x = input.const_data_ptr<float>(), *gs = grad_spikes.const_data_ptr<float>();
    const int spikes = static_cast<int>(max_spikes);
    const float f0 = static_cast<float>(p0), f1 = static_cast<float>(p1);
    if (from_input)
        launch(input, "exodus_layer_lif_backward_from_input", [&](void *stream) {
            return lib.exodus_layer_lif_backward_from_input(
                out(grad_input), out(am_g), out(as_g), out(v0_g), out(i0_g), gs, gvl, gil, x, v0, i0, am, as, c, th, lo,
                apply_low, spikes, decay_early, norm_input, kind, f0, f1, surr, gvr, gir, uniform, b, t, m, stream);
        });
    else
        launch(input, "exodus_layer_lif_backward", [&](void *stream) {
            return lib.exodus_layer_lif_backward(
                out(grad_input), out(am_g), out(as_g), out(v0_g), out(i0_g), gs, gvl, gil, x, cv, ci, v0, i0, am, as, c, th, lo,
                apply_low, spikes, decay_early, norm_input, kind, f0, f1, surr, gvr, gir, uniform, b, t, m, stream);
        });
    return {grad_input, am_g, as_g, v0_g, i0_g};
}

// -> (out, v_last, total)
Three layer_leaky_forward_decays(const exodus_layer_decays *decays, const Tensor &input, const Tensor &v_init, const Tensor &alpha,
                              bool decay_early, bool norm_input, const std::optional<Shape> &state_shape, bool want_sum,
                              const py::handle place)
{
    three(input, "input");
    const int64_t b = input.size(0), t = input.size(1), m = input.size(2), n = b * m;
    const float *v0 = rows(v_init, "vmemInitial", input, n), *a = rows(alpha, "alpha", input, n);
    const Shape shape{b, t, m}, states = state_shape_of(state_shape, n);
    const Tensor result = large(shape, input, place), v_last = fresh(states, input);
    Tensor total, work;
    if (want_sum) total_and_work(input, total, work);
    if (t == 0) v_last.copy_(v_init.reshape(states));
    const bool worked_out = decays && decays->tau_mem;
    launch(input, worked_out ? "exodus_layer_leaky_forward_decays" : "exodus_layer_leaky_forward_total", [&](void *stream) {
        return lib.exodus_layer_leaky_forward_decays(out(result), out(v_last), out64(total), out64(work), decays,
                                                     input.const_data_ptr<float>(), v0, a, decay_early, norm_input, b, t, m,
                                                     stream);
    });
    return {result, v_last, total};
}

Three layer_leaky_forward(const Tensor &input, const Tensor &v_init, const Tensor &alpha, bool decay_early, bool norm_input,
                          const std::optional<Shape> &state_shape, bool want_sum, const py::handle place)
{
    return layer_leaky_forward_decays(nullptr, input, v_init, alpha, decay_early, norm_input, state_shape, want_sum, place);
}

// -> (grad_input, alpha, v_init)
Three layer_leaky_backward(const Tensor &grad_out, const Maybe &grad_v_last, const Maybe &forward_out, const Maybe &input,
                               const Maybe &v_init, const Tensor &alpha, bool decay_early, bool norm_input, bool want_alpha,
                               const std::optional<Shape> &uniform_shape, const py::handle place)
{
    const bool uniform = uniform_shape.has_value();
    Shape shape;
    if (uniform) {
        if (dev(grad_out, "gradOut").numel() != 1) refuse("gradOut must hold one value when shape is given");
        shape = *uniform_shape;
        if (shape.size() != 3) throw py::value_error("shape must be (batch, time, neurons)");
    } else {
        three(grad_out, "gradOut");
        shape = grad_out.sizes().vec();
    }
    const int64_t b = shape[0], t = shape[1], m = shape[2], n = b * m;
    const float *a = rows(alpha, "alpha", grad_out, n);
    const float *gvl = nullptr;
    if (has(grad_v_last)) {
        if (dev(*grad_v_last, "gradVLast", &grad_out).numel() != n)
            refuse("gradVLast must hold " + std::to_string(n) + " values");
        gvl = grad_v_last->const_data_ptr<float>();
    }
    const auto full = [&](const Maybe &x, const char *name) {
        if (three(present(x, name), name, &grad_out).sizes() != c10::IntArrayRef(shape))
            refuse(std::string(name) + " must have the shape of gradOut");
        return x->const_data_ptr<float>();
    };
    const float *o = want_alpha ? full(forward_out, "out") : nullptr;
    const float *v0 = want_alpha ? rows(v_init, "vmemInitial", grad_out, n) : nullptr;
    const float *x = want_alpha && (decay_early || norm_input) ? full(input, "input") : nullptr;
    const Tensor grad_input = large(shape, grad_out, place);
    const int64_t many = want_alpha ? 2 : 1;
    const Tensor block = t == 0 ? at::zeros({many, n}, grad_out.options()) : fresh({many, n}, grad_out);
    const Tensor v0_g = block.select(0, 0), a_g = want_alpha ? block.select(0, 1) : Tensor();
    if (t == 0 && gvl) v0_g.copy_(grad_v_last->reshape({-1}));
    launch(grad_out, "exodus_layer_leaky_backward", [&](void *stream) {
        return lib.exodus_layer_leaky_backward(out(grad_input), out(a_g), out(v0_g), grad_out.const_data_ptr<float>(), gvl, o, x,
                                               v0, a, decay_early, norm_input, uniform, b, t, m, stream);
    });
    return {grad_input, a_g, v0_g};
}

// -> (alpha, copy of tau)
Two decay_expand(const Tensor &tau, int64_t batch, int64_t neurons)
{
    dev(tau, "tau");
    const Tensor alpha = fresh({batch * neurons}, tau), kept = fresh(tau.sizes(), tau);
    launch(tau, "exodus_decay_expand", [&](void *stream) {
        return lib.exodus_decay_expand(out(alpha), out(kept), tau.const_data_ptr<float>(), batch, neurons, tau.numel(), stream);
    });
    return {alpha, kept};
}

Tensor decay_grad(const Tensor &grad_alpha, const Tensor &tau, int64_t batch, int64_t neurons)
{
    const float *g = rows(grad_alpha, "gradAlpha", dev(tau, "tau"), batch * neurons);
    if (batch * neurons == 0) return at::zeros_like(tau);
    const Tensor result = fresh(tau.sizes(), tau);
    const int64_t wanted = lib.exodus_decay_work(batch, neurons, tau.numel());
    const Tensor work = wanted ? fresh({wanted}, tau, at::kDouble) : Tensor();
    launch(tau, "exodus_decay_grad", [&](void *stream) {
        return lib.exodus_decay_grad(out(result), out64(work), g, tau.const_data_ptr<float>(), batch, neurons, tau.numel(),
                                     stream);
    });
    return result;
}

// ---------------------------------------------------------------------------------------------
// what shows that a layer's parameters are the ones of the call before
// ---------------------------------------------------------------------------------------------
// An entry stands for a value at one moment: a tensor's holds the tensor itself, its version and a detached alias, so neither
// its object nor its memory can be given to another tensor while the entry is alive; a number's is its float.
bool unchanged(PyObject *entry, PyObject *value)
{
    if (THPVariable_Check(value)) {
        if (!PyTuple_CheckExact(entry) || PyTuple_GET_ITEM(entry, 0) != value) return false;
        const Tensor &x = THPVariable_Unpack(value), &alias = THPVariable_Unpack(PyTuple_GET_ITEM(entry, 2));
        return PyLong_AsLongLong(PyTuple_GET_ITEM(entry, 1)) == x._version() && alias.const_data_ptr() == x.const_data_ptr() &&
               alias.sizes() == x.sizes() && alias.strides() == x.strides();
    }
    if (value == Py_None) return entry == Py_None;
    if (!PyFloat_CheckExact(entry)) return false;
    const py::object number = py::reinterpret_steal<py::object>(PyNumber_Float(value));
    if (!number) {
        PyErr_Clear();
        return false;
    }
    const double was = PyFloat_AS_DOUBLE(entry), is = PyFloat_AS_DOUBLE(number.ptr());
    return std::memcmp(&was, &is, sizeof was) == 0;            // bits: a number that is none is itself, -0 is not 0
}

py::object entry_of(PyObject *value)
{
    if (THPVariable_Check(value)) {
        const Tensor &x = THPVariable_Unpack(value);
        return py::make_tuple(py::reinterpret_borrow<py::object>(value), static_cast<int64_t>(x._version()), x.detach());
    }
    if (value == Py_None) return py::none();
    py::object number = py::reinterpret_steal<py::object>(PyNumber_Float(value));
    if (number) return number;
    PyErr_Clear();                                             // what is no number is never the same again
    return py::reinterpret_steal<py::object>(PyObject_CallNoArgs(reinterpret_cast<PyObject *>(&PyBaseObject_Type)));
}

// One entry per value.  `kept` is what an earlier call returned, or None: its entries are handed on for the values that have not
// changed since, and it is returned itself if none has.
py::object stamps(const py::object &kept, const py::tuple &values)
{
    const size_t n = values.size();
    const bool comparable = PyTuple_CheckExact(kept.ptr()) && static_cast<size_t>(PyTuple_GET_SIZE(kept.ptr())) == n;
    size_t same = 0;
    if (comparable)
        while (same < n && unchanged(PyTuple_GET_ITEM(kept.ptr(), same), values[same].ptr())) ++same;
    if (comparable && same == n) return kept;
    py::tuple result(n);
    for (size_t k = 0; k < n; ++k) {
        PyObject *const was = comparable ? PyTuple_GET_ITEM(kept.ptr(), k) : nullptr, *const value = values[k].ptr();
        result[k] = was && (k < same || (k > same && unchanged(was, value))) ? py::reinterpret_borrow<py::object>(was)
                                                                             : entry_of(value);
    }
    return std::move(result);
}

// ---------------------------------------------------------------------------------------------
// (rows, time) matrices
// ---------------------------------------------------------------------------------------------
void lif_forward(const Tensor &spikes, const Tensor &v_mem, const Tensor &input, const Tensor &v_init, const Tensor &alpha,
                 const Tensor &subtract, const Tensor &theta, const Maybe &theta_low, bool apply_low, int64_t max_spikes)
{
    two(input, "input");
    const int64_t n = input.size(0), t = input.size(1);
    matrix(spikes, "outputSpikes", input, n, t);
    matrix(v_mem, "vmem", input, n, t);
    const float *v0 = rows(v_init, "vmemPostInitial", input, n), *a = rows(alpha, "alpha", input, n);
    const float *c = rows(subtract, "membrSubtract", input, n), *th = rows(theta, "theta", input, n);
    const float *lo = apply_low ? rows(theta_low, "thetaLow", input, n) : nullptr;
    launch(input, "exodus_lif_forward", [&](void *stream) {
        return lib.exodus_lif_forward(out(spikes), out(v_mem), input.const_data_ptr<float>(), v0, a, c, th, lo, apply_low,
                                      static_cast<int>(max_spikes), n, t, stream);
    });
}

// the per-row gradients of a backward call (every entry is written if there is a step to walk)
Tensor per_row(const Tensor &alpha, int64_t n, int64_t t)
{
    return n == 0 || t == 0 ? at::zeros_like(alpha) : fresh(alpha.sizes(), alpha);
}

// -> (grad_input, alpha, v_init)
Three lif_backward_fused(const Tensor &grad_spikes, const Maybe &grad_vmem, const Tensor &v_mem, const Maybe &v_init,
                             const Tensor &alpha, const Tensor &subtract, const Tensor &theta, const Maybe &theta_low,
                             bool apply_low, int64_t max_spikes, int kind, double p0, double p1, const Maybe &surr_given,
                             bool want_alpha, const Maybe &grad_input_given, const py::handle place)
{
    two(v_mem, "vmem");
    const int64_t n = v_mem.size(0), t = v_mem.size(1);
    const float *gs = matrix(grad_spikes, "gradSpikes", v_mem, n, t);
    const float *gv = has(grad_vmem) ? matrix(*grad_vmem, "gradVmem", v_mem, n, t) : nullptr;
    const float *a = rows(alpha, "alpha", v_mem, n), *c = rows(subtract, "membrSubtract", v_mem, n);
    const float *th = rows(theta, "theta", v_mem, n);
    const float *lo = apply_low ? rows(theta_low, "thetaLow", v_mem, n) : nullptr;
    const float *v0 = want_alpha ? rows(v_init, "vmemPostInitial", v_mem, n) : nullptr;
    const float *surr = kind == EXODUS_SURR_TENSOR ? matrix(present(surr_given, "surr"), "surr", v_mem, n, t) : nullptr;
    if (has(grad_input_given)) matrix(*grad_input_given, "inputGrad", v_mem, n, t);
    const Tensor grad_input = has(grad_input_given) ? *grad_input_given : large(v_mem.sizes(), v_mem, place);
    const Tensor v0_g = per_row(alpha, n, t), a_g = want_alpha ? per_row(alpha, n, t) : Tensor();
    launch(v_mem, "exodus_lif_backward_fused", [&](void *stream) {
        return lib.exodus_lif_backward_fused(out(grad_input), out(a_g), out(v0_g), gs, gv, v_mem.const_data_ptr<float>(), surr, v0,
                                             a, c, th, lo, apply_low, static_cast<int>(max_spikes), kind,
                                             static_cast<float>(p0), static_cast<float>(p1), n, t, stream);
    });
    return {grad_input, a_g, v0_g};
}

Tensor leaky_forward(const Tensor &input, const Tensor &v_init, const Tensor &alpha, const Maybe &given, const py::handle place)
{
    two(input, "input");
    const int64_t n = input.size(0), t = input.size(1);
    const float *v0 = rows(v_init, "vmemInitial", input, n), *a = rows(alpha, "alpha", input, n);
    if (has(given)) matrix(*given, "output", input, n, t);
    const Tensor result = has(given) ? *given : large(input.sizes(), input, place);
    launch(input, "exodus_leaky_forward", [&](void *stream) {
        return lib.exodus_leaky_forward(out(result), input.const_data_ptr<float>(), v0, a, n, t, stream);
    });
    return result;
}

// -> (grad_input, alpha, v_init)
Three leaky_backward_fused(const Tensor &grad_out, const Tensor &alpha, const Maybe &forward_out, const Maybe &v_init,
                               bool want_alpha, const Maybe &grad_input_given, const py::handle place)
{
    two(grad_out, "outputGrad");
    const int64_t n = grad_out.size(0), t = grad_out.size(1);
    const float *a = rows(alpha, "alpha", grad_out, n);
    const float *o = want_alpha ? matrix(present(forward_out, "output"), "output", grad_out, n, t) : nullptr;
    const float *v0 = want_alpha ? rows(v_init, "vmemInitial", grad_out, n) : nullptr;
    if (has(grad_input_given)) matrix(*grad_input_given, "inputGrad", grad_out, n, t);
    const Tensor grad_input = has(grad_input_given) ? *grad_input_given : large(grad_out.sizes(), grad_out, place);
    const Tensor v0_g = per_row(alpha, n, t), a_g = want_alpha ? per_row(alpha, n, t) : Tensor();
    launch(grad_out, "exodus_leaky_backward_fused", [&](void *stream) {
        return lib.exodus_leaky_backward_fused(out(grad_input), out(a_g), out(v0_g), grad_out.const_data_ptr<float>(), o, v0, a, n,
                                               t, stream);
    });
    return {grad_input, a_g, v0_g};
}

// ---------------------------------------------------------------------------------------------
// layers as nodes of the autograd graph
// ---------------------------------------------------------------------------------------------
// What layer_function.py's two Functions do, for the calls that need no Python on the way back (a surrogate that the kernels
// know): the same tensors saved in the same order, the same gradients.  The engine runs a backward pass on a thread of its own,
// where Python means the interpreter lock, cold caches and thirteen unpacked tensors; and the input's shape is taken and given
// back here instead of by reshapes that are nodes of their own.  us per training step with Python Functions and with these nodes (and the
// kernels that came with them): IAF (8, 100, 256) 134 / 96, LIF (32, 100, 512) with a trained time constant 154 / 113, LIF with synapses
// (4, 2000, 512), both constants trained, 194 / 139; with the constants written to between the steps, as an optimizer does, 216 / 180
// and 263 / 222 (with the same write to other tensors 179 / 136 and 225 / 174).
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// the tensor in another shape, for the calls above and as a result of a node: no view in autograd's books
Tensor shaped(const Tensor &x, c10::IntArrayRef shape) { return x.sizes() == shape ? x : at::_unsafe_view(x, shape); }
Maybe shaped(const Maybe &x, c10::IntArrayRef shape) { return has(x) ? Maybe(shaped(*x, shape)) : Maybe(); }

Shape three_of(const Tensor &x)
{
    if (x.dim() < 2) refuse("the input must have the dimensions batch, time, neurons");
    return {x.size(0), x.size(1), elements(Shape(x.sizes().begin() + 2, x.sizes().end()))};
}

// What allocates the large results of a backward pass, as of now; held until the call has returned, as nobody else need hold it.
// The interpreter lock is taken a second time only where something was found.
class PlaceNow {
    PyObject *found = Py_None;                                 // None: not held

public:
    explicit PlaceNow(const Tensor &like)
    {
        if (place_of == nullptr) return;
        py::gil_scoped_acquire locked;
        py::object place = py::reinterpret_borrow<py::object>(place_of)(like);
        if (!place.is_none()) found = place.release().ptr();
    }
    PlaceNow(const PlaceNow &) = delete;
    PlaceNow &operator=(const PlaceNow &) = delete;
    ~PlaceNow()
    {
        if (found == Py_None) return;
        py::gil_scoped_acquire locked;
        Py_DECREF(found);
    }
    operator py::handle() const { return found; }
};

// One value that `grad` repeats everywhere (the gradient of a sum of the output), as a tensor of one element.
Tensor one_value(const Tensor &grad)
{
    if (!grad.defined() || grad.numel() < 2 || grad.scalar_type() != at::kFloat) return Tensor();
    for (const int64_t stride : grad.strides())
        if (stride != 0) return Tensor();
    return grad.as_strided({1}, {1});
}

// The gradient of a layer's output as the kernels take it, from what arrived at the output and at its total: dense, or one value
// for every element (then `uniform`) where `allowed`.
Tensor joined_gradient(const Tensor &grad, const Tensor &grad_total, const Shape &shape, const Tensor &like, bool allowed, bool &uniform)
{
    const auto options = like.options().dtype(at::kFloat);
    uniform = false;
    if (allowed && elements(shape) > 1) {
        Tensor one = grad.defined() ? one_value(grad) : (grad_total.defined() ? Tensor() : at::zeros({1}, options));
        if (grad_total.defined() && (one.defined() || !grad.defined())) {
            const Tensor total = grad_total.to(at::kFloat).reshape({1});
            one = one.defined() ? at::add(one, total) : total;
        }
        if (one.defined()) {
            uniform = true;
            return one;
        }
    }
    Tensor dense = grad.defined() ? grad.reshape(shape) : at::zeros(shape, options);
    if (grad_total.defined()) dense = at::add(dense, grad_total.to(dense.scalar_type()));
    return dense.contiguous();
}

Maybe dense(const Tensor &grad) { return grad.defined() ? Maybe(grad.contiguous()) : Maybe(); }
Maybe dense(const Tensor &grad, const Shape &shape) { return grad.defined() ? Maybe(grad.reshape(shape).contiguous()) : Maybe(); }
Maybe maybe(const Tensor &x) { return x.defined() ? Maybe(x) : Maybe(); }

// The place among a node's edges of each of its arguments, -1 for one that is absent (absent tensors get no edge).
struct Edges {
    int next = 0;
    int add(bool given) { return given ? next++ : -1; }
};

// What a node keeps besides tensors is one list of integers: compiled autograd looks into it.
int64_t bits(double x)
{
    int64_t n;
    std::memcpy(&n, &x, sizeof n);
    return n;
}
double from_bits(int64_t n)
{
    double x;
    std::memcpy(&x, &n, sizeof x);
    return x;
}

// What a forward kernel is to work out from the time constant `tau`, where nobody has (`alpha` absent): allocates alpha and kept.
void to_work_out(const Maybe &tau, Maybe &alpha, Maybe &kept, const float *&source, int64_t &period, float *&to, float *&copy,
                 const Tensor &like, int64_t neurons, int64_t n)
{
    if (!has(tau) || has(alpha)) return;
    dev(*tau, "tau", &like);
    if (tau->numel() != 1 && tau->numel() != neurons) refuse("tau must hold one value or one per neuron");
    alpha = fresh({n}, like);
    kept = fresh(tau->sizes(), like);
    source = tau->const_data_ptr<float>();
    period = tau->numel();
    to = out(*alpha);
    copy = out(*kept);
}

struct LifCall {
    const exodus_layer_decays *decays;
    bool syn, apply_low, decay_early, norm_input, records, need_grad;
    int64_t max_spikes, kind;
    double p0, p1;
    const Shape &states;
    const Maybe &kept_mem, &kept_syn;                          // the time constants as the forward pass saw them
    py::handle place;
};

struct LifLayer : torch::autograd::Function<LifLayer> {
    static variable_list forward(AutogradContext *ctx, const Tensor &input, const Tensor &alpha_mem, const Maybe &alpha_syn,
                                 const Tensor &v_init, const Maybe &i_init, const Maybe &tau_mem, const Maybe &tau_syn,
                                 const Tensor &theta, const Tensor &subtract, const Maybe &theta_low,
                                 const LifCall &c)
    {
        const Shape shape = three_of(input);
        const int64_t n = shape[0] * shape[2];
        Edges edges;
        edges.add(true);                                       // the input
        const int e_am = edges.add(true), e_as = edges.add(has(alpha_syn)), e_v0 = edges.add(true), e_i0 = edges.add(has(i_init));
        const int e_tm = edges.add(has(tau_mem)), e_ts = edges.add(has(tau_syn));
        const auto [spikes, v_last, i_last, ckpt_v, ckpt_i, v_rec, i_rec, total] = layer_lif_forward_decays(
            c.decays, shaped(input, shape), shaped(v_init, {n}), shaped(i_init, {n}), alpha_mem, alpha_syn, subtract, theta, theta_low,
            c.apply_low, c.max_spikes, c.decay_early, c.norm_input, c.need_grad, c.records, false, true, Maybe(), c.states, c.place);
        ctx->set_materialize_grads(false);
        if (c.need_grad)
            ctx->save_for_backward({input, ckpt_v, ckpt_i, v_init, i_init.value_or(Tensor()), alpha_mem,
                                    alpha_syn.value_or(Tensor()), subtract, theta, theta_low.value_or(Tensor()),
                                    c.kept_mem.value_or(Tensor()), c.kept_syn.value_or(Tensor())});
        ctx->saved_data["call"] = Shape{c.syn, c.apply_low, c.decay_early, c.norm_input, c.records, c.max_spikes, c.kind, bits(c.p0),
                                        bits(c.p1), e_am, e_as, e_v0, e_i0, e_tm, e_ts};
        variable_list outputs{shaped(spikes, input.sizes()), v_last, total};
        if (c.syn) outputs.push_back(i_last);
        if (c.records) outputs.push_back(shaped(v_rec, input.sizes()));
        if (c.records && c.syn) outputs.push_back(shaped(i_rec, input.sizes()));
        return outputs;
    }

    static variable_list backward(AutogradContext *ctx, const variable_list &grads)
    {
        const at::AutoGradMode no_graph(false);
        const Shape call = ctx->saved_data.at("call").toIntVector();
        const bool syn = call[0], apply_low = call[1], decay_early = call[2], norm_input = call[3], records = call[4];
        const int e_am = call[9], e_as = call[10], e_v0 = call[11], e_i0 = call[12], e_tm = call[13], e_ts = call[14];
        const variable_list saved = ctx->get_saved_variables();
        variable_list result(11);
        bool any = false;
        for (const Tensor &g : grads) any = any || g.defined();
        if (!any) return result;
        size_t at = 3;
        const Tensor &grad_spikes = grads[0], &grad_v_last = grads[1], &grad_total = grads[2];
        const Tensor grad_i_last = syn ? grads[at++] : Tensor(), grad_v_rec = records ? grads[at++] : Tensor();
        const Tensor grad_i_rec = records && syn ? grads[at++] : Tensor();
        const Tensor &input = saved[0], &v_init = saved[3], &i_init = saved[4];
        const Shape shape = three_of(input);
        const int64_t n = shape[0] * shape[2];
        const auto needs = [&](int edge) { return edge >= 0 && ctx->needs_input_grad(edge); };
        const bool tau_mem = needs(e_tm), tau_syn = needs(e_ts);
        bool uniform;
        const Tensor gs = joined_gradient(grad_spikes, grad_total, shape, input, !grad_v_rec.defined() && !grad_i_rec.defined(), uniform);
        const auto [g_x, g_am, g_as, g_v0, g_i0] = layer_lif_backward(
            gs, dense(grad_v_last), dense(grad_i_last), shaped(input, shape), maybe(saved[1]), maybe(saved[2]), shaped(v_init, {n}),
            shaped(maybe(i_init), {n}), saved[5], maybe(saved[6]), saved[7], saved[8], maybe(saved[9]), apply_low, call[5],
            decay_early, norm_input, static_cast<int>(call[6]), from_bits(call[7]), from_bits(call[8]), Maybe(), Maybe(),
            dense(grad_v_rec, shape), dense(grad_i_rec, shape), needs(e_am) || tau_mem, needs(e_as) || tau_syn, needs(e_v0),
            needs(e_i0), uniform, PlaceNow(input));
        if (ctx->needs_input_grad(0)) result[0] = shaped(g_x, input.sizes());
        if (needs(e_am)) result[1] = g_am;
        if (needs(e_as)) result[2] = g_as;
        if (needs(e_v0)) result[3] = shaped(g_v0, v_init.sizes());
        if (needs(e_i0)) result[4] = shaped(g_i0, i_init.sizes());
        if (tau_mem) result[5] = decay_grad(g_am, saved[10], shape[0], shape[2]);
        if (tau_syn) result[6] = decay_grad(g_as, saved[11], shape[0], shape[2]);
        return result;
    }
};

bool graph_wanted(std::initializer_list<const Tensor *> given, std::initializer_list<const Maybe *> optional)
{
    if (!at::GradMode::is_enabled()) return false;
    for (const Tensor *x : given)
        if (x->requires_grad()) return true;
    for (const Maybe *x : optional)
        if (has(*x) && (*x)->requires_grad()) return true;
    return false;
}

// -> (spikes, v_last, total, i_last, v_rec, i_rec) in the input's shape and the states' shape, with their place in the graph.
// tau_mem / tau_syn: the parameters that alpha_mem / alpha_syn were worked out from (decay_expand, which also made kept_mem /
// kept_syn) and whose gradients are wanted in the place of theirs; without factors the forward kernel works them out.
Eight layer_lif(const Tensor &input, Maybe alpha_mem, Maybe alpha_syn, const Tensor &v_init, const Maybe &i_init,
                const Maybe &tau_mem, const Maybe &tau_syn, Maybe kept_mem, Maybe kept_syn, const Tensor &theta,
                const Tensor &subtract, const Maybe &theta_low, int kind, double p0, double p1, int64_t max_spikes, bool decay_early,
                bool norm_input, bool records, const Shape &states, const py::handle place)
{
    const Shape shape = three_of(input);
    const int64_t n = shape[0] * shape[2];
    exodus_layer_decays decays{};
    // (a call without steps launches nothing that would write the factors)
    if (input.numel() > 0) {
        to_work_out(tau_mem, alpha_mem, kept_mem, decays.tau_mem, decays.period_mem, decays.alpha_mem, decays.kept_mem, input, shape[2], n);
        to_work_out(tau_syn, alpha_syn, kept_syn, decays.tau_syn, decays.period_syn, decays.alpha_syn, decays.kept_syn, input, shape[2], n);
    } else {
        if (has(tau_mem) && !has(alpha_mem)) std::tie(alpha_mem, kept_mem) = decay_expand(*tau_mem, shape[0], shape[2]);
        if (has(tau_syn) && !has(alpha_syn)) std::tie(alpha_syn, kept_syn) = decay_expand(*tau_syn, shape[0], shape[2]);
    }
    const bool syn = has(alpha_syn);
    const Tensor &am = present(alpha_mem, "alphaMem");
    const bool need_grad = graph_wanted({&input, &am, &v_init, &theta, &subtract}, {&alpha_syn, &i_init, &tau_mem, &tau_syn,
                                                                                           &theta_low});
    const LifCall call{&decays, syn, has(theta_low), decay_early, norm_input, records, need_grad, max_spikes, kind, p0, p1, states,
                       kept_mem, kept_syn, place};
    const variable_list out = LifLayer::apply(input, am, alpha_syn, v_init, i_init, tau_mem, tau_syn, theta, subtract,
                                              theta_low, call);
    const auto nth = [&](bool given, size_t k) { return given ? out[k] : Tensor(); };
    const size_t rec = syn ? 4 : 3;
    return {out[0], out[1], out[2], nth(syn, 3), nth(records, rec), nth(records && syn, rec + 1), Tensor(), Tensor()};
}

struct LeakyCall {
    const exodus_layer_decays *decays;
    bool decay_early, norm_input, need_grad, need_alpha;
    const Shape &states;
    const Maybe &kept;
    py::handle place;
};

struct LeakyLayer : torch::autograd::Function<LeakyLayer> {
    static variable_list forward(AutogradContext *ctx, const Tensor &input, const Tensor &alpha, const Tensor &v_init, const Maybe &tau,
                                 const LeakyCall &c)
    {
        const Shape shape = three_of(input);
        auto [flat, v_last, total] = layer_leaky_forward_decays(c.decays, shaped(input, shape),
                                                                shaped(v_init, {shape[0] * shape[2]}), alpha,
                                                         c.decay_early, c.norm_input, c.states, true, c.place);
        const Tensor result = shaped(flat, input.sizes());
        ctx->set_materialize_grads(false);
        if (c.need_grad && c.need_alpha)
            ctx->save_for_backward({alpha, v_init, result, c.decay_early || c.norm_input ? input : Tensor(),
                                    c.kept.value_or(Tensor())});
        else if (c.need_grad)
            ctx->save_for_backward({alpha});
        Shape call{c.decay_early, c.norm_input, c.need_alpha, has(tau), input.dim()};
        call.insert(call.end(), input.sizes().begin(), input.sizes().end());
        call.insert(call.end(), v_init.sizes().begin(), v_init.sizes().end());
        ctx->saved_data["call"] = call;
        return {result, v_last, total};
    }

    static variable_list backward(AutogradContext *ctx, const variable_list &grads)
    {
        const at::AutoGradMode no_graph(false);
        const Shape call = ctx->saved_data.at("call").toIntVector();
        const bool decay_early = call[0], norm_input = call[1], need_alpha = call[2], tau = call[3];
        const c10::IntArrayRef sizes = c10::IntArrayRef(call).slice(5), full = sizes.slice(0, call[4]), states = sizes.slice(call[4]);
        const Shape shape{full[0], full[1], elements(Shape(full.begin() + 2, full.end()))};
        variable_list saved = ctx->get_saved_variables();
        saved.resize(5);
        variable_list result(5);
        if (!grads[0].defined() && !grads[1].defined() && !grads[2].defined()) return result;
        const Tensor &alpha = saved[0], &out = saved[2], &input = saved[3];
        const int64_t n = shape[0] * shape[2];
        bool uniform;
        const Tensor g = joined_gradient(grads[0], grads[2], shape, alpha, true, uniform);
        // what of the results is allocated elsewhere depends on their size: the same kind of tensor as the gradient, expanded
        const auto [g_x, g_a, g_v0] = layer_leaky_backward(
            g, dense(grads[1]), need_alpha ? maybe(shaped(out, shape)) : Maybe(),
            input.defined() ? maybe(shaped(input, shape)) : Maybe(), need_alpha ? maybe(shaped(saved[1], {n})) : Maybe(), alpha,
            decay_early, norm_input, need_alpha, uniform ? std::optional<Shape>(shape) : std::nullopt,
            PlaceNow(uniform ? g.expand(shape) : g));
        if (ctx->needs_input_grad(0)) result[0] = shaped(g_x, full);
        if (tau) {
            if (ctx->needs_input_grad(3)) result[3] = decay_grad(g_a, saved[4], shape[0], shape[2]);
        } else if (ctx->needs_input_grad(1)) {
            result[1] = g_a;
        }
        if (ctx->needs_input_grad(2)) result[2] = shaped(g_v0, states);
        return result;
    }
};

// -> (out in the input's shape, v_last, total); tau as above, in the place of alpha_given
Three layer_leaky(const Tensor &input, Maybe alpha_given, const Tensor &v_init, const Maybe &tau, bool decay_early, bool norm_input,
                  const Shape &states, const py::handle place)
{
    const Shape shape = three_of(input);
    Maybe kept;
    exodus_layer_decays decays{};
    if (has(tau) && input.numel() == 0) std::tie(alpha_given, kept) = decay_expand(*tau, shape[0], shape[2]);
    to_work_out(tau, alpha_given, kept, decays.tau_mem, decays.period_mem, decays.alpha_mem, decays.kept_mem, input, shape[2],
                shape[0] * shape[2]);
    const Tensor &alpha = present(alpha_given, "alpha");
    const bool need_alpha = has(tau) ? tau->requires_grad() : alpha.requires_grad();
    const bool need_grad = graph_wanted({&input, &alpha, &v_init}, {&tau});
    const LeakyCall call{&decays, decay_early, norm_input, need_grad, need_alpha, states, kept, place};
    const variable_list out = LeakyLayer::apply(input, alpha, v_init, tau, call);
    return {out[0], out[1], out[2]};
}

}  // namespace

PYBIND11_MODULE(_exodus_torch, module)
{
    module.attr("built_for") = EXODUS_BUILT_FOR;                // the loader compares it with what is running
    // torch's own exceptions reach the caller as what they are (out of memory as torch.OutOfMemoryError)
    module.def("bind", torch::wrap_pybind_function(bind), py::arg("addresses"), py::arg("on_status"), py::arg("on_place") = py::none());
    // The calls run without the interpreter lock from their checks to their launch: an allocation may have to free memory and
    // wait for the device, and other Python threads go on meanwhile.  One release for all of it, as taking the lock back is what
    // a busy interpreter makes a caller wait for.
    module.def("layer_lif_forward", torch::wrap_pybind_function_no_gil(layer_lif_forward));
    module.def("layer_lif_backward", torch::wrap_pybind_function_no_gil(layer_lif_backward));
    module.def("layer_leaky_forward", torch::wrap_pybind_function_no_gil(layer_leaky_forward));
    module.def("layer_leaky_backward", torch::wrap_pybind_function_no_gil(layer_leaky_backward));
    module.def("layer_lif", torch::wrap_pybind_function_no_gil(layer_lif));
    module.def("layer_leaky", torch::wrap_pybind_function_no_gil(layer_leaky));
    module.def("stamps", torch::wrap_pybind_function(stamps));
    module.def("decay_expand", torch::wrap_pybind_function_no_gil(decay_expand));
    module.def("decay_grad", torch::wrap_pybind_function_no_gil(decay_grad));
    module.def("lif_forward", torch::wrap_pybind_function_no_gil(lif_forward));
    module.def("lif_backward_fused", torch::wrap_pybind_function_no_gil(lif_backward_fused));
    module.def("leaky_forward", torch::wrap_pybind_function_no_gil(leaky_forward));
    module.def("leaky_backward_fused", torch::wrap_pybind_function_no_gil(leaky_backward_fused));
}
