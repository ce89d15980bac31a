// The host side of a layer call: tensors in, autograd node out, one call into the kernel library per pass.
//
// A training step of a small layer is as long as the host takes to issue it.  Written in Python (a torch.autograd.Function
// with 37 torch.empty, 130 data_ptr and two ctypes calls per step) that was 240 to 480 us at B=2 L=128 E=768, of which
// the library's own launches were 75; here a pass is a few allocations for its intermediates, the launches, and a node
// that the engine runs without taking the interpreter's lock.
#include <algorithm>
#include <dlfcn.h>

#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/autograd/variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>

#include "../../include/substation_amd.h"

namespace py = pybind11;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

namespace {

// The kernel library, at the path the Python package has loaded it from.
struct Lib {
    decltype(&sub_last_error) last_error = nullptr;
    decltype(&sub_set_stream) set_stream = nullptr;
    decltype(&sub_get_option) get_option = nullptr;
    decltype(&sub_attention_in_registers) attention_in_registers = nullptr;
    decltype(&sub_set_attention_mask) set_attention_mask = nullptr;
    decltype(&sub_set_rng_counter) set_rng_counter = nullptr;
    decltype(&sub_forget_staged) forget_staged = nullptr;
    decltype(&sub_forward_form) forward_form = nullptr;
    decltype(&sub_set_forward_form) set_forward_form = nullptr;
    decltype(&sub_forward_alone) forward_alone = nullptr;
    decltype(&sub_encoder_forward) encoder_forward = nullptr;
    decltype(&sub_encoder_backward) encoder_backward = nullptr;
} lib;
PyObject* g_error = nullptr;          // substation_amd._lib.SubstationError

void load(const std::string& path, py::object error) {
    void* so = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
    if (!so) throw std::runtime_error(std::string("substation_amd host: ") + dlerror());
    auto get = [&](auto& fn, const char* name) {
        fn = reinterpret_cast<std::decay_t<decltype(fn)>>(dlsym(so, name));
        if (!fn) throw std::runtime_error(std::string("substation_amd host: the library has no ") + name);
    };
    get(lib.last_error, "sub_last_error");
    get(lib.set_stream, "sub_set_stream");
    get(lib.get_option, "sub_get_option");
    get(lib.attention_in_registers, "sub_attention_in_registers");
    get(lib.set_attention_mask, "sub_set_attention_mask");
    get(lib.set_rng_counter, "sub_set_rng_counter");
    get(lib.forget_staged, "sub_forget_staged");
    get(lib.forward_form, "sub_forward_form");
    get(lib.set_forward_form, "sub_set_forward_form");
    get(lib.forward_alone, "sub_forward_alone");
    get(lib.encoder_forward, "sub_encoder_forward");
    get(lib.encoder_backward, "sub_encoder_backward");
    g_error = error.release().ptr();
}

// An error of the library as the exception the Python binding raises for it; from any thread.
[[noreturn]] void raise(const std::string& what, PyObject* type = nullptr) {
    py::gil_scoped_acquire gil;
    PyErr_SetString(type ? type : g_error, what.c_str());
    python_error e;
    e.persist();
    throw e;
}
void check(int rc, const char* what) {
    if (rc < 0) raise(std::string(what) + ": " + lib.last_error());
}

void use_current_stream(void* handle, c10::DeviceIndex device) {
    check(lib.set_stream(handle, c10::hip::getCurrentHIPStream(device).stream()), "sub_set_stream");
}

// A list of buffers, side by side in allocations of up to 32 MiB (a larger buffer has one of its own), each from a multiple
// of 256 bytes on.  Not all of them in one: torch's allocator had to ask the device for a block of that size again
// wherever a program had since put tensors into the one it had given back, 1 ms and more on a layer's first pass at
// B=8 L=512 E=1024.  Not one for each: 37 per training step took 0.2 ms there where blocks had to be split and joined.
struct Buffers {
    static constexpr int64_t kMost = 16 << 20;    // halves
    std::vector<std::pair<int, int64_t>> where;   // allocation, offset in halves
    std::vector<int64_t> sizes;                   // of the allocations, in halves
    explicit Buffers(const std::vector<int64_t>& numels) {
        for (int64_t n : numels) {
            n = (n + 127) / 128 * 128;
            if (sizes.empty() || sizes.back() + n > kMost) sizes.push_back(0);
            where.emplace_back((int)sizes.size() - 1, sizes.back());
            sizes.back() += n;
        }
    }
    std::vector<at::Tensor> allocate(const at::TensorOptions& opt) const {
        std::vector<at::Tensor> ts;
        ts.reserve(sizes.size());
        for (int64_t n : sizes) ts.push_back(at::empty({n}, opt));
        return ts;
    }
    void pointers(const at::Tensor* ts, std::vector<void*>& out) const {
        for (const auto& [t, o] : where) out.push_back(static_cast<char*>(ts[t].data_ptr()) + 2 * o);
    }
};

// What the node below has no answer for and a Python autograd function has (a refusal, a traced call, a rule): tangents of
// forward-mode differentiation, functorch's transforms, dispatch modes and tensor subclasses, tracing.
bool has_tangent(const at::Tensor& t) {
    const auto* m = torch::autograd::impl::get_autograd_meta(t);
    return m && m->fw_grad_;
}
bool plain(const at::Tensor& X, const std::vector<at::Tensor>& params) {
    if (torch::jit::tracer::isTracing() || c10::impl::TorchDispatchModeTLS::any_modes_set() ||
        c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode))
        return false;
    auto odd = [](const at::Tensor& t) { return has_tangent(t) || t.key_set().has(c10::DispatchKey::Python); };
    return !odd(X) && std::none_of(params.begin(), params.end(), odd);
}

// A saved tensor as the backward pass needs it: dense, and 16-byte aligned where the forward pass found it so (a hook may
// restore it as a slice of a larger buffer, or with other strides).  On another device, of another type or size it is
// refused: the kernels are handed bare pointers.
bool misaligned(const at::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) & 15; }
struct Saved {
    SavedVariable variable;
    at::Device device;
    at::ScalarType type;
    int64_t numel;
    bool was_misaligned;
    explicit Saved(const at::Tensor& t)
        : variable(t, false), device(t.device()), type(t.scalar_type()), numel(t.numel()), was_misaligned(misaligned(t)) {}
    at::Tensor unpack() const {
        at::Tensor t = variable.unpack();
        if (t.device() != device || t.scalar_type() != type || t.numel() != numel)
            raise("a tensor that the forward pass has saved was restored on another device, with another type or another size",
                  PyExc_RuntimeError);
        if (t.is_contiguous() && (was_misaligned || !misaligned(t))) return t;
        at::NoGradGuard no_grad;
        t = t.contiguous();
        return misaligned(t) && !was_misaligned ? t.clone() : t;
    }
};

// An additive attention mask and the order of its dims.
struct Mask {
    at::Tensor values;
    std::string layout;
};

struct EncoderLayer : std::enable_shared_from_this<EncoderLayer> {
    void* handle;
    py::object keep_alive;            // the Python object that owns `handle`
    std::vector<int64_t> in_shape, out_shape;
    std::vector<std::vector<int64_t>> param_shapes;
    Buffers fwd, bwd;
    bool persistent, need_registers, need_relu_gate;
    // persistent: allocates (or finds) the two lists of tensors, given (which, tensor of the device)
    py::object workspace;
    std::vector<at::Tensor> kept_fwd, kept_bwd;
    uint64_t generation = 0;
    uint64_t passes = 0;              // forward and backward passes begun
    // What `handle` holds a bare pointer to from one call to the next.  Kept here and not on the module: a backward pass
    // that runs after its module is gone keeps this object.
    std::shared_ptr<Mask> mask;
    std::optional<at::Tensor> step_counter;

    EncoderLayer(uintptr_t handle_, py::object owner, std::vector<int64_t> in, std::vector<int64_t> out,
                 std::vector<std::vector<int64_t>> params, const std::vector<int64_t>& fwd_numels,
                 const std::vector<int64_t>& bwd_numels, bool persistent_, bool need_registers_, bool need_relu_gate_,
                 py::object workspace_)
        : handle(reinterpret_cast<void*>(handle_)), keep_alive(std::move(owner)), in_shape(std::move(in)),
          out_shape(std::move(out)), param_shapes(std::move(params)), fwd(fwd_numels), bwd(bwd_numels),
          persistent(persistent_), need_registers(need_registers_), need_relu_gate(need_relu_gate_),
          workspace(std::move(workspace_)) {}
    ~EncoderLayer() {
        if (!Py_IsInitialized()) { keep_alive.release(); workspace.release(); return; }
        py::gil_scoped_acquire gil;
        keep_alive = py::object();
        workspace = py::object();
    }

    // A layer built with token buffers for what its path leaves alone must be on that path.
    void check_compact() const {
        int v = 0;
        if (need_registers) {
            check(lib.attention_in_registers(handle, &v), "sub_attention_in_registers");
            if (!v)
                raise("this Encoder was built with compact_attention=True but the attention kernels that keep the scores "
                      "in registers are switched off", PyExc_RuntimeError);
        }
        check_relu_gate();
    }
    void check_relu_gate() const {
        int v = 0;
        if (!need_relu_gate) return;
        check(lib.get_option(handle, SUB_OPT_RELU_FROM_OUTPUT, &v), "sub_get_option");
        if (!v)
            raise("this Encoder was built with compact_activation=True but the ReLU gate from the dropout output (option 6) "
                  "is switched off: LIN1 and DROP2MASK would be written through 8-element buffers", PyExc_RuntimeError);
    }
    // (the old tensor is let go only once the handle points to the new one)
    void use_mask(std::shared_ptr<Mask> m) {
        if (m == mask) return;
        check(lib.set_attention_mask(handle, m ? m->values.data_ptr() : nullptr, m ? m->layout.c_str() : "JK"),
              "sub_set_attention_mask");
        mask = std::move(m);
    }
    void set_attention_mask(const std::optional<at::Tensor>& values, const std::string& layout) {
        use_mask(values ? std::make_shared<Mask>(Mask{*values, layout}) : nullptr);
    }
    void set_step_counter(const std::optional<at::Tensor>& counter) {
        check(lib.set_rng_counter(handle, counter ? static_cast<uint32_t*>(counter->data_ptr()) : nullptr),
              "sub_set_rng_counter");
        step_counter = counter;
    }
    // Only the pass right behind its forward pass (number `forward` of them all) can know the handle's staged copies by the
    // addresses they were made from: hooks may have dropped and restored the saved tensors, at addresses of others' by now.
    void begin_backward(uint64_t forward, int form) {
        if (passes != forward) check(lib.forget_staged(handle), "sub_forget_staged");
        check(lib.set_forward_form(handle, form), "sub_set_forward_form");
        ++passes;
    }
    // What the forward pass that has just run left (see sub_forward_form).
    int form() const {
        int v = 0;
        check(lib.forward_form(handle, &v), "sub_forward_form");
        return v;
    }
    void keep(std::vector<at::Tensor>& list, const char* which, const at::Tensor& X) {
        if (list.empty() || list[0].device() != X.device()) list = workspace(which, X).cast<std::vector<at::Tensor>>();
    }

    std::optional<at::Tensor> forward(const at::Tensor& X, const std::vector<at::Tensor>& params);
};

// A backward pass under the mask of its forward pass, whatever has been set since.
struct MaskScope {
    EncoderLayer& layer;
    const std::shared_ptr<Mask> now;
    MaskScope(EncoderLayer& l, const std::shared_ptr<Mask>& m) : layer(l), now(l.mask) { layer.use_mask(m); }
    ~MaskScope() {
        try { layer.use_mask(now); } catch (...) {}   // (one that the handle has taken before)
    }
};

struct EncoderBackward : Node {
    std::shared_ptr<EncoderLayer> layer;
    std::shared_ptr<Mask> mask;          // of the forward pass
    // the parameters as the forward pass read them, X, and the forward intermediates (those of a layer that keeps its own
    // too: what hooks on saved tensors see does not depend on who holds the memory)
    std::vector<Saved> saved;
    int form = 0;                        // what the forward pass left (sub_forward_form)
    uint64_t generation = 0, pass = 0;

    std::string name() const override { return "EncoderFunctionBackward"; }
    void release_variables() override {
        for (auto& s : saved) s.variable.reset_data();
    }

    variable_list apply(variable_list&& grads) override {
        EncoderLayer& l = *layer;
        if (l.persistent && generation != l.generation)
            raise("persistent_workspace: forward() ran again before this backward pass; what it had saved has been "
                  "overwritten", PyExc_RuntimeError);
        l.check_relu_gate();
        variable_list in;
        in.reserve(saved.size());
        for (const auto& s : saved) in.push_back(s.unpack());
        const size_t np = l.param_shapes.size();
        const at::Tensor& X = in[np];
        const c10::DeviceGuard guard(X.device());
        at::Tensor DY = grads[0].defined() ? grads[0].contiguous() : at::zeros(l.out_shape, X.options());
        variable_list out;
        out.reserve(1 + l.param_shapes.size());
        const auto opt = X.options();
        out.push_back(at::empty(l.in_shape, DY.options()));
        for (const auto& s : l.param_shapes) out.push_back(at::empty(s, opt));
        std::vector<at::Tensor> scratch;
        std::vector<void*> p;
        p.reserve(96);
        p.push_back(DY.data_ptr());
        for (size_t i = 1; i < out.size(); ++i) p.push_back(out[i].data_ptr());
        if (l.persistent) {
            for (const auto& t : l.kept_bwd) p.push_back(t.data_ptr());
        } else {
            scratch = l.bwd.allocate(opt);
            l.bwd.pointers(scratch.data(), p);
        }
        for (size_t i = 0; i < np; ++i) p.push_back(in[i].data_ptr());
        if (l.persistent) for (size_t i = np + 1; i < in.size(); ++i) p.push_back(in[i].data_ptr());
        else l.fwd.pointers(in.data() + np + 1, p);
        p.push_back(X.data_ptr());
        p.push_back(out[0].data_ptr());
        use_current_stream(l.handle, X.device().index());
        const MaskScope own(l, mask);
        l.begin_backward(pass, form);
        check(lib.encoder_backward(l.handle, p.data(), (int)p.size()), "encoder_backward");
        return out;
    }
};

// None where the caller is to take the Python function.
std::optional<at::Tensor> EncoderLayer::forward(const at::Tensor& X_, const std::vector<at::Tensor>& params) {
    if (!plain(X_, params)) return std::nullopt;
    if (!X_.is_cuda()) raise("Encoder.forward needs a tensor on the GPU", PyExc_RuntimeError);
    if (X_.sizes() != at::IntArrayRef(in_shape)) {
        std::ostringstream m;
        m << "X has shape " << X_.sizes() << ", the configured input layout needs " << at::IntArrayRef(in_shape);
        raise(m.str(), PyExc_ValueError);
    }
    check_compact();
    const c10::DeviceGuard guard(X_.device());
    bool grad = false;
    if (at::GradMode::is_enabled()) {
        grad = X_.requires_grad();
        for (size_t i = 0; !grad && i < params.size(); ++i) grad = params[i].requires_grad();
    }
    at::Tensor X, Y;
    std::vector<at::Tensor> w, interm;
    std::vector<void*> p;
    p.reserve(48);
    {
        at::NoGradGuard no_grad;
        X = X_.contiguous();
        w.reserve(params.size());
        for (const auto& t : params) w.push_back(t.contiguous());
        // same element count as X, shaped in the output's own dimension order
        Y = at::empty(out_shape, X.options().requires_grad(false));
        p.push_back(X.data_ptr());
        for (const auto& t : w) p.push_back(t.data_ptr());
        if (persistent) {
            keep(kept_fwd, "forward_interm", X);
            if (grad) keep(kept_bwd, "backward_interm", X);
            for (const auto& t : kept_fwd) p.push_back(t.data_ptr());
        } else {
            interm = fwd.allocate(Y.options());
            fwd.pointers(interm.data(), p);
        }
        p.push_back(Y.data_ptr());
    }
    ++generation;
    ++passes;
    {
        py::gil_scoped_release nogil;
        use_current_stream(handle, X.device().index());
        // (a workspace that stays with the module can be looked at, these intermediates are gone when this returns)
        if (!grad && !persistent) check(lib.forward_alone(handle), "sub_forward_alone");
        check(lib.encoder_forward(handle, p.data(), (int)p.size()), "encoder_forward");
    }
    if (grad) {
        std::shared_ptr<EncoderBackward> node(new EncoderBackward(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(X_, params));
        node->layer = shared_from_this();
        node->mask = mask;
        const std::vector<at::Tensor>& held = persistent ? kept_fwd : interm;
        node->saved.reserve(w.size() + 1 + held.size());
        for (const auto& t : w) node->saved.emplace_back(t);
        node->saved.emplace_back(X);
        for (const auto& t : held) node->saved.emplace_back(t);
        node->form = form();
        node->generation = generation;
        node->pass = passes;
        torch::autograd::set_history(Y, node);
    }
    return Y;
}

}  // namespace

PYBIND11_MODULE(_host, m) {
    m.def("load", &load);
    py::class_<Mask, std::shared_ptr<Mask>>(m, "Mask");
    py::class_<EncoderLayer, std::shared_ptr<EncoderLayer>>(m, "EncoderLayer")
        .def(py::init<uintptr_t, py::object, std::vector<int64_t>, std::vector<int64_t>, std::vector<std::vector<int64_t>>,
                      const std::vector<int64_t>&, const std::vector<int64_t>&, bool, bool, bool, py::object>())
        .def_readwrite("generation", &EncoderLayer::generation)
        .def_readwrite("passes", &EncoderLayer::passes)
        .def("begin_backward", &EncoderLayer::begin_backward)
        .def("form", &EncoderLayer::form)
        .def("check_compact", &EncoderLayer::check_compact)
        .def("check_relu_gate", &EncoderLayer::check_relu_gate)
        .def("set_attention_mask", &EncoderLayer::set_attention_mask)
        .def_property("mask", [](const EncoderLayer& l) { return l.mask; }, &EncoderLayer::use_mask)
        .def("set_step_counter", &EncoderLayer::set_step_counter)
        .def("forward", &EncoderLayer::forward);
}
