// The host side of a layer call: tensors in, autograd node out, one call into the kernel library per pass.
//
// A training step of a small layer is as long as the host takes to issue it.  Written in Python (a torch.autograd.Function
// with 37 torch.empty, 130 data_ptr and two ctypes calls per step) that was 240 to 480 us at B=2 L=128 E=768, of which
// the library's own launches were 75; here a pass is a few allocations for its intermediates, the launches, and a node
// that the engine runs without taking the interpreter's lock.
#include <algorithm>
#include <dlfcn.h>
#include <mutex>

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
    decltype(&sub_set_rng) set_rng = nullptr;
    decltype(&sub_ops_defer) ops_defer = nullptr;
    decltype(&sub_op_einsum) einsum = nullptr;
    decltype(&sub_op_einsum_add) einsum_add = nullptr;
    decltype(&sub_op_einsum_bad) einsum_bad = nullptr;
    decltype(&sub_op_einsum_bdrlb) einsum_bdrlb = nullptr;
    decltype(&sub_op_einsum_group) einsum_group = nullptr;
    decltype(&sub_op_attention_forward) attention_forward = nullptr;
    decltype(&sub_op_attention_backward_biases) attention_backward = nullptr;
    decltype(&sub_op_bdrln) bdrln = nullptr;
    decltype(&sub_op_bad) bad = nullptr;
    decltype(&sub_op_bdrlb) bdrlb = nullptr;
    decltype(&sub_op_ln_backward) ln_backward = nullptr;
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
    get(lib.set_rng, "sub_set_rng");
    get(lib.ops_defer, "sub_ops_defer");
    get(lib.einsum, "sub_op_einsum");
    get(lib.einsum_add, "sub_op_einsum_add");
    get(lib.einsum_bad, "sub_op_einsum_bad");
    get(lib.einsum_bdrlb, "sub_op_einsum_bdrlb");
    get(lib.einsum_group, "sub_op_einsum_group");
    get(lib.attention_forward, "sub_op_attention_forward");
    get(lib.attention_backward, "sub_op_attention_backward_biases");
    get(lib.bdrln, "sub_op_bdrln");
    get(lib.bad, "sub_op_bad");
    get(lib.bdrlb, "sub_op_bdrlb");
    get(lib.ln_backward, "sub_op_ln_backward");
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

// The operators of a decoder layer's two passes (substation_amd/decoder.py), in the order of the reference's statements
// (substation/transformer.py:288-441).  Issued from Python (some 55 ctypes calls and 60 torch.empty) they kept the host for 717 us at
// B=8, lengths 256 and 512, E 1024, where their kernels took 530; from here the host takes 430 to 470 and a
// pass 524, of which 494 to 501 are kernels.
struct DecoderPasses {
    enum Parameter { SATTN_WKQV, SATTN_IN_B, SATTN_WO, SATTN_OUT_B, EDATTN_WQ, EDATTN_WK, EDATTN_WV, EDATTN_IN_B, EDATTN_WO, EDATTN_OUT_B,
                     NORM1_SCALE, NORM1_BIAS, NORM2_SCALE, NORM2_BIAS, NORM3_SCALE, NORM3_BIAS, LINEAR1_W, LINEAR1_B, LINEAR2_W, LINEAR2_B,
                     PARAMETERS };
    // what a forward pass leaves for its backward pass
    enum Kept { KQV, STATS1, KEEP1, GAMMA1, MASK1, DIFF1, LN1, NORMED1, ISTD1, Q2, K2, V2, STATS2, KEEP2, GAMMA2, MASK2, DIFF2, LN2, NORMED2,
                ISTD2, LIN1, MASK3, FF1, BITS, MASK4, DIFF3, LN3, ISTD3, KEPT };
    typedef std::optional<at::Tensor> Maybe;

    void* target;                     // the handles of the two sizes
    void* source;
    py::object keep_alive;
    int64_t B, Lt, Ls, H, P, E, U;
    double p_sattn, p_edattn, p_linear1, p_ff;
    uint32_t site_sattn, site_edattn, site_linear1, site_ff;
    bool relu;
    float scale;
    std::mutex busy;                  // a pass is a sequence of calls on the same two handles

    DecoderPasses(uintptr_t target_, uintptr_t source_, py::object owner, const std::vector<int64_t>& sizes,
                  const std::vector<double>& probs, const std::vector<uint32_t>& sites, bool relu_, double scale_)
        : target(reinterpret_cast<void*>(target_)), source(reinterpret_cast<void*>(source_)), keep_alive(std::move(owner)),
          B(sizes.at(0)), Lt(sizes.at(1)), Ls(sizes.at(2)), H(sizes.at(3)), P(sizes.at(4)), E(sizes.at(5)), U(sizes.at(6)),
          p_sattn(probs.at(0)), p_edattn(probs.at(1)), p_linear1(probs.at(2)), p_ff(probs.at(3)),
          site_sattn(sites.at(0)), site_edattn(sites.at(1)), site_linear1(sites.at(2)), site_ff(sites.at(3)),
          relu(relu_), scale((float)scale_) {}
    ~DecoderPasses() {
        if (!Py_IsInitialized()) { keep_alive.release(); return; }
        py::gil_scoped_acquire gil;
        keep_alive = py::object();
    }

    static void* at_(const at::Tensor& t) {
        if (!(t.is_cuda() && t.scalar_type() == at::kHalf && t.is_contiguous()))
            raise("operators take contiguous fp16 CUDA tensors", PyExc_ValueError);
        return t.data_ptr();
    }
    static void* at_(const Maybe& t) { return t ? at_(*t) : nullptr; }
    // The kernels are handed bare pointers: what a caller brings, or hooks on saved tensors restore, has as many elements as the layer's
    // sizes say, or the pass is refused before its first launch.
    static void holds(const at::Tensor& t, int64_t numel, const char* what) {
        if (t.numel() == numel) return;
        raise("DecoderLayer: " + std::string(what) + " has " + std::to_string(t.numel()) + " elements, the sizes of the layer need " +
              std::to_string(numel), PyExc_ValueError);
    }
    void check_sizes(const at::Tensor& x, const at::Tensor& enc, const std::vector<at::Tensor>& w, const Maybe& mask) const {
        const int64_t EE = E * H * P, in_b = 3 * H * P;
        const struct { const char* name; int64_t numel; } parameters[PARAMETERS] = {
            {"sattn_wkqv", 3 * EE}, {"sattn_in_b", in_b}, {"sattn_wo", EE}, {"sattn_out_b", E}, {"edattn_wq", EE}, {"edattn_wk", EE},
            {"edattn_wv", EE}, {"edattn_in_b", in_b}, {"edattn_wo", EE}, {"edattn_out_b", E}, {"norm1_scale", E}, {"norm1_bias", E},
            {"norm2_scale", E}, {"norm2_bias", E}, {"norm3_scale", E}, {"norm3_bias", E}, {"linear1_w", U * E}, {"linear1_b", U},
            {"linear2_w", E * U}, {"linear2_b", E}};
        if (w.size() != PARAMETERS) raise("DecoderLayer: 20 parameters", PyExc_ValueError);
        for (int i = 0; i < PARAMETERS; ++i) holds(w[i], parameters[i].numel, parameters[i].name);
        holds(x, B * Lt * E, "x");
        holds(enc, B * Ls * E, "the encoder's output");
        if (mask) holds(*mask, Lt * Lt, "the mask of the self-attention");
    }
    void check_kept(const std::vector<Maybe>& k, const at::Tensor& dy) const {
        const int64_t bji = B * Lt * E, bki = B * Ls * E, bj = B * Lt, bju = B * Lt * U, rows = H * B * Lt;
        const int64_t numels[KEPT] = {3 * bji, 2 * rows, rows * (Lt / 32), bji, bji, bji, bji, bji, bj, bji, bki, bki, 2 * rows, rows * (Ls / 32), bji,
                                      bji, bji, bji, bji, bj, bju, bju, bju, bju / 8, bji, bji, bji, bj};
        if (k.size() < KEPT) raise("DecoderLayer: not what a forward pass has saved", PyExc_ValueError);
        for (int i = 0; i < KEPT; ++i) {
            if (k[i]) holds(*k[i], numels[i], "what a forward pass has saved");
            else if (i != LIN1 && i != MASK3 && i != BITS) raise("DecoderLayer: not what a forward pass has saved", PyExc_ValueError);
        }
        holds(dy, bji, "the gradient of the output");
    }
    static char* part(const at::Tensor& t, int64_t i, int64_t of) { return static_cast<char*>(at_(t)) + 2 * (t.numel() / of) * i; }

    // A pass: the current device's stream, tensors on that device.
    struct Place {
        at::TensorOptions half;
        explicit Place(DecoderPasses& d) {
            const c10::DeviceIndex device = c10::hip::current_device();
            half = at::TensorOptions().dtype(at::kHalf).device(c10::Device(c10::kCUDA, device));
            use_current_stream(d.target, device);
            if (d.source != d.target) use_current_stream(d.source, device);
        }
        at::Tensor operator()(at::IntArrayRef shape) const { return at::empty(shape, half); }
        at::Tensor operator()(at::IntArrayRef shape, at::ScalarType type) const { return at::empty(shape, half.dtype(type)); }
    };

    std::vector<Maybe> forward(const at::Tensor& x, const at::Tensor& enc, const std::vector<at::Tensor>& w, const Maybe& mask, uint64_t seed,
                               uint32_t step, bool epilogues) {
        py::gil_scoped_release nogil;
        const std::lock_guard<std::mutex> one(busy);
        check_sizes(x, enc, w, mask);
        const Place e(*this);
        check(lib.set_rng(target, seed, step), "sub_set_rng");
        check(lib.set_rng(source, seed, step), "sub_set_rng");
        std::vector<Maybe> k(KEPT + 1);                      // and the output
        std::vector<void*> wp;
        wp.reserve(PARAMETERS);
        for (const auto& t : w) wp.push_back(at_(t));
        const auto make = [&](Kept i, at::IntArrayRef shape) { k[i] = e(shape); return k[i]->data_ptr(); };
        const std::initializer_list<int64_t> bji = {B, Lt, E}, bj = {B, Lt}, bjhp = {B, Lt, H, P}, bkhp = {B, Ls, H, P}, bju = {B, Lt, U};
        // All that reads the layer's inputs: the projections of the self-attention and, of the encoder's output, the keys and values of
        // the other.  In one call their tiles share a round (8 x 256 on 512, E 1024: 22.4, 18.5 and 13.6 us in three launches, 37.4
        // now).  Not in front
        // of a ReLU, where another order of the sums moves gates.
        make(KQV, {3, B, Lt, H, P}); make(K2, bkhp); make(V2, bkhp);
        const at::Tensor& in_b = w[EDATTN_IN_B];
        const SubEinsum inputs[] = {
            {target, at_(x), "BJI", wp[SATTN_WKQV], "QHPI", wp[SATTN_IN_B], "QHP", at_(k[KQV]), "QBJHP", 1.f},
            {source, at_(enc), "BKI", wp[EDATTN_WK], "HPI", part(in_b, 1, 3), "HP", at_(k[K2]), "BKHP", 1.f},
            {source, at_(enc), "BKI", wp[EDATTN_WV], "HPI", part(in_b, 2, 3), "HP", at_(k[V2]), "BKHP", 1.f}};
        const auto alone = [](const SubEinsum& q) {
            check(lib.einsum_add(q.sizes, q.A, q.l_A, q.B, q.l_B, q.T, q.l_T, q.C, q.l_C, q.alpha), "einsum_add");
        };
        if (relu) alone(inputs[0]);
        else check(lib.einsum_group(target, inputs, 3), "einsum_group");
        // masked self-attention, residual, norm1
        const auto workspace = [&](Kept stats, Kept keep, int64_t keys) {
            k[stats] = e({2 * H * B * Lt}, at::kFloat);
            k[keep] = e({H * B * Lt * (keys / 32)}, at::kInt);
        };
        workspace(STATS1, KEEP1, Lt);
        make(GAMMA1, bjhp);
        check(lib.attention_forward(target, (int)Lt, (int)Lt, part(*k[KQV], 1, 3), "BJHP", part(*k[KQV], 0, 3), part(*k[KQV], 2, 3), "BKHP",
                                    at_(k[GAMMA1]), "BJHP", k[STATS1]->data_ptr(), k[KEEP1]->data_ptr(), at_(mask), "JK", scale, 0.f, 0),
              "attention_forward");
        const at::Tensor att1 = e(bji);
        check(lib.einsum(target, wp[SATTN_WO], "IHP", at_(k[GAMMA1]), "BJHP", at_(att1), "BJI", 1.f), "einsum");
        const auto norm = [&](const at::Tensor& in, const at::Tensor& residual, Parameter b, Parameter s, Kept m, Kept diff, Kept ln, int normed,
                              Kept istd, double p, uint32_t site) {
            make(m, bji); make(diff, bji); make(ln, bji); make(istd, bj);
            k[normed] = e(bji);
            check(lib.bdrln(target, at_(in), "BJI", at_(residual), "BJI", wp[b], wp[s], wp[s + 1], at_(in), "BJI", at_(k[m]), "BJI",
                            at_(k[diff]), "BJI", at_(k[ln]), "BJI", at_(k[normed]), "BJI", at_(k[istd]), "BJ", (float)p, site), "bdrln");
        };
        norm(att1, x, SATTN_OUT_B, NORM1_SCALE, MASK1, DIFF1, LN1, NORMED1, ISTD1, p_sattn, site_sattn);
        // encoder-decoder attention, residual, norm2
        make(Q2, bjhp);
        check(lib.einsum_add(target, at_(k[NORMED1]), "BJI", wp[EDATTN_WQ], "HPI", part(in_b, 0, 3), "HP", at_(k[Q2]), "BJHP", 1.f), "einsum_add");
        if (relu) { alone(inputs[1]); alone(inputs[2]); }
        workspace(STATS2, KEEP2, Ls);
        make(GAMMA2, bjhp);
        check(lib.attention_forward(target, (int)Lt, (int)Ls, at_(k[Q2]), "BJHP", at_(k[K2]), at_(k[V2]), "BKHP", at_(k[GAMMA2]), "BJHP",
                                    k[STATS2]->data_ptr(), k[KEEP2]->data_ptr(), nullptr, "JK", scale, 0.f, 0), "attention_forward");
        const at::Tensor att2 = e(bji);
        check(lib.einsum(target, wp[EDATTN_WO], "IHP", at_(k[GAMMA2]), "BJHP", at_(att2), "BJI", 1.f), "einsum");
        norm(att2, *k[NORMED1], EDATTN_OUT_B, NORM2_SCALE, MASK2, DIFF2, LN2, NORMED2, ISTD2, p_edattn, site_edattn);
        // feed-forward, residual, norm3: linear1 with bias, activation and dropout in its epilogue where the product qualifies (the keep
        // bits then travel as bits, no mask tensor; ReLU needs no pre-activation either); else operator by operator
        make(FF1, bju);
        if (!relu) make(LIN1, bju);
        int applied = 0;
        if (epilogues) {
            k[BITS] = e({B * Lt * U / 8}, at::kByte);
            check(lib.einsum_bad(target, at_(k[NORMED2]), "BJI", wp[LINEAR1_W], "UI", wp[LINEAR1_B], "U", at_(k[LIN1]), at_(k[FF1]), "BJU",
                                 k[BITS]->data_ptr(), (float)p_linear1, site_linear1, &applied), "einsum_bad");
        }
        if (!applied) {
            k[BITS].reset();
            make(LIN1, bju); make(MASK3, bju);
            check(lib.einsum(target, at_(k[NORMED2]), "BJI", wp[LINEAR1_W], "UI", at_(k[LIN1]), "BJU", 1.f), "einsum");
            check(lib.bad(target, at_(k[LIN1]), "BJU", wp[LINEAR1_B], at_(k[LIN1]), "BJU", at_(k[MASK3]), "BJU", at_(k[FF1]), "BJU",
                          (float)p_linear1, site_linear1), "bad");
        }
        const at::Tensor ff = e(bji);
        check(lib.einsum(target, at_(k[FF1]), "BJU", wp[LINEAR2_W], "IU", at_(ff), "BJI", 1.f), "einsum");
        norm(ff, *k[NORMED2], LINEAR2_B, NORM3_SCALE, MASK4, DIFF3, LN3, KEPT, ISTD3, p_ff, site_ff);
        return k;
    }

    // The second stage of every column sum of a pass in one launch at its end (whatever becomes of the pass).
    struct Deferred {
        std::vector<void*> handles;
        Deferred() = default;
        // (by way of the constructor above: from there on a refusal of the second handle runs the destructor for the first)
        explicit Deferred(const DecoderPasses& d) : Deferred() {
            for (void* h : {d.target, d.source}) {
                if (std::find(handles.begin(), handles.end(), h) != handles.end()) continue;
                handles.push_back(h);
                check(lib.ops_defer(h, 1), "sub_ops_defer");
            }
        }
        void finish() {
            while (!handles.empty()) {
                void* h = handles.back();
                handles.pop_back();
                check(lib.ops_defer(h, 0), "sub_ops_defer");
            }
        }
        ~Deferred() {
            for (; !handles.empty(); handles.pop_back()) lib.ops_defer(handles.back(), 0);
        }
    };

    // The gradients of x, of the encoder's output and of the parameters.
    std::vector<at::Tensor> backward(const at::Tensor& x, const at::Tensor& enc, std::vector<at::Tensor> w, const std::vector<Maybe>& k,
                                     const at::Tensor& dy, const Maybe& mask) {
        py::gil_scoped_release nogil;
        const std::lock_guard<std::mutex> one(busy);
        check_sizes(x, enc, w, mask);
        check_kept(k, dy);
        // (the products with an epilogue need whole 16-byte words, wherever a parameter lies or was restored to)
        for (const Parameter i : {LINEAR2_W, EDATTN_WV, SATTN_WKQV})
            if (misaligned(w[i])) w[i] = w[i].clone();
        const Place e(*this);
        std::vector<at::Tensor> out(2);                      // dx and d(encoder output), then the parameters'
        std::vector<void*> wp, g;
        wp.reserve(PARAMETERS); g.reserve(PARAMETERS);
        for (const auto& t : w) {
            wp.push_back(at_(t));
            out.push_back(at::empty_like(t));
            g.push_back(at_(out.back()));
        }
        const at::Tensor unused = at::empty_like(out[2 + SATTN_OUT_B]);      // norm1's column sums of the third input are not needed
        // (behind all that receives such a sum: what a refusal further down leaves on the list is launched on the way out, into memory
        // that must still be this pass's)
        Deferred deferred(*this);
        const std::initializer_list<int64_t> bji = {B, Lt, E}, bjhp = {B, Lt, H, P}, bkhp = {B, Ls, H, P}, bju = {B, Lt, U};
        // a LayerNorm's backward pass, its dropout's and (second: with a second gradient) the sums next to it
        struct Norm { at::Tensor dln, dres, ddrop; };
        const auto norm = [&](Kept ln, Parameter s, const at::Tensor& dout, Kept istd, Kept diff, Kept m, const at::Tensor* dout2,
                              const at::Tensor* dlinear, void* dlinear_bias, void* dout_bias) {
            Norm n{e(bji), e(bji), e(bji)};
            check(lib.ln_backward(target, dout2 ? 1 : 0, at_(k[ln]), "BJI", wp[s], at_(dout), "BJI", dout2 ? at_(*dout2) : nullptr, "BJI",
                                  dlinear ? at_(*dlinear) : nullptr, "BJI", at_(k[istd]), "BJ", at_(k[diff]), "BJI", at_(k[m]), "BJI",
                                  at_(n.dln), "BJI", at_(n.dres), "BJI", at_(n.ddrop), "BJI", g[s], g[s + 1], dlinear_bias, dout_bias),
                  "ln_backward");
            return n;
        };
        // norm3, residual, feed-forward
        const Norm n3 = norm(LN3, NORM3_SCALE, dy, ISTD3, DIFF3, MASK4, nullptr, nullptr, nullptr, nullptr);
        const at::Tensor& dff = n3.ddrop;
        const at::Tensor dlin1 = e(bju);
        int applied = 0;
        if (k[BITS])
            check(lib.einsum_bdrlb(target, at_(dff), "BJI", wp[LINEAR2_W], "IU", at_(k[relu ? FF1 : LIN1]), "BJU", k[BITS]->data_ptr(), at_(dlin1),
                                   "BJU", g[LINEAR1_B], &applied), "einsum_bdrlb");
        if (!applied) {
            if (!k[MASK3])
                raise("DecoderLayer: the forward pass ran linear1 with its activation epilogue, the backward pass cannot", PyExc_RuntimeError);
            const at::Tensor dff1 = e(bju);
            check(lib.einsum(target, at_(dff), "BJI", wp[LINEAR2_W], "IU", at_(dff1), "BJU", 1.f), "einsum");
            check(lib.bdrlb(target, at_(dff1), "BJU", at_(k[MASK3]), "BJU", at_(k[LIN1]), "BJU", at_(dlin1), "BJU", g[LINEAR1_B]), "bdrlb");
        }
        // (weight gradients feed nothing: all of them run at the end, where their tiles fill each other's rounds.  Kernels of
        // 8 x 256 on 512, E 1024: 526 us, 639 with each next to its data gradient; 8 x 512 on 512: a pass 1004 -> 873)
        const at::Tensor dnormed2 = e(bji);
        check(lib.einsum(target, at_(dlin1), "BJU", wp[LINEAR1_W], "UI", at_(dnormed2), "BJI", 1.f), "einsum");
        // norm2, residual, encoder-decoder attention
        const Norm n2 = norm(LN2, NORM2_SCALE, n3.dres, ISTD2, DIFF2, MASK2, &dnormed2, &dff, g[LINEAR2_B], g[EDATTN_OUT_B]);
        const at::Tensor& datt2 = n2.ddrop;
        const at::Tensor dgamma2 = e(bjhp);
        check(lib.einsum(target, wp[EDATTN_WO], "IHP", at_(datt2), "BJI", at_(dgamma2), "BJHP", 1.f), "einsum");
        const at::Tensor dq2 = e(bjhp), dk2 = e(bkhp), dv2 = e(bkhp);
        const at::Tensor& d_in_b = out[2 + EDATTN_IN_B];
        check(lib.attention_backward(target, (int)Lt, (int)Ls, at_(k[Q2]), "BJHP", at_(k[K2]), at_(k[V2]), "BKHP", at_(k[GAMMA2]), "BJHP",
                                     at_(dgamma2), "BJHP", k[STATS2]->data_ptr(), k[KEEP2]->data_ptr(), at_(dq2), "BJHP", at_(dk2), at_(dv2), "BKHP",
                                     nullptr, "JK", scale, part(d_in_b, 0, 3), part(d_in_b, 1, 3), part(d_in_b, 2, 3)), "attention_backward");
        const at::Tensor dnormed1 = e(bji);
        out[1] = e({B, Ls, E});
        void* const denc = at_(out[1]);
        const auto group = [&](std::initializer_list<SubEinsum> products) {
            check(lib.einsum_group(target, products.begin(), (int)products.size()), "einsum_group");
        };
        group({{nullptr, at_(dq2), "BJHP", wp[EDATTN_WQ], "HPI", nullptr, nullptr, at_(dnormed1), "BJI", 1.f},
               {source, at_(dk2), "BKHP", wp[EDATTN_WK], "HPI", nullptr, nullptr, denc, "BKI", 1.f}});
        // norm1, residual, self-attention
        const Norm n1 = norm(LN1, NORM1_SCALE, n2.dres, ISTD1, DIFF1, MASK1, &dnormed1, &datt2, at_(unused), g[SATTN_OUT_B]);
        const at::Tensor& datt1 = n1.ddrop;
        const at::Tensor dgamma1 = e(bjhp);
        check(lib.einsum(target, wp[SATTN_WO], "IHP", at_(datt1), "BJI", at_(dgamma1), "BJHP", 1.f), "einsum");
        const at::Tensor dkqv = e({3, B, Lt, H, P});
        const at::Tensor &kqv = *k[KQV], &ds_in_b = out[2 + SATTN_IN_B];
        check(lib.attention_backward(target, (int)Lt, (int)Lt, part(kqv, 1, 3), "BJHP", part(kqv, 0, 3), part(kqv, 2, 3), "BKHP", at_(k[GAMMA1]),
                                     "BJHP", at_(dgamma1), "BJHP", k[STATS1]->data_ptr(), k[KEEP1]->data_ptr(), part(dkqv, 1, 3), "BJHP",
                                     part(dkqv, 0, 3), part(dkqv, 2, 3), "BKHP", at_(mask), "JK", scale, part(ds_in_b, 1, 3), part(ds_in_b, 0, 3),
                                     part(ds_in_b, 2, 3)), "attention_backward");
        out[0] = e(bji);
        group({{nullptr, wp[SATTN_WKQV], "QHPI", at_(dkqv), "QBJHP", at_(n1.dres), "BJI", at_(out[0]), "BJI", 1.f},
               {source, at_(dv2), "BKHP", wp[EDATTN_WV], "HPI", denc, "BKI", denc, "BKI", 1.f},
               {source, at_(dv2), "BKHP", at_(enc), "BKI", nullptr, nullptr, g[EDATTN_WV], "HPI", 1.f},
               {source, at_(dk2), "BKHP", at_(enc), "BKI", nullptr, nullptr, g[EDATTN_WK], "HPI", 1.f},
               {nullptr, at_(dkqv), "QBJHP", at_(x), "BJI", nullptr, nullptr, g[SATTN_WKQV], "QHPI", 1.f},
               {nullptr, at_(datt1), "BJI", at_(k[GAMMA1]), "BJHP", nullptr, nullptr, g[SATTN_WO], "IHP", 1.f},
               {nullptr, at_(dq2), "BJHP", at_(k[NORMED1]), "BJI", nullptr, nullptr, g[EDATTN_WQ], "HPI", 1.f},
               {nullptr, at_(datt2), "BJI", at_(k[GAMMA2]), "BJHP", nullptr, nullptr, g[EDATTN_WO], "IHP", 1.f},
               {nullptr, at_(dlin1), "BJU", at_(k[NORMED2]), "BJI", nullptr, nullptr, g[LINEAR1_W], "UI", 1.f},
               {nullptr, at_(dff), "BJI", at_(k[FF1]), "BJU", nullptr, nullptr, g[LINEAR2_W], "IU", 1.f}});
        deferred.finish();
        return out;
    }
};

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
    py::class_<DecoderPasses> decoder(m, "DecoderPasses");
    decoder
        .def(py::init<uintptr_t, uintptr_t, py::object, const std::vector<int64_t>&, const std::vector<double>&, const std::vector<uint32_t>&, bool,
                      double>())
        .def("forward", &DecoderPasses::forward)
        .def("backward", &DecoderPasses::backward);
    // places in what a forward pass returns
    decoder.attr("MASK1") = (int)DecoderPasses::MASK1;
    decoder.attr("MASK2") = (int)DecoderPasses::MASK2;
    decoder.attr("MASK3") = (int)DecoderPasses::MASK3;
    decoder.attr("BITS") = (int)DecoderPasses::BITS;
    decoder.attr("MASK4") = (int)DecoderPasses::MASK4;
    decoder.attr("OUTPUT") = (int)DecoderPasses::KEPT;
}
