// The host side of eager calls, in native code: allocation, launches and autograd nodes on torch tensors.
//
// A small call is bound by the host.  Autograd runs a backward pass on a thread of its own, so everything a Python
// node touches there (its objects, the interpreter's, the launch path's) moves from one core's caches to another's
// twice per pass: forward and backward of a tiny scan took 167 us as a Python node, of which the forward by itself
// is 20 and the backward by itself 54; a built-in node with one launch each way takes 46.  The nodes here run their
// backward without the interpreter.
//
// What a node takes is what its kernels read in place: plain dense CUDA tensors of the right types.  Everything
// else (other types and layouts, tracing, modes, transforms) stays with the Python functions, to which a backward
// pass that is itself recorded, or is handed a gradient of another kind, goes as well.
//
// The kernels are reached through the C ABI of libhawk_hip.so, by addresses that Python hands over (so that both
// sides use one copy of the library); the workspaces belong to Python and are looked up there once per stream.
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/mm.h>
#include <ATen/ops/zeros.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <optional>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/hawk_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Variable;
using torch::autograd::variable_list;
namespace py = pybind11;

constexpr auto kBF16 = at::kBFloat16;
constexpr auto kF32 = at::kFloat;

// ---------------------------------------------------------------------------------------
// The library and Python's part
// ---------------------------------------------------------------------------------------
#define HAWK_FUNCTIONS(X)                                                                                             \
    X(hawk_scan_workspace_bytes) X(hawk_rglru_scan_fwd_mixed) X(hawk_rglru_scan_bwd_mixed)                            \
    X(hawk_rglru_scan_gated_fwd) X(hawk_rglru_scan_gated_bwd) X(hawk_conv1d_fwd) X(hawk_conv1d_fwd_strided)           \
    X(hawk_conv1d_bwd) X(hawk_conv1d_bwd_workspace_bytes) X(hawk_gate_proj_fwd) X(hawk_gate_weights_to_bf16)          \
    X(hawk_gate_proj_bwd_weights_workspace_bytes) X(hawk_block_core_fwd) X(hawk_block_core_grads)                     \
    X(hawk_block_core_grads_conv_workspace_bytes)                                                                     \
    X(hawk_decode_core_workspace_bytes) X(hawk_decode_core_step_ws) X(hawk_decode_layer_tail)                         \
    X(hawk_decode_norm_linear) X(hawk_cast) X(hawk_add_norm_fwd) X(hawk_add_norm_bwd)                                 \
    X(hawk_add_norm_bwd_workspace_bytes) X(hawk_gelu_mul_fwd) X(hawk_gelu_mul_bwd) X(hawk_cross_entropy_fwd)          \
    X(hawk_cross_entropy_bwd) X(hawk_embedding_bwd) X(hawk_weight_grads) X(hawk_weight_grad_supported)                \
    X(hawk_weight_grads_workspace_bytes) X(hawk_linear_supported) X(hawk_linear_workspace_bytes)           \
    X(hawk_linear_fwd) X(hawk_input_grad) X(hawk_input_grad_workspace_bytes)
struct Library {
#define X(name) decltype(&::name) name = nullptr;
    HAWK_FUNCTIONS(X)
#undef X
};
Library lib;
int64_t placed_from_bytes = 0;   // _lib.activation_empty places tensors from this size on

// Python callables by name; never destroyed (the interpreter may be gone before this library is).
py::dict* python = nullptr;

// Runs f with the interpreter held; an error it raises travels on through C++ as the engine expects it.
template <typename F>
auto in_python(F f) {
    py::gil_scoped_acquire held;
    try {
        return f();
    } catch (py::error_already_set& e) {
        e.restore();
        python_error error;
        error.persist();
        throw error;
    }
}
py::object callable(const char* name) { return (*python)[name]; }

void check(const char* name, int status) {
    if (status != HAWK_OK) in_python([&] { callable("check")(name, status); });
}

// A binding's body, without the interpreter; errors from Python come out as themselves.
template <typename F>
auto entry(F f) {
    try {
        py::gil_scoped_release released;
        return f();
    } catch (python_error& e) {
        e.restore();
        throw py::error_already_set();
    }
}

int code(at::ScalarType t) { return t == kBF16 ? HAWK_DTYPE_BF16 : HAWK_DTYPE_F32; }
template <typename T = void>
T* data(const Tensor& t) { return static_cast<T*>(t.data_ptr()); }
template <typename T = void>
T* data_or_null(const Tensor& t) { return t.defined() && t.numel() > 0 ? static_cast<T*>(t.data_ptr()) : nullptr; }

bool aligned(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

Tensor dense16(const Tensor& t) {
    Tensor d = t.contiguous();
    return aligned(d) ? d : d.clone(at::MemoryFormat::Contiguous);
}
std::vector<Tensor> dense16(const std::vector<Tensor>& ts) {
    std::vector<Tensor> out;
    for (const Tensor& t : ts) out.push_back(dense16(t));
    return out;
}

// Device and stream of a call, and the guards of its body: no autograd, no autocast.
struct Call {
    c10::DeviceGuard guard;
    at::AutoDispatchBelowADInplaceOrView below;
    c10::impl::ExcludeDispatchKeyGuard no_autocast{c10::autocast_dispatch_keyset};
    at::Device dev;
    void* st;
    explicit Call(at::Device d) : guard(d), dev(d), st(c10::hip::getCurrentHIPStream(d.index()).stream()) {}

    Tensor empty(at::IntArrayRef shape, at::ScalarType t) const {
        return at::empty(shape, at::TensorOptions().dtype(t).device(dev));
    }
    // as _lib.activation_empty, which places large ones
    Tensor activation(at::IntArrayRef shape, at::ScalarType t) const {
        if (c10::multiply_integers(shape) * (int64_t)c10::elementSize(t) < placed_from_bytes) return empty(shape, t);
        return in_python([&] {
            return callable("activation_empty")(shape.vec(), t == kBF16, (int)dev.index()).cast<Tensor>();
        });
    }
};

// Workspaces that Python keeps per (device, stream), seen once per stream; inside a capture Python is asked every time.
// Between Python's answer and the entry here another thread may have it replaced or dropped (clear()): such an answer
// serves its call, which holds it, and is not kept.
struct Workspaces {
    const char* name;
    std::mutex mutex;
    std::map<std::pair<int, void*>, Tensor> kept;
    uint64_t cleared = 0;

    explicit Workspaces(const char* n) : name(n) {}
    Tensor get(const Call& c, size_t bytes) {
        const bool capturing = c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None;
        const std::pair<int, void*> key{c.dev.index(), c.st};
        uint64_t before = 0;
        if (!capturing) {
            std::lock_guard<std::mutex> lock(mutex);
            auto it = kept.find(key);
            if (it != kept.end() && (size_t)it->second.numel() >= bytes) return it->second;
            before = cleared;
        }
        // (Python clears in here too, where it makes or replaces a buffer: the stream's next call keeps that one)
        Tensor ws = in_python([&] { return callable(name)((int)c.dev.index(), bytes).cast<Tensor>(); });
        if (!capturing) {
            std::lock_guard<std::mutex> lock(mutex);
            if (cleared == before) kept[key] = ws;
        }
        return ws;
    }
    void clear() {
        std::map<std::pair<int, void*>, Tensor> old;
        std::lock_guard<std::mutex> lock(mutex);
        old.swap(kept);
        ++cleared;
    }
};
Workspaces& scan_workspaces() { static auto* w = new Workspaces("scan_workspace"); return *w; }
Workspaces& gate_workspaces() { static auto* w = new Workspaces("gate_workspace"); return *w; }
Workspaces& decode_workspaces() { static auto* w = new Workspaces("decode_workspace"); return *w; }

// ---------------------------------------------------------------------------------------
// What the nodes take
// ---------------------------------------------------------------------------------------
// Exactly torch.Tensor or Parameter; defined only then.
Tensor exact(const py::handle& h) {
    return THPVariable_CheckExact(h.ptr()) ? THPVariable_Unpack(h.ptr()) : Tensor();
}
// A CUDA tensor without wrapper, lazy conjugate or the like.
bool plain(const Tensor& t) {
    constexpr c10::DispatchKeySet odd({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                       c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
                                       c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                       c10::DispatchKey::ZeroTensor});
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(odd);
}
bool dense(const Tensor& t, at::Device dev, at::ScalarType type) {
    return plain(t) && t.device() == dev && t.scalar_type() == type && t.is_contiguous() && aligned(t);
}
bool dense(const Tensor& t, at::Device dev, at::ScalarType type, at::IntArrayRef shape) {
    return dense(t, dev, type) && t.sizes() == shape;
}
// Elements between consecutive rows of a [B, T, D] tensor whose row b * T + t starts at (b * T + t) times that; 0 if
// it is not laid out like this.  (scan_fused._row_stride is the same in Python, which a tracing compiler sees through.)
int64_t row_stride(const Tensor& t) {
    const int64_t b = t.size(0), sq = t.size(1), d = t.size(2);
    if (t.stride(2) != 1 && d > 1) return 0;
    const int64_t ld = sq > 1 ? t.stride(1) : (b > 1 ? t.stride(0) : d);
    return ld < d || (b > 1 && t.stride(0) != sq * ld) ? 0 : ld;
}
// Whether something watches or rewrites operator calls on this thread; forward passes have looked before they came
// here, a backward pass looks for itself.
bool watched() {
    return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::PythonTorchFunctionTLS::stack_len() != 0 ||
           torch::jit::tracer::isTracing() ||
           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}
// Whether a node's backward can launch on these; otherwise Python's backward function gets them.
bool launches(const variable_list& saved, const Tensor& grad, at::ScalarType type, const Tensor& like) {
    if (at::GradMode::is_enabled() || watched() || !dense(grad, like.device(), type, like.sizes())) return false;
    for (const Tensor& t : saved)
        if (!plain(t) || t.device() != grad.device()) return false;
    return true;
}
variable_list backward_in_python(const char* name, const variable_list& args, size_t gradients) {
    variable_list out = in_python([&] {
        py::tuple packed(args.size());
        for (size_t k = 0; k < args.size(); ++k) packed[k] = py::cast(args[k]);
        py::tuple got = callable(name)(*packed);
        variable_list tensors;
        for (auto g : got) tensors.push_back(g.is_none() ? Tensor() : g.cast<Tensor>());
        return tensors;
    });
    out.resize(gradients);
    return out;
}
Tensor gradient_or_zeros(const Tensor& grad, const Tensor& like, at::ScalarType type) {
    return grad.defined() ? grad : at::zeros(like.sizes(), like.options().dtype(type));
}

// ---------------------------------------------------------------------------------------
// Launches: allocate the outputs, call the library.  (Python's launch functions are these.)
// ---------------------------------------------------------------------------------------
Tensor scan_fwd(const Tensor& x_, const Tensor& xg_, const Tensor& ag_, const Tensor& lam_, bool h_bf16) {
    Call c(x_.device());
    const Tensor x = dense16(x_), xg = dense16(xg_), ag = dense16(ag_), lam = dense16(lam_);
    const int B = x.size(0), T = x.size(1), D = x.size(2), in = code(x.scalar_type());
    const auto out = h_bf16 ? kBF16 : x.scalar_type();
    Tensor h = c.activation(x.sizes(), out);
    const Tensor ws = scan_workspaces().get(c, lib.hawk_scan_workspace_bytes(B, T, D, in));
    check("hawk_rglru_scan_fwd_mixed", lib.hawk_rglru_scan_fwd_mixed(
        data(x), data(xg), data(ag), data<float>(lam), data(h), B, T, D, in, code(out), data(ws), ws.numel(), c.st));
    return h;
}

std::tuple<Tensor, Tensor, Tensor, Tensor> scan_bwd(const Tensor& x_, const Tensor& xg_, const Tensor& ag_,
                                                    const Tensor& lam_, const Tensor& h_, const Tensor& go_) {
    Call c(x_.device());
    const Tensor x = dense16(x_), xg = dense16(xg_), ag = dense16(ag_), lam = dense16(lam_), h = dense16(h_), go = dense16(go_);
    const int B = x.size(0), T = x.size(1), D = x.size(2), in = code(x.scalar_type());
    Tensor dx = c.activation(x.sizes(), x.scalar_type()), dxg = c.activation(x.sizes(), x.scalar_type()),
           dag = c.activation(x.sizes(), x.scalar_type()), dlam = c.empty({D}, kF32);
    const Tensor ws = scan_workspaces().get(c, lib.hawk_scan_workspace_bytes(B, T, D, in));
    check("hawk_rglru_scan_bwd_mixed", lib.hawk_rglru_scan_bwd_mixed(
        data(x), data(xg), data(ag), data<float>(lam), data(h), data(go), data(dx), data(dxg), data(dag),
        data<float>(dlam), B, T, D, in, code(h.scalar_type()), data(ws), ws.numel(), c.st));
    return {dx, dxg, dag, dlam};
}

// y as the gated kernels read it: evenly spaced rows of the state's type, and the distance between them.
std::pair<Tensor, int64_t> gate_rows(const Tensor& y, at::ScalarType type) {
    const Tensor t = y.scalar_type() == type ? y : y.to(type);
    if (const int64_t ld = row_stride(t)) return {t, ld};
    return {dense16(t), t.size(2)};
}

std::tuple<Tensor, Tensor, Tensor> gated_fwd(const Tensor& x_, const Tensor& xg_, const Tensor& ag_, const Tensor& lam_,
                                             const Tensor& y_, bool h_bf16, bool want_h, bool want_last) {
    Call c(x_.device());
    const Tensor x = dense16(x_), xg = dense16(xg_), ag = dense16(ag_), lam = dense16(lam_);
    const int B = x.size(0), T = x.size(1), D = x.size(2), in = code(x.scalar_type());
    const auto type = h_bf16 ? kBF16 : x.scalar_type();
    const auto [y, ldy] = gate_rows(y_, type);
    Tensor out = c.activation(x.sizes(), type), h = want_h ? c.activation(x.sizes(), type) : c.empty({0}, type),
           last = want_last ? c.empty({B, 1, D}, type) : c.empty({0}, type);
    const Tensor ws = scan_workspaces().get(c, lib.hawk_scan_workspace_bytes(B, T, D, in));
    check("hawk_rglru_scan_gated_fwd", lib.hawk_rglru_scan_gated_fwd(
        data(x), data(xg), data(ag), data<float>(lam), data(y), ldy, data_or_null(h), data(out), data_or_null(last), B, T,
        D, in, code(type), data(ws), ws.numel(), c.st));
    return {out, h, last};
}

std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor> gated_bwd(const Tensor& x_, const Tensor& xg_, const Tensor& ag_,
                                                             const Tensor& lam_, const Tensor& y_, const Tensor& h_,
                                                             const Tensor& go_) {
    Call c(x_.device());
    const Tensor x = dense16(x_), xg = dense16(xg_), ag = dense16(ag_), lam = dense16(lam_), h = dense16(h_), go = dense16(go_);
    const int B = x.size(0), T = x.size(1), D = x.size(2), in = code(x.scalar_type());
    const auto [y, ldy] = gate_rows(y_, h.scalar_type());
    Tensor dx = c.activation(x.sizes(), x.scalar_type()), dxg = c.activation(x.sizes(), x.scalar_type()),
           dag = c.activation(x.sizes(), x.scalar_type()), dy = c.activation(x.sizes(), h.scalar_type()),
           dlam = c.empty({D}, kF32);
    const Tensor ws = scan_workspaces().get(c, lib.hawk_scan_workspace_bytes(B, T, D, in));
    check("hawk_rglru_scan_gated_bwd", lib.hawk_rglru_scan_gated_bwd(
        data(x), data(xg), data(ag), data<float>(lam), data(y), ldy, data(h), data(go), data(dx), data(dxg), data(dag),
        data(dy), D, data<float>(dlam), B, T, D, in, code(h.scalar_type()), data(ws), ws.numel(), c.st));
    return {dx, dxg, dag, dlam, dy};
}

Tensor conv_fwd(const Tensor& x_, const Tensor& w_, const Tensor& b_, const std::optional<Tensor>& state_, bool out_fp32) {
    Call c(x_.device());
    const Tensor x = dense16(x_), w = dense16(w_), b = dense16(b_);
    const Tensor state = state_.has_value() ? dense16(*state_) : Tensor();
    const int B = x.size(0), T = x.size(1), D = x.size(2), W = w.size(0);
    const auto type = out_fp32 ? kF32 : kBF16;
    Tensor y = c.activation(x.sizes(), type);
    check("hawk_conv1d_fwd", lib.hawk_conv1d_fwd(data(x), data<float>(w), data<float>(b),
                                                 state.defined() ? data(state) : nullptr, data(y), B, T, D, W,
                                                 code(x.scalar_type()), code(type), c.st));
    return y;
}

std::tuple<Tensor, Tensor, Tensor> conv_bwd(const Tensor& gy_, const Tensor& x_, const Tensor& w_) {
    Call c(x_.device());
    const Tensor gy = dense16(gy_), x = dense16(x_), w = dense16(w_);
    const int B = x.size(0), T = x.size(1), D = x.size(2), W = w.size(0);
    Tensor dx = c.activation(x.sizes(), x.scalar_type()), dw = c.empty({W, D}, kF32), db = c.empty({D}, kF32);
    const Tensor ws = c.empty({(int64_t)lib.hawk_conv1d_bwd_workspace_bytes(B, T, D, W)}, at::kByte);
    check("hawk_conv1d_bwd", lib.hawk_conv1d_bwd(data(gy), data(x), data<float>(w), data(dx), data<float>(dw),
                                                 data<float>(db), B, T, D, W, code(x.scalar_type()),
                                                 code(gy.scalar_type()), data(ws), ws.numel(), c.st));
    return {dx, dw, db};
}

// The core's kernels are told sizes and one type for both gates' weights: everything else they read has to agree with that.
void check_core_sizes(int64_t D, const Tensor& cw, const Tensor& wi, const Tensor& wa, const Tensor& lam) {
    TORCH_CHECK(wi.dim() == 3 && wi.size(1) == wi.size(2) && wi.size(0) * wi.size(1) == D && wa.sizes() == wi.sizes(),
                "gate weights must be [num_blocks, width, width] of ", D, " channels, got ", wi.sizes(), " and ", wa.sizes());
    TORCH_CHECK(wi.scalar_type() == kBF16 || wi.scalar_type() == kF32, "gate weights must be bf16 or fp32, got ", wi.scalar_type());
    TORCH_CHECK(cw.dim() == 2 && cw.size(1) == D && cw.scalar_type() == kF32, "the conv's weight must be fp32 [width, ", D,
                "], got ", cw.sizes());
    TORCH_CHECK(lam.numel() == D && lam.scalar_type() == kF32, "a_param must be fp32 [", D, "], got ", lam.sizes());
}
void check_core_vector(const char* what, const Tensor& t, int64_t D) {
    TORCH_CHECK(t.numel() == D && t.scalar_type() == kF32, what, " must hold ", D, " fp32 values, got ", t.sizes());
}
Tensor as_type(const Tensor& t, at::ScalarType type) { return t.scalar_type() == type ? t : t.to(type); }

constexpr int kFusedConvMinT = 32;   // hawk_block_core_fwd needs T >= 32 and a temporal width of 4

// (out, u, xg, ag, h, h_last)
std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor> core_fwd(
    const Tensor& xy_, const Tensor& cw_, const Tensor& cb_, const Tensor& wi_, const Tensor& bi_, const Tensor& wa_,
    const Tensor& ba_, const Tensor& lam_, bool want_h, bool want_last) {
    Call c(xy_.device());
    const Tensor xy = aligned(xy_) ? xy_ : xy_.clone(at::MemoryFormat::Contiguous);
    const int64_t B = xy.size(0), T = xy.size(1), D = xy.size(2) / 2, ld = row_stride(xy);
    TORCH_CHECK(xy.scalar_type() == kBF16, "xy must be bf16");
    check_core_sizes(D, cw_, wi_, wa_, lam_);
    check_core_vector("the conv's bias", cb_, D);
    check_core_vector("a gate's bias", bi_, D);
    check_core_vector("a gate's bias", ba_, D);
    const Tensor cw = dense16(cw_), cb = dense16(cb_), wi = dense16(wi_), bi = dense16(bi_),
                 wa = dense16(as_type(wa_, wi_.scalar_type())), ba = dense16(ba_), lam = dense16(lam_);
    const int W = cw.size(0), nb = wi.size(0), wt = code(wi.scalar_type()), bf = HAWK_DTYPE_BF16;
    Tensor u = c.activation({B, T, D}, kBF16), xg = c.activation({B, T, D}, kBF16), ag = c.activation({B, T, D}, kBF16),
           out = c.activation({B, T, D}, kBF16), h = want_h ? c.activation({B, T, D}, kBF16) : c.empty({0}, kBF16),
           last = want_last ? c.empty({B, 1, D}, kBF16) : c.empty({0}, kBF16);
    const Tensor ws = scan_workspaces().get(c, lib.hawk_scan_workspace_bytes(B, T, D, bf));
    if (W == 4 && T >= kFusedConvMinT) {
        // conv and both projections, then the gated scan, in one call
        check("hawk_block_core_fwd", lib.hawk_block_core_fwd(
            data(xy), ld, data<float>(cw), data<float>(cb), data(wi), data<float>(bi), data(wa), data<float>(ba), wt,
            nullptr, data<float>(lam), data(u), data(xg), data(ag), data_or_null(h), data(out), data_or_null(last), B, T, D,
            nb, W, data(ws), ws.numel(), c.st));
    } else {
        check("hawk_conv1d_fwd_strided", lib.hawk_conv1d_fwd_strided(
            data(xy), ld, data<float>(cw), data<float>(cb), nullptr, data(u), D, B, T, D, W, bf, bf, c.st));
        check("hawk_gate_proj_fwd", lib.hawk_gate_proj_fwd(data(u), data(wi), data<float>(bi), data(wa), data<float>(ba),
                                                           data(xg), data(ag), B * T, D, nb, bf, wt, bf, c.st));
        check("hawk_rglru_scan_gated_fwd", lib.hawk_rglru_scan_gated_fwd(
            data(u), data(xg), data(ag), data<float>(lam), static_cast<char*>(data(xy)) + 2 * D, ld, data_or_null(h),
            data(out), data_or_null(last), B, T, D, bf, bf, data(ws), ws.numel(), c.st));
    }
    return {out, u, xg, ag, h, last};
}

// (d_xy, d_conv_w, d_conv_b, dw_i, db_i, dw_a, db_a, dlam).  What the forward pass saved may come back in another layout:
// hooks that pack saved tensors return what they like.
std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor> core_bwd(
    const Tensor& xy_, const Tensor& u_, const Tensor& xg_, const Tensor& ag_, const Tensor& h_, const Tensor& cw_,
    const Tensor& wi_, const Tensor& wa_, const Tensor& lam_, const Tensor& go_) {
    Call c(xy_.device());
    const Tensor xy = aligned(xy_) && row_stride(xy_) % 8 == 0 && row_stride(xy_) > 0 ? xy_ : xy_.clone(at::MemoryFormat::Contiguous);
    const int64_t B = xy.size(0), T = xy.size(1), D = xy.size(2) / 2;
    check_core_sizes(D, cw_, wi_, wa_, lam_);
    const at::IntArrayRef states[] = {u_.sizes(), xg_.sizes(), ag_.sizes(), h_.sizes(), go_.sizes()};
    for (const auto& size : states) TORCH_CHECK(size == at::IntArrayRef({B, T, D}), "expected [", B, ", ", T, ", ", D, "], got ", size);
    for (const Tensor* t : {&xy_, &u_, &xg_, &ag_, &h_, &go_}) TORCH_CHECK(t->scalar_type() == kBF16, "the core's tensors must be bf16");
    const Tensor u = dense16(u_), xg = dense16(xg_), ag = dense16(ag_), h = dense16(h_), cw = dense16(cw_), wi = dense16(wi_),
                 wa = dense16(as_type(wa_, wi_.scalar_type())), lam = dense16(lam_), go = dense16(go_);
    const int64_t W = cw.size(0), nb = wi.size(0), bw = wi.size(1);
    Tensor d_xy = c.activation(xy.sizes(), kBF16), du = c.activation({B, T, D}, kBF16), dxg = c.activation({B, T, D}, kBF16),
           dag = c.activation({B, T, D}, kBF16);
    Tensor dlam = c.empty({D}, kF32), dwi = c.empty({nb, bw, bw}, kF32), dwa = c.empty({nb, bw, bw}, kF32),
           dbi = c.empty({D}, kF32), dba = c.empty({D}, kF32), dcb = c.empty({D}, kF32), dcw = c.empty({W, D}, kF32);
    const Tensor ws = scan_workspaces().get(c, lib.hawk_scan_workspace_bytes(B, T, D, HAWK_DTYPE_BF16));
    const Tensor gws = gate_workspaces().get(c, lib.hawk_gate_proj_bwd_weights_workspace_bytes(B * T, D, nb));
    const Tensor cws = c.empty({(int64_t)lib.hawk_block_core_grads_conv_workspace_bytes(B, T, D, W)}, at::kByte);
    // scan (with the output gate) -> projections' input gradient onto the scan's and the conv ->
    // projections' weight gradients, and one launch for the three closing reductions
    check("hawk_block_core_grads", lib.hawk_block_core_grads(
        data(xy), row_stride(xy), data(u), data(xg), data(ag), data(h), data<float>(cw), data(wi), data(wa),
        code(wi.scalar_type()), data<float>(lam), data(go), data(d_xy), 2 * D, data(du), data(dxg), data(dag),
        data<float>(dcw), data<float>(dcb), data<float>(dwi), data<float>(dbi), data<float>(dwa), data<float>(dba),
        data<float>(dlam), B, T, D, nb, W, data(ws), ws.numel(), data(gws), gws.numel(), data(cws), cws.numel(), c.st));
    return {d_xy, dcw, dcb, dwi, dbi, dwa, dba, dlam};
}

// Both gates' fp32 weights rounded to bf16 by one launch.
std::tuple<Tensor, Tensor> gate_weights_to_bf16(const Tensor& wi_, const Tensor& wa_) {
    Call c(wi_.device());
    const Tensor wi = dense16(wi_), wa = dense16(wa_);
    const int64_t nb = wi.size(0), bw = wi.size(1);
    const Tensor both = c.empty({2, nb, bw, bw}, kBF16);
    const Tensor i = both.select(0, 0), a = both.select(0, 1);
    check("hawk_gate_weights_to_bf16", lib.hawk_gate_weights_to_bf16(data<float>(wi), data<float>(wa), data(i), data(a),
                                                                     nb, bw, c.st));
    return {i, a};
}

// ---------------------------------------------------------------------------------------
// Autograd nodes
// ---------------------------------------------------------------------------------------
struct Scan : torch::autograd::Function<Scan> {
    static Variable forward(AutogradContext* ctx, const Variable& x, const Variable& xg, const Variable& ag,
                            const Variable& lam, bool h_bf16) {
        ctx->set_materialize_grads(false);
        Tensor h = scan_fwd(x, xg, ag, lam, h_bf16);
        ctx->save_for_backward({x, xg, ag, lam, h});
        return h;
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        const variable_list s = ctx->get_saved_variables();
        const Tensor go = gradient_or_zeros(grads[0], s[4], s[4].scalar_type());
        if (!launches(s, go, s[4].scalar_type(), s[4]))
            return backward_in_python("scan_backward", {s[0], s[1], s[2], s[3], s[4], go}, 5);
        auto [dx, dxg, dag, dlam] = scan_bwd(s[0], s[1], s[2], s[3], s[4], go);
        return {dx, dxg, dag, dlam, Tensor()};
    }
};

struct GatedScan : torch::autograd::Function<GatedScan> {
    static variable_list forward(AutogradContext* ctx, const Variable& x, const Variable& xg, const Variable& ag,
                                 const Variable& lam, const Variable& y, bool h_bf16, bool want_h, bool want_last) {
        ctx->set_materialize_grads(false);
        auto [out, h, last] = gated_fwd(x, xg, ag, lam, y, h_bf16, want_h, want_last);
        if (want_h) ctx->save_for_backward({x, xg, ag, lam, y, h});
        ctx->mark_non_differentiable({last});
        return {out, last};
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        const variable_list s = ctx->get_saved_variables();
        const Tensor go = gradient_or_zeros(grads[0], s[5], s[5].scalar_type());
        if (!launches(s, go, s[5].scalar_type(), s[5]))
            return backward_in_python("gated_backward", {s[0], s[1], s[2], s[3], s[4], s[5], go}, 8);
        auto [dx, dxg, dag, dlam, dy] = gated_bwd(s[0], s[1], s[2], s[3], s[4], s[5], go);
        return {dx, dxg, dag, dlam, dy, Tensor(), Tensor(), Tensor()};
    }
};

struct Conv : torch::autograd::Function<Conv> {
    static Variable forward(AutogradContext* ctx, const Variable& x, const Variable& w, const Variable& b, bool out_fp32) {
        ctx->set_materialize_grads(false);
        ctx->save_for_backward({x, w});
        ctx->saved_data["type"] = (int64_t)(out_fp32 ? kF32 : kBF16);
        return conv_fwd(x, w, b, std::nullopt, out_fp32);
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        const variable_list s = ctx->get_saved_variables();
        const auto type = (at::ScalarType)ctx->saved_data["type"].toInt();
        const Tensor go = gradient_or_zeros(grads[0], s[0], type);
        if (!launches(s, go, type, s[0])) return backward_in_python("conv_backward", {go, s[0], s[1]}, 4);
        auto [dx, dw, db] = conv_bwd(go, s[0], s[1]);
        return {dx, dw, db, Tensor()};
    }
};

// What the forward pass of a core has computed, handed to its node past autograd.
struct CoreResult {
    Tensor out, u, xg, ag, h, last;
    Tensor cw, wi, wa, lam;    // as the kernels read them
};

struct Core : torch::autograd::Function<Core> {
    static variable_list forward(AutogradContext* ctx, const Variable& xy, const Variable& cw, const Variable& cb,
                                 const Variable& wi, const Variable& bi, const Variable& wa, const Variable& ba,
                                 const Variable& lam, const CoreResult& r) {
        ctx->set_materialize_grads(false);
        ctx->save_for_backward({xy, r.u, r.xg, r.ag, r.h, r.cw, r.wi, r.wa, r.lam});
        std::vector<int64_t> types;
        for (const Tensor* t : {&cw, &cb, &wi, &bi, &wa, &ba, &lam}) types.push_back((int64_t)t->scalar_type());
        ctx->saved_data["types"] = types;
        ctx->mark_non_differentiable({r.last});
        return {r.out, r.last};
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        const variable_list s = ctx->get_saved_variables();
        const Tensor go = gradient_or_zeros(grads[0], s[4], kBF16);
        variable_list g;
        if (launches(s, go, kBF16, s[4])) {
            auto [d_xy, dcw, dcb, dwi, dbi, dwa, dba, dlam] = core_bwd(s[0], s[1], s[2], s[3], s[4], s[5], s[6], s[7], s[8], go);
            g = {d_xy, dcw, dcb, dwi, dbi, dwa, dba, dlam};
        } else {
            g = backward_in_python("core_backward", {s[0], s[1], s[2], s[3], s[4], s[5], s[6], s[7], s[8], go}, 8);
        }
        const std::vector<int64_t> types = ctx->saved_data["types"].toIntVector();
        const int64_t nb = s[6].size(0), bw = s[6].size(1);
        for (size_t k = 1; k < 8; ++k) {
            if (k == 4 || k == 6) g[k] = g[k].reshape({nb, bw});
            const auto type = (at::ScalarType)types[k - 1];
            if (g[k].scalar_type() != type) g[k] = g[k].to(type);
        }
        g.emplace_back();
        return g;
    }
};

// ---------------------------------------------------------------------------------------
// Entries of the nodes: None where the operands are not what the kernels read in place
// ---------------------------------------------------------------------------------------
bool scan_operands(const Tensor& x, const Tensor& xg, const Tensor& ag, const Tensor& lam) {
    if (!plain(x) || x.dim() != 3 || x.numel() == 0 || x.size(2) % 64 != 0) return false;
    const auto type = x.scalar_type();
    return (type == kBF16 || type == kF32) && dense(x, x.device(), type) && dense(xg, x.device(), type, x.sizes()) &&
           dense(ag, x.device(), type, x.sizes()) && dense(lam, x.device(), kF32, {x.size(2)});
}

py::object scan_node(py::handle x_, py::handle xg_, py::handle ag_, py::handle lam_) {
    const Tensor x = exact(x_), xg = exact(xg_), ag = exact(ag_), lam = exact(lam_);
    if (!scan_operands(x, xg, ag, lam)) return py::none();
    const bool h_bf16 = x.scalar_type() == kBF16 || at::autocast::is_autocast_enabled(at::kCUDA);
    return py::cast(entry([&] { return Scan::apply(x, xg, ag, lam, h_bf16); }));
}

py::object gated_node(py::handle x_, py::handle xg_, py::handle ag_, py::handle lam_, py::handle y_, bool want_last) {
    const Tensor x = exact(x_), xg = exact(xg_), ag = exact(ag_), lam = exact(lam_), y = exact(y_);
    if (!scan_operands(x, xg, ag, lam)) return py::none();
    const bool h_bf16 = x.scalar_type() == kBF16 || at::autocast::is_autocast_enabled(at::kCUDA);
    const auto type = h_bf16 ? kBF16 : kF32;
    if (!plain(y) || y.device() != x.device() || y.scalar_type() != type || y.sizes() != x.sizes() || row_stride(y) == 0)
        return py::none();
    bool want_h = false;
    if (at::GradMode::is_enabled())
        for (const Tensor* t : {&x, &xg, &ag, &lam, &y}) want_h |= t->requires_grad();
    const variable_list out = entry([&] { return GatedScan::apply(x, xg, ag, lam, y, h_bf16, want_h, want_last); });
    return py::make_tuple(out[0], out[1]);
}

py::object conv_node(py::handle x_, py::handle w_, py::handle b_, bool out_fp32) {
    const Tensor x = exact(x_), w = exact(w_), b = exact(b_);
    if (!plain(x) || x.dim() != 3 || x.numel() == 0) return py::none();
    const auto type = x.scalar_type();
    if ((type != kBF16 && type != kF32) || !dense(x, x.device(), type) || !dense(w, x.device(), kF32) || w.dim() != 2 ||
        w.size(1) != x.size(2) || !dense(b, x.device(), kF32, {x.size(2)}))
        return py::none();
    return py::cast(entry([&] { return Conv::apply(x, w, b, out_fp32); }));
}

// The node of a core whose forward pass has run: (out, h_last).
py::object core_node(const std::vector<Tensor>& params, const std::vector<Tensor>& result, const std::vector<Tensor>& read) {
    const CoreResult r{result[0], result[1], result[2], result[3], result[4], result[5], read[0], read[1], read[2], read[3]};
    const variable_list out = entry([&] {
        return Core::apply(params[0], params[1], params[2], params[3], params[4], params[5], params[6], params[7], r);
    });
    return py::make_tuple(out[0], out[1]);
}

// ---------------------------------------------------------------------------------------
// Decode steps
// ---------------------------------------------------------------------------------------
// A parameter that a kernel reads as it is: exactly a Parameter or tensor of this type, shape and device, dense, aligned.
bool dense_parameter(py::handle t_, const std::vector<int64_t>& shape, bool bf16, int index) {
    const Tensor t = exact(t_);
    return t.defined() && t.is_cuda() && t.get_device() == index && t.scalar_type() == (bf16 ? kBF16 : kF32) &&
           t.sizes() == at::IntArrayRef(shape) && t.is_contiguous() && aligned(t);
}

// Distance between the rows of a bf16 [B, 1, D] tensor with unit column stride, 0 if it is none.
int64_t decode_rows(const Tensor& t, at::Device dev, int64_t B, int64_t D) {
    if (!plain(t) || t.device() != dev || t.scalar_type() != kBF16 || t.sizes() != at::IntArrayRef({B, 1, D}) ||
        t.stride(2) != 1 || t.stride(0) < D)
        return 0;
    return B > 1 ? t.stride(0) : D;
}

// One decode step of a recurrent core; None where an operand is not dense or of another type.
py::object decode_core(py::handle x_, py::handle y_, py::handle conv_state_, py::handle state_, py::handle cw_,
                       py::handle cb_, py::handle wi_, py::handle bi_, py::handle wa_, py::handle ba_, py::handle lam_) {
    const Tensor x = exact(x_), y = exact(y_), conv_state = exact(conv_state_), state = exact(state_), cw = exact(cw_),
                 cb = exact(cb_), wi = exact(wi_), bi = exact(bi_), wa = exact(wa_), ba = exact(ba_), lam = exact(lam_);
    if (!plain(x) || x.dim() != 3 || x.numel() == 0 || !plain(cw) || cw.dim() != 2 || !plain(wi) || wi.dim() != 3 ||
        !plain(state))
        return py::none();
    const at::Device dev = x.device();
    const int64_t B = x.size(0), D = cw.size(1), W = cw.size(0), nb = wi.size(0), bw = wi.size(1);
    const auto wt = wi.scalar_type(), stt = state.scalar_type();
    const int64_t ldx = decode_rows(x, dev, B, D), ldy = decode_rows(y, dev, B, D);
    if (nb * bw != D || (bw != 32 && bw != 64 && bw != 128 && bw != 256) || W < 1 || W > 8 || (wt != kBF16 && wt != kF32) ||
        (stt != kBF16 && stt != kF32) || ldx == 0 || ldx % 8 != 0 || !aligned(x) || ldy == 0 ||
        !dense(conv_state, dev, kBF16, {B, W - 1, D}) || !dense(state, dev, stt) || state.numel() != B * D ||
        !dense(cw, dev, kF32) || !dense(cb, dev, kF32, {D}) || !dense(wi, dev, wt, {nb, bw, bw}) ||
        !dense(wa, dev, wt, {nb, bw, bw}) || !dense(bi, dev, kF32, {nb, bw}) || !dense(ba, dev, kF32, {nb, bw}) ||
        !dense(lam, dev, kF32, {D}))
        return py::none();
    return py::cast(entry([&] {
        Call c(dev);
        Tensor out = c.empty({B, 1, D}, kBF16);
        const Tensor ws = decode_workspaces().get(c, lib.hawk_decode_core_workspace_bytes(B, D, nb));
        check("hawk_decode_core_step_ws", lib.hawk_decode_core_step_ws(
            data(conv_state), data(x), ldx, data<float>(cw), data<float>(cb), data(wi), data<float>(bi), data(wa),
            data<float>(ba), data<float>(lam), data(y), ldy, data(state), data(out), B, D, nb, W, HAWK_DTYPE_BF16, code(wt),
            code(stt), data(ws), ws.numel(), c.st));
        return out;
    }));
}

Tensor decode_first(const Tensor& hidden, const Tensor& norm, double eps, const Tensor& w, const Tensor& ws) {
    Call c(hidden.device());
    const int M = hidden.size(0), H = hidden.size(1), N = w.size(0);
    Tensor out = c.empty({M, N}, kBF16);
    check("hawk_decode_norm_linear", lib.hawk_decode_norm_linear(data(hidden), data(norm), (float)eps, data(w), data(out),
                                                                 M, N, H, data(ws), ws.numel(), c.st));
    return out;
}

Tensor decode_tail(const Tensor& hidden, const Tensor& gated, const Tensor& w_resid, const Tensor& norm, double eps,
                   const Tensor& w_gate_up, const Tensor& w_down, const Tensor& next_norm, double next_eps,
                   const Tensor& w_next, const Tensor& ws, int R, int inter) {
    Call c(hidden.device());
    const int M = hidden.size(0), H = hidden.size(1), N = w_next.size(0);
    Tensor out = c.empty({M, N}, kBF16);
    check("hawk_decode_layer_tail", lib.hawk_decode_layer_tail(
        data(gated), data(w_resid), data(hidden), data(norm), (float)eps, data(w_gate_up), data(w_down), data(next_norm),
        (float)next_eps, data(w_next), data(out), M, H, R, inter, N, data(ws), ws.numel(), c.st));
    return out;
}

// ---------------------------------------------------------------------------------------
// Training passes (train_fused.py holds the nodes)
// ---------------------------------------------------------------------------------------
// Dense, 16-byte aligned tensors of one type (fp32 or bf16) in the other, by one launch.
std::vector<Tensor> cast_in(const Call& c, const std::vector<Tensor>& in, at::ScalarType type) {
    std::vector<Tensor> out;
    std::vector<const void*> src;
    std::vector<void*> dst;
    std::vector<unsigned long long> counts;
    for (const Tensor& t : in) {
        out.push_back(c.empty(t.sizes(), type));
        src.push_back(data(t));
        dst.push_back(data(out.back()));
        counts.push_back(t.numel());
    }
    check("hawk_cast", lib.hawk_cast(src.data(), dst.data(), counts.data(), (int)in.size(), type == kBF16, c.st));
    return out;
}

// (hidden + delta, its norm in bf16, 1 / rms) of [n, D] rows.
std::tuple<Tensor, Tensor, Tensor> add_norm(const Tensor& hidden, const std::optional<Tensor>& delta, const Tensor& weight,
                                            double eps) {
    Call c(hidden.device());
    const int n = hidden.size(0), D = hidden.size(1);
    Tensor total = delta.has_value() ? c.empty({n, D}, kF32) : hidden, out = c.empty({n, D}, kBF16), rstd = c.empty({n}, kF32);
    check("hawk_add_norm_fwd", lib.hawk_add_norm_fwd(
        data<float>(hidden), delta.has_value() ? data(*delta) : nullptr, data<float>(weight), (float)eps,
        delta.has_value() ? data<float>(total) : nullptr, data(out), data<float>(rstd), n, D, c.st));
    return {total, out, rstd};
}

// (gradient of the sum in fp32, its bf16 rounding, gradient of the weight)
std::tuple<Tensor, std::optional<Tensor>, Tensor> add_norm_bwd(const Tensor& dout, const Tensor& total, const Tensor& rstd,
                                                               const Tensor& weight, const std::optional<Tensor>& direct,
                                                               bool want_delta) {
    Call c(total.device());
    const int n = total.size(0), D = total.size(1);
    Tensor d_sum = c.empty({n, D}, kF32), d_weight = c.empty({D}, kF32);
    std::optional<Tensor> d_delta;
    if (want_delta) d_delta = c.empty({n, D}, kBF16);
    const Tensor ws = c.empty({(int64_t)lib.hawk_add_norm_bwd_workspace_bytes(n, D)}, at::kByte);
    check("hawk_add_norm_bwd", lib.hawk_add_norm_bwd(
        data(dout), data<float>(total), data<float>(rstd), data<float>(weight),
        direct.has_value() ? data<float>(*direct) : nullptr, data<float>(d_sum), want_delta ? data(*d_delta) : nullptr,
        data<float>(d_weight), n, D, data(ws), ws.numel(), c.st));
    return {d_sum, d_delta, d_weight};
}

// Whether the library's product, with its result in fp32, takes a weight gradient [rows, columns] over a sum of n: results
// of more than 256 tiles of 128 x 128 over more than 2048 rows, or 4096 and more wide both ways over more than 1024.
// Kernel / library in us, replayed:
//   the four weights of a layer in one launch, or those of more than 256 tiles by the library
//              1024 channels, MLP 2048: 45 / 43 at 1100 rows, 53 / 49 at 1500, 130 / 130 at 4096 (all four by the library
//              77, 96, 167); 1536 and 4608: 115 / 128, 127 / 160, 292 / 298; 2560 and 7680: 273 / 291, 345 / 364, at 2048
//              431 / 396, at 3000 618 / 599; 4096 and 12288: 700 / 567, 885 / 708, 1111 / 825, 1532 / 1177; 5120 and 15360
//              1027 / 945, 1305 / 1187, 1684 / 1352
//   a head's   32000 x 512 65 / 54 at 1100 rows, 78 / 66 at 1500, 97 / 79 at 2048, 171 / 146 at 4096; 32000 x 768 91 / 87,
//              111 / 126, 135 / 116; 8192 x 1024 32 / 34, 37 / 43, 52 / 44; 32000 x 4096 462 / 366, 576 / 461, 727 / 538
// Up to 2048 rows of a narrow head the difference does not show in a pass (two layers, replayed, kernel and library: 512
// channels 756 / 761 at 1100 rows, 814 / 818 at 1500, 905 / 902 at 2048; 768 921 / 941, 1030 / 1066, 1200 / 1191; 1024
// 1124 / 1131, 1283 / 1278, 1434 / 1411), and the library's call costs the host 13 us more.
bool library_weight_grad(int64_t n, int64_t rows, int64_t columns) {
    const int64_t tiles = ((rows + 127) / 128) * ((columns + 127) / 128);
    return tiles > 256 && (n > 2048 || (n > 1024 && std::min(rows, columns) >= 4096));
}
// dy^T x of [n, N] and [n, K] each, in fp32: together in one launch, but for those that the library takes.
std::vector<Tensor> weight_grads(const std::vector<std::pair<Tensor, Tensor>>& products) {
    Call c(products[0].first.device());
    const int n = products[0].first.size(0);
    std::vector<Tensor> out(products.size());
    std::vector<const void*> dy, x;
    std::vector<float*> dw;
    std::vector<int> N, K;
    for (size_t k = 0; k < products.size(); ++k) {
        const auto& [g, in] = products[k];
        const int rows = g.size(1), cols = in.size(1);
        if (library_weight_grad(n, rows, cols) || !lib.hawk_weight_grad_supported(n, rows, cols)) {
            out[k] = at::mm(g.t(), in, kF32);
            continue;
        }
        out[k] = c.empty({rows, cols}, kF32);
        dy.push_back(data(g)), x.push_back(data(in)), dw.push_back(data<float>(out[k])), N.push_back(rows), K.push_back(cols);
    }
    if (dy.empty()) return out;
    const size_t bytes = lib.hawk_weight_grads_workspace_bytes(dy.size(), n, N.data(), K.data());
    const Tensor ws = c.empty({(int64_t)bytes}, at::kByte);
    check("hawk_weight_grads", lib.hawk_weight_grads(dy.size(), dy.data(), x.data(), dw.data(), n, N.data(), K.data(),
                                                     data_or_null(ws), bytes, c.st));
    return out;
}
Tensor weight_grad(const Tensor& dy, const Tensor& x) { return weight_grads({{dy, x}})[0]; }

// x w^T of [n, K] and [N, K], and dy w of [n, N] and [N, K]: by own kernels up to 256 tiles of 128 x 128 of results; their
// launch costs the host 4 us, a library product 17.
// An input gradient's operand lies across the sum, and the library's products of that kind are the slower ones: of 120
// sizes of 512 to 4096 channels and heads of 32000 at 100 to 4096 rows the kernels are ahead at 98 (dx of 15360 x 2560 at
// 1024 rows 146 / 204 us, 9216 x 1536 at 512 41 / 61, 32000 x 512 at 2048 107 / 210), level within 9 % at 17 and behind at
// five (4096 x 1024 at 1500 and 3000 rows 33 / 28 and 47 / 41, 2560 x 2560 at 1500 41 / 29).
bool own_product(int64_t rows, int64_t columns, int64_t sum) {
    return ((rows + 127) / 128) * ((columns + 127) / 128) <= 256 && lib.hawk_linear_supported(rows, columns, sum);
}
// An output's operands lie along the sum.  The kernels are ahead up to 2^31 multiply-adds (own / library in us: 1024 x 1024 at
// 1024 rows 7.1 / 9.0 and at 2048 10.3 / 10.6, 4096 x 1024 at 512 10.0 / 10.7, 1024 x 512 at 4096 9.7 / 11.1, 9216 x 1536
// at 100 16.3 / 18.7), 1 to 4 us behind from there to 2^32 (2048 x 1024 at 2048 15.2 / 13.1, 2560 x 2560 at 512 18.5 / 15.5,
// 15360 x 2560 at 100 30.6 / 25.0), less than their launch saves the host (with the line at 2^31 passes of three layers
// of 768 over 2000 rows took 1430 us instead of 1414, of 1024 over 1500 rows 1567 instead of 1551), and further beyond
// (1536 x 4608 at 1024 37.7 / 28.0, 2560 x 7680 at 1024 79.0 / 63.4, 32000 x 4096 at 100 72.8 / 57.4), but for one tile of
// rows over a sum longer than the row of results, which they split (4096 x 12288 at 100 32.4 / 41.6).
bool own_output(int64_t rows, int64_t columns, int64_t sum) {
    return own_product(rows, columns, sum) && (rows * columns * sum <= (int64_t)1 << 32 || (rows <= 128 && sum > columns));
}
Tensor layer_linear(const Tensor& x, const Tensor& w) {
    const int n = x.size(0), N = w.size(0), K = w.size(1);
    if (!own_output(n, N, K)) return at::mm(x, w.t());
    Call c(x.device());
    Tensor out = c.empty({n, N}, kBF16);
    const size_t bytes = lib.hawk_linear_workspace_bytes(n, N, K);
    const Tensor ws = bytes > 0 ? c.empty({(int64_t)bytes}, at::kByte) : Tensor();
    check("hawk_linear_fwd", lib.hawk_linear_fwd(data(x), data(w), data(out), n, N, K, data_or_null(ws), bytes, c.st));
    return out;
}
Tensor input_grad(const Tensor& dy, const Tensor& w) {
    const int n = dy.size(0), N = w.size(0), K = w.size(1);
    if (!own_product(n, K, N)) return at::mm(dy, w);
    Call c(dy.device());
    Tensor dx = c.empty({n, K}, kBF16);
    const size_t bytes = lib.hawk_input_grad_workspace_bytes(n, N, K);
    const Tensor ws = bytes > 0 ? c.empty({(int64_t)bytes}, at::kByte) : Tensor();
    check("hawk_input_grad", lib.hawk_input_grad(data(dy), data(w), data(dx), n, N, K, data_or_null(ws), bytes, c.st));
    return dx;
}

Tensor gelu_mul(const Tensor& gu, int rows, int inter) {
    Call c(gu.device());
    Tensor act = c.empty({rows, inter}, kBF16);
    check("hawk_gelu_mul_fwd", lib.hawk_gelu_mul_fwd(data(gu), data(act), rows, inter, c.st));
    return act;
}

// A layer's forward pass.  params: n1, n2, w_in, w_out, w_gu, w_dn, cw, cb, wi, bi, wa, ba, lam; wi and wa as the
// kernels read them.  Returns (total2, out) and what the backward reads: w_in16, w_out16, w_gu16, w_dn16, total1, x1,
// rstd1, xy, u, xg, ag, h, gated, x2, rstd2, gu, act.
std::vector<Tensor> layer_fwd(const Tensor& hidden, const std::optional<Tensor>& delta, double eps1, double eps2,
                              const std::vector<Tensor>& p, bool want_h) {
    Call c(hidden.device());
    const int64_t B = hidden.size(0), T = hidden.size(1), H = hidden.size(2), rows = B * T, R = p[3].size(1), inter = p[5].size(1);
    const std::vector<Tensor> w16 = cast_in(c, {p[2], p[3], p[4], p[5]}, kBF16);
    std::optional<Tensor> d;
    if (delta.has_value()) d = delta->view({rows, H});
    auto [total1, x1, rstd1] = add_norm(hidden.view({rows, H}), d, p[0], eps1);
    const Tensor xy = layer_linear(x1, w16[0]).view({B, T, 2 * R});
    auto [gated, u, xg, ag, h, last] = core_fwd(xy, p[6], p[7], p[8], p[9], p[10], p[11], p[12], want_h, false);
    const Tensor mixed = layer_linear(gated.view({rows, R}), w16[1]);
    auto [total2, x2, rstd2] = add_norm(total1, mixed, p[1], eps2);
    const Tensor gu = layer_linear(x2, w16[2]);
    const Tensor act = gelu_mul(gu, rows, inter);
    const Tensor out = layer_linear(act, w16[3]);
    return {total2.view({B, T, H}), out.view({B, T, H}), w16[0], w16[1], w16[2], w16[3], total1, x1, rstd1, xy, u, xg, ag, h,
            gated, total2, x2, rstd2, gu, act};
}

// Its backward pass.  s: n1, n2, cw, lam, wi, wa and what layer_fwd returned behind (total2, out), in its order.
// Returns d_hidden, d_delta (undefined without want_delta), d_n1, d_n2, d_w_in, d_w_out, d_w_gu, d_w_dn, d_cw, d_cb,
// d_wi, d_bi, d_wa, d_ba, d_lam, all in fp32 but d_delta.
std::vector<Tensor> layer_bwd(const std::vector<Tensor>& saved, const Tensor& d_total_, const Tensor& d_out_, bool want_delta) {
    Call c(d_total_.device());
    const std::vector<Tensor> s = dense16(saved);
    const Tensor &n1 = s[0], &n2 = s[1], &cw = s[2], &lam = s[3], &wi = s[4], &wa = s[5], &w_in = s[6], &w_out = s[7],
                 &w_gu = s[8], &w_dn = s[9], &total1 = s[10], &x1 = s[11], &rstd1 = s[12], &xy = s[13], &u = s[14],
                 &xg = s[15], &ag = s[16], &h = s[17], &gated = s[18], &total2 = s[19], &x2 = s[20], &rstd2 = s[21],
                 &gu = s[22], &act = s[23];
    const int64_t B = xy.size(0), T = xy.size(1), rows = B * T, H = total1.size(1), R = gated.size(2), inter = act.size(1);
    auto as = [&](const Tensor& t, at::ScalarType type) { return dense16(t.scalar_type() == type ? t : t.to(type)).view({rows, H}); };
    const Tensor d_total = as(d_total_, kF32), d_out = as(d_out_, kBF16);
    const Tensor d_act = input_grad(d_out, w_dn);
    const Tensor d_gu = c.empty(gu.sizes(), kBF16);
    check("hawk_gelu_mul_bwd", lib.hawk_gelu_mul_bwd(data(gu), data(d_act), data(d_gu), rows, inter, c.st));
    const Tensor d_x2 = input_grad(d_gu, w_gu);
    auto [d_total1, d_mixed, g_n2] = add_norm_bwd(d_x2, total2, rstd2, n2, d_total, true);
    const Tensor d_gated = input_grad(*d_mixed, w_out);
    auto [d_xy_, dcw, dcb, dwi, dbi, dwa, dba, dlam] = core_bwd(xy, u, xg, ag, h, cw, wi, wa, lam, d_gated.view({B, T, R}));
    const Tensor d_xy = d_xy_.view({rows, 2 * R});
    const Tensor d_x1 = input_grad(d_xy, w_in);
    // (all four at the end: each alone is too few tiles for the chip)
    const std::vector<Tensor> g = weight_grads({{d_gu, x2}, {d_out, act}, {d_xy, x1}, {*d_mixed, gated.view({rows, R})}});
    auto [d_hidden, d_delta, g_n1] = add_norm_bwd(d_x1, total1, rstd1, n1, d_total1, want_delta);
    const int64_t nb = wi.size(0), bw = wi.size(1);
    return {d_hidden.view({B, T, H}), d_delta.has_value() ? d_delta->view({B, T, H}) : Tensor(), g_n1, g_n2, g[2], g[3], g[0],
            g[1], dcw, dcb, dwi, dbi.view({nb, bw}), dwa, dba.view({nb, bw}), dlam};
}

// Final norm, head and mean cross entropy: the loss and head16, total, x, rstd, logits, lse, mean.
std::vector<Tensor> loss_fwd(const Tensor& hidden, const std::optional<Tensor>& delta, double eps, const Tensor& norm,
                             const Tensor& head, const Tensor& labels) {
    Call c(hidden.device());
    const int64_t B = hidden.size(0), T = hidden.size(1), H = hidden.size(2), rows = B * T, V = head.size(0);
    const Tensor head16 = cast_in(c, {head}, kBF16)[0];
    std::optional<Tensor> d;
    if (delta.has_value()) d = delta->view({rows, H});
    auto [total, x, rstd] = add_norm(hidden.view({rows, H}), d, norm, eps);
    // (every row: the last of a sequence is left out of the loss, not cut out of the tensor)
    const Tensor logits = layer_linear(x, head16);
    const Tensor lse = c.empty({rows}, kF32), each = c.empty({rows}, kF32), mean = c.empty({2}, kF32);
    check("hawk_cross_entropy_fwd", lib.hawk_cross_entropy_fwd(
        data(logits), data<const long long>(labels), data<float>(lse), data<float>(each), data<float>(mean), B, T, V, c.st));
    return {mean.select(0, 0).clone(), head16, total, x, rstd, logits, lse, mean};
}

// s: norm, head16, total, x, rstd, logits, lse, mean.  Returns d_hidden, d_delta, d_norm, d_head.
std::vector<Tensor> loss_bwd(const std::vector<Tensor>& saved, const Tensor& labels_, const Tensor& d_loss_,
                             at::IntArrayRef shape, bool want_delta) {
    Call c(saved[0].device());
    const std::vector<Tensor> s = dense16(saved);
    const Tensor labels = labels_.contiguous();
    const Tensor d_loss = d_loss_.scalar_type() == kF32 ? d_loss_ : d_loss_.to(kF32);
    const Tensor &logits = s[5];
    const Tensor d_logits = c.empty(logits.sizes(), kBF16);
    check("hawk_cross_entropy_bwd", lib.hawk_cross_entropy_bwd(
        data(logits), data<const long long>(labels), data<float>(s[6]), data<float>(s[7]), data<float>(d_loss),
        data(d_logits), shape[0], shape[1], s[1].size(0), c.st));
    const Tensor d_x = input_grad(d_logits, s[1]);
    const Tensor d_head = weight_grad(d_logits, s[3]);
    auto [d_hidden, d_delta, d_norm] = add_norm_bwd(d_x, s[2], s[4], s[0], std::nullopt, want_delta);
    return {d_hidden.view(shape), d_delta.has_value() ? d_delta->view(shape) : Tensor(), d_norm, d_head};
}

Tensor embedding_bwd(const Tensor& ids_, const Tensor& d_out_, int64_t V) {
    Call c(d_out_.device());
    const Tensor ids = ids_.contiguous();
    const Tensor d_out = dense16(d_out_.scalar_type() == kF32 ? d_out_ : d_out_.to(kF32));
    const int64_t D = d_out.size(-1);
    Tensor dweight = at::zeros({V, D}, at::TensorOptions().dtype(kF32).device(c.dev));
    check("hawk_embedding_bwd", lib.hawk_embedding_bwd(data<const long long>(ids), data<float>(d_out), data<float>(dweight),
                                                       ids.numel(), V, D, c.st));
    return dweight;
}

py::object optional_list(const std::vector<Tensor>& ts) {
    py::tuple out(ts.size());
    for (size_t k = 0; k < ts.size(); ++k) out[k] = ts[k].defined() ? py::cast(ts[k]) : py::none();
    return out;
}

// A launch function as a binding.
template <typename R, typename... A>
auto bound(R (*f)(A...)) {
    return [f](A... a) { return entry([&] { return f(a...); }); };
}

}  // namespace

PYBIND11_MODULE(_hawk_torch, m) {
    m.def("bind", [](const py::dict& addresses, const py::dict& callables, int64_t placed_from) {
#define X(name) lib.name = reinterpret_cast<decltype(lib.name)>(addresses[#name].cast<uintptr_t>());
        HAWK_FUNCTIONS(X)
#undef X
        python = new py::dict(callables);
        placed_from_bytes = placed_from;
    });
    m.def("functions", [] {
        std::vector<std::string> names;
#define X(name) names.push_back(#name);
        HAWK_FUNCTIONS(X)
#undef X
        return names;
    });
    m.def("forget", [](const std::string& which) {
        entry([&] {
            if (which == "scan_workspace") scan_workspaces().clear();
            if (which == "gate_workspace") gate_workspaces().clear();
            if (which == "decode_workspace") decode_workspaces().clear();
            return 0;
        });
    });
    m.def("scan_fwd", bound(scan_fwd));
    m.def("scan_bwd", bound(scan_bwd));
    m.def("gated_fwd", bound(gated_fwd));
    m.def("gated_bwd", bound(gated_bwd));
    m.def("conv_fwd", bound(conv_fwd));
    m.def("conv_bwd", bound(conv_bwd));
    m.def("core_fwd", bound(core_fwd));
    m.def("core_bwd", bound(core_bwd));
    m.def("gate_weights_to_bf16", bound(gate_weights_to_bf16));
    m.def("scan_node", scan_node);
    m.def("gated_node", gated_node);
    m.def("conv_node", conv_node);
    m.def("core_node", core_node);
    m.def("dense_parameter", dense_parameter);
    m.def("decode_core", decode_core);
    m.def("decode_first", bound(decode_first));
    m.def("decode_tail", bound(decode_tail));
    m.def("add_norm", bound(add_norm));
    m.def("add_norm_bwd", bound(add_norm_bwd));
    m.def("weight_grad", bound(weight_grad));
    m.def("layer_fwd", bound(layer_fwd));
    m.def("layer_bwd", [](const std::vector<Tensor>& s, const Tensor& d_total, const Tensor& d_out, bool want_delta) {
        return optional_list(entry([&] { return layer_bwd(s, d_total, d_out, want_delta); }));
    });
    m.def("loss_fwd", bound(loss_fwd));
    m.def("loss_bwd", [](const std::vector<Tensor>& s, const Tensor& labels, const Tensor& d_loss,
                         const std::vector<int64_t>& shape, bool want_delta) {
        return optional_list(entry([&] { return loss_bwd(s, labels, d_loss, shape, want_delta); }));
    });
    m.def("embedding_bwd", bound(embedding_bwd));
}
