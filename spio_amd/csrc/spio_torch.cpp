// Native call path of the package's operators (host C++, no device code): what a call of
// spio::conv2d_gw8 or spio::layernorm_2d does between the Python call and the kernel launch.
//
// The Python definitions (spio_amd/functional) register the operators with torch and carry every
// rule of them: argument checks, fake tensors, autocast, autograd, tracing.  They cost 20 us per
// inference call and 220 us per training step, several times what the kernels take at ordinary
// sizes.  The functions here run the plain case (dense GPU tensors, eager mode, no tracing or
// dispatch mode in the way) without touching Python: look up the launch plan of the shape, allocate
// the result, launch, record one autograd node.  Anything else returns NotImplemented and the
// Python definition runs, so its checks and errors are the operator's.
//
// A launch plan is made once per shape by the Python side (tuner, compiler, kernel caches) and
// holds what a launch needs.  spio_amd/native.py drops the plans whenever the kernels behind them
// may change and switches this path off while an overlay, a logger or a timer wants to see every
// launch.
#include <torch/extension.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>

#include <atomic>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <shared_mutex>
#include <unordered_map>

#include "spio_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

constexpr auto CL = at::MemoryFormat::ChannelsLast;

// ---- launch plans ---------------------------------------------------------------------------

enum Kind : int64_t { FPROP = 0, DGRAD = 1, WGRAD = 2, BGRAD = 3, NORM = 4, NORM_BWD = 5 };

// What selects a plan: the kind, the device and the numbers of the problem.
struct Key {
    int64_t v[12];
    bool operator==(const Key& o) const { return std::memcmp(v, o.v, sizeof v) == 0; }
};
struct KeyHash {
    size_t operator()(const Key& k) const {
        uint64_t h = 0x9e3779b97f4a7c15ull;
        for (int64_t x : k.v) {
            h ^= static_cast<uint64_t>(x);
            h *= 0xff51afd7ed558ccdull;
            h ^= h >> 32;
        }
        return h;
    }
};

struct Stage {
    void* function = nullptr;
    unsigned grid[3] = {0, 0, 0}, block[3] = {0, 0, 0}, lds = 0;
};
struct Plan {
    Stage main, second;         // `second` of two-stage kernels
    Stage second_half;          // the second stage that stores grad_weight as float16
    int64_t workspace = 0;      // bytes of partial results between the stages
    bool present = false;       // false: the shape does not use this kind (no fused backward, no float32 output)
    bool overwrites = false;    // the kernel stores its sums whole instead of adding to them
    std::shared_ptr<PyObject> kernel;  // the Python kernel whose code object `main` and `second` point into
};
using PlanPtr = std::shared_ptr<const Plan>;

std::shared_mutex g_plans_mutex;
using Plans = std::unordered_map<Key, PlanPtr, KeyHash>;
Plans& g_plans = *new Plans;            // never destroyed: the plans hold Python objects
std::atomic<int64_t> g_bypass{1};      // > 0: every call takes the Python path
std::atomic<uint64_t> g_generation{0};  // of the plans: a plan made before a forget() is not kept
PyObject* g_make_plan = nullptr;        // Python: (key values) -> plan description

PlanPtr find_plan(const Key& key) {
    {
        std::shared_lock<std::shared_mutex> lock(g_plans_mutex);
        auto it = g_plans.find(key);
        if (it != g_plans.end()) return it->second;
    }
    const uint64_t generation = g_generation.load();
    auto plan = std::make_shared<Plan>();
    {
        // tunes and compiles on a shape's first use; its errors travel to the caller
        py::gil_scoped_acquire gil;
        py::tuple values(12);
        for (int i = 0; i < 12; ++i) values[i] = py::int_(key.v[i]);
        py::object made = py::reinterpret_borrow<py::object>(g_make_plan)(values);
        if (!made.is_none()) {
            auto t = made.cast<py::tuple>();  // (stages, workspace bytes, overwrites, kernel)
            auto stages = t[0].cast<py::list>();
            for (size_t i = 0; i < stages.size(); ++i) {
                auto s = stages[i].cast<std::vector<uint64_t>>();
                Stage& stage = i == 0 ? plan->main : i == 1 ? plan->second : plan->second_half;
                stage.function = reinterpret_cast<void*>(s[0]);
                for (int d = 0; d < 3; ++d) {
                    stage.grid[d] = static_cast<unsigned>(s[1 + d]);
                    stage.block[d] = static_cast<unsigned>(s[4 + d]);
                }
                stage.lds = static_cast<unsigned>(s[7]);
            }
            plan->workspace = t[1].cast<int64_t>();
            plan->overwrites = t[2].cast<bool>();
            plan->present = true;
            // the last owner may be a thread without the GIL
            plan->kernel = {py::object(t[3]).release().ptr(), [](PyObject* kernel) {
                                py::gil_scoped_acquire gil;
                                Py_DECREF(kernel);
                            }};
        }
    }
    std::unique_lock<std::shared_mutex> lock(g_plans_mutex);
    if (g_bypass.load() == 0 && g_generation.load() == generation) g_plans.emplace(key, plan);
    return plan;
}

void launch(const Stage& stage, hipStream_t stream, std::initializer_list<const void*> args) {
    const void* values[8];
    void* params[8];
    int n = 0;
    for (const void* a : args) {
        values[n] = a;
        params[n] = &values[n];
        ++n;
    }
    const int rc = spio_hip_launch(stage.function, stage.grid[0], stage.grid[1], stage.grid[2], stage.block[0],
                                   stage.block[1], stage.block[2], stage.lds, stream, params, n);
    TORCH_CHECK_VALUE(rc == 0, "kernel launch failed: ", spio_hip_last_error());
}

const void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

Tensor empty_cl(at::IntArrayRef sizes, at::ScalarType dtype, const Tensor& like) {
    return at::detail::empty_cuda(sizes, dtype, like.device(), CL);
}
Tensor empty_1d(int64_t n, at::ScalarType dtype, const Tensor& like) {
    return at::detail::empty_cuda({n}, dtype, like.device(), std::nullopt);
}
// Clears one or two tensors (undefined: none) in one launch.
void zero(const Tensor& a, const Tensor& b, hipStream_t stream) {
    auto bytes = [](const Tensor& t) { return t.defined() ? static_cast<size_t>(t.nbytes()) : 0; };
    const int rc = spio_hip_zero_fill_pair_async(const_cast<void*>(ptr(a)), bytes(a), const_cast<void*>(ptr(b)), bytes(b), stream);
    TORCH_CHECK_VALUE(rc == 0, "zero fill failed: ", spio_hip_last_error());
}

// ---- which calls take this path -------------------------------------------------------------

// A dense GPU tensor with no wrapper, transform or lazy view on it.
bool is_plain(const Tensor& t) {
    static const c10::DispatchKeySet dense =
        c10::DispatchKeySet(c10::DispatchKey::CUDA) | c10::DispatchKeySet(c10::DispatchKey::AutogradCUDA) |
        c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView) | c10::DispatchKeySet(c10::DispatchKey::AutocastCUDA);
    return t.defined() && t.is_cuda() && dense.has_all(t.key_set()) && !t._fw_grad(0).defined();
}

// Eager mode: no tracing, functionalisation, transform or Python mode above the operator.
bool eager_mode() {
    static const c10::DispatchKeySet usual = c10::DispatchKeySet(c10::DispatchKey::BackendSelect) |
                                             c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView);
    return usual.has_all(c10::impl::tls_local_dispatch_key_set().included_) &&
           !at::impl::torch_function_mode_enabled();
}

// Whether a backward pass goes to the Python operators: somebody has come to see every launch, or to trace or
// transform the call, since the forward pass, or its gradients are to be differentiated (create_graph=True).
bool stands_aside(const Tensor& grad) {
    return g_bypass.load(std::memory_order_relaxed) != 0 || !eager_mode() || !is_plain(grad) || at::GradMode::is_enabled();
}

// What a profiler that records shapes is told of a call; evaluated only if one is active.
std::vector<c10::IValue> tensors(std::initializer_list<Tensor> args) {
    std::vector<c10::IValue> values;
    for (const Tensor& t : args) values.emplace_back(t);
    return values;
}

bool wants_grad(const Tensor& t) { return t.defined() && t.requires_grad(); }

std::optional<Tensor> optional(const Tensor& t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; }

struct Conv {  // the numbers of one convolution
    int64_t n, c, h, w, r, s, py, px;
    bool bias;
    int64_t p() const { return h + 2 * py - r + 1; }
    int64_t q() const { return w + 2 * px - s + 1; }
    Key key(Kind kind, int64_t device, int64_t mode = 0) const {
        return {{kind, device, n, c, h, w, r, s, py, px, bias, mode}};
    }
};

// SPIO_FUSED_BACKWARD as the Python operator reads it: 0 never, 1 whenever possible, 2 by time.
int64_t fused_mode() {
    const char* v = std::getenv("SPIO_FUSED_BACKWARD");
    if (!v) return 2;
    std::string s(v);
    const auto from = s.find_first_not_of(" \t\n");
    s = from == std::string::npos ? "" : s.substr(from, s.find_last_not_of(" \t\n") - from + 1);
    for (char& ch : s) ch = static_cast<char>(std::tolower(static_cast<unsigned char>(ch)));
    if (s == "0" || s == "false" || s == "off" || s == "no") return 0;
    if (s == "1" || s == "true" || s == "on" || s == "yes") return 1;
    return 2;
}

// ---- convolution ----------------------------------------------------------------------------

// Bits of a key's mode.  WIDE: the kernel stores its activations as float32.  HALF_WEIGHT: the caller's weights,
// and so their gradient, are float16.  READ_F32, WEIGHT_F32: it reads a float32 source (x forward, grad_output
// backward), float32 weights.  KEEP: it stores what it rounded of these as float16.
constexpr int64_t WIDE = 4, HALF_WEIGHT = 8, READ_F32 = 16, WEIGHT_F32 = 32, KEEP = 64;

// What the kernels read: float16, channels_last; the tensor itself where it is that already.
Tensor to_half_cl(const Tensor& t) {
    if (t.scalar_type() == at::kHalf) return t.is_contiguous(CL) ? t : t.contiguous(CL);
    return t.to(at::kHalf, /*non_blocking=*/false, /*copy=*/false, CL).contiguous(CL);
}
// A float32 tensor that a kernel can read as it is, in the order and with the alignment of its 16-byte loads.
bool readable_f32(const Tensor& t) {
    return t.scalar_type() == at::kFloat && t.is_contiguous(CL) && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

struct ConvOutput {
    Tensor y, x, w;  // x, w: the float16 tensors that the products were taken of (wanted: `keep`)
};

// The result is in the type of `x` where the kernel has such a version, else float16, for the caller to convert.
ConvOutput conv_forward(const Conv& cv, const Tensor& x, const Tensor& w, const Tensor& bias, bool keep) {
    const auto device = x.get_device();
    hipStream_t stream = c10::hip::getCurrentHIPStream(device);
    const int64_t wide = x.scalar_type() == at::kFloat ? WIDE : 0;
    const int64_t reads = (readable_f32(x) ? READ_F32 : 0) | (readable_f32(w) ? WEIGHT_F32 : 0);
    if (reads) {
        const auto plan = find_plan(cv.key(FPROP, device, wide | reads | (keep ? KEEP : 0)));
        if (plan->present) {
            ConvOutput o;
            o.y = empty_cl({cv.n, cv.c, cv.p(), cv.q()}, wide ? at::kFloat : at::kHalf, x);
            const Tensor xr = reads & READ_F32 ? x : to_half_cl(x), wr = reads & WEIGHT_F32 ? w : to_half_cl(w);
            if (keep) {
                o.x = reads & READ_F32 ? empty_cl(x.sizes(), at::kHalf, x) : xr;
                o.w = reads & WEIGHT_F32 ? empty_cl(w.sizes(), at::kHalf, w) : wr;
                launch(plan->main, stream, {ptr(o.y), ptr(xr), ptr(wr), ptr(bias), ptr(o.x), ptr(o.w)});
            } else {
                launch(plan->main, stream, {ptr(o.y), ptr(xr), ptr(wr), ptr(bias)});
            }
            return o;
        }
    }
    ConvOutput o{Tensor(), to_half_cl(x), to_half_cl(w)};
    PlanPtr plan;
    if (wide) plan = find_plan(cv.key(FPROP, device, WIDE));
    const bool store_wide = plan && plan->present;
    if (!store_wide) plan = find_plan(cv.key(FPROP, device));
    o.y = empty_cl({cv.n, cv.c, cv.p(), cv.q()}, store_wide ? at::kFloat : at::kHalf, x);
    launch(plan->main, stream, {ptr(o.y), ptr(o.x), ptr(o.w), ptr(bias)});
    return o;
}

struct ConvGrads {
    Tensor x, w, b;
};

// The backward operator, x and w on channels_last tensors: one fused kernel where the shape uses it and
// both gradients are wanted, else the weight and the data gradient one after the other.
// `x_dtype`, `w_dtype`: what the caller's tensors are; a gradient is stored in that type where the kernel
// can (a two-stage one's grad_weight), else in the operator's and the caller converts it.
ConvGrads conv_backward(const Conv& cv, const Tensor& x, const Tensor& w, const Tensor& grad, bool need_x,
                        bool need_w, bool need_b, at::ScalarType x_dtype, at::ScalarType w_dtype) {
    ConvGrads g;
    const auto device = grad.get_device();
    hipStream_t stream = c10::hip::getCurrentHIPStream(device);
    const int64_t weight_mode = w_dtype == at::kHalf ? HALF_WEIGHT : 0;
    const bool read_f32 = readable_f32(grad);
    // grad as float16, made when a kernel that wants it comes first
    Tensor half_grad;
    auto dy = [&]() -> const Tensor& {
        if (!half_grad.defined()) half_grad = to_half_cl(grad);
        return half_grad;
    };
    // The version of a kernel for the caller's types: one whose grad_input is float32, one that reads a float32
    // grad_output (and leaves a float16 copy), where these are wanted and there is one.
    int64_t types = 0;
    auto version = [&](const PlanPtr& plan, Kind kind, int64_t mode, int64_t keep) {
        const int64_t wide = x_dtype == at::kFloat ? WIDE : 0;
        for (const int64_t t : {wide | (read_f32 ? READ_F32 | keep : 0), wide}) {
            if (t == 0) continue;
            const auto v = find_plan(cv.key(kind, device, mode | t));
            if (!v->present) continue;
            types = t;
            return v;
        }
        return plan;
    };
    auto make_grad_input = [&] { g.x = empty_cl({cv.n, cv.c, cv.h, cv.w}, types & WIDE ? at::kFloat : at::kHalf, grad); };
    // atomic kernels add into zeroed sums, two-stage ones store them whole
    auto sums = [&](const Plan& plan, bool with_bias, bool bias_is_stored) {
        g.w = empty_cl({cv.c, 8, cv.r, cv.s}, weight_mode && plan.second_half.function ? at::kHalf : at::kFloat, grad);
        if (with_bias) g.b = empty_1d(cv.c, at::kFloat, grad);
        // one launch for both: a launch is all that the fill of such small sums costs
        zero(plan.overwrites ? Tensor() : g.w, bias_is_stored ? Tensor() : g.b, stream);
    };
    auto second = [&](const Plan& plan) -> const Stage& {
        return g.w.scalar_type() == at::kHalf ? plan.second_half : plan.second;
    };
    auto data_gradient = [&](int64_t keep) {
        const auto plan = version(find_plan(cv.key(DGRAD, device)), DGRAD, 0, keep);
        make_grad_input();
        if (types & KEEP) half_grad = empty_cl(grad.sizes(), at::kHalf, grad);
        if (types & KEEP)
            launch(plan->main, stream, {ptr(g.x), ptr(grad), ptr(w), nullptr, ptr(half_grad), nullptr});
        else
            launch(plan->main, stream, {ptr(g.x), types & READ_F32 ? ptr(grad) : ptr(dy()), ptr(w), nullptr});
    };
    PlanPtr fused;
    if (need_x && need_w) {
        const int64_t mode = fused_mode();
        if (mode != 0) fused = find_plan(cv.key(BGRAD, device, mode | weight_mode));
        if (fused && !fused->present) fused.reset();
        if (fused) fused = version(fused, BGRAD, mode | weight_mode, 0);
    }
    if (fused) {
        make_grad_input();
        sums(*fused, cv.bias && need_b, fused->overwrites);
        Tensor workspace;
        if (fused->second.function) workspace = empty_1d(fused->workspace, at::kByte, grad);
        const void* dw = workspace.defined() ? ptr(workspace) : ptr(g.w);
        const void* dy_ptr = types & READ_F32 ? ptr(grad) : ptr(dy());
        if (cv.bias)
            launch(fused->main, stream, {ptr(g.x), dw, ptr(x), dy_ptr, ptr(w), ptr(g.b)});
        else
            launch(fused->main, stream, {ptr(g.x), dw, ptr(x), dy_ptr, ptr(w)});
        if (workspace.defined()) launch(second(*fused), stream, {ptr(g.w), ptr(workspace), ptr(g.b)});
    } else if (need_w) {
        // a data gradient that reads float32 goes first: it leaves the copy that the weight gradient reads
        if (need_x && read_f32) data_gradient(KEEP);
        const auto plan = find_plan(cv.key(WGRAD, device, weight_mode));
        // the second stage that stores float16 stores the bias sums as well; the other adds them with atomics
        const bool half = weight_mode && plan->second_half.function;
        sums(*plan, cv.bias && need_b, half);
        Tensor workspace;
        if (plan->second.function) workspace = empty_1d(plan->workspace, at::kByte, grad);
        const void* dw = workspace.defined() ? ptr(workspace) : ptr(g.w);
        if (cv.bias)
            launch(plan->main, stream, {dw, ptr(x), ptr(dy()), half ? nullptr : ptr(g.b)});
        else
            launch(plan->main, stream, {dw, ptr(x), ptr(dy())});
        if (half && cv.bias)
            launch(plan->second_half, stream, {ptr(g.w), ptr(workspace), ptr(g.b)});
        else if (workspace.defined())
            launch(second(*plan), stream, {ptr(g.w), ptr(workspace)});
    }
    if (need_b && !g.b.defined()) g.b = dy().sum({0, 2, 3}, /*keepdim=*/false, at::kFloat);
    if (need_x && !g.x.defined()) data_gradient(0);
    return g;
}

// Whether a saved tensor still is what the forward pass saved, up to its layout: hooks on saved tensors may
// unpack it with other strides (a copy packed into host memory, say) or elsewhere altogether.
bool is_again(const Tensor& t, const Tensor& grad, at::IntArrayRef sizes, at::ScalarType dtype = at::kHalf) {
    return is_plain(t) && t.sizes() == sizes && t.device() == grad.device() && t.scalar_type() == dtype;
}
// A float32 vector of channels.
Tensor to_float_1d(const Tensor& t) {
    if (!t.defined() || (t.scalar_type() == at::kFloat && t.is_contiguous())) return t;
    return t.to(at::kFloat).contiguous();
}

PyObject* g_backward_op = nullptr;  // the Python operator: gradients that are differentiated again

// A saved copy (`cast`) of input number `input` of the node that is running, made to depend on that input
// again: the forward pass cast it with gradients off.  What is computed from it then leads back to the input,
// by way of a node that refuses to be run, so that a gradient of it is never taken for a constant.
Tensor with_history(const Tensor& copy, bool cast, size_t input) {
    const auto node = torch::autograd::get_current_node();
    if (!cast || !node || input >= node->num_outputs() || !node->next_edge(input).is_valid()) return copy;
    Tensor t = copy.variable_data();
    torch::autograd::set_history(t, std::make_shared<torch::autograd::Error>(
        "spio::conv2d_gw8: second derivatives have no autograd formula", torch::autograd::edge_list{node->next_edge(input)}));
    return t;
}

struct ConvFunction : torch::autograd::Function<ConvFunction> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w,
                          const std::optional<Tensor>& bias_arg, const Conv& cv) {
        const Tensor bias = bias_arg.value_or(Tensor());
        const Tensor bf = to_float_1d(bias);
        const auto [y, xh, wh] = conv_forward(cv, x, w, bf, /*keep=*/true);
        // the caller's own tensors unless their type was cast: with their history and their version, which
        // a second differentiation and a write to one of them before the backward pass are noticed by
        ctx->save_for_backward({x.scalar_type() == at::kHalf ? x : xh, w.scalar_type() == at::kHalf ? w : wh,
                                bias.defined() && bias.scalar_type() == at::kFloat ? bias : bf});
        ctx->saved_data["v"] = std::vector<int64_t>{
            cv.n, cv.c, cv.h, cv.w, cv.r, cv.s, cv.py, cv.px, cv.bias, static_cast<int64_t>(x.scalar_type()),
            static_cast<int64_t>(w.scalar_type()),
            bias.defined() ? static_cast<int64_t>(bias.scalar_type()) : static_cast<int64_t>(at::kFloat)};
        return y.to(x.scalar_type());
    }

    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const auto v = ctx->saved_data["v"].toIntVector();
        const Conv cv{v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8] != 0};
        const auto saved = ctx->get_saved_variables();
        const Tensor &x = saved[0], &w = saved[1];
        const bool native = !stands_aside(grads[0]) && is_again(x, grads[0], {cv.n, cv.c, cv.h, cv.w}) &&
                            is_again(w, grads[0], {cv.c, 8, cv.r, cv.s});
        const bool need_x = ctx->needs_input_grad(0), need_w = ctx->needs_input_grad(1),
                   need_b = cv.bias && ctx->needs_input_grad(2);
        ConvGrads g;
        if (!native) {  // the Python operator, which refuses second derivatives and tensors it does not take
            const Tensor xa = with_history(x, v[9] != static_cast<int64_t>(at::kHalf), 0),
                         wa = with_history(w, v[10] != static_cast<int64_t>(at::kHalf), 1),
                         ba = with_history(saved[2], v[11] != static_cast<int64_t>(at::kFloat), 2);
            py::gil_scoped_acquire gil;
            py::tuple r = py::reinterpret_borrow<py::object>(g_backward_op)(
                xa, wa, ba.defined() ? py::cast(ba) : py::none(), grads[0].to(at::kHalf), cv.py, cv.px, need_x, need_w, need_b);
            auto get = [&](int i) { return r[i].is_none() ? Tensor() : r[i].cast<Tensor>(); };
            g = {get(0), get(1), get(2)};
        } else {
            RECORD_FUNCTION("spio::conv2d_gw8_backward", tensors({x, w, saved[2], grads[0]}));
            g = conv_backward(cv, to_half_cl(x), to_half_cl(w), grads[0], need_x, need_w, need_b,
                              static_cast<at::ScalarType>(v[9]), static_cast<at::ScalarType>(v[10]));
        }
        auto typed = [&](const Tensor& t, int i) {
            return t.defined() ? t.to(static_cast<at::ScalarType>(v[i])) : t;
        };
        return {typed(g.x, 9), typed(g.w, 10), typed(g.b, 11), Tensor()};
    }
};

// ---- layer norm -----------------------------------------------------------------------------

struct Norm {
    int64_t n, c, h, w;
    double eps;
    Key key(Kind kind, int64_t device, bool weight, bool bias) const {
        int64_t bits;
        std::memcpy(&bits, &eps, sizeof bits);
        return {{kind, device, n, c, h, w, bits, weight, bias, 0, 0, 0}};
    }
};

Tensor norm_forward(const Norm& nm, const Tensor& x, const Tensor& weight, const Tensor& bias) {
    const auto plan = find_plan(nm.key(NORM, x.get_device(), weight.defined(), bias.defined()));
    Tensor y = empty_cl({nm.n, nm.c, nm.h, nm.w}, at::kHalf, x);
    launch(plan->main, c10::hip::getCurrentHIPStream(x.get_device()), {ptr(y), ptr(x), ptr(weight), ptr(bias)});
    return y;
}

constexpr int64_t NORM_BACKWARD_MAX_CHANNELS = 1024;  // of the backward kernel
PyObject* g_norm_gradients = nullptr;  // Python: the gradients, by kernel or torch operations

struct NormFunction : torch::autograd::Function<NormFunction> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const std::optional<Tensor>& weight_arg,
                          const std::optional<Tensor>& bias_arg, const Norm& nm) {
        const Tensor weight = weight_arg.value_or(Tensor()), bias = bias_arg.value_or(Tensor());
        const Tensor xc = to_half_cl(x);
        Tensor y = norm_forward(nm, xc, to_float_1d(weight), to_float_1d(bias));
        ctx->save_for_backward({x, weight});  // as in ConvFunction
        ctx->saved_data["v"] = std::vector<int64_t>{
            nm.n, nm.c, nm.h, nm.w, bias.defined(),
            weight.defined() ? static_cast<int64_t>(weight.scalar_type()) : static_cast<int64_t>(at::kFloat)};
        ctx->saved_data["eps"] = nm.eps;
        return y;
    }

    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const auto v = ctx->saved_data["v"].toIntVector();
        const Norm nm{v[0], v[1], v[2], v[3], ctx->saved_data["eps"].toDouble()};
        const auto saved = ctx->get_saved_variables();
        const Tensor &x = saved[0], &weight = saved[1];
        const bool native = !stands_aside(grads[0]) && !std::getenv("SPIO_LAYERNORM_BACKWARD") &&
                            is_again(x, grads[0], {nm.n, nm.c, nm.h, nm.w}) &&
                            (!weight.defined() || is_again(weight, grads[0], {nm.c}, static_cast<at::ScalarType>(v[5])));
        // absent tensors have no edge: the bias's follows the weight's or the input's
        const bool has_weight = weight.defined();
        const bool need_x = ctx->needs_input_grad(0), need_w = has_weight && ctx->needs_input_grad(1),
                   need_b = v[4] != 0 && ctx->needs_input_grad(has_weight ? 2 : 1);
        if (!native) {
            py::gil_scoped_acquire gil;
            py::tuple r = py::reinterpret_borrow<py::object>(g_norm_gradients)(
                x, has_weight ? py::cast(weight) : py::none(), grads[0], nm.eps, need_x, need_w, need_b);
            auto get = [&](int i) { return r[i].is_none() ? Tensor() : r[i].cast<Tensor>(); };
            return {get(0), get(1), get(2), Tensor()};
        }
        RECORD_FUNCTION("spio::layernorm_2d_backward", tensors({x, grads[0], weight}));
        const Tensor dy = to_half_cl(grads[0]), xc = to_half_cl(x);
        const Tensor w = to_float_1d(weight);
        const auto device = dy.get_device();
        hipStream_t stream = c10::hip::getCurrentHIPStream(device);
        const auto plan = find_plan(nm.key(NORM_BWD, device, w.defined(), false));
        const Tensor dx = empty_cl({nm.n, nm.c, nm.h, nm.w}, at::kHalf, dy);
        const Tensor sums = at::detail::empty_cuda({2, nm.c}, at::kFloat, dy.device(), std::nullopt);
        const Tensor workspace = empty_1d(plan->workspace, at::kByte, dy);
        launch(plan->main, stream, {ptr(workspace), ptr(dx), ptr(xc), ptr(dy), ptr(w)});
        launch(plan->second, stream, {ptr(sums), ptr(workspace)});
        return {need_x ? dx : Tensor(), need_w ? sums.select(0, 0).to(weight.scalar_type()) : Tensor(),
                need_b ? sums.select(0, 1) : Tensor(), Tensor()};
    }
};

// ---- Python boundary ------------------------------------------------------------------------

// Arguments of a Python call by position or keyword; false if they do not fit the names.
template <size_t N>
bool parse(PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames, PyObject* const (&names)[N], PyObject* (&out)[N]) {
    if (nargs > static_cast<Py_ssize_t>(N)) return false;
    for (Py_ssize_t i = 0; i < nargs; ++i) out[i] = args[i];
    const Py_ssize_t nkw = kwnames ? PyTuple_GET_SIZE(kwnames) : 0;
    for (Py_ssize_t k = 0; k < nkw; ++k) {
        PyObject* name = PyTuple_GET_ITEM(kwnames, k);
        size_t i = 0;
        while (i < N && name != names[i]) ++i;
        if (i == N) {
            i = 0;
            while (i < N && PyUnicode_Compare(name, names[i]) != 0) ++i;
        }
        if (i == N || out[i]) return false;
        out[i] = args[nargs + k];
    }
    return true;
}

bool tensor_arg(PyObject* o, Tensor* t) {
    if (!o || !THPVariable_CheckExact(o)) return false;
    *t = THPVariable_Unpack(o);
    return true;
}
bool int_arg(PyObject* o, int64_t* v) {
    if (!o) return true;
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    *v = PyLong_AsLongLongAndOverflow(o, &overflow);
    return overflow == 0;
}

PyObject* not_implemented() { Py_RETURN_NOTIMPLEMENTED; }

// Paddings above this are the Python operator's to refuse: twice one near 2^63 would wrap around to a small image.
constexpr int64_t MAX_PADDING = 1 << 24;

// conv2d_gw8(inputs, weight, bias=None, stride=1, padding_y=0, padding_x=0, dilation=1, groups=1)
PyObject* conv2d_gw8(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
    HANDLE_TH_ERRORS
    static PyObject* const names[8] = {
        PyUnicode_InternFromString("inputs"),    PyUnicode_InternFromString("weight"),
        PyUnicode_InternFromString("bias"),      PyUnicode_InternFromString("stride"),
        PyUnicode_InternFromString("padding_y"), PyUnicode_InternFromString("padding_x"),
        PyUnicode_InternFromString("dilation"),  PyUnicode_InternFromString("groups")};
    if (g_bypass.load(std::memory_order_relaxed) != 0 || !eager_mode()) return not_implemented();
    PyObject* a[8] = {};
    if (!parse(args, nargs, kwnames, names, a)) return not_implemented();
    Tensor x, w, bias;
    int64_t stride = 1, py = 0, px = 0, dilation = 1, groups = 1;
    if (!tensor_arg(a[0], &x) || !tensor_arg(a[1], &w) || (a[2] && a[2] != Py_None && !tensor_arg(a[2], &bias)) ||
        !int_arg(a[3], &stride) || !int_arg(a[4], &py) || !int_arg(a[5], &px) || !int_arg(a[6], &dilation) ||
        !int_arg(a[7], &groups))
        return not_implemented();
    if (!is_plain(x) || !is_plain(w) || x.dim() != 4 || w.dim() != 4 || w.device() != x.device())
        return not_implemented();
    if (bias.defined() && (!is_plain(bias) || bias.dim() != 1 || bias.device() != x.device() || bias.size(0) != w.size(0)))
        return not_implemented();
    const Conv cv{x.size(0), x.size(1), x.size(2), x.size(3), w.size(2), w.size(3), py, px, bias.defined()};
    if (stride != 1 || dilation != 1 || groups != cv.c / 8 || cv.c % 8 || w.size(0) != cv.c || w.size(1) != 8 || py < 0 ||
        px < 0 || py > MAX_PADDING || px > MAX_PADDING || cv.r < 1 || cv.r > 7 || cv.s < 1 || cv.s > 7 || cv.n < 1 ||
        cv.c < 8 || cv.h < 1 || cv.w < 1 || cv.p() < 1 || cv.q() < 1)
        return not_implemented();
    const bool autocast = at::autocast::is_autocast_enabled(at::kCUDA);
    auto floating = [](const Tensor& t) { return t.scalar_type() == at::kFloat || t.scalar_type() == at::kHalf; };
    if (autocast) {  // any of the two types is cast to what the kernels take; others are the Python operator's
        if (!floating(x) || !floating(w) || (bias.defined() && !floating(bias))) return not_implemented();
    } else if (x.scalar_type() != at::kHalf || w.scalar_type() != at::kHalf ||
               (bias.defined() && bias.scalar_type() != at::kFloat)) {
        return not_implemented();
    }
    Tensor y;
    {
        py::gil_scoped_release no_gil;
        c10::DeviceGuard device(x.device());
        RECORD_FUNCTION("spio::conv2d_gw8", tensors({x, w, bias}));
        // the casts and copies inside are the operator's own, whatever autocast thinks of them
        c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::autocast_dispatch_keyset);
        if (at::GradMode::is_enabled() && (wants_grad(x) || wants_grad(w) || wants_grad(bias))) {
            y = ConvFunction::apply(x, w, optional(bias), cv);
        } else {
            at::AutoDispatchBelowADInplaceOrView below;
            y = conv_forward(cv, x, w, to_float_1d(bias), /*keep=*/false).y.to(x.scalar_type());
        }
    }
    return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

// layernorm_2d(inputs, weight=None, bias=None, eps=1e-6)
PyObject* layernorm_2d(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
    HANDLE_TH_ERRORS
    static PyObject* const names[4] = {PyUnicode_InternFromString("inputs"), PyUnicode_InternFromString("weight"),
                                       PyUnicode_InternFromString("bias"), PyUnicode_InternFromString("eps")};
    if (g_bypass.load(std::memory_order_relaxed) != 0 || !eager_mode()) return not_implemented();
    PyObject* a[4] = {};
    if (!parse(args, nargs, kwnames, names, a)) return not_implemented();
    Tensor x, weight, bias;
    if (!tensor_arg(a[0], &x) || (a[1] && a[1] != Py_None && !tensor_arg(a[1], &weight)) ||
        (a[2] && a[2] != Py_None && !tensor_arg(a[2], &bias)) || (a[3] && !PyFloat_CheckExact(a[3])))
        return not_implemented();
    if (!is_plain(x) || x.dim() != 4 || x.scalar_type() != at::kHalf) return not_implemented();
    const Norm nm{x.size(0), x.size(1), x.size(2), x.size(3), a[3] ? PyFloat_AS_DOUBLE(a[3]) : 1e-6};
    for (const Tensor& t : {weight, bias})
        if (t.defined() && (!is_plain(t) || t.dim() != 1 || t.size(0) != nm.c || t.device() != x.device() ||
                            (t.scalar_type() != at::kFloat && t.scalar_type() != at::kHalf)))
            return not_implemented();
    if (nm.n < 1 || nm.h < 1 || nm.w < 1 || nm.c < 8 || nm.c % 8 || !(nm.eps > 0)) return not_implemented();
    const bool record = at::GradMode::is_enabled() && (wants_grad(x) || wants_grad(weight) || wants_grad(bias));
    // the backward pass by torch operations is the Python operator's
    if (record && nm.c > NORM_BACKWARD_MAX_CHANNELS) return not_implemented();
    Tensor y;
    {
        py::gil_scoped_release no_gil;
        c10::DeviceGuard device(x.device());
        RECORD_FUNCTION("spio::layernorm_2d", tensors({x, weight, bias}));
        if (record) {
            y = NormFunction::apply(x, optional(weight), optional(bias), nm);
        } else {
            at::AutoDispatchBelowADInplaceOrView below;
            y = norm_forward(nm, to_half_cl(x), to_float_1d(weight), to_float_1d(bias));
        }
    }
    return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

PyMethodDef g_methods[] = {
    {"layernorm_2d", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(layernorm_2d)),
     METH_FASTCALL | METH_KEYWORDS, "spio::layernorm_2d on plain GPU tensors, else NotImplemented"},
    {"conv2d_gw8", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(conv2d_gw8)),
     METH_FASTCALL | METH_KEYWORDS, "spio::conv2d_gw8 on plain GPU tensors, else NotImplemented"},
    {nullptr, nullptr, 0, nullptr}};

}  // namespace

// Found in the built file by spio_amd/build.py.
#define SPIO_TEXT_(x) #x
#define SPIO_TEXT(x) SPIO_TEXT_(x)

PYBIND11_MODULE(_native, m) {
    m.attr("built_from") = "spio-built-from:" SPIO_TEXT(SPIO_BUILT_FROM);
    m.attr("WIDE") = WIDE;
    m.attr("HALF_WEIGHT") = HALF_WEIGHT;
    m.attr("READ_F32") = READ_F32;
    m.attr("WEIGHT_F32") = WEIGHT_F32;
    m.attr("KEEP") = KEEP;
    m.def("configure", [](py::object make_plan, py::object backward_op, py::object norm_gradients) {
        g_make_plan = make_plan.release().ptr();
        g_backward_op = backward_op.release().ptr();
        g_norm_gradients = norm_gradients.release().ptr();
    });
    m.def("bypass", [](int64_t change) { g_bypass.fetch_add(change); });
    m.def("forget", [] {
        g_generation.fetch_add(1);
        Plans dropped;  // destroyed behind the lock: a kernel that goes with its plan runs Python code
        std::unique_lock<std::shared_mutex> lock(g_plans_mutex);
        dropped.swap(g_plans);
    });
    m.def("plans", [] {
        std::shared_lock<std::shared_mutex> lock(g_plans_mutex);
        return g_plans.size();
    });
    PyModule_AddFunctions(m.ptr(), g_methods);
}
