// Autograd kernels of the torch operators, in C++: an operator whose first k = 3 or 4 tensor arguments are differentiable
// (the rest are index tensors) and whose derivative is another operator of the dispatcher.
//
//   op(t_1 .. t_k, index ..) -> outputs          next(t_1 .. t_k, dout_1 .. dout_m, index ..) -> [dt_1 .. dt_k]
//
// What they do per call is what an autograd.Function in Python does, without entering the interpreter for it: the same
// small step costs tens of microseconds there, as much as the kernels of a molecular-dynamics step.
//
// Below them, the operators' GPU kernels (NativeKernel): the checks, output allocations and the call of the C library for
// ordinary tensors, without the interpreter either.  A pass back runs in a thread of torch's, where Python code first
// waits for the interpreter's lock and then runs with cold caches: a training step over 5183 edges, 64 channels, took 144 us
// with Python kernels (47 until the forward returned, 60 more until the backward's C call), 78 with these (17), a forward
// of 1000 rows 11 and 6.8; torch's own product of three tensors takes 80 in the same process.  Whatever they
// do not take - other layouts, alignments, devices, empty tensors, errors to be reported, a stream capture, the first call
// on a stream - goes to the operator's general implementation in Python, which also owns the workspaces lent to them.
#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/library.h>

#include "../../include/oeq_hip.h"

#include <algorithm>
#include <atomic>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

namespace {

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

struct Rule {
    c10::OperatorHandle op, next;
    size_t differentiable;
    bool list;                    // the operator returns Tensor[] (else one Tensor)
};

// Rules live as long as the process, as the operators they belong to do; a node of a graph names its rule by position.
std::mutex g_mutex;
std::vector<std::unique_ptr<Rule>>& rules() {
    static auto* r = new std::vector<std::unique_ptr<Rule>>();
    return *r;
}
std::vector<std::unique_ptr<torch::Library>>& libraries() {
    static auto* l = new std::vector<std::unique_ptr<torch::Library>>();
    return *l;
}
const Rule& rule(int64_t id) {
    std::lock_guard<std::mutex> lock(g_mutex);
    return *rules().at(static_cast<size_t>(id));
}

// What a node needs besides the differentiable tensors.
struct Call {
    int64_t id;
    c10::DispatchKeySet below;
    const variable_list& index;
};

// Where a node keeps argument i.  Each by itself, not as a list: torch's compiled autograd makes inputs of its graph only of
// tensors that are entries of saved_data themselves.
std::string slot(size_t i) { return "t" + std::to_string(i); }

variable_list run_forward(AutogradContext* ctx, const variable_list& tensors, const Call& call) {
    const Rule& r = rule(call.id);
    // (kept as data of the node, not as saved variables: the operators' arguments are not checked for changes in place)
    for (size_t i = 0; i < tensors.size(); ++i) ctx->saved_data[slot(i)] = tensors[i];
    for (size_t i = 0; i < call.index.size(); ++i) ctx->saved_data[slot(tensors.size() + i)] = call.index[i];
    ctx->saved_data["rule"] = call.id;
    torch::jit::Stack stack;
    stack.reserve(tensors.size() + call.index.size());
    for (const auto& t : tensors) stack.emplace_back(t);
    for (const auto& t : call.index) stack.emplace_back(t);
    at::AutoDispatchBelowAutograd guard;
    r.op.redispatchBoxed(call.below, &stack);
    return r.list ? stack.back().toTensorVector() : variable_list{stack.back().toTensor()};
}

variable_list run_backward(AutogradContext* ctx, const variable_list& grads) {
    const Rule& r = rule(ctx->saved_data["rule"].toInt());
    const size_t n = r.op.schema().arguments().size();
    torch::jit::Stack stack;
    stack.reserve(n + grads.size());
    for (size_t i = 0; i < r.differentiable; ++i) stack.push_back(ctx->saved_data.at(slot(i)));
    for (const auto& t : grads) stack.emplace_back(t);
    for (size_t i = r.differentiable; i < n; ++i) stack.push_back(ctx->saved_data.at(slot(i)));
    r.next.callBoxed(&stack);
    variable_list out = stack.back().toTensorVector();
    TORCH_CHECK(out.size() == r.differentiable, "a derivative returned ", out.size(), " gradients for ", r.differentiable, " tensors");
    out.emplace_back();                                     // nothing for the Call
    return out;
}

struct First : torch::autograd::Function<First> {           // of a product: x, y, w
    static variable_list forward(AutogradContext* ctx, const at::Tensor& a, const at::Tensor& b, const at::Tensor& c,
                                 const Call& call) {
        return run_forward(ctx, {a, b, c}, call);
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) { return run_backward(ctx, grads); }
};

struct Second : torch::autograd::Function<Second> {         // of its backward: x, y, w, dz
    static variable_list forward(AutogradContext* ctx, const at::Tensor& a, const at::Tensor& b, const at::Tensor& c,
                                 const at::Tensor& d, const Call& call) {
        return run_forward(ctx, {a, b, c, d}, call);
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) { return run_backward(ctx, grads); }
};

struct AutogradKernel final : c10::OperatorKernel {
    const int64_t id;
    explicit AutogradKernel(int64_t i) : id(i) {}

    void operator()(const c10::OperatorHandle& op, c10::DispatchKeySet keys, torch::jit::Stack* stack) {
        const Rule& r = rule(id);
        const size_t n = op.schema().arguments().size(), first = stack->size() - n;
        const auto below = keys & c10::after_autograd_keyset;
        bool graph = false;
        if (at::GradMode::is_enabled())
            for (size_t i = 0; i < n && !graph; ++i) graph = (*stack)[first + i].toTensor().requires_grad();
        if (!graph) {
            at::AutoDispatchBelowAutograd guard;
            op.redispatchBoxed(below, stack);
            return;
        }
        variable_list t, index;
        for (size_t i = 0; i < n; ++i) (i < r.differentiable ? t : index).push_back((*stack)[first + i].toTensor());
        torch::jit::drop(*stack, n);
        const Call call{id, below, index};
        variable_list out = r.differentiable == 3 ? First::apply(t[0], t[1], t[2], call) : Second::apply(t[0], t[1], t[2], t[3], call);
        if (r.list)
            stack->emplace_back(c10::List<at::Tensor>(out));
        else
            stack->emplace_back(out.at(0));
    }
};

// Gives the operator `ns::name` the derivative `ns::next`.
void register_derivative(const std::string& ns, const std::string& name, const std::string& next, int64_t differentiable) {
    auto& dispatcher = c10::Dispatcher::singleton();
    auto op = dispatcher.findSchemaOrThrow((ns + "::" + name).c_str(), "");
    auto nx = dispatcher.findSchemaOrThrow((ns + "::" + next).c_str(), "");
    TORCH_CHECK((differentiable == 3 || differentiable == 4) && static_cast<size_t>(differentiable) <= op.schema().arguments().size(),
                "three or four differentiable arguments are supported, got ", differentiable);
    const bool list = op.schema().returns().at(0).type()->kind() == c10::TypeKind::ListType;
    int64_t id;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        id = static_cast<int64_t>(rules().size());
        rules().push_back(std::unique_ptr<Rule>(new Rule{op, nx, static_cast<size_t>(differentiable), list}));
    }
    auto lib = std::make_unique<torch::Library>(torch::Library::IMPL, ns, std::make_optional(c10::DispatchKey::Autograd), __FILE__, __LINE__);
    lib->impl(name.c_str(), torch::CppFunction::makeFromBoxedFunctor(std::make_unique<AutogradKernel>(id)));
    std::lock_guard<std::mutex> lock(g_mutex);
    libraries().push_back(std::move(lib));
}

// ---------------------------------------------------------------------------------------------- GPU kernels
// Entry points of the C library, as the interpreter has loaded it (native_library).
struct Library {
    decltype(&oeq_tp_forward) tp_forward;
    decltype(&oeq_tp_backward) tp_backward;
    decltype(&oeq_tp_double_backward) tp_double;
    decltype(&oeq_conv_forward_on) conv_forward;
    decltype(&oeq_conv_backward_on) conv_backward;
    decltype(&oeq_conv_double_backward_on) conv_double;
    decltype(&oeq_last_error) last_error;
} g_lib;

// Bytes of a convolution's workspace, the numbers that codegen/uvu_det.py's workspace_bytes takes.
struct Bytes {
    int64_t fixed, node, edge, spill, flags, chunks, row, long_node, piece_min;
    static int64_t up(int64_t b) { return (b + 255) & ~int64_t(255); }
    int64_t operator()(int64_t e, int64_t n) const {
        int64_t b = fixed + node * n + edge * e;
        if (spill) b = up(b) + spill * e;
        b = up(b + (flags ? 8 + 4 * ((e + 255) / 256) : 0));
        if (!long_node || !e || !n) return b;
        const int64_t t = std::max(piece_min, long_node * ((e + n - 1) / n)), tiles = (e + t - 1) / t;
        return b + 256 + up(16 * chunks * tiles) + 2 * tiles * row;
    }
};
int64_t largest(const std::vector<Bytes>& all, int64_t e, int64_t n) {
    int64_t b = 0;
    for (const auto& f : all) b = std::max(b, f(e, n));
    return b;
}

// Scratch that an operator in Python lends for one stream, and a convolution's record of the counters in it.
struct Lease {
    int64_t device, stream, size;
    at::Tensor buffer;
    oeq_conv_counters* counters;
};

// A backward of the unsorted convolution: by float atomics into zeros, or over edges grouped by sender.
struct Variant {
    void* handle;
    bool overwrites;
    int64_t kind;
};

struct Native {
    at::ScalarType dtype, index;
    int64_t d1, d2, d3, wn, scratch;
    bool conv, shared, deterministic, overwrites;    // overwrites: the main set's backward writes every row of dX
    std::atomic<void*> main, few;                    // kernel sets: general, for few rows,
    void* twice;                                     // ... of the double backward
    std::atomic<int64_t> few_forward, few_backward;  // largest batches of the kernels for few rows
    std::vector<Bytes> first_order, second_order;

    std::mutex mutex;                                // of everything below, and of a convolution's launches
    std::vector<Lease> leases;
    std::map<std::pair<int64_t, int64_t>, Variant> variants;
    bool enabled = true, double_ready = false, tuned = false;      // tuned: the backward's variant is measured per size class

    Lease* lease(int64_t device, int64_t stream) {
        for (auto& l : leases)
            if (l.device == device && l.stream == stream) return &l;
        return nullptr;
    }
};
std::vector<std::unique_ptr<Native>>& natives() {
    static auto* n = new std::vector<std::unique_ptr<Native>>();
    return *n;
}
Native& native(int64_t id) {
    std::lock_guard<std::mutex> lock(g_mutex);
    return *natives().at(static_cast<size_t>(id));
}

bool capturing() {
    return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None;
}
int64_t bits(int64_t v) {
    int64_t b = 0;
    for (; v; v >>= 1) ++b;
    return b;
}
void done(int status) {
    if (status) throw std::runtime_error(g_lib.last_error());
}

enum Kind { TP_FORWARD, TP_BACKWARD, TP_DOUBLE, CONV_FORWARD, CONV_BACKWARD, CONV_DOUBLE };

struct NativeKernel final : c10::OperatorKernel {
    Native& n;
    const c10::OperatorHandle general;
    const Kind kind;
    NativeKernel(Native& n_, c10::OperatorHandle g, Kind k) : n(n_), general(g), kind(k) {}

    void operator()(const c10::OperatorHandle& op, c10::DispatchKeySet keys, torch::jit::Stack* stack) {
        const size_t count = op.schema().arguments().size();
        const at::Tensor* t[10];
        for (size_t i = 0; i < count; ++i) t[i] = &(*stack)[stack->size() - count + i].toTensor();
        std::vector<at::Tensor> out;
        if (!run(t, count, out)) {
            general.redispatchBoxed(keys, stack);
            return;
        }
        torch::jit::drop(*stack, count);
        if (kind == TP_FORWARD || kind == CONV_FORWARD)
            stack->emplace_back(std::move(out[0]));
        else
            stack->emplace_back(c10::List<at::Tensor>(std::move(out)));
    }

    // An ordinary operand: on the device of the call, contiguous, of this shape, 16-byte aligned.
    bool takes(const at::Tensor& t, c10::Device device, int64_t rows, int64_t width) const {
        return t.defined() && t.device() == device && t.scalar_type() == n.dtype && t.dim() == 2 && t.size(0) == rows
            && t.size(1) == width && t.is_contiguous() && reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0;
    }

    bool run(const at::Tensor* const* t, size_t count, std::vector<at::Tensor>& out) {
        const at::Tensor& x = *t[0];
        if (!x.defined() || !x.is_cuda() || x.dim() != 2) return false;
        const c10::Device device = x.device();
        if (device.index() != c10::hip::current_device() || capturing()) return false;
        const int64_t nodes = x.size(0);
        int64_t rows = nodes;
        size_t operands = kind == TP_FORWARD || kind == CONV_FORWARD ? 3 : kind == TP_BACKWARD || kind == CONV_BACKWARD ? 4 : 7;
        if (n.conv) {
            if (!t[operands]->defined() || t[operands]->dim() != 1) return false;
            rows = t[operands]->size(0);
            for (size_t i = operands; i < count; ++i) {
                const at::Tensor& q = *t[i];
                if (!q.defined() || q.device() != device || q.scalar_type() != n.index || q.dim() != 1 || q.size(0) != rows
                    || !q.is_contiguous())
                    return false;
            }
            if (nodes >= int64_t(1) << 31 || rows >= int64_t(1) << 32) return false;
        }
        if (!nodes || !rows) return false;
        for (size_t i = 0; i < operands; ++i) {
            const size_t which = i < 4 ? i : i - 4;                  // x, y, w, dz, and the cotangents of the first three
            if (which == 2 && n.shared) {
                const at::Tensor& w = *t[i];
                if (!w.defined() || w.device() != device || w.scalar_type() != n.dtype || w.dim() != 1 || w.size(0) != n.wn
                    || !w.is_contiguous() || reinterpret_cast<uintptr_t>(w.const_data_ptr()) % 16)
                    return false;
            } else if (!takes(*t[i], device, which == 1 || which == 2 ? rows : nodes,
                              which == 0 ? n.d1 : which == 1 ? n.d2 : which == 2 ? n.wn : n.d3))
                return false;
        }
        void* stream = c10::hip::getCurrentHIPStream(device.index()).stream();
        const int64_t at_stream = reinterpret_cast<int64_t>(stream);
        return n.conv ? convolution(t, operands, nodes, rows, device, stream, at_stream, out)
                      : product(t, rows, device, stream, at_stream, out);
    }

    static const void* in(const at::Tensor* t) { return t->const_data_ptr(); }
    static void* to(const at::Tensor& t) { return t.data_ptr(); }

    bool product(const at::Tensor* const* t, int64_t rows, c10::Device device, void* stream, int64_t at_stream,
                 std::vector<at::Tensor>& out) {
        void* scratch = nullptr;
        if (n.scratch && kind != TP_DOUBLE) {
            std::lock_guard<std::mutex> lock(n.mutex);
            Lease* l = n.lease(device.index(), at_stream);
            if (!l) return false;
            scratch = to(l->buffer);                     // (of fixed size, never replaced)
        }
        const at::Tensor &x = *t[0], &y = *t[1], &w = *t[2];
        if (kind == TP_FORWARD) {
            out.push_back(at::empty({rows, n.d3}, x.options()));
            auto* h = static_cast<oeq_tp*>(rows <= n.few_forward ? n.few.load() : n.main.load());
            done(g_lib.tp_forward(h, rows, in(&x), in(&y), to(out[0]), in(&w), scratch, stream));
        } else if (kind == TP_BACKWARD) {
            for (const at::Tensor* a : {&x, &y, &w}) out.push_back(at::empty_like(*a));
            auto* h = static_cast<oeq_tp*>(rows <= n.few_backward ? n.few.load() : n.main.load());
            done(g_lib.tp_backward(h, rows, in(&x), to(out[0]), in(&y), to(out[1]), in(&w), to(out[2]), in(t[3]), scratch, stream));
        } else {
            for (size_t i = 0; i < 4; ++i) out.push_back(at::empty_like(*t[i]));
            done(g_lib.tp_double(static_cast<oeq_tp*>(n.twice), rows, in(&x), in(&y), in(&w), in(t[3]), in(t[4]), in(t[5]), in(t[6]),
                                 to(out[0]), to(out[1]), to(out[2]), to(out[3]), stream));
        }
        return true;
    }

    bool convolution(const at::Tensor* const* t, size_t operands, int64_t nodes, int64_t edges, c10::Device device, void* stream,
                     int64_t at_stream, std::vector<at::Tensor>& out) {
        const at::Tensor &x = *t[0], &y = *t[1], &w = *t[2];
        const void *rows = in(t[operands]), *cols = in(t[operands + 1]), *perm = n.deterministic ? in(t[operands + 2]) : nullptr;
        std::lock_guard<std::mutex> lock(n.mutex);
        if (!n.enabled) return false;
        Lease* l = n.lease(device.index(), at_stream);
        const int64_t first = largest(n.first_order, edges, nodes);
        if (!l || l->counters->captured || l->size < (kind == CONV_DOUBLE ? std::max(first, largest(n.second_order, edges, nodes)) : first))
            return false;
        const at::Tensor buffer = l->buffer;             // (held until the launches name it)
        if (kind == CONV_FORWARD) {
            out.push_back(at::empty({nodes, n.d3}, x.options()));
            done(g_lib.conv_forward(static_cast<oeq_conv*>(n.main.load()), in(&x), in(&y), in(&w), to(out[0]), rows, cols, edges, nodes,
                                    to(buffer), perm, stream, 0, l->counters, 1));
        } else if (kind == CONV_BACKWARD) {
            Variant v{n.main, n.overwrites, 1};
            if (n.tuned) {
                const auto found = n.variants.find({bits(edges), bits(nodes)});
                if (found == n.variants.end()) return false;
                v = found->second;
            }
            out.push_back(v.overwrites ? at::empty_like(x) : at::zeros_like(x));
            out.push_back(at::empty_like(y));
            out.push_back(at::empty_like(w));
            done(g_lib.conv_backward(static_cast<oeq_conv*>(v.handle), in(&x), to(out[0]), in(&y), to(out[1]), in(&w), to(out[2]),
                                     in(t[3]), rows, cols, edges, nodes, to(buffer), perm, stream, 0, l->counters, v.kind));
        } else {
            if (!n.double_ready) return false;
            for (size_t i = 0; i < 4; ++i) out.push_back(at::empty_like(*t[i]));
            // (both groupings are built in the scratch of the first-order kernels: kind 0)
            done(g_lib.conv_double(static_cast<oeq_conv*>(n.twice), in(&x), in(&y), in(&w), in(t[3]), in(t[4]), in(t[5]), in(t[6]),
                                   to(out[0]), to(out[1]), to(out[2]), to(out[3]), rows, cols, edges, nodes, to(buffer), perm, stream, 0, l->counters, 0));
        }
        return true;
    }
};

// The second derivatives where the fused kernel gives them: all cotangents there, no graph of them asked for.
struct DerivativeKernel final : c10::OperatorKernel {
    Native& n;
    const c10::OperatorHandle fused, general;
    DerivativeKernel(Native& n_, c10::OperatorHandle f, c10::OperatorHandle g) : n(n_), fused(f), general(g) {}

    void operator()(const c10::OperatorHandle& op, c10::DispatchKeySet, torch::jit::Stack* stack) {
        const size_t count = op.schema().arguments().size();
        bool direct = !at::GradMode::is_enabled();
        for (size_t i = 0; i < count && direct; ++i) direct = (*stack)[stack->size() - count + i].toTensor().defined();
        if (direct && n.conv) {
            std::lock_guard<std::mutex> lock(n.mutex);
            direct = n.double_ready;
        }
        (direct ? fused : general).callBoxed(stack);
    }
};

c10::OperatorHandle find(const std::string& ns, const std::string& name) {
    return c10::Dispatcher::singleton().findSchemaOrThrow((ns + "::" + name).c_str(), "");
}
void keep(const std::string& ns, c10::DispatchKey key, const std::string& name, torch::CppFunction f) {
    auto lib = std::make_unique<torch::Library>(torch::Library::IMPL, ns, std::make_optional(key), __FILE__, __LINE__);
    lib->impl(name.c_str(), std::move(f));
    std::lock_guard<std::mutex> lock(g_mutex);
    libraries().push_back(std::move(lib));
}

void native_library(at::IntArrayRef address) {
    TORCH_CHECK(address.size() == 7, "seven entry points are wanted");
    void** out[] = {(void**)&g_lib.tp_forward, (void**)&g_lib.tp_backward, (void**)&g_lib.tp_double, (void**)&g_lib.conv_forward,
                    (void**)&g_lib.conv_backward, (void**)&g_lib.conv_double, (void**)&g_lib.last_error};
    for (size_t i = 0; i < 7; ++i) *out[i] = reinterpret_cast<void*>(address[i]);
}

// Numbers of an operator -> its id.  ``v``: fp64, index64, d1, d2, d3, wn, scratch bytes, conv, shared, deterministic, overwrites, handles
// (main, few, double), limits of the kernels for few rows; ``first`` / ``second``: nine numbers (Bytes) for each workspace rule.
int64_t native_operator(at::IntArrayRef v, at::IntArrayRef first, at::IntArrayRef second) {
    TORCH_CHECK(v.size() == 16 && first.size() % 9 == 0 && second.size() % 9 == 0, "bad argument");
    auto n = std::make_unique<Native>();
    n->dtype = v[0] ? at::kDouble : at::kFloat;
    n->index = v[1] ? at::kLong : at::kInt;
    n->d1 = v[2]; n->d2 = v[3]; n->d3 = v[4]; n->wn = v[5]; n->scratch = v[6];
    n->conv = v[7]; n->shared = v[8]; n->deterministic = v[9]; n->overwrites = v[10];
    n->main = reinterpret_cast<void*>(v[11]); n->few = reinterpret_cast<void*>(v[12]); n->twice = reinterpret_cast<void*>(v[13]);
    n->few_forward = n->few ? v[14] : 0;
    n->few_backward = n->few ? v[15] : 0;
    for (auto [from, into] : {std::make_pair(first, &n->first_order), std::make_pair(second, &n->second_order)})
        for (size_t i = 0; i < from.size(); i += 9)
            into->push_back({from[i], from[i + 1], from[i + 2], from[i + 3], from[i + 4], from[i + 5], from[i + 6], from[i + 7], from[i + 8]});
    std::lock_guard<std::mutex> lock(g_mutex);
    natives().push_back(std::move(n));
    return static_cast<int64_t>(natives().size()) - 1;
}

// Operator `name` runs natively, `general` what that leaves.
void native_kernel(const std::string& ns, const std::string& name, const std::string& general, int64_t id, int64_t kind) {
    auto g = find(ns, general);
    keep(ns, c10::DispatchKey::CUDA, name, torch::CppFunction::makeFromBoxedFunctor(std::make_unique<NativeKernel>(native(id), g, static_cast<Kind>(kind))));
}
void native_derivative(const std::string& ns, const std::string& name, const std::string& fused, const std::string& general, int64_t id) {
    auto f = find(ns, fused), g = find(ns, general);
    keep(ns, c10::DispatchKey::CompositeImplicitAutograd, name,
         torch::CppFunction::makeFromBoxedFunctor(std::make_unique<DerivativeKernel>(native(id), f, g)));
}

// Scratch for a stream, in place of what was lent for it before.  Nothing is known of the counters in it, whatever a call in
// what it replaces has left in the record until now.
void native_lease(int64_t id, const at::Tensor& buffer, int64_t device, int64_t stream, int64_t counters) {
    Native& n = native(id);
    std::lock_guard<std::mutex> lock(n.mutex);
    Lease l{device, stream, buffer.numel(), buffer, reinterpret_cast<oeq_conv_counters*>(counters)};
    if (l.counters) l.counters->forward[2] = l.counters->backward[2] = 0;
    if (Lease* old = n.lease(device, stream))
        *old = l;
    else
        n.leases.push_back(l);
}
// The backward variant of a size class; without a handle, no class has one any more.
void native_variant(int64_t id, int64_t edge_bits, int64_t node_bits, int64_t handle, bool overwrites, int64_t kind) {
    Native& n = native(id);
    std::lock_guard<std::mutex> lock(n.mutex);
    if (handle)
        n.variants[{edge_bits, node_bits}] = Variant{reinterpret_cast<void*>(handle), overwrites, kind};
    else
        n.variants.clear();
}
void native_bytes(int64_t id, at::IntArrayRef more) {
    TORCH_CHECK(more.size() == 9, "bad argument");
    Native& n = native(id);
    std::lock_guard<std::mutex> lock(n.mutex);
    n.first_order.push_back({more[0], more[1], more[2], more[3], more[4], more[5], more[6], more[7], more[8]});
}
void native_enable(int64_t id, bool enabled, bool double_ready, bool tuned) {
    Native& n = native(id);
    std::lock_guard<std::mutex> lock(n.mutex);
    n.enabled = enabled;
    n.double_ready = n.double_ready || double_ready;
    n.tuned = tuned;
}
void native_kernels(int64_t id, int64_t main, int64_t few, int64_t forward, int64_t backward) {
    Native& n = native(id);
    n.main = reinterpret_cast<void*>(main);
    n.few_forward = n.few_backward = 0;
    n.few = reinterpret_cast<void*>(few);
    if (few) {
        n.few_forward = forward;
        n.few_backward = backward;
    }
}
int64_t native_workspace_bytes(int64_t id, bool second, int64_t edges, int64_t nodes) {
    Native& n = native(id);
    std::lock_guard<std::mutex> lock(n.mutex);
    return largest(second ? n.second_order : n.first_order, edges, nodes);
}

}  // namespace

TORCH_LIBRARY_FRAGMENT(openequivariance_amd, m) {
    m.def("register_derivative(str ns, str name, str next, int differentiable) -> ()", register_derivative);
    m.def("native_library(int[] address) -> ()", native_library);
    m.def("native_operator(int[] v, int[] first, int[] second) -> int", native_operator);
    m.def("native_kernel(str ns, str name, str general, int id, int kind) -> ()", native_kernel);
    m.def("native_derivative(str ns, str name, str fused, str general, int id) -> ()", native_derivative);
    m.def("native_lease(int id, Tensor buffer, int device, int stream, int counters) -> ()", native_lease);
    m.def("native_variant(int id, int edge_bits, int node_bits, int handle, bool overwrites, int kind) -> ()", native_variant);
    m.def("native_bytes(int id, int[] more) -> ()", native_bytes);
    m.def("native_enable(int id, bool enabled, bool double_ready, bool tuned) -> ()", native_enable);
    m.def("native_kernels(int id, int main, int few, int forward, int backward) -> ()", native_kernels);
    m.def("native_workspace_bytes(int id, bool second, int edges, int nodes) -> int", native_workspace_bytes);
}
