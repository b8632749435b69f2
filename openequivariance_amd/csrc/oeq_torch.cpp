// Autograd kernels of the torch operators, in C++: an operator whose first k = 3 or 4 tensor arguments are differentiable
// (the rest are index tensors) and whose derivative is another operator of the dispatcher.
//
//   op(t_1 .. t_k, index ..) -> outputs          next(t_1 .. t_k, dout_1 .. dout_m, index ..) -> [dt_1 .. dt_k]
//
// What they do per call is what an autograd.Function in Python does, without entering the interpreter for it: the same
// small step costs tens of microseconds there, as much as the kernels of a molecular-dynamics step.  The kernels
// themselves are launched by the operators' GPU implementations below this dispatch level.
#include <ATen/core/dispatch/Dispatcher.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/library.h>

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

}  // namespace

TORCH_LIBRARY_FRAGMENT(openequivariance_amd, m) {
    m.def("register_derivative(str ns, str name, str next, int differentiable) -> ()", register_derivative);
}
