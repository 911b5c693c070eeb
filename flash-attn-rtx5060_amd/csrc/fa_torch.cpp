// The part of the PyTorch binding that runs on every call: what __init__.py works out once per combination of shapes, strides,
// types and options (a filled parameter block and sizes, "a plan") is applied here to new tensors, and the differentiable
// operator is a C++ autograd function, so that neither direction of a training step runs Python once its plan is known.
//
// Host time only: under autograd the Python function was called back in the engine's own thread, behind a hand-over of the
// interpreter's lock, and took three times as long there as in the caller's.  One call and its gradients, B1 H4 S128 D64
// (25 us of kernels): 105 us through a Python autograd.Function, 78 here; a forward call alone 7.5, 6.2 (its kernel takes 6.8).
// All arithmetic stays in the library (its entry points come in as addresses); nothing here keeps a tensor, an address or an
// object's identity from one call for the next.
#include <torch/extension.h>

#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>

#include <cstring>
#include <mutex>
#include <string>
#include <unordered_map>

#include "fa_bwd.h"
#include "fa_fwd.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

typedef int (*ForwardFn)(const fa_fwd_params *, void *);
typedef int (*BackwardFn)(const fa_bwd_params *, void *, unsigned long long, void *);
ForwardFn g_forward = nullptr, g_forward_static = nullptr;
BackwardFn g_backward = nullptr;
// The binding's Python functions for a combination that has no plan here yet; they do every check, make the call and return
// its results and, where the call may be repeated from a plan, that plan.  (Never released: the interpreter may be gone first.)
PyObject *g_first_forward = nullptr, *g_first_backward = nullptr;

void *raw_stream(const Tensor &t) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream(); }
Tensor bytes_like(const Tensor &t, int64_t n) { return at::empty({n}, t.options().dtype(at::kByte)); }

// flash_attention_forward with its plan at hand, into a tensor for O that the caller has made (of q's class, where that is a subclass):
// the status, O and the logsumexp (or None).
typedef std::tuple<int, Tensor, c10::optional<Tensor>> Planned;
Planned forward_planned_into(Tensor out, const std::string &block, const Tensor &q, const Tensor &k, const Tensor &v, const c10::optional<Tensor> &slopes,
                             unsigned long long seed, bool want_lse, int64_t workspace_bytes, bool static_scratch)
{
    py::gil_scoped_release release;
    fa_fwd_params p;
    TORCH_CHECK(block.size() == sizeof(p), "not a forward plan");
    std::memcpy(&p, block.data(), sizeof(p));
    if (!out.defined()) out = at::empty_like(q);
    c10::optional<Tensor> lse;
    p.Q = q.data_ptr(); p.K = k.data_ptr(); p.V = v.data_ptr(); p.O = out.data_ptr();
    p.seed = seed;
    if (want_lse) {
        lse = at::empty({q.size(0), q.size(1), q.size(2)}, q.options().dtype(at::kFloat));
        p.L = lse->data_ptr<float>();
    }
    if (slopes) p.alibi_slopes_ptr = static_cast<float *>(slopes->data_ptr());
    Tensor workspace;                                   // stream-ordered: freed after the launch
    if (workspace_bytes > 0) {
        workspace = bytes_like(q, workspace_bytes);
        p.workspace = workspace.data_ptr();
    }
    const int status = (static_scratch ? g_forward_static : g_forward)(&p, raw_stream(q));
    return {status, out, lse};
}
Planned forward_planned(const std::string &block, const Tensor &q, const Tensor &k, const Tensor &v, const c10::optional<Tensor> &slopes, unsigned long long seed,
                        bool want_lse, int64_t workspace_bytes, bool static_scratch)
{
    return forward_planned_into(Tensor(), block, q, k, v, slopes, seed, want_lse, workspace_bytes, static_scratch);
}

// ---- the differentiable operator
struct Call : torch::CustomClassHolder {                // one call's options
    c10::optional<double> scale;
    bool causal = false;
    int window_left = -1, window_right = -1;
    c10::optional<Tensor> slopes;
    double dropout = 0.0;
    unsigned long long seed = 0;
};
struct ForwardPlan {
    fa_fwd_params block;
};
struct BackwardPlan {
    fa_bwd_params block;
    int64_t total, parts_at;
    unsigned long long parts;
};
constexpr size_t kMostPlans = 1024;
std::mutex g_mutex;
std::unordered_map<std::string, ForwardPlan> g_forward_plans;
std::unordered_map<std::string, BackwardPlan> g_backward_plans;

// What a plan follows from: shape, strides, type and device of every tensor, and every option but the seed.
struct Key {
    std::string bytes;
    template <class T> void add(const T &x) { bytes.append(reinterpret_cast<const char *>(&x), sizeof(x)); }
    void add_tensor(const Tensor &t)
    {
        add((int)t.dim());
        add((int)t.scalar_type());
        add((int)t.device().type());
        add((int)t.device().index());
        for (int64_t n : t.sizes()) add(n);
        for (int64_t n : t.strides()) add(n);
    }
    explicit Key(const Call &c)
    {
        bytes.reserve(640);
        add((char)c.scale.has_value()); add(c.scale.value_or(0.0));
        add((char)c.causal); add(c.window_left); add(c.window_right); add(c.dropout);
        add((char)c.slopes.has_value());
        if (c.slopes) add_tensor(*c.slopes);
    }
};
template <class P> bool find_plan(const std::unordered_map<std::string, P> &plans, const Key &key, P *plan)
{
    std::lock_guard<std::mutex> lock(g_mutex);
    const auto it = plans.find(key.bytes);
    if (it == plans.end()) return false;
    *plan = it->second;
    return true;
}
template <class P> void keep_plan(std::unordered_map<std::string, P> &plans, const Key &key, const P &plan)
{
    std::lock_guard<std::mutex> lock(g_mutex);
    if (plans.size() >= kMostPlans) plans.clear();
    plans[key.bytes] = plan;
}
py::tuple options_of(const Call &c)
{
    return py::make_tuple(c.scale ? py::object(py::float_(*c.scale)) : py::object(py::none()), c.causal, c.window_left, c.window_right,
                          c.slopes ? py::cast(*c.slopes) : py::object(py::none()), c.dropout, c.seed);
}

struct Attention : torch::autograd::Function<Attention> {
    static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v, const c10::intrusive_ptr<Call> &call)
    {
        Key key(*call);
        key.add_tensor(q); key.add_tensor(k); key.add_tensor(v);
        Tensor out, lse;
        ForwardPlan plan;
        if (find_plan(g_forward_plans, key, &plan)) {
            fa_fwd_params &p = plan.block;
            out = at::empty_like(q);
            lse = at::empty({q.size(0), q.size(1), q.size(2)}, q.options().dtype(at::kFloat));
            p.Q = q.data_ptr(); p.K = k.data_ptr(); p.V = v.data_ptr(); p.O = out.data_ptr(); p.L = lse.data_ptr<float>();
            p.seed = call->seed;
            if (call->slopes) p.alibi_slopes_ptr = static_cast<float *>(call->slopes->data_ptr());
            if (g_forward(&p, raw_stream(q)) != FA_OK) out = Tensor();        // (the call below raises what this was)
        }
        if (!out.defined()) {
            py::gil_scoped_acquire gil;
            const py::tuple r = py::reinterpret_borrow<py::object>(g_first_forward)(q, k, v, options_of(*call)).cast<py::tuple>();
            out = r[0].cast<Tensor>();
            lse = r[1].cast<Tensor>();
            if (!r[2].is_none()) {
                const std::string block = r[2].cast<std::string>();
                TORCH_CHECK(block.size() == sizeof(plan.block), "not a forward plan");
                std::memcpy(&plan.block, block.data(), sizeof(plan.block));
                keep_plan(g_forward_plans, key, plan);
            }
        }
        ctx->save_for_backward({q, k, v, out, lse});
        ctx->saved_data["call"] = c10::IValue::make_capsule(call);
        return out;
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const variable_list saved = ctx->get_saved_variables();
        const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &o = saved[3], &lse = saved[4], &go = grads[0];
        const auto call = c10::static_intrusive_pointer_cast<Call>(ctx->saved_data["call"].toCapsule());
        Key key(*call);
        for (const Tensor &t : saved) key.add_tensor(t);
        key.add_tensor(go);
        BackwardPlan plan;
        if (find_plan(g_backward_plans, key, &plan)) {
            Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);      // (first: they need no less when memory is short)
            Tensor workspace;
            try {
                workspace = bytes_like(q, plan.total);          // stream-ordered: freed after the launch
            } catch (const c10::OutOfMemoryError &) {
                dq = dk = dv = Tensor();                        // (the smaller sizes are tried below)
            }
            if (workspace.defined()) {
                fa_bwd_params &p = plan.block;
                p.Q = q.data_ptr(); p.K = k.data_ptr(); p.V = v.data_ptr(); p.O = o.data_ptr(); p.dO = go.data_ptr(); p.L = lse.data_ptr<float>();
                p.dQ = dq.data_ptr(); p.dK = dk.data_ptr(); p.dV = dv.data_ptr();
                p.seed = call->seed;
                char *at_ = static_cast<char *>(workspace.data_ptr());
                p.workspace = at_;
                if (call->slopes) p.alibi_slopes_ptr = static_cast<float *>(call->slopes->data_ptr());
                if (g_backward(&p, plan.parts ? at_ + plan.parts_at : nullptr, plan.parts, raw_stream(q)) == FA_OK) return {dq, dk, dv, Tensor()};
            }
        }
        py::gil_scoped_acquire gil;
        const py::tuple r = py::reinterpret_borrow<py::object>(g_first_backward)(q, k, v, o, lse, go, options_of(*call)).cast<py::tuple>();
        if (!r[3].is_none()) {
            const py::tuple made = r[3].cast<py::tuple>();
            const std::string block = made[0].cast<std::string>();
            TORCH_CHECK(block.size() == sizeof(plan.block), "not a backward plan");
            std::memcpy(&plan.block, block.data(), sizeof(plan.block));
            plan.total = made[1].cast<int64_t>();
            plan.parts_at = made[2].cast<int64_t>();
            plan.parts = made[3].cast<unsigned long long>();
            keep_plan(g_backward_plans, key, plan);
        }
        return {r[0].cast<Tensor>(), r[1].cast<Tensor>(), r[2].cast<Tensor>(), Tensor()};
    }
};

Tensor attention(const Tensor &q, const Tensor &k, const Tensor &v, c10::optional<double> scale, bool causal, int window_left, int window_right,
                 c10::optional<Tensor> slopes, double dropout, unsigned long long seed)
{
    auto call = c10::make_intrusive<Call>();
    call->scale = scale;
    call->causal = causal;
    call->window_left = window_left;
    call->window_right = window_right;
    call->slopes = std::move(slopes);
    call->dropout = dropout;
    call->seed = seed;
    py::gil_scoped_release release;
    return Attention::apply(q, k, v, call);
}

void set_up(uint64_t forward, uint64_t forward_static, uint64_t backward, py::object first_forward, py::object first_backward)
{
    g_forward = reinterpret_cast<ForwardFn>(forward);
    g_forward_static = reinterpret_cast<ForwardFn>(forward_static);
    g_backward = reinterpret_cast<BackwardFn>(backward);
    g_first_forward = first_forward.release().ptr();
    g_first_backward = first_backward.release().ptr();
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    m.def("set_up", &set_up);
    m.def("forward_planned", &forward_planned);
    m.def("forward_planned_into", &forward_planned_into);
    m.def("attention", &attention);
}
