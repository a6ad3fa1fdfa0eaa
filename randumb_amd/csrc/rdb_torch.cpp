// The eager path of ops.linear without Python in it: autograd functions over the C ABI of librandumb_hip.so, as the extension
// module randumb_amd._rdb_torch.
//
// Why it exists: a layer's forward and backward are three to eight kernel launches of 5 to 40 us.  Issued from Python (an
// autograd.Function, ctypes with a dozen arguments a call, a torch.empty per output, device and stream look-ups) they cost 60
// to 75 us of host time, more than the kernels of a headline layer take (8192 tokens x 768 -> 3072, k = 256: 76 us of kernels,
// 130 us of wall time) and twice what a single-token forward takes.  Nothing here computes: it sizes and allocates outputs
// and workspaces with torch's allocator and calls the library.  Under torch.compile ops.linear takes the registered operators.
#include <ATen/ATen.h>
#include <ATen/core/Reduction.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/autograd.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_cpp_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <atomic>
#include <initializer_list>
#include <optional>

#include "../../include/randumb_hip.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

PyObject *g_error_class = nullptr;   // randumb_amd._lib.RandumbHipError
PyObject *g_tick = nullptr;          // hip's look at the give-up counter: called with (device index, calls)

// ----------------------------------------------------------------------------------------------- errors, device, stream
// A Python exception of the package's class, from whatever thread (the backward pass runs on autograd's).
[[noreturn]] void fail(PyObject *cls, const std::string &msg)
{
    pybind11::gil_scoped_acquire gil;
    PyErr_SetString(cls, msg.c_str());
    python_error err;
    err.persist();
    throw std::move(err);
}
void check(int rc, const char *what)
{
    if (rc == 0) return;
    fail(g_error_class ? g_error_class : PyExc_RuntimeError,
         std::string(what) + ": " + (rc < 0 ? "argument error " : "HIP error ") + std::to_string(rc) + ": " + rdb_last_error_string());
}

// The library takes raw pointers and looks at none of them: everything a call reads has to lie on the device it runs on.  Called
// with all tensor arguments before the first launch.
void same_device(const char *who, const Tensor &at, std::initializer_list<const Tensor *> others)
{
    auto check_one = [&](const Tensor &t) {
        if (!t.is_cuda()) fail(PyExc_NotImplementedError, std::string("Unsupported CPU implementation of ") + who + " called.");
        if (t.device() != at.device())
            fail(PyExc_RuntimeError, std::string(who) + ": expected all tensors on " + at.device().str() + ", found one on " + t.device().str());
    };
    check_one(at);
    for (const Tensor *t : others)
        if (t && t->defined()) check_one(*t);
}
const Tensor *address(const OptTensor &t) { return t ? &*t : nullptr; }

// Whether a call on these tensors may go past the dispatcher: not under a mode that wants to see it (tracing, fake tensors, counters),
// and not on tensors that stand for something else than their memory (fake, batched, tracked by functorch) or carry a forward-mode
// tangent.  The entry points return None for the others, and their callers take the general path.
bool past_dispatcher(std::initializer_list<const Tensor *> tensors)
{
    static const c10::DispatchKeySet special({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::BatchedNestedTensor,
                                              c10::DispatchKey::Batched, c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize});
    if (c10::impl::TorchDispatchModeTLS::any_modes_set()) return false;
    for (const Tensor *t : tensors)
        if (t && t->defined() && (t->key_set().has_any(special) || t->layout() != at::kStrided || t->_fw_grad(0).defined())) return false;
    return true;
}
// What a backward pass gets back of a tensor that it saved.  Saved-tensor hooks put in between may return anything: it is used only
// if it lies on the gradient's device and is what was saved, as far as the kernels rely on it.
const Tensor &restored(const char *who, const Tensor &t, const Tensor &grad, at::IntArrayRef sizes)
{
    if (!t.defined()) fail(PyExc_RuntimeError, std::string(who) + ": a saved tensor is missing");
    same_device(who, grad, {&t});
    if (t.sizes() != sizes) fail(PyExc_RuntimeError, std::string(who) + ": a saved tensor came back with another shape");
    return t;
}
// ... of `numel` values (at least) that are read by address
const Tensor &restored_values(const char *who, const Tensor &t, const Tensor &grad, at::ScalarType type, int64_t numel)
{
    if (!t.defined()) fail(PyExc_RuntimeError, std::string(who) + ": a saved tensor is missing");
    same_device(who, grad, {&t});
    if (t.scalar_type() != type || !t.is_contiguous() || t.numel() < numel || numel < 0)
        fail(PyExc_RuntimeError, std::string(who) + ": a saved tensor came back as something else");
    return t;
}

void *stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

// Entry points that may run a kernel whose blocks wait for each other are counted; every 16 of them hip looks at the
// counter of waits that gave up (which raises if there are new ones).
void tick(const Tensor &t)
{
    constexpr unsigned every = 16;
    static std::atomic<unsigned> calls[64];
    const int dev = t.get_device();
    if ((calls[dev & 63].fetch_add(1, std::memory_order_relaxed) + 1) % every || !g_tick) return;
    pybind11::gil_scoped_acquire gil;
    PyObject *r = PyObject_CallFunction(g_tick, "iI", dev, every);
    if (!r) {
        python_error err;
        err.persist();
        throw std::move(err);
    }
    Py_DECREF(r);
}

// ----------------------------------------------------------------------------------------------- tensors as the library reads them
bool readable(at::ScalarType t) { return t == at::kFloat || t == at::kBFloat16; }
int code(at::ScalarType t) { return t == at::kBFloat16 ? RDB_BF16 : RDB_F32; }

Tensor native(const Tensor &t) { return (readable(t.scalar_type()) ? t : t.to(at::kFloat)).contiguous(); }

// 2-D activation with unit inner stride in a dtype the kernels compute in
Tensor act(const Tensor &t0)
{
    if (t0.dim() != 2) fail(PyExc_ValueError, "activations must be 2-D (tokens, features)");
    const Tensor t = readable(t0.scalar_type()) ? t0 : t0.to(at::kFloat);
    return t.stride(1) == 1 && t.stride(0) >= t.size(1) ? t : t.contiguous();
}

// ... whose rows lie no farther apart than one launch addresses (2^29 elements): slices of very wide matrices are copied.  For the
// calls that keep something for the backward pass; the others fall through to kernels that take any stride.
Tensor near_act(const Tensor &t0)
{
    const Tensor t = act(t0);
    return t.size(0) * t.stride(0) >= (1ll << 29) ? t.contiguous() : t;
}

// ... of the input as a backward pass gets it back, in the gradient's dtype, as the kernels that read both by address take it (hooks on saved tensors may
// keep it in another one)
Tensor near_input(const Tensor &x, const Tensor &dy) { return near_act(x.to(dy.scalar_type())); }

Tensor bytes(int64_t n, const Tensor &like) { return n > 0 ? at::empty({n}, like.options().dtype(at::kByte)) : Tensor(); }
void *ptr(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }

struct Layer {
    int64_t in_f, out_f, sO, sI;
    uint32_t seed;
};

rdb_linear_desc desc(int64_t tokens, const Layer &l, int64_t k, int64_t coef_rows, at::ScalarType a, at::ScalarType c)
{
    rdb_linear_desc d;
    d.tokens = tokens;
    d.in_f = l.in_f;
    d.out_f = l.out_f;
    d.k = k;
    d.coef_rows = coef_rows;
    d.sO = l.sO;
    d.sI = l.sI;
    d.seed = l.seed;
    d.act_dtype = code(a);
    d.coef_dtype = code(c);
    d.algo = RDB_ALGO_AUTO;
    return d;
}
rdb_linear_desc desc(const Tensor &rows, const Layer &l, const Tensor &c)
{
    return desc(rows.size(0), l, c.size(-1), c.dim() == 1 ? 0 : c.size(0), rows.scalar_type(), c.scalar_type());
}

// ----------------------------------------------------------------------------------------------- pseudorandom vectors and biases
// n values of a contiguous vector-coef tensor, b[o] = sum_m noise(PRIME*o + m) coef[m] (+ s noise1d(o)), in the coefficients' dtype
Tensor coef_values(const Tensor &coef, const OptTensor &scale_bias, int64_t n, int64_t seed)
{
    const Tensor c = native(coef), sb = scale_bias && scale_bias->defined() ? native(*scale_bias).to(c.scalar_type()) : Tensor();
    const c10::OptionalDeviceGuard guard(c.device());
    Tensor out = at::empty({n}, c.options().dtype(at::kFloat));
    check(rdb_materialize_fwd(out.data_ptr<float>(), c.data_ptr(), code(c.scalar_type()), 0, c.numel(), 0, 1, n, 0, 1, (uint32_t)seed, ptr(sb), stream_of(c)),
          "rdb_materialize_fwd");
    return out.to(coef.scalar_type());
}
// ... and the adjoint: fp32 gradients of coef (k values) and s from the gradient of the values
std::pair<Tensor, Tensor> coef_grads(const Tensor &grad, int64_t k, int64_t seed, bool want_coef, bool want_scale)
{
    const Tensor d = native(grad);
    const c10::OptionalDeviceGuard guard(d.device());
    const auto f32 = d.options().dtype(at::kFloat);
    Tensor dc, ds;
    if (want_coef) {
        const int64_t need = rdb_materialize_bwd_workspace_bytes(0, k, 0, d.numel());
        const Tensor ws = bytes(need, d);
        dc = at::empty({k}, f32);
        check(rdb_materialize_bwd(dc.data_ptr<float>(), d.data_ptr(), code(d.scalar_type()), 0, k, 0, d.numel(), (uint32_t)seed, ptr(ws), need, stream_of(d)),
              "rdb_materialize_bwd");
    }
    if (want_scale) {
        const int64_t need = rdb_scale_bias_bwd_workspace_bytes(d.numel());
        const Tensor ws = bytes(need, d);
        ds = at::empty({1}, f32);
        check(rdb_scale_bias_bwd(ds.data_ptr<float>(), d.data_ptr(), code(d.scalar_type()), d.numel(), (uint32_t)seed, ptr(ws), need, stream_of(d)),
              "rdb_scale_bias_bwd");
    }
    return {dc, ds};
}

// A layer's bias: a dense vector (seed < 0), or a pseudorandom one given by its coefficients (and, with a fused random bias, its scale)
struct Bias {
    OptTensor coef, scale;
    int64_t seed = -1;
    explicit operator bool() const { return coef.has_value(); }
    int tensors() const { return (coef ? 1 : 0) + (scale ? 1 : 0); }
    Tensor values(int64_t n, at::ScalarType dtype) const
    {
        if (!coef) return Tensor();
        return (seed < 0 ? *coef : coef_values(*coef, scale, n, seed)).to(dtype).contiguous();
    }
    // ... as the library's calls take it that form them into `values` on the side (see beside); the tensors are the caller's
    rdb_pseudo_bias ref(const Tensor &c, const Tensor &s, const Tensor &values) const
    {
        return {c.data_ptr<float>(), s.defined() ? s.data_ptr<float>() : nullptr, values.data_ptr<float>(), c.numel(), (uint32_t)seed};
    }
    // Whether the values may be formed by a launch that a layer with fp32 rows makes anyway; the bounds: the summation order of coef_values
    bool beside(int64_t n, at::ScalarType dtype) const
    {
        return coef && seed >= 0 && dtype == at::kFloat && coef->scalar_type() == at::kFloat && coef->numel() >= 8 && n > 0 && n <= (1 << 15) &&
               (!scale || !scale->defined() || (scale->scalar_type() == at::kFloat && scale->numel() >= 1));
    }
    // what its gradient needs of it: whether there is one, length, seed, dtypes
    std::vector<int64_t> meta() const
    {
        return {coef ? coef->numel() : -1, seed, coef ? (int64_t)coef->scalar_type() : 0, scale ? (int64_t)scale->scalar_type() : -1};
    }
};
// The gradients of a pseudorandom bias in fp32, as a call of the library takes them (none wanted: ref.k < 0), and in the bias's dtypes
struct BiasGrads {
    Tensor dc, ds;
    rdb_pseudo_bias_grad ref = {nullptr, nullptr, -1, 0};
    BiasGrads(AutogradContext *ctx, const Tensor &dy, const std::vector<int64_t> &m, int at)
    {
        if (m[0] < 0 || m[1] < 0) return;
        const bool want_c = ctx->needs_input_grad(at), want_s = m[3] >= 0 && ctx->needs_input_grad(at + 1);
        if (!want_c && !want_s) return;
        const auto f32 = dy.options().dtype(at::kFloat);
        if (want_c) dc = at::empty({m[0]}, f32);
        if (want_s) ds = at::empty({1}, f32);
        ref = {want_c ? dc.data_ptr<float>() : nullptr, want_s ? ds.data_ptr<float>() : nullptr, m[0], (uint32_t)m[1]};
    }
    std::pair<Tensor, Tensor> done(const std::vector<int64_t> &m) const
    {
        return {dc.defined() ? dc.to((at::ScalarType)m[2]) : Tensor(), ds.defined() ? ds.to((at::ScalarType)m[3]) : Tensor()};
    }
};
// (gradient of the bias or its coefficients, gradient of its scale) from the column sums of dy; `at` is the bias's index among the
// function's tensor inputs
std::pair<Tensor, Tensor> bias_grads(AutogradContext *ctx, const Tensor &dy0, const std::vector<int64_t> &m, int at)
{
    if (m[0] < 0) return {};
    const bool want_c = ctx->needs_input_grad(at), want_s = m[3] >= 0 && ctx->needs_input_grad(at + 1);
    if (!want_c && !want_s) return {};
    if (m[1] < 0) return {dy0.sum(0).to((at::ScalarType)m[2]), Tensor()};
    const Tensor dy = act(dy0);
    const c10::OptionalDeviceGuard guard(dy.device());
    const BiasGrads g(ctx, dy, m, at);
    const int64_t need = rdb_bias_bwd_workspace_bytes(dy.size(0), dy.size(1));
    const Tensor ws = bytes(need, dy);
    check(rdb_bias_bwd(g.ref.dcoef, g.ref.dscale, dy.data_ptr(), code(dy.scalar_type()), dy.stride(0), dy.size(0), dy.size(1), g.ref.k, g.ref.seed, ptr(ws), need,
                       stream_of(dy)),
          "rdb_bias_bwd");
    return g.done(m);
}

// ----------------------------------------------------------------------------------------------- the library's calls
Tensor linear_fwd(const Tensor &x0, const Tensor &coefs, const Layer &l, const OptTensor &scale_bias, const Bias &bias)
{
    const Tensor x = act(x0), c = native(coefs);
    const Tensor sb = scale_bias ? native(*scale_bias).to(c.scalar_type()) : Tensor();
    const c10::OptionalDeviceGuard guard(x.device());
    const Tensor b = bias.values(l.out_f, x.scalar_type());
    Tensor y = at::empty({x.size(0), l.out_f}, x.options());
    const rdb_linear_desc d = desc(x, l, c);
    const int64_t need = rdb_linear_workspace_bytes(RDB_OP_LINEAR_FWD, &d);
    const Tensor ws = bytes(need, x);
    check(rdb_linear_fwd(y.data_ptr(), y.stride(0), x.data_ptr(), x.stride(0), c.data_ptr(), ptr(sb), ptr(b), &d, ptr(ws), need, stream_of(x)),
          "rdb_linear_fwd");
    tick(x);
    return y;
}

Tensor linear_bwd_dx(const Tensor &dy0, const Tensor &coefs, const Layer &l, const Tensor &scale_bias)
{
    const Tensor dy = act(dy0), c = native(coefs);
    const Tensor sb = scale_bias.defined() ? native(scale_bias).to(c.scalar_type()) : Tensor();
    const c10::OptionalDeviceGuard guard(dy.device());
    Tensor dx = at::empty({dy.size(0), l.in_f}, dy.options());
    const rdb_linear_desc d = desc(dy, l, c);
    const int64_t need = rdb_linear_workspace_bytes(RDB_OP_LINEAR_BWD_DX, &d);
    const Tensor ws = bytes(need, dy);
    check(rdb_linear_bwd_dx(dx.data_ptr(), dx.stride(0), dy.data_ptr(), dy.stride(0), c.data_ptr(), ptr(sb), &d, ptr(ws), need, stream_of(dy)),
          "rdb_linear_bwd_dx");
    tick(dy);
    return dx;
}

// (dx, gradient of the random bias's scale) from one pass over the random-bias product; undefined where the library has no such kernel
std::pair<Tensor, Tensor> linear_bwd_dx_dscale(const Tensor &dy0, const Tensor &x0, const Tensor &coefs, const Layer &l, const Tensor &scale_bias)
{
    if (dy0.scalar_type() != at::kBFloat16 || coefs.scalar_type() != at::kBFloat16 || coefs.dim() != 2) return {};
    const Tensor dy = act(dy0), x = act(x0).to(dy.scalar_type()), c = native(coefs), sb = native(scale_bias).to(c.scalar_type());
    const c10::OptionalDeviceGuard guard(dy.device());
    const rdb_linear_desc d = desc(dy, l, c);
    const int64_t need = rdb_linear_workspace_bytes(RDB_OP_LINEAR_BWD_DX_DSCALE, &d);
    if (need <= 0) return {};
    Tensor dx = at::empty({dy.size(0), l.in_f}, dy.options()), ds = at::empty({1}, dy.options().dtype(at::kFloat));
    const Tensor ws = bytes(need, dy);
    const int rc = rdb_linear_bwd_dx_dscale(dx.data_ptr(), dx.stride(0), ds.data_ptr<float>(), dy.data_ptr(), dy.stride(0), x.data_ptr(), x.stride(0),
                                            c.data_ptr(), sb.data_ptr(), &d, ptr(ws), need, stream_of(dy));
    if (rc == RDB_E_UNSUPPORTED) return {};   // nothing was launched
    check(rc, "rdb_linear_bwd_dx_dscale");
    return {dx, ds};
}

std::pair<Tensor, Tensor> linear_bwd_dcoef(const Tensor &dy0, const Tensor &x0, const Tensor &coefs, const Layer &l, bool want_scale)
{
    const Tensor dy = act(dy0), x = act(x0).to(dy.scalar_type());
    const int64_t k = coefs.size(-1), rows = coefs.dim() == 1 ? 0 : coefs.size(0);
    const c10::OptionalDeviceGuard guard(dy.device());
    const auto f32 = dy.options().dtype(at::kFloat);
    Tensor dc = rows ? at::empty({rows, k}, f32) : at::empty({k}, f32), ds = want_scale ? at::empty({1}, f32) : Tensor();
    const rdb_linear_desc d = desc(dy.size(0), l, k, rows, dy.scalar_type(), at::kFloat);
    const int64_t need = rdb_linear_workspace_bytes(RDB_OP_LINEAR_BWD_DCOEF, &d);
    const Tensor ws = bytes(need, dy);
    check(rdb_linear_bwd_dcoef(dc.data_ptr<float>(), want_scale ? ds.data_ptr<float>() : nullptr, dy.data_ptr(), dy.stride(0), x.data_ptr(), x.stride(0),
                               &d, ptr(ws), need, stream_of(dy)),
          "rdb_linear_bwd_dcoef");
    return {dc, ds};
}

rdb_linear_desc rbias_desc(const Tensor &rows, const Layer &l) { return desc(rows.size(0), l, 8, l.out_f, at::kBFloat16, at::kBFloat16); }

// First derivatives that a function's backward pass computes under create_graph without a graph, having no second ones: they are there,
// and going through them again raises (a result without a graph would pass for one that depends on nothing).  dy: the incoming
// gradient; inputs: which of the function's tensor inputs the derivative depends on.  The raising node leads to what these come
// from, so that it is on the way to all of them, whichever of them a derivative is asked for.
Tensor once_differentiable(const char *who, const Tensor &grad, const Tensor &dy, std::initializer_list<int> inputs)
{
    if (!at::GradMode::is_enabled() || !grad.defined()) return grad;
    torch::autograd::edge_list edges;
    auto depends_on = [&](const torch::autograd::Edge &e) {
        if (e.is_valid()) edges.push_back(e);
    };
    if (dy.requires_grad()) depends_on(torch::autograd::impl::gradient_edge(dy));
    const auto node = torch::autograd::get_current_node();
    for (int i : inputs)
        if (node && i >= 0 && i < (int)node->num_outputs()) depends_on(node->next_edge(i));
    if (edges.empty()) return grad;   // a constant
    const Tensor out = grad.tensor_data();
    torch::autograd::set_history(out, std::make_shared<torch::autograd::Error>(std::string(who) + " has no second derivative", std::move(edges)));
    return out;
}
// bias_grads under create_graph: linear in dy, by differentiable operators
std::pair<Tensor, Tensor> bias_grads_with_graph(const Tensor &dy, const std::vector<int64_t> &m);
// What a matrix-coef layer's backward pass returns, under create_graph too: dx depends on dy, the coefficients and the scale; dC and the scale's
// gradient on dy and x.  x is input 0, the coefficients are 1, the scale is `scale` (negative: none).
void layer_gradients(const Tensor &dy, int scale, Tensor &dx, Tensor &dc, Tensor &ds, std::pair<Tensor, Tensor> &db, const std::vector<int64_t> &bias)
{
    if (!at::GradMode::is_enabled()) return;
    dx = once_differentiable("linear", dx, dy, {1, scale});
    dc = once_differentiable("linear", dc, dy, {0});
    ds = once_differentiable("linear", ds, dy, {0});
    if (dy.requires_grad() && (db.first.defined() || db.second.defined())) {
        const auto again = bias_grads_with_graph(dy, bias);
        if (db.first.defined()) db.first = again.first;
        if (db.second.defined()) db.second = again.second;
    }
}

// ----------------------------------------------------------------------------------------------- one-call form
// y = x.W^T (+ bias) with x saved; the three products of the layer as three calls, or, for the layers of which the library keeps
// z = x.N^T (rdb_linear_kept_bytes), that saved and one call each way.
class OneCallLinear : public Function<OneCallLinear> {
  public:
    static Tensor forward(AutogradContext *ctx, const Tensor &x0, const Tensor &coefs, const OptTensor &scale_bias, const OptTensor &bias,
                          const OptTensor &bias_scale, int64_t bias_seed, const Layer &l)
    {
        const Bias b{bias, bias_scale, bias_seed};
        ctx->saved_data["layer"] = std::vector<int64_t>{l.in_f, l.out_f, l.sO, l.sI, (int64_t)l.seed, scale_bias ? 1 : 0, coefs.size(0), coefs.size(-1)};
        ctx->saved_data["bias"] = b.meta();
        const Tensor x = act(x0);
        const bool same = x.scalar_type() == coefs.scalar_type() && readable(coefs.scalar_type()) && (!scale_bias || scale_bias->numel() == 1);
        const rdb_linear_desc d = desc(x, l, coefs);
        const int64_t keep = same && coefs.dim() == 2 && coefs.size(0) == l.out_f ? rdb_linear_kept_bytes(&d) : 0;
        if (!keep) {
            ctx->save_for_backward({x0, coefs, scale_bias.value_or(Tensor()), Tensor()});
            return linear_fwd(x0, coefs, l, scale_bias, b);
        }
        const c10::OptionalDeviceGuard guard(x.device());
        const Tensor c = coefs.contiguous(), sb = scale_bias ? scale_bias->to(c.scalar_type()) : Tensor();
        const Tensor xn = near_act(x);
        Tensor y = at::empty({x.size(0), l.out_f}, x.options()), kept = bytes(keep, x);
        const int64_t room = rdb_linear_workspace_bytes(RDB_OP_LINEAR_FWD_KEPT, &d);
        const Tensor ws = bytes(room, x);
        auto call = [&](const Tensor &values, const rdb_pseudo_bias *pseudo) {
            check(rdb_linear_fwd_kept_ws(y.data_ptr(), l.out_f, kept.data_ptr(), xn.data_ptr(), xn.stride(0), c.data_ptr(), ptr(sb), ptr(values), pseudo, &d, ptr(ws),
                                         room, stream_of(x)),
                  "rdb_linear_fwd_kept");
        };
        if (b.beside(l.out_f, x.scalar_type())) {
            const Tensor bc = b.coef->contiguous(), bs = b.scale && b.scale->defined() ? b.scale->contiguous() : Tensor(), bv = at::empty({l.out_f}, x.options());
            const rdb_pseudo_bias pb = b.ref(bc, bs, bv);
            call(Tensor(), &pb);
        } else {
            call(b.values(l.out_f, x.scalar_type()), nullptr);
        }
        ctx->save_for_backward({scale_bias ? x0 : Tensor(), coefs, scale_bias.value_or(Tensor()), kept});
        return y;
    }
    static variable_list backward(AutogradContext *ctx, const variable_list &grads)
    {
        Tensor dx, dc, ds;
        std::pair<Tensor, Tensor> db;
        gradients(ctx, grads, dx, dc, ds, db);
        layer_gradients(grads[0], ctx->saved_data["layer"].toIntVector()[5] ? 2 : -1, dx, dc, ds, db, ctx->saved_data["bias"].toIntVector());
        return {dx, dc, ds, db.first, db.second, Tensor(), Tensor()};
    }
    static void gradients(AutogradContext *ctx, const variable_list &grads, Tensor &dx, Tensor &dc, Tensor &dsb, std::pair<Tensor, Tensor> &db)
    {
        const auto saved = ctx->get_saved_variables();
        const Tensor &x = saved[0], &coefs = saved[1], &sb = saved[2], &kept = saved[3];
        const auto m = ctx->saved_data["layer"].toIntVector();
        const Layer l{m[0], m[1], m[2], m[3], (uint32_t)m[4]};
        const bool has_sb = m[5] != 0;
        constexpr const char *who = "linear (backward)";
        restored(who, coefs, grads[0], at::IntArrayRef(&m[6], coefs.dim() == 1 ? 1 : 2));
        if (x.defined()) restored(who, x, grads[0], {grads[0].size(0), l.in_f});
        if (has_sb) restored(who, sb, grads[0], sb.sizes());
        const at::AutoGradMode no_grad(false);
        const bool want_dx = ctx->needs_input_grad(0), want_dc = ctx->needs_input_grad(1);
        bool want_sb = has_sb && ctx->needs_input_grad(2);
        const Tensor dy = kept.defined() ? near_act(grads[0]) : grads[0].contiguous();
        if (kept.defined()) {
            if (want_dx || want_dc || want_sb) {
                const c10::OptionalDeviceGuard guard(dy.device());
                const Tensor c = coefs.contiguous(), xs = want_sb ? near_input(x, dy) : Tensor(), s = has_sb ? sb.to(c.scalar_type()) : Tensor();
                const rdb_linear_desc d = desc(dy, l, c);
                const int64_t kept_bytes = rdb_linear_kept_bytes(&d);   // 0: the coefficients came back in another dtype
                restored_values(who, kept, dy, at::kByte, kept_bytes ? kept_bytes : -1);
                if (want_dx) dx = at::empty({dy.size(0), l.in_f}, dy.options());
                if (want_dc) dc = at::empty({c.size(0), c.size(1)}, c.options());
                if (want_sb) dsb = at::empty({1}, dy.options().dtype(at::kFloat));
                const auto bias = ctx->saved_data["bias"].toIntVector();
                const BiasGrads g(ctx, dy, bias, has_sb ? 3 : 2);
                const int64_t least = rdb_linear_workspace_bytes(RDB_OP_LINEAR_BWD_KEPT, &d);
                if (g.ref.k >= 0) {
                    const int64_t need = std::max(least, rdb_bias_bwd_workspace_bytes(d.tokens, d.out_f));
                    const Tensor ws = bytes(need, dy);
                    check(rdb_linear_bwd_kept_pseudo_bias(ptr(dx), l.in_f, ptr(dc), code(c.scalar_type()), want_sb ? dsb.data_ptr<float>() : nullptr, dy.data_ptr(),
                                                          dy.stride(0), ptr(xs), want_sb ? xs.stride(0) : l.in_f, kept.data_ptr(), c.data_ptr(), ptr(s), &g.ref, &d,
                                                          ptr(ws), need, stream_of(dy)),
                          "rdb_linear_bwd_kept");
                    if (want_sb) dsb = dsb.to(sb.scalar_type());
                    db = g.done(bias);
                    return;
                }
                const Tensor ws = bytes(least, dy);
                check(rdb_linear_bwd_kept(ptr(dx), l.in_f, ptr(dc), code(c.scalar_type()), want_sb ? dsb.data_ptr<float>() : nullptr, dy.data_ptr(), dy.stride(0),
                                          ptr(xs), want_sb ? xs.stride(0) : l.in_f, kept.data_ptr(), c.data_ptr(), ptr(s), &d, ptr(ws), least, stream_of(dy)),
                      "rdb_linear_bwd_kept");
                if (want_sb) dsb = dsb.to(sb.scalar_type());
            }
            db = bias_grads(ctx, dy, ctx->saved_data["bias"].toIntVector(), has_sb ? 3 : 2);
            return;
        }
        if (want_dx && want_sb && l.sO == l.in_f && l.sI == 1) {
            // the random-bias product dy.R that dx needs anyway also gives the gradient of the bias's scale (reduced against x
            // in the same pass), so the coefficient gradient below comes from the factored kernels and dW is never formed
            auto both = linear_bwd_dx_dscale(dy, x, coefs, l, sb);
            if (both.first.defined()) {
                dx = both.first;
                dsb = both.second.to(sb.scalar_type());
                want_sb = false;
            }
        }
        if (want_dx && !dx.defined()) dx = linear_bwd_dx(dy, coefs, l, sb);
        if (want_dc || want_sb) {
            auto both = linear_bwd_dcoef(dy, x, coefs, l, want_sb);
            dc = both.first.to(coefs.scalar_type());
            if (want_sb) dsb = both.second.to(sb.scalar_type());
        }
        db = bias_grads(ctx, dy, ctx->saved_data["bias"].toIntVector(), has_sb ? 3 : 2);
    }
};

// ----------------------------------------------------------------------------------------------- projected form
Tensor dense(const Tensor &t);
Tensor relu_squared(const Tensor &x, const Tensor &dy = Tensor());   // relu(x)^2, or with dy its gradient
Tensor relu_squared_with_graph(const Tensor &x, const Tensor &dy);
// The forward pass keeps z = x.N^T (and, in bf16, the transposed coefficients) for the backward pass, which needs nothing else
// of x; with the fused random bias its full-rank share is added on top in both directions and x is saved as well.
// square: where relu(y)^2 is left beside y, for a layer of that input (or NULL).
// squared: the layer's input is relu(x)^2 of an x that wants a gradient, formed here unless `formed` is that, which nothing keeps, and its gradient goes through that on its way to
// memory (8192 tokens x 3072 -> 768, k = 256: backward and a pass over its dx 62.8 us, 47.7 so); x is saved for it.
class ProjectedLinear : public Function<ProjectedLinear> {
  public:
    static Tensor forward(AutogradContext *ctx, const Tensor &x0, const Tensor &coefs, const OptTensor &bias, const OptTensor &bias_scale, int64_t bias_seed,
                          const OptTensor &scale_bias, const Layer &l, bool squared, const Tensor *formed = nullptr, Tensor *square = nullptr)
    {
        const Bias pb{bias, bias_scale, bias_seed};
        const c10::OptionalDeviceGuard guard(x0.device());
        const Tensor x = !squared ? near_act(x0) : formed ? *formed : relu_squared(x0), c = coefs.contiguous();
        const rdb_linear_desc d = desc(x, l, c);
        const int64_t need = rdb_linear_projection_bytes(&d);
        Tensor state = bytes(need, x), y = at::empty({x.size(0), l.out_f}, x.options());
        const Tensor b = pb.values(l.out_f, x.scalar_type());
        void *s = stream_of(x);
        const int64_t one_product = scale_bias ? rdb_linear_workspace_bytes(RDB_OP_LINEAR_PROJECT_FWD_RBIAS, &d) : 0;
        if (one_product) {
            const Tensor sb = native(*scale_bias).to(at::kBFloat16), ws = bytes(one_product, x);
            check(rdb_linear_project_fwd_rbias(y.data_ptr(), l.out_f, ptr(state), x.data_ptr(), x.stride(0), c.data_ptr(), sb.data_ptr(), ptr(b), &d, ptr(ws),
                                               one_product, s),
                  "rdb_linear_project_fwd_rbias");
        } else {
            const int64_t room = rdb_linear_workspace_bytes(RDB_OP_LINEAR_PROJECT, &d);
            const Tensor ws = bytes(room, x);
            if (square) *square = at::empty_like(y);
            check(square ? rdb_linear_project_fwd_relu_square(y.data_ptr(), square->data_ptr(), ptr(state), x.data_ptr(), x.stride(0), c.data_ptr(), &d, ptr(ws), room, s)
                         : rdb_linear_project_fwd_ws(y.data_ptr(), l.out_f, ptr(state), x.data_ptr(), x.stride(0), c.data_ptr(), ptr(b), &d, ptr(ws), room, s),
                  "rdb_linear_project_fwd");
        }
        if (scale_bias && !one_product) {
            const Tensor sb = native(*scale_bias).to(at::kBFloat16);
            const rdb_linear_desc r = rbias_desc(x, l);
            const int64_t room = rdb_linear_workspace_bytes(RDB_OP_LINEAR_RBIAS_FWD, &r);
            const Tensor ws = bytes(room, x);
            check(rdb_linear_rbias_fwd_ws(y.data_ptr(), l.out_f, x.data_ptr(), x.stride(0), sb.data_ptr(), &r, ptr(ws), room, s), "rdb_linear_rbias_fwd");
        }
        tick(x);
        ctx->save_for_backward({state, coefs, scale_bias.value_or(Tensor()), scale_bias || squared ? x0 : Tensor()});
        ctx->saved_data["layer"] = std::vector<int64_t>{l.in_f, l.out_f, (int64_t)l.seed, scale_bias ? 1 : 0, pb.tensors(), coefs.size(1), squared ? 1 : 0};
        ctx->saved_data["bias"] = pb.meta();
        return y;
    }
    static variable_list backward(AutogradContext *ctx, const variable_list &grads)
    {
        Tensor dx, dc, ds;
        std::pair<Tensor, Tensor> db;
        const auto m = ctx->saved_data["layer"].toIntVector();
        const bool graph = at::GradMode::is_enabled();   // relu(x)^2 is then gone through by stock operators, which have further derivatives
        gradients(ctx, grads, dx, dc, ds, db, m[6] && !graph);
        layer_gradients(grads[0], m[3] ? (int)(2 + m[4]) : -1, dx, dc, ds, db, ctx->saved_data["bias"].toIntVector());
        if (m[6] && graph && dx.defined()) dx = relu_squared_with_graph(ctx->get_saved_variables()[3], dx);
        return {dx, dc, db.first, db.second, Tensor(), ds, Tensor(), Tensor(), Tensor(), Tensor()};
    }
    // through: dx is to be the gradient behind relu(x)^2
    static void gradients(AutogradContext *ctx, const variable_list &grads, Tensor &dx, Tensor &dc, Tensor &dsb, std::pair<Tensor, Tensor> &db, bool through)
    {
        const auto saved = ctx->get_saved_variables();
        const Tensor &state = saved[0], &coefs = saved[1], &scale_bias = saved[2];
        const auto m = ctx->saved_data["layer"].toIntVector();
        const Layer l{m[0], m[1], m[0], 1, (uint32_t)m[2]};
        const bool has_sb = m[3] != 0;
        constexpr const char *who = "linear (backward)";
        restored(who, coefs, grads[0], {l.out_f, m[5]});
        if (has_sb) restored(who, scale_bias, grads[0], scale_bias.sizes());
        if (has_sb || m[6]) restored(who, saved[3], grads[0], {grads[0].size(0), l.in_f});
        const at::AutoGradMode no_grad(false);
        through = through && ctx->needs_input_grad(0);
        const Tensor gate = through ? dense(saved[3]) : Tensor();
        if (through) restored_values(who, gate, grads[0], at::kBFloat16, grads[0].size(0) * l.in_f);
        const bool want_x = ctx->needs_input_grad(0), want_dc = ctx->needs_input_grad(1), want_sb = has_sb && ctx->needs_input_grad(2 + m[4]);
        const bool want_dx = want_x || want_sb;   // the gradient of the scale comes out of the random-bias share of dx
        Tensor dy = near_act(grads[0]);
        const bool f32 = coefs.scalar_type() == at::kFloat;
        if (!f32 && (dy.stride(0) % 8 || (uintptr_t)dy.data_ptr() % 16)) dy = dy.contiguous();   // rows with a leading dimension are read in place
        const Tensor c = coefs.contiguous();
        const c10::OptionalDeviceGuard guard(dy.device());
        const rdb_linear_desc d = desc(dy, l, c);
        if (c.scalar_type() != dy.scalar_type()) fail(PyExc_RuntimeError, std::string(who) + ": the saved coefficients came back in another dtype");
        restored_values(who, state, dy, at::kByte, rdb_linear_projection_bytes(&d));
        void *s = stream_of(dy);
        // with the fused random bias: both shares of dx, all gradients, in one call where the layer has such a form (it refuses what the two calls refuse)
        const int64_t both_shares = has_sb && !f32 && want_dx && want_dc ? rdb_linear_workspace_bytes(RDB_OP_LINEAR_BWD_PROJECTED_RBIAS, &d) : 0;
        if (both_shares) {
            const Tensor x = want_sb ? near_input(saved[3], dy) : Tensor(), sb = native(scale_bias).to(at::kBFloat16), ws = bytes(both_shares, dy);
            const auto dt = scale_bias.scalar_type() == at::kBFloat16 ? at::kBFloat16 : at::kFloat;
            dx = at::empty({dy.size(0), l.in_f}, dy.options());
            dc = at::empty({c.size(0), c.size(1)}, dy.options().dtype(at::kBFloat16));
            if (want_sb) dsb = at::empty({1}, dy.options().dtype(dt));
            check(rdb_linear_bwd_projected_rbias(dx.data_ptr(), l.in_f, dc.data_ptr(), RDB_BF16, ptr(dsb), code(dt), dy.data_ptr(), dy.stride(0), state.data_ptr(),
                                                 ptr(x), want_sb ? x.stride(0) : 0, c.data_ptr(), sb.data_ptr(), &d, ptr(ws), both_shares, s),
                  "rdb_linear_bwd_projected_rbias");
            if (want_sb) dsb = dsb.to(scale_bias.scalar_type());
        } else if (want_dc && (want_dx || f32)) {
            // bf16 coefficients: their gradient leaves the kernel that adds it up in bf16, where the layer runs as one chunk of tokens
            const bool to_bf16 = !f32 && rdb_linear_projection_chunks(&d, nullptr) == 1;
            const int64_t need = rdb_linear_workspace_bytes(to_bf16 ? RDB_OP_LINEAR_BWD_PROJECTED_TO : RDB_OP_LINEAR_BWD_PROJECTED, &d);
            const Tensor ws = bytes(need, dy);
            if (want_dx) dx = at::empty({dy.size(0), l.in_f}, dy.options());
            dc = at::empty({c.size(0), c.size(1)}, dy.options().dtype(to_bf16 ? at::kBFloat16 : at::kFloat));
            if (through && to_bf16 && rdb_linear_bwd_projected_takes_relu_square(&d) && (uintptr_t)dx.data_ptr() % 128 == 0) {
                check(rdb_linear_bwd_projected_relu_square(dx.data_ptr(), dc.data_ptr(), dy.data_ptr(), dy.stride(0), state.data_ptr(), c.data_ptr(), gate.data_ptr(), &d,
                                                           ptr(ws), need, s),
                      "rdb_linear_bwd_projected_relu_square");
                through = false;
            } else {
                check(to_bf16 ? rdb_linear_bwd_projected_to(ptr(dx), l.in_f, dc.data_ptr(), RDB_BF16, dy.data_ptr(), dy.stride(0), state.data_ptr(), c.data_ptr(),
                                                            &d, ptr(ws), need, s)
                              : rdb_linear_bwd_projected(ptr(dx), l.in_f, dc.data_ptr<float>(), dy.data_ptr(), dy.stride(0), state.data_ptr(), c.data_ptr(), &d,
                                                         ptr(ws), need, s),
                      "rdb_linear_bwd_projected");
            }
            dc = dc.to(c.scalar_type());
        } else if (want_dx) {
            dx = linear_bwd_dx(dy, c, l, Tensor());
        } else if (want_dc) {
            dc = at::empty({c.size(0), c.size(1)}, dy.options().dtype(at::kFloat));
            check(rdb_linear_bwd_dcoef_projected(dc.data_ptr<float>(), dy.data_ptr(), dy.stride(0), state.data_ptr(), &d, s), "rdb_linear_bwd_dcoef_projected");
            dc = dc.to(c.scalar_type());
        }
        if (has_sb && dx.defined() && !both_shares) {
            const Tensor x = near_input(saved[3], dy), sb = native(scale_bias).to(at::kBFloat16);
            const rdb_linear_desc r = rbias_desc(dy, l);
            const int64_t need = rdb_linear_workspace_bytes(RDB_OP_LINEAR_RBIAS_BWD_FULL, &r);
            const Tensor ws = bytes(need, dy);
            if (want_sb) {
                const auto dt = scale_bias.scalar_type() == at::kBFloat16 ? at::kBFloat16 : at::kFloat;
                dsb = at::empty({1}, dy.options().dtype(dt));
                check(rdb_linear_rbias_bwd_to(dx.data_ptr(), l.in_f, dsb.data_ptr(), code(dt), dy.data_ptr(), dy.stride(0), x.data_ptr(), x.stride(0),
                                              sb.data_ptr(), &r, ptr(ws), need, s),
                      "rdb_linear_rbias_bwd");
                dsb = dsb.to(scale_bias.scalar_type());
            } else {
                check(rdb_linear_rbias_bwd(dx.data_ptr(), l.in_f, nullptr, dy.data_ptr(), dy.stride(0), nullptr, 0, sb.data_ptr(), &r, ptr(ws), need, s),
                      "rdb_linear_rbias_bwd");
            }
        }
        if (!want_x) dx = Tensor();
        if (through && dx.defined()) dx = relu_squared(gate, dx);
        db = bias_grads(ctx, dy, ctx->saved_data["bias"].toIntVector(), 2);
    }
};

// ----------------------------------------------------------------------------------------------- the vector-coef layer
// Gradient of the values of a vector-coef tensor -> gradients of its coefficients and scale, differentiable (for create_graph).
class CoefGrads : public Function<CoefGrads> {
  public:
    static variable_list forward(AutogradContext *ctx, const Tensor &dvalues, int64_t k, int64_t seed, bool want_scale)
    {
        ctx->saved_data["n"] = dvalues.numel();
        ctx->saved_data["seed"] = seed;
        ctx->saved_data["dtype"] = (int64_t)dvalues.scalar_type();
        ctx->saved_data["sizes"] = dvalues.sizes().vec();
        const auto g = coef_grads(dvalues, k, seed, true, want_scale);
        return want_scale ? variable_list{g.first, g.second} : variable_list{g.first};
    }
    static variable_list backward(AutogradContext *ctx, const variable_list &grads);   // by CoefValues
};
// The values themselves, differentiable in coef and scale.
class CoefValues : public Function<CoefValues> {
  public:
    static Tensor forward(AutogradContext *ctx, const Tensor &coef, const OptTensor &scale_bias, int64_t n, int64_t seed)
    {
        ctx->saved_data["m"] = std::vector<int64_t>{coef.numel(), seed, (int64_t)coef.scalar_type(), scale_bias ? (int64_t)scale_bias->scalar_type() : -1};
        return coef_values(coef, scale_bias, n, seed);
    }
    static variable_list backward(AutogradContext *ctx, const variable_list &grads)
    {
        const auto m = ctx->saved_data["m"].toIntVector();
        const auto g = CoefGrads::apply(grads[0].contiguous(), m[0], m[1], m[3] >= 0);
        return {g[0].to((at::ScalarType)m[2]), m[3] >= 0 ? g[1].to((at::ScalarType)m[3]) : Tensor(), Tensor(), Tensor()};
    }
};

variable_list CoefGrads::backward(AutogradContext *ctx, const variable_list &grads)
{
    const Tensor v = CoefValues::apply(grads[0], grads.size() > 1 ? OptTensor(grads[1]) : OptTensor(), ctx->saved_data["n"].toInt(), ctx->saved_data["seed"].toInt());
    return {v.to((at::ScalarType)ctx->saved_data["dtype"].toInt()).view(ctx->saved_data["sizes"].toIntVector()), Tensor(), Tensor(), Tensor()};
}

std::pair<Tensor, Tensor> bias_grads_with_graph(const Tensor &dy, const std::vector<int64_t> &m)
{
    const Tensor db = dy.sum(0, false, at::kFloat);
    if (m[1] < 0) return {db.to((at::ScalarType)m[2]), Tensor()};
    const auto g = CoefGrads::apply(db, m[0], m[1], m[3] >= 0);
    return {g[0].to((at::ScalarType)m[2]), m[3] >= 0 ? g[1].to((at::ScalarType)m[3]) : Tensor()};
}

// out [M x N], contiguous, = A . B^T (+ bias); A [M x K], B [N x K], or stored transposed (across).  fp32: the library's own product;
// bf16: torch's.  out is the caller's, because what an autograd function returns must not be a view (in-place changes of it are refused)
const Tensor &product(const Tensor &out, const Tensor &a, bool a_across, const Tensor &b, bool b_across, const Tensor &bias)
{
    const int64_t M = a.size(a_across ? 1 : 0), K = a.size(a_across ? 0 : 1), N = b.size(b_across ? 1 : 0);
    if (a.scalar_type() == at::kFloat) {
        const int64_t need = rdb_product_f32_workspace_bytes(M, N, K);
        const Tensor ws = bytes(need, a);
        const int rc = rdb_product_f32(out.data_ptr<float>(), a.data_ptr<float>(), a.stride(0), a_across, b.data_ptr<float>(), b.stride(0), b_across,
                                       bias.defined() ? bias.data_ptr<float>() : nullptr, M, N, K, ptr(ws), need, stream_of(a));
        if (rc != RDB_E_UNSUPPORTED) {
            check(rc, "rdb_product_f32");
            return out;
        }
    }
    const Tensor l = a_across ? a.t() : a, r = b_across ? b : b.t();
    Tensor to = out.view({M, N});
    if (bias.defined()) at::addmm_out(to, bias, l, r);
    else at::mm_out(to, l, r);
    return out;
}

// y = x.W^T (+ b) with W and b vector-coef tensors: W is formed (k hashed values per element), multiplied as a dense matrix, and
// in the backward pass dW = dy^T.x is formed and contracted with the hashed values.  Forming W is the most expensive step of the
// layer, and the backward pass needs it again for dx: it is kept for that where it takes no more memory than the activations x
// and y of this pass, which the program holds anyway; otherwise it is formed again, so that a layer never holds more than twice
// what its activations take (1024 tokens x 768 -> 3072, k = 256: 9.4 MB beside 15.7 MB).
class VectorLinear : public Function<VectorLinear> {
  public:
    static Tensor forward(AutogradContext *ctx, const Tensor &x0, const Tensor &coef, const OptTensor &scale, const OptTensor &bias, const OptTensor &bias_scale,
                          int64_t bias_seed, const Layer &l)
    {
        const Bias b{bias, bias_scale, bias_seed};
        const c10::OptionalDeviceGuard guard(x0.device());
        Tensor W, bv;
        if (b.beside(l.out_f, x0.scalar_type()) && coef.scalar_type() == at::kFloat && (!scale || !scale->defined() || scale->scalar_type() == at::kFloat)) {
            const Tensor c = coef.contiguous(), sc = scale && scale->defined() ? scale->contiguous() : Tensor();
            const Tensor bc = b.coef->contiguous(), bs = b.scale && b.scale->defined() ? b.scale->contiguous() : Tensor();
            W = at::empty({l.out_f, l.in_f}, c.options());
            bv = at::empty({l.out_f}, c.options());
            const rdb_pseudo_bias pb = b.ref(bc, bs, bv);
            check(rdb_materialize_weight_and_bias(W.data_ptr<float>(), W.numel(), c.data_ptr<float>(), c.numel(), l.seed, sc.defined() ? sc.data_ptr<float>() : nullptr,
                                                  &pb, l.out_f, stream_of(c)),
                  "rdb_materialize_weight_and_bias");
        } else {
            W = coef_values(coef, scale, l.out_f * l.in_f, l.seed).view({l.out_f, l.in_f});
            bv = b.values(l.out_f, x0.scalar_type());
        }
        Tensor y = values(x0, W, bv, l);
        const bool keep = ctx != nullptr && W.numel() <= x0.numel() + y.numel();
        if (ctx) {
            ctx->save_for_backward({x0, coef, scale.value_or(Tensor()), keep && x0.requires_grad() ? W : Tensor()});
            ctx->saved_data["layer"] = std::vector<int64_t>{l.in_f, l.out_f, (int64_t)l.seed, scale ? (int64_t)scale->scalar_type() : -1, coef.numel()};
            ctx->saved_data["bias"] = b.meta();
            ctx->saved_data["x"] = x0.sizes().vec();
        }
        return y;
    }
    static Tensor values(const Tensor &x0, const Tensor &W, const Tensor &bias, const Layer &l)
    {
        auto sizes = x0.sizes().vec();
        sizes.back() = l.out_f;
        return product(at::empty(sizes, x0.options()), act(x0.reshape({-1, l.in_f})), false, W, false, bias);
    }
    static variable_list backward(AutogradContext *ctx, const variable_list &grads)
    {
        const auto saved = ctx->get_saved_variables();
        const auto m = ctx->saved_data["layer"].toIntVector();
        const Layer l{m[0], m[1], m[0], 1, (uint32_t)m[2]};
        const bool has_scale = m[3] >= 0;
        const bool want_x = ctx->needs_input_grad(0), want_c = ctx->needs_input_grad(1), want_s = has_scale && ctx->needs_input_grad(2);
        const Tensor &x0 = saved[0], &coef = saved[1];
        const OptTensor scale = has_scale ? OptTensor(saved[2]) : OptTensor();
        constexpr const char *who = "linear (backward)";
        restored(who, x0, grads[0], ctx->saved_data["x"].toIntVector());
        restored(who, coef, grads[0], {m[4]});
        if (has_scale) restored(who, saved[2], grads[0], saved[2].sizes());
        const c10::OptionalDeviceGuard guard(x0.device());
        Tensor dx, dc, ds;
        const Tensor dy = act(grads[0].reshape({-1, l.out_f}));
        if (at::GradMode::is_enabled()) {   // create_graph: the same products from differentiable operators
            const Tensor x = x0.reshape({-1, l.in_f});
            if (want_x) dx = dy.mm(CoefValues::apply(coef, scale, l.out_f * l.in_f, (int64_t)l.seed).view({l.out_f, l.in_f})).view(x0.sizes());
            if (want_c || want_s) {
                const auto g = CoefGrads::apply(dy.t().mm(x), coef.numel(), (int64_t)l.seed, want_s);
                if (want_c) dc = g[0].to(coef.scalar_type());
                if (want_s) ds = g[1].to((at::ScalarType)m[3]);
            }
            const auto bm = ctx->saved_data["bias"].toIntVector();
            const auto db = bm[0] < 0 ? std::pair<Tensor, Tensor>() : bias_grads_with_graph(dy, bm);
            return {dx, dc, ds, db.first, db.second, Tensor(), Tensor()};
        }
        const auto bm = ctx->saved_data["bias"].toIntVector();
        const int bias_at = has_scale ? 3 : 2;
        Tensor W;
        if (want_x) {
            const bool kept = saved[3].defined();
            if (kept) restored(who, restored_values(who, saved[3], dy, x0.scalar_type(), l.out_f * l.in_f), dy, {l.out_f, l.in_f});
            W = kept ? saved[3] : coef_values(coef, scale, l.out_f * l.in_f, l.seed).view({l.out_f, l.in_f});
        }
        // the gradients that a layer without a fused random bias asks for, together
        const bool b_coef = bm[0] >= 0 && ctx->needs_input_grad(bias_at), b_scale = bm[0] >= 0 && bm[3] >= 0 && ctx->needs_input_grad(bias_at + 1);
        if (want_c && !want_s && !b_scale && !(b_coef && bm[1] < 0) && dy.scalar_type() == at::kFloat && x0.scalar_type() == at::kFloat && dy.numel() && x0.numel()) {
            const int64_t k = coef.numel(), bk = b_coef ? bm[0] : 0, need = rdb_vector_linear_bwd_workspace_bytes(dy.size(0), l.in_f, l.out_f, k, want_x, bk > 0);
            if (need > 0 && rdb_vector_linear_bwd_pays(dy.size(0), l.in_f, l.out_f, want_x, bk > 0)) {
                const Tensor x = act(x0.reshape({-1, l.in_f})), ws = bytes(need, dy);
                const auto f32 = dy.options();
                if (want_x) dx = at::empty(x0.sizes(), f32);
                dc = at::empty({k}, f32);
                Tensor db = b_coef ? at::empty({bk}, f32) : Tensor();
                const int rc = rdb_vector_linear_bwd(want_x ? dx.data_ptr<float>() : nullptr, dc.data_ptr<float>(), bk > 0 ? db.data_ptr<float>() : nullptr, dy.data_ptr<float>(),
                                                     dy.stride(0), x.data_ptr<float>(), x.stride(0), want_x ? W.data_ptr<float>() : nullptr, dy.size(0), l.in_f, l.out_f, k,
                                                     l.seed, bk, (uint32_t)std::max<int64_t>(bm[1], 0), ptr(ws), need, stream_of(dy));
                if (rc != RDB_E_UNSUPPORTED) {
                    check(rc, "rdb_vector_linear_bwd");
                    dc = dc.to(coef.scalar_type());
                    if (b_coef) db = db.to((at::ScalarType)bm[2]);
                    return {dx, dc, ds, db, Tensor(), Tensor(), Tensor()};
                }
            }
        }
        if (want_x) dx = product(at::empty(x0.sizes(), dy.options()), dy, false, W, true, Tensor());
        if (want_c || want_s) {
            const Tensor dW = product(at::empty({l.out_f, l.in_f}, dy.options()), dy, true, act(x0.reshape({-1, l.in_f})), true, Tensor());
            const auto g = coef_grads(dW, coef.numel(), l.seed, want_c, want_s);
            if (want_c) dc = g.first.to(coef.scalar_type());
            if (want_s) ds = g.second.to((at::ScalarType)m[3]);
        }
        const auto db = bias_grads(ctx, dy, bm, bias_at);
        return {dx, dc, ds, db.first, db.second, Tensor(), Tensor()};
    }
};

// Gradient of f(inputs...) with a graph of its own (create_graph), by f's stock operators.  Inputs without a gradient to come: undefined.
// f takes views of the inputs: a gradient taken at an input itself runs the hooks on it, and they run on the whole of its gradient
// in the pass that this is part of.
template <typename F> variable_list stock_gradient(F f, variable_list inputs, const variable_list &grads)
{
    variable_list wanted;
    for (Tensor &t : inputs)
        if (t.requires_grad()) wanted.push_back(t = t.alias());
    variable_list out(inputs.size());
    if (wanted.empty()) return out;
    const variable_list got = torch::autograd::grad(f(inputs), wanted, grads, true, true, true);
    size_t n = 0;
    for (size_t i = 0; i < inputs.size(); ++i)
        if (inputs[i].requires_grad()) out[i] = got[n++];
    return out;
}

// rows idx of a (*, rowsize) vector-coef table, fp32
class EmbedRows : public Function<EmbedRows> {
  public:
    static Tensor forward(AutogradContext *ctx, const Tensor &idx0, const Tensor &coef, int64_t rowsize, int64_t seed)
    {
        const Tensor idx = idx0.to(at::kLong).contiguous();
        if (ctx) {
            ctx->save_for_backward({idx});
            ctx->saved_data["m"] = std::vector<int64_t>{coef.numel(), rowsize, seed, (int64_t)coef.scalar_type()};
        }
        return rows(idx, coef, rowsize, seed);
    }
    static Tensor rows(const Tensor &idx, const Tensor &coef, int64_t rowsize, int64_t seed)
    {
        const Tensor c = native(coef);
        const c10::OptionalDeviceGuard guard(c.device());
        auto sizes = idx.sizes().vec();
        sizes.push_back(rowsize);
        Tensor out = at::empty(sizes, c.options().dtype(at::kFloat));
        check(rdb_embed_fwd(out.data_ptr<float>(), idx.data_ptr<int64_t>(), idx.numel(), c.data_ptr(), code(c.scalar_type()), c.numel(), rowsize, (uint32_t)seed,
                            stream_of(c)),
              "rdb_embed_fwd");
        return out;
    }
    static variable_list backward(AutogradContext *ctx, const variable_list &grads)
    {
        const Tensor idx = ctx->get_saved_variables()[0];
        const auto m = ctx->saved_data["m"].toIntVector();
        return {Tensor(), once_differentiable("embed_fwd", gradient(idx, grads[0], m), grads[0], {}), Tensor(), Tensor()};
    }
    static Tensor gradient(const Tensor &idx, const Tensor &grad, const std::vector<int64_t> &m)
    {
        const at::AutoGradMode no_grad(false);
        const Tensor d = native(grad);
        restored_values("embedding (backward)", idx, d, at::kLong, m[1] ? d.numel() / m[1] : 0);
        const c10::OptionalDeviceGuard guard(d.device());
        Tensor dc = at::empty({m[0]}, d.options().dtype(at::kFloat));
        const int64_t need = rdb_embed_bwd_workspace_bytes(idx.numel(), m[1], m[0]);
        const Tensor ws = bytes(need, d);
        check(rdb_embed_bwd(dc.data_ptr<float>(), idx.data_ptr<int64_t>(), idx.numel(), d.data_ptr(), code(d.scalar_type()), m[0], m[1], (uint32_t)m[2], ptr(ws),
                            need, stream_of(d)),
              "rdb_embed_bwd");
        return dc.to((at::ScalarType)m[3]);
    }
};

// ----------------------------------------------------------------------------------------------- the rest of a transformer block
// bf16 on the GPU; what gpt.py calls when its tensors are that.
void need_bf16(const char *who, const Tensor &t)
{
    if (!t.is_cuda() || t.scalar_type() != at::kBFloat16) fail(PyExc_ValueError, std::string(who) + " needs bf16 tensors on the GPU");
}
// Contiguous from a 16-byte boundary on: the kernels read 8 and 16 bytes at a time, and a contiguous slice may begin anywhere.
Tensor dense(const Tensor &t)
{
    const Tensor c = t.contiguous();
    return (uintptr_t)c.data_ptr() % 16 ? c.clone() : c;
}
int64_t row_count(const Tensor &x) { return x.size(-1) ? x.numel() / x.size(-1) : 0; }

// A gradient asked for under create_graph is computed by the stock operators, from the inputs as they were given.

// x -> x / rms(x) over the last dimension
class RmsNorm : public Function<RmsNorm> {
  public:
    static Tensor forward(AutogradContext *ctx, const Tensor &x0, double eps)
    {
        const Tensor x = dense(x0);
        const c10::OptionalDeviceGuard guard(x.device());
        Tensor y = at::empty_like(x), rstd = at::empty({row_count(x)}, x.options().dtype(at::kFloat));
        check(rdb_rms_norm_fwd(y.data_ptr(), nullptr, rstd.data_ptr<float>(), x.data_ptr(), nullptr, row_count(x), x.size(-1), (float)eps, stream_of(x)),
              "rdb_rms_norm_fwd");
        ctx->save_for_backward({x0, rstd});
        ctx->saved_data["eps"] = eps;
        return y;
    }
    static Tensor stock(const Tensor &x, double eps) { return at::rms_norm(x, {x.size(-1)}, {}, eps); }
    static variable_list backward(AutogradContext *ctx, const variable_list &grads)
    {
        const auto saved = ctx->get_saved_variables();
        constexpr const char *who = "rms_norm (backward)";
        restored(who, saved[0], grads[0], grads[0].sizes());
        if (at::GradMode::is_enabled()) {
            const double eps = ctx->saved_data["eps"].toDouble();
            return {stock_gradient([&](const variable_list &in) { return variable_list{stock(in[0], eps)}; }, {saved[0]}, {grads[0]})[0], Tensor()};
        }
        const Tensor x = dense(saved[0]), dy = dense(grads[0]);
        restored_values(who, x, dy, at::kBFloat16, dy.numel());
        restored_values(who, saved[1], dy, at::kFloat, row_count(dy));
        const c10::OptionalDeviceGuard guard(x.device());
        Tensor dx = at::empty_like(x);
        check(rdb_rms_norm_bwd(dx.data_ptr(), dy.data_ptr(), x.data_ptr(), nullptr, saved[1].data_ptr<float>(), row_count(x), x.size(-1), stream_of(x)),
              "rdb_rms_norm_bwd");
        return {dx, Tensor()};
    }
};

// (x, delta) -> (x + delta, its normalisation)
class AddRmsNorm : public Function<AddRmsNorm> {
  public:
    static variable_list forward(AutogradContext *ctx, const Tensor &x0, const Tensor &delta0, double eps)
    {
        const Tensor x = dense(x0), delta = dense(delta0);
        const c10::OptionalDeviceGuard guard(x.device());
        Tensor y = at::empty_like(x), sum = at::empty_like(x), rstd = at::empty({row_count(x)}, x.options().dtype(at::kFloat));
        check(rdb_rms_norm_fwd(y.data_ptr(), sum.data_ptr(), rstd.data_ptr<float>(), x.data_ptr(), delta.data_ptr(), row_count(x), x.size(-1), (float)eps,
                               stream_of(x)),
              "rdb_rms_norm_fwd");
        ctx->save_for_backward({sum, rstd});
        ctx->saved_data["eps"] = eps;
        ctx->set_materialize_grads(false);
        return {sum, y};
    }
    static variable_list backward(AutogradContext *ctx, const variable_list &grads)
    {
        const auto saved = ctx->get_saved_variables();
        if (!grads[1].defined()) return {grads[0], grads[0], Tensor()};
        const Tensor &x = saved[0];   // the sum: an output, with this function behind it
        constexpr const char *who = "add_rms_norm (backward)";
        restored(who, x, grads[1], grads[1].sizes());
        if (at::GradMode::is_enabled()) {
            const double eps = ctx->saved_data["eps"].toDouble();
            Tensor d = stock_gradient([&](const variable_list &in) { return variable_list{RmsNorm::stock(in[0], eps)}; }, {x}, {grads[1]})[0];
            if (d.defined() && grads[0].defined()) d = d + grads[0];
            return {d, d, Tensor()};
        }
        const Tensor dy = dense(grads[1]), dsum = grads[0].defined() ? dense(grads[0]) : Tensor();
        restored_values(who, x, dy, at::kBFloat16, dy.numel());
        restored_values(who, saved[1], dy, at::kFloat, row_count(dy));
        const c10::OptionalDeviceGuard guard(x.device());
        Tensor dx = at::empty_like(x);
        check(rdb_rms_norm_bwd(dx.data_ptr(), dy.data_ptr(), x.data_ptr(), ptr(dsum), saved[1].data_ptr<float>(), row_count(x), x.size(-1), stream_of(x)),
              "rdb_rms_norm_bwd");
        return {dx, dx, Tensor()};
    }
};

Tensor relu_squared(const Tensor &x0, const Tensor &dy0)
{
    const Tensor x = dense(x0), dy = dy0.defined() ? dense(dy0) : Tensor();
    const c10::OptionalDeviceGuard guard(x.device());
    Tensor out = at::empty_like(x);
    check(rdb_relu_square(out.data_ptr(), x.data_ptr(), ptr(dy), x.numel(), stream_of(x)), "rdb_relu_square");
    return out;
}
Tensor relu_squared_with_graph(const Tensor &x, const Tensor &dy)
{
    return stock_gradient([](const variable_list &in) { return variable_list{at::relu(in[0]).square()}; }, {x}, {dy})[0];
}
class ReluSquare : public Function<ReluSquare> {
  public:
    static Tensor forward(AutogradContext *ctx, const Tensor &x0)
    {
        ctx->save_for_backward({x0});
        return relu_squared(x0);
    }
    static variable_list backward(AutogradContext *ctx, const variable_list &grads)
    {
        const Tensor x0 = ctx->get_saved_variables()[0];
        constexpr const char *who = "relu_square (backward)";
        restored(who, x0, grads[0], grads[0].sizes());
        if (at::GradMode::is_enabled()) return {relu_squared_with_graph(x0, grads[0])};
        const Tensor x = dense(x0), dy = dense(grads[0]);
        restored_values(who, x, dy, at::kBFloat16, dy.numel());
        return {relu_squared(x, dy)};
    }
};

// rows idx of a dense bf16 table; the gradient is the table's, in one launch
class EmbedDense : public Function<EmbedDense> {
  public:
    static Tensor forward(AutogradContext *ctx, const Tensor &weight, const Tensor &idx)
    {
        ctx->save_for_backward({idx});
        ctx->saved_data["m"] = std::vector<int64_t>{weight.size(0), weight.size(1), idx.numel()};
        return at::embedding(weight, idx);
    }
    static variable_list backward(AutogradContext *ctx, const variable_list &grads)
    {
        const Tensor idx0 = ctx->get_saved_variables()[0];
        const auto m = ctx->saved_data["m"].toIntVector();
        constexpr const char *who = "embedding (backward)";
        restored(who, idx0, grads[0], grads[0].sizes().slice(0, grads[0].dim() - 1));
        if (at::GradMode::is_enabled() || grads[0].scalar_type() != at::kBFloat16 || (idx0.scalar_type() != at::kLong && idx0.scalar_type() != at::kInt))
            return {at::embedding_dense_backward(grads[0], idx0, m[0], -1, false), Tensor()};
        const Tensor idx = idx0.contiguous(), dy = dense(grads[0]);
        restored_values(who, idx, dy, idx.scalar_type(), m[2]);
        const c10::OptionalDeviceGuard guard(dy.device());
        Tensor dw = at::empty({m[0], m[1]}, dy.options());
        check(rdb_embedding_bwd(dw.data_ptr(), idx.data_ptr(), (int)idx.element_size(), dy.data_ptr(), m[2], m[0], m[1], stream_of(dy)), "rdb_embedding_bwd");
        return {dw, Tensor()};
    }
};

// mean cross entropy of bf16 logits (rows, classes), computed in fp32
class CrossEntropy : public Function<CrossEntropy> {
  public:
    static Tensor forward(AutogradContext *ctx, const Tensor &logits0, const Tensor &target0, int64_t ignore)
    {
        const Tensor logits = dense(logits0), target = target0.contiguous();
        const c10::OptionalDeviceGuard guard(logits.device());
        const int64_t rows = logits.size(0);
        Tensor loss = at::empty({}, logits.options().dtype(at::kFloat)), scratch = at::empty({2 * rows + 1}, loss.options());
        check(rdb_cross_entropy_fwd(loss.data_ptr<float>(), scratch.data_ptr<float>(), logits.data_ptr(), target.data_ptr<int64_t>(), rows, logits.size(1), ignore,
                                    stream_of(logits)),
              "rdb_cross_entropy_fwd");
        ctx->save_for_backward({logits0, target, scratch});
        ctx->saved_data["m"] = std::vector<int64_t>{rows, logits.size(1), ignore};
        return loss;
    }
    static variable_list backward(AutogradContext *ctx, const variable_list &grads)
    {
        const auto saved = ctx->get_saved_variables();
        const auto m = ctx->saved_data["m"].toIntVector();   // rows, classes, ignored label
        constexpr const char *who = "cross_entropy (backward)";
        restored(who, saved[0], grads[0], {m[0], m[1]});
        restored_values(who, saved[1], grads[0], at::kLong, m[0]);
        if (at::GradMode::is_enabled()) {
            const auto loss = [&](const variable_list &in) {
                return variable_list{at::cross_entropy_loss(in[0].to(at::kFloat), saved[1], {}, at::Reduction::Mean, m[2])};
            };
            return {stock_gradient(loss, {saved[0]}, {grads[0]})[0], Tensor(), Tensor()};
        }
        const Tensor logits = dense(saved[0]), dloss = grads[0].to(at::kFloat).contiguous();
        restored_values(who, logits, dloss, at::kBFloat16, m[0] * m[1]);
        restored_values(who, saved[2], dloss, at::kFloat, 2 * m[0] + 1);
        const c10::OptionalDeviceGuard guard(logits.device());
        Tensor d = at::empty_like(logits);
        check(rdb_cross_entropy_bwd(d.data_ptr(), logits.data_ptr(), saved[1].data_ptr<int64_t>(), saved[2].data_ptr<float>(), dloss.data_ptr<float>(),
                                    m[0], m[1], m[2], stream_of(logits)),
              "rdb_cross_entropy_bwd");
        return {d, Tensor(), Tensor()};
    }
};

// qkv (B, T, 3 * heads * 64) -> causal self-attention with normalised, rotated q and k (B, T, heads * 64)
class CausalAttention : public Function<CausalAttention> {
  public:
    static Tensor forward(AutogradContext *ctx, const Tensor &qkv0, const Tensor &inv_freq0, int64_t heads, double eps)
    {
        const Tensor qkv = dense(qkv0), inv_freq = native(inv_freq0);
        const c10::OptionalDeviceGuard guard(qkv.device());
        const int64_t B = qkv.size(0), T = qkv.size(1);
        Tensor y = at::empty({B, T, heads * 64}, qkv.options()), q = at::empty({B * heads, T, 64}, qkv.options()), k = at::empty_like(q);
        Tensor scratch = at::empty({rdb_causal_attention_scratch_floats(B, T, heads)}, qkv.options().dtype(at::kFloat));
        check(rdb_causal_attention_fwd(y.data_ptr(), q.data_ptr(), k.data_ptr(), scratch.data_ptr<float>(), qkv.data_ptr(), inv_freq.data_ptr(),
                                       code(inv_freq.scalar_type()), B, T, heads, (float)eps, stream_of(qkv)),
              "rdb_causal_attention_fwd");
        ctx->save_for_backward({qkv, y, q, k, scratch});
        ctx->saved_data["heads"] = heads;
        ctx->saved_data["eps"] = eps;
        return y;
    }
    static variable_list backward(AutogradContext *ctx, const variable_list &grads)
    {
        const auto saved = ctx->get_saved_variables();
        return {once_differentiable("causal_attention", gradient(ctx, saved, grads[0]), grads[0], {0}), Tensor(), Tensor(), Tensor()};
    }
    static Tensor gradient(AutogradContext *ctx, const variable_list &saved, const Tensor &grad)
    {
        const at::AutoGradMode no_grad(false);
        const Tensor &qkv = saved[0], dy = dense(grad);
        constexpr const char *who = "causal_attention (backward)";
        const int64_t B = dy.size(0), T = dy.size(1), heads = ctx->saved_data["heads"].toInt();
        restored(who, restored_values(who, qkv, dy, at::kBFloat16, 3 * dy.numel()), dy, {B, T, 3 * heads * 64});
        for (int i = 1; i < 4; ++i) restored_values(who, saved[i], dy, at::kBFloat16, dy.numel());
        restored_values(who, saved[4], dy, at::kFloat, rdb_causal_attention_scratch_floats(B, T, heads));
        const c10::OptionalDeviceGuard guard(qkv.device());
        Tensor d = at::empty_like(qkv);
        check(rdb_causal_attention_bwd(d.data_ptr(), dy.data_ptr(), saved[1].data_ptr(), saved[2].data_ptr(), saved[3].data_ptr(), saved[4].data_ptr<float>(),
                                       qkv.data_ptr(), B, T, heads, (float)ctx->saved_data["eps"].toDouble(),
                                       stream_of(qkv)),
              "rdb_causal_attention_bwd");
        return d;
    }
};

// The sizes the descriptor states are those of the tensors: the library is told in_f and out_f and reads that far.
void check_sizes(const char *who, const Tensor &x, const Tensor &c, const Layer &l, const OptTensor &scale, const Bias &b)
{
    auto wrong = [&](const char *what, const Tensor &t) {
        std::string sizes;
        for (int64_t n : t.sizes()) sizes += (sizes.empty() ? "" : ", ") + std::to_string(n);
        fail(PyExc_RuntimeError, std::string(who) + ": a layer " + std::to_string(l.in_f) + " -> " + std::to_string(l.out_f) + " cannot take " + what + " of shape (" +
                                     sizes + ")");
    };
    if (x.dim() < 1 || x.size(-1) != l.in_f) wrong("an input", x);
    if (c.dim() != 1 && c.dim() != 2) wrong("coefficients", c);
    if (scale && scale->numel() < 1) wrong("a scale", *scale);
    if (b.coef && (b.seed < 0 ? b.coef->numel() != l.out_f : b.coef->dim() != 1)) wrong(b.seed < 0 ? "a bias" : "bias coefficients", *b.coef);
    if (b.scale && b.scale->numel() < 1) wrong("a bias scale", *b.scale);
}

// ----------------------------------------------------------------------------------------------- Python methods
// They return None for requests that are not to go past the dispatcher (past_dispatcher).
struct BadArgument {};

const Tensor &tensor_arg(PyObject *o)
{
    if (!THPVariable_Check(o)) {
        PyErr_SetString(PyExc_TypeError, "expected a tensor");
        throw BadArgument();
    }
    return THPVariable_Unpack(o);
}
OptTensor opt_arg(PyObject *o) { return o == Py_None ? OptTensor() : OptTensor(tensor_arg(o)); }
int64_t int_arg(PyObject *o)
{
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw BadArgument();
    return v;
}
uint32_t seed_arg(PyObject *o)
{
    const int64_t v = int_arg(o);
    if (v < 0 || v >= (1ll << 32)) {
        PyErr_Format(PyExc_ValueError, "seed must fit in 32 unsigned bits, got %lld", (long long)v);
        throw BadArgument();
    }
    return (uint32_t)v;
}
void count_args(Py_ssize_t n, Py_ssize_t want)
{
    if (n == want) return;
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
    throw BadArgument();
}
bool wants_grad(const OptTensor &t) { return t && t->requires_grad(); }

template <typename F> PyObject *guarded(F f)
{
    try {
        return f();
    } catch (const BadArgument &) {
        return nullptr;
    } catch (python_error &e) {
        e.restore();
        return nullptr;
    } catch (const std::exception &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

// takes_projected(x, coefs, in_f, out_f, sO, sI, scale_bias, bias): whether ops.linear runs the projected form
PyObject *py_takes_projected(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        count_args(n, 8);
        const Tensor &x = tensor_arg(a[0]), &c = tensor_arg(a[1]);
        const Layer l{int_arg(a[2]), int_arg(a[3]), int_arg(a[4]), int_arg(a[5]), 0};
        bool yes = c.dim() == 2 && c.size(0) == l.out_f && l.sO == l.in_f && l.sI == 1 && x.is_cuda() && x.dim() == 2 && readable(x.scalar_type()) &&
                   c.scalar_type() == x.scalar_type();
        if (yes && a[6] != Py_None) yes = x.scalar_type() == at::kBFloat16 && l.in_f % 8 == 0 && l.out_f % 8 == 0 && tensor_arg(a[6]).numel() == 1;
        if (yes && a[7] != Py_None) yes = tensor_arg(a[7]).scalar_type() == x.scalar_type();
        if (yes) {
            const rdb_linear_desc d = desc(x, l, c);
            yes = rdb_linear_projection_preferred(&d) != 0;
        }
        return PyBool_FromLong(yes);
    });
}

// A bias is passed as three arguments: a dense vector, None, -1; or a pseudorandom vector's coefficients, scale (or None), seed.
Bias bias_arg(PyObject *const *a)
{
    Bias b{opt_arg(a[0]), opt_arg(a[1]), int_arg(a[2])};
    if (b.seed >= (1ll << 32)) {
        PyErr_SetString(PyExc_ValueError, "the bias's seed must fit in 32 unsigned bits");
        throw BadArgument();
    }
    return b;
}
bool wants_grad(const Bias &b) { return wants_grad(b.coef) || wants_grad(b.scale); }

// linear_projected(x, coefs, in_f, out_f, seed, bias, bias_scale, bias_seed, scale_bias)
PyObject *py_linear_projected(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        count_args(n, 9);
        const Tensor &x = tensor_arg(a[0]), &c = tensor_arg(a[1]);
        const Layer l{int_arg(a[2]), int_arg(a[3]), int_arg(a[2]), 1, seed_arg(a[4])};
        const Bias b = bias_arg(a + 5);
        const OptTensor sb = opt_arg(a[8]);
        same_device("linear_fwd", x, {&c, address(b.coef), address(b.scale), address(sb)});
        check_sizes("linear_fwd", x, c, l, sb, b);
        if (!past_dispatcher({&x, &c, address(b.coef), address(b.scale), address(sb)})) Py_RETURN_NONE;
        // without a backward pass to come there is no state to keep: the one-call forward
        if (!at::GradMode::is_enabled() || !(x.requires_grad() || c.requires_grad() || wants_grad(b) || wants_grad(sb)))
            return THPVariable_Wrap(linear_fwd(x, c, l, sb, b));
        return THPVariable_Wrap(ProjectedLinear::apply(x, c, b.coef, b.scale, b.seed, sb, l, false, (const Tensor *)nullptr, (Tensor *)nullptr));
    });
}

// relu_square_linear(x, coefs, in_f, out_f, seed): linear_projected of relu(x)^2, for a gradient of x to come; None without one: the node would save nothing of the
// backward pass, and keep x for it
PyObject *py_relu_square_linear(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        count_args(n, 5);
        const Tensor &x = tensor_arg(a[0]), &c = tensor_arg(a[1]);
        const Layer l{int_arg(a[2]), int_arg(a[3]), int_arg(a[2]), 1, seed_arg(a[4])};
        same_device("linear_fwd", x, {&c});
        check_sizes("linear_fwd", x, c, l, OptTensor(), Bias{});
        if (!past_dispatcher({&x, &c}) || !at::GradMode::is_enabled() || !x.requires_grad()) Py_RETURN_NONE;
        need_bf16("relu_square_linear", x);
        return THPVariable_Wrap(ProjectedLinear::apply(x, c, OptTensor(), OptTensor(), -1, OptTensor(), l, true, (const Tensor *)nullptr, (Tensor *)nullptr));
    });
}

// squared_relu_mlp(x, coefs 1, coefs 2, in_f, hidden, out_f, seed 1, seed 2): linear_projected, relu(.)^2 and linear_projected, each a node of its own but for the
// activation, which is the second one's and leaves the first one's kernel beside its input; None without a backward pass to come
PyObject *py_squared_relu_mlp(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        count_args(n, 8);
        const Tensor &x = tensor_arg(a[0]), &c1 = tensor_arg(a[1]), &c2 = tensor_arg(a[2]);
        const int64_t in_f = int_arg(a[3]), hidden = int_arg(a[4]), out_f = int_arg(a[5]);
        const Layer l1{in_f, hidden, in_f, 1, seed_arg(a[6])}, l2{hidden, out_f, hidden, 1, seed_arg(a[7])};
        same_device("linear_fwd", x, {&c1, &c2});
        check_sizes("linear_fwd", x, c1, l1, OptTensor(), Bias{});
        if (!past_dispatcher({&x, &c1, &c2}) || !at::GradMode::is_enabled() || !(x.requires_grad() || c1.requires_grad())) Py_RETURN_NONE;
        need_bf16("squared_relu_mlp", x);
        Tensor square;
        const Tensor h = ProjectedLinear::apply(x, c1, OptTensor(), OptTensor(), -1, OptTensor(), l1, false, (const Tensor *)nullptr, &square);
        check_sizes("linear_fwd", h, c2, l2, OptTensor(), Bias{});
        return THPVariable_Wrap(ProjectedLinear::apply(h, c2, OptTensor(), OptTensor(), -1, OptTensor(), l2, true, (const Tensor *)&square, (Tensor *)nullptr));
    });
}

// linear_one_call(x, coefs, in_f, out_f, sO, sI, seed, scale_bias, bias, bias_scale, bias_seed)
PyObject *py_linear_one_call(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        count_args(n, 11);
        const Tensor &x = tensor_arg(a[0]), &c = tensor_arg(a[1]);
        const Layer l{int_arg(a[2]), int_arg(a[3]), int_arg(a[4]), int_arg(a[5]), seed_arg(a[6])};
        const OptTensor sb = opt_arg(a[7]);
        const Bias b = bias_arg(a + 8);
        same_device("linear_fwd", x, {&c, address(b.coef), address(b.scale), address(sb)});
        check_sizes("linear_fwd", x, c, l, sb, b);
        if (!past_dispatcher({&x, &c, address(b.coef), address(b.scale), address(sb)})) Py_RETURN_NONE;
        if (!at::GradMode::is_enabled() || !(x.requires_grad() || c.requires_grad() || wants_grad(b) || wants_grad(sb)))
            return THPVariable_Wrap(linear_fwd(x, c, l, sb, b));
        return THPVariable_Wrap(OneCallLinear::apply(x, c, sb, b.coef, b.scale, b.seed, l));
    });
}

// linear_vector(x, coef, in_f, out_f, seed, scale_bias, bias, bias_scale, bias_seed): x (..., in_f)
PyObject *py_linear_vector(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        count_args(n, 9);
        const Tensor &x = tensor_arg(a[0]), &c = tensor_arg(a[1]);
        const Layer l{int_arg(a[2]), int_arg(a[3]), int_arg(a[2]), 1, seed_arg(a[4])};
        const OptTensor sb = opt_arg(a[5]);
        const Bias b = bias_arg(a + 6);
        same_device("linear_vector", x, {&c, address(b.coef), address(b.scale), address(sb)});
        check_sizes("linear_vector", x, c, l, sb, b);
        if (!past_dispatcher({&x, &c, address(b.coef), address(b.scale), address(sb)})) Py_RETURN_NONE;
        if (!at::GradMode::is_enabled() || !(x.requires_grad() || c.requires_grad() || wants_grad(b) || wants_grad(sb)))
            return THPVariable_Wrap(VectorLinear::forward(nullptr, x, c, sb, b.coef, b.scale, b.seed, l));
        return THPVariable_Wrap(VectorLinear::apply(x, c, sb, b.coef, b.scale, b.seed, l));
    });
}

// embed_rows(idx, coef, rowsize, seed)
PyObject *py_embed_rows(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        count_args(n, 4);
        const Tensor &idx = tensor_arg(a[0]), &c = tensor_arg(a[1]);
        const int64_t rowsize = int_arg(a[2]), seed = seed_arg(a[3]);
        same_device("embed_fwd", idx, {&c});
        if (c._fw_grad(0).defined()) fail(PyExc_NotImplementedError, "embed_fwd has no forward-mode derivative");   // the operator would drop it
        if (!past_dispatcher({&idx, &c})) Py_RETURN_NONE;
        if (!at::GradMode::is_enabled() || !c.requires_grad()) return THPVariable_Wrap(EmbedRows::forward(nullptr, idx, c, rowsize, seed));
        return THPVariable_Wrap(EmbedRows::apply(idx, c, rowsize, seed));
    });
}

double float_arg(PyObject *o)
{
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw BadArgument();
    return v;
}

// rms_norm(x, eps)
PyObject *py_rms_norm(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        count_args(n, 2);
        const Tensor &x = tensor_arg(a[0]);
        if (!past_dispatcher({&x})) Py_RETURN_NONE;
        need_bf16("rms_norm", x);
        return THPVariable_Wrap(RmsNorm::apply(x, float_arg(a[1])));
    });
}

// add_rms_norm(x, delta, eps) -> (x + delta, its normalisation)
PyObject *py_add_rms_norm(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        count_args(n, 3);
        const Tensor &x = tensor_arg(a[0]), &delta = tensor_arg(a[1]);
        if (!past_dispatcher({&x, &delta})) Py_RETURN_NONE;
        need_bf16("add_rms_norm", x);
        need_bf16("add_rms_norm", delta);
        same_device("add_rms_norm", x, {&delta});
        if (x.sizes() != delta.sizes()) fail(PyExc_ValueError, "add_rms_norm needs tensors of one shape");
        const auto r = AddRmsNorm::apply(x, delta, float_arg(a[2]));
        PyObject *s = THPVariable_Wrap(r[0]), *y = THPVariable_Wrap(r[1]);
        return Py_BuildValue("NN", s, y);
    });
}

PyObject *py_relu_square(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        count_args(n, 1);
        const Tensor &x = tensor_arg(a[0]);
        if (!past_dispatcher({&x})) Py_RETURN_NONE;
        need_bf16("relu_square", x);
        return THPVariable_Wrap(ReluSquare::apply(x));
    });
}

// embedding(weight, idx): rows of a dense bf16 table; None without a backward pass to come, or for sizes that the stock operator is faster at
PyObject *py_embedding(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        count_args(n, 2);
        const Tensor &w = tensor_arg(a[0]), &idx = tensor_arg(a[1]);
        if (!past_dispatcher({&w, &idx}) || !at::GradMode::is_enabled() || !w.requires_grad()) Py_RETURN_NONE;
        need_bf16("embedding", w);
        same_device("embedding", w, {&idx});
        if (w.dim() != 2 || !idx.dim() || (idx.scalar_type() != at::kLong && idx.scalar_type() != at::kInt) || !rdb_embedding_bwd_takes(idx.numel(), w.size(0), w.size(1)))
            Py_RETURN_NONE;
        return THPVariable_Wrap(EmbedDense::apply(w, idx));
    });
}

// cross_entropy(logits, target, ignore_index): mean over the rows that count
PyObject *py_cross_entropy(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        count_args(n, 3);
        const Tensor &x = tensor_arg(a[0]), &t = tensor_arg(a[1]);
        if (!past_dispatcher({&x, &t})) Py_RETURN_NONE;
        need_bf16("cross_entropy", x);
        if (x.dim() != 2 || t.dim() != 1 || t.size(0) != x.size(0) || t.scalar_type() != at::kLong || t.device() != x.device())
            fail(PyExc_ValueError, "cross_entropy needs logits (rows, classes) and int64 targets (rows) on one device");
        return THPVariable_Wrap(CrossEntropy::apply(x, t, int_arg(a[2])));
    });
}

// causal_attention(qkv, inv_freq, heads, eps)
PyObject *py_causal_attention(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        count_args(n, 4);
        const Tensor &qkv = tensor_arg(a[0]), &f = tensor_arg(a[1]);
        const int64_t heads = int_arg(a[2]);
        if (!past_dispatcher({&qkv, &f})) Py_RETURN_NONE;
        need_bf16("causal_attention", qkv);
        if (qkv.dim() != 3 || qkv.size(2) != 3 * heads * 64 || f.numel() != 32 || f.device() != qkv.device())
            fail(PyExc_ValueError, "causal_attention needs qkv (B, T, 3 * heads * 64) and 32 frequencies on one device");
        return THPVariable_Wrap(CausalAttention::apply(qkv, f, heads, float_arg(a[3])));
    });
}

// once_differentiable(grad, dy, input, input): for the functions in Python, called from their backward passes (negative: no input)
PyObject *py_once_differentiable(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        count_args(n, 4);
        return THPVariable_Wrap(once_differentiable("linear", tensor_arg(a[0]), tensor_arg(a[1]), {(int)int_arg(a[2]), (int)int_arg(a[3])}));
    });
}

// set_hooks(error class, tick)
PyObject *py_set_hooks(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        count_args(n, 2);
        Py_INCREF(a[0]);
        Py_INCREF(a[1]);
        Py_XSETREF(g_error_class, a[0]);
        Py_XSETREF(g_tick, a[1]);
        Py_RETURN_NONE;
    });
}

#define RDB_METHOD(name) {#name, (PyCFunction)(void (*)(void))py_##name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {RDB_METHOD(takes_projected),   RDB_METHOD(linear_projected), RDB_METHOD(linear_one_call), RDB_METHOD(relu_square_linear), RDB_METHOD(squared_relu_mlp),
                         RDB_METHOD(linear_vector),     RDB_METHOD(embed_rows),       RDB_METHOD(set_hooks),
                         RDB_METHOD(rms_norm),          RDB_METHOD(add_rms_norm),     RDB_METHOD(relu_square),
                         RDB_METHOD(embedding),
                         RDB_METHOD(cross_entropy),     RDB_METHOD(causal_attention), RDB_METHOD(once_differentiable),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_rdb_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// The name under which a function's node shows up as grad_fn in Python.
template <typename F> static void name_node(const char *name)
{
    static PyTypeObject type = {PyVarObject_HEAD_INIT(nullptr, 0)};
    torch::autograd::_initFunctionPyTypeObject(type, name, nullptr, nullptr);
    torch::autograd::registerCppFunction(typeid(torch::autograd::CppNode<F>), &type);
}

PyMODINIT_FUNC PyInit__rdb_torch(void)
{
    name_node<OneCallLinear>("OneCallLinearBackward");
    name_node<ProjectedLinear>("ProjectedLinearBackward");
    name_node<VectorLinear>("VectorLinearBackward");
    name_node<EmbedRows>("EmbedRowsBackward");
    name_node<CoefValues>("CoefValuesBackward");
    name_node<CoefGrads>("CoefGradsBackward");
    name_node<RmsNorm>("RmsNormBackward");
    name_node<AddRmsNorm>("AddRmsNormBackward");
    name_node<ReluSquare>("ReluSquareBackward");
    name_node<CrossEntropy>("CrossEntropyBackward");
    name_node<CausalAttention>("CausalAttentionBackward");
    return PyModule_Create(&module);
}
