// The host side of the layers, native: what bgemm_linear.py and lowbit_kernel.py would do on every call in Python (argument
// checks, allocation, the stream, the calls into the C ABI, autograd bookkeeping).  A small layer's kernels take a few
// microseconds, less than those steps cost in Python.  Host code only: plain CPython functions on torch's C++ API, linked against
// libbgemm_mi355x.so beside it.  This part: training; torch_infer.cpp: inference and attention.  Functions that find a case they do not
// take return None, and the caller goes the Python way.
#include "torch_common.h"

#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>

#include <utility>
#include <vector>

namespace {

using namespace bgemm_native;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

// The interpreter's pending exception as a C++ one that outlives the lock and the thread it was raised on.
[[noreturn]] void throw_pending()
{
    python_error e;
    e.persist();
    throw e;
}

// A node of the layers: its inputs are four tensors and perhaps a bias, whose gradient is the upstream one (the engine adds it up).
struct LayerNode : public torch::autograd::Node {
    bool has_bias, released_by_bias = false;

    // The bias's gradient alone needs nothing that is kept, and giving it takes nothing away: the addition of the bias is the last of
    // the separate operations, and the only one that would run.
    bool bias_alone()
    {
        bool alone = has_bias;
        for (int i = 0; i < 4; i++) alone &= !task_should_compute_output(i);
        std::lock_guard<std::mutex> lock(mutex_);
        released_by_bias = alone;
        return alone;
    }
    // Whether release_variables() (under its lock) follows such a pass.
    bool nothing_to_release() { return std::exchange(released_by_bias, false); }

    // No gradient from above: zeros for the inputs `which`, as the binary product's Function among the separate operations gives them.
    variable_list zeros_for(std::initializer_list<size_t> which)
    {
        variable_list r(num_outputs());
        for (const size_t i : which)
            if (task_should_compute_output(i)) r[i] = next_edge(i).function->input_metadata(next_edge(i).input_nr).zeros_like();
        return r;
    }

    // Whether torch has to see the operations of this gradient: it will itself be differentiated (in either mode), or it is no plain
    // tensor (a batch of vmap's), or something listens.
    static bool by_operations(const Tensor& grad) { return c10::GradMode::is_enabled() || !is_memory(grad) || has_tangent(grad) || is_watched(); }

    // fn(the four gradients wanted, tensors .., number) of bgemm_linear.py: a tuple of the four gradients.  Holds the interpreter's lock.
    variable_list python_grads(const char* fn, std::initializer_list<Tensor> tensors, const double number)
    {
        PyObject* const module = PyImport_ImportModule("bgemm_linear");
        if (!module) throw_pending();
        PyObject* const f = PyObject_GetAttrString(module, fn);
        Py_DECREF(module);
        if (!f) throw_pending();
        PyObject* const args = PyTuple_New(tensors.size() + 2), * const need = PyTuple_New(4);
        for (int i = 0; i < 4; i++) PyTuple_SET_ITEM(need, i, PyBool_FromLong(task_should_compute_output(i)));
        PyTuple_SET_ITEM(args, 0, need);
        int at = 1;
        for (const Tensor& t : tensors) PyTuple_SET_ITEM(args, at++, THPVariable_Wrap(t));
        PyTuple_SET_ITEM(args, at, PyFloat_FromDouble(number));
        PyObject* const got = PyObject_CallObject(f, args);
        Py_DECREF(f); Py_DECREF(args);
        if (!got) throw_pending();
        variable_list r;
        for (int i = 0; i < 4; i++) r.push_back(tensor_or_none(PyTuple_GET_ITEM(got, i)));
        Py_DECREF(got);
        if (has_bias) r.push_back(task_should_compute_output(4) ? *(tensors.end() - 1) : Tensor());
        return r;
    }
};

// A fresh tensor that stands for a value of the forward pass in operations whose graph goes on through the input it came from.
Tensor stand_in(const Tensor& value, const torch::autograd::Edge& edge)
{
    const Tensor t = value.detach();
    if (edge.is_valid()) torch::autograd::impl::set_gradient_edge(t, edge);
    return t;
}

// Numbers whose sign bits and zeros are those of a packed operand: [rows, K] of +-1 and +-0.
Tensor signs_of(const int32_t* sign, const int32_t* nonzero, const int64_t rows, const int64_t K, const at::TensorOptions& like)
{
    const c10::NoGradGuard no_grad;
    const auto ints = like.dtype(at::kInt);
    const Tensor shifts = at::arange(31, -1, -1, ints);
    auto bits = [&](const int32_t* tiled) {
        const Tensor words = at::empty({rows, (K + 31) / 32}, ints);
        check(bgemm_logical_from_tiled(tiled, rows, K, (uint32_t*)words.data_ptr(), stream_of(words)));
        return words.unsqueeze(-1).bitwise_right_shift(shifts).bitwise_and(1).reshape({rows, -1}).narrow(1, 0, K).to(like.dtype());
    };
    return bits(nonzero) * (1 - 2 * bits(sign));
}

// ---- the scaled binary Linear as one autograd node -----------------------------------------------------------------------------
// y = fn(x - zpa, w - zpw) * sw * sa (+ bias) (tests/python/bgemm_linear.py:479-484): two launches forward, two backward.  What is kept
// for the backward pass is bits, the sign and nonzero planes of both operands; for Bi-Real half(x - zpa); and the scales, as the two
// products by them keep them: themselves (changed by an in-place operation they are refused) where what they multiply has a
// gradient, and the first product's values for the gradient of sa.
struct LinearNode : public LayerNode {
    int64_t N, K, M, words_x, words_w;
    bool bireal, operands_recorded, sa_kept;        // x or w has a gradient; sa is kept
    Tensor planes;                                  // [x sign | x nonzero | w sign | w nonzero | sw then]
    Tensor centred;                                 // Bi-Real with a gradient of x: half(x - zpa)
    SavedVariable sw_, sa_;
    std::vector<int64_t> x_shape, sa_shape;
    at::ScalarType type;

    std::string name() const override { return "ScaledBinaryLinearBackward"; }

    void release_variables() override
    {
        std::lock_guard<std::mutex> lock(mutex_);
        if (nothing_to_release()) return;
        planes.reset(); centred.reset();
        sw_.reset_data(); sa_.reset_data();
    }

    variable_list apply(variable_list&& grads) override
    {
        if (bias_alone()) return {Tensor(), Tensor(), Tensor(), Tensor(), grads[0]};
        const bool want_x = task_should_compute_output(0), want_w = task_should_compute_output(1), want_sw = task_should_compute_output(2),
                   want_sa = task_should_compute_output(3), want_b = has_bias && task_should_compute_output(4);
        std::unique_lock<std::mutex> lock(mutex_);
        TORCH_CHECK(planes.defined(), torch::autograd::ERR_BACKWARD_TWICE);
        if (!grads[0].defined()) return zeros_for({0, 1});
        const c10::OptionalDeviceGuard guard(planes.device());
        const int32_t* const p = planes.data_ptr<int32_t>();
        const int32_t* const pw = p + 2 * words_x;
        const Tensor then = planes.narrow(0, 2 * (words_x + words_w), planes.numel() - 2 * (words_x + words_w)).view(type).narrow(0, 0, M);
        Tensor sw = then, sa = then;                // (sa: not read for what is wanted where it is not kept)
        if (sa_kept && (want_x || want_w || want_sw || want_sa)) sa = sa_.unpack();
        if (operands_recorded && (want_x || want_w || want_sw)) sw = sw_.unpack();
        if (by_operations(grads[0])) {
            const auto like = planes.options().dtype(type);
            const Tensor x = stand_in((centred.defined() ? centred.to(type) : signs_of(p, p + words_x, N, K, like)).view(x_shape), next_edge(0));
            const Tensor w = stand_in(signs_of(pw, pw + words_w, M, K, like), next_edge(1));
            const Tensor sw_then = stand_in(then.clone(), next_edge(2));
            lock.unlock();                          // (whoever waits for the lock may hold the interpreter's)
            pybind11::gil_scoped_acquire gil;
            return python_grads("_scaled_linear_grads", {x, w, sw, sw_then, sa, grads[0]}, bireal ? 1. : 0.);
        }
        const Tensor g = grads[0].contiguous();
        Tensor gx, gw, gb, gsw, gsa;
        if (want_x) gx = at::empty(x_shape, g.options());
        if (want_w) gw = at::empty({M, K}, g.options());
        if (want_sw) gsw = at::empty({M}, g.options());
        if (want_sa) gsa = at::empty(sa_shape, g.options());
        if (want_b) gb = at::empty({M}, g.options());
        const size_t bytes = bgemm_linear_backward_workspace_bytes(N, M, K, want_x, want_w);
        const Tensor ws = at::empty({(int64_t)bytes}, g.options().dtype(at::kByte));
        check(bgemm_linear_backward(pw, pw + words_w, p, p + words_x, g.data_ptr(), src_type(g), N, M, K, sw.data_ptr(), sa.data_ptr(), then.data_ptr(),
                                    data_or_null(centred), data_or_null(gx), data_or_null(gw), data_or_null(gb), data_or_null(gsw), data_or_null(gsa),
                                    ws.data_ptr(), bytes, stream_of(g)));
        variable_list r = {gx, gw, gsw, gsa};
        if (has_bias) r.push_back(gb);
        return r;
    }
};

// torch.Tensor or Parameter themselves, the bias (argument 4) or None, and nothing that listens.
bool plain_call(PyObject* const* args, const int tensors)
{
    for (int i = 0; i < tensors; i++)
        if (!THPVariable_CheckExact(args[i]) && !(i == 4 && args[i] == Py_None)) return false;
    // (saved-tensor hooks - checkpointing, offloading - get the tensors the separate operations keep: bit planes mean nothing to them)
    return !is_watched() && !at::SavedTensorDefaultHooks::get_hooks().has_value();
}

bool one_scalar(const Tensor& t) { return t.numel() == 1 && t.dim() <= 1; }

// Whether a recorded forward is the one-node form: the module's own arithmetic on one device and in one type, zero points that
// are no parameters, and sizes the kernels take.
bool one_node(const Tensor& x, const Tensor& w, const Tensor& sw, const Tensor& sa, const Tensor& bias, const Tensor& zpa, const Tensor& zpw)
{
    if (!c10::GradMode::is_enabled() || !x.is_cuda() || !is_param_type(w.scalar_type()) || w.dim() != 2 || x.dim() < 1 || x.numel() == 0) return false;
    const int64_t M = w.size(0), K = w.size(1);
    if (M < 2 || M > (1 << 20) || K >= (1 << 24) || x.size(-1) != K || x.numel() / K > (1 << 20) ||
        !bgemm_linear_backward_workspace_bytes(x.numel() / K, M, K, x.requires_grad(), w.requires_grad()))
        return false;
    for (const Tensor* t : {&x, &w, &sw, &sa, &zpa, &zpw})
        if (t->scalar_type() != w.scalar_type() || t->device() != x.device() || !is_memory(*t) || has_tangent(*t)) return false;
    if (!one_scalar(sa) || !one_scalar(zpa) || !one_scalar(zpw) || zpa.requires_grad() || zpw.requires_grad()) return false;
    if (sw.dim() != 1 || sw.size(0) != M || !sw.is_contiguous()) return false;
    // (a single vector and a bias: the addition refuses them)
    return !bias.defined() || (x.dim() > 1 && is_memory(bias) && !has_tangent(bias) && bias.scalar_type() == w.scalar_type() && bias.device() == x.device() && bias.dim() == 1 && bias.size(0) == M && bias.is_contiguous());
}

// linear_train(x, weight, sw, sa, bias | None, zpa, zpw, bireal) -> y, or None where the separate operations have to run
PyObject* linear_train(PyObject*, PyObject* const* args, const Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n == 8, "linear_train takes 8 arguments");
    if (!plain_call(args, 7)) Py_RETURN_NONE;
    const Tensor &x = tensor_at(args[0]), &w = tensor_at(args[1]), &sw = tensor_at(args[2]), &sa = tensor_at(args[3]);
    const Tensor bias = tensor_or_none(args[4]);
    const Tensor &zpa = tensor_at(args[5]), &zpw = tensor_at(args[6]);
    if (!one_node(x, w, sw, sa, bias, zpa, zpw)) Py_RETURN_NONE;
    const bool bireal = PyObject_IsTrue(args[7]);
    Tensor out;
    {
        const WithoutGil no_gil;
        std::shared_ptr<LinearNode> node;
        bool recorded = bias.defined() && bias.requires_grad();
        for (const Tensor* t : {&x, &w, &sw, &sa}) recorded |= t->requires_grad();
        const int64_t K = w.size(1), M = w.size(0), N = x.numel() / K;
        const int64_t words_x = bgemm_tiled_words(N, K), words_w = bgemm_tiled_words(M, K);
        Tensor planes, centred;
        {
            const c10::NoGradGuard no_grad;
            const c10::OptionalDeviceGuard guard(x.device());
            const Rows x2 = rows_2d(x), w2 = rows_2d(w);
            planes = at::empty({2 * (words_x + words_w) + M}, x.options().dtype(at::kInt));
            if (bireal && x.requires_grad()) centred = at::empty({N, K}, x.options().dtype(at::kHalf));
            std::vector<int64_t> shape = x.sizes().vec();
            shape.back() = M;
            out = at::empty(shape, x.options());
            int32_t* const p = planes.data_ptr<int32_t>();
            int32_t* const pw = p + 2 * words_x;
            check(bgemm_linear_train_forward(x2.t.data_ptr(), x2.ld, zpa.data_ptr(), w2.t.data_ptr(), w2.ld, zpw.data_ptr(), src_type(x), N, M, K,
                                             sw.data_ptr(), sa.data_ptr(), data_or_null(bias), p, p + words_x, pw, pw + words_w,
                                             recorded ? pw + 2 * words_w : nullptr, data_or_null(centred), out.data_ptr(), stream_of(x)));
        }
        if (recorded) {
            node = std::shared_ptr<LinearNode>(new LinearNode(), torch::autograd::deleteNode);
            node->N = N; node->K = K; node->M = M; node->words_x = words_x; node->words_w = words_w;
            node->bireal = bireal; node->has_bias = bias.defined();
            node->planes = planes; node->centred = centred;
            node->x_shape = x.sizes().vec(); node->sa_shape = sa.sizes().vec(); node->type = x.scalar_type();
            node->operands_recorded = x.requires_grad() || w.requires_grad();
            node->sa_kept = node->operands_recorded || sw.requires_grad();
            if (node->operands_recorded) node->sw_ = SavedVariable(sw, false);
            if (node->sa_kept) node->sa_ = SavedVariable(sa, false);
            if (bias.defined()) node->set_next_edges(torch::autograd::collect_next_edges(x, w, sw, sa, bias));
            else node->set_next_edges(torch::autograd::collect_next_edges(x, w, sw, sa));
            torch::autograd::set_history(out, node);
        }
    }
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// ---- the learned-scale layer as one autograd node ----------------------------------------------------------------------------------
// (half(acc) * sa) * sw (+ bias) of xs = (x - mean(x)) / sa and ws = w - mean(w) (tests/python/bgemm_linear.py:350-457, :538-564): three
// launches forward, two backward.  Kept: xs and ws as the separate operations keep them, so that nothing done to the operands or
// scales between the passes matters, and their sign and nonzero planes.
struct ElasticNode : public LayerNode {
    int64_t N, K, M, words_x, words_w;
    double grad_scale;
    Tensor planes;                                  // [x sign | x nonzero | w sign | w nonzero | scratch | xs | ws]
    std::vector<int64_t> x_shape;

    // xs and ws in the same memory as the planes: each allocation is a microsecond of a small layer's step.
    int64_t xs_at() const { return 2 * (words_x + words_w) + BGEMM_ELASTIC_SCRATCH; }
    int64_t ws_at() const { return xs_at() + N * K; }

    std::string name() const override { return "ElasticBinaryLinearBackward"; }

    void release_variables() override
    {
        std::lock_guard<std::mutex> lock(mutex_);
        if (nothing_to_release()) return;
        planes.reset();
    }

    variable_list apply(variable_list&& grads) override
    {
        if (bias_alone()) return {Tensor(), Tensor(), Tensor(), Tensor(), grads[0]};
        std::unique_lock<std::mutex> lock(mutex_);
        TORCH_CHECK(planes.defined(), torch::autograd::ERR_BACKWARD_TWICE);
        if (!grads[0].defined()) return zeros_for({0, 1, 2, 3});
        if (by_operations(grads[0])) {
            const Tensor x = planes.narrow(0, xs_at(), N * K).view(at::kFloat).view(x_shape), w = planes.narrow(0, ws_at(), M * K).view(at::kFloat).view({M, K});
            lock.unlock();                          // (whoever waits for the lock may hold the interpreter's)
            pybind11::gil_scoped_acquire gil;
            return python_grads("_elastic_grads", {x, w, grads[0]}, grad_scale);
        }
        const c10::OptionalDeviceGuard guard(planes.device());
        const bool want_x = task_should_compute_output(0), want_sa = task_should_compute_output(2);
        const bool need_x = want_x || want_sa, need_w = task_should_compute_output(1) || task_should_compute_output(3);
        const Tensor g = grads[0].contiguous();
        Tensor gx, gw, gb, gsw, gsa;
        if (need_x) gx = at::empty(x_shape, g.options());
        if (want_sa) gsa = at::empty({}, g.options());
        if (need_w) {
            gw = at::empty({M, K}, g.options());
            gsw = at::empty({M}, g.options());
        }
        if (has_bias && task_should_compute_output(4)) gb = at::empty({M}, g.options());
        const size_t bytes = bgemm_elastic_backward_workspace_bytes(N, M, K, need_x, need_w);
        const Tensor work = at::empty({(int64_t)bytes}, g.options().dtype(at::kByte));
        const int32_t* const p = planes.data_ptr<int32_t>();
        const int32_t* const pw = p + 2 * words_x;
        check(bgemm_elastic_backward(p, p + words_x, pw, pw + words_w, g.data_ptr(), p + xs_at(), p + ws_at(), (float)grad_scale, N, M, K,
                                     data_or_null(gx), data_or_null(gw), data_or_null(gb), data_or_null(gsw), data_or_null(gsa), work.data_ptr(), bytes,
                                     stream_of(g)));
        variable_list r = {want_x ? gx : Tensor(), gw, gsa, gsw};
        if (has_bias) r.push_back(gb);
        return r;
    }
};

// elastic_train(x, weight, sa, sw, bias | None, grad_scale) -> y, or None where the separate operations have to run
PyObject* elastic_train(PyObject*, PyObject* const* args, const Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n == 6, "elastic_train takes 6 arguments");
    if (!plain_call(args, 5)) Py_RETURN_NONE;
    const Tensor &x = tensor_at(args[0]), &w = tensor_at(args[1]), &sa = tensor_at(args[2]), &sw = tensor_at(args[3]);
    const Tensor bias = tensor_or_none(args[4]);
    const double grad_scale = PyFloat_AsDouble(args[5]);
    if (grad_scale == -1.0 && PyErr_Occurred()) throw python_error();
    if (!c10::GradMode::is_enabled() || !x.is_cuda() || w.dim() != 2 || x.dim() < 1 || x.numel() == 0 || sa.dim() != 0) Py_RETURN_NONE;
    const int64_t M = w.size(0), K = w.size(1), N = x.numel() / (K ? K : 1);
    if (M < 2 || M > (1 << 20) || K < 1 || K >= (1 << 24) || x.size(-1) != K || N > (1 << 20)) Py_RETURN_NONE;
    for (const Tensor* t : {&x, &w, &sa, &sw})
        if (t->scalar_type() != at::kFloat || t->device() != x.device() || !is_memory(*t) || has_tangent(*t)) Py_RETURN_NONE;
    if (!bgemm_elastic_backward_workspace_bytes(N, M, K, x.requires_grad() || sa.requires_grad(), w.requires_grad() || sw.requires_grad())) Py_RETURN_NONE;
    if (sw.dim() != 1 || sw.size(0) != M || !sw.is_contiguous()) Py_RETURN_NONE;
    if (bias.defined() && (x.dim() < 2 || !is_memory(bias) || has_tangent(bias) || bias.scalar_type() != at::kFloat || bias.device() != x.device() || bias.dim() != 1 || bias.size(0) != M || !bias.is_contiguous())) Py_RETURN_NONE;
    Tensor out;
    {
        const WithoutGil no_gil;
        bool recorded = bias.defined() && bias.requires_grad();
        for (const Tensor* t : {&x, &w, &sa, &sw}) recorded |= t->requires_grad();
        const int64_t words_x = bgemm_tiled_words(N, K), words_w = bgemm_tiled_words(M, K);
        const int64_t bits = 2 * (words_x + words_w) + BGEMM_ELASTIC_SCRATCH;
        Tensor planes;
        {
            const c10::NoGradGuard no_grad;
            const c10::OptionalDeviceGuard guard(x.device());
            const Tensor x2 = x.contiguous(), w2 = w.contiguous();
            planes = at::empty({bits + (recorded ? (N + M) * K : 0)}, x.options().dtype(at::kInt));
            std::vector<int64_t> shape = x.sizes().vec();
            shape.back() = M;
            out = at::empty(shape, x.options());
            int32_t* const p = planes.data_ptr<int32_t>();
            int32_t* const pw = p + 2 * words_x;
            check(bgemm_elastic_forward(x2.data_ptr(), w2.data_ptr(), N, M, K, sa.data_ptr(), sw.data_ptr(), data_or_null(bias), p, p + words_x,
                                        recorded ? p + bits : nullptr, pw, pw + words_w, recorded ? p + bits + N * K : nullptr, pw + 2 * words_w,
                                        out.data_ptr(), stream_of(x)));
        }
        if (recorded) {
            auto node = std::shared_ptr<ElasticNode>(new ElasticNode(), torch::autograd::deleteNode);
            node->N = N; node->K = K; node->M = M; node->words_x = words_x; node->words_w = words_w;
            node->grad_scale = grad_scale; node->has_bias = bias.defined();
            node->planes = planes;
            node->x_shape = x.sizes().vec();
            if (bias.defined()) node->set_next_edges(torch::autograd::collect_next_edges(x, w, sa, sw, bias));
            else node->set_next_edges(torch::autograd::collect_next_edges(x, w, sa, sw));
            torch::autograd::set_history(out, node);
        }
    }
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// ---- attention's products as one autograd node each ----------------------------------------------------------------------------------
// bgemm_matmul and bgemm_attn_matmul on batches of fp16 matrices (bgemm_linear.py).  Kept are the operands themselves, as the Functions
// keep them: changed in place they are refused.  As Python Functions the two took 45 of the 155 us of a step of 4 x 512 tokens, 12 heads
// of 64, half of that waiting for the interpreter's lock on the engine's thread.
struct ProductNode : public torch::autograd::Node {
    bool context;
    int64_t longest, narrow, most;
    SavedVariable x_, right_;

    std::string name() const override { return context ? "BinaryContextBackward" : "BinaryScoresBackward"; }

    void release_variables() override
    {
        std::lock_guard<std::mutex> lock(mutex_);
        x_.reset_data();
        right_.reset_data();
    }

    variable_list apply(variable_list&& grads) override
    {
        // (what has no gradient has zeros, as the Functions have it)
        if (!grads[0].defined()) grads[0] = input_metadata(0).zeros_like();
        const bool need0 = task_should_compute_output(0), need1 = task_should_compute_output(1);
        std::unique_lock<std::mutex> lock(mutex_);
        const Tensor x = x_.unpack(), right = right_.unpack();
        lock.unlock();
        const Tensor& g = grads[0];
        if (!LayerNode::by_operations(g) && g.scalar_type() == at::kHalf && !has_tangent(x) && !has_tangent(right)) {
            Tensor g0, g1;
            const bool done = context ? attention_grads(true, x, g, right, need0, need1, longest, narrow, most, g0, g1)
                                      : attention_grads(false, g, x, right.transpose(-1, -2), need0, need1, longest, narrow, most, g0, g1);
            if (done) return {g0, !context && g1.defined() ? g1.transpose(-1, -2) : g1};
        }
        pybind11::gil_scoped_acquire gil;
        PyObject* const module = PyImport_ImportModule("bgemm_linear");
        if (!module) throw_pending();
        PyObject* const f = PyObject_GetAttrString(module, context ? "_context_grads" : "_scores_grads");
        Py_DECREF(module);
        if (!f) throw_pending();
        PyObject* const args = PyTuple_New(4), * const need = PyTuple_New(2);
        PyTuple_SET_ITEM(need, 0, PyBool_FromLong(need0));
        PyTuple_SET_ITEM(need, 1, PyBool_FromLong(need1));
        PyTuple_SET_ITEM(args, 0, need);
        PyTuple_SET_ITEM(args, 1, THPVariable_Wrap(x));
        PyTuple_SET_ITEM(args, 2, THPVariable_Wrap(right));
        PyTuple_SET_ITEM(args, 3, THPVariable_Wrap(g));
        PyObject* const got = PyObject_CallObject(f, args);
        Py_DECREF(f); Py_DECREF(args);
        if (!got) throw_pending();
        variable_list r = {tensor_or_none(PyTuple_GET_ITEM(got, 0)), tensor_or_none(PyTuple_GET_ITEM(got, 1))};
        Py_DECREF(got);
        return r;
    }
};

// product_train(x [.., N, K], right [.., K, M], mode, longest, narrow, most) -> fp16 [.., N, M], or None where the Function has to run
PyObject* product_train(PyObject*, PyObject* const* args, const Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n == 6, "product_train takes 6 arguments");
    if (!c10::GradMode::is_enabled() || !plain_call(args, 2)) Py_RETURN_NONE;
    const Tensor &x = tensor_at(args[0]), &right = tensor_at(args[1]);
    const int mode = (int)PyLong_AsLong(args[2]);
    const int64_t longest = PyLong_AsLongLong(args[3]), narrow = PyLong_AsLongLong(args[4]), most = PyLong_AsLongLong(args[5]);
    if (PyErr_Occurred()) throw python_error();
    if (!x.requires_grad() && !right.requires_grad()) Py_RETURN_NONE;
    for (const Tensor* t : {&x, &right})
        if (!t->is_cuda() || !is_memory(*t) || has_tangent(*t) || t->scalar_type() != at::kHalf) Py_RETURN_NONE;
    Tensor out;
    {
        const WithoutGil no_gil;
        {
            const c10::NoGradGuard no_grad;
            out = batched_product_of(x, right, mode);
        }
        if (out.defined()) {
            auto node = std::shared_ptr<ProductNode>(new ProductNode(), torch::autograd::deleteNode);
            node->context = mode == BGEMM_MODE_ATTN_X;
            node->longest = longest; node->narrow = narrow; node->most = most;
            node->x_ = SavedVariable(x, false);
            node->right_ = SavedVariable(right, false);
            node->set_next_edges(torch::autograd::collect_next_edges(x, right));
            torch::autograd::set_history(out, node);
        }
    }
    if (!out.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

const PyMethodDef train_methods[] = {
    {"product_train", (PyCFunction)(void (*)(void))product_train, METH_FASTCALL, "batched product of two binarised operands, recorded as one autograd node"},
    {"elastic_train", (PyCFunction)(void (*)(void))elastic_train, METH_FASTCALL, "forward of a learned-scale binary Linear, recorded as one autograd node"},
    {"linear_train", (PyCFunction)(void (*)(void))linear_train, METH_FASTCALL, "forward of a scaled binary Linear, recorded as one autograd node"}};

// both parts' functions and the end mark
PyMethodDef* all_methods()
{
    static std::vector<PyMethodDef> all;
    if (all.empty()) {
        for (const PyMethodDef& m : train_methods) all.push_back(m);
        for (int i = 0; i < infer_method_count; i++) all.push_back(infer_methods[i]);
        all.push_back({nullptr, nullptr, 0, nullptr});
    }
    return all.data();
}

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_bgemm_native", "host side of the binary layers", -1, nullptr, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__bgemm_native(void)
{
    module_def.m_methods = all_methods();
    PyObject* const module = PyModule_Create(&module_def);
    // what it was built for: an older one lacks functions that the Python side calls
    if (module && (PyModule_AddIntConstant(module, "abi_version", BGEMM_ABI_VERSION) != 0 || PyModule_AddIntConstant(module, "native_version", NATIVE_VERSION) != 0)) {
        Py_DECREF(module);
        return nullptr;
    }
    return module;
}
