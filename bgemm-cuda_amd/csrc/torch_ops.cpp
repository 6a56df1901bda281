// The host side of the layers, native: what bgemm_linear.py and lowbit_kernel.py would do on every call in Python (argument
// checks, allocation, the stream, the calls into the C ABI, autograd bookkeeping).  A small layer's kernels take a few
// microseconds, less than those steps cost in Python.  Host code only: plain CPython functions on torch's C++ API, linked against
// libbgemm_mi355x.so beside it.  Functions that find a case they do not take return None, and the caller goes the Python way.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>

#include "../../include/bgemm_mi355x.h"

namespace {

using at::Tensor;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

// Turns a negative status into the exception _lib.check() raises.
void check(const int rc)
{
    if (rc == BGEMM_OK) return;
    const std::string msg = bgemm_last_error();
    if (rc == BGEMM_EINVAL || rc == BGEMM_ENULL || rc == BGEMM_EALIGN || rc == BGEMM_EWORKSPACE) TORCH_CHECK_VALUE(false, msg);
    TORCH_CHECK(false, msg);
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
bool is_param_type(const at::ScalarType t) { return t == at::kFloat || t == at::kHalf; }
int src_type(const Tensor& t) { return t.scalar_type() == at::kFloat ? BGEMM_SRC_F32 : BGEMM_SRC_F16; }
void* data_or_null(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
const Tensor& tensor_at(PyObject* o) { return THPVariable_Unpack(o); }
Tensor tensor_or_none(PyObject* o) { return o == Py_None ? Tensor() : THPVariable_Unpack(o); }

// Kernels are enqueued and memory is allocated without the interpreter's lock.
struct WithoutGil {
    PyThreadState* state = PyEval_SaveThread();
    ~WithoutGil() { PyEval_RestoreThread(state); }
};

// [..., C] as rows [R, C] whose elements are dense (a row stride larger than C is fine).
Tensor rows_2d(const Tensor& t)
{
    const int64_t C = t.size(-1);
    Tensor r = t.dim() == 2 ? t : t.reshape({t.numel() / C, C});
    return r.stride(1) == 1 && r.stride(0) >= C ? r : r.contiguous();
}

// ---- the scaled binary Linear as one autograd node -----------------------------------------------------------------------------
// y = fn(x - zpa, w - zpw) * sw * sa (+ bias) (tests/python/bgemm_linear.py:479-484): two launches forward, five backward.  What is
// kept for the backward pass is bits: sign and nonzero planes of both operands.
struct LinearNode : public torch::autograd::Node {
    int64_t N, K, M, words_x, words_w;
    bool bireal;
    Tensor planes;                                  // [x sign | x nonzero | w sign | w nonzero]
    Tensor sw, sa;                                  // the values of now, as with any operation's saved operands
    uint32_t sw_version, sa_version;
    std::vector<int64_t> x_shape;
    at::IntArrayRef sa_shape() const { return sa.sizes(); }
    // only needed to differentiate twice, and (x, zpa) by Bi-Real's surrogate
    SavedVariable x_, weight_, sw_, sa_, bias_, zpa_, zpw_;
    bool has_bias;

    std::string name() const override { return "ScaledBinaryLinearBackward"; }

    void release_variables() override
    {
        std::lock_guard<std::mutex> lock(mutex_);
        planes.reset();
        for (SavedVariable* s : {&x_, &weight_, &sw_, &sa_, &bias_, &zpa_, &zpw_}) s->reset_data();
    }

    // A gradient that will itself be differentiated: the separate operations, whose graph autograd knows.
    variable_list differentiable(const Tensor& grad)
    {
        pybind11::gil_scoped_acquire gil;
        const Tensor x = x_.unpack(), w = weight_.unpack(), sw0 = sw_.unpack(), sa0 = sa_.unpack(), zpa = zpa_.unpack(), zpw = zpw_.unpack();
        const Tensor bias = has_bias ? bias_.unpack() : Tensor();
        PyObject* const module = PyImport_ImportModule("bgemm_linear");
        if (!module) throw python_error();
        PyObject* const need = PyTuple_New(5);
        for (int i = 0; i < 5; i++) PyTuple_SET_ITEM(need, i, PyBool_FromLong(i < (has_bias ? 5 : 4) && task_should_compute_output(i)));
        PyObject* const got = PyObject_CallMethod(module, "_scaled_linear_grads", "iNNNNNNNNN", (int)bireal, THPVariable_Wrap(x), THPVariable_Wrap(w),
                                                  THPVariable_Wrap(sw0), THPVariable_Wrap(sa0), THPVariable_Wrap(bias), THPVariable_Wrap(zpa),
                                                  THPVariable_Wrap(zpw), THPVariable_Wrap(grad), need);
        Py_DECREF(module);
        if (!got) throw python_error();
        variable_list r;
        for (int i = 0; i < (has_bias ? 5 : 4); i++) r.push_back(tensor_or_none(PyTuple_GET_ITEM(got, i)));
        Py_DECREF(got);
        return r;
    }

    variable_list apply(variable_list&& grads) override
    {
        std::lock_guard<std::mutex> lock(mutex_);
        const size_t inputs = has_bias ? 5 : 4;
        if (!grads[0].defined()) return variable_list(inputs);
        TORCH_CHECK(planes.defined(), torch::autograd::ERR_BACKWARD_TWICE);
        if (c10::GradMode::is_enabled()) return differentiable(grads[0]);
        TORCH_CHECK(sw._version() == sw_version && sa._version() == sa_version,
                    "a scale of the binary layer was modified by an inplace operation between its forward and backward pass");
        const c10::OptionalDeviceGuard guard(planes.device());
        const bool need_x = task_should_compute_output(0), need_w = task_should_compute_output(1);
        const Tensor g = grads[0].contiguous();
        Tensor gx, gw, gb, zpa, x2;
        if (need_x) gx = at::empty(x_shape, g.options());
        if (need_w) gw = at::empty({M, K}, g.options());
        if (has_bias && task_should_compute_output(4)) gb = at::empty({M}, g.options());
        const Tensor gsw = at::empty({M}, g.options()), gsa = at::empty(sa.sizes(), g.options());
        if (bireal && need_x) {
            x2 = rows_2d(x_.unpack());
            zpa = zpa_.unpack();
        }
        const size_t bytes = bgemm_linear_backward_workspace_bytes(N, M, K, need_x, need_w);
        const Tensor ws = at::empty({(int64_t)bytes}, g.options().dtype(at::kByte));
        const int32_t* const p = planes.data_ptr<int32_t>();
        check(bgemm_linear_backward(p + 2 * words_x, p + 2 * words_x + words_w, p, p + words_x, g.data_ptr(), src_type(g), N, M, K, sw.data_ptr(),
                                    sa.data_ptr(), data_or_null(x2), x2.defined() ? x2.stride(0) : 0, data_or_null(zpa), data_or_null(gx),
                                    data_or_null(gw), data_or_null(gb), gsw.data_ptr(), gsa.data_ptr(), ws.data_ptr(), bytes, stream_of(g)));
        variable_list r = {gx, gw, gsw, gsa};
        if (has_bias) r.push_back(gb);
        return r;
    }
};

bool one_scalar(const Tensor& t) { return t.numel() == 1 && t.dim() <= 1; }

// Whether a recorded forward is the one-node form: the module's own arithmetic on one device and in one type, zero points that
// are no parameters, and sizes the kernels take.
bool one_node(const Tensor& x, const Tensor& w, const Tensor& sw, const Tensor& sa, const Tensor& bias, const Tensor& zpa, const Tensor& zpw)
{
    if (!c10::GradMode::is_enabled() || !x.is_cuda() || !is_param_type(w.scalar_type()) || w.dim() != 2 || x.dim() < 1 || x.numel() == 0) return false;
    const int64_t M = w.size(0), K = w.size(1);
    if (M < 2 || M > (1 << 20) || K >= (1 << 24) || x.size(-1) != K || x.numel() / K > (1 << 20)) return false;
    for (const Tensor* t : {&x, &w, &sw, &sa, &zpa, &zpw})
        if (t->scalar_type() != w.scalar_type() || t->device() != x.device() || t->layout() != at::kStrided) return false;
    if (!one_scalar(sa) || !one_scalar(zpa) || !one_scalar(zpw) || zpa.requires_grad() || zpw.requires_grad()) return false;
    if (sw.dim() != 1 || sw.size(0) != M || !sw.is_contiguous()) return false;
    return !bias.defined() || (bias.scalar_type() == w.scalar_type() && bias.device() == x.device() && bias.dim() == 1 && bias.size(0) == M && bias.is_contiguous());
}

// linear_train(x, weight, sw, sa, bias | None, zpa, zpw, bireal) -> y, or None where the separate operations have to run
PyObject* linear_train(PyObject*, PyObject* const* args, const Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n == 8, "linear_train takes 8 arguments");
    for (int i = 0; i < 7; i++)
        if (!THPVariable_Check(args[i]) && !(i == 4 && args[i] == Py_None)) Py_RETURN_NONE;
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
        Tensor planes;
        {
            const c10::NoGradGuard no_grad;
            const c10::OptionalDeviceGuard guard(x.device());
            const Tensor x2 = rows_2d(x), w2 = rows_2d(w);
            planes = at::empty({2 * (words_x + words_w)}, x.options().dtype(at::kInt));
            std::vector<int64_t> shape = x.sizes().vec();
            shape.back() = M;
            out = at::empty(shape, x.options());
            int32_t* const p = planes.data_ptr<int32_t>();
            void* const st = stream_of(x);
            check(bgemm_pack_sign_nonzero_pair(x2.data_ptr(), N, x2.stride(0), zpa.data_ptr(), p, p + words_x, w2.data_ptr(), M, w2.stride(0),
                                               zpw.data_ptr(), p + 2 * words_x, p + 2 * words_x + words_w, src_type(x), K, st));
            check(bgemm_packed_forward_scaled(BGEMM_MODE_XOR, p + 2 * words_x, p, nullptr, out.data_ptr(),
                                              src_type(x) == BGEMM_SRC_F32 ? BGEMM_OUT_F32_SCALED : BGEMM_OUT_F16_SCALED, 1, M, N, K, 0, 0, N * M, 8,
                                              BGEMM_VARIANT_AUTO, nullptr, 0, nullptr, 0, sw.data_ptr(), sa.data_ptr(), data_or_null(bias), st));
        }
        if (recorded) {
            node = std::shared_ptr<LinearNode>(new LinearNode(), torch::autograd::deleteNode);
            node->N = N; node->K = K; node->M = M; node->words_x = words_x; node->words_w = words_w;
            node->bireal = bireal; node->has_bias = bias.defined();
            node->planes = planes;
            node->sw = sw.detach(); node->sa = sa.detach();
            node->sw_version = sw._version(); node->sa_version = sa._version();
            node->x_shape = x.sizes().vec();
            node->x_ = SavedVariable(x, false); node->weight_ = SavedVariable(w, false);
            node->sw_ = SavedVariable(sw, false); node->sa_ = SavedVariable(sa, false);
            node->zpa_ = SavedVariable(zpa, false); node->zpw_ = SavedVariable(zpw, false);
            if (bias.defined()) {
                node->bias_ = SavedVariable(bias, false);
                node->set_next_edges(torch::autograd::collect_next_edges(x, w, sw, sa, bias));
            } else
                node->set_next_edges(torch::autograd::collect_next_edges(x, w, sw, sa));
            torch::autograd::set_history(out, node);
        }
    }
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// ---- the learned-scale layer as one autograd node ----------------------------------------------------------------------------------
// (half(acc) * sa) * sw (+ bias) of (x - mean(x)) / sa and w - mean(w) (tests/python/bgemm_linear.py:350-457, :538-564): three launches
// forward, two backward.  Kept: sign and nonzero planes of both operands, the means, and the operands themselves (as references).
struct ElasticNode : public torch::autograd::Node {
    int64_t N, K, M, words_x, words_w;
    double grad_scale;
    Tensor planes;                                  // [x sign | x nonzero | w sign | w nonzero | stats]
    SavedVariable x_, weight_, sa_, sw_, bias_;
    bool has_bias;

    std::string name() const override { return "ElasticBinaryLinearBackward"; }

    void release_variables() override
    {
        std::lock_guard<std::mutex> lock(mutex_);
        planes.reset();
        for (SavedVariable* s : {&x_, &weight_, &sa_, &sw_, &bias_}) s->reset_data();
    }

    variable_list differentiable(const Tensor& grad)
    {
        pybind11::gil_scoped_acquire gil;
        const Tensor bias = has_bias ? bias_.unpack() : Tensor();
        PyObject* const module = PyImport_ImportModule("bgemm_linear");
        if (!module) throw python_error();
        PyObject* const need = PyTuple_New(5);
        for (int i = 0; i < 5; i++) PyTuple_SET_ITEM(need, i, PyBool_FromLong(i < (has_bias ? 5 : 4) && task_should_compute_output(i)));
        PyObject* const got = PyObject_CallMethod(module, "_elastic_grads", "NNNNNdNN", THPVariable_Wrap(x_.unpack()), THPVariable_Wrap(weight_.unpack()),
                                                  THPVariable_Wrap(sa_.unpack()), THPVariable_Wrap(sw_.unpack()), THPVariable_Wrap(bias), grad_scale,
                                                  THPVariable_Wrap(grad), need);
        Py_DECREF(module);
        if (!got) throw python_error();
        variable_list r;
        for (int i = 0; i < (has_bias ? 5 : 4); i++) r.push_back(tensor_or_none(PyTuple_GET_ITEM(got, i)));
        Py_DECREF(got);
        return r;
    }

    variable_list apply(variable_list&& grads) override
    {
        std::lock_guard<std::mutex> lock(mutex_);
        const size_t inputs = has_bias ? 5 : 4;
        if (!grads[0].defined()) return variable_list(inputs);
        TORCH_CHECK(planes.defined(), torch::autograd::ERR_BACKWARD_TWICE);
        if (c10::GradMode::is_enabled()) return differentiable(grads[0]);
        const c10::OptionalDeviceGuard guard(planes.device());
        const bool want_x = task_should_compute_output(0), want_sa = task_should_compute_output(2);
        const bool need_x = want_x || want_sa, need_w = task_should_compute_output(1) || task_should_compute_output(3);
        const Tensor g = grads[0].contiguous(), x = x_.unpack().contiguous(), w = weight_.unpack().contiguous(), sa = sa_.unpack();
        Tensor gx, gw, gb, gsw, gsa;
        const bool need_b = has_bias && task_should_compute_output(4);
        if (!need_x && !need_w) {
            if (need_b) gb = g.reshape({N, M}).sum(0);
        } else {
            if (need_x) gx = at::empty(x.sizes(), g.options());
            if (want_sa) gsa = at::empty({}, g.options());
            if (need_w) {
                gw = at::empty({M, K}, g.options());
                gsw = at::empty({M}, g.options());
            }
            if (need_b) gb = at::empty({M}, g.options());
            const size_t bytes = bgemm_elastic_backward_workspace_bytes(N, M, K, need_x, need_w);
            const Tensor ws = at::empty({(int64_t)bytes}, g.options().dtype(at::kByte));
            const int32_t* const p = planes.data_ptr<int32_t>();
            const int32_t* const pw = p + 2 * words_x;
            check(bgemm_elastic_backward(p, p + words_x, pw, pw + words_w, g.data_ptr(), x.data_ptr(), w.data_ptr(), pw + 2 * words_w, sa.data_ptr(),
                                         (float)grad_scale, N, M, K, data_or_null(gx), data_or_null(gw), data_or_null(gb), data_or_null(gsw),
                                         data_or_null(gsa), ws.data_ptr(), bytes, stream_of(g)));
        }
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
    for (int i = 0; i < 5; i++)
        if (!THPVariable_Check(args[i]) && !(i == 4 && args[i] == Py_None)) Py_RETURN_NONE;
    const Tensor &x = tensor_at(args[0]), &w = tensor_at(args[1]), &sa = tensor_at(args[2]), &sw = tensor_at(args[3]);
    const Tensor bias = tensor_or_none(args[4]);
    const double grad_scale = PyFloat_AsDouble(args[5]);
    if (grad_scale == -1.0 && PyErr_Occurred()) throw python_error();
    if (!c10::GradMode::is_enabled() || !x.is_cuda() || w.dim() != 2 || x.dim() < 1 || x.numel() == 0 || sa.dim() != 0) Py_RETURN_NONE;
    const int64_t M = w.size(0), K = w.size(1), N = x.numel() / (K ? K : 1);
    if (M < 2 || M > (1 << 20) || K < 1 || K >= (1 << 24) || x.size(-1) != K || N > (1 << 20)) Py_RETURN_NONE;
    for (const Tensor* t : {&x, &w, &sa, &sw})
        if (t->scalar_type() != at::kFloat || t->device() != x.device() || t->layout() != at::kStrided) Py_RETURN_NONE;
    if (sw.dim() != 1 || sw.size(0) != M || !sw.is_contiguous()) Py_RETURN_NONE;
    if (bias.defined() && (bias.scalar_type() != at::kFloat || bias.device() != x.device() || bias.dim() != 1 || bias.size(0) != M || !bias.is_contiguous())) Py_RETURN_NONE;
    Tensor out;
    {
        const WithoutGil no_gil;
        bool recorded = bias.defined() && bias.requires_grad();
        for (const Tensor* t : {&x, &w, &sa, &sw}) recorded |= t->requires_grad();
        const int64_t words_x = bgemm_tiled_words(N, K), words_w = bgemm_tiled_words(M, K);
        Tensor planes;
        {
            const c10::NoGradGuard no_grad;
            const c10::OptionalDeviceGuard guard(x.device());
            const Tensor x2 = x.contiguous(), w2 = w.contiguous();
            planes = at::empty({2 * (words_x + words_w) + BGEMM_ELASTIC_STATS}, x.options().dtype(at::kInt));
            std::vector<int64_t> shape = x.sizes().vec();
            shape.back() = M;
            out = at::empty(shape, x.options());
            int32_t* const p = planes.data_ptr<int32_t>();
            int32_t* const pw = p + 2 * words_x;
            check(bgemm_elastic_forward(x2.data_ptr(), w2.data_ptr(), N, M, K, sa.data_ptr(), sw.data_ptr(), data_or_null(bias), p, p + words_x, pw,
                                        pw + words_w, pw + 2 * words_w, out.data_ptr(), stream_of(x)));
        }
        if (recorded) {
            auto node = std::shared_ptr<ElasticNode>(new ElasticNode(), torch::autograd::deleteNode);
            node->N = N; node->K = K; node->M = M; node->words_x = words_x; node->words_w = words_w;
            node->grad_scale = grad_scale; node->has_bias = bias.defined();
            node->planes = planes;
            node->x_ = SavedVariable(x, false); node->weight_ = SavedVariable(w, false);
            node->sa_ = SavedVariable(sa, false); node->sw_ = SavedVariable(sw, false);
            if (bias.defined()) {
                node->bias_ = SavedVariable(bias, false);
                node->set_next_edges(torch::autograd::collect_next_edges(x, w, sa, sw, bias));
            } else
                node->set_next_edges(torch::autograd::collect_next_edges(x, w, sa, sw));
            torch::autograd::set_history(out, node);
        }
    }
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"elastic_train", (PyCFunction)(void (*)(void))elastic_train, METH_FASTCALL, "forward of a learned-scale binary Linear, recorded as one autograd node"},
    {"linear_train", (PyCFunction)(void (*)(void))linear_train, METH_FASTCALL, "forward of a scaled binary Linear, recorded as one autograd node"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_bgemm_native", "host side of the binary layers", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__bgemm_native(void) { return PyModule_Create(&module_def); }
