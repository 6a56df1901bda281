// The native host side of inference and of the attention products (see torch_ops.cpp): a decode layer's kernel takes five
// microseconds and its checks, key, allocation and call took ten in Python.  Every function looks at its arguments on each call, keeps
// nothing between calls, and returns None for whatever it does not take: the Python form behind it then runs, or raises what it raises.
#include "torch_common.h"

#include <torch/csrc/DynamicTypes.h>

#include <algorithm>
#include <vector>

namespace bgemm_native {
namespace {

PyObject* interned(const char* s) { return PyUnicode_InternFromString(s); }

// Borrowed reference or null; no error is left behind.
PyObject* item(PyObject* dict, PyObject* key)
{
    PyObject* const v = PyDict_GetItemWithError(dict, key);
    if (!v) PyErr_Clear();
    return v;
}

bool exact(PyObject* o) { return o && THPVariable_CheckExact(o); }
bool plain_gpu(PyObject* o) { return exact(o) && tensor_at(o).is_cuda() && is_memory(tensor_at(o)); }
bool fits(const Tensor& t, const at::ScalarType dt, const c10::Device dev) { return t.scalar_type() == dt && t.device() == dev && is_memory(t); }
// a tiled operand's plane
bool is_plane(const Tensor& t, const c10::Device dev, const int64_t batch, const int64_t rows, const int64_t K)
{
    return fits(t, at::kInt, dev) && t.is_contiguous() && t.dim() == 2 && t.size(0) == batch && t.size(1) == bgemm_tiled_words(rows, K);
}
Tensor new_plane(const Tensor& like, const int64_t batch, const int64_t rows, const int64_t K)
{
    return at::empty({batch, bgemm_tiled_words(rows, K)}, like.options().dtype(at::kInt).requires_grad(false));
}
int scaled_kind(const bool f32) { return f32 ? BGEMM_OUT_F32_SCALED : BGEMM_OUT_F16_SCALED; }
int bits_kind(const bool f32) { return f32 ? BGEMM_OUT_BITS_F32 : BGEMM_OUT_BITS_F16; }
std::vector<int64_t> with_last(const Tensor& x, const int64_t M)
{
    std::vector<int64_t> shape = x.sizes().vec();
    shape.back() = M;
    return shape;
}

// ---- scaled layers ------------------------------------------------------------------------------------------------------------------
// What a BGEMMLinear's inference reads, from the module's own dictionaries: parameters and zero points of one type on one device, and
// the packed weight it keeps, if that is the weight's as it is now (the same key as BGEMMLinear._weight_key).
struct Layer {
    Tensor weight, sw, sa, bias, zpa, packed;
    int64_t M, K;

    // (kept: the packed weight as well)
    bool read(PyObject* dict, const Tensor& x, const bool kept = true)
    {
        static PyObject* const k_params = interned("_parameters"), * const k_weight = interned("weight"), * const k_bias = interned("bias"),
                       * const k_sw = interned("sw"), * const k_sa = interned("sa"), * const k_zpa = interned("zpa"), * const k_zpw = interned("zpw"),
                       * const k_wp = interned("_wp"), * const k_key = interned("_wp_key"), * const k_data = interned("data"), * const k_data2 = interned("data2"),
                       * const k_fuse = interned("fuse_inference"), * const k_init = interned("initialized");
        if (!PyDict_CheckExact(dict) || item(dict, k_init) != Py_True) return false;
        PyObject* const fuse = item(dict, k_fuse);                    // the instance's own (the class's is asked in Python)
        if (fuse && fuse != Py_True) return false;
        PyObject* const params = item(dict, k_params);
        if (!params || !PyDict_Check(params)) return false;
        PyObject* const pw = item(params, k_weight), * const psw = item(params, k_sw), * const psa = item(params, k_sa), * const pb = item(params, k_bias);
        PyObject* const pza = item(dict, k_zpa), * const pzw = item(dict, k_zpw), * const wp = item(dict, k_wp), * const key = item(dict, k_key);
        if (!exact(pw) || !exact(psw) || !exact(psa) || !pb || (pb != Py_None && !exact(pb)) || !exact(pza) || !exact(pzw)) return false;
        weight = tensor_at(pw); sw = tensor_at(psw); sa = tensor_at(psa); zpa = tensor_at(pza);
        bias = pb == Py_None ? Tensor() : tensor_at(pb);
        const at::ScalarType dt = x.scalar_type();
        const c10::Device dev = x.device();
        if (weight.dim() != 2 || !is_param_type(dt)) return false;
        M = weight.size(0); K = weight.size(1);
        if (!fits(weight, dt, dev) || !fits(sw, dt, dev) || !fits(sa, dt, dev) || !fits(zpa, dt, dev) || sw.dim() != 1 || sw.size(0) != M || !sw.is_contiguous() ||
            sa.numel() != 1 || zpa.numel() != 1 || (bias.defined() && (!fits(bias, dt, dev) || bias.dim() != 1 || bias.size(0) != M || !bias.is_contiguous())))
            return false;
        if (!kept) return true;
        // the kept bits
        if (!wp || !key) return false;
        const Tensor& zpw = tensor_at(pzw);
        if (weight.is_inference() || zpw.is_inference() || !zpw.defined() || !zpw.has_storage()) return false;
        if (!PyTuple_CheckExact(key) || PyTuple_GET_SIZE(key) != 6) return false;
        auto is = [&](const int i, const int64_t v) {
            PyObject* const o = PyTuple_GET_ITEM(key, i);
            if (!PyLong_CheckExact(o)) return false;
            const unsigned long long u = PyLong_AsUnsignedLongLongMask(o);
            if (u == (unsigned long long)-1 && PyErr_Occurred()) PyErr_Clear();
            return u == (unsigned long long)v;
        };
        if (!is(0, weight._version()) || !is(1, (int64_t)(intptr_t)weight.data_ptr()) || PyTuple_GET_ITEM(key, 2) != (PyObject*)torch::getTHPDtype(dt) ||
            !is(3, (int64_t)(intptr_t)pzw) || !is(4, zpw._version()) || !is(5, (int64_t)(intptr_t)zpw.data_ptr()))
            return false;
        PyObject* const data = PyObject_GetAttr(wp, k_data), * const data2 = PyObject_GetAttr(wp, k_data2);
        bool ok = false;
        if (exact(data) && data2 == Py_None) {
            packed = tensor_at(data);
            ok = is_plane(packed, dev, 1, M, K);
        }
        PyErr_Clear();
        Py_XDECREF(data); Py_XDECREF(data2);
        return ok;
    }

    bgemm_rows_layer rows_layer(void* out, const void* next = nullptr) const
    {
        return {packed.data_ptr(), zpa.data_ptr(), sw.data_ptr(), sa.data_ptr(), data_or_null(bias), next, out};
    }
};

// Whether a call without a gradient may go past torch's operations at all.
bool quiet_call(PyObject* x) { return !c10::GradMode::is_enabled() && plain_gpu(x) && !is_watched(); }

// Packed weights x rows as they are, with the scratch that the size needs.
void unpacked(const int mode, const Tensor& w, const Rows& x, const Tensor& zp, const Tensor& out, const int kind, const int64_t M, const int64_t N, const int64_t K,
              const Tensor& sw, const Tensor& sa, const Tensor& bias)
{
    void* const st = stream_of(out);
    const size_t bytes = bgemm_unpacked_workspace_bytes_on(mode, x.t.data_ptr(), src_type(x.t), x.ld, M, N, K, st);
    Tensor ws;
    if (bytes) ws = at::empty({(int64_t)bytes}, x.t.options().dtype(at::kByte).requires_grad(false));
    check(bgemm_unpacked_forward(mode, w.data_ptr(), x.t.data_ptr(), src_type(x.t), x.ld, data_or_null(zp), out.data_ptr(), kind, M, N, K, data_or_null(sw),
                                 data_or_null(sa), data_or_null(bias), data_or_null(ws), bytes, st));
}

// linear_infer(module.__dict__, x) -> y
PyObject* linear_infer(PyObject*, PyObject* const* args, const Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n == 2, "linear_infer takes 2 arguments");
    if (!quiet_call(args[1])) Py_RETURN_NONE;
    const Tensor& x = tensor_at(args[1]);
    Layer l;
    if (x.dim() < 1 || x.numel() == 0 || !l.read(args[0], x) || x.size(-1) != l.K || l.M == 0) Py_RETURN_NONE;
    const int64_t N = x.numel() / l.K;
    Tensor out;
    {
        const WithoutGil no_gil;
        const c10::OptionalDeviceGuard guard(x.device());
        const Rows r = rows_2d(x);
        const bool f32 = x.scalar_type() == at::kFloat;
        const int kind = scaled_kind(f32);
        out = at::empty(with_last(x, l.M), x.options().requires_grad(false));
        void* const st = stream_of(x);
        if (bgemm_packed_weight_forward_supported(BGEMM_MODE_XOR, l.M, N, l.K))
            check(bgemm_packed_weight_forward(BGEMM_MODE_XOR, l.packed.data_ptr(), r.t.data_ptr(), src_type(x), r.ld, l.zpa.data_ptr(), out.data_ptr(), kind, l.M, N, l.K,
                                              BGEMM_VARIANT_AUTO, l.sw.data_ptr(), l.sa.data_ptr(), data_or_null(l.bias), nullptr, st));
        else if (bgemm_linear_rows_supported(N, l.M, l.K, 1, kind) == 2) {
            const bgemm_rows_layer layer = l.rows_layer(out.data_ptr());
            check(bgemm_linear_rows_forward(r.t.data_ptr(), src_type(x), r.ld, N, l.M, l.K, 1, &layer, kind, nullptr, 0, st));
        } else {
            unpacked(BGEMM_MODE_XOR, l.packed, r, l.zpa, out, kind, l.M, N, l.K, l.sw, l.sa, l.bias);
        }
    }
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// chain_infer([module.__dict__, ..], x) -> y: only bits between the layers
PyObject* chain_infer(PyObject*, PyObject* const* args, const Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n == 2 && PyList_CheckExact(args[0]), "chain_infer takes a list and a tensor");
    const Py_ssize_t layers = PyList_GET_SIZE(args[0]);
    if (layers < 2 || !quiet_call(args[1])) Py_RETURN_NONE;
    const Tensor& x = tensor_at(args[1]);
    if (x.dim() < 1 || x.numel() == 0) Py_RETURN_NONE;
    const int64_t K0 = x.size(-1), N = x.numel() / K0;
    std::vector<Layer> l(layers);
    int64_t K = K0, most = 0;                 // words of the largest operand between two layers
    for (Py_ssize_t i = 0; i < layers; i++) {
        if (!l[i].read(PyList_GET_ITEM(args[0], i), x) || l[i].K != K || l[i].M == 0) Py_RETURN_NONE;
        K = l[i].M;
        if (i + 1 < layers) most = std::max(most, bgemm_tiled_words(N, K));
    }
    Tensor out;
    {
        const WithoutGil no_gil;
        const c10::OptionalDeviceGuard guard(x.device());
        const Rows r = rows_2d(x);
        const bool f32 = x.scalar_type() == at::kFloat;
        void* const st = stream_of(x);
        // The call's own bits, so that other streams and threads may be in the same modules: a layer reads one half and writes the other.
        const c10::DataPtr planes = c10::GetAllocator(x.device().type())->allocate((layers > 2 ? 2 : 1) * most * sizeof(int32_t));
        int32_t* const half[2] = {static_cast<int32_t*>(planes.get()), static_cast<int32_t*>(planes.get()) + (layers > 2 ? most : 0)};
        const void* in = nullptr;             // the operand of the layer at hand; null: x itself
        Tensor first;
        if (bgemm_linear_rows_supported(N, l[0].M, K0, 1, bits_kind(f32)) != 2) {
            first = new_plane(x, 1, N, K0);
            in = first.data_ptr();
            check(bgemm_pack_batched(r.t.data_ptr(), src_type(x), 0, l[0].zpa.data_ptr(), 1, 1, N, K0, r.ld, 0, 0, first.data_ptr(), nullptr, st));
        }
        out = at::empty(with_last(x, l.back().M), x.options().requires_grad(false));
        for (Py_ssize_t i = 0; i < layers; i++) {
            const Layer& a = l[i];
            if (i + 1 == layers)
                check(bgemm_packed_forward_scaled(BGEMM_MODE_XOR, a.packed.data_ptr(), in, nullptr, out.data_ptr(), scaled_kind(f32), 1, a.M, N, a.K, 0, 0, N * a.M,
                                                  8, BGEMM_VARIANT_AUTO, nullptr, 0, nullptr, 0, a.sw.data_ptr(), a.sa.data_ptr(), data_or_null(a.bias), st));
            else {
                const void* const next = l[i + 1].zpa.data_ptr();
                int32_t* const bits = half[i & 1];
                if (!in) {
                    const bgemm_rows_layer layer = a.rows_layer(bits, next);
                    check(bgemm_linear_rows_forward(r.t.data_ptr(), src_type(x), r.ld, N, a.M, a.K, 1, &layer, bits_kind(f32), nullptr, 0, st));
                } else
                    check(bgemm_packed_forward_bits(BGEMM_MODE_XOR, a.packed.data_ptr(), in, nullptr, bits, bits_kind(f32), 1, a.M, N, a.K, 0, 0,
                                                    bgemm_tiled_words(N, a.M), 8, BGEMM_VARIANT_AUTO, nullptr, 0, nullptr, 0, a.sw.data_ptr(), a.sa.data_ptr(),
                                                    data_or_null(a.bias), next, st));
                in = bits;
            }
        }
    }
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// block_ready([module.__dict__, ..], x [batch, seq, features], heads, head size) -> whether these layers are projections of x into such heads, in
// x's type, and the attention kernel takes those
PyObject* block_ready(PyObject*, PyObject* const* args, const Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n == 4 && PyList_CheckExact(args[0]), "block_ready takes a list, a tensor and two numbers");
    if (!quiet_call(args[1])) Py_RETURN_FALSE;
    const Tensor& x = tensor_at(args[1]);
    const int64_t heads = PyLong_AsLongLong(args[2]), size = PyLong_AsLongLong(args[3]);
    if (PyErr_Occurred()) throw python_error();
    if (x.dim() != 3 || x.numel() == 0 || !bgemm_attention_supported(x.size(0), x.size(1), heads, size)) Py_RETURN_FALSE;
    Layer l;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(args[0]); i++)
        if (!l.read(PyList_GET_ITEM(args[0], i), x, false) || l.K != x.size(-1) || l.M != heads * size) Py_RETURN_FALSE;
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// rows_bits([module.__dict__, ..], x) -> a tuple of planes: the sign bits of every layer's output
PyObject* rows_bits(PyObject*, PyObject* const* args, const Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n == 2 && PyList_CheckExact(args[0]), "rows_bits takes a list and a tensor");
    const Py_ssize_t layers = PyList_GET_SIZE(args[0]);
    if (layers < 1 || layers > 3 || !quiet_call(args[1])) Py_RETURN_NONE;
    const Tensor& x = tensor_at(args[1]);
    if (x.dim() < 1 || x.numel() == 0) Py_RETURN_NONE;
    Layer l[3];
    for (Py_ssize_t i = 0; i < layers; i++)
        if (!l[i].read(PyList_GET_ITEM(args[0], i), x) || l[i].K != x.size(-1) || l[i].M != l[0].M) Py_RETURN_NONE;
    const int64_t N = x.numel() / l[0].K;
    const bool f32 = x.scalar_type() == at::kFloat;
    if (!bgemm_linear_rows_supported(N, l[0].M, l[0].K, (int)layers, bits_kind(f32))) Py_RETURN_NONE;
    Tensor out[3];
    {
        const WithoutGil no_gil;
        const c10::OptionalDeviceGuard guard(x.device());
        const Rows r = rows_2d(x);
        bgemm_rows_layer layer[3];
        for (Py_ssize_t i = 0; i < layers; i++) {
            out[i] = new_plane(x, 1, N, l[i].M);
            layer[i] = l[i].rows_layer(out[i].data_ptr());
        }
        check(bgemm_linear_rows_forward(r.t.data_ptr(), src_type(x), r.ld, N, l[0].M, l[0].K, (int)layers, layer, bits_kind(f32), nullptr, 0, stream_of(x)));
    }
    PyObject* const t = PyTuple_New(layers);
    for (Py_ssize_t i = 0; i < layers; i++) PyTuple_SET_ITEM(t, i, THPVariable_Wrap(out[i]));
    return t;
    END_HANDLE_TH_ERRORS
}

// rows_residual(module.__dict__, plane of centred sign bits, residual, norm) -> the layer's output plus the residual, in the residual's
// shape; norm: None, or (gamma | None, beta | None, eps) of a layer norm over that
PyObject* rows_residual(PyObject*, PyObject* const* args, const Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n == 4, "rows_residual takes 4 arguments");
    if (!quiet_call(args[2]) || !plain_gpu(args[1])) Py_RETURN_NONE;
    const Tensor &bits = tensor_at(args[1]), &res = tensor_at(args[2]);
    Layer l;
    if (res.dim() < 1 || res.numel() == 0 || !res.is_contiguous() || !l.read(args[0], res) || res.size(-1) != l.M) Py_RETURN_NONE;
    const int64_t N = res.numel() / l.M;
    const int kind = scaled_kind(res.scalar_type() == at::kFloat);
    if (!is_plane(bits, res.device(), 1, N, l.K)) Py_RETURN_NONE;
    const bool norm = args[3] != Py_None;
    Tensor gamma, beta;
    double eps = 0;
    if (norm) {
        if (!PyTuple_CheckExact(args[3]) || PyTuple_GET_SIZE(args[3]) != 3 || kind != BGEMM_OUT_F32_SCALED || !bgemm_linear_rows_norm_supported(N, l.M, l.K)) Py_RETURN_NONE;
        Tensor* const to[2] = {&gamma, &beta};
        for (int i = 0; i < 2; i++) {
            PyObject* const o = PyTuple_GET_ITEM(args[3], i);
            if (o == Py_None) continue;
            if (!exact(o) || !fits(tensor_at(o), at::kFloat, res.device()) || tensor_at(o).dim() != 1 || tensor_at(o).size(0) != l.M || !tensor_at(o).is_contiguous()) Py_RETURN_NONE;
            *to[i] = tensor_at(o);
        }
        eps = PyFloat_AsDouble(PyTuple_GET_ITEM(args[3], 2));
        if (PyErr_Occurred()) throw python_error();
    } else if (!bgemm_linear_rows_supported(N, l.M, l.K, 1, kind))
        Py_RETURN_NONE;
    Tensor out;
    {
        const WithoutGil no_gil;
        const c10::OptionalDeviceGuard guard(res.device());
        out = at::empty(res.sizes(), res.options().requires_grad(false));
        const bgemm_rows_layer layer = l.rows_layer(out.data_ptr());
        check(norm ? bgemm_linear_rows_norm_forward(bits.data_ptr(), N, l.M, l.K, &layer, res.data_ptr(), data_or_null(gamma), data_or_null(beta), eps, stream_of(res))
                   : bgemm_linear_rows_forward(bits.data_ptr(), BGEMM_SRC_BITS, 0, N, l.M, l.K, 1, &layer, kind, res.data_ptr(), 0, stream_of(res)));
    }
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// ---- packed operands --------------------------------------------------------------------------------------------------------------------
// packed_weight_forward(w plane, w rows, K, x, mode, output kind, sw | None, sa, bias | None, zero point | None) -> y
PyObject* packed_weight_forward(PyObject*, PyObject* const* args, const Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n == 10, "packed_weight_forward takes 10 arguments");
    if (!plain_gpu(args[0]) || !plain_gpu(args[3]) || is_watched()) Py_RETURN_NONE;
    const Tensor &w = tensor_at(args[0]), &x = tensor_at(args[3]);
    const int64_t M = PyLong_AsLongLong(args[1]), K = PyLong_AsLongLong(args[2]);
    const int mode = (int)PyLong_AsLong(args[4]), kind = (int)PyLong_AsLong(args[5]);
    if (PyErr_Occurred()) throw python_error();
    if (x.dim() != 2 || x.size(1) != K || x.numel() == 0 || !is_param_type(x.scalar_type()) || M < 1 || !is_plane(w, x.device(), 1, M, K)) Py_RETURN_NONE;
    const bool scaled = args[6] != Py_None, ternary = mode == BGEMM_MODE_BWTA;
    Tensor sw, sa, bias, zp;
    at::ScalarType out_type = kind == BGEMM_OUT_F16 ? at::kHalf : at::kInt;
    if (scaled) {
        if (!exact(args[6]) || !exact(args[7]) || (args[8] != Py_None && !exact(args[8]))) Py_RETURN_NONE;
        sw = tensor_at(args[6]); sa = tensor_at(args[7]); bias = tensor_or_none(args[8]);
        out_type = sw.scalar_type();
        if (!is_param_type(out_type) || kind != scaled_kind(out_type == at::kFloat)) Py_RETURN_NONE;
        if (!fits(sw, out_type, x.device()) || sw.numel() != M || !sw.is_contiguous() || !fits(sa, out_type, x.device()) || sa.numel() != 1 ||
            (bias.defined() && (!fits(bias, out_type, x.device()) || bias.numel() != M || !bias.is_contiguous())))
            Py_RETURN_NONE;
    } else if (kind != BGEMM_OUT_I32 && kind != BGEMM_OUT_F16)
        Py_RETURN_NONE;
    if (args[9] != Py_None) {
        if (ternary || !exact(args[9])) Py_RETURN_NONE;
        zp = tensor_at(args[9]);
        if (!fits(zp, x.scalar_type(), x.device()) || zp.numel() != 1) Py_RETURN_NONE;
    }
    const int64_t N = x.size(0);
    Tensor out;
    {
        const WithoutGil no_gil;
        const c10::OptionalDeviceGuard guard(x.device());
        const c10::NoGradGuard no_grad;
        const Rows r = rows_2d(x);
        void* const st = stream_of(x);
        out = at::empty({N, M}, x.options().dtype(out_type).requires_grad(false));
        if (bgemm_packed_weight_forward_supported(mode, M, N, K))
            check(bgemm_packed_weight_forward(mode, w.data_ptr(), r.t.data_ptr(), src_type(x), r.ld, data_or_null(zp), out.data_ptr(), kind, M, N, K, BGEMM_VARIANT_AUTO,
                                              data_or_null(sw), data_or_null(sa), data_or_null(bias), nullptr, st));
        else if (scaled && mode == BGEMM_MODE_XOR && out_type == x.scalar_type() && bgemm_linear_rows_supported(N, M, K, 1, kind) == 2) {
            const bgemm_rows_layer layer = {w.data_ptr(), data_or_null(zp), sw.data_ptr(), sa.data_ptr(), data_or_null(bias), nullptr, out.data_ptr()};
            check(bgemm_linear_rows_forward(r.t.data_ptr(), src_type(x), r.ld, N, M, K, 1, &layer, kind, nullptr, 0, st));
        } else {
            unpacked(mode, w, r, zp, out, kind, M, N, K, sw, sa, bias);
        }
    }
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// packed_forward(w plane, w batch, w rows, K, x plane, x second plane | None, x batch, x rows, mode, output kind) -> [batch, N, M]
PyObject* packed_forward(PyObject*, PyObject* const* args, const Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n == 10, "packed_forward takes 10 arguments");
    if (!plain_gpu(args[0]) || !plain_gpu(args[4]) || (args[5] != Py_None && !plain_gpu(args[5])) || is_watched()) Py_RETURN_NONE;
    const Tensor &w = tensor_at(args[0]), &x = tensor_at(args[4]);
    const Tensor x2 = tensor_or_none(args[5]);
    const int64_t wb = PyLong_AsLongLong(args[1]), M = PyLong_AsLongLong(args[2]), K = PyLong_AsLongLong(args[3]), xb = PyLong_AsLongLong(args[6]), N = PyLong_AsLongLong(args[7]);
    const int mode = (int)PyLong_AsLong(args[8]), kind = (int)PyLong_AsLong(args[9]);
    if (PyErr_Occurred()) throw python_error();
    const int64_t batch = wb > xb ? wb : xb;
    if (wb < 1 || xb < 1 || M < 1 || N < 1 || K < 1 || (wb != 1 && wb != batch) || (xb != 1 && xb != batch) || (mode == BGEMM_MODE_BWTA) != x2.defined() ||
        (kind != BGEMM_OUT_I32 && kind != BGEMM_OUT_F16) || !is_plane(w, w.device(), wb, M, K) || !is_plane(x, w.device(), xb, N, K) ||
        (x2.defined() && !is_plane(x2, w.device(), xb, N, K)))
        Py_RETURN_NONE;
    Tensor out;
    {
        const WithoutGil no_gil;
        const c10::OptionalDeviceGuard guard(w.device());
        out = at::empty({batch, N, M}, w.options().dtype(kind == BGEMM_OUT_F16 ? at::kHalf : at::kInt));
        check(bgemm_packed_forward(mode, w.data_ptr(), x.data_ptr(), data_or_null(x2), out.data_ptr(), kind, batch, M, N, K, wb > 1 ? w.size(1) : 0, xb > 1 ? x.size(1) : 0,
                                   N * M, 1, BGEMM_VARIANT_AUTO, nullptr, 0, nullptr, 0, stream_of(w)));
    }
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// f16_forward(x, w, splitK, INSTR) -> [N, M]
PyObject* f16_forward(PyObject*, PyObject* const* args, const Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n == 4, "f16_forward takes 4 arguments");
    if (!plain_gpu(args[0]) || !plain_gpu(args[1]) || is_watched() || !PyLong_CheckExact(args[2]) || !PyLong_CheckExact(args[3])) Py_RETURN_NONE;
    const Tensor &x0 = tensor_at(args[0]), &w0 = tensor_at(args[1]);
    const long split = PyLong_AsLong(args[2]), instr = PyLong_AsLong(args[3]);
    if (PyErr_Occurred()) throw python_error();
    if (x0.dim() != 2 || w0.dim() != 2 || x0.scalar_type() != at::kHalf || w0.scalar_type() != at::kHalf || x0.size(1) != w0.size(1) || x0.device() != w0.device() ||
        instr < BGEMM_MODE_AND || instr > BGEMM_MODE_ATTN || split < 1 || split > 65535 || x0.numel() == 0 || w0.numel() == 0)
        Py_RETURN_NONE;
    Tensor out;
    {
        const WithoutGil no_gil;
        const c10::OptionalDeviceGuard guard(x0.device());
        const c10::NoGradGuard no_grad;
        const Tensor x = x0.contiguous(), w = w0.contiguous();
        const int64_t N = x.size(0), K = x.size(1), M = w.size(0);
        out = at::empty({N, M}, x.options().requires_grad(false));
        const size_t bytes = bgemm_f16_workspace_bytes(M, N, K, (int)split);
        const Tensor ws = at::empty({(int64_t)(bytes ? bytes : 1)}, x.options().dtype(at::kByte).requires_grad(false));
        check(bgemm_f16_forward(w.data_ptr(), x.data_ptr(), out.data_ptr(), M, N, K, ws.data_ptr(), bytes, (int)split, (int)instr, stream_of(x)));
    }
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// ---- attention's products -----------------------------------------------------------------------------------------------------------------
struct Batch { int64_t outer, inner, so, si; };
Batch batch_of(const Tensor& t)
{
    return t.dim() == 3 ? Batch{1, t.size(0), 0, t.stride(0)} : Batch{t.size(0), t.size(1), t.stride(0), t.stride(1)};
}

// Whether the one-launch kernels are ahead of two packs and a GEMM (us, batch x rows x columns, D).  The scores' is until what it writes
// outgrows the caches, where the GEMM's own store order is as good: 48 x 512^2, 64 14.5 -> 7.0; 192 x 512^2, 128 37.6 -> 30.5;
// 192 x 340^2, 96 31.9 -> 23.7; 2 x 32^2, 32 10.3 -> 3.4; but 128 x 1024^2, 128 67.9 -> 70.4, 16 x 4096^2, 32 96.4 -> 101.3.
bool scores_in_one(const int64_t batch, const int64_t N, const int64_t M, const int64_t D)
{
    return (D == 32 || D == 64 || D == 96 || D == 128) && N <= 1 << 20 && M <= 1 << 20 && N * M < 1 << 27 && batch * N * M < 1 << 27;
}

// The context's packs a matrix' [M][D] values again in each block, which has to stay a small part of its work: 48 x 512^2, 64 20.5 -> 10.8;
// 192 x 256^2, 128 24.7 -> 21.7; 192 x 1024^2, 32 98.6 -> 86.1; 12 x 1024^2, 64 22.2 -> 15.8; 2 x 2048^2, 32 17.3 -> 16.3; but one
// 2048^2, 32 14.8 -> 16.3, 192 x 1024^2, 64 110.6 -> 112.8, 192 x 512^2, 128 40.9 -> 40.8, 64 x 1024^2, 128 44.1 -> 56.6.
bool context_in_one(const int64_t batch, const int64_t N, const int64_t M, const int64_t D)
{
    return (D == 32 || D == 64 || D == 96 || D == 128) && N <= 1 << 20 && M >= 8 && (M * D <= 1 << 15 || (M * D <= 1 << 16 && D <= 64 && batch > 1 && batch * N * M < 1 << 27));
}

}  // namespace

// One launch on fp16 operands of an attention product's form, else both operands packed where they lie and one GEMM over the batch.
Tensor batched_product_of(const Tensor& x, const Tensor& right, const int mode)
{
    const int64_t d = x.dim();
    if ((d != 3 && d != 4) || right.dim() != d || !is_param_type(x.scalar_type()) || !is_param_type(right.scalar_type()) || right.device() != x.device() || x.numel() == 0 ||
        right.numel() == 0 || x.size(-1) != right.size(-2) || x.size(0) != right.size(0) || (d == 4 && x.size(1) != right.size(1)))
        return Tensor();
    const int64_t N = x.size(-2), K = x.size(-1), M = right.size(-1);
    // rows read where they lie; the right operand row by row of its transpose if that is dense, else column by column
    const bool by_rows = right.stride(-2) == 1 && right.stride(-1) >= K, by_columns = right.stride(-1) == 1 && right.stride(-2) >= M;
    if (x.stride(-1) != 1 || x.stride(-2) < K || !(by_rows || by_columns)) return Tensor();
    const Batch bx = batch_of(x), br = batch_of(right);
    if (bx.so < 0 || bx.si < 0 || br.so < 0 || br.si < 0) return Tensor();
    const int64_t batch = bx.outer * bx.inner;
    Tensor out;
    const c10::OptionalDeviceGuard guard(x.device());
    const auto options = x.options().requires_grad(false);
    std::vector<int64_t> shape = x.sizes().vec();
    shape.back() = M;
    out = at::empty(shape, options.dtype(at::kHalf));
    void* const st = stream_of(x);
    const bool half = x.scalar_type() == at::kHalf && right.scalar_type() == at::kHalf;
    const bool scores = half && (mode == BGEMM_MODE_XOR || mode == BGEMM_MODE_AND) && by_rows && scores_in_one(batch, N, M, K);
    const bool context = half && mode == BGEMM_MODE_ATTN_X && by_columns && context_in_one(batch, N, K, M);
    if (scores || context) {
        const int64_t strides[6] = {bx.so, bx.si, x.stride(-2), br.so, br.si, scores ? right.stride(-1) : right.stride(-2)};
        check(scores ? bgemm_scores_forward(mode, x.data_ptr(), right.data_ptr(), strides, batch, bx.inner, N, M, K, out.data_ptr(), st)
                     : bgemm_context_forward(x.data_ptr(), right.data_ptr(), strides, batch, bx.inner, N, K, M, out.data_ptr(), st));
    } else {
        const int64_t wx = bgemm_tiled_words(N, K), wr = bgemm_tiled_words(M, K);
        const Tensor planes = at::empty({batch * (wx + wr)}, options.dtype(at::kInt));
        int32_t* const px = planes.data_ptr<int32_t>();
        int32_t* const pr = px + batch * wx;
        check(bgemm_pack_batched(x.data_ptr(), src_type(x), 0, nullptr, bx.outer, bx.inner, N, K, x.stride(-2), bx.so, bx.si, px, nullptr, st));
        if (by_rows)
            check(bgemm_pack_batched(right.data_ptr(), src_type(right), 0, nullptr, br.outer, br.inner, M, K, right.stride(-1), br.so, br.si, pr, nullptr, st));
        else
            check(bgemm_pack_transposed_batched(right.data_ptr(), src_type(right), br.outer, br.inner, M, K, right.stride(-2), br.so, br.si, pr, st));
        check(bgemm_packed_forward(mode, pr, px, nullptr, out.data_ptr(), BGEMM_OUT_F16, batch, M, N, K, batch > 1 ? wr : 0, batch > 1 ? wx : 0, N * M, 1, BGEMM_VARIANT_AUTO,
                                   nullptr, 0, nullptr, 0, st));
    }
    return out;
}

namespace {

// batched_product(x [.., N, K], right [.., K, M], mode) -> fp16 [.., N, M]
PyObject* batched_product(PyObject*, PyObject* const* args, const Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n == 3, "batched_product takes 3 arguments");
    if (!plain_gpu(args[0]) || !plain_gpu(args[1]) || is_watched()) Py_RETURN_NONE;
    const int mode = (int)PyLong_AsLong(args[2]);
    if (PyErr_Occurred()) throw python_error();
    Tensor out;
    {
        const WithoutGil no_gil;
        out = batched_product_of(tensor_at(args[0]), tensor_at(args[1]), mode);
    }
    if (!out.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// (outer, inner, row) strides of [.., rows, D], zero where there is one of something
void head_view(const Tensor& t, int64_t* s)
{
    s[0] = s[1] = s[2] = 0;
    const int64_t d = t.dim();
    for (int64_t i = 0; i < d - 1; i++)
        if (t.size(i) > 1) s[3 - (d - 1) + i] = t.stride(i);
}

bool head_operand(const Tensor& t)
{
    if (t.scalar_type() != at::kHalf || (t.dim() != 3 && t.dim() != 4) || t.numel() == 0 || t.stride(-1) != 1 || ((uintptr_t)t.data_ptr() & 15)) return false;
    const int64_t D = t.size(-1);
    if (D != 32 && D != 64 && D != 96 && D != 128) return false;
    int64_t s[3];
    head_view(t, s);
    return ((s[0] | s[1] | s[2]) & 7) == 0;
}

// Operands that the gradients' kernels read where they lie, and no more rows than `longest`.
bool grads_in_one(const Tensor& a, const Tensor& b, const int64_t longest)
{
    if (a.device() != b.device() || !head_operand(a) || !head_operand(b)) return false;
    const int64_t N = a.size(-2), M = b.size(-2), batch = a.numel() / (N * a.size(-1));
    return N <= longest && M <= longest && batch * ((N + 63) / 64) * ((M + 63) / 64 + 1) < (int64_t)(1LL << 31) - (1 << 24);
}

// one_launch_grads(matrix, a, b, longest) -> whether the products' gradients go to their kernels (bgemm_linear._one_launch_grads)
PyObject* one_launch_grads(PyObject*, PyObject* const* args, const Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n == 4, "one_launch_grads takes 4 arguments");
    if (c10::GradMode::is_enabled() || is_watched()) Py_RETURN_FALSE;
    for (int i = 0; i < 3; i++)
        if (!plain_gpu(args[i]) || has_tangent(tensor_at(args[i]))) Py_RETURN_FALSE;
    const Tensor &m = tensor_at(args[0]), &a = tensor_at(args[1]), &b = tensor_at(args[2]);
    const int64_t longest = PyLong_AsLongLong(args[3]);
    if (PyErr_Occurred()) throw python_error();
    if (m.scalar_type() != at::kHalf || m.device() != a.device() || !grads_in_one(a, b, longest)) Py_RETURN_FALSE;
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// An uninitialised gradient in the operand's own strides, or dense where those have gaps that end its rows.
Tensor grad_like(const Tensor& t)
{
    const Tensor g = at::empty_like(t);
    return g.stride(-1) == 1 ? g : at::empty_like(t, at::MemoryFormat::Contiguous);
}

// The matrix and the operands of one product, such as its kernel takes.
bool grads_match(const Tensor& m, const Tensor& a, const Tensor& b)
{
    if (!head_operand(a) || !head_operand(b) || a.dim() != b.dim() || a.size(-1) != b.size(-1) || m.scalar_type() != at::kHalf || m.device() != a.device() ||
        b.device() != a.device() || m.dim() != a.dim() || m.size(-2) != a.size(-2) || m.size(-1) != b.size(-2))
        return false;
    for (int64_t i = 0; i < a.dim() - 2; i++)
        if (a.size(i) != b.size(i) || a.size(i) != m.size(i)) return false;
    return true;
}

void launch_grads(const bool context, const Tensor& m0, const Tensor& a, const Tensor& b, const bool need0, const bool need1, Tensor& g0, Tensor& g1)
{
    const c10::OptionalDeviceGuard guard(a.device());
    const Tensor m = context && !need1 ? Tensor() : m0.contiguous();
    int64_t s[12] = {0};
    head_view(a, s);
    head_view(b, s + 3);
    const int64_t inner = a.size(-3), batch = a.dim() == 4 ? a.size(0) * inner : inner, N = a.size(-2), M = b.size(-2), D = a.size(-1);
    if (context) {
        if (need0) g0 = at::empty(m0.sizes(), m0.options().requires_grad(false));
        if (need1) { g1 = grad_like(b); head_view(g1, s + 9); }
        check(bgemm_context_backward(data_or_null(m), a.data_ptr(), b.data_ptr(), s, batch, inner, N, M, D, data_or_null(g0), data_or_null(g1), stream_of(a)));
    } else {
        if (need0) { g0 = grad_like(a); head_view(g0, s + 6); }
        if (need1) { g1 = grad_like(b); head_view(g1, s + 9); }
        check(bgemm_scores_backward(m.data_ptr(), a.data_ptr(), b.data_ptr(), s, batch, inner, N, M, D, data_or_null(g0), data_or_null(g1), stream_of(a)));
    }
}

}  // namespace

bool attention_grads(const bool context, const Tensor& m, const Tensor& a, const Tensor& b, const bool need0, const bool need1, const int64_t longest,
                     const int64_t narrow, const int64_t most, Tensor& g0, Tensor& g1)
{
    if (!is_memory(m) || !is_memory(a) || !is_memory(b) || !grads_match(m, a, b) || !grads_in_one(a, b, longest)) return false;
    if (a.size(-1) > narrow && a.numel() * b.size(-2) >= most) return false;
    launch_grads(context, m, a, b, need0, need1, g0, g1);
    return true;
}

namespace {

// attention_backward(context, m | None, a, b, need a (context: the probabilities), need b) -> (gradient | None, gradient | None); operands
// that one_launch_grads has looked at
PyObject* attention_backward(PyObject*, PyObject* const* args, const Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n == 6, "attention_backward takes 6 arguments");
    const bool context = args[0] == Py_True, need0 = PyObject_IsTrue(args[4]), need1 = PyObject_IsTrue(args[5]);
    for (int i = 1; i < 4; i++)
        if (!plain_gpu(args[i])) Py_RETURN_NONE;
    const Tensor &m = tensor_at(args[1]), &a = tensor_at(args[2]), &b = tensor_at(args[3]);
    if (c10::GradMode::is_enabled() || !grads_match(m, a, b)) Py_RETURN_NONE;
    Tensor g0, g1;
    {
        const WithoutGil no_gil;
        launch_grads(context, m, a, b, need0, need1, g0, g1);
    }
    PyObject* const t = PyTuple_New(2);
    PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(g0));
    PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(g1));
    return t;
    END_HANDLE_TH_ERRORS
}

// attention_forward(q, k, v planes, rows, hidden, batch, heads, fp32, zero point | None) -> (scores, context or its plane)
PyObject* attention_forward(PyObject*, PyObject* const* args, const Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n == 9, "attention_forward takes 9 arguments");
    for (int i = 0; i < 3; i++)
        if (!plain_gpu(args[i])) Py_RETURN_NONE;
    const Tensor &q = tensor_at(args[0]), &k = tensor_at(args[1]), &v = tensor_at(args[2]);
    const int64_t rows = PyLong_AsLongLong(args[3]), hidden = PyLong_AsLongLong(args[4]), batch = PyLong_AsLongLong(args[5]), heads = PyLong_AsLongLong(args[6]);
    const bool f32 = args[7] == Py_True, bits = args[8] != Py_None;
    if (PyErr_Occurred()) throw python_error();
    if (rows < 1 || hidden < 1 || batch < 1 || heads < 1 || rows % batch || hidden % heads || !is_plane(q, q.device(), 1, rows, hidden) ||
        !is_plane(k, q.device(), 1, rows, hidden) || !is_plane(v, q.device(), 1, rows, hidden) || is_watched() || (bits && !exact(args[8])))
        Py_RETURN_NONE;
    const Tensor zp = tensor_or_none(args[8]);
    const at::ScalarType dt = f32 ? at::kFloat : at::kHalf;
    if (bits && (!fits(zp, dt, q.device()) || zp.numel() != 1)) Py_RETURN_NONE;
    const int64_t seq = rows / batch;
    Tensor scores, context;
    {
        const WithoutGil no_gil;
        const c10::OptionalDeviceGuard guard(q.device());
        scores = at::empty({batch, heads, seq, seq}, q.options().dtype(at::kHalf));
        context = bits ? new_plane(q, 1, rows, hidden) : at::empty({batch, seq, hidden}, q.options().dtype(dt));
        const int src = f32 ? BGEMM_SRC_F32 : BGEMM_SRC_F16;
        if (bits)
            check(bgemm_attention_forward_bits(q.data_ptr(), k.data_ptr(), v.data_ptr(), batch, seq, heads, hidden / heads, scores.data_ptr(), context.data_ptr(), zp.data_ptr(), src,
                                               stream_of(q)));
        else
            check(bgemm_attention_forward(q.data_ptr(), k.data_ptr(), v.data_ptr(), batch, seq, heads, hidden / heads, scores.data_ptr(), context.data_ptr(), src, stream_of(q)));
    }
    PyObject* const t = PyTuple_New(2);
    PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(scores));
    PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(context));
    return t;
    END_HANDLE_TH_ERRORS
}

#define BGEMM_FAST(f) (PyCFunction)(void (*)(void))f, METH_FASTCALL

}  // namespace

PyMethodDef infer_methods[] = {
    {"linear_infer", BGEMM_FAST(linear_infer), "a BGEMMLinear without a gradient"},
    {"chain_infer", BGEMM_FAST(chain_infer), "BGEMMLinear layers with only bits between them"},
    {"block_ready", BGEMM_FAST(block_ready), "whether three layers are an attention block's projections"},
    {"rows_bits", BGEMM_FAST(rows_bits), "sign bits of up to three BGEMMLinear layers of one input"},
    {"rows_residual", BGEMM_FAST(rows_residual), "a BGEMMLinear on packed rows plus a residual"},
    {"packed_weight_forward", BGEMM_FAST(packed_weight_forward), "prepacked weights x activations as they are"},
    {"packed_forward", BGEMM_FAST(packed_forward), "GEMM on packed operands"},
    {"f16_forward", BGEMM_FAST(f16_forward), "GEMM on fp16 operands"},
    {"batched_product", BGEMM_FAST(batched_product), "batched product of two binarised operands"},
    {"one_launch_grads", BGEMM_FAST(one_launch_grads), "whether a batched product's gradients go to their one-launch kernel"},
    {"attention_backward", BGEMM_FAST(attention_backward), "gradients of a batched product in one launch"},
    {"attention_forward", BGEMM_FAST(attention_forward), "binary self-attention on packed operands"}};
const int infer_method_count = sizeof infer_methods / sizeof infer_methods[0];

}  // namespace bgemm_native
