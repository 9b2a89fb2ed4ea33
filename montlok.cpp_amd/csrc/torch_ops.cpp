// The operators of montlok._C that make one launch each, from tensors to the C
// ABI of libmlk_hip.so: argument checks (the texts of montlok.cpp:43-65 and the
// operators' own), output allocation and the call, on the current stream.
//
// In Python these steps took 9 to 13 us per operator (27 attribute reads and
// comparisons, torch.cuda.current_stream() 2.8 us, torch.empty 1.8 us, ctypes'
// conversion of 12 to 26 arguments 2 us) against 1.5 us for the launch itself,
// more than most kernels of a small batch run; here the whole call takes about
// 4 us. The library is opened by path at bind(), not linked, so that MLK_HIP_LIB
// selects it here as it does for ctypes.

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/utils/pybind.h>

#include <optional>
#include <stdexcept>
#include <string>
#include <tuple>

#include "../../include/mlk_hip.h"

namespace {
// Arguments taken as Python's int() and float() take them: a count may be any whole number (4.0, a numpy or torch
// scalar), a real anything with a value (the text "1e-5", as YAML reads it, among them).
struct Count {
    int64_t value = 0;
    operator int64_t() const { return value; }
};
struct Real {
    double value = 0.0;
    operator double() const { return value; }
};
bool no_error() {
    const bool failed = PyErr_Occurred() != nullptr;
    if (failed) PyErr_Clear();
    return !failed;
}
}  // namespace

namespace pybind11::detail {
template <>
struct type_caster<Count> {
    PYBIND11_TYPE_CASTER(Count, const_name("int"));
    bool load(handle source, bool) {
        const object whole = reinterpret_steal<object>(PyNumber_Long(source.ptr()));
        const bool same = whole && PyObject_RichCompareBool(source.ptr(), whole.ptr(), Py_EQ) == 1;
        if (same) value.value = PyLong_AsLongLong(whole.ptr());
        return no_error() && same;
    }
};
template <>
struct type_caster<Real> {
    PYBIND11_TYPE_CASTER(Real, const_name("float"));
    bool load(handle source, bool) {
        const object number = reinterpret_steal<object>(PyNumber_Float(source.ptr()));
        if (number) value.value = PyFloat_AsDouble(number.ptr());
        return no_error();
    }
};
}  // namespace pybind11::detail

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

[[noreturn]] void fail(const std::string& message) { throw std::runtime_error(message); }
#define REQUIRE(cond, message) \
    do {                     \
        if (!(cond)) fail(message); \
    } while (0)

#define MLK_FUNCTIONS(X)                                                                                           \
    X(mlk_last_error) X(mlk_rms_norm) X(mlk_add_rms_norm) X(mlk_layer_norm) X(mlk_swiglu) X(mlk_linear)            \
    X(mlk_linear_residual) X(mlk_rms_norm_linear) X(mlk_linear_swiglu) X(mlk_mhc_prepare) X(mlk_mhc_combine) X(mlk_mhc_combine_prepare) \
    X(mlk_mamba3_workspace_bytes) X(mlk_mamba3_siso_forward) X(mlk_mamba3_siso_step)                               \
    X(mlk_rms_norm_mamba3_forward) X(mlk_mla_rope_qk) X(mlk_attention)

struct Library {
#define X(name) decltype(&::name) name = nullptr;
    MLK_FUNCTIONS(X)
#undef X
};
Library lib;

void bind(const std::string& path) {
    void* handle = dlopen(path.c_str(), RTLD_NOW);
    if (handle == nullptr) fail(dlerror());
    Library found;
#define X(name)                                                              \
    found.name = reinterpret_cast<decltype(found.name)>(dlsym(handle, #name)); \
    if (found.name == nullptr) fail(path + " has no symbol " #name);
    MLK_FUNCTIONS(X)
#undef X
    lib = found;
}

void done(mlk_status status) {
    if (status != MLK_OK) fail(lib.mlk_last_error());
}

mlk_stream_t stream() { return c10::hip::getCurrentHIPStream().stream(); }

const Tensor& f32_gpu(const OptTensor& t, const char* name) {
    REQUIRE(t.has_value() && t->defined(), std::string(name) + " must be defined");
    REQUIRE(t->is_cuda(), std::string(name) + " must be on the GPU");
    REQUIRE(t->scalar_type() == at::kFloat, std::string(name) + " must be float32");
    return *t;
}

const float* data(const Tensor& t) { return static_cast<const float*>(t.const_data_ptr()); }
float* out_data(const Tensor& t) { return static_cast<float*>(t.data_ptr()); }
const float* data(const OptTensor& t) { return t.has_value() ? data(*t) : nullptr; }

Tensor dense(const OptTensor& t, int64_t numel, const char* name) {
    f32_gpu(t, name);
    REQUIRE(t->numel() == numel, std::string(name) + " must have " + std::to_string(numel) + " elements, got " + std::to_string(t->numel()));
    return t->contiguous();
}

// A parameter that may be None or empty.
OptTensor dense_or_none(const OptTensor& t, int64_t numel, const char* name) {
    if (!t.has_value() || !t->defined() || t->numel() == 0) return std::nullopt;
    return dense(t, numel, name);
}

Tensor empty(at::IntArrayRef sizes, const Tensor& like) { return at::empty(sizes, at::TensorOptions().dtype(at::kFloat).device(like.device())); }

// [..., dim] as rows of dense floats, like x.reshape(-1, dim) (montlok.cpp:921-924).
struct Rows {
    Tensor t;
    int64_t count, stride;
};
Rows rows_of(const Tensor& x, int64_t dim) {
    if (dim > 0 && x.is_contiguous()) return {x, x.numel() / dim, dim};
    Tensor r = x.reshape({-1, dim});
    if (r.stride(1) != 1 && dim != 1) r = r.contiguous();
    return {r, r.size(0), r.size(0) > 1 ? r.stride(0) : dim};
}

Tensor weight_of(const OptTensor& w, const char* name = "weight") {
    const std::string n(name);
    REQUIRE(w.has_value() && w->defined(), n + " must be defined");
    REQUIRE(w->is_cuda(), n + " must be on the GPU");
    REQUIRE(w->scalar_type() == at::kFloat || w->scalar_type() == at::kBFloat16, n + " must be float32 or bfloat16");
    REQUIRE(w->dim() == 2, n + " must be [out_features, in_features]");
    return w->contiguous();
}
int32_t dtype_of(const Tensor& w) { return w.scalar_type() == at::kBFloat16 ? MLK_DTYPE_BF16 : MLK_DTYPE_F32; }

std::vector<int64_t> with_last(const Tensor& x, int64_t n) {
    std::vector<int64_t> s = x.sizes().vec();
    s.back() = n;
    return s;
}

// ------------------------------------------------------------------ norms

Tensor rms_norm(const OptTensor& x_, const OptTensor& weight, Real eps, Count groups) {
    const Tensor& x = f32_gpu(x_, "x");
    REQUIRE(x.dim() >= 1, "x must have at least one dimension");
    const int64_t dim = x.size(-1);
    REQUIRE(groups > 0 && dim % groups == 0, "groups must divide the normalised dimension");
    const Tensor w = dense(weight, dim, "weight");
    const Rows r = rows_of(x, dim);
    const Tensor out = empty(x.sizes(), x);
    done(lib.mlk_rms_norm(data(r.t), r.count, dim, r.stride, data(w), eps, groups, out_data(out), stream()));
    return out;
}

std::tuple<Tensor, Tensor> add_rms_norm(const OptTensor& left, const OptTensor& right, const OptTensor& weight, Real eps,
                                        Count groups) {
    f32_gpu(left, "left");
    f32_gpu(right, "right");
    REQUIRE(left->sizes() == right->sizes() && left->dim() >= 1, "residual operands must have the same shape");
    const int64_t dim = left->size(-1);
    REQUIRE(groups > 0 && dim % groups == 0, "groups must divide the normalized dimension");
    const Tensor l = left->reshape({-1, dim}).contiguous(), r = right->reshape({-1, dim}).contiguous();
    const Tensor w = dense(weight, dim, "weight");
    const Tensor residual = empty(left->sizes(), *left), normalized = empty(left->sizes(), *left);
    done(lib.mlk_add_rms_norm(data(l), data(r), l.size(0), dim, data(w), eps, groups, out_data(residual), out_data(normalized), stream()));
    return {residual, normalized};
}

Tensor layer_norm(const OptTensor& x_, const OptTensor& weight, const OptTensor& bias, Real eps) {
    const Tensor& x = f32_gpu(x_, "x");
    REQUIRE(x.dim() >= 1, "x must have at least one dimension");
    const int64_t dim = x.size(-1);
    const Tensor w = dense(weight, dim, "weight");
    const OptTensor b = dense_or_none(bias, dim, "bias");
    const Rows r = rows_of(x, dim);
    const Tensor out = empty(x.sizes(), x);
    done(lib.mlk_layer_norm(data(r.t), r.count, dim, r.stride, data(w), data(b), eps, out_data(out), stream()));
    return out;
}

Tensor swiglu(const OptTensor& x_) {
    const Tensor& x = f32_gpu(x_, "x");
    REQUIRE(x.dim() >= 1 && x.size(-1) % 2 == 0, "x must end in an even dimension [gate | up]");
    const int64_t width = x.size(-1), hidden = width / 2;
    const Rows r = rows_of(x, width);
    const Tensor out = empty(with_last(x, hidden), x);
    done(lib.mlk_swiglu(data(r.t), r.count, hidden, r.stride, out_data(out), stream()));
    return out;
}

// ------------------------------------------------------------------ linear

Tensor linear(const OptTensor& input, const OptTensor& weight, const OptTensor& bias) {
    const Tensor& x = f32_gpu(input, "input");
    const Tensor w = weight_of(weight);
    const int64_t n = w.size(0), k = w.size(1);
    REQUIRE(x.dim() >= 1 && x.size(-1) == k, "input must end in in_features=" + std::to_string(k));
    const OptTensor b = dense_or_none(bias, n, "bias");
    const Rows r = rows_of(x, k);
    const Tensor out = empty(with_last(x, n), x);
    done(lib.mlk_linear(data(r.t), r.count, k, r.stride, w.const_data_ptr(), dtype_of(w), data(b), n, out_data(out), n, stream()));
    return out;
}

Tensor linear_residual(const OptTensor& input, const OptTensor& weight, const OptTensor& bias, const OptTensor& residual) {
    const Tensor& x = f32_gpu(input, "input");
    f32_gpu(residual, "residual");
    const Tensor w = weight_of(weight);
    const int64_t n = w.size(0), k = w.size(1);
    REQUIRE(x.dim() >= 1 && x.size(-1) == k, "input must end in in_features=" + std::to_string(k));
    const std::vector<int64_t> shape = with_last(x, n);
    REQUIRE(residual->sizes() == at::IntArrayRef(shape), "residual must have the output's shape");
    const OptTensor b = dense_or_none(bias, n, "bias");
    const Rows r = rows_of(x, k);
    const Tensor res = residual->reshape({r.count, n}).contiguous();
    const Tensor out = empty(shape, x);
    done(lib.mlk_linear_residual(data(r.t), r.count, k, r.stride, w.const_data_ptr(), dtype_of(w), data(b), n, data(res), n,
                                 out_data(out), n, stream()));
    return out;
}

// None where the shape has no fused form.
OptTensor rms_norm_linear(const OptTensor& x_, const OptTensor& norm_weight, Real eps, Count groups, const OptTensor& weight,
                          const OptTensor& bias) {
    const Tensor& x = f32_gpu(x_, "x");
    REQUIRE(x.dim() >= 1, "x must have at least one dimension");
    const int64_t dim = x.size(-1);
    REQUIRE(groups > 0 && dim % groups == 0, "groups must divide the normalised dimension");
    const Tensor nw = dense(norm_weight, dim, "weight");
    const Tensor w = weight_of(weight);
    const int64_t n = w.size(0), k = w.size(1);
    REQUIRE(k == dim, "input must end in in_features=" + std::to_string(k));
    const OptTensor b = dense_or_none(bias, n, "bias");
    const Rows r = rows_of(x, dim);
    const Tensor out = empty(with_last(x, n), x);
    const mlk_status status = lib.mlk_rms_norm_linear(data(r.t), r.count, k, r.stride, data(nw), eps, groups, w.const_data_ptr(),
                                                      dtype_of(w), data(b), n, out_data(out), n, stream());
    if (status == MLK_ERR_UNSUPPORTED) return std::nullopt;
    done(status);
    return out;
}

// swiglu(linear(input, weight, bias)); None where the shape has no fused form.
OptTensor linear_swiglu(const OptTensor& input, const OptTensor& weight, const OptTensor& bias) {
    const Tensor& x = f32_gpu(input, "input");
    const Tensor w = weight_of(weight);
    const int64_t n = w.size(0), k = w.size(1);
    REQUIRE(x.dim() >= 1 && x.size(-1) == k, "input must end in in_features=" + std::to_string(k));
    const OptTensor b = dense_or_none(bias, n, "bias");
    REQUIRE(n % 2 == 0, "x must end in an even dimension [gate | up]");
    const Rows r = rows_of(x, k);
    const Tensor out = empty(with_last(x, n / 2), x);
    const mlk_status status = lib.mlk_linear_swiglu(data(r.t), r.count, k, r.stride, w.const_data_ptr(), dtype_of(w), data(b), n / 2,
                                                    out_data(out), n / 2, stream());
    if (status == MLK_ERR_UNSUPPORTED) return std::nullopt;
    done(status);
    return out;
}

// ------------------------------------------------------------------ mHC

// montlok.cpp:535-557 (StreamsView): [B,L,n,d] or the broadcast [B,L,d] backbone.
struct Streams {
    int64_t B, L, n, d, sd, ts;
};
Streams streams_of(const OptTensor& s_, int64_t n_streams) {
    const Tensor& s = f32_gpu(s_, "streams");
    REQUIRE(s.is_contiguous(), "streams must be contiguous");
    Streams v;
    if (s.dim() == 4) {
        v.n = s.size(2);
        v.sd = v.d = s.size(3);
        REQUIRE(n_streams <= 0 || n_streams == v.n,
              "streams has " + std::to_string(v.n) + " streams, expected " + std::to_string(n_streams));
    } else {
        REQUIRE(s.dim() == 3, "streams must be [B,L,n,d] or a broadcast [B,L,d]");
        REQUIRE(n_streams > 0, "n_streams is required for a broadcast [B,L,d] streams");
        v.n = n_streams;
        v.d = s.size(2);
        v.sd = 0;
    }
    v.B = s.size(0);
    v.L = s.size(1);
    v.ts = v.sd == 0 ? v.d : v.n * v.d;
    REQUIRE(v.n > 0 && v.d > 0, "streams must be non-empty");
    return v;
}

Tensor scalar(const OptTensor& t, const char* name) {
    f32_gpu(t, name);
    REQUIRE(t->numel() == 1, std::string(name) + " must be a scalar");
    return *t;
}

// montlok.cpp:568-649 (mhc_prepare_plan).
struct Prepare {
    Tensor nw, pb, qb, rb, proj, pa, qa, ra;
    OptTensor anw;
};
Prepare prepare_of(int64_t n, int64_t d, const OptTensor& norm_w, const OptTensor& proj_w, const OptTensor& pre_bias,
                   const OptTensor& post_bias, const OptTensor& res_bias, const OptTensor& pre_alpha, const OptTensor& post_alpha,
                   const OptTensor& res_alpha, int64_t iters, const OptTensor& agg_norm_w) {
    REQUIRE(iters >= 0, "sinkhorn_iters must be non-negative");
    Prepare p;
    p.nw = dense(norm_w, d, "dyn_norm.weight");
    p.pb = dense(pre_bias, n, "pre_bias");
    p.qb = dense(post_bias, n, "post_bias");
    p.rb = dense(res_bias, n * n, "res_bias");
    REQUIRE(proj_w.has_value() && proj_w->is_cuda() && proj_w->scalar_type() == at::kDouble && proj_w->is_contiguous(),
          "proj_w must be a contiguous float64 GPU tensor");
    REQUIRE(proj_w->dim() == 2 && proj_w->size(0) == 2 * n + n * n && proj_w->size(1) == d, "proj_w must be [2n + n*n, d]");
    p.proj = *proj_w;
    p.pa = scalar(pre_alpha, "pre_alpha");
    p.qa = scalar(post_alpha, "post_alpha");
    p.ra = scalar(res_alpha, "res_alpha");
    p.anw = dense_or_none(agg_norm_w, d, "agg_norm_w");
    return p;
}

std::tuple<Tensor, Tensor, Tensor, Tensor> mhc_prepare(const OptTensor& streams, const OptTensor& norm_w, Real eps,
                                                       const OptTensor& proj_w, const OptTensor& pre_bias,
                                                       const OptTensor& post_bias, const OptTensor& res_bias,
                                                       const OptTensor& pre_alpha, const OptTensor& post_alpha,
                                                       const OptTensor& res_alpha, Count iters, Count n_streams,
                                                       const OptTensor& agg_norm_w, Real agg_norm_eps) {
    const Streams v = streams_of(streams, n_streams);
    const Prepare p = prepare_of(v.n, v.d, norm_w, proj_w, pre_bias, post_bias, res_bias, pre_alpha, post_alpha, res_alpha, iters, agg_norm_w);
    const Tensor agg = empty({v.B, v.L, v.d}, *streams), pre = empty({v.B, v.L, v.n}, *streams);
    const Tensor post = empty({v.B, v.L, v.n}, *streams), res = empty({v.B, v.L, v.n, v.n}, *streams);
    done(lib.mlk_mhc_prepare(data(*streams), v.B * v.L, v.n, v.d, v.sd, v.ts, data(p.nw), eps,
                             static_cast<const double*>(p.proj.const_data_ptr()), data(p.pb), data(p.qb), data(p.rb), data(p.pa),
                             data(p.qa), data(p.ra), iters, data(p.anw), agg_norm_eps, out_data(agg), out_data(pre), out_data(post),
                             out_data(res), stream()));
    return {agg, pre, post, res};
}

Streams combine_inputs(const OptTensor& streams, const OptTensor& res, const OptTensor& post, const OptTensor& out) {
    const Streams v = streams_of(streams, res.has_value() && res->dim() == 4 ? res->size(-1) : 0);
    f32_gpu(res, "res");
    f32_gpu(post, "post");
    f32_gpu(out, "out");
    REQUIRE(res->sizes() == at::IntArrayRef({v.B, v.L, v.n, v.n}) && res->is_contiguous(), "res must be contiguous [B,L,n,n]");
    REQUIRE(post->sizes() == at::IntArrayRef({v.B, v.L, v.n}) && post->is_contiguous(), "post must be contiguous [B,L,n]");
    REQUIRE(out->sizes() == at::IntArrayRef({v.B, v.L, v.d}) && out->is_contiguous(), "out must be contiguous [B,L,d]");
    return v;
}

Tensor mhc_combine(const OptTensor& streams, const OptTensor& res, const OptTensor& post, const OptTensor& out, bool collapse) {
    const Streams v = combine_inputs(streams, res, post, out);
    const Tensor result = collapse ? empty({v.B, v.L, v.d}, *streams) : empty({v.B, v.L, v.n, v.d}, *streams);
    done(lib.mlk_mhc_combine(data(*streams), v.B * v.L, v.n, v.d, v.sd, v.ts, data(*res), data(*post), data(*out),
                             collapse ? nullptr : out_data(result), collapse ? out_data(result) : nullptr, stream()));
    return result;
}

std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor> mhc_combine_prepare(
    const OptTensor& streams, const OptTensor& res, const OptTensor& post, const OptTensor& out, const OptTensor& norm_w, Real eps,
    const OptTensor& proj_w, const OptTensor& pre_bias, const OptTensor& post_bias, const OptTensor& res_bias,
    const OptTensor& pre_alpha, const OptTensor& post_alpha, const OptTensor& res_alpha, Count iters, const OptTensor& agg_norm_w,
    Real agg_norm_eps, bool reuse_streams, const std::optional<std::tuple<Tensor, Tensor, Tensor, Tensor>>& into) {
    const Streams v = combine_inputs(streams, res, post, out);
    const Prepare p = prepare_of(v.n, v.d, norm_w, proj_w, pre_bias, post_bias, res_bias, pre_alpha, post_alpha, res_alpha, iters, agg_norm_w);
    Tensor fresh, agg, pre_o, post_o, res_o;
    if (reuse_streams) {
        REQUIRE(streams->dim() == 4 && v.sd == v.d && v.ts == v.n * v.d && v.n <= 8,
              "in-place mHC requires contiguous materialised streams with at most eight lanes");
        fresh = *streams;
    } else {
        fresh = empty({v.B, v.L, v.n, v.d}, *streams);
    }
    if (into.has_value()) {
        std::tie(agg, pre_o, post_o, res_o) = *into;
        auto fits = [](const Tensor& t, const std::vector<int64_t>& shape, const char* name) {
            std::string text = "[";
            for (size_t i = 0; i < shape.size(); ++i) text += (i ? ", " : "") + std::to_string(shape[i]);
            REQUIRE(t.scalar_type() == at::kFloat && t.is_contiguous() && t.sizes() == at::IntArrayRef(shape),
                  std::string(name) + " workspace must be contiguous float32 " + text + "]");
        };
        fits(agg, {v.B, v.L, v.d}, "agg");
        fits(pre_o, {v.B, v.L, v.n}, "pre");
        fits(post_o, {v.B, v.L, v.n}, "post");
        fits(res_o, {v.B, v.L, v.n, v.n}, "res");
    } else {
        agg = empty({v.B, v.L, v.d}, *streams);
        pre_o = empty({v.B, v.L, v.n}, *streams);
        post_o = empty({v.B, v.L, v.n}, *streams);
        res_o = empty({v.B, v.L, v.n, v.n}, *streams);
    }
    done(lib.mlk_mhc_combine_prepare(data(*streams), v.B * v.L, v.n, v.d, v.sd, v.ts, data(*res), data(*post), data(*out), data(p.nw),
                                     eps, static_cast<const double*>(p.proj.const_data_ptr()), data(p.pb), data(p.qb), data(p.rb),
                                     data(p.pa), data(p.qa), data(p.ra), iters, data(p.anw), agg_norm_eps, out_data(fresh),
                                     out_data(agg), out_data(pre_o), out_data(post_o), out_data(res_o), stream()));
    return {fresh, agg, pre_o, post_o, res_o};
}

// ------------------------------------------------------------------ Mamba-3

struct Mixer {
    Tensor b_bias, c_bias, b_norm_w, c_norm_w, dt_bias, skip;
};
Mixer mixer_of(const OptTensor& b_bias, const OptTensor& c_bias, const OptTensor& b_norm_w, const OptTensor& c_norm_w,
               const OptTensor& dt_bias, const OptTensor& skip, int64_t d_state, int64_t nheads) {
    return {dense(b_bias, nheads * d_state, "B_bias"), dense(c_bias, nheads * d_state, "C_bias"),
            dense(b_norm_w, d_state, "B_norm.weight"), dense(c_norm_w, d_state, "C_norm.weight"),
            dense(dt_bias, nheads, "dt_bias"), dense(skip, nheads, "D")};
}

void inner_dense(const Tensor& t, const char* name) {
    REQUIRE(t.dim() >= 1 && (t.stride(-1) == 1 || t.size(-1) == 1), std::string(name) + " must be contiguous along its last dimension");
}

Tensor mamba3_siso_forward(const OptTensor& projected_, const OptTensor& gate, const OptTensor& b_bias, const OptTensor& c_bias,
                           const OptTensor& b_norm_w, const OptTensor& c_norm_w, const OptTensor& dt_bias, const OptTensor& skip,
                           int64_t d_state, int64_t ngroups, int64_t nheads, int64_t headdim, int64_t angles, Real b_eps,
                           Real c_eps, Real a_floor) {
    const Tensor& projected = f32_gpu(projected_, "projected");
    const bool logits = !gate.has_value() || gate->numel() == 0;
    if (!logits) f32_gpu(gate, "gate");
    REQUIRE(projected.dim() == 3, "projected must be [B,L,W]");
    REQUIRE(d_state > 0 && ngroups > 0 && nheads > 0 && headdim > 0, "invalid Mamba-3 geometry");
    REQUIRE(nheads % ngroups == 0, "nheads must be divisible by ngroups");
    REQUIRE(angles >= 0 && 2 * angles <= d_state, "num_rope_angles must fit in d_state");
    inner_dense(projected, "projected");
    const int64_t B = projected.size(0), L = projected.size(1), W = projected.size(2), d_inner = nheads * headdim;
    if (!logits) {
        inner_dense(*gate, "gate");
        REQUIRE(gate->sizes() == at::IntArrayRef({B, L, d_inner}), "gate must be [B,L,d_inner]");
    }
    const int64_t expected = 2 * d_inner + 2 * ngroups * d_state + 3 * nheads + angles;
    REQUIRE(W == expected, "projected width " + std::to_string(W) + " does not match the Mamba-3 layout width " + std::to_string(expected));
    const Mixer m = mixer_of(b_bias, c_bias, b_norm_w, c_norm_w, dt_bias, skip, d_state, nheads);
    const Tensor out = empty({B, L, d_inner}, projected);
    const int64_t bytes = static_cast<int64_t>(lib.mlk_mamba3_workspace_bytes(B, L, nheads, d_state, angles));
    const Tensor ws = at::empty({bytes > 4 ? bytes : 4}, at::TensorOptions().dtype(at::kByte).device(projected.device()));
    done(lib.mlk_mamba3_siso_forward(data(projected), B, L, W, projected.stride(0), projected.stride(1), logits ? nullptr : data(*gate),
                                     logits ? 0 : gate->stride(0), logits ? 0 : gate->stride(1), data(m.b_bias), data(m.c_bias),
                                     data(m.b_norm_w), data(m.c_norm_w), data(m.dt_bias), data(m.skip), d_state, ngroups, nheads,
                                     headdim, angles, b_eps, c_eps, a_floor, out_data(out), ws.data_ptr(),
                                     static_cast<size_t>(ws.numel()), stream()));
    return out;
}

Tensor mamba3_siso_step(const OptTensor& projected_, const OptTensor& ssm, const OptTensor& k, const OptTensor& v,
                        const OptTensor& angle, bool started, const OptTensor& b_bias, const OptTensor& c_bias,
                        const OptTensor& b_norm_w, const OptTensor& c_norm_w, const OptTensor& dt_bias, const OptTensor& skip,
                        int64_t d_state, int64_t ngroups, int64_t nheads, int64_t headdim, int64_t angles, Real b_eps,
                        Real c_eps, Real a_floor) {
    const Tensor& projected = f32_gpu(projected_, "projected");
    REQUIRE(projected.dim() == 2, "projected must be [S,W]");
    inner_dense(projected, "projected");
    const int64_t S = projected.size(0), W = projected.size(1), d_inner = nheads * headdim;
    const int64_t expected = 2 * d_inner + 2 * ngroups * d_state + 3 * nheads + angles;
    REQUIRE(W == expected, "projected width " + std::to_string(W) + " does not match the Mamba-3 layout width " + std::to_string(expected));
    auto state = [](const OptTensor& t, const std::vector<int64_t>& shape, const char* key, at::ScalarType type) {
        std::string text = "(";
        for (size_t i = 0; i < shape.size(); ++i) text += (i ? ", " : "") + std::to_string(shape[i]);
        REQUIRE(t.has_value() && t->sizes() == at::IntArrayRef(shape) && t->is_contiguous() && t->is_cuda(),
              std::string("state['") + key + "'] must be a contiguous GPU tensor of shape " + text + ")");
        REQUIRE(t->scalar_type() == type, std::string("state['") + key + "'] has the wrong dtype");
    };
    state(ssm, {S, nheads, d_state, headdim}, "ssm", at::kFloat);
    state(k, {S, nheads, d_state}, "k", at::kFloat);
    state(v, {S, nheads, headdim}, "v", at::kFloat);
    state(angle, {S, nheads, angles > 1 ? angles : 1}, "angle", at::kDouble);
    const Mixer m = mixer_of(b_bias, c_bias, b_norm_w, c_norm_w, dt_bias, skip, d_state, nheads);
    const Tensor out = empty({S, d_inner}, projected);
    done(lib.mlk_mamba3_siso_step(data(projected), S, projected.stride(0), data(m.b_bias), data(m.c_bias), data(m.b_norm_w),
                                  data(m.c_norm_w), data(m.dt_bias), data(m.skip), d_state, ngroups, nheads, headdim, angles, b_eps,
                                  c_eps, a_floor, out_data(*ssm), out_data(*k), out_data(*v), static_cast<double*>(angle->data_ptr()),
                                  started ? 1 : 0, out_data(out), stream()));
    return out;
}

// None where the geometry has no one-launch kernel.
OptTensor rms_norm_mamba3_forward(const OptTensor& inputs, const OptTensor& norm_weight, Real norm_eps, Count norm_groups,
                                  const OptTensor& in_weight, const OptTensor& b_bias, const OptTensor& c_bias,
                                  const OptTensor& b_norm_w, const OptTensor& c_norm_w, const OptTensor& dt_bias,
                                  const OptTensor& skip, int64_t d_state, int64_t ngroups, int64_t nheads, int64_t headdim,
                                  int64_t angles, Real b_eps, Real c_eps, Real a_floor) {
    const Tensor& x = f32_gpu(inputs, "inputs");
    REQUIRE(x.dim() == 3, "inputs must be [B,L,d_model]");
    const int64_t B = x.size(0), L = x.size(1), dm = x.size(2);
    REQUIRE(norm_groups > 0 && dm % norm_groups == 0, "groups must divide the normalised dimension");
    const Tensor nw = dense(norm_weight, dm, "weight");
    const Tensor w = weight_of(in_weight);
    const int64_t d_inner = nheads * headdim, width = 2 * d_inner + 2 * ngroups * d_state + 3 * nheads + angles;
    REQUIRE(w.size(0) == width && w.size(1) == dm, "in_proj weight must be [" + std::to_string(width) + ", " + std::to_string(dm) + "]");
    const Mixer m = mixer_of(b_bias, c_bias, b_norm_w, c_norm_w, dt_bias, skip, d_state, nheads);
    if (x.stride(-1) != 1) return std::nullopt;
    const Tensor out = empty({B, L, d_inner}, x);
    const mlk_status status = lib.mlk_rms_norm_mamba3_forward(
        data(x), B, L, dm, x.stride(0), x.stride(1), data(nw), norm_eps, norm_groups, w.const_data_ptr(), dtype_of(w), data(m.b_bias),
        data(m.c_bias), data(m.b_norm_w), data(m.c_norm_w), data(m.dt_bias), data(m.skip), d_state, ngroups, nheads, headdim, angles,
        b_eps, c_eps, a_floor, out_data(out), stream());
    if (status == MLK_ERR_UNSUPPORTED) return std::nullopt;
    done(status);
    return out;
}

// ------------------------------------------------------------------ MLA

Tensor mla_rope_qk(const OptTensor& q_, const OptTensor& kv_, const OptTensor& k_rope_, const OptTensor& cos_, const OptTensor& sin_,
                   int64_t nope) {
    const Tensor &q = f32_gpu(q_, "q"), &kv = f32_gpu(kv_, "kv"), &kr = f32_gpu(k_rope_, "k_rope");
    const Tensor &cos = f32_gpu(cos_, "cos"), &sin = f32_gpu(sin_, "sin");
    REQUIRE(q.dim() == 4, "q must be [B,Lq,H,head_dim]");
    REQUIRE(kv.dim() == 4 && kv.is_contiguous(), "kv must be contiguous [B,L,H,nope_dim+head_dim]");
    const int64_t batch = q.size(0), q_length = q.size(1), heads = q.size(2), head_dim = q.size(3), length = kv.size(1);
    const int64_t rope = head_dim - nope;
    REQUIRE(nope >= 0 && rope > 0 && rope % 2 == 0, "head_dim - nope_dim must be a positive even rope_dim");
    REQUIRE(1 <= q_length && q_length <= length, "q must cover between 1 and L trailing positions");
    REQUIRE((q.stride(3) == 1 || head_dim == 1) && (q.stride(2) == head_dim || heads == 1) &&
              (q.stride(0) == q_length * q.stride(1) || batch == 1),
          "q must be dense within a token with a uniform token stride");
    REQUIRE(kv.sizes() == at::IntArrayRef({batch, length, heads, nope + head_dim}), "kv must be [B,L,H,nope_dim+head_dim]");
    REQUIRE(kr.sizes() == at::IntArrayRef({batch, length, rope}), "k_rope must be [B,L,rope_dim]");
    REQUIRE((kr.stride(2) == 1 || rope == 1) && (kr.stride(0) == length * kr.stride(1) || batch == 1),
          "k_rope must be dense within a token with a uniform token stride");
    REQUIRE(cos.sizes() == at::IntArrayRef({length, rope}) && cos.is_contiguous(), "cos must be contiguous [L,rope_dim]");
    REQUIRE(sin.sizes() == cos.sizes() && sin.is_contiguous(), "sin must be contiguous [L,rope_dim]");
    const Tensor k = empty({batch, length, heads, head_dim}, q);
    const int64_t q_ts = q_length > 1 || batch == 1 ? q.stride(1) : q.stride(0), kr_ts = length > 1 ? kr.stride(1) : kr.stride(0);
    done(lib.mlk_mla_rope_qk(out_data(q), std::max(q_ts, heads * head_dim), q_length, data(kv), data(kr), std::max(kr_ts, rope),
                             data(cos), data(sin), batch, length, heads, head_dim, nope, out_data(k), stream()));
    return k;
}

// (token stride, head stride) of a [B, L, H, hd] view whose sequences are L tokens apart.
std::pair<int64_t, int64_t> token_strides(const Tensor& t, const char* name) {
    const int64_t B = t.size(0), L = t.size(1), H = t.size(2), hd = t.size(3);
    REQUIRE(t.stride(3) == 1 || hd == 1, std::string(name) + " must be dense in head_dim");
    const int64_t ts = L > 1 ? t.stride(1) : (B > 1 ? t.stride(0) : H * t.stride(2));
    REQUIRE(B == 1 || t.stride(0) == L * ts, std::string(name) + " must have a uniform token stride");
    return {ts, H > 1 ? t.stride(2) : hd};
}

Tensor attention(const OptTensor& q_, const OptTensor& k_, const OptTensor& v_, Count mask, Real scale, bool bf16) {
    const Tensor& q = f32_gpu(q_, "q");
    REQUIRE(q.dim() == 4, "q must be [B,L,H,head_dim]");
    const Tensor& k = f32_gpu(k_, "k");
    REQUIRE(k.dim() == 4, "k must be [B,L,H,head_dim]");
    const Tensor& v = f32_gpu(v_, "v");
    REQUIRE(v.dim() == 4, "v must be [B,L,H,head_dim]");
    const int64_t B = q.size(0), Lq = q.size(1), H = q.size(2), hd = q.size(3), Lk = k.size(1);
    REQUIRE(k.sizes() == at::IntArrayRef({B, Lk, H, hd}) && v.sizes() == at::IntArrayRef({B, Lk, H, hd}), "k and v must be [B,L,H,head_dim]");
    const auto qs = token_strides(q, "q"), ks = token_strides(k, "k"), vs = token_strides(v, "v");
    const Tensor out = empty({B, Lq, H, hd}, q);
    done(lib.mlk_attention(data(q), qs.first, qs.second, data(k), ks.first, ks.second, data(v), vs.first, vs.second, B, H, Lq, Lk, hd,
                           static_cast<int32_t>(mask), scale, bf16 ? MLK_DTYPE_BF16 : MLK_DTYPE_F32, out_data(out), stream()));
    return out;
}

}  // namespace

PYBIND11_MODULE(_torch_ops, m) {
    m.def("bind", &bind);
    m.def("current_stream", [] { return reinterpret_cast<uintptr_t>(stream()); });
    // The operators run without the interpreter's lock: the allocator and a full queue can make a call wait, and
    // other threads have streams of their own to serve.
#define OPERATOR(name) m.def(#name, &name, py::call_guard<py::gil_scoped_release>())
    OPERATOR(rms_norm);
    OPERATOR(add_rms_norm);
    OPERATOR(layer_norm);
    OPERATOR(swiglu);
    OPERATOR(linear);
    OPERATOR(linear_residual);
    OPERATOR(rms_norm_linear);
    OPERATOR(linear_swiglu);
    OPERATOR(mhc_prepare);
    OPERATOR(mhc_combine);
    OPERATOR(mhc_combine_prepare);
    OPERATOR(mamba3_siso_forward);
    OPERATOR(mamba3_siso_step);
    OPERATOR(rms_norm_mamba3_forward);
    OPERATOR(mla_rope_qk);
    OPERATOR(attention);
#undef OPERATOR
}
