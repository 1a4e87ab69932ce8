// The host side of the Python entry points for arrays that are already as the kernels take them (on the GPU, dense, one
// element type): argument checks, buffers, launches and the autograd rules in one native call.  The same path in Python
// took 23 us for a forward and 105 to 210 us for a forward and backward, more than the kernels of a small call; here it
// is about a third of that.  Everything else (other layouts and types, function transforms, error messages) stays in
// gla.py, which calls this again once the arrays are converted, and whose backward rules are called where a transform is active.
#include <ATen/TracerMode.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <ATen/ops/zeros.h>
#include <ATen/ops/zeros_like.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/utils/pybind.h>

#include <optional>

#include "../../include/gla_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// A status of the library as gla_jax_amd._lib.GlaError.  The Python error itself is thrown: out of a backward the autograd
// engine carries it to the caller as it is, while any exception of this file's own would arrive as a plain RuntimeError.
PyObject *gla_error = nullptr;
void check(const char *fn, int status)
{
    if (status == 0) return;
    const py::gil_scoped_acquire gil;
    PyErr_SetObject(gla_error, py::handle(gla_error)(fn, status, gla_status_string(status)).ptr());
    throw py::error_already_set();
}

void *stream_of(const Tensor &t)
{
    return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

bool known(at::ScalarType s) { return s == at::kFloat || s == at::kBFloat16; }
gla_dtype code(const Tensor &t) { return t.scalar_type() == at::kFloat ? GLA_F32 : GLA_BF16; }
bool dense_on_gpu(const Tensor &t) { return t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.is_contiguous(); }

struct Dims {
    int64_t B, T, H, D;
};
Dims dims_of(const Tensor &k)
{
    const auto s = k.sizes();
    const size_t n = s.size();
    int64_t B = 1;
    for (size_t i = 0; i + 3 < n; ++i) B *= s[i];
    return {B, s[n - 3], s[n - 2], s[n - 1]};
}

// The arrays can go to the kernels as they are: see gla.py's _prep for the contract.
bool canonical_rows(const Tensor &g, const Tensor &v, const Tensor &k, const Tensor &q)
{
    for (const Tensor *t : {&g, &v, &k, &q})
        if (!dense_on_gpu(*t) || t->device() != k.device()) return false;
    const auto s = k.sizes();
    if (s.size() < 3 || q.sizes() != s || g.sizes() != s || v.sizes() != s) return false;
    return g.scalar_type() == at::kFloat && known(v.scalar_type()) && k.scalar_type() == v.scalar_type() &&
           q.scalar_type() == v.scalar_type();
}
std::vector<int64_t> state_sizes(const Tensor &k)
{
    std::vector<int64_t> s = k.sizes().vec();
    const size_t n = s.size();
    s[n - 3] = s[n - 2];
    s[n - 2] = s[n - 1];
    return s;
}
bool canonical(const Tensor &h0, const Tensor &g, const Tensor &v, const Tensor &k, const Tensor &q)
{
    return canonical_rows(g, v, k, q) && dense_on_gpu(h0) && h0.device() == k.device() && known(h0.scalar_type()) &&
           h0.sizes() == at::IntArrayRef(state_sizes(k));
}

Tensor bytes_like(size_t n, const Tensor &t) { return at::empty({(int64_t)n}, t.options().dtype(at::kByte)); }

[[noreturn]] void no_double_backward(const char *name)
{
    TORCH_CHECK_NOT_IMPLEMENTED(false, name, ": second-order gradients are not provided (the reference defines first-order "
                                             "custom_vjp rules only)");
    std::abort();
}

// The call goes through the autograd function: a gradient may be asked for, or an array carries a forward-mode tangent,
// which the function refuses (a call past it would drop the tangent without a word).
bool wants_grad(const Tensor &h0, const Tensor &g, const Tensor &v, const Tensor &k, const Tensor &q)
{
    for (const Tensor *t : {&h0, &g, &v, &k, &q})
        if ((at::GradMode::is_enabled() && t->requires_grad()) || t->_fw_grad(/*level=*/0).defined()) return true;
    return false;
}

// ---- chunk_gla ----------------------------------------------------------------------------------
struct ChunkOut {
    Tensor hT, out, states;
};
ChunkOut chunk_forward(const Tensor &h0, const Tensor &g, const Tensor &v, const Tensor &k, const Tensor &q, int64_t chunk,
                       bool residual)
{
    const c10::DeviceGuard guard(k.device());
    const Dims d = dims_of(k);
    const gla_dtype dt = code(v);
    const size_t nws = gla_chunk_fwd_workspace_bytes(d.B, d.T, d.H, d.D, d.D, chunk, dt);
    const size_t nst = residual ? gla_chunk_states_bytes(d.B, d.T, d.H, d.D, d.D, chunk, dt) : 0;
    if (nws == 0) check("gla_chunk_fwd", GLA_ERR_UNSUPPORTED);
    ChunkOut r{at::empty_like(h0), at::empty_like(v), Tensor()};
    // as B rows of bytes, which is how gla.py's rules map them
    if (residual) r.states = at::empty({d.B, (int64_t)(nst + d.B - 1) / d.B}, v.options().dtype(at::kByte));
    const Tensor ws = bytes_like(nws, v);
    check("gla_chunk_fwd",
          gla_chunk_fwd(stream_of(k), d.B, d.T, d.H, d.D, d.D, chunk, dt, code(h0), h0.data_ptr(), (const float *)g.data_ptr(),
                        v.data_ptr(), k.data_ptr(), q.data_ptr(), r.hT.data_ptr(), r.out.data_ptr(),
                        residual ? r.states.data_ptr() : nullptr, ws.data_ptr(), nws));
    return r;
}

variable_list chunk_backward(const Tensor &states, const Tensor &g, const Tensor &v, const Tensor &k, const Tensor &q,
                             const Tensor &dhT, const Tensor &dout, int64_t chunk)
{
    const c10::DeviceGuard guard(k.device());
    const Dims d = dims_of(k);
    const gla_dtype dt = code(v);
    const size_t nws = gla_chunk_bwd_workspace_bytes(d.B, d.T, d.H, d.D, d.D, chunk, dt);
    const Tensor ws = bytes_like(nws, v);
    Tensor dh0 = at::empty_like(dhT), dg = at::empty_like(g), dv = at::empty_like(v), dk = at::empty_like(k),
           dq = at::empty_like(q);
    check("gla_chunk_bwd",
          gla_chunk_bwd(stream_of(k), d.B, d.T, d.H, d.D, d.D, chunk, dt, code(dhT), (const float *)g.data_ptr(), v.data_ptr(),
                        k.data_ptr(), q.data_ptr(), states.data_ptr(), dhT.data_ptr(), dout.data_ptr(), dh0.data_ptr(),
                        (float *)dg.data_ptr(), dv.data_ptr(), dk.data_ptr(), dq.data_ptr(), ws.data_ptr(), nws));
    return {dh0, dg, dv, dk, dq};
}

// What autograd saved: a saved-tensor hook may hand it back in another layout (taken as it is, the kernels would read other
// values), or as another array altogether (refused).
void check_saved(bool as_saved)
{
    TORCH_CHECK(as_saved, "a saved-tensor hook handed back an array of another type, shape or device");
}
variable_list saved_dense(AutogradContext *ctx)
{
    variable_list s = ctx->get_saved_variables();
    for (Tensor &t : s)
        if (t.defined() && !t.is_contiguous()) t = t.contiguous();
    return s;
}
bool holds(const Tensor &bytes, size_t n, const Tensor &like)
{
    return bytes.scalar_type() == at::kByte && bytes.device() == like.device() && (size_t)bytes.numel() >= n;
}
// A function transform can be active in the backward alone (torch.func.vmap over torch.autograd.grad): the cotangents then
// are wrappers without memory of their own, and the rules of gla.py, which know how to map, take over.  The older mapping
// behind is_grads_batched reaches no rule of a custom function.
bool transforms_active()
{
    return c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}
// a cotangent as the kernels take it: zeros where autograd has none, dense, in the type of what it belongs to
Tensor cotangent(const Tensor &d, at::IntArrayRef sizes, at::ScalarType type, const Tensor &like)
{
    if (!d.defined()) return at::zeros(sizes, like.options().dtype(type));
    check_saved(d.sizes() == sizes && d.device() == like.device());
    TORCH_CHECK_NOT_IMPLEMENTED(d.has_storage() || transforms_active(), "batched cotangents (is_grads_batched, jacobian with "
                                "vectorize=True) are not provided: map torch.autograd.grad by torch.func.vmap");
    // (each operation on a tensor that changes nothing costs a microsecond of a small step's hundred)
    return d.scalar_type() == type && d.is_contiguous() ? d : d.to(type).contiguous();
}

template <typename... Args> variable_list python_rule(const char *name, Args &&...args)
{
    const py::gil_scoped_acquire gil;
    const py::object r = py::module_::import("gla_jax_amd.gla").attr(name).attr("apply")(std::forward<Args>(args)...);
    return r.cast<variable_list>();
}

// The backward rules as functions of their own, used where a graph of the gradients is asked for: what they return can
// be differentiated no further, and says so.
struct ChunkBackward : torch::autograd::Function<ChunkBackward> {
    static variable_list forward(AutogradContext *, const Tensor &states, const Tensor &g, const Tensor &v, const Tensor &k,
                                 const Tensor &q, const Tensor &dhT, const Tensor &dout, int64_t chunk)
    {
        return chunk_backward(states, g, v, k, q, dhT, dout, chunk);
    }
    static variable_list backward(AutogradContext *, variable_list) { no_double_backward("chunk_gla"); }
};

struct Chunk : torch::autograd::Function<Chunk> {      // gla.py:483-550, 552-625
    static variable_list forward(AutogradContext *ctx, const Tensor &h0, const Tensor &g, const Tensor &v, const Tensor &k,
                                 const Tensor &q, int64_t chunk)
    {
        ChunkOut r = chunk_forward(h0, g, v, k, q, chunk, true);
        ctx->save_for_backward({r.states, g, v, k, q});      // residuals of gla.py:542-549
        ctx->saved_data["chunk"] = chunk;
        ctx->saved_data["hidden"] = (int64_t)h0.scalar_type();
        ctx->set_materialize_grads(false);
        return {r.hT, r.out};
    }
    static variable_list backward(AutogradContext *ctx, variable_list d)
    {
        const variable_list s = saved_dense(ctx);
        const int64_t chunk = ctx->saved_data["chunk"].toInt();
        check_saved(canonical_rows(s[1], s[2], s[3], s[4]));
        const Dims n = dims_of(s[3]);
        check_saved(holds(s[0], gla_chunk_states_bytes(n.B, n.T, n.H, n.D, n.D, chunk, code(s[2])), s[3]));
        const Tensor dhT = cotangent(d[0], state_sizes(s[3]), (at::ScalarType)ctx->saved_data["hidden"].toInt(), s[3]);
        const Tensor dout = cotangent(d[1], s[2].sizes(), s[2].scalar_type(), s[2]);
        variable_list r = transforms_active() ? python_rule("_ChunkGLABwd", s[0], s[1], s[2], s[3], s[4], dhT, dout, chunk)
                          : at::GradMode::is_enabled() ? ChunkBackward::apply(s[0], s[1], s[2], s[3], s[4], dhT, dout, chunk)
                                                       : chunk_backward(s[0], s[1], s[2], s[3], s[4], dhT, dout, chunk);
        r.emplace_back();
        return r;
    }
};

// ---- recurrent_gla ------------------------------------------------------------------------------
// residual: what the forward can leave for the backward (undefined where sequences run whole), if that is wanted
std::pair<Tensor, Tensor> recurrent_forward(const Tensor &h0, const Tensor &g, const Tensor &v, const Tensor &k,
                                            const Tensor &q, bool reverse, bool out_fp32, Tensor *residual = nullptr)
{
    const c10::DeviceGuard guard(k.device());
    const Dims d = dims_of(k);
    const gla_dtype dt = code(v);
    Tensor hT = at::empty_like(h0), out = out_fp32 ? at::empty_like(v, v.options().dtype(at::kFloat)) : at::empty_like(v), ws;
    // a workspace where the library can use one (head dimension 256, few sequences)
    const size_t nws = gla_recurrent_fwd_workspace_bytes(d.B, d.T, d.H, d.D, d.D, dt);
    if (nws) ws = bytes_like(nws, v);
    const size_t nres = residual ? gla_recurrent_residual_bytes(d.B, d.T, d.H, d.D, d.D, dt) : 0;
    if (nres) *residual = bytes_like(nres, v);
    check("gla_recurrent_fwd_res",
          gla_recurrent_fwd_res(stream_of(k), d.B, d.T, d.H, d.D, d.D, dt, code(h0), out_fp32 ? GLA_F32 : dt, reverse,
                               h0.data_ptr(), (const float *)g.data_ptr(), v.data_ptr(), k.data_ptr(), q.data_ptr(),
                               hT.data_ptr(), out.data_ptr(), nres ? residual->data_ptr() : nullptr,
                               nws ? ws.data_ptr() : nullptr, nws));
    return {hT, out};
}

variable_list recurrent_backward(const Tensor &h0, const Tensor &g, const Tensor &v, const Tensor &k, const Tensor &q,
                                 const Tensor &hT, const Tensor &residual, const Tensor &dhT, const Tensor &dout, bool reverse,
                                 bool out_fp32)
{
    const c10::DeviceGuard guard(k.device());
    const Dims d = dims_of(k);
    const gla_dtype dt = code(v);
    Tensor dh0 = at::empty_like(h0), dg = at::empty_like(g), dv = at::empty_like(v), dk = at::empty_like(k),
           dq = at::empty_like(q), ws;
    const size_t nws = gla_recurrent_bwd_workspace_bytes(d.B, d.T, d.H, d.D, d.D, dt);
    if (nws) ws = bytes_like(nws, v);
    check("gla_recurrent_bwd_res",
          gla_recurrent_bwd_res(stream_of(k), d.B, d.T, d.H, d.D, d.D, dt, code(h0), out_fp32 ? GLA_F32 : dt, reverse,
                               h0.data_ptr(), (const float *)g.data_ptr(), v.data_ptr(), k.data_ptr(), q.data_ptr(),
                               hT.data_ptr(), dhT.data_ptr(), dout.data_ptr(), dh0.data_ptr(), (float *)dg.data_ptr(),
                               dv.data_ptr(), dk.data_ptr(), dq.data_ptr(), residual.defined() ? residual.data_ptr() : nullptr,
                               nws ? ws.data_ptr() : nullptr, nws));
    return {dh0, dg, dv, dk, dq};
}

struct RecurrentBackward : torch::autograd::Function<RecurrentBackward> {
    static variable_list forward(AutogradContext *, const Tensor &h0, const Tensor &g, const Tensor &v, const Tensor &k,
                                 const Tensor &q, const Tensor &hT, const std::optional<Tensor> &residual, const Tensor &dhT,
                                 const Tensor &dout, bool reverse, bool out_fp32)
    {
        return recurrent_backward(h0, g, v, k, q, hT, residual.value_or(Tensor()), dhT, dout, reverse, out_fp32);
    }
    static variable_list backward(AutogradContext *, variable_list) { no_double_backward("recurrent_gla"); }
};

struct Recurrent : torch::autograd::Function<Recurrent> {      // gla.py:99-170, 172-269
    static variable_list forward(AutogradContext *ctx, const Tensor &h0, const Tensor &g, const Tensor &v, const Tensor &k,
                                 const Tensor &q, bool reverse, bool out_fp32)
    {
        Tensor residual;
        auto [hT, out] = recurrent_forward(h0, g, v, k, q, reverse, out_fp32, &residual);
        ctx->save_for_backward({h0, g, v, k, q, hT, residual});          // residuals of gla.py:169, and the segments' states
        ctx->saved_data["reverse"] = reverse;
        ctx->saved_data["out_fp32"] = out_fp32;
        ctx->set_materialize_grads(false);
        return {hT, out};
    }
    static variable_list backward(AutogradContext *ctx, variable_list d)
    {
        const variable_list s = saved_dense(ctx);
        check_saved(canonical(s[0], s[1], s[2], s[3], s[4]) && dense_on_gpu(s[5]) && s[5].sizes() == s[0].sizes());
        const Dims n = dims_of(s[3]);
        check_saved(!s[6].defined() || holds(s[6], gla_recurrent_residual_bytes(n.B, n.T, n.H, n.D, n.D, code(s[2])), s[3]));
        const bool reverse = ctx->saved_data["reverse"].toBool(), out_fp32 = ctx->saved_data["out_fp32"].toBool();
        const Tensor dhT = cotangent(d[0], s[0].sizes(), s[0].scalar_type(), s[0]);
        const Tensor dout = cotangent(d[1], s[2].sizes(), out_fp32 ? at::kFloat : s[2].scalar_type(), s[2]);
        variable_list r = transforms_active()
                              ? python_rule("_RecurrentGLABwd", s[0], s[1], s[2], s[3], s[4], s[5], dhT, dout, reverse, out_fp32)
                          : at::GradMode::is_enabled()
                              ? RecurrentBackward::apply(s[0], s[1], s[2], s[3], s[4], s[5], std::optional<Tensor>(s[6]), dhT, dout, reverse, out_fp32)
                              : recurrent_backward(s[0], s[1], s[2], s[3], s[4], s[5], s[6], dhT, dout, reverse, out_fp32);
        r.resize(7);
        return r;
    }
};

// ---- module -------------------------------------------------------------------------------------
typedef std::optional<std::vector<Tensor>> Result;       // none: not for this path

// A tracer records an autograd function of Python's as a call of it; of a native call it would record the buffers that are
// allocated here, and replay those.
bool traced() { return at::tracer::impl::is_dispatch_enabled(); }

Result chunk(const Tensor &h0, const Tensor &g, const Tensor &v, const Tensor &k, const Tensor &q, int64_t size)
{
    if (traced() || !canonical(h0, g, v, k, q) || size <= 0 || (size & (size - 1)) || dims_of(k).T % size) return std::nullopt;
    if (wants_grad(h0, g, v, k, q)) return Chunk::apply(h0, g, v, k, q, size);
    ChunkOut r = chunk_forward(h0, g, v, k, q, size, false);
    return std::vector<Tensor>{r.hT, r.out};
}

Result recurrent(const Tensor &h0, const Tensor &g, const Tensor &v, const Tensor &k, const Tensor &q, bool reverse,
                 bool out_fp32)
{
    if (traced() || !canonical(h0, g, v, k, q) || k.size(-1) < 16) return std::nullopt;
    if (wants_grad(h0, g, v, k, q)) return Recurrent::apply(h0, g, v, k, q, reverse, out_fp32);
    auto [hT, out] = recurrent_forward(h0, g, v, k, q, reverse, out_fp32);
    return std::vector<Tensor>{hT, out};
}

bool plain_f32(const Tensor &t) { return dense_on_gpu(t) && t.scalar_type() == at::kFloat; }

std::optional<Tensor> cumsum(const Tensor &src, int64_t axis, const std::optional<Tensor> &init, bool reverse)
{
    const int64_t n = src.dim();
    if (!plain_f32(src) || axis < 0 || axis >= n) return std::nullopt;
    int64_t outer = 1, inner = 1;
    for (int64_t i = 0; i < axis; ++i) outer *= src.size(i);
    for (int64_t i = axis + 1; i < n; ++i) inner *= src.size(i);
    if (outer < 1 || outer > 65535) return std::nullopt;
    if (init) {
        if (!plain_f32(*init) || init->dim() != n - 1 || init->device() != src.device()) return std::nullopt;
        for (int64_t i = 0; i < n - 1; ++i)
            if (init->size(i) != src.size(i < axis ? i : i + 1)) return std::nullopt;
    }
    const c10::DeviceGuard guard(src.device());
    Tensor dst = at::empty_like(src), ws;
    const size_t nws = gla_cumsum_workspace_bytes(outer, src.size(axis), inner);
    if (nws) ws = bytes_like(nws, src);
    check("gla_cumsum_f32", gla_cumsum_f32_ws(stream_of(src), (const float *)src.data_ptr(),
                                              init ? (const float *)init->data_ptr() : nullptr, (float *)dst.data_ptr(), outer,
                                              src.size(axis), inner, reverse, nws ? ws.data_ptr() : nullptr, nws));
    return dst;
}

std::optional<std::pair<Tensor, Tensor>> rnn(const Tensor &a, const Tensor &b, const std::optional<Tensor> &ia,
                                             const std::optional<Tensor> &ib, bool reverse)
{
    const int64_t n = b.dim();
    if (!plain_f32(a) || !plain_f32(b) || (n != 3 && n != 4) || a.dim() != n - 1 || a.device() != b.device()) return std::nullopt;
    for (int64_t i = 0; i < n - 1; ++i)
        if (a.size(i) != b.size(i)) return std::nullopt;
    if ((bool)ia != (bool)ib) return std::nullopt;
    const int64_t B = n == 4 ? b.size(0) : 1, T = b.size(n - 3), K = b.size(n - 2), V = b.size(n - 1);
    // the initial pair is read as B rows of K (and K x V) whatever its shape: the number of values is what has to fit
    if (ia && (!plain_f32(*ia) || !plain_f32(*ib) || ia->numel() != B * K || ib->numel() != B * K * V ||
               ia->device() != b.device() || ib->device() != b.device()))
        return std::nullopt;
    const c10::DeviceGuard guard(b.device());
    Tensor oa = at::empty_like(a), ox = at::empty_like(b);
    check("gla_rnn_scan_f32",
          gla_rnn_scan_f32(stream_of(b), (const float *)a.data_ptr(), (const float *)b.data_ptr(),
                           ia ? (const float *)ia->data_ptr() : nullptr, ib ? (const float *)ib->data_ptr() : nullptr,
                           (float *)oa.data_ptr(), (float *)ox.data_ptr(), B, T, K, V, reverse));
    return std::make_pair(oa, ox);
}

}  // namespace

PYBIND11_MODULE(_gla_torch, m)
{
    gla_error = py::object(py::module_::import("gla_jax_amd._lib").attr("GlaError")).release().ptr();
    typedef py::call_guard<py::gil_scoped_release> NoGil;
    m.def("chunk", &chunk, NoGil());
    m.def("recurrent", &recurrent, NoGil());
    m.def("cumsum", &cumsum, NoGil());
    m.def("rnn", &rnn, NoGil());
}
