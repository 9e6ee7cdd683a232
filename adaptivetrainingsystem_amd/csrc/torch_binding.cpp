// Host side of the calls whose kernels are shorter than a Python wrapper around them: checks, allocation, launch and autograd
// node in one native call.
//
// A normalisation, a rotation or a projection of a decoding step runs 3-15 us on the card; its wrapper in Python, an
// allocation and a foreign call with 8 to 30 arguments took 8-17 us, and a Python node in the backward pass 40 us more on the
// engine's thread.  Every function here serves the ordinary form of its call and returns None for any other (types, strides,
// devices, sizes of nothing, tensor subclasses, tracing, function transforms, forward-mode gradients): the caller then takes the
// general path, which converts, records or raises.  The kernels, their arguments and the results are those of that path.
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include "../../include/ats_gfx950.h"

// An argument that is a torch.Tensor or a Parameter; of any other subclass nothing is taken over (an undefined tensor).
struct Plain : at::Tensor {};
namespace pybind11::detail {
template <>
struct type_caster<Plain> {
    PYBIND11_TYPE_CASTER(Plain, const_name("torch.Tensor"));
    bool load(handle src, bool) {
        if (!THPVariable_Check(src.ptr())) return false;
        if (THPVariable_CheckExact(src.ptr())) static_cast<at::Tensor&>(value) = THPVariable_Unpack(src.ptr());
        return true;
    }
};
}  // namespace pybind11::detail

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

PyObject* g_error = nullptr;      // AtsError

// in_backward: on the engine's thread, whose errors keep their type only as python_error
void check(int rc, const char* what, bool in_backward = false) {
    if (rc == ATS_OK) return;
    pybind11::gil_scoped_acquire gil;
    PyErr_Format(g_error ? g_error : PyExc_RuntimeError, "%s failed with code %d: %s", what, rc, ats_last_error_string());
    if (!in_backward) throw pybind11::error_already_set();
    python_error e;
    e.persist();
    throw e;
}

ats_stream_t stream() { return reinterpret_cast<ats_stream_t>(c10::hip::getCurrentHIPStream().stream()); }
bool served(at::ScalarType t) { return t == at::kFloat || t == at::kBFloat16; }
int tag(const Tensor& t) { return t.scalar_type() == at::kFloat ? ATS_F32 : ATS_BF16; }
bool on_gpu(const Tensor& t) { return t.defined() && t.is_cuda() && t.layout() == at::kStrided; }
// Function transforms (vmap, grad, ..) wrap their tensors, dispatch modes and torch.jit.trace record what is called: the general path
// has its own answer to them (a trace keeps a Python autograd function, of a node in here only its allocation).
bool transformed() {
    using c10::DispatchKey;
    using c10::impl::tls_is_dispatch_key_included;
    return tls_is_dispatch_key_included(DispatchKey::FuncTorchDynamicLayerFrontMode) ||
           tls_is_dispatch_key_included(DispatchKey::Python) || tls_is_dispatch_key_included(DispatchKey::Tracer);
}
bool has_tangent(const Tensor& t) { return t.defined() && t._fw_grad(0).defined(); }
bool wants_grad(const Tensor& a, const Tensor& b) {
    return at::GradMode::is_enabled() && (a.requires_grad() || (b.defined() && b.requires_grad()));
}

// ------------------------------------------------------------------ normalisation
Tensor rmsnorm_fwd(const Tensor& x, const Tensor& w, double eps) {
    const int64_t H = x.size(-1);
    Tensor y = at::empty_like(x);
    check(ats_rmsnorm_fwd(x.data_ptr(), w.defined() ? w.data_ptr() : nullptr, y.data_ptr(), x.numel() / H, (int)H, (float)eps,
                          tag(x), w.defined() ? tag(w) : ATS_F32, stream()), "ats_rmsnorm_fwd");
    return y;
}

struct RMSNormFunction : torch::autograd::Function<RMSNormFunction> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, double eps) {
        ctx->save_for_backward({x, w});
        ctx->saved_data["eps"] = eps;
        return rmsnorm_fwd(x, w, eps);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const Tensor x = saved[0].contiguous(), w = saved[1].defined() ? saved[1].contiguous() : saved[1];
        const Tensor dy = grads[0].to(x.scalar_type()).contiguous();
        const int64_t H = x.size(-1), rows = x.numel() / H;
        const bool need_dw = w.defined() && ctx->needs_input_grad(1);
        Tensor dx = at::empty_like(x), dw, ws;
        size_t bytes = 0;
        if (need_dw) {
            dw = at::empty({H}, x.options().dtype(at::kFloat));
            bytes = ats_rmsnorm_bwd_workspace(rows, (int)H);
            ws = at::empty({(int64_t)(bytes > 0 ? bytes : 1)}, x.options().dtype(at::kByte));
        }
        check(ats_rmsnorm_bwd(x.data_ptr(), w.defined() ? w.data_ptr() : nullptr, dy.data_ptr(), dx.data_ptr(),
                              need_dw ? static_cast<float*>(dw.data_ptr()) : nullptr, rows, (int)H,
                              (float)ctx->saved_data["eps"].toDouble(), tag(x), w.defined() ? tag(w) : ATS_F32,
                              need_dw ? ws.data_ptr() : nullptr, bytes, stream()), "ats_rmsnorm_bwd", true);
        if (need_dw && w.scalar_type() != at::kFloat) dw = dw.to(w.scalar_type());
        return {dx, dw, Tensor()};
    }
};

std::optional<Tensor> rmsnorm(const Plain& input, const std::optional<Plain>& weight, double eps) {
    const Tensor& x = input;      // (a node's inputs are found by their type)
    const Tensor w = weight.has_value() ? static_cast<const Tensor&>(*weight) : Tensor();
    if (!on_gpu(x) || !served(x.scalar_type()) || x.dim() < 1 || x.numel() == 0 || !x.is_contiguous() || transformed()) return {};
    if (has_tangent(x) || has_tangent(w)) return {};
    if (weight.has_value() && (!on_gpu(w) || w.device() != x.device() || !served(w.scalar_type()) || w.numel() != x.size(-1) ||
                        !w.is_contiguous()))
        return {};
    if (wants_grad(x, w)) return RMSNormFunction::apply(x, w, eps);
    at::AutoDispatchBelowADInplaceOrView below;
    return rmsnorm_fwd(x, w, eps);
}

// ------------------------------------------------------------------ rotation
variable_list rotate(const Tensor& q, const Tensor& k, const Tensor& cos, const Tensor& sin, int64_t offset) {
    const int64_t B = q.size(0), Hq = q.size(1), L = q.size(2), D = q.size(3), Hkv = k.size(1);
    Tensor qo = at::empty({B, Hq, L, D}, q.options()), ko = at::empty({B, Hkv, L, D}, k.options());
    check(ats_rope_fwd(q.data_ptr(), k.data_ptr(), qo.data_ptr(), ko.data_ptr(), static_cast<const float*>(cos.data_ptr()),
                       static_cast<const float*>(sin.data_ptr()), (int)cos.stride(0), (int)cos.size(0), (int)B, (int)Hq, (int)Hkv,
                       (int)L, (int)D, (int)offset, q.stride(0), q.stride(1), q.stride(2), k.stride(0), k.stride(1), k.stride(2),
                       tag(q), stream()), "ats_rope_fwd");
    return {qo, ko};
}

// heads behind positions in memory, as projections leave them
bool positions_first(const Tensor& t) { return !t.is_contiguous() && t.transpose(1, 2).is_contiguous(); }
Tensor empty_heads(const Tensor& like, bool positions_first) {
    const int64_t B = like.size(0), h = like.size(1), L = like.size(2), D = like.size(3);
    return positions_first ? at::empty({B, L, h, D}, like.options()).transpose(1, 2) : at::empty({B, h, L, D}, like.options());
}

// The gradients are written in the layout of their inputs: what autograd adds up, or keeps for a leaf, has that layout, and
// from head-major gradients it made it with two copies (q [4, 16, 2048, 128], k [4, 4, 2048, 128] bfloat16: 31 us of 100; the
// pass with the norm beside it 93 -> 65 us).
struct RoPEFunction : torch::autograd::Function<RoPEFunction> {
    static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& cos, const Tensor& sin,
                                 int64_t offset) {
        ctx->save_for_backward({cos, sin});
        ctx->saved_data["offset"] = offset;
        ctx->saved_data["q"] = positions_first(q);
        ctx->saved_data["k"] = positions_first(k);
        return rotate(q, k, cos, sin, offset);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const Tensor dq = grads[0].stride(3) == 1 ? grads[0] : grads[0].contiguous();
        const Tensor dk = grads[1].stride(3) == 1 ? grads[1] : grads[1].contiguous();
        const Tensor gq = empty_heads(dq, ctx->saved_data["q"].toBool()), gk = empty_heads(dk, ctx->saved_data["k"].toBool());
        const void* in[3] = {dq.data_ptr(), dk.data_ptr(), nullptr};
        void* out[3] = {gq.data_ptr(), gk.data_ptr(), nullptr};
        const int64_t is[9] = {dq.stride(0), dq.stride(1), dq.stride(2), dk.stride(0), dk.stride(1), dk.stride(2), 0, 0, 0};
        const int64_t os[9] = {gq.stride(0), gq.stride(1), gq.stride(2), gk.stride(0), gk.stride(1), gk.stride(2), 0, 0, 0};
        const int heads[3] = {(int)dq.size(1), (int)dk.size(1), 0};
        check(ats_rope_strided(in, out, is, os, static_cast<const float*>(saved[0].data_ptr()),
                               static_cast<const float*>(saved[1].data_ptr()), (int)saved[0].stride(0), (int)saved[0].size(0),
                               (int)dq.size(0), heads, (int)dq.size(2), (int)dq.size(3), (int)ctx->saved_data["offset"].toInt(), 1,
                               tag(dq), stream()), "ats_rope_strided", true);
        return {gq, gk, Tensor(), Tensor(), Tensor()};
    }
};

// a table as the kernels read it: float32 rows of unit stride
bool tables_ok(const Tensor& cos, const Tensor& sin) {
    return on_gpu(cos) && on_gpu(sin) && cos.scalar_type() == at::kFloat && sin.scalar_type() == at::kFloat && cos.dim() == 2 &&
           cos.sizes() == sin.sizes() && cos.stride(1) == 1 && sin.stride(1) == 1 && cos.stride(0) == sin.stride(0);
}
bool heads_ok(const Tensor& t) { return on_gpu(t) && t.dim() == 4 && t.numel() > 0 && t.stride(3) == 1 && served(t.scalar_type()); }
bool heads_match(const Tensor& q, const Tensor& k) {
    return k.scalar_type() == q.scalar_type() && k.size(0) == q.size(0) && k.size(2) == q.size(2) && k.size(3) == q.size(3);
}

std::optional<std::tuple<Tensor, Tensor>> rope(const Plain& q_in, const Plain& k_in, const Plain& cos_in, const Plain& sin_in,
                                                   int64_t offset) {
    const Tensor &q = q_in, &k = k_in, &cos = cos_in, &sin = sin_in;
    if (!heads_ok(q) || !heads_ok(k) || !heads_match(q, k) || !tables_ok(cos, sin) || transformed()) return {};
    if (has_tangent(q) || has_tangent(k)) return {};
    if (wants_grad(q, k)) {
        const auto r = RoPEFunction::apply(q, k, cos, sin, offset);
        return std::make_tuple(r[0], r[1]);
    }
    at::AutoDispatchBelowADInplaceOrView below;
    const auto r = rotate(q, k, cos, sin, offset);
    return std::make_tuple(r[0], r[1]);
}

// ------------------------------------------------------------------ the launches of an attention sub-layer, inference
// (their callers have decided that no gradient is wanted)
std::optional<Tensor> rope_append(const Plain& q, const Plain& k, const Plain& v, const Plain& cos, const Plain& sin,
                                  const Plain& k_cache, const Plain& v_cache, int64_t cache_pos, int64_t offset) {
    if (!heads_ok(q) || !heads_ok(k) || !heads_ok(v) || !heads_match(q, k) || v.sizes() != k.sizes() ||
        v.scalar_type() != q.scalar_type() || !tables_ok(cos, sin) || !heads_ok(k_cache) || !heads_ok(v_cache) ||
        k_cache.scalar_type() != q.scalar_type() || v_cache.scalar_type() != q.scalar_type() || v_cache.sizes() != k_cache.sizes() ||
        v_cache.strides() != k_cache.strides() || k_cache.size(0) != q.size(0) || k_cache.size(1) != k.size(1) ||
        k_cache.size(3) != q.size(3) || transformed())
        return {};
    const int64_t B = q.size(0), Hq = q.size(1), L = q.size(2), D = q.size(3);
    at::AutoDispatchBelowADInplaceOrView below;
    Tensor qo = at::empty({B, Hq, L, D}, q.options());
    check(ats_rope_fwd_append(q.data_ptr(), k.data_ptr(), v.data_ptr(), qo.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
                              static_cast<const float*>(cos.data_ptr()), static_cast<const float*>(sin.data_ptr()),
                              (int)cos.stride(0), (int)cos.size(0), (int)B, (int)Hq, (int)k.size(1), (int)L, (int)D, (int)offset,
                              q.stride(0), q.stride(1), q.stride(2), k.stride(0), k.stride(1), k.stride(2), v.stride(0), v.stride(1),
                              v.stride(2), k_cache.stride(0), k_cache.stride(1), k_cache.stride(2), cache_pos, k_cache.size(2),
                              tag(q), stream()), "ats_rope_fwd_append");
    return qo;
}

// x [T, K] against one [N, K] matrix whose address is table[0]; splits as the caller's rule gives them
std::optional<Tensor> linear(const Plain& x, const Tensor& table, const Tensor& start, const Tensor& count, int64_t N, int64_t splits) {
    if (!on_gpu(x) || !served(x.scalar_type()) || x.dim() != 2 || !x.is_contiguous() || x.numel() == 0 || transformed()) return {};
    const int64_t T = x.size(0), K = x.size(1);
    const void* const* b = static_cast<const void* const*>(table.data_ptr());
    const int32_t* rs = static_cast<const int32_t*>(start.data_ptr());
    const int32_t* rc = static_cast<const int32_t*>(count.data_ptr());
    at::AutoDispatchBelowADInplaceOrView below;
    Tensor out = at::empty({T, N}, x.options());
    if (splits > 1) {
        Tensor parts = at::empty({splits, T, N}, x.options().dtype(at::kFloat));
        float* const p = static_cast<float*>(parts.data_ptr());
        check(ats_grouped_down_splitk(x.data_ptr(), b, p, rs, rc, 1, T, T, (int)N, (int)K, (int)splits, tag(x), stream()),
              "ats_grouped_down_splitk");
        check(ats_sum_partials(p, (int)splits, T * N, out.data_ptr(), T * N, tag(x), stream()), "ats_sum_partials");
    } else {
        check(ats_linear_nt(x.data_ptr(), b, out.data_ptr(), rs, rc, T, (int)N, (int)K, tag(x), stream()), "ats_linear_nt");
    }
    return out;
}

// linear of stacked q, k, v weights with splits > 1, its sum fused with rope_append: x [B * L, K] -> rotated q [B, Hq, L, D]
std::optional<Tensor> linear_rope_append(const Plain& x, const Tensor& table, const Tensor& start, const Tensor& count, int64_t splits,
                                         const Plain& cos, const Plain& sin, const Plain& k_cache, const Plain& v_cache,
                                         int64_t cache_pos, int64_t Hq, int64_t L) {
    auto aligned = [](const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; };
    if (!on_gpu(x) || !served(x.scalar_type()) || x.dim() != 2 || !x.is_contiguous() || x.numel() == 0 || !tables_ok(cos, sin) ||
        !heads_ok(k_cache) || !heads_ok(v_cache) || k_cache.scalar_type() != x.scalar_type() ||
        v_cache.scalar_type() != x.scalar_type() || v_cache.sizes() != k_cache.sizes() || v_cache.strides() != k_cache.strides() ||
        k_cache.size(0) * L != x.size(0) || k_cache.size(3) % 8 || k_cache.stride(0) % 4 || k_cache.stride(1) % 4 ||
        k_cache.stride(2) % 4 || cos.stride(0) % 4 || !aligned(k_cache) || !aligned(v_cache) || !aligned(cos) || !aligned(sin) ||
        transformed())
        return {};
    const int64_t T = x.size(0), K = x.size(1), B = k_cache.size(0), Hkv = k_cache.size(1), D = k_cache.size(3);
    const int64_t N = (Hq + 2 * Hkv) * D;
    at::AutoDispatchBelowADInplaceOrView below;
    Tensor qo = at::empty({B, Hq, L, D}, x.options());
    Tensor parts = at::empty({splits, T, N}, x.options().dtype(at::kFloat));
    float* const p = static_cast<float*>(parts.data_ptr());
    check(ats_grouped_down_splitk(x.data_ptr(), static_cast<const void* const*>(table.data_ptr()), p,
                                  static_cast<const int32_t*>(start.data_ptr()), static_cast<const int32_t*>(count.data_ptr()), 1, T, T,
                                  (int)N, (int)K, (int)splits, tag(x), stream()), "ats_grouped_down_splitk");
    check(ats_rope_sum_append(p, (int)splits, T * N, qo.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
                              static_cast<const float*>(cos.data_ptr()), static_cast<const float*>(sin.data_ptr()),
                              (int)cos.stride(0), (int)cos.size(0), (int)B, (int)Hq, (int)Hkv, (int)L, (int)D, k_cache.stride(0),
                              k_cache.stride(1), k_cache.stride(2), cache_pos, k_cache.size(2), tag(x), stream()),
          "ats_rope_sum_append");
    return qo;
}

// causal attention without masks, dropout or log-sum-exp
std::optional<Tensor> attention(const Plain& q, const Plain& k, const Plain& v, double scale, bool split_keys) {
    if (!heads_ok(q) || !heads_ok(k) || !heads_ok(v) || q.scalar_type() != at::kBFloat16 || k.scalar_type() != q.scalar_type() ||
        v.scalar_type() != q.scalar_type() || v.sizes() != k.sizes() || k.size(0) != q.size(0) || k.size(3) != q.size(3) ||
        q.size(1) % k.size(1) != 0 || k.size(2) < q.size(2) || !q.is_contiguous() || transformed())
        return {};
    const int64_t B = q.size(0), Hq = q.size(1), L = q.size(2), D = q.size(3), Hkv = k.size(1), Lk = k.size(2);
    auto aligned = [](const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; };
    if (k.stride(2) != D || k.stride(0) % 8 || k.stride(1) % 8 || !aligned(k) || v.stride(0) % 8 || v.stride(1) % 8 ||
        v.stride(2) % 8 || v.stride(2) < D || !aligned(v))
        return {};
    at::AutoDispatchBelowADInplaceOrView below;
    Tensor out = at::empty({B, L, Hq * D}, q.options()), ws;
    const size_t bytes = split_keys ? ats_attention_fwd_workspace((int)B, (int)Hq, (int)Hkv, (int)L, (int)Lk, (int)D) : 0;
    if (bytes) ws = at::empty({(int64_t)bytes}, q.options().dtype(at::kByte));
    check(ats_attention_fwd_ex(q.data_ptr(), k.data_ptr(), k.stride(0), k.stride(1), v.data_ptr(), v.stride(0), v.stride(2),
                               v.stride(1), nullptr, nullptr, 0, 0, 0.f, 0, out.data_ptr(), nullptr, (int)B, (int)Hq, (int)Hkv,
                               (int)L, (int)Lk, (int)D, (float)scale, bytes ? ws.data_ptr() : nullptr, bytes, stream()),
          "ats_attention_fwd_ex");
    return out;
}

// causal attention of a prompt on its stacked projections qkv [B * L, (Hq + 2 Hkv) * D]: keys rotated (with the values beside them:
// the prompt's cache), queries rotated as the attention loads them -> out, k, v
std::optional<std::tuple<Tensor, Tensor, Tensor>> prompt_attention(const Plain& qkv, const Plain& cos, const Plain& sin, int64_t B,
                                                                   int64_t Hkv, int64_t D, double scale, bool keep_values) {
    auto aligned = [](const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; };
    if (!on_gpu(qkv) || qkv.scalar_type() != at::kBFloat16 || !qkv.is_contiguous() || !tables_ok(cos, sin) || cos.stride(0) % 4 ||
        !aligned(qkv) || !aligned(cos) || !aligned(sin) || transformed())
        return {};
    const int64_t L = qkv.size(0) / B, N = qkv.size(1), Hq = N / D - 2 * Hkv;
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor rows = qkv.view({B, L, N / D, D}).transpose(1, 2);
    const Tensor k_in = rows.narrow(1, Hq, Hkv), v_in = rows.narrow(1, Hq + Hkv, Hkv);
    const Tensor k = at::empty({B, Hkv, L, D}, qkv.options());
    const Tensor v = keep_values ? at::empty({B, Hkv, L, D}, qkv.options()) : v_in;
    const float* const c = static_cast<const float*>(cos.data_ptr());
    const float* const s = static_cast<const float*>(sin.data_ptr());
    const void* in[3] = {nullptr, k_in.data_ptr(), v_in.data_ptr()};
    void* to[3] = {nullptr, k.data_ptr(), v.data_ptr()};
    const int64_t is[9] = {0, 0, 0, L * N, D, N, L * N, D, N}, os[9] = {0, 0, 0, Hkv * L * D, L * D, D, Hkv * L * D, L * D, D};
    const int heads[3] = {0, (int)Hkv, keep_values ? (int)Hkv : 0};
    check(ats_rope_strided(in, to, is, os, c, s, (int)cos.stride(0), (int)cos.size(0), (int)B, heads, (int)L, (int)D, 0, 0, tag(qkv),
                           stream()), "ats_rope_strided");
    Tensor out = at::empty({B, L, Hq * D}, qkv.options());
    check(ats_attention_fwd_rope(qkv.data_ptr(), L * N, D, N, c, s, (int)cos.stride(0), (int)cos.size(0), k.data_ptr(), k.stride(0),
                                 k.stride(1), v.data_ptr(), v.stride(0), v.stride(2), v.stride(1), out.data_ptr(), (int)B, (int)Hq,
                                 (int)Hkv, (int)L, (int)L, (int)D, (float)scale, stream()), "ats_attention_fwd_rope");
    return std::make_tuple(out, k, v);
}

}  // namespace

// The interpreter lock is released through every call, as ctypes releases it: other threads run while a launch waits for a full
// queue.  (check takes it again to raise.)
PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.def("set_error", [](pybind11::object e) { g_error = e.release().ptr(); });
    auto def = [&m](const char* name, auto function) { m.def(name, function, pybind11::call_guard<pybind11::gil_scoped_release>()); };
    def("rmsnorm", &rmsnorm);
    def("rope", &rope);
    def("rope_append", &rope_append);
    def("linear", &linear);
    def("linear_rope_append", &linear_rope_append);
    def("attention", &attention);
    def("prompt_attention", &prompt_attention);
}
