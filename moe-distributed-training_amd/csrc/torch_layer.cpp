// The autograd side of the package in C++: the layer, the expert MLP, a single grouped projection and the router as
// torch::autograd functions over the C ABI of libmoe_hip.so (include/moe_hip.h).  No device code and no arithmetic here:
// shape checks, allocation of outputs and interims, and the order of the library calls, all on the current stream.
//
// Why native: a small layer step enqueues some twenty kernels of a few microseconds each; with the same sequence in Python
// the host spent about 10 us per library call (argument conversion, allocation, stream lookup, the interpreter lock of the
// backward thread) and the GPU waited for it.
#include <torch/extension.h>
#include <torch/library.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/utils/pybind.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include "../../include/moe_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;
using OptTensor = std::optional<Tensor>;

// Python's assert statements of the reference's entry points: an AssertionError there, and here
struct AssertionFailure : torch::PyTorchError {
    explicit AssertionFailure(const std::string& m) : PyTorchError(m) {}
    PyObject* python_type() override { return PyExc_AssertionError; }
};
#define MOE_ASSERT(cond, msg) do { if (!(cond)) throw AssertionFailure(msg); } while (0)

inline void check(int status, const char* what)
{
    TORCH_CHECK(status == MOE_OK, what, " failed: ", moe_hip_strerror(status), " (status ", status, ")");
}

inline int dtype_code(const Tensor& t)
{
    switch (t.scalar_type()) {
    case at::kBFloat16: return MOE_BF16;
    case at::kHalf: return MOE_F16;
    case at::kFloat: return MOE_F32;
    default: TORCH_CHECK_TYPE(false, "unsupported dtype ", t.scalar_type(), ": the HIP kernels take bfloat16, float16 or float32");
    }
}

inline int is64(const Tensor& t)
{
    if (t.scalar_type() == at::kLong) return 1;
    TORCH_CHECK_TYPE(t.scalar_type() == at::kInt, "index tensors must be int32 or int64, got ", t.scalar_type());
    return 0;
}

inline void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
inline void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

inline void require_gpu(std::initializer_list<const Tensor*> ts)
{
    const Tensor* first = nullptr;
    for (const Tensor* t : ts) {
        if (!t->defined()) continue;
        TORCH_CHECK(t->has_storage(), "function transforms (torch.func, vmap) are not supported: their tensors hold no memory that a kernel could read");
        TORCH_CHECK(t->is_cuda(), "moe_distributed_training_amd runs on the GPU only (got a CPU tensor); there is no host fallback");
        if (!first) first = t;
        TORCH_CHECK(t->device() == first->device(), "all tensors must live on the same device");
    }
}

// gates (T, k): one weight per row of the product; the combine takes its sizes from them
inline void check_gates(const Tensor& gates, int64_t rows)
{
    TORCH_CHECK(!gates.defined() || (gates.dim() == 2 && gates.numel() == rows), "gates of ", gates.defined() ? gates.sizes() : at::IntArrayRef(),
                " must be (tokens, experts per token) with one weight for each of the ", rows, " assignments");
}

// inclusive row counts: the kernels read one per expert
inline void check_offsets(const Tensor& offsets, int64_t E)
{
    TORCH_CHECK(offsets.numel() >= E, "expert offsets of ", offsets.sizes(), " do not cover ", E, " experts");
}

inline Tensor bytes_on(const Tensor& like, size_t n)
{
    return at::empty({(int64_t)(n < 256 ? 256 : n)}, like.options().dtype(at::kByte));
}

// the gate weights one after the other, as the kernels read them (a saved-tensor hook may hand them back with strides that a reshape keeps)
inline Tensor flat_gates(const Tensor& g) { return g.defined() ? g.reshape({-1}).contiguous() : Tensor(); }

inline Tensor unit_inner(const Tensor& t) { return t.stride(-1) == 1 ? t : t.contiguous(); }

// Whether the call has to go through its autograd node: a gradient is recorded, or an input carries a forward-mode tangent
// (which the node refuses; the plain sequence of library calls would drop it).
inline bool needs_node(std::initializer_list<const Tensor*> ts)
{
    const bool grad = at::GradMode::is_enabled();
    for (const Tensor* t : ts)
        if (t->defined() && ((grad && t->requires_grad()) || t->_fw_grad(0).defined())) return true;
    return false;
}

inline Tensor val(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }
// (an autograd function takes an absent tensor as an empty optional, not as an undefined tensor)
inline OptTensor opt(const Tensor& t) { return t.defined() ? OptTensor(t) : OptTensor(); }

// ---------------------------------------------------------------------------------------------------------------
// library calls with their allocations
// ---------------------------------------------------------------------------------------------------------------
Tensor combine(const Tensor& y, const Tensor& gates, const int32_t* inv, int64_t k, int64_t T, const float* extra_coef = nullptr,
               const Tensor& extra_rows = Tensor(), int64_t n_extra = 0)
{
    Tensor out = at::empty({T, y.size(1)}, y.options());
    check(moe_combine(ptr(y), y.stride(0), ptr(out), out.stride(0), ptr(gates), gates.defined() ? dtype_code(gates) : 0, inv, (int)k, T, y.size(1),
                      dtype_code(y), extra_coef, ptr(extra_rows), extra_rows.defined() ? extra_rows.stride(0) : 0, (int)n_extra, stream_of(y)),
          "moe_combine");
    return out;
}

Tensor combine_dgates(const Tensor& y, const Tensor& dout, int64_t k, at::ScalarType dt, const int32_t* inv)
{
    Tensor dg = at::empty({dout.size(0), k}, y.options().dtype(dt));
    check(moe_combine_dgates(ptr(y), y.stride(0), ptr(dout), dout.stride(0), ptr(dg), dtype_code(dg), inv, (int)k, dout.size(0), y.size(1),
                             dtype_code(y), stream_of(y)), "moe_combine_dgates");
    return dg;
}

Tensor group_rows(const Tensor& src, const void* pos, int pos64, int64_t n, int64_t fan_out, const Tensor& coeff = Tensor())
{
    Tensor out = at::empty({n, src.size(1)}, src.options());
    check(moe_group_rows(ptr(src), src.stride(0), ptr(out), out.stride(0), pos, pos64, (int)fan_out, ptr(coeff),
                         coeff.defined() ? dtype_code(coeff) : 0, n, src.size(1), dtype_code(src), stream_of(src)), "moe_group_rows");
    return out;
}

Tensor group_bwd_w(const Tensor& dy, const Tensor& x, const void* offsets, int off64, int64_t E)
{
    Tensor dw = at::empty({E, x.size(1), dy.size(1)}, dy.options());
    check(moe_group_bwd_w(ptr(dy), dy.stride(0), dy.stride(1), ptr(x), x.stride(0), x.stride(1), ptr(dw), dw.stride(0), dw.stride(1), dw.stride(2),
                          offsets, off64, (int)E, x.size(0), x.size(1), dy.size(1), dtype_code(dy), stream_of(dy)), "moe_group_bwd_w");
    return dw;
}

Tensor scatter2scatter(const Tensor& X, const Tensor& W, const Tensor& A, const Tensor& B, double scaling, const Tensor& ssi, const Tensor& eo,
                       int64_t k, bool x_grouped, bool y_grouped, const Tensor& into = Tensor())
{
    const int64_t L = ssi.size(0), E = W.size(0), K = W.size(1), N = W.size(2);
    const int rank = A.defined() ? (int)A.size(2) : 0;
    Tensor out = into.defined() ? into : at::empty({L, N}, X.options());
    if (L == 0) return out;
    Tensor ws = bytes_on(X, moe_scatter2scatter_workspace_bytes(L, (int)E, K, N, rank));
    auto st = [](const Tensor& t, int i) { return t.defined() ? t.stride(i) : (int64_t)0; };
    check(moe_scatter2scatter(ptr(X), X.stride(0), X.stride(1), ptr(W), W.stride(0), W.stride(1), W.stride(2), ptr(A), st(A, 0), st(A, 1), st(A, 2),
                              ptr(B), st(B, 0), st(B, 1), st(B, 2), rank, (float)scaling, ptr(out), out.stride(0), out.stride(1), ptr(ssi), is64(ssi),
                              ptr(eo), is64(eo), (int)E, L, K, N, (int)k, x_grouped, y_grouped, dtype_code(X), ptr(ws), (size_t)ws.numel(), stream_of(X)),
          "moe_scatter2scatter");
    return out;
}

Tensor offsets_from_sorted(const Tensor& sei, int64_t E)
{
    Tensor s = sei.contiguous(), out = at::empty({E}, s.options());
    check(moe_expert_offsets(ptr(s), is64(s), s.numel(), (int)E, ptr(out), is64(out), stream_of(s)), "moe_expert_offsets");
    return out;
}

// ---------------------------------------------------------------------------------------------------------------
// adapters: the six factors as views (E, K, r) / (E, r, N), or in the storage of the block module --
// A.weight (E*hidden, r) and B.weight (E*ffn, r) per projection, w2's factors swapped (megablocks_utils/peft_utils.py:37-38,68-70)
// ---------------------------------------------------------------------------------------------------------------
struct Lora {
    const void* p[6] = {};
    int64_t s[18] = {};
    int rank = 0;
    const void* const* ptrs() const { return rank ? p : nullptr; }
    const int64_t* strides() const { return rank ? s : nullptr; }
};

// order a1, b1, a3, b3, a2, b2
Lora describe_lora(const Tensor* t, bool storage, int64_t d, int64_t f)
{
    Lora l;
    if (!t[0].defined()) return l;
    l.rank = (int)t[0].size(-1);
    const int64_t r = l.rank;
    for (int i = 0; i < 6; ++i) {
        int64_t* s = l.s + 3 * i;
        l.p[i] = t[i].data_ptr();
        if (!storage) { for (int j = 0; j < 3; ++j) s[j] = t[i].stride(j); continue; }
        const bool on_ffn = i == 1 || i == 3 || i == 4;        // b1, b3 and a2 live in (E*ffn, r) storage
        s[0] = (on_ffn ? f : d) * r;
        const bool a_like = i % 2 == 0;                        // (E, K, r): k stride r, rank stride 1; else (E, r, N)
        s[1] = a_like ? r : 1;
        s[2] = a_like ? 1 : r;
    }
    return l;
}

// (E, f, d), or in the storage of the block module (E*f, d): the launches take the sizes of all three from E, f and d
void check_expert_weight(const Tensor& w, int64_t E, int64_t f, int64_t d)
{
    const bool fits = w.dim() == 3 ? w.size(0) == E && w.size(1) == f && w.size(2) == d : w.dim() == 2 && w.size(0) == E * f && w.size(1) == d;
    TORCH_CHECK(fits, "expert weights of ", w.sizes(), " do not fit ", E, " experts of ", f, " x ", d);
}

// The six factors, all of the rank of the first: views (E, K, r) / (E, r, N), or the block's storage.  The launches take every extent
// from E, f, d and that rank, and the gradients are allocated like the factors.
void check_factors(const Tensor* t, bool storage, int64_t E, int64_t f, int64_t d)
{
    if (!t[0].defined()) return;
    const int64_t rank = t[0].dim() ? t[0].size(-1) : 0;
    for (int i = 0; i < 6; ++i) {
        const bool on_ffn = i == 1 || i == 3 || i == 4, a_like = i % 2 == 0;
        const int64_t rows = on_ffn ? f : d;
        const bool fits = t[i].defined() && (storage ? t[i].dim() >= 2 && t[i].size(-1) == rank && t[i].numel() == E * rows * rank
                                                     : t[i].dim() == 3 && t[i].size(0) == E && t[i].size(a_like ? 1 : 2) == rows && t[i].size(a_like ? 2 : 1) == rank);
        TORCH_CHECK(fits, "adapter factor of ", t[i].defined() ? t[i].sizes() : at::IntArrayRef(), " does not fit ", E, " experts of ", rows,
                    " rows and rank ", rank);
    }
}

// what the fused launches take (the same limits the library checks before it enqueues anything)
bool fast_path_ok(const Tensor& x, const Tensor& w1, const Tensor& w2, const Tensor& w3, const Tensor* lora, bool storage, int64_t E, int64_t d,
                  int64_t f)
{
    (void)E;
    if (x.scalar_type() != at::kBFloat16 && x.scalar_type() != at::kHalf) return false;
    if (w1.scalar_type() != x.scalar_type() || w2.scalar_type() != x.scalar_type() || w3.scalar_type() != x.scalar_type()) return false;
    const bool has = lora[0].defined();
    for (int i = 0; i < 6 && has; ++i)
        if (lora[i].scalar_type() != x.scalar_type() || (storage && !lora[i].is_contiguous())) return false;
    if (d % 64 || f % 64 || x.stride(-1) != 1 || x.stride(0) % 8) return false;
    if (!w1.is_contiguous() || !w2.is_contiguous() || !w3.is_contiguous()) return false;
    if (has && lora[0].size(-1) > 128) return false;   // up to eight 16-wide rank chunks
    // gathered activation rows and one expert's matrix are addressed with 32-bit byte offsets
    return (x.size(0) * x.stride(0) + d) * 2 < ((int64_t)1 << 32) && (f * d + d) * 2 < ((int64_t)1 << 32);
}

// lora: empty, or six factors in the order a1, b1, a3, b3, a2, b2
void take_factors(const std::vector<Tensor>& lora, Tensor* t)
{
    TORCH_CHECK(lora.empty() || lora.size() == 6, "an expert MLP has six adapter factors, got ", lora.size());
    for (size_t i = 0; i < lora.size(); ++i) t[i] = lora[i];
}

struct MlpShape { int64_t E, d, f, R; int fan_out; double scaling; };

struct MlpOut { Tensor gate, up, h, y, saved; };

// save: keep gate, up (only the backward pass reads them)
MlpOut mlp_forward(const Tensor& x, const Tensor& w1, const Tensor& w3, const Tensor& w2, const Lora& lora, const MlpShape& s, const void* ssi,
                   int ssi64, const void* offsets, int off64, bool y_grouped, bool save)
{
    MlpOut o;
    if (save) {
        o.gate = at::empty({s.R, s.f}, x.options());
        o.up = at::empty({s.R, s.f}, x.options());
    }
    o.h = at::empty({s.R, s.f}, x.options());
    o.y = at::empty({s.R, s.d}, x.options());
    o.saved = bytes_on(x, moe_mlp_saved_bytes(s.R, lora.rank));
    Tensor ws = bytes_on(x, moe_mlp_workspace_bytes(s.R, (int)s.E, s.d, s.f, lora.rank));
    check(moe_mlp_fwd(ptr(x), x.stride(0), ptr(w1), ptr(w3), ptr(w2), lora.ptrs(), lora.strides(), lora.rank, (float)s.scaling, ptr(o.gate), ptr(o.up),
                      ptr(o.h), ptr(o.y), o.y.stride(0), ssi, ssi64, offsets, off64, (int)s.E, s.R, s.d, s.f, s.fan_out, y_grouped, dtype_code(x),
                      ptr(o.saved), ptr(ws), (size_t)ws.numel(), stream_of(x)), "moe_mlp_fwd");
    return o;
}

struct MlpGrads { Tensor dx_rows, dgate, dup, lora[6]; };

MlpGrads mlp_backward(const Tensor& dy, bool dy_grouped, int64_t dy_fan_out, const float* row_scale, const Tensor& x, const Tensor& w1, const Tensor& w3,
                      const Tensor& w2, const Tensor* lora_t, const Lora& lora, const MlpShape& s, const Tensor& gate, const Tensor& up, const Tensor& h,
                      const Tensor& saved, const void* ssi, int ssi64, const void* offsets, int off64)
{
    MlpGrads g;
    g.dgate = at::empty({s.R, s.f}, x.options());
    g.dup = at::empty({s.R, s.f}, x.options());
    g.dx_rows = at::empty({s.R, s.d}, x.options());
    Tensor ws = bytes_on(x, moe_mlp_workspace_bytes(s.R, (int)s.E, s.d, s.f, lora.rank));
    void* gp[6] = {};
    int64_t gs[18] = {};
    if (lora.rank)
        for (int i = 0; i < 6; ++i) {
            g.lora[i] = at::empty_like(lora_t[i]);   // storage and, for views, strides of the factor
            gp[i] = g.lora[i].data_ptr();
            for (int j = 0; j < 3; ++j) gs[3 * i + j] = g.lora[i].dim() == 3 ? g.lora[i].stride(j) : lora.s[3 * i + j];
        }
    check(moe_mlp_bwd(ptr(dy), dy.stride(0), dy_grouped, (int)dy_fan_out, row_scale, ptr(x), x.stride(0), ptr(w1), ptr(w3), ptr(w2), lora.ptrs(),
                      lora.strides(), lora.rank ? gp : nullptr, lora.rank ? gs : nullptr, lora.rank, (float)s.scaling, ptr(gate), ptr(up), ptr(h),
                      ptr(g.dgate), ptr(g.dup), ptr(g.dx_rows), g.dx_rows.stride(0), 0, ssi, ssi64, offsets, off64, (int)s.E, s.R, s.d, s.f, s.fan_out,
                      dtype_code(x), ptr(saved), ptr(ws), (size_t)ws.numel(), stream_of(x)), "moe_mlp_bwd");
    return g;
}

// Gradients of the stored (E, f, d) expert weights (full fine-tuning; the reference gets them from scattermoe's group_bwd_W):
// dW2[e] = h_e^T dy_e, dW1[e] = dgate_e^T x_e, dW3[e] = dup_e^T x_e over each expert's rows -- already in the storage
// orientation.  coeff: the per-assignment gate weights folded into dy (or undefined).
void base_weight_grads(const bool* needs /* w1, w3, w2 */, const Tensor& x, const Tensor& dy, bool dy_grouped, int64_t dy_fan_out, const Tensor& coeff,
                       const MlpGrads& g, const Tensor& h, const void* ssi, int ssi64, const void* offsets, int off64, const MlpShape& s, Tensor* dw)
{
    if (needs[0] || needs[1]) {
        Tensor x_g = group_rows(x, ssi, ssi64, s.R, s.fan_out);
        if (needs[0]) dw[0] = group_bwd_w(x_g, g.dgate, offsets, off64, s.E);
        if (needs[1]) dw[1] = group_bwd_w(x_g, g.dup, offsets, off64, s.E);
    }
    if (needs[2]) dw[2] = group_bwd_w(dy_grouped ? dy : group_rows(dy, ssi, ssi64, s.R, dy_fan_out, coeff), h, offsets, off64, s.E);
}

// ---------------------------------------------------------------------------------------------------------------
// router
// ---------------------------------------------------------------------------------------------------------------
Tensor router_input_grad(const Tensor& dlogits, const Tensor& weight, at::ScalarType dt)
{
    Tensor w = unit_inner(weight.scalar_type() == dt ? weight : weight.to(dt));
    const int64_t T = dlogits.size(0);
    Tensor out = at::empty({T, w.size(1)}, w.options());
    check(moe_combine(nullptr, 0, ptr(out), out.stride(0), nullptr, 0, nullptr, 0, T, w.size(1), dtype_code(out), (const float*)ptr(dlogits), ptr(w),
                      w.stride(0), (int)dlogits.size(1), stream_of(w)), "moe_combine (router input gradient)");
    return out;
}

Tensor router_weight_grad(const Tensor& x, const Tensor& dlogits)
{
    const int64_t T = x.size(0), d = x.size(1), E = dlogits.size(1);
    Tensor out = at::empty({E, d}, x.options());
    Tensor ws = bytes_on(x, moe_router_weight_grad_workspace_bytes(T, d, (int)E));
    check(moe_router_weight_grad(ptr(x), x.stride(0), (const float*)ptr(dlogits), ptr(out), out.stride(0), T, d, (int)E, dtype_code(x), ptr(ws),
                                 (size_t)ws.numel(), stream_of(x)), "moe_router_weight_grad");
    return out;
}

struct RouterOut { Tensor scores, weights, indices; };

RouterOut router_outputs(const Tensor& x, const Tensor& wg, int64_t k)
{
    const int64_t T = x.size(0), E = wg.size(0);
    MOE_ASSERT(wg.scalar_type() == x.scalar_type() && wg.size(1) == x.size(1), "router weight and input do not fit");
    MOE_ASSERT(k >= 1 && k <= E, "top_k must be between 1 and the number of experts");
    const auto f32 = x.options().dtype(at::kFloat);
    return {at::empty({T, E}, f32), at::empty({T, k}, f32), at::empty({T, k}, x.options().dtype(at::kInt))};
}

RouterOut router_forward(const Tensor& x, const Tensor& wg, int64_t k, bool normalize)
{
    const int64_t T = x.size(0), d = x.size(1), E = wg.size(0);
    RouterOut o = router_outputs(x, wg, k);
    Tensor logits = at::empty_like(o.scores);
    check(moe_router_forward(ptr(x), x.stride(0), ptr(wg), wg.stride(0), dtype_code(x), (float*)ptr(logits), (float*)ptr(o.scores), (float*)ptr(o.weights),
                             (int32_t*)ptr(o.indices), T, d, (int)E, (int)k, normalize, stream_of(x)), "moe_router_forward");
    return o;
}

Tensor router_topk_bwd(const Tensor& dw, const Tensor& weights_, const Tensor& indices_, const Tensor& scores_, bool normalize)
{
    const Tensor weights = weights_.contiguous(), indices = indices_.contiguous(), scores = scores_.contiguous();   // (as in flat_gates)
    Tensor d = dw.contiguous().to(at::kFloat), dl = at::empty_like(scores);
    check(moe_router_topk_bwd((const float*)ptr(d), (const float*)ptr(weights), (const int32_t*)ptr(indices), (const float*)ptr(scores), (float*)ptr(dl),
                              scores.size(0), (int)scores.size(1), (int)weights.size(1), normalize, stream_of(scores)), "moe_router_topk_bwd");
    return dl;
}

struct RouterFn : Function<RouterFn> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& wg, int64_t k, bool normalize)
    {
        RouterOut o = router_forward(x, wg, k, normalize);
        ctx->save_for_backward({x, wg, o.scores, o.weights, o.indices});
        ctx->saved_data["normalize"] = normalize;
        ctx->mark_non_differentiable({o.indices});
        ctx->set_materialize_grads(false);
        return {o.scores, o.weights, o.indices};
    }
    static variable_list backward(AutogradContext* ctx, variable_list g)
    {
        const auto sv = ctx->get_saved_variables();
        const Tensor &x = sv[0], &wg = sv[1], &scores = sv[2], &w = sv[3], &idx = sv[4];
        const c10::DeviceGuard guard(x.device());
        Tensor dl = router_topk_bwd(g[1].defined() ? g[1] : at::zeros_like(w), w, idx, scores, ctx->saved_data["normalize"].toBool());
        if (g[0].defined()) {
            // softmax backward for a gradient that reaches the full score matrix (e.g. an auxiliary loss)
            Tensor ds = g[0].to(at::kFloat);
            dl = dl + scores * (ds - (ds * scores).sum(-1, true));
        }
        return {ctx->needs_input_grad(0) ? router_input_grad(dl, wg, x.scalar_type()) : Tensor(),
                ctx->needs_input_grad(1) ? router_weight_grad(x, dl) : Tensor(), Tensor(), Tensor()};
    }
};

variable_list router(const Tensor& x_, const Tensor& wg_, int64_t k, bool normalize)
{
    require_gpu({&x_, &wg_});
    TORCH_CHECK(x_.dim() == 2 && wg_.dim() == 2, "the router takes (tokens, hidden size) and a weight of (experts, hidden size), got ", x_.sizes(), " and ", wg_.sizes());
    const c10::DeviceGuard guard(x_.device());
    Tensor x = unit_inner(x_), wg = unit_inner(wg_);
    if (needs_node({&x, &wg})) return RouterFn::apply(x, wg, k, normalize);
    RouterOut o = router_forward(x, wg, k, normalize);
    return {o.scores, o.weights, o.indices};
}

// ---------------------------------------------------------------------------------------------------------------
// one grouped projection, with or without adapters: scattermoe_utils/parallel_linear_lora.py:11-149 of the reference
// ---------------------------------------------------------------------------------------------------------------
struct LinearCfg { double scaling, scaling_ab; int64_t k; bool grouped_in, grouped_out; };   // scaling_ab: of the adapters' gradients

Tensor linear_rows(const Tensor& x, const Tensor& W, const Tensor& A, const Tensor& B, const Tensor& ssi, const Tensor& eo, const LinearCfg& c)
{
    return scatter2scatter(x, W, A, B, c.scaling, ssi, eo, c.k, c.grouped_in, c.grouped_out);
}

struct LinearFn : Function<LinearFn> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& W, const OptTensor& A_, const OptTensor& B_, const OptTensor& gates_,
                          const Tensor& ssi, const Tensor& eo, const LinearCfg& c)
    {
        const Tensor A = val(A_), B = val(B_), gates = val(gates_);
        Tensor y = linear_rows(x, W, A, B, ssi, eo, c), y_rows;
        if (gates.defined()) {   // rows of y are token-major (t*k+j): weighted sum of each token's k rows (reference :30-35)
            y_rows = y;
            y = combine(y_rows, gates, nullptr, gates.size(1), gates.size(0));
        }
        ctx->save_for_backward({x, W, A, B, gates, ssi, eo, y_rows});
        ctx->saved_data["scaling"] = c.scaling;
        ctx->saved_data["scaling_ab"] = c.scaling_ab;
        ctx->saved_data["k"] = c.k;
        ctx->saved_data["flags"] = (int64_t)(c.grouped_in | (c.grouped_out << 1));
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list g)
    {
        const auto sv = ctx->get_saved_variables();
        const Tensor &x = sv[0], &W = sv[1], &A = sv[2], &B = sv[3], &gates = sv[4], &ssi = sv[5], &eo = sv[6], &y_rows = sv[7];
        const c10::DeviceGuard guard(x.device());
        const double scaling = ctx->saved_data["scaling"].toDouble();
        const int64_t k = ctx->saved_data["k"].toInt(), flags = ctx->saved_data["flags"].toInt(), E = W.size(0), L = ssi.size(0);
        const bool grouped_in = flags & 1, grouped_out = flags & 2;
        MOE_ASSERT(k >= 1, "no gradients without assignments per row of X");
        MOE_ASSERT(!grouped_out || g[0].size(0) == L, "gates combine rows in token order: no gradients for them with a grouped output");
        Tensor dout = g[0].contiguous(), d_gates, coeff, dA, dB, dW;
        int64_t gate_fan = 1;
        if (gates.defined()) {
            d_gates = combine_dgates(y_rows, dout, gates.size(1), gates.scalar_type(), nullptr);   // reference :70-72
            coeff = flat_gates(gates);
            gate_fan = gates.size(1);
        }
        // All of it from the rows where they lie.  What the matrix-core paths do not take by its type or sizes goes on below before anything is
        // allocated for them (fp16 with gates: see moe_linear_lora_bwd), what they refuse by its strides or alignment after.
        const bool by_type = x.scalar_type() == at::kBFloat16 || (x.scalar_type() == at::kHalf && !gates.defined());
        const size_t ws_bytes = by_type && A.defined() && !grouped_in && !grouped_out && scaling == ctx->saved_data["scaling_ab"].toDouble() && L > 0 && W.numel() > 0
                                    ? moe_linear_lora_bwd_workspace_bytes(L, (int)E, x.size(1), W.size(2), (int)A.size(2)) : 0;
        if (ws_bytes) {
            const int64_t K = x.size(1), N = W.size(2), r = A.size(2);
            dA = at::empty({E, K, r}, dout.options());
            dB = at::empty({E, r, N}, dout.options());
            Tensor dx = at::empty({L, K}, x.options()), ws = bytes_on(x, ws_bytes);
            const int rc = moe_linear_lora_bwd(ptr(dout), dout.stride(0), (int)gate_fan, ptr(coeff), gates.defined() ? dtype_code(gates) : 0, ptr(x), x.stride(0), (int)k, ptr(W), W.stride(0),
                                               W.stride(1), W.stride(2), ptr(A), A.stride(0), A.stride(1), A.stride(2), ptr(B), B.stride(0), B.stride(1), B.stride(2),
                                               (int)r, (float)scaling, ptr(dA), dA.stride(0), dA.stride(1), dA.stride(2), ptr(dB), dB.stride(0), dB.stride(1),
                                               dB.stride(2), ptr(dx), dx.stride(0), ptr(ssi), is64(ssi), ptr(eo), is64(eo), (int)E, L, K, N, dtype_code(x), ptr(ws),
                                               (size_t)ws.numel(), stream_of(x));
            if (rc != MOE_ERR_UNSUPPORTED) {
                check(rc, "moe_linear_lora_bwd");
                ws = Tensor();   // given back before the fan-out sum takes its output
                if (k != 1) dx = combine(dx, Tensor(), nullptr, k, L / k);
                return {dx, Tensor(), dA, dB, d_gates, Tensor(), Tensor(), Tensor()};
            }
        }
        // Gradients of adapters and weights need dY and X in expert-grouped order (reference :83-99); nobody else reads the latter.
        // (dY does not go into the saved rows of Y: a second backward pass over the same graph reads those again.)
        Tensor dy_g = grouped_out ? dout : group_rows(dout, ptr(ssi), is64(ssi), L, gate_fan, coeff);
        Tensor x_g = grouped_in ? x : A.defined() || ctx->needs_input_grad(1) ? group_rows(x, ptr(ssi), is64(ssi), L, k) : Tensor();
        if (A.defined()) {
            const int64_t K = x_g.size(1), N = dy_g.size(1), r = A.size(2);
            dA = at::empty({E, K, r}, dy_g.options());
            dB = at::empty({E, r, N}, dy_g.options());
            const int dt = dtype_code(dy_g);
            Tensor ws = bytes_on(x, moe_group_bwd_ab_workspace_bytes(L, (int)E, K, N, (int)r, dt));
            check(moe_group_bwd_ab(ptr(dy_g), dy_g.stride(0), dy_g.stride(1), ptr(x_g), x_g.stride(0), x_g.stride(1), ptr(A), A.stride(0), A.stride(1),
                                   A.stride(2), ptr(B), B.stride(0), B.stride(1), B.stride(2), (int)r,
                                   (float)ctx->saved_data["scaling_ab"].toDouble(), ptr(dA), dA.stride(0), dA.stride(1),
                                   dA.stride(2), ptr(dB), dB.stride(0), dB.stride(1), dB.stride(2), ptr(eo), is64(eo), (int)E, L, K, N, dt, ptr(ws),
                                   (size_t)ws.numel(), stream_of(x)), "moe_group_bwd_ab");
        } else if (ctx->needs_input_grad(1)) {
            dW = group_bwd_w(dy_g, x_g, ptr(eo), is64(eo), E);
        }
        // dX = dY W^T + s (dY B^T) A^T: the same grouped GEMM on transposed views (reference :116-128), then the fan-out sum (:134).  Its rows
        // take the place of the gathered X, which has had its readers: as large as dX before that sum, and freed with it
        Tensor dx = scatter2scatter(dy_g, W.transpose(1, 2), A.defined() ? B.transpose(1, 2) : Tensor(), A.defined() ? A.transpose(1, 2) : Tensor(), scaling,
                                    ssi, eo, 1, true, grouped_in, grouped_in ? Tensor() : x_g);
        if (k != 1) dx = combine(dx, Tensor(), nullptr, k, dx.size(0) / k);
        return {dx, dW, dA, dB, d_gates, Tensor(), Tensor(), Tensor()};
    }
};

Tensor linear_checked(const Tensor& x_, const Tensor& W, const Tensor& A, const Tensor& B, double scaling, double scaling_ab, int64_t k, const Tensor& sei, const Tensor& ssi_,
                      const Tensor& eo_, const Tensor& gates_, bool grouped_in, bool grouped_out)
{
    require_gpu({&x_, &W, &A, &B, &sei, &ssi_, &eo_, &gates_});
    MOE_ASSERT(ssi_.size(0) == sei.size(0), "sorted_scattered_idxs and sorted_expert_idxs differ in length");
    MOE_ASSERT(ssi_.size(0) == x_.size(0) * k, "the number of assignments is not rows of X times k");
    MOE_ASSERT(x_.dim() == 2 && W.dim() == 3 && x_.size(1) == W.size(1), "X and W have inconsistent inner dims.");
    MOE_ASSERT(!grouped_in || k == 1, "grouped rows of X are one for each assignment: k is 1 with them");
    MOE_ASSERT(W.scalar_type() == x_.scalar_type(), "X and W must share a dtype");
    if (A.defined()) {
        MOE_ASSERT(W.size(1) == A.size(1), "A has incorrect input size.");
        MOE_ASSERT(W.size(2) == B.size(2), "B has incorrect output size.");
        MOE_ASSERT(A.size(2) == B.size(1), "A and B have inconsistent inner dims.");
        MOE_ASSERT(A.dim() == 3 && B.dim() == 3 && A.size(0) >= W.size(0) && B.size(0) >= W.size(0), "A and B must hold a factor for every expert.");
        MOE_ASSERT(A.scalar_type() == x_.scalar_type() && B.scalar_type() == x_.scalar_type(), "A, B and X must share a dtype");
    }
    if (eo_.defined()) check_offsets(eo_, W.size(0));
    check_gates(gates_, ssi_.size(0));
    const c10::DeviceGuard guard(x_.device());
    Tensor x = unit_inner(x_), ssi = ssi_.contiguous(), eo = eo_.defined() ? eo_.contiguous() : offsets_from_sorted(sei, W.size(0));
    Tensor gates = gates_.defined() ? gates_.contiguous() : Tensor();
    const LinearCfg c{scaling, scaling_ab, k, grouped_in, grouped_out};
    if (needs_node({&x, &W, &A, &B, &gates})) return LinearFn::apply(x, W, opt(A), opt(B), opt(gates), ssi, eo, c);
    Tensor y = linear_rows(x, W, A, B, ssi, eo, c);
    return gates.defined() ? combine(y, gates, nullptr, gates.size(1), gates.size(0)) : y;
}

// lora_r: the rank the caller names (it scales the adapters' gradients, reference :102); the forward product is scaled by the factors' own
Tensor linear(const Tensor& x, const Tensor& W, const OptTensor& A, const OptTensor& B, double lora_r, double lora_alpha, int64_t k, const Tensor& sei,
              const Tensor& ssi, const OptTensor& eo, const OptTensor& gates, bool grouped_in, bool grouped_out)
{
    const Tensor a = val(A);
    return linear_checked(x, W, a, val(B), a.defined() ? lora_alpha / (double)a.size(2) : 0.0, a.defined() ? lora_alpha / lora_r : 0.0, k, sei, ssi, val(eo),
                          val(gates), grouped_in, grouped_out);
}

// ---------------------------------------------------------------------------------------------------------------
// pieces of the unfused route
// ---------------------------------------------------------------------------------------------------------------
Tensor swiglu_forward(const Tensor& gate, const Tensor& up)
{
    Tensor h = at::empty_like(gate);
    check(moe_swiglu(ptr(gate), ptr(up), ptr(h), gate.numel(), dtype_code(gate), stream_of(gate)), "moe_swiglu");
    return h;
}

struct SwigluFn : Function<SwigluFn> {
    static Tensor forward(AutogradContext* ctx, const Tensor& gate, const Tensor& up)
    {
        ctx->save_for_backward({gate, up});
        return swiglu_forward(gate, up);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g)
    {
        const auto sv = ctx->get_saved_variables();
        const c10::DeviceGuard guard(sv[0].device());
        Tensor dh = g[0].contiguous(), dg = at::empty_like(sv[0]), du = at::empty_like(sv[1]);
        check(moe_swiglu_bwd(ptr(sv[0]), ptr(sv[1]), ptr(dh), ptr(dg), ptr(du), dh.numel(), dtype_code(dh), stream_of(dh)), "moe_swiglu_bwd");
        return {dg, du};
    }
};

Tensor swiglu(const Tensor& gate_, const Tensor& up_)
{
    require_gpu({&gate_, &up_});
    const c10::DeviceGuard guard(gate_.device());
    Tensor gate = gate_.contiguous(), up = up_.contiguous();
    return needs_node({&gate, &up}) ? SwigluFn::apply(gate, up) : swiglu_forward(gate, up);
}

// out[t] = sum_j w[t,j] * y_grouped[inv[t*k+j]]  (megablocks ops.scatter, config_utils.py:251)
struct GatherCombineFn : Function<GatherCombineFn> {
    static Tensor forward(AutogradContext* ctx, const Tensor& y, const Tensor& w, const Tensor& inv, const Tensor& ssi)
    {
        ctx->save_for_backward({y, w, inv, ssi});
        return combine(y, w, (const int32_t*)ptr(inv), w.size(1), w.size(0));
    }
    static variable_list backward(AutogradContext* ctx, variable_list g)
    {
        const auto sv = ctx->get_saved_variables();
        const Tensor &y = sv[0], &w = sv[1], &inv = sv[2], &ssi = sv[3];
        const c10::DeviceGuard guard(y.device());
        Tensor dout = g[0].contiguous();
        Tensor d_w = combine_dgates(y, dout, w.size(1), w.scalar_type(), (const int32_t*)ptr(inv));
        // dy_grouped[i] = w[pos_i] * dout[pos_i // k]; pos, the inverse of inv, is the sort's own sorted_scattered_idxs
        Tensor d_y = group_rows(dout, ptr(ssi), is64(ssi), ssi.numel(), w.size(1), flat_gates(w));
        return {d_y, d_w, Tensor(), Tensor()};
    }
};

// int32, one buffer: sorted expert ids, sorted positions, inverse permutation (R each), inclusive offsets (E)
struct Sorted {
    Tensor ints;
    int64_t R = 0, E = 0;
    int32_t* at(int64_t i) const { return (int32_t*)ints.data_ptr() + i; }
    int32_t* sei() const { return at(0); }
    int32_t* ssi() const { return at(R); }
    int32_t* inv() const { return at(2 * R); }
    int32_t* offsets() const { return at(3 * R); }
};

Sorted sort_assignments(const Tensor& indices, int64_t E)
{
    const int64_t R = indices.numel();
    Sorted s{at::empty({3 * R + E}, indices.options()), R, E};
    Tensor ws = bytes_on(indices, moe_sort_workspace_bytes(R, (int)E));
    check(moe_sort_by_expert(ptr(indices), 0, R, (int)E, 128, s.sei(), s.ssi(), 0, nullptr, s.offsets(), nullptr, 0, nullptr, s.inv(), ptr(ws), (size_t)ws.numel(), stream_of(indices)), "moe_sort_by_expert");
    return s;
}

// router_forward and sort_assignments of its choices, one launch where the library has one
void router_and_sort(const Tensor& x, const Tensor& wg, int64_t k, bool normalize, RouterOut& rt, Sorted& s)
{
    const int64_t T = x.size(0), E = wg.size(0), R = T * k;
    rt = router_outputs(x, wg, k);
    Tensor logits = at::empty_like(rt.scores);
    s = Sorted{at::empty({3 * R + E}, rt.indices.options()), R, E};
    Tensor ws = bytes_on(x, moe_sort_workspace_bytes(R, (int)E));
    check(moe_router_forward_sorted(ptr(x), x.stride(0), ptr(wg), wg.stride(0), dtype_code(x), (float*)ptr(logits), (float*)ptr(rt.scores), (float*)ptr(rt.weights),
                                    (int32_t*)ptr(rt.indices), T, x.size(1), (int)E, (int)k, normalize, s.sei(), s.ssi(), s.inv(), s.offsets(), ptr(ws),
                                    (size_t)ws.numel(), stream_of(x)), "moe_router_forward_sorted");
}

// ---------------------------------------------------------------------------------------------------------------
// expert MLP on expert-grouped assignments (the reference's scattermoe_permute_and_compute, config_utils.py:99-185)
// ---------------------------------------------------------------------------------------------------------------
struct MlpCfg { double scaling; int64_t fan_out; bool y_grouped; };

struct ExpertMlpFn : Function<ExpertMlpFn> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w1, const Tensor& w3, const Tensor& w2, const OptTensor& a1, const OptTensor& b1,
                          const OptTensor& a3, const OptTensor& b3, const OptTensor& a2, const OptTensor& b2, const OptTensor& gates_,
                          const Tensor& ssi, const Tensor& offsets, const MlpCfg& c)
    {
        const Tensor lt[6] = {val(a1), val(b1), val(a3), val(b3), val(a2), val(b2)}, gates = val(gates_);
        const Lora lora = describe_lora(lt, false, w1.size(2), w1.size(1));
        const MlpShape s{w1.size(0), w1.size(2), w1.size(1), ssi.numel(), (int)c.fan_out, c.scaling};
        MlpOut o = mlp_forward(x, w1, w3, w2, lora, s, ptr(ssi), is64(ssi), ptr(offsets), is64(offsets), c.y_grouped, true);
        Tensor out = gates.defined() ? combine(o.y, gates, nullptr, gates.size(1), gates.size(0)) : o.y;
        ctx->save_for_backward({x, w1, w3, w2, lt[0], lt[1], lt[2], lt[3], lt[4], lt[5], gates, ssi, offsets, o.gate, o.up, o.h, o.saved, gates.defined() ? o.y : Tensor()});
        ctx->saved_data["scaling"] = c.scaling;
        ctx->saved_data["fan_out"] = c.fan_out;
        ctx->saved_data["y_grouped"] = c.y_grouped;
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list g_)
    {
        const auto sv = ctx->get_saved_variables();
        const Tensor &x = sv[0], &w1 = sv[1], &w3 = sv[2], &w2 = sv[3], &gates = sv[10], &ssi = sv[11], &offsets = sv[12];
        const c10::DeviceGuard guard(x.device());
        const Lora lora = describe_lora(&sv[4], false, w1.size(2), w1.size(1));
        const MlpShape s{w1.size(0), w1.size(2), w1.size(1), ssi.numel(), (int)ctx->saved_data["fan_out"].toInt(), ctx->saved_data["scaling"].toDouble()};
        Tensor dout = g_[0].contiguous(), d_gates, row_scale;
        bool dy_grouped = ctx->saved_data["y_grouped"].toBool();
        int64_t dy_fan = 1;
        if (gates.defined()) {
            dy_fan = gates.size(1);
            dy_grouped = false;
            d_gates = combine_dgates(sv[17], dout, dy_fan, gates.scalar_type(), nullptr);
            row_scale = group_rows(gates.reshape({-1, 1}).to(at::kFloat), ptr(ssi), is64(ssi), s.R, 1);   // gate of each sorted position
        }
        MlpGrads g = mlp_backward(dout, dy_grouped, dy_fan, (const float*)ptr(row_scale), x, w1, w3, w2, &sv[4], lora, s, sv[13], sv[14], sv[15], sv[16],
                                  ptr(ssi), is64(ssi), ptr(offsets), is64(offsets));
        Tensor d_x = s.fan_out == 1 ? g.dx_rows : combine(g.dx_rows, Tensor(), nullptr, s.fan_out, s.R / s.fan_out);
        Tensor dw[3];
        const bool needs[3] = {ctx->needs_input_grad(1), ctx->needs_input_grad(2), ctx->needs_input_grad(3)};
        if (needs[0] || needs[1] || needs[2])
            base_weight_grads(needs, x, dout, dy_grouped, dy_fan, flat_gates(gates), g, sv[15], ptr(ssi), is64(ssi),
                              ptr(offsets), is64(offsets), s, dw);
        return {d_x, dw[0], dw[1], dw[2], g.lora[0], g.lora[1], g.lora[2], g.lora[3], g.lora[4], g.lora[5], d_gates, Tensor(), Tensor(), Tensor()};
    }
};

bool mlp_fast_path(const Tensor& x, const Tensor& w1, const Tensor& w2, const Tensor& w3, const std::vector<Tensor>& lora)
{
    Tensor lt[6];
    take_factors(lora, lt);
    return fast_path_ok(x, w1, w2, w3, lt, false, w1.size(0), w1.size(2), w1.size(1));
}

// lora: empty, or the six factor views a1, b1, a3, b3, a2, b2
Tensor expert_mlp(const Tensor& x, const Tensor& w1, const Tensor& w2, const Tensor& w3, int64_t fan_out, const Tensor& ssi_, const Tensor& offsets_,
                  const std::vector<Tensor>& lora, double lora_alpha, const OptTensor& gates_, bool grouped_out)
{
    const Tensor gates_in = val(gates_);
    Tensor lt[6];
    take_factors(lora, lt);
    require_gpu({&x, &w1, &w2, &w3, &ssi_, &offsets_, &gates_in, &lt[0], &lt[1], &lt[2], &lt[3], &lt[4], &lt[5]});
    check_gates(gates_in, ssi_.numel());
    TORCH_CHECK(x.dim() == 2 && w1.dim() == 3 && x.size(1) == w1.size(2), "rows of ", x.sizes(), " do not fit expert weights of ", w1.sizes());
    for (const Tensor* w : {&w2, &w3}) check_expert_weight(*w, w1.size(0), w1.size(1), w1.size(2));
    check_factors(lt, false, w1.size(0), w1.size(1), w1.size(2));
    check_offsets(offsets_, w1.size(0));
    // Positions name rows of x (position / fan_out) and, unless the output stays grouped, its rows as well: there they are a permutation.
    // (A grouped output may hold a row of x any number of times.)
    TORCH_CHECK(fan_out >= 1 && ((grouped_out && !gates_in.defined()) || ssi_.numel() <= x.size(0) * fan_out), "positions of ",
                ssi_.sizes(), " do not fit ", x.size(0), " rows with a fan-out of ", fan_out);
    TORCH_CHECK(fast_path_ok(x, w1, w2, w3, lt, false, w1.size(0), w1.size(2), w1.size(1)),
                "fused_expert_mlp needs bf16 or fp16 throughout, contiguous (E,f,d) weights, d and f multiples of 64 and rank <= 128; use "
                "scattermoe_permute_and_compute for other cases");
    const c10::DeviceGuard guard(x.device());
    Tensor ssi = ssi_.contiguous(), offsets = offsets_.contiguous(), gates = gates_in.defined() ? gates_in.contiguous() : Tensor();
    const MlpCfg c{lt[0].defined() ? lora_alpha / (double)lt[0].size(2) : 0.0, fan_out, grouped_out && !gates.defined()};
    if (needs_node({&x, &w1, &w2, &w3, &lt[0], &lt[1], &lt[2], &lt[3], &lt[4], &lt[5], &gates}))
        return ExpertMlpFn::apply(x, w1, w3, w2, opt(lt[0]), opt(lt[1]), opt(lt[2]), opt(lt[3]), opt(lt[4]), opt(lt[5]), opt(gates), ssi, offsets, c);
    const MlpShape s{w1.size(0), w1.size(2), w1.size(1), ssi.numel(), (int)fan_out, c.scaling};
    MlpOut o = mlp_forward(x, w1, w3, w2, describe_lora(lt, false, s.d, s.f), s, ptr(ssi), is64(ssi), ptr(offsets), is64(offsets), c.y_grouped, false);
    return gates.defined() ? combine(o.y, gates, nullptr, gates.size(1), gates.size(0)) : o.y;
}

// ---------------------------------------------------------------------------------------------------------------
// whole layer: router -> sort -> expert MLP -> weighted combine, one autograd node
// ---------------------------------------------------------------------------------------------------------------
struct LayerCfg { double scaling; int64_t E, d, f, k; bool normalize, storage; };

struct LayerOut { RouterOut rt; Sorted so; MlpOut mlp; Tensor out; };

LayerOut layer_forward(const Tensor& x, const Tensor& wg, const Tensor& w1, const Tensor& w3, const Tensor& w2, const Tensor* lt, const LayerCfg& c, bool save)
{
    LayerOut o;
    router_and_sort(x, unit_inner(wg), c.k, c.normalize, o.rt, o.so);
    const MlpShape s{c.E, c.d, c.f, x.size(0) * c.k, (int)c.k, c.scaling};
    o.mlp = mlp_forward(x, w1, w3, w2, describe_lora(lt, c.storage, c.d, c.f), s, o.so.ssi(), 0, o.so.offsets(), 0, false, save);
    o.out = combine(o.mlp.y, o.rt.weights, nullptr, c.k, x.size(0));
    return o;
}

struct LayerFn : Function<LayerFn> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& wg, const Tensor& w1, const Tensor& w3, const Tensor& w2,
                                 const OptTensor& a1, const OptTensor& b1, const OptTensor& a3, const OptTensor& b3, const OptTensor& a2,
                                 const OptTensor& b2, const LayerCfg& c)
    {
        const Tensor lt[6] = {val(a1), val(b1), val(a3), val(b3), val(a2), val(b2)};
        LayerOut o = layer_forward(x, wg, w1, w3, w2, lt, c, true);
        ctx->save_for_backward({x, wg, w1, w3, w2, lt[0], lt[1], lt[2], lt[3], lt[4], lt[5], o.rt.scores, o.rt.weights, o.rt.indices, o.so.ints, o.mlp.gate, o.mlp.up,
                                o.mlp.h, o.mlp.y, o.mlp.saved});
        ctx->saved_data["scaling"] = c.scaling;
        ctx->saved_data["sizes"] = std::vector<int64_t>{c.E, c.d, c.f, c.k, c.normalize, c.storage};
        ctx->mark_non_differentiable({o.rt.indices});
        ctx->set_materialize_grads(false);   // an unused expert_weights output must not cost a zero-fill per step
        return {o.out, o.rt.weights, o.rt.indices};
    }
    static variable_list backward(AutogradContext* ctx, variable_list g_)
    {
        const auto sv = ctx->get_saved_variables();
        const Tensor &x = sv[0], &wg = sv[1], &w1 = sv[2], &w3 = sv[3], &w2 = sv[4], &y = sv[18];
        const Tensor scores = sv[11].contiguous(), weights = sv[12].contiguous(), indices = sv[13].contiguous();   // (a saved-tensor hook may hand back other strides)
        const c10::DeviceGuard guard(x.device());
        const auto sz = ctx->saved_data["sizes"].toIntVector();
        const int64_t k = sz[3], T = x.size(0);
        const Sorted so{sv[14], T * k, sz[0]};
        const bool normalize = sz[4] != 0, storage = sz[5] != 0;
        const MlpShape s{sz[0], sz[1], sz[2], T * k, (int)k, ctx->saved_data["scaling"].toDouble()};
        const Lora lora = describe_lora(&sv[5], storage, s.d, s.f);
        Tensor dout = g_[0].defined() ? g_[0].contiguous() : at::zeros_like(x);
        const Tensor d_w = g_[1].defined() ? g_[1].to(at::kFloat).contiguous() : Tensor();   // the caller also used the returned expert weights (e.g. in an auxiliary loss)
        Tensor dlogits = at::empty_like(scores), row_scale = at::empty({s.R}, scores.options());
        check(moe_gates_bwd(ptr(y), y.stride(0), ptr(dout), dout.stride(0), dtype_code(y), (const float*)ptr(d_w), (const float*)ptr(weights),
                            (const int32_t*)ptr(indices), (const float*)ptr(scores), so.inv(), (float*)ptr(dlogits), (float*)ptr(row_scale), T, y.size(1), (int)s.E,
                            (int)k, normalize, stream_of(y)), "moe_gates_bwd");
        MlpGrads g = mlp_backward(dout, false, k, (const float*)ptr(row_scale), x, w1, w3, w2, &sv[5], lora, s, sv[15], sv[16], sv[17], sv[19], so.ssi(), 0,
                                  so.offsets(), 0);
        Tensor dw[3];
        const bool needs[3] = {ctx->needs_input_grad(2), ctx->needs_input_grad(3), ctx->needs_input_grad(4)};
        if (needs[0] || needs[1] || needs[2]) {
            base_weight_grads(needs, x, dout, false, k, weights.view({-1}), g, sv[17], so.ssi(), 0, so.offsets(), 0, s, dw);
            const Tensor* w[3] = {&w1, &w3, &w2};
            for (int i = 0; i < 3; ++i)
                if (dw[i].defined()) dw[i] = dw[i].view(w[i]->sizes());
        }
        // fan-out sum of the k expert rows of each token plus the router's contribution dlogits @ wg, one pass
        Tensor d_x = combine(g.dx_rows, Tensor(), nullptr, k, T, (const float*)ptr(dlogits), unit_inner(wg), s.E);
        Tensor d_wg = ctx->needs_input_grad(1) ? router_weight_grad(x, dlogits) : Tensor();
        return {d_x, d_wg, dw[0], dw[1], dw[2], g.lora[0], g.lora[1], g.lora[2], g.lora[3], g.lora[4], g.lora[5], Tensor()};
    }
};

// The factors as views (E, K, r) / (E, r, N) of their storage
void lora_storage_to_views(Tensor* lt, int64_t E, int64_t d, int64_t f, int64_t rank)
{
    for (int i = 0; i < 6; ++i) {
        const bool on_ffn = i == 1 || i == 3 || i == 4;
        Tensor v = lt[i].view({E, on_ffn ? f : d, rank});
        lt[i] = i % 2 == 0 ? v : v.transpose(1, 2);
    }
}

// x (T, d); wg (E, d); expert weights (E, f, d), or (E*f, d) with `storage`; lora: empty, or six factors -- views, or with
// `storage` the block's A.weight / B.weight as a1, b1, a3, b3, a2 (= B of w2), b2 (= A of w2).
// -> out (T, d), expert weights (T, k) fp32, expert indices (T, k) int32
variable_list layer(const Tensor& x, const Tensor& wg, const Tensor& w1_, const Tensor& w2_, const Tensor& w3_, int64_t E, int64_t f, int64_t k,
                    const std::vector<Tensor>& lora, double lora_alpha, bool normalize, bool storage)
{
    Tensor lt[6];
    take_factors(lora, lt);
    require_gpu({&x, &wg, &w1_, &w2_, &w3_, &lt[0], &lt[1], &lt[2], &lt[3], &lt[4], &lt[5]});
    TORCH_CHECK(x.dim() == 2, "the layer takes (tokens, hidden size), got ", x.sizes());
    const int64_t d = x.size(1);
    TORCH_CHECK(wg.dim() == 2 && wg.size(0) == E, "router weight of ", wg.sizes(), " does not fit ", E, " experts");
    for (const Tensor* w : {&w1_, &w2_, &w3_}) {
        check_expert_weight(*w, E, f, d);
        MOE_ASSERT(w->scalar_type() == x.scalar_type(), "X and W must share a dtype");
    }
    check_factors(lt, storage, E, f, d);
    const c10::DeviceGuard guard(x.device());
    const Tensor w1 = w1_.contiguous(), w2 = w2_.contiguous(), w3 = w3_.contiguous();   // storage order, as the launches address it
    const int64_t rank = lt[0].defined() ? lt[0].size(-1) : 0;
    const double scaling = rank ? lora_alpha / (double)rank : 0.0;
    if (rank && storage) {
        bool contiguous = true;
        for (int i = 0; i < 6; ++i) contiguous = contiguous && lt[i].is_contiguous();
        if (!contiguous) {
            lora_storage_to_views(lt, E, d, f, rank);
            storage = false;
        }
    }
    if (fast_path_ok(x, w1, w2, w3, lt, storage, E, d, f)) {
        const LayerCfg c{scaling, E, d, f, k, normalize, storage};
        if (needs_node({&x, &wg, &w1, &w2, &w3, &lt[0], &lt[1], &lt[2], &lt[3], &lt[4], &lt[5]}))
            return LayerFn::apply(x, wg, w1, w3, w2, opt(lt[0]), opt(lt[1]), opt(lt[2]), opt(lt[3]), opt(lt[4]), opt(lt[5]), c);
        LayerOut o = layer_forward(x, wg, w1, w3, w2, lt, c, false);
        return {o.out, o.rt.weights, o.rt.indices};
    }
    // unfused route: the reference's three projections (config_utils.py:127-166), the combine of ops.scatter (:251)
    const variable_list rt = router(x, wg, k, normalize);
    const Sorted so = sort_assignments(rt[2], E);
    const Tensor sei = so.ints.narrow(0, 0, so.R), ssi = so.ints.narrow(0, so.R, so.R), inv = so.ints.narrow(0, 2 * so.R, so.R),
                 offsets = so.ints.narrow(0, 3 * so.R, E);
    if (storage && rank) lora_storage_to_views(lt, E, d, f, rank);
    auto proj = [&](const Tensor& in, const Tensor& w, bool n_contiguous, int ia, int64_t fan, bool gin) {
        Tensor W = w.view({E, f, d});
        return linear_checked(in, n_contiguous ? W : W.transpose(1, 2), lt[ia], lt[ia + 1], scaling, scaling, fan, sei, ssi, offsets, Tensor(), gin, true);
    };
    Tensor h;
    if (!rank && x.scalar_type() == at::kFloat && so.R > 0 && d > 0 && f > 0 && !needs_node({&x, &w1, &w3})) {   // both projections and their product in one launch (three: 256 tokens, d=128, f=256: 20 us, one 10.4)
        h = at::empty({so.R, f}, x.options());
        check(moe_swiglu_pair(ptr(x), x.stride(0), x.stride(1), ptr(w1), ptr(w3), f * d, 1, d, ptr(h), h.stride(0), so.ssi(), 0, so.offsets(), 0, (int)E, so.R, d, f, (int)k,
                              dtype_code(x), stream_of(x)), "moe_swiglu_pair");
    } else h = swiglu(proj(x, w1, false, 0, k, false), proj(x, w3, false, 2, k, false));
    Tensor y = proj(h, w2, true, 4, 1, true);
    Tensor out = needs_node({&y, &rt[1]}) ? GatherCombineFn::apply(y, rt[1], inv, ssi) : combine(y, rt[1], so.inv(), k, x.size(0));
    return {out, rt[1], rt[2]};
}

}  // namespace

// Called from Python without the interpreter lock.  The wrapper carries a Python exception that is raised below (a saved-tensor
// hook's, such as the one that ends a recomputation of activation checkpointing early) through as itself.
PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    m.def("router", torch::wrap_pybind_function_no_gil(router));
    m.def("linear", torch::wrap_pybind_function_no_gil(linear));
    m.def("swiglu", torch::wrap_pybind_function_no_gil(swiglu));
    m.def("mlp_fast_path", torch::wrap_pybind_function(mlp_fast_path));
    m.def("expert_mlp", torch::wrap_pybind_function_no_gil(expert_mlp));
    m.def("layer", torch::wrap_pybind_function_no_gil(layer));
}

// The same functions as dispatcher operators, for torch.jit.trace: a trace records operators, and of the functions above it
// would see their allocations only.  (Calls outside a trace take the functions above, which cost less to enter.)
TORCH_LIBRARY(moe_hip, m)
{
    m.def("router", [](const Tensor& x, const Tensor& wg, int64_t k, bool normalize) { return router(x, wg, k, normalize); });
    m.def("linear", [](const Tensor& x, const Tensor& W, const OptTensor& A, const OptTensor& B, double lora_r, double lora_alpha, int64_t k,
                       const Tensor& sei, const Tensor& ssi, const OptTensor& eo, const OptTensor& gates, bool grouped_in, bool grouped_out) {
        return linear(x, W, A, B, lora_r, lora_alpha, k, sei, ssi, eo, gates, grouped_in, grouped_out);
    });
    m.def("swiglu", [](const Tensor& gate, const Tensor& up) { return swiglu(gate, up); });
    m.def("expert_mlp", [](const Tensor& x, const Tensor& w1, const Tensor& w2, const Tensor& w3, int64_t fan_out, const Tensor& ssi,
                           const Tensor& offsets, at::TensorList lora, double lora_alpha, const OptTensor& gates, bool grouped_out) {
        return expert_mlp(x, w1, w2, w3, fan_out, ssi, offsets, lora.vec(), lora_alpha, gates, grouped_out);
    });
    m.def("layer", [](const Tensor& x, const Tensor& wg, const Tensor& w1, const Tensor& w2, const Tensor& w3, int64_t E, int64_t f, int64_t k,
                      at::TensorList lora, double lora_alpha, bool normalize, bool storage) {
        return layer(x, wg, w1, w2, w3, E, f, k, lora.vec(), lora_alpha, normalize, storage);
    });
}
