// Host side of the operator for torch tensors: checks, output and workspace tensors, launches through the C ABI of
// libmhffn_hip.so, and the autograd nodes.  The same steps written in Python (two autograd.Function nodes, ctypes calls, a
// dozen attribute look-ups) take 20 us per forward and 100 us per forward + backward of the operator on the host, several
// times what the kernels of a short sequence take on the GPU.
//
// What each function computes and returns is described in flash_mlp_moe.py, head_gate.py and mhffn_layer.py, which call
// these.  Errors carry the exception types of the reference: TypeError for dtypes, ValueError for the expert and head
// dims, RuntimeError otherwise (kernels/triton/flash_mlp_moe.py:758-766, kernels/thunderkittens/flash_ffn_moe.cu:943-958).
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/utils/pybind.h>
#include <ATen/ATen.h>
#include <ATen/record_function.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include "../../include/mhffn.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

void raise_for_code(int code, const char* what)
{
    if (code == MHFFN_OK) return;
    const char* text = mhffn_strerror(code);
    TORCH_CHECK_TYPE(code != MHFFN_ERR_DTYPE, what, ": ", text, " (code ", code, ")");
    TORCH_CHECK_VALUE(code != MHFFN_ERR_EXPERT_DIM && code != MHFFN_ERR_HEAD_DIM, what, ": ", text, " (code ", code, ")");
    TORCH_CHECK(false, what, ": ", text, " (code ", code, ")");
}

int dtype_code(at::ScalarType t)
{
    return t == at::kBFloat16 ? MHFFN_DTYPE_BF16 : t == at::kFloat ? MHFFN_DTYPE_F32 : -1;
}

// Workspace bytes of a shape, remembered per thread: the slots of a direct-mapped table.
struct Plan {
    mhffn_dims dims;
    int dtype;
    size_t fwd_bytes, bwd_bytes, bwd_min_bytes;
};
const Plan& plan_for(const mhffn_dims& d, int dtype)
{
    static thread_local Plan table[64] = {};
    unsigned h = (unsigned)d.S * 2654435761u ^ (unsigned)d.B * 40503u ^ (unsigned)d.d_e * 97u ^ (unsigned)d.E * 31u ^
                 (unsigned)d.H * 7u ^ (unsigned)d.Hkuv * 3u ^ (unsigned)d.d_h ^ (unsigned)dtype;
    Plan& p = table[(h ^ (h >> 13)) & 63];
    if (memcmp(&p.dims, &d, sizeof d) != 0 || p.dtype != dtype) {
        raise_for_code(mhffn_check_dims(&d, dtype), "mhffn");
        p = Plan{d, dtype, mhffn_fwd_workspace_bytes(&d, dtype), mhffn_bwd_workspace_bytes(&d, dtype),
                 mhffn_bwd_workspace_min_bytes(&d, dtype)};
    }
    return p;
}

// The library launches on the current device: a guard only where the tensors live on another one.
struct OnDevice {
    c10::OptionalDeviceGuard guard;
    explicit OnDevice(const Tensor& t)
    {
        if (t.device().index() != c10::hip::current_device()) guard.reset_device(t.device());
    }
};
void* stream() { return (void*)c10::hip::getCurrentHIPStream().stream(); }

Tensor empty_like_layout(const Tensor& t) { return at::detail::empty_strided_cuda(t.sizes(), t.strides(), t.scalar_type(), t.device()); }
Tensor empty_of(at::IntArrayRef sizes, at::ScalarType dtype, const Tensor& on)
{
    return at::detail::empty_cuda(sizes, dtype, on.device(), std::nullopt);
}
Tensor scratch(size_t bytes, const Tensor& on)
{
    return bytes ? empty_of({(int64_t)bytes}, at::kByte, on) : Tensor();
}
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

bool token_major(const Tensor& t)      // [B, H, S, d] seen through the transposed view of a contiguous [B, S, H, d]
{
    const auto s = t.strides(), n = t.sizes();
    return (s[3] == 1 || n[3] == 1) && (s[1] == n[3] || n[1] == 1) && (s[2] == n[1] * n[3] || n[2] == 1) &&
           (s[0] == n[2] * n[1] * n[3] || n[0] == 1);
}

void check_inputs(const Tensor& Q, const Tensor& K, const Tensor& U, const Tensor& V, const Tensor& R)
{
    TORCH_CHECK(Q.dim() == 4 && K.dim() == 4 && R.dim() == 4, "expected Q [B,H,S,d_h], K/U/V [Hkuv,E,d_e,d_h], R [B,H,S,E]");
    const auto dt = Q.scalar_type();
    TORCH_CHECK_TYPE((dt == at::kBFloat16 || dt == at::kFloat) && K.scalar_type() == dt && V.scalar_type() == dt && U.scalar_type() == dt,
                     "FlashMLPFunction expects all inputs in torch.bfloat16 (or all in torch.float32), got Q=", dt, ", K=",
                     K.scalar_type(), ", V=", V.scalar_type(), ", U=", U.scalar_type());
    TORCH_CHECK_TYPE(R.scalar_type() == at::kFloat, "R must be float32 (the router gate is computed in fp32), got ", R.scalar_type());
    TORCH_CHECK(U.sizes() == K.sizes() && V.sizes() == K.sizes(), "K, U, V must share one shape, got ", K.sizes(), ", ", U.sizes(),
                ", ", V.sizes());
    TORCH_CHECK(R.size(0) == Q.size(0) && R.size(1) == Q.size(1) && R.size(2) == Q.size(2) && R.size(3) == K.size(1),
                "R must be [B,H,S,E] = [", Q.size(0), ", ", Q.size(1), ", ", Q.size(2), ", ", K.size(1), "], got ", R.sizes());
    TORCH_CHECK_VALUE(dt != at::kBFloat16 || K.size(2) % 32 == 0, "Expert dimension ", K.size(2), " must be divisible by 32");
    TORCH_CHECK(Q.is_cuda(), "flashmhf_amd runs on the GPU only; there is no CPU path");
    for (const Tensor* t : {&K, &U, &V, &R})
        TORCH_CHECK(t->device() == Q.device(), "K, U, V and R must be on the device of Q, ", Q.device(), "; one is on ", t->device());
    TORCH_CHECK(Q.size(3) == K.size(3), "head dim mismatch: Q has ", Q.size(3), ", K has ", K.size(3));
}

mhffn_dims dims_of(const Tensor& Q, const Tensor& K)
{
    return mhffn_dims{(int)Q.size(0), (int)Q.size(1), (int)K.size(0), (int)Q.size(2), (int)Q.size(3), (int)K.size(1), (int)K.size(2)};
}

// (the tensor to pass, its layout): [B,H,S,d_h] contiguous, or the transposed view of a contiguous [B,S,H,d_h]
std::pair<Tensor, int> laid_out(const Tensor& Q)
{
    if (Q.is_contiguous()) return {Q, MHFFN_TOKENS_BHSD};
    if (token_major(Q)) return {Q, MHFFN_TOKENS_BSHD};
    return {Q.contiguous(), MHFFN_TOKENS_BHSD};
}
Tensor as_layout(const Tensor& t, int layout)
{
    if (layout == MHFFN_TOKENS_BHSD) return t.contiguous();
    return token_major(t) ? t : t.transpose(1, 2).contiguous().transpose(1, 2);
}
Tensor contig(const Tensor& t) { return t.is_contiguous() ? t : t.contiguous(); }

Tensor op_forward(const Tensor& Q0, const Tensor& K0, const Tensor& U0, const Tensor& V0, const Tensor& R0, bool one_part)
{
    check_inputs(Q0, K0, U0, V0, R0);
    auto [Q, layout] = laid_out(Q0);
    const Tensor K = contig(K0), U = contig(U0), V = contig(V0), R = contig(R0);
    const int dt = dtype_code(Q.scalar_type());
    const Plan& p = plan_for(dims_of(Q, K), dt);
    OnDevice guard(Q);
    Tensor O = empty_like_layout(Q), ws = scratch(one_part ? 0 : p.fwd_bytes, Q);
    raise_for_code(mhffn_fwd_layout(ptr(Q), ptr(K), ptr(U), ptr(V), (const float*)ptr(R), ptr(O), ptr(ws), p.fwd_bytes, &p.dims, dt,
                                    layout, stream(), MHFFN_FWD_ALL | (one_part ? MHFFN_ONE_PART : 0)),
                   "mhffn_fwd");
    return O;
}

variable_list op_backward(const Tensor& Q0, const Tensor& K0, const Tensor& U0, const Tensor& V0, const Tensor& R0,
                          const Tensor& dO0, at::ScalarType grad_w, bool one_part)
{
    check_inputs(Q0, K0, U0, V0, R0);
    TORCH_CHECK(dO0.sizes() == Q0.sizes(), "grad_output shape should be the same as Q");
    auto [Q, layout] = laid_out(Q0);
    const Tensor K = contig(K0), U = contig(U0), V = contig(V0), R = contig(R0);
    const Tensor dO = as_layout(dO0.scalar_type() == Q.scalar_type() ? dO0 : dO0.to(Q.scalar_type()), layout);
    const int dt = dtype_code(Q.scalar_type()), wdt = dtype_code(grad_w);
    const Plan& p = plan_for(dims_of(Q, K), dt);
    OnDevice guard(Q);
    const size_t ws_bytes = one_part ? p.bwd_min_bytes : p.bwd_bytes;
    Tensor dQ = empty_like_layout(Q), dR = empty_of(R.sizes(), at::kFloat, Q), ws = scratch(ws_bytes, Q);
    Tensor dK = empty_of(K.sizes(), grad_w, Q), dU = empty_of(K.sizes(), grad_w, Q), dV = empty_of(K.sizes(), grad_w, Q);
    raise_for_code(mhffn_bwd_layout(ptr(Q), ptr(K), ptr(U), ptr(V), (const float*)ptr(R), ptr(dO), ptr(dQ), ptr(dK), ptr(dU), ptr(dV),
                                    (float*)ptr(dR), wdt, ptr(ws), ws_bytes, &p.dims, dt, layout, stream(),
                                    MHFFN_BWD_ALL | (one_part ? MHFFN_ONE_PART : 0)),
                   "mhffn_bwd");
    return {dQ, dK, dU, dV, dR};
}

bool records_grad(std::initializer_list<const Tensor*> ts)
{
    if (!at::GradMode::is_enabled()) return false;
    for (const Tensor* t : ts)
        if (t->defined() && t->requires_grad()) return true;
    return false;
}

// O = fused(Q, K, U, V, R), gradients in the inputs' types.  (The ThunderKittens wrapper returns float32 gradients,
// kernels/thunderkittens/flash_ffn_moe_torch.py:17-21, which autograd rounds to the inputs' types before anyone sees
// them: the same values, so the kernels write those at once.)
struct OpNode : torch::autograd::Function<OpNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& Q, const Tensor& K, const Tensor& U, const Tensor& V, const Tensor& R,
                          bool one_part)
    {
        ctx->save_for_backward({Q, K, U, V, R});
        ctx->saved_data["one_part"] = one_part;
        return op_forward(Q, K, U, V, R, one_part);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g)
    {
        const auto s = ctx->get_saved_variables();
        auto out = op_backward(s[0], s[1], s[2], s[3], s[4], g[0], s[1].scalar_type(), ctx->saved_data["one_part"].toBool());
        out.emplace_back();
        return out;
    }
};
Tensor op(const Tensor& Q, const Tensor& K, const Tensor& U, const Tensor& V, const Tensor& R, bool one_part)
{
    if (!records_grad({&Q, &K, &U, &V, &R})) return op_forward(Q, K, U, V, R, one_part);
    return OpNode::apply(Q, K, U, V, R, one_part);
}

// The single-expert operator: Q [B,H,S,d_h], K/U/V [Hkuv, rows, d_h], gate 1.
Tensor ones_gate(const Tensor& Q) { return at::ones({Q.size(0), Q.size(1), Q.size(2), 1}, Q.options().dtype(at::kFloat)); }
struct SingleNode : torch::autograd::Function<SingleNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& Q, const Tensor& K, const Tensor& U, const Tensor& V, bool one_part)
    {
        const Tensor R = ones_gate(Q);
        ctx->save_for_backward({Q, K, U, V, R});
        ctx->saved_data["one_part"] = one_part;
        return op_forward(Q, K.unsqueeze(1), U.unsqueeze(1), V.unsqueeze(1), R, one_part);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g)
    {
        const auto s = ctx->get_saved_variables();
        auto out = op_backward(s[0], s[1].unsqueeze(1), s[2].unsqueeze(1), s[3].unsqueeze(1), s[4], g[0], s[1].scalar_type(),
                               ctx->saved_data["one_part"].toBool());
        return {out[0], out[1].squeeze(1), out[2].squeeze(1), out[3].squeeze(1), Tensor()};
    }
};
Tensor single(const Tensor& Q, const Tensor& K, const Tensor& U, const Tensor& V, bool one_part)
{
    if (!records_grad({&Q, &K, &U, &V})) return op_forward(Q, K.unsqueeze(1), U.unsqueeze(1), V.unsqueeze(1), ones_gate(Q), one_part);
    return SingleNode::apply(Q, K, U, V, one_part);
}

// ---- head prologue -------------------------------------------------------------------------------------------------
mhffn_dims gate_dims(const Tensor& x4, const Tensor& wn, const Tensor& router)
{
    TORCH_CHECK(x4.dim() == 4 && router.dim() == 3, "expected x [B,S,H,d_h] and router [H,d_h,E]");
    TORCH_CHECK_TYPE(x4.scalar_type() == at::kBFloat16, "head_norm_gate expects bfloat16 heads, got ", x4.scalar_type());
    const auto n = x4.sizes();
    TORCH_CHECK(router.size(0) == n[2] && router.size(1) == n[3], "router must be [H,d_h,E] = [", n[2], ",", n[3], ",E], got ",
                router.sizes());
    TORCH_CHECK(!wn.defined() || (wn.dim() == 2 && wn.size(0) == n[2] && wn.size(1) == n[3]), "norm_weight must be [H,d_h] = [", n[2],
                ",", n[3], "], got ", wn.defined() ? wn.sizes() : at::IntArrayRef());
    TORCH_CHECK(x4.is_cuda(), "flashmhf_amd runs on the GPU only; there is no CPU path");
    TORCH_CHECK(router.device() == x4.device() && (!wn.defined() || wn.device() == x4.device()),
                "router and norm_weight must be on the device of x, ", x4.device());
    return mhffn_dims{(int)n[0], (int)n[2], (int)n[2], (int)n[1], (int)n[3], (int)router.size(2), 32};
}

struct GateForward {
    Tensor x4, wn, wr, q4, R;      // contiguous x and weights, normalised heads [B,S,H,d_h] (x4 without a norm), gate
};
// `t` contiguous on a 16-byte boundary (a view into a flat buffer of parameters may start anywhere)
Tensor on_boundary(const Tensor& t)
{
    const Tensor c = contig(t);
    return (reinterpret_cast<uintptr_t>(c.data_ptr()) & 15) == 0 ? c : c.clone();
}
Tensor gate_param(const Tensor& w)      // contiguous and on a boundary, float32 or bfloat16
{
    if (!w.defined()) return w;
    return on_boundary(w.scalar_type() == at::kBFloat16 || w.scalar_type() == at::kFloat ? w : w.to(at::kFloat));
}
int param_code(const Tensor& w) { return w.defined() ? dtype_code(w.scalar_type()) : MHFFN_DTYPE_F32; }
GateForward gate_forward(const Tensor& x, const Tensor& norm_weight, const Tensor& router, double eps)
{
    const mhffn_dims d = gate_dims(x, norm_weight, router);
    GateForward f;
    f.x4 = contig(x);
    f.wn = gate_param(norm_weight);
    f.wr = gate_param(router);
    OnDevice guard(f.x4);
    f.q4 = f.wn.defined() ? empty_of(x.sizes(), at::kBFloat16, f.x4) : f.x4;
    f.R = empty_of({d.B, d.H, d.S, d.E}, at::kFloat, f.x4);
    raise_for_code(mhffn_gate_fwd_typed(ptr(f.x4), ptr(f.wn), param_code(f.wn), (float)eps, ptr(f.wr), param_code(f.wr),
                                        f.wn.defined() ? ptr(f.q4) : nullptr, (float*)ptr(f.R), &d, stream()),
                   "mhffn_gate_fwd");
    return f;
}
// {dx, d_norm_weight, d_router}; dQ, dR may be undefined (zero)
variable_list gate_backward(const Tensor& x4, const Tensor& norm_weight, const Tensor& router, const Tensor& wn, const Tensor& wr,
                            double eps, Tensor dQ, Tensor dR)
{
    const mhffn_dims d = gate_dims(x4, norm_weight, router);
    OnDevice guard(x4);
    if (!dQ.defined()) dQ = at::zeros_like(x4).transpose(1, 2);
    if (!dR.defined()) dR = at::zeros({d.B, d.H, d.S, d.E}, x4.options().dtype(at::kFloat));
    int layout = MHFFN_TOKENS_BSHD;
    if (!token_major(dQ)) {
        layout = MHFFN_TOKENS_BHSD;
        dQ = dQ.contiguous();
    }
    dR = contig(dR.scalar_type() == at::kFloat ? dR : dR.to(at::kFloat));
    Tensor dx = empty_of(x4.sizes(), at::kBFloat16, x4), dwn, dwr = empty_of(wr.sizes(), wr.scalar_type(), x4);
    if (wn.defined()) dwn = empty_of(wn.sizes(), wn.scalar_type(), x4);
    const size_t ws_bytes = mhffn_gate_bwd_workspace_bytes(&d);
    Tensor ws = scratch(ws_bytes, x4);
    raise_for_code(mhffn_gate_bwd_into(ptr(x4), ptr(wn), param_code(wn), (float)eps, ptr(wr), param_code(wr), ptr(dQ), layout,
                                       (const float*)ptr(dR), ptr(dx), ptr(dwn), ptr(dwr), ptr(ws), ws_bytes, &d, stream()),
                   "mhffn_gate_bwd");
    return {dx, dwn.defined() ? dwn.to(norm_weight.scalar_type()) : dwn, dwr.to(router.scalar_type())};
}

struct GateNode : torch::autograd::Function<GateNode> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const std::optional<Tensor>& norm_weight, const Tensor& router,
                                 double eps)
    {
        const Tensor nw = norm_weight.value_or(Tensor());
        GateForward f = gate_forward(x, nw, router, eps);
        ctx->save_for_backward({f.x4, nw, router, f.wn, f.wr});
        ctx->saved_data["eps"] = eps;
        return {f.q4.transpose(1, 2), f.R};
    }
    static variable_list backward(AutogradContext* ctx, variable_list g)
    {
        const auto s = ctx->get_saved_variables();
        auto out = gate_backward(s[0], s[1], s[2], s[3], s[4], ctx->saved_data["eps"].toDouble(), g[0], g[1]);
        out.emplace_back();
        return out;
    }
};
std::pair<Tensor, Tensor> gate(const Tensor& x, const std::optional<Tensor>& norm_weight, const Tensor& router, double eps)
{
    const Tensor nw = norm_weight.value_or(Tensor());
    if (!records_grad({&x, &nw, &router})) {
        GateForward f = gate_forward(x, nw, router, eps);
        return {f.q4.transpose(1, 2), f.R};
    }
    auto out = GateNode::apply(x, norm_weight, router, eps);
    return {out[0], out[1]};
}

// ---- products of the block's projections ----------------------------------------------------------------------------
// Whether a tensor on the GPU is its memory and nothing more: no code of a subclass, a transform (batches) or a lazy view (negation) is
// to run for it, and no tangent goes with it (forward mode, which may be entered for the backward alone).  Asked before its pointer:
// some of the others have none.
bool memory_alone(const Tensor& t)
{
    using Key = c10::DispatchKey;
    constexpr c10::DispatchKeySet plain_keys({Key::CUDA, Key::AutogradCUDA, Key::ADInplaceOrView, Key::AutocastCUDA});
    return (t.key_set().raw_repr() & ~plain_keys.raw_repr()) == 0 && !t._fw_grad(0).defined();
}
// A plain matrix that the product kernels read as it lies.
bool plain(const Tensor& t)
{
    return memory_alone(t) && t.is_contiguous() && t.scalar_type() == at::kBFloat16 &&
           (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
}
// Whose products: the library's, these kernels', or these kernels' where the library was found to take each element's sum in the order
// of the summed index, as the tile kernels do, so that both have the same bits (a model's layers amplify a different rounding, see
// MHFFNDecoder in mhffn_layer.py).  Found by comparing bits, 11,700 products of 512 to 4,096 columns and summed indexes to 8,192, of
// 17 to 8,192 rows: the library splits the summed index, or adds in another order,
//   NT  below 32 rows, and with more than 1,024 of the summed index only where there are no more than 2^18 results
//   NN  at 16 rows and fewer, and with more than 1,024 of the summed index only where there are no more than 2^18 results
//   TN  of 16 rows and fewer, and of more than 16,384 (compared to 32,768).  Those of more stay here, in order: the gradient of a
//       weight goes into no other layer's (hidden 1024, 32,768 rows: 128 us, the library's 198).
// It is a table of another library's choices, not a promise of it: tests/test_gpu_product.py compares.
enum Whose { LIBRARY = 0, OWN = 1, OWN_IN_ORDER = 2 };
bool library_in_order(int form, int64_t M, int64_t N, int64_t K)
{
    if (form == MHFFN_PRODUCT_TN) return K > 16;
    return M > (form == MHFFN_PRODUCT_NT ? 31 : 16) && (K <= 1024 || M * N > (1 << 18));
}
// Whether an M x N product with inner extent K may run in these kernels: not where its bits are to be the library's and are not, not
// under a dispatch mode (which is to see the call) nor where autograd is to record the call.
bool own_may(int form, Whose whose, const Tensor& a, const Tensor& b, int64_t M, int64_t N, int64_t K)
{
    if (whose == LIBRARY || (whose == OWN_IN_ORDER && !library_in_order(form, M, N, K))) return false;
    if (at::GradMode::is_enabled() && (a.requires_grad() || b.requires_grad())) return false;
    if (!plain(a) || !plain(b) || a.device() != b.device() || c10::impl::TorchDispatchModeTLS::any_modes_set()) return false;
    return std::max({M, N, K}) <= INT_MAX;
}
// That product into `out_sizes`, or an undefined tensor where it is the library's: also where that is faster
Tensor own_product(int form, Whose whose, const Tensor& a, const Tensor& b, int64_t M, int64_t N, int64_t K, at::IntArrayRef out_sizes)
{
    if (!own_may(form, whose, a, b, M, N, K) || !mhffn_product_faster(form, whose == OWN_IN_ORDER, (int)M, (int)N, (int)K)) return {};
    RECORD_FUNCTION("mhffn::product", std::vector<c10::IValue>());
    OnDevice on_device(a);
    Tensor c = empty_of(out_sizes, at::kBFloat16, a);
    raise_for_code(mhffn_product(form, whose == OWN_IN_ORDER, ptr(a), ptr(b), ptr(c), (int)M, (int)N, (int)K, stream()), "mhffn_product");
    return c;
}
// x w^T, x [.., in], w [out, in]
Tensor project(const Tensor& x, const Tensor& w, Whose whose)
{
    if (x.dim() > 0 && w.dim() == 2 && x.size(-1) == w.size(1) && w.size(1) > 0) {
        at::DimVector sizes(x.sizes());
        sizes.back() = w.size(0);
        Tensor y = own_product(MHFFN_PRODUCT_NT, whose, x, w, x.numel() / w.size(1), w.size(0), w.size(1), sizes);
        if (y.defined()) return y;
    }
    return at::linear(x, w);
}
// dy w and dy^T x of matrices
Tensor product_nn(const Tensor& a, const Tensor& b, Whose whose)
{
    Tensor c = own_product(MHFFN_PRODUCT_NN, whose, a, b, a.size(0), b.size(1), a.size(1), {a.size(0), b.size(1)});
    return c.defined() ? c : at::mm(a, b);
}
Tensor product_tn(const Tensor& a, const Tensor& b, Whose whose)
{
    Tensor c = own_product(MHFFN_PRODUCT_TN, whose, a, b, a.size(1), b.size(1), a.size(0), {a.size(1), b.size(1)});
    return c.defined() ? c : at::mm(a.t(), b);
}

// Both gradients of a linear layer, {dy w, dy^T x} of matrices: in one launch where that is faster.
std::pair<Tensor, Tensor> product_pair(const Tensor& dy, const Tensor& w, const Tensor& x, Whose whose)
{
    const int64_t M = dy.size(0), N = dy.size(1), K = w.size(1);
    if (w.size(0) == N && x.size(0) == M && x.size(1) == K && own_may(MHFFN_PRODUCT_NN, whose, dy, w, M, K, N) &&
        own_may(MHFFN_PRODUCT_TN, whose, dy, x, N, K, M) && mhffn_product_pair_faster(whose == OWN_IN_ORDER, (int)M, (int)N, (int)K)) {
        OnDevice on_device(dy);
        Tensor dx, dw;
        {
            RECORD_FUNCTION("mhffn::product", std::vector<c10::IValue>());      // (one for each product)
            dx = empty_of({M, K}, at::kBFloat16, dy);
        }
        RECORD_FUNCTION("mhffn::product", std::vector<c10::IValue>());
        dw = empty_of({N, K}, at::kBFloat16, dy);
        raise_for_code(mhffn_product_pair(ptr(dy), ptr(w), ptr(x), ptr(dx), ptr(dw), (int)M, (int)N, (int)K, stream()), "mhffn_product_pair");
        return {dx, dw};
    }
    return {product_nn(dy, w, whose), product_tn(dy, x, whose)};
}

// A linear layer without bias (Projection in mhffn_layer.py).
struct LinearNode : torch::autograd::Function<LinearNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, int64_t whose)
    {
        ctx->saved_data["whose"] = whose;
        // (each gradient needs the other factor)
        ctx->save_for_backward({w.requires_grad() ? x : Tensor(), x.requires_grad() ? w : Tensor()});
        return project(x, w, Whose(whose));
    }
    static variable_list backward(AutogradContext* ctx, variable_list g)
    {
        const auto s = ctx->get_saved_variables();
        const Tensor &x = s[0], &w = s[1];
        const Whose whose = Whose(ctx->saved_data["whose"].toInt());
        const Tensor dy = g[0].reshape({-1, g[0].size(-1)});
        Tensor dx, dw;
        const bool need_x = ctx->needs_input_grad(0), need_w = ctx->needs_input_grad(1);
        if (need_x && need_w) std::tie(dx, dw) = product_pair(dy, w, x.reshape({-1, x.size(-1)}), whose);
        else if (need_x) dx = product_nn(dy, w, whose);
        else if (need_w) dw = product_tn(dy, x.reshape({-1, x.size(-1)}), whose);
        if (need_x) {
            at::DimVector sizes(g[0].sizes());
            sizes.back() = w.size(1);
            dx = dx.view(sizes);
        }
        return {dx, dw, Tensor()};
    }
};
Tensor linear(const Tensor& x, const Tensor& w, Whose whose)
{
    if (!records_grad({&x, &w})) return project(x, w, whose);
    // (torch's node where the products are the library's, and where a dispatch mode is to see them)
    if (whose == LIBRARY || x.dim() == 0 || w.dim() != 2 || x.numel() == 0 || x.size(-1) != w.size(1) || !plain(x) || !plain(w) ||
        c10::impl::TorchDispatchModeTLS::any_modes_set())
        return at::linear(x, w);
    return LinearNode::apply(x, w, (int64_t)whose);
}

// ---- the whole block: w_self, prologue, operator, w_self_2 ---------------------------------------------------------
struct BlockForward {
    GateForward g;
    Tensor O4, Y;      // operator output [B,S,H,d_h], block output
};
BlockForward block_forward(const Tensor& x, const Tensor& w1, const Tensor& norm_weight, const Tensor& router, const Tensor& K,
                           const Tensor& U, const Tensor& V, const Tensor& w2, double eps, bool one_part, Whose whose)
{
    BlockForward f;
    const int64_t B = x.size(0), S = x.size(1), hid = x.size(2);
    f.g = gate_forward(project(x, w1, whose).view({B, S, router.size(0), router.size(1)}), norm_weight, router, eps);
    f.O4 = op_forward(f.g.q4.transpose(1, 2), K, U, V, f.g.R, one_part).transpose(1, 2);
    f.Y = project(f.O4.view({B, S, hid}), w2, whose);
    return f;
}

Tensor stepwise_O4(const Tensor& x, const Tensor& w1, const Tensor& nw, const Tensor& router, const Tensor& K, const Tensor& U,
                   const Tensor& V, double eps, bool one_part, Whose whose)
{
    auto [Q, R] = gate(linear(x, w1, whose).view({x.size(0), x.size(1), router.size(0), router.size(1)}),
                       nw.defined() ? std::optional<Tensor>(nw) : std::nullopt, router, eps);
    return op(Q, K, U, V, R, one_part).transpose(1, 2);
}

// Only where every parameter takes a gradient (block() below): what it saves is then what the steps' own nodes would.
struct BlockNode : torch::autograd::Function<BlockNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w1, const std::optional<Tensor>& norm_weight,
                          const Tensor& router, const Tensor& K, const Tensor& U, const Tensor& V, const Tensor& w2, double eps,
                          bool one_part, int64_t whose_)
    {
        const Whose whose = Whose(whose_);
        const Tensor nw = norm_weight.value_or(Tensor());
        BlockForward f = block_forward(x, w1, nw, router, K, U, V, w2, eps, one_part, whose);
        ctx->save_for_backward({x, w1, nw, router, K, U, V, w2, f.g.x4, f.g.wn, f.g.wr, f.g.q4, f.g.R, f.O4});
        ctx->saved_data["eps"] = eps;
        ctx->saved_data["one_part"] = one_part;
        ctx->saved_data["whose"] = whose_;
        return f.Y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const auto s = ctx->get_saved_variables();
        const Tensor &x = s[0], &w1 = s[1], &nw = s[2], &router = s[3], &K = s[4], &U = s[5], &V = s[6], &w2 = s[7], &x4 = s[8],
                     &wn = s[9], &wr = s[10], &q4 = s[11], &R = s[12];
        const double eps = ctx->saved_data["eps"].toDouble();
        const bool one_part = ctx->saved_data["one_part"].toBool();
        const Whose whose = Whose(ctx->saved_data["whose"].toInt());
        const int64_t hid = x.size(2);
        // What this pass asks for (torch.autograd.grad may name a few inputs): a step whose results nobody asked for is left
        // out, as the engine leaves out a node of its own.  The numbers count the tensors that went in: x, w1, nw if there is
        // one, router, K, U, V, w2.
        const size_t after_nw = nw.defined() ? 3 : 2;
        auto asked = [&](size_t from, size_t to) {
            for (size_t i = from; i < to; ++i)
                if (ctx->needs_input_grad(i)) return true;
            return false;
        };
        const bool prologue = asked(0, after_nw + 1), experts = asked(after_nw + 1, after_nw + 4);
        Tensor dx, dw1, dw2;
        variable_list g(5), h(3);
        // (the products of a linear layer's own backward: d_in = d_out w, d_w = d_out^T in)
        const Tensor dY = grads[0].reshape({-1, hid});
        auto both = [&](bool need_in, bool need_w, const Tensor& d, const Tensor& w, const Tensor& in) -> std::pair<Tensor, Tensor> {
            if (need_in && need_w) return product_pair(d, w, in, whose);
            return {need_in ? product_nn(d, w, whose) : Tensor(), need_w ? product_tn(d, in, whose) : Tensor()};
        };
        const bool need_w2 = asked(after_nw + 4, after_nw + 5);
        {
            Tensor dO, O4 = s[13];      // (dO goes with this scope: the prologue's gradients take its place)
            if (need_w2 && at::GradMode::is_enabled())      // create_graph: dw2 is a function of O, as a linear layer's own backward has it
                O4 = stepwise_O4(x, w1, nw, router, K, U, V, eps, one_part, whose);
            std::tie(dO, dw2) = both(prologue || experts, need_w2, dY, w2, O4.reshape({-1, hid}));
            if (prologue || experts)
                g = op_backward(q4.transpose(1, 2), K, U, V, R, dO.view(s[13].sizes()).transpose(1, 2), K.scalar_type(), one_part);
        }
        if (prologue) {
            h = gate_backward(x4, nw, router, wn, wr, eps, g[0], g[4]);
            std::tie(dx, dw1) = both(ctx->needs_input_grad(0), ctx->needs_input_grad(1), h[0].view({-1, hid}), w1, x.reshape({-1, hid}));
            if (dx.defined()) dx = dx.view(x.sizes());
        }
        return {dx, dw1, h[1], h[2], g[1], g[2], g[3], dw2, Tensor(), Tensor(), Tensor()};
    }
};
Tensor block(const Tensor& x, const Tensor& w1, const std::optional<Tensor>& norm_weight, const Tensor& router, const Tensor& K,
             const Tensor& U, const Tensor& V, const Tensor& w2, double eps, bool one_part, int64_t whose_)
{
    const Whose whose = Whose(whose_);
    const Tensor nw = norm_weight.value_or(Tensor());
    if (!records_grad({&x, &w1, &nw, &router, &K, &U, &V, &w2}))
        return block_forward(x, w1, nw, router, K, U, V, w2, eps, one_part, whose).Y;
    // With anything frozen (adapters, training of the experts alone) the steps record their own nodes: each saves what its
    // own gradients need, and what nobody asks for is neither kept nor computed.
    // So with plain data for x: the node would keep w1 as well, which nothing but dx needs.  (17 us of host time on calls of a few rows,
    // 116 against 99 us of a training call on 32 tokens; from 600 tokens on the GPU takes longer than either.)
    for (const Tensor* t : {&x, &w1, &nw, &router, &K, &U, &V, &w2})
        if (t->defined() && !t->requires_grad())
            return linear(stepwise_O4(x, w1, nw, router, K, U, V, eps, one_part, whose).reshape(x.sizes()), w2, whose);
    return BlockNode::apply(x, w1, norm_weight, router, K, U, V, w2, eps, one_part, whose_);
}

// ---- the decoder's rotary positions --------------------------------------------------------------------------------
struct RopeForward {
    Tensor q, k, v;      // [B, H, S, d] views: q, k of [B, S, H, d] memory, v of qkv itself
};
RopeForward rope_forward(const Tensor& qkv, const Tensor& cos, const Tensor& sin, int64_t H)
{
    TORCH_CHECK(qkv.dim() == 3 && qkv.is_contiguous() && qkv.is_cuda() && cos.is_contiguous() && sin.is_contiguous() &&
                    cos.sizes() == sin.sizes() && cos.dim() == 2 && cos.size(0) == qkv.size(1) && qkv.size(2) == 3 * H * cos.size(1),
                "expected qkv [B,S,3*H*d] contiguous on the GPU and cos, sin [S,d]");
    for (const Tensor* t : {&qkv, &cos, &sin}) {
        TORCH_CHECK_TYPE(t->scalar_type() == at::kBFloat16, "rotary positions are bfloat16 here");
        TORCH_CHECK(t->device() == qkv.device(), "cos and sin must be on the device of qkv, ", qkv.device());
    }
    const int64_t B = qkv.size(0), S = qkv.size(1), d = cos.size(1);
    OnDevice guard(qkv);
    RopeForward f;
    f.q = empty_of({B, S, H, d}, at::kBFloat16, qkv);
    f.k = empty_of({B, S, H, d}, at::kBFloat16, qkv);
    const Tensor src = on_boundary(qkv), c = on_boundary(cos), s = on_boundary(sin);
    raise_for_code(mhffn_rope_fwd(ptr(src), ptr(c), ptr(s), ptr(f.q), ptr(f.k), (int)B, (int)S, (int)H, (int)d, stream()), "mhffn_rope");
    f.q = f.q.transpose(1, 2);
    f.k = f.k.transpose(1, 2);
    f.v = qkv.view({B, S, 3, H, d}).select(2, 2).transpose(1, 2);
    return f;
}
// dqkv [B,S,3*H*d] of gradients of q, k, v [B,H,S,d] of any strides
Tensor rope_backward(Tensor dq, Tensor dk, Tensor dv, const Tensor& cos, const Tensor& sin)
{
    long strides[9];
    Tensor* g[3] = {&dq, &dk, &dv};
    for (int w = 0; w < 3; ++w) {
        if (g[w]->stride(3) != 1) *g[w] = g[w]->contiguous();
        for (int i = 0; i < 3; ++i) strides[3 * w + i] = g[w]->stride(i);
    }
    const int64_t B = dq.size(0), H = dq.size(1), S = dq.size(2), d = dq.size(3);
    OnDevice guard(dq);
    Tensor dqkv = empty_of({B, S, 3 * H * d}, at::kBFloat16, dq);
    raise_for_code(mhffn_rope_bwd(ptr(dq), ptr(dk), ptr(dv), strides, ptr(cos), ptr(sin), ptr(dqkv), (int)B, (int)S, (int)H, (int)d,
                                  stream()),
                   "mhffn_rope");
    return dqkv;
}
std::tuple<Tensor, Tensor, Tensor> rope(const Tensor& qkv, const Tensor& cos, const Tensor& sin, int64_t H);

// The same in torch's operations, for tensors that are more than their memory.
std::tuple<Tensor, Tensor, Tensor> rope_by_elements(const Tensor& qkv, const Tensor& cos, const Tensor& sin, int64_t H)
{
    const int64_t d = cos.size(1), half = d / 2;
    auto rotate = [&](const Tensor& x) {
        return x * cos + at::cat({-x.narrow(-1, half, half), x.narrow(-1, 0, half)}, -1) * sin;
    };
    const Tensor x = qkv.view({qkv.size(0), qkv.size(1), 3, H, d}).permute({2, 0, 3, 1, 4});
    return {rotate(x.select(0, 0)), rotate(x.select(0, 1)), x.select(0, 2)};
}
Tensor rope_backward_by_elements(const Tensor& dq, const Tensor& dk, const Tensor& dv, const Tensor& cos, const Tensor& sin)
{
    const int64_t half = cos.size(1) / 2;
    auto back = [&](const Tensor& g) {
        const Tensor s = g * sin;
        return g * cos + at::cat({s.narrow(-1, half, half), -s.narrow(-1, 0, half)}, -1);
    };
    return at::stack({back(dq), back(dk), dv}, 0).permute({1, 3, 0, 2, 4}).reshape({dq.size(0), dq.size(2), 3 * dq.size(1) * dq.size(3)});
}

// The backward as a node of its own, for create_graph: the map is linear in dq, dk, dv and its transpose is the forward.
struct RopeBackNode : torch::autograd::Function<RopeBackNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& dq, const Tensor& dk, const Tensor& dv, const Tensor& cos, const Tensor& sin)
    {
        ctx->save_for_backward({cos, sin});
        ctx->saved_data["H"] = dq.size(1);
        return rope_backward(dq, dk, dv, cos, sin);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g)
    {
        const auto s = ctx->get_saved_variables();
        auto [q, k, v] = rope(contig(g[0]), s[0], s[1], ctx->saved_data["H"].toInt());
        return {q, k, v, Tensor(), Tensor()};
    }
};

struct RopeNode : torch::autograd::Function<RopeNode> {
    static variable_list forward(AutogradContext* ctx, const Tensor& qkv, const Tensor& cos, const Tensor& sin, int64_t H)
    {
        RopeForward f = rope_forward(qkv, cos, sin, H);
        ctx->save_for_backward({on_boundary(cos), on_boundary(sin)});
        return {f.q, f.k, f.v};
    }
    static variable_list backward(AutogradContext* ctx, variable_list g)
    {
        const auto s = ctx->get_saved_variables();
        Tensor any;
        bool memory = true;
        for (const Tensor& t : g)
            if (t.defined()) {
                any = t;
                memory = memory && memory_alone(t);
            }
        for (Tensor& t : g)
            if (!t.defined()) t = at::zeros_like(any);
        if (!memory) return {rope_backward_by_elements(g[0], g[1], g[2], s[0], s[1]), Tensor(), Tensor(), Tensor()};
        const Tensor dqkv = records_grad({&g[0], &g[1], &g[2]}) ? RopeBackNode::apply(g[0], g[1], g[2], s[0], s[1])
                                                                : rope_backward(g[0], g[1], g[2], s[0], s[1]);
        return {dqkv, Tensor(), Tensor(), Tensor()};
    }
};
std::tuple<Tensor, Tensor, Tensor> rope(const Tensor& qkv, const Tensor& cos, const Tensor& sin, int64_t H)
{
    if (!memory_alone(qkv) || !memory_alone(cos) || !memory_alone(sin)) return rope_by_elements(qkv, cos, sin, H);
    if (!records_grad({&qkv})) {
        RopeForward f = rope_forward(qkv, cos, sin, H);
        return {f.q, f.k, f.v};
    }
    auto out = RopeNode::apply(qkv, cos, sin, H);
    return {out[0], out[1], out[2]};
}

}  // namespace

PYBIND11_MODULE(_native, m)
{
    // (all without the interpreter lock, as a ctypes call is)
    m.def("op_forward", torch::wrap_pybind_function_no_gil(op_forward));
    m.def("op_backward", torch::wrap_pybind_function_no_gil(
                             [](const Tensor& Q, const Tensor& K, const Tensor& U, const Tensor& V, const Tensor& R, const Tensor& dO,
                                bool f32_grad_w, bool one_part) {
                                 return op_backward(Q, K, U, V, R, dO, f32_grad_w ? at::kFloat : at::kBFloat16, one_part);
                             }));
    m.def("op", torch::wrap_pybind_function_no_gil(op));
    m.def("single", torch::wrap_pybind_function_no_gil(single));
    m.def("gate", torch::wrap_pybind_function_no_gil(gate));
    m.def("gate_backward", torch::wrap_pybind_function_no_gil(
                               [](const Tensor& x, const std::optional<Tensor>& norm_weight, const Tensor& router, double eps,
                                  const std::optional<Tensor>& dQ, const std::optional<Tensor>& dR) {
                                   const Tensor nw = norm_weight.value_or(Tensor());
                                   variable_list g = gate_backward(contig(x), nw, router, gate_param(nw), gate_param(router), eps,
                                                                   dQ.value_or(Tensor()), dR.value_or(Tensor()));
                                   return std::make_tuple(g[0], g[1].defined() ? std::optional<Tensor>(g[1]) : std::nullopt, g[2]);
                               }));
    m.def("linear", torch::wrap_pybind_function_no_gil([](const Tensor& x, const Tensor& w, int64_t whose) { return linear(x, w, Whose(whose)); }));
    m.def("rope", torch::wrap_pybind_function_no_gil(rope));
    m.def("block", torch::wrap_pybind_function_no_gil(block));
}
