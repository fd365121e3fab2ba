// C ABI of libmhffn_hip.so: argument validation, error codes, dispatch.  No torch, no pybind, no allocation.
#include "../../include/mhffn.h"
#include "mhffn_common.hpp"
#include "mhffn_product.hpp"

// Scratch of mhffn_bwd_static: device memory that belongs to this code object, so the call needs no allocation.  Every
// GPU the library is loaded on holds its own copy at its own address until the process ends.  In host code the array's
// name is only a handle for hipGetSymbolAddress; kernels get the address that call returned, never the name.
static __device__ __align__(256) unsigned char scratch[MHFFN_STATIC_SCRATCH_BYTES];

namespace {

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int check_dims_impl(const mhffn_dims* d, int dtype)
{
    if (!d) return MHFFN_ERR_NULL_POINTER;
    if (dtype != MHFFN_DTYPE_BF16 && dtype != MHFFN_DTYPE_F32) return MHFFN_ERR_DTYPE;
    if (d->B <= 0 || d->H <= 0 || d->Hkuv <= 0 || d->S <= 0 || d->E <= 0 || d->d_e <= 0 || d->d_h <= 0)
        return MHFFN_ERR_SHAPE;
    if (d->H % d->Hkuv != 0) return MHFFN_ERR_SHAPE;
    if (dtype == MHFFN_DTYPE_F32) {           // fp32 correctness path: generic tiles, no MFMA
        if (d->d_h % 8 != 0 || d->d_h > 128) return MHFFN_ERR_HEAD_DIM;
    } else {
        if (d->d_h != 64 && d->d_h != 96 && d->d_h != 128) return MHFFN_ERR_HEAD_DIM;
        if (d->d_e % 32 != 0) return MHFFN_ERR_EXPERT_DIM;
    }
    // index arithmetic inside the kernels is 64-bit for rows, 32-bit for per-(b,h) token indices and grid extents
    if ((long long)d->B > 65535 || (long long)d->S > (1ll << 30)) return MHFFN_ERR_SHAPE;
    if ((long long)d->B * d->H * d->S >= (1ll << 31)) return MHFFN_ERR_SHAPE;   // token rows are counted in 32 bits
    return MHFFN_OK;
}

mhffn::Dims to_dims(const mhffn_dims* d, int token_layout = 0)
{
    return mhffn::Dims{d->B, d->H, d->Hkuv, d->S, d->d_h, d->E, d->d_e, token_layout};
}

std::atomic<void*> scratch_addr[mhffn::LDS_OPTIN_MAX_DEVICES];   // per device, looked up on the first call there

hipError_t static_scratch_of_current_device(void** out)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= mhffn::LDS_OPTIN_MAX_DEVICES) return hipErrorInvalidDevice;
    void* p = scratch_addr[dev].load(std::memory_order_acquire);
    if (!p) {
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (!p) return hipErrorInvalidSymbol;
        scratch_addr[dev].store(p, std::memory_order_release);
    }
    *out = p;
    return hipSuccess;
}

}  // namespace

extern "C" {

const char* mhffn_strerror(int code)
{
    switch (code) {
        case MHFFN_OK: return "ok";
        case MHFFN_ERR_NULL_POINTER: return "null pointer argument";
        case MHFFN_ERR_DTYPE: return "unsupported dtype (Q, K, U, V must all be bfloat16 or all float32; R float32)";
        case MHFFN_ERR_HEAD_DIM: return "unsupported head dim (bf16: d_h must be 64, 96 or 128; fp32: a multiple of 8 up to 128)";
        case MHFFN_ERR_EXPERT_DIM: return "unsupported expert dim (bf16: d_e must be a multiple of 32)";
        case MHFFN_ERR_SHAPE:
            return "invalid extents (all must be positive, H a multiple of Hkuv; gate kernels: E <= 64), token layout or phase mask";
        case MHFFN_ERR_WORKSPACE: return "workspace missing or too small";
        case MHFFN_ERR_LAUNCH: return "kernel launch failed";
        case MHFFN_ERR_ALIGNMENT: return "pointer not 16-byte aligned";
        case MHFFN_ERR_STATIC_SCRATCH:
            return "problem too large for mhffn_bwd_static's fixed scratch (MHFFN_STATIC_SCRATCH_BYTES); use mhffn_bwd";
    }
    return "unknown error code";
}

int mhffn_is_supported(int d_h, int d_e, int dtype)
{
    if (dtype == MHFFN_DTYPE_F32) return d_h > 0 && d_h % 8 == 0 && d_h <= 128 && d_e > 0;
    if (dtype != MHFFN_DTYPE_BF16) return 0;
    return (d_h == 64 || d_h == 96 || d_h == 128) && d_e > 0 && d_e % 32 == 0;
}

int mhffn_check_dims(const mhffn_dims* dims, int dtype) { return check_dims_impl(dims, dtype); }

size_t mhffn_fwd_workspace_bytes(const mhffn_dims* dims, int dtype)
{
    if (check_dims_impl(dims, dtype) != MHFFN_OK) return 0;
    if (dtype == MHFFN_DTYPE_F32) return mhffn::fwd_workspace_bytes_f32(to_dims(dims));
    return mhffn::fwd_workspace_bytes_bf16(to_dims(dims));
}

size_t mhffn_bwd_workspace_bytes(const mhffn_dims* dims, int dtype)
{
    if (check_dims_impl(dims, dtype) != MHFFN_OK) return 0;
    if (dtype == MHFFN_DTYPE_F32) return mhffn::bwd_workspace_bytes_f32(to_dims(dims));
    return mhffn::bwd_workspace_bytes_bf16(to_dims(dims));
}

size_t mhffn_bwd_workspace_min_bytes(const mhffn_dims* dims, int dtype)
{
    if (check_dims_impl(dims, dtype) != MHFFN_OK) return 0;
    return dtype == MHFFN_DTYPE_F32 ? mhffn::bwd_min_workspace_bytes_f32(to_dims(dims)) : mhffn::bwd_min_workspace_bytes_bf16(to_dims(dims));
}

int mhffn_launch_plan(const mhffn_dims* dims, int dtype, size_t fwd_workspace_bytes, size_t bwd_workspace_bytes, int phases,
                      mhffn_plan* plan)
{
    const int rc = check_dims_impl(dims, dtype);
    if (rc != MHFFN_OK) return rc;
    if (!plan) return MHFFN_ERR_NULL_POINTER;
    if (phases & ~(MHFFN_BWD_ALL | MHFFN_ONE_PART)) return MHFFN_ERR_SHAPE;
    if (bwd_workspace_bytes < mhffn_bwd_workspace_min_bytes(dims, dtype)) return MHFFN_ERR_WORKSPACE;
    const mhffn::Dims d = to_dims(dims);
    const bool f32 = dtype == MHFFN_DTYPE_F32;
    const mhffn::Pick f = f32 ? mhffn::fwd_pick_f32(d, fwd_workspace_bytes, phases) : mhffn::fwd_pick_bf16(d, fwd_workspace_bytes, phases);
    const mhffn::Pick q = f32 ? mhffn::dq_pick_f32(d, bwd_workspace_bytes, phases) : mhffn::dq_pick_bf16(d, bwd_workspace_bytes, phases);
    *plan = mhffn_plan{f.tile_rows, f.nsplit, q.tile_rows, q.nsplit,
                       f32 ? mhffn::dw_slices_f32(d) : mhffn::dw_slices_bf16(d, bwd_workspace_bytes)};
    return MHFFN_OK;
}

int mhffn_launch_forms(const mhffn_dims* dims, int dtype, size_t fwd_workspace_bytes, size_t bwd_workspace_bytes, int phases)
{
    mhffn_plan plan;
    const int rc = mhffn_launch_plan(dims, dtype, fwd_workspace_bytes, bwd_workspace_bytes, phases, &plan);
    if (rc != MHFFN_OK) return rc;
    const mhffn::Dims d = to_dims(dims);
    const mhffn::Pick f{plan.fwd_tile_rows, plan.fwd_parts}, q{plan.dqdr_tile_rows, plan.dqdr_parts};
    const bool f32 = dtype == MHFFN_DTYPE_F32;
    auto padded = [&](const mhffn::Pick& p) { return (f32 ? mhffn::grid_of_part_f32(d, p) : mhffn::whole_xcds(d, p, 2)) != mhffn::tiles_of(d, p); };
    int forms = (padded(f) ? MHFFN_FORM_FWD_PADDED : 0) | (padded(q) ? MHFFN_FORM_DQDR_PADDED : 0);
    if (f32) return forms;
    if (mhffn::fwd_reads_past(d, f)) forms |= MHFFN_FORM_WEIGHTS_PAST_CACHES;
    if (mhffn::dw_token_halves(d, bwd_workspace_bytes)) forms |= MHFFN_FORM_TOKEN_HALVES;
    if (mhffn::gate_fwd_whole_rows(d)) forms |= MHFFN_FORM_GATE_FWD_WHOLE_ROWS;
    if (mhffn::gate_bwd_whole_rows(d)) forms |= MHFFN_FORM_GATE_BWD_WHOLE_ROWS;
    return forms;
}

int mhffn_fwd_layout(const void* Q, const void* K, const void* U, const void* V, const float* R, void* O,
                     void* workspace, size_t workspace_bytes, const mhffn_dims* dims, int dtype, int token_layout,
                     void* stream, int phases)
{
    const int rc = check_dims_impl(dims, dtype);
    if (rc != MHFFN_OK) return rc;
    if (token_layout != MHFFN_TOKENS_BHSD && token_layout != MHFFN_TOKENS_BSHD) return MHFFN_ERR_SHAPE;
    if (phases & ~(MHFFN_FWD_ALL | MHFFN_ONE_PART)) return MHFFN_ERR_SHAPE;       // a bit this build does not define: refuse, do not ignore
    if (!Q || !K || !U || !V || !R || !O) return MHFFN_ERR_NULL_POINTER;
    if (!aligned16(Q) || !aligned16(K) || !aligned16(U) || !aligned16(V) || !aligned16(R) || !aligned16(O) ||
        !aligned16(workspace))
        return MHFFN_ERR_ALIGNMENT;
    const mhffn::Dims d = to_dims(dims, token_layout);
    if (dtype == MHFFN_DTYPE_F32) {
        if (!(phases & MHFFN_FWD_MAIN)) return MHFFN_OK;
        return mhffn::launch_fwd_f32(Q, K, U, V, R, O, workspace, workspace_bytes, d, (hipStream_t)stream, phases) == hipSuccess
                   ? MHFFN_OK
                   : MHFFN_ERR_LAUNCH;
    }
    const hipError_t err = mhffn::launch_fwd_bf16(Q, K, U, V, R, O, workspace, workspace_bytes, d, (hipStream_t)stream, phases);
    return err == hipSuccess ? MHFFN_OK : MHFFN_ERR_LAUNCH;
}

int mhffn_fwd_phases(const void* Q, const void* K, const void* U, const void* V, const float* R, void* O,
                     void* workspace, size_t workspace_bytes, const mhffn_dims* dims, int dtype, void* stream,
                     int phases)
{
    return mhffn_fwd_layout(Q, K, U, V, R, O, workspace, workspace_bytes, dims, dtype, MHFFN_TOKENS_BHSD, stream, phases);
}

int mhffn_fwd(const void* Q, const void* K, const void* U, const void* V, const float* R, void* O,
              void* workspace, size_t workspace_bytes, const mhffn_dims* dims, int dtype, void* stream)
{
    return mhffn_fwd_phases(Q, K, U, V, R, O, workspace, workspace_bytes, dims, dtype, stream, MHFFN_FWD_ALL);
}

int mhffn_bwd_layout(const void* Q, const void* K, const void* U, const void* V, const float* R, const void* dO,
                     void* dQ, void* dK, void* dU, void* dV, float* dR, int grad_w_dtype,
                     void* workspace, size_t workspace_bytes, const mhffn_dims* dims, int dtype, int token_layout,
                     void* stream, int phases)
{
    const int rc = check_dims_impl(dims, dtype);
    if (rc != MHFFN_OK) return rc;
    if (token_layout != MHFFN_TOKENS_BHSD && token_layout != MHFFN_TOKENS_BSHD) return MHFFN_ERR_SHAPE;
    if (grad_w_dtype != MHFFN_DTYPE_BF16 && grad_w_dtype != MHFFN_DTYPE_F32) return MHFFN_ERR_DTYPE;
    if (phases & ~(MHFFN_BWD_ALL | MHFFN_ONE_PART)) return MHFFN_ERR_SHAPE;       // a bit this build does not define: refuse, do not ignore
    if (!Q || !K || !U || !V || !R || !dO || !dQ || !dK || !dU || !dV || !dR) return MHFFN_ERR_NULL_POINTER;
    const void* ptrs[] = {Q, K, U, V, R, dO, dQ, dK, dU, dV, dR, workspace};
    for (const void* p : ptrs)
        if (!aligned16(p)) return MHFFN_ERR_ALIGNMENT;
    const mhffn::Dims d = to_dims(dims, token_layout);
    const size_t ws_bytes = workspace ? workspace_bytes : 0;
    if (ws_bytes < mhffn_bwd_workspace_min_bytes(dims, dtype)) return MHFFN_ERR_WORKSPACE;
    if (dtype == MHFFN_DTYPE_F32)
        return mhffn::launch_bwd_f32(Q, K, U, V, R, dO, dQ, dK, dU, dV, dR, grad_w_dtype == MHFFN_DTYPE_F32, workspace,
                                     ws_bytes, d, (hipStream_t)stream, phases) == hipSuccess
                   ? MHFFN_OK
                   : MHFFN_ERR_LAUNCH;
    const hipError_t err = mhffn::launch_bwd_bf16(Q, K, U, V, R, dO, dQ, dK, dU, dV, dR,
                                                  grad_w_dtype == MHFFN_DTYPE_F32, workspace, ws_bytes, d,
                                                  (hipStream_t)stream, phases);
    return err == hipSuccess ? MHFFN_OK : MHFFN_ERR_LAUNCH;
}

int mhffn_bwd_static(const void* Q, const void* K, const void* U, const void* V, const float* R, const void* dO,
                     void* dQ, void* dK, void* dU, void* dV, float* dR, int grad_w_dtype,
                     const mhffn_dims* dims, int dtype, int token_layout, void* stream)
{
    const int rc = check_dims_impl(dims, dtype);
    if (rc != MHFFN_OK) return rc;
    if (token_layout != MHFFN_TOKENS_BHSD && token_layout != MHFFN_TOKENS_BSHD) return MHFFN_ERR_SHAPE;
    if (grad_w_dtype != MHFFN_DTYPE_BF16 && grad_w_dtype != MHFFN_DTYPE_F32) return MHFFN_ERR_DTYPE;
    if (!Q || !K || !U || !V || !R || !dO || !dQ || !dK || !dU || !dV || !dR) return MHFFN_ERR_NULL_POINTER;
    const void* ptrs[] = {Q, K, U, V, R, dO, dQ, dK, dU, dV, dR};
    for (const void* p : ptrs)
        if (!aligned16(p)) return MHFFN_ERR_ALIGNMENT;
    const mhffn::Dims d = to_dims(dims, token_layout);
    // The bfloat16 launch runs with as many token slices and parts as the array holds partial sums for (with one it needs
    // none), so it never exceeds the array.  So does the float32 launch with its parts; its token slices are fixed.
    const size_t need = dtype == MHFFN_DTYPE_F32 ? mhffn::bwd_min_workspace_bytes_f32(d) : 0;
    if (need > MHFFN_STATIC_SCRATCH_BYTES) return MHFFN_ERR_STATIC_SCRATCH;
    void* ws = nullptr;
    if (static_scratch_of_current_device(&ws) != hipSuccess) return MHFFN_ERR_LAUNCH;
    hipError_t err;
    if (dtype == MHFFN_DTYPE_F32)
        err = mhffn::launch_bwd_f32(Q, K, U, V, R, dO, dQ, dK, dU, dV, dR, grad_w_dtype == MHFFN_DTYPE_F32, ws,
                                    (size_t)MHFFN_STATIC_SCRATCH_BYTES, d, (hipStream_t)stream, MHFFN_BWD_ALL);
    else
        err = mhffn::launch_bwd_bf16(Q, K, U, V, R, dO, dQ, dK, dU, dV, dR, grad_w_dtype == MHFFN_DTYPE_F32, ws,
                                     (size_t)MHFFN_STATIC_SCRATCH_BYTES, d, (hipStream_t)stream, MHFFN_BWD_ALL);
    return err == hipSuccess ? MHFFN_OK : MHFFN_ERR_LAUNCH;
}

int mhffn_bwd_phases(const void* Q, const void* K, const void* U, const void* V, const float* R, const void* dO,
                     void* dQ, void* dK, void* dU, void* dV, float* dR, int grad_w_dtype,
                     void* workspace, size_t workspace_bytes, const mhffn_dims* dims, int dtype, void* stream,
                     int phases)
{
    return mhffn_bwd_layout(Q, K, U, V, R, dO, dQ, dK, dU, dV, dR, grad_w_dtype, workspace, workspace_bytes, dims, dtype,
                            MHFFN_TOKENS_BHSD, stream, phases);
}

int mhffn_bwd(const void* Q, const void* K, const void* U, const void* V, const float* R, const void* dO,
              void* dQ, void* dK, void* dU, void* dV, float* dR, int grad_w_dtype,
              void* workspace, size_t workspace_bytes, const mhffn_dims* dims, int dtype, void* stream)
{
    return mhffn_bwd_phases(Q, K, U, V, R, dO, dQ, dK, dU, dV, dR, grad_w_dtype, workspace, workspace_bytes, dims,
                            dtype, stream, MHFFN_BWD_ALL);
}

static int check_gate_dims(const mhffn_dims* d)
{
    if (!d) return MHFFN_ERR_NULL_POINTER;
    if (d->B <= 0 || d->H <= 0 || d->S <= 0 || d->E <= 0 || d->d_h <= 0) return MHFFN_ERR_SHAPE;
    if (d->d_h != 64 && d->d_h != 96 && d->d_h != 128) return MHFFN_ERR_HEAD_DIM;
    if (d->E > 64 || d->B > 65535 || d->H > 65535 || (long long)d->S > (1ll << 30)) return MHFFN_ERR_SHAPE;
    if ((long long)d->B * d->H * d->S >= (1ll << 31)) return MHFFN_ERR_SHAPE;
    return MHFFN_OK;
}

static bool param_dtypes_ok(int norm_dtype, int router_dtype)
{
    return (norm_dtype == MHFFN_DTYPE_BF16 || norm_dtype == MHFFN_DTYPE_F32) &&
           (router_dtype == MHFFN_DTYPE_BF16 || router_dtype == MHFFN_DTYPE_F32);
}

int mhffn_gate_fwd_typed(const void* X, const void* norm_weight, int norm_dtype, float eps, const void* router, int router_dtype,
                         void* Qn, float* R, const mhffn_dims* dims, void* stream)
{
    const int rc = check_gate_dims(dims);
    if (rc != MHFFN_OK) return rc;
    if (!param_dtypes_ok(norm_dtype, router_dtype)) return MHFFN_ERR_DTYPE;
    if (!X || !router || !R || (norm_weight && !Qn)) return MHFFN_ERR_NULL_POINTER;
    if (!aligned16(X) || !aligned16(Qn) || !aligned16(R) || !aligned16(router) || !aligned16(norm_weight))
        return MHFFN_ERR_ALIGNMENT;
    return mhffn::launch_gate_fwd(X, norm_weight, norm_dtype == MHFFN_DTYPE_BF16, eps, router, router_dtype == MHFFN_DTYPE_BF16, Qn, R,
                                  to_dims(dims), (hipStream_t)stream) == hipSuccess
               ? MHFFN_OK
               : MHFFN_ERR_LAUNCH;
}

int mhffn_gate_fwd(const void* X, const float* norm_weight, float eps, const float* router, void* Qn, float* R,
                   const mhffn_dims* dims, void* stream)
{
    return mhffn_gate_fwd_typed(X, norm_weight, MHFFN_DTYPE_F32, eps, router, MHFFN_DTYPE_F32, Qn, R, dims, stream);
}

static int gate_bwd(const void* X, const void* norm_weight, int norm_dtype, float eps, const void* router, int router_dtype,
                    const void* dQ, int dq_token_layout, const float* dR, void* dX, void* d_norm_weight, void* d_router, void* workspace,
                    const mhffn_dims* dims, void* stream)
{
    if (dq_token_layout != MHFFN_TOKENS_BHSD && dq_token_layout != MHFFN_TOKENS_BSHD) return MHFFN_ERR_SHAPE;
    if (!X || !router || !dQ || !dR || !dX || !d_router || (norm_weight && !d_norm_weight)) return MHFFN_ERR_NULL_POINTER;
    const void* ptrs[] = {X, norm_weight, router, dQ, dR, dX, d_norm_weight, d_router, workspace};
    for (const void* p : ptrs)
        if (!aligned16(p)) return MHFFN_ERR_ALIGNMENT;
    return mhffn::launch_gate_bwd(X, norm_weight, norm_dtype == MHFFN_DTYPE_BF16, eps, router, router_dtype == MHFFN_DTYPE_BF16, dQ,
                                  dq_token_layout, dR, dX, d_norm_weight, d_router, workspace, to_dims(dims), (hipStream_t)stream) == hipSuccess
               ? MHFFN_OK
               : MHFFN_ERR_LAUNCH;
}

int mhffn_gate_bwd(const void* X, const float* norm_weight, float eps, const float* router, const void* dQ,
                   int dq_token_layout, const float* dR, void* dX, float* d_norm_weight, float* d_router,
                   const mhffn_dims* dims, void* stream)
{
    const int rc = check_gate_dims(dims);
    if (rc != MHFFN_OK) return rc;
    return gate_bwd(X, norm_weight, MHFFN_DTYPE_F32, eps, router, MHFFN_DTYPE_F32, dQ, dq_token_layout, dR, dX, d_norm_weight, d_router,
                    nullptr, dims, stream);
}

size_t mhffn_gate_bwd_workspace_bytes(const mhffn_dims* dims)
{
    return check_gate_dims(dims) == MHFFN_OK ? mhffn::gate_bwd_workspace_bytes(to_dims(dims)) : 0;
}

int mhffn_gate_bwd_into(const void* X, const void* norm_weight, int norm_dtype, float eps, const void* router, int router_dtype,
                        const void* dQ, int dq_token_layout, const float* dR, void* dX, void* d_norm_weight, void* d_router, void* workspace,
                        size_t workspace_bytes, const mhffn_dims* dims, void* stream)
{
    const int rc = check_gate_dims(dims);
    if (rc != MHFFN_OK) return rc;
    if (!param_dtypes_ok(norm_dtype, router_dtype)) return MHFFN_ERR_DTYPE;
    if (!workspace || workspace_bytes < mhffn::gate_bwd_workspace_bytes(to_dims(dims))) return MHFFN_ERR_WORKSPACE;
    return gate_bwd(X, norm_weight, norm_dtype, eps, router, router_dtype, dQ, dq_token_layout, dR, dX, d_norm_weight, d_router,
                    workspace, dims, stream);
}

static int check_rope_dims(int B, int S, int H, int d)
{
    if (B <= 0 || S <= 0 || H <= 0 || d <= 0 || (double)B * S * H * (d / 16) >= 2147483648.0) return MHFFN_ERR_SHAPE;
    return d % 16 == 0 ? MHFFN_OK : MHFFN_ERR_HEAD_DIM;
}

int mhffn_rope_fwd(const void* qkv, const void* cos, const void* sin, void* q, void* k, int B, int S, int H, int d, void* stream)
{
    const int rc = check_rope_dims(B, S, H, d);
    if (rc != MHFFN_OK) return rc;
    const void* ptrs[] = {qkv, cos, sin, q, k};
    for (const void* p : ptrs) {
        if (!p) return MHFFN_ERR_NULL_POINTER;
        if (!aligned16(p)) return MHFFN_ERR_ALIGNMENT;
    }
    return mhffn::launch_rope_fwd(qkv, cos, sin, q, k, B, S, H, d, (hipStream_t)stream) == hipSuccess ? MHFFN_OK : MHFFN_ERR_LAUNCH;
}

int mhffn_rope_bwd(const void* dq, const void* dk, const void* dv, const long* strides, const void* cos, const void* sin, void* dqkv,
                   int B, int S, int H, int d, void* stream)
{
    const int rc = check_rope_dims(B, S, H, d);
    if (rc != MHFFN_OK) return rc;
    if (!dq || !dk || !dv || !strides || !cos || !sin || !dqkv) return MHFFN_ERR_NULL_POINTER;
    if (!aligned16(cos) || !aligned16(sin) || !aligned16(dqkv)) return MHFFN_ERR_ALIGNMENT;
    const void* grads[3] = {dq, dk, dv};
    return mhffn::launch_rope_bwd(grads, reinterpret_cast<const long(*)[3]>(strides), cos, sin, dqkv, B, S, H, d,
                                  (hipStream_t)stream) == hipSuccess
               ? MHFFN_OK
               : MHFFN_ERR_LAUNCH;
}

int mhffn_product_preferred(int M, int N) { return M > 0 && N > 0 && mhffn::product_preferred(M, N); }

static int check_product(int form, int M, int N, int K)
{
    if (form != MHFFN_PRODUCT_NT && form != MHFFN_PRODUCT_NN && form != MHFFN_PRODUCT_TN) return MHFFN_ERR_SHAPE;
    const int ld = form == MHFFN_PRODUCT_TN ? M : K;      // with N the lengths of the rows in memory
    if (M <= 0 || N <= 0 || K <= 0 || N % 8 != 0 || ld % 8 != 0) return MHFFN_ERR_SHAPE;
    // (a stage's lane offsets, at most 128 rows, are 32-bit, and so is the number of tiles)
    if (N > (1 << 22) || ld > (1 << 22) || (double)M * N >= 1024.0 * 2147483648.0) return MHFFN_ERR_SHAPE;
    return MHFFN_OK;
}

int mhffn_product_tile(int form, int in_order, int M, int N, int K)
{
    return check_product(form, M, N, K) == MHFFN_OK ? mhffn::product_tile(form, in_order != 0, M, N, K) : 0;
}

int mhffn_product_faster(int form, int in_order, int M, int N, int K)
{
    return check_product(form, M, N, K) == MHFFN_OK && mhffn::product_faster(form, in_order != 0, M, N, K);
}

int mhffn_product(int form, int in_order, const void* A, const void* B, void* C, int M, int N, int K, void* stream)
{
    const int rc = check_product(form, M, N, K);
    if (rc != MHFFN_OK) return rc;
    const void* ptrs[] = {A, B, C};
    for (const void* p : ptrs) {
        if (!p) return MHFFN_ERR_NULL_POINTER;
        if (!aligned16(p)) return MHFFN_ERR_ALIGNMENT;
    }
    return mhffn::launch_product(form, in_order != 0, A, B, C, M, N, K, (hipStream_t)stream) == hipSuccess ? MHFFN_OK : MHFFN_ERR_LAUNCH;
}

static int check_pair(int M, int N, int K)
{
    const int rc = check_product(MHFFN_PRODUCT_NN, M, K, N);
    return rc == MHFFN_OK ? check_product(MHFFN_PRODUCT_TN, N, K, M) : rc;
}

int mhffn_product_pair_faster(int in_order, int M, int N, int K)
{
    return check_pair(M, N, K) == MHFFN_OK && mhffn::product_pair_faster(in_order != 0, M, N, K);
}

int mhffn_product_pair(const void* dy, const void* w, const void* x, void* dx, void* dw, int M, int N, int K, void* stream)
{
    const int rc = check_pair(M, N, K);
    if (rc != MHFFN_OK) return rc;
    const void* ptrs[] = {dy, w, x, dx, dw};
    for (const void* p : ptrs) {
        if (!p) return MHFFN_ERR_NULL_POINTER;
        if (!aligned16(p)) return MHFFN_ERR_ALIGNMENT;
    }
    return mhffn::launch_product_pair(dy, w, x, dx, dw, M, N, K, (hipStream_t)stream) == hipSuccess ? MHFFN_OK : MHFFN_ERR_LAUNCH;
}

}  // extern "C"
