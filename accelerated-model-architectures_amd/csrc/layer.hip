// The layer's forward and backward as one call each: the launches of the single ops in their order, on buffers that the caller
// has laid out.  Host code only.  A pass of a handful of tokens is as long as what the host does between its launches; with one
// call per op that is a dozen trips through the language binding, its argument checks and allocations.  Forward of 7 tokens through
// 128 experts of H = 576, I = 256: 83 -> 35 us, the time of its five kernels; forward and backward of small layers 375 -> 238.
#include "common.hpp"

namespace {

#define RUN(call)              \
    do {                       \
        const int rc = (call); \
        if (rc) return rc;     \
    } while (0)

// forward-type GEMM through the entry point that the caller has chosen
int gemm(const xma_rocm_moe *m, int64_t few, const void *X, const void *W, int64_t w_es, int64_t ldw, int w_is_kn, void *out, void *aux,
         int64_t ldaux, void *aux2, const void *scale, const void *bias, int64_t N, int64_t K, int64_t fan_out, int x_grouped, int y_grouped,
         int epilogue, void *stream, float *dots = nullptr) {
    const int64_t M = m->T * m->k, ldo = epilogue == XMA_ROCM_EPI_SWIGLU_BWD ? 2 * N : N;
    if (epilogue >= XMA_ROCM_EPI_GELU_TANH && !few) { // no epilogue of the 256 x 256 kernels: a pass of its own
        const int form = epilogue >= XMA_ROCM_EPI_GELU_ERF, bwd = epilogue & 1;
        RUN(gemm(m, 0, X, W, w_es, ldw, w_is_kn, out, nullptr, 0, nullptr, scale, bias, N, K, fan_out, x_grouped, y_grouped, XMA_ROCM_EPI_STORE, stream));
        return bwd ? xma_rocm_gelu_backward(aux, out, out, M * N, form, (int)m->dtype, stream) : xma_rocm_gelu_forward(out, aux, M * N, form, (int)m->dtype, stream);
    }
    const int64_t *idx = (const int64_t *)m->sorted_scattered_idxs, *offs = (const int64_t *)m->expert_offsets;
    if (few)
        return xma_rocm_scatter2scatter_few_rows(X, K, W, w_es, ldw, w_is_kn, idx, offs, out, ldo, aux, ldaux, aux2, aux2 ? N : 0, scale, bias,
                                                 bias ? N : 0, M, (int32_t)N, (int32_t)K, (int32_t)m->E, (int32_t)fan_out, x_grouped, y_grouped,
                                                 epilogue, (int)m->dtype, m->workspace, (size_t)m->workspace_bytes, stream);
    if (dots)
        return xma_down_projection_dx_dots(X, K, W, w_es, ldw, idx, offs, aux, ldaux, out, ldo, aux2, N, scale, M, (int32_t)N, (int32_t)K,
                                           (int32_t)m->E, (int32_t)fan_out, (int)m->dtype, m->workspace, (size_t)m->workspace_bytes, stream, dots);
    // the 256 x 256 kernels split the last round of tiles where there is a workspace, and refuse one that is too small for it
    if (aux2)
        return xma_rocm_down_projection_dx_swiglu(X, K, W, w_es, ldw, idx, offs, aux, ldaux, out, ldo, aux2, N, scale, M, (int32_t)N, (int32_t)K,
                                                  (int32_t)m->E, (int32_t)fan_out, (int)m->dtype, m->workspace, (size_t)m->workspace_bytes, stream);
    return xma_rocm_scatter2scatter_bias(X, K, W, w_es, ldw, w_is_kn, idx, offs, out, ldo, aux, ldaux, scale, bias, bias ? N : 0, M, (int32_t)N,
                                         (int32_t)K, (int32_t)m->E, (int32_t)fan_out, x_grouped, y_grouped, epilogue, (int)m->dtype,
                                         m->workspace, (size_t)m->workspace_bytes, stream);
}

// Before a pass's first launch: the workspace holds the K slices of a GEMM by the 256 x 256 kernels (0 bytes: none, and without a
// workspace at all they split nothing).  Few-row launches and route check it themselves.
int check_workspace(const xma_rocm_moe *m, int64_t few, int64_t N, int64_t K, const char *what) {
    if (few || !m->workspace || m->dtype == XMA_ROCM_F32) return XMA_ROCM_OK;
    const size_t need = xma_rocm_scatter2scatter_workspace_bytes(m->T * m->k, (int32_t)N, (int32_t)K, (int32_t)m->E);
    XMA_REQUIRE((size_t)m->workspace_bytes >= need, XMA_ROCM_EWORKSPACE, "%s: workspace of %lld bytes, %zu needed", what,
                (long long)m->workspace_bytes, need);
    return XMA_ROCM_OK;
}

int dw(const xma_rocm_moe *m, int64_t few, const void *DY, int dy_grouped, const void *scale, const void *X, int x_grouped, void *DW,
       int64_t N_out, int64_t K_in, void *stream) {
    const int64_t *idx = (const int64_t *)m->sorted_scattered_idxs, *offs = (const int64_t *)m->expert_offsets;
    const int32_t dy_fan = dy_grouped ? 1 : (int32_t)m->k, x_fan = x_grouped ? 1 : (int32_t)m->k;
    if (few)
        return xma_rocm_group_bwd_W_few_rows(DY, N_out, dy_grouped, dy_fan, scale, X, K_in, x_grouped, x_fan, idx, offs, DW, N_out * K_in, K_in,
                                             (int32_t)N_out, (int32_t)K_in, (int32_t)m->E, m->T * m->k, (int)m->dtype, stream);
    return xma_group_bwd_W(DY, N_out, dy_grouped, dy_fan, scale, X, K_in, x_grouped, x_fan, idx, offs, DW, N_out * K_in, K_in, (int32_t)N_out,
                           (int32_t)K_in, (int32_t)m->E, m->T * m->k, (int)m->dtype, stream);
}

int down_projection(const xma_rocm_moe *m, void *stream) {
    return gemm(m, m->few_down, m->h, m->w_proj, m->H * m->I, m->I, 0, m->expert_out, nullptr, 0, nullptr, nullptr, m->b_proj, m->H, m->I, 1, 1, 0,
                XMA_ROCM_EPI_STORE, stream);
}

int check(const xma_rocm_moe *m, const char *what) {
    XMA_REQUIRE(m && m->size == (int64_t)sizeof(xma_rocm_moe), XMA_ROCM_EINVAL, "%s: argument block of another size", what);
    XMA_REQUIRE(m->T >= 1 && m->T < ((int64_t)1 << 31) && m->H >= 8 && m->I >= 8 && m->E >= 1 && m->k >= 1 && m->k <= m->E && m->T * m->k < ((int64_t)1 << 31) &&
                    m->H < ((int64_t)1 << 30) && m->I < ((int64_t)1 << 29) && m->E <= 16384,
                XMA_ROCM_EINVAL, "%s: T=%lld H=%lld I=%lld E=%lld k=%lld", what, (long long)m->T, (long long)m->H, (long long)m->I,
                (long long)m->E, (long long)m->k);
    XMA_REQUIRE(m->workspace_bytes >= 0, XMA_ROCM_EINVAL, "%s: workspace of %lld bytes", what, (long long)m->workspace_bytes);
    XMA_REQUIRE(m->x && m->w_fc && m->w_proj && m->router_weights && m->expert_ids && m->expert_offsets && m->sorted_scattered_idxs && m->z &&
                    m->expert_out,
                XMA_ROCM_EINVAL, "%s: null buffer", what);
    XMA_REQUIRE(m->activation == 0 || ((m->activation == 1 || m->activation == 2) && !m->recompute && m->dw2_form != 1), XMA_ROCM_EINVAL,
                "%s: activation %lld goes without recomputation and scaled activations", what, (long long)m->activation);
    return XMA_ROCM_OK;
}

int64_t up_width(const xma_rocm_moe *m) { return m->activation ? m->I : 2 * m->I; }
int epilogue_of(const xma_rocm_moe *m, int bwd) {
    if (m->activation == 0) return bwd ? XMA_ROCM_EPI_SWIGLU_BWD : XMA_ROCM_EPI_SWIGLU;
    return (m->activation == 1 ? XMA_ROCM_EPI_GELU_TANH : XMA_ROCM_EPI_GELU_ERF) + bwd;
}

} // namespace

extern "C" int xma_rocm_moe_forward(const xma_rocm_moe *m, void *stream) {
    RUN(check(m, "moe_forward"));
    XMA_REQUIRE(m->logits && m->h && m->y && m->counts, XMA_ROCM_EINVAL, "moe_forward: null buffer");
    const int dtype = (int)m->dtype;
    const int64_t M = m->T * m->k, U = up_width(m);
    RUN(check_workspace(m, m->few_up, U, m->H, "moe_forward"));
    RUN(check_workspace(m, m->few_down, m->H, m->I, "moe_forward"));
    if (m->gate_weight) {
        RUN(xma_router_gate_route(m->x, m->H, m->gate_weight, m->H, m->T, (int32_t)m->H, (int32_t)m->E, (int32_t)m->k, dtype, m->logits, m->E,
                                  m->router_weights, m->expert_ids, (uint32_t *)m->counts, (int64_t *)m->expert_offsets,
                                  (int64_t *)m->sorted_scattered_idxs, m->workspace, (size_t)m->workspace_bytes, stream));
    } else {
        RUN(xma_rocm_router_topk(m->logits, m->E, m->T, (int32_t)m->E, (int32_t)m->k, dtype, m->router_weights, m->expert_ids, 0, stream));
        RUN(xma_rocm_route(m->expert_ids, 0, M, (int32_t)m->E, (uint32_t *)m->counts, (int64_t *)m->expert_offsets, nullptr, nullptr,
                           (int64_t *)m->sorted_scattered_idxs, m->workspace, (size_t)m->workspace_bytes, stream));
    }
    RUN(gemm(m, m->few_up, m->x, m->w_fc, U * m->H, m->H, 0, m->z, m->h, m->I, nullptr, nullptr, m->b_fc, U, m->H, m->k, 0, 1, epilogue_of(m, 0), stream));
    RUN(down_projection(m, stream));
    return xma_rocm_combine(m->expert_out, m->H, m->router_weights, m->y, m->H, m->T, (int32_t)m->k, (int32_t)m->H, dtype, stream);
}

static int check_recompute(const xma_rocm_moe *m, const char *what, bool dots) {
    return m->recompute && !dots ? check_workspace(m, m->few_down, m->H, m->I, what) : XMA_ROCM_OK;
}
// The activations and expert outputs again where neither was kept: h from z, the expert outputs by the down-projection.  Where dX2
// leaves the router weights' gradient (`dots`), nothing reads the expert outputs, and h only dW2.
static int recompute(const xma_rocm_moe *m, bool dots, void *stream) {
    if (!m->recompute) return XMA_ROCM_OK;
    if (!dots || m->dw2_form != 1)
        RUN(xma_rocm_swiglu_packed_forward(m->z, 2 * m->I, m->h, m->I, m->T * m->k, (int32_t)m->I, (int)m->dtype, stream));
    return dots ? XMA_ROCM_OK : down_projection(m, stream);
}

static int64_t dots_parts(const xma_rocm_moe *m) { return (m->I + 127) / 128; }

// Where dX2 by the 256 x 256 kernels leaves <d h, h> of each row and 128 columns: in the workspace, behind the K slices of that launch, if it
// is large enough.  A bias of the down-projection would add <dy, bias> to the gradient, which <d h, h> lacks.
static float *dots_place(const xma_rocm_moe *m) {
    if (m->few_dx2 || m->activation || m->b_proj || m->dtype == XMA_ROCM_F32 || !m->workspace || m->k > 32) return nullptr;
    const int64_t M = m->T * m->k, I = m->I, H = m->H, E = m->E;
    if (M * dots_parts(m) >= ROUTER_GRADIENT_MAX) return nullptr;
    const size_t need = xma_rocm_down_projection_dx_swiglu_router_workspace_bytes(M, (int32_t)I, (int32_t)H, (int32_t)E);
    return (size_t)m->workspace_bytes >= need ? (float *)((char *)m->workspace + need) - M * dots_parts(m) : nullptr;
}

// The gradient of the router's logits: what the gate's own products need before the rest of the backward.
extern "C" int xma_rocm_moe_backward_router(const xma_rocm_moe *m, void *stream) {
    RUN(check(m, "moe_backward_router"));
    XMA_REQUIRE(m->logits && m->dy && m->d_router_weights && m->d_logits && (!m->recompute || m->h), XMA_ROCM_EINVAL,
                "moe_backward_router: null buffer");
    const int dtype = (int)m->dtype;
    RUN(check_recompute(m, "moe_backward_router", false));
    RUN(recompute(m, false, stream));
    RUN(xma_rocm_combine_bwd(m->expert_out, m->H, m->dy, m->H, m->d_router_weights, m->T, (int32_t)m->k, (int32_t)m->H, dtype, stream));
    return xma_rocm_router_topk_bwd(m->logits, m->E, m->T, (int32_t)m->E, (int32_t)m->k, dtype, m->expert_ids, 0, m->d_router_weights, m->d_logits,
                                    m->E, stream);
}

// What the part below asks of its arguments, before the first launch.
static int check_experts(const xma_rocm_moe *m, const char *what) {
    XMA_REQUIRE(m->dy && m->dz && m->d_w_fc && m->d_w_proj && m->scattered && m->d_x && (m->dw2_form == 1 || m->h) &&
                    (m->dw2_form == 0 || m->dw2_operand) && (!m->d_b_fc || m->b_fc) && (!m->d_b_proj || m->b_proj),
                XMA_ROCM_EINVAL, "%s: null buffer", what);
    // the column sums that make d_b_proj want dy scaled, in a copy or beside the scaled activations: the loader of form 0 keeps none
    XMA_REQUIRE(m->dw2_form >= 0 && m->dw2_form <= 2 && !(m->dw2_form == 0 && m->d_b_proj), XMA_ROCM_EINVAL,
                "%s: dw2_form %lld%s", what, (long long)m->dw2_form, m->d_b_proj ? " with d_b_proj (forms 1 and 2 only)" : "");
    RUN(check_workspace(m, m->few_dx2, m->I, m->H, what));
    return check_workspace(m, m->few_dx1, m->H, up_width(m), what);
}

// Everything of the backward between the router's part and the sum over the k slots: `scattered` holds dX1 then.  With `dots`, d_router_weights
// too: the router weights' gradient or, with logits, that of the selected logits.
static int backward_experts(const xma_rocm_moe *m, float *dots, const void *logits, void *stream) {
    const int dtype = (int)m->dtype;
    const int64_t M = m->T * m->k, H = m->H, I = m->I, U = up_width(m);
    const int64_t *idx = (const int64_t *)m->sorted_scattered_idxs, *offs = (const int64_t *)m->expert_offsets;
    // dX2 + SwiGLU', with the scaled activations for dW2 where that takes dy through the index
    RUN(gemm(m, m->few_dx2, m->dy, m->w_proj, H * I, I, 1, m->dz, m->z, U, m->dw2_form == 1 ? m->dw2_operand : nullptr, m->router_weights,
             nullptr, I, H, m->k, 0, 1, epilogue_of(m, 1), stream, dots));
    if (dots) // before dX1, whose K slices take their place
        RUN(xma_dots_router_bwd(dots, dots_parts(m), logits, (const int32_t *)m->expert_ids, m->T, (int32_t)m->E, (int32_t)m->k, dtype,
                                m->d_router_weights, (hipStream_t)stream));
    if (m->dw2_form == 1) {
        RUN(dw(m, m->few_dw2, m->dy, 0, nullptr, m->dw2_operand, 1, m->d_w_proj, H, I, stream));
        if (m->d_b_proj)
            RUN(xma_rocm_expert_column_sums(m->dy, H, idx, (int32_t)m->k, m->router_weights, offs, m->d_b_proj, H, (int32_t)H, (int32_t)m->E, dtype, stream));
    } else if (m->dw2_form == 2) { // a scaled grouped copy of dy
        RUN(xma_rocm_group(m->dy, H, idx, m->dw2_operand, H, m->router_weights, M, (int32_t)H, (int32_t)m->k, dtype, stream));
        RUN(dw(m, m->few_dw2, m->dw2_operand, 1, nullptr, m->h, 1, m->d_w_proj, H, I, stream));
        if (m->d_b_proj)
            RUN(xma_rocm_expert_column_sums(m->dw2_operand, H, nullptr, 1, nullptr, offs, m->d_b_proj, H, (int32_t)H, (int32_t)m->E, dtype, stream));
    } else { // the loader of the few-row kernel gathers and scales
        RUN(dw(m, m->few_dw2, m->dy, 0, m->router_weights, m->h, 1, m->d_w_proj, H, I, stream));
    }
    RUN(dw(m, m->few_dw1, m->dz, 1, nullptr, m->x, 0, m->d_w_fc, U, H, stream));
    if (m->d_b_fc)
        RUN(xma_rocm_expert_column_sums(m->dz, U, nullptr, 1, nullptr, offs, m->d_b_fc, U, (int32_t)U, (int32_t)m->E, dtype, stream));
    return gemm(m, m->few_dx1, m->dz, m->w_fc, U * H, H, 1, m->scattered, nullptr, 0, nullptr, nullptr, nullptr, H, U, 1, 1, 0,
                XMA_ROCM_EPI_STORE, stream);
}

extern "C" int xma_rocm_moe_backward(const xma_rocm_moe *m, void *stream) {
    RUN(check(m, "moe_backward"));
    RUN(check_experts(m, "moe_backward"));
    RUN(backward_experts(m, nullptr, nullptr, stream));
    return xma_rocm_combine_add(m->scattered, m->H, nullptr, m->d_x_addend, m->H, m->d_x, m->H, m->T, (int32_t)m->k, (int32_t)m->H, (int)m->dtype, stream);
}

// The order of the launches is that of the ops: whether the router weights' gradient comes from dX2 does not depend on what else hangs on
// the logits, and d_logits waits for it.
extern "C" int xma_rocm_moe_backward_logits(const xma_rocm_moe *m, void *stream) {
    RUN(check(m, "moe_backward_logits"));
    XMA_REQUIRE(m->logits && m->dy && m->d_router_weights && m->d_logits && (!m->recompute || m->h), XMA_ROCM_EINVAL,
                "moe_backward_logits: null buffer");
    const int dtype = (int)m->dtype;
    float *const dots = dots_place(m);
    RUN(check_recompute(m, "moe_backward_logits, as moe_backward_router", dots != nullptr));
    RUN(check_experts(m, "moe_backward_logits, as moe_backward"));
    RUN(recompute(m, dots != nullptr, stream));
    if (!dots)
        RUN(xma_rocm_combine_bwd(m->expert_out, m->H, m->dy, m->H, m->d_router_weights, m->T, (int32_t)m->k, (int32_t)m->H, dtype, stream));
    RUN(backward_experts(m, dots, nullptr, stream));
    return xma_rocm_router_topk_bwd(m->logits, m->E, m->T, (int32_t)m->E, (int32_t)m->k, dtype, m->expert_ids, 0, m->d_router_weights, m->d_logits,
                                    m->E, stream);
}

extern "C" int xma_rocm_moe_backward_gated(const xma_rocm_moe *m, void *d_gate_weight, void *stream) {
    RUN(check(m, "moe_backward_gated"));
    XMA_REQUIRE(m->gate_weight && m->logits && m->dy && m->d_router_weights && m->d_x && m->scattered && (!m->recompute || m->h), XMA_ROCM_EINVAL,
                "moe_backward_gated: null buffer");
    const int dtype = (int)m->dtype;
    XMA_REQUIRE(xma_rocm_gate_bwd_supported((int32_t)m->H, (int32_t)m->E, (int32_t)m->k, dtype), XMA_ROCM_EUNSUPPORTED,
                "moe_backward_gated: H=%lld E=%lld k=%lld dtype=%d", (long long)m->H, (long long)m->E, (long long)m->k, dtype);
    float *const dots = dots_place(m);
    RUN(check_recompute(m, "moe_backward_gated, as moe_backward_router", dots != nullptr));
    RUN(check_experts(m, "moe_backward_gated, as moe_backward"));
    RUN(xma_gate_bwd_check("moe_backward_gated", m->x, m->H, m->gate_weight, m->d_router_weights, (const int32_t *)m->expert_ids, m->scattered, m->d_x,
                           d_gate_weight, m->T, (int32_t)m->H, (int32_t)m->E, (int32_t)m->k, dtype, m->workspace, (size_t)m->workspace_bytes));
    RUN(recompute(m, dots != nullptr, stream));
    if (!dots)
        RUN(xma_combine_router_bwd(m->expert_out, m->dy, m->logits, (const int32_t *)m->expert_ids, m->T, (int32_t)m->H, (int32_t)m->E, (int32_t)m->k,
                                   dtype, m->d_router_weights, (hipStream_t)stream));
    RUN(backward_experts(m, dots, m->logits, stream));
    return xma_gate_bwd(m->x, m->H, m->gate_weight, m->d_router_weights, (const int32_t *)m->expert_ids, m->scattered, m->d_x, d_gate_weight, m->T,
                        (int32_t)m->H, (int32_t)m->E, (int32_t)m->k, dtype, m->workspace, (size_t)m->workspace_bytes, (hipStream_t)stream);
}
