"""KernelBackend.rocm implementation of the MoE expert computation.

Mirrors the op-level interface of the reference's Triton implementation
(xma/layers/moe/triton_implementation/__init__.py): ``scatter2scatter``,
``group``, ``group_bwd_W`` and the two autograd Functions behind
``up_projection_experts`` / ``down_projection_experts``; adds ``route`` (one op
for sort + histogram + offsets), ``router_topk`` (top-k + softmax behind the gate) and ``fused_swiglu_experts`` (the whole expert
computation with SwiGLU folded into the GEMM epilogues).

Differences from the reference's data flow, all of which remove HBM passes:
  * dW reads its gathered operand through the index instead of a materialised
    ``grouped_x`` / ``grouped_grad_out`` copy, and writes every element of dW
    (no zeros_like fill);
  * the router-weight scaling of dy is applied in the dX2 epilogue; dW2 reads one scaled grouped copy of dy, or, from
    four experts per token on in the fused SwiGLU path, dy through the index and activations that the dX2 epilogue
    wrote already scaled (then h is not kept for the backward either);
  * backward reuses the un-weighted expert outputs saved by forward instead of
    recomputing them with another GEMM (triton_implementation/__init__.py:117-128);
  * combine and its backward are dedicated coalesced kernels, not bmm;
  * with packed SwiGLU or GELU the layer is one autograd node (``layer``), and each direction one call of the library.
"""

from __future__ import annotations

import struct
from functools import lru_cache

import torch

from ...rocm import ops
from ...rocm.loader import check, get_library


# ----------------------------------------------------------------------------------------- routing
@torch.no_grad()
def route(selected_experts: torch.Tensor, num_experts: int):
    """(counts uint32 (E,), inclusive offsets int64 (E,), exclusive offsets int64 (E,),
    sorted_expert_idxs, sorted_scattered_idxs int64) of the flattened (T, k) selection; stable order."""
    ids = selected_experts.flatten().contiguous()
    n, dev = ids.numel(), ids.device
    counts = torch.empty(num_experts, dtype=torch.uint32, device=dev)
    incl = torch.empty(num_experts, dtype=torch.int64, device=dev)
    excl = torch.empty(num_experts, dtype=torch.int64, device=dev)
    sorted_expert_idxs = torch.empty_like(ids)
    sorted_scattered_idxs = torch.empty(n, dtype=torch.int64, device=dev)
    ops.route_rocm(ids, counts, incl, excl, sorted_expert_idxs, sorted_scattered_idxs, None)
    return counts, incl, excl, sorted_expert_idxs, sorted_scattered_idxs


def route_offsets(selected_experts: torch.Tensor, num_experts: int):
    """(inclusive offsets int64 (E,), sorted_scattered_idxs int64): the two of `route` that the fused experts read"""
    ids = selected_experts.flatten().contiguous()
    n, dev = ids.numel(), ids.device
    counts = torch.empty(num_experts, dtype=torch.uint32, device=dev)
    incl = torch.empty(num_experts, dtype=torch.int64, device=dev)
    sorted_scattered_idxs = torch.empty(n, dtype=torch.int64, device=dev)
    ops.route_rocm(ids, counts, incl, None, None, sorted_scattered_idxs, None)
    return incl, sorted_scattered_idxs


class _RouterTopK(torch.autograd.Function):
    """top-k + fp32 softmax over the selected logits + cast, and the gradient of the logits
    (xma/layers/moe/__init__.py:186-193, 256-262)"""

    @staticmethod
    def forward(ctx, router_logits: torch.Tensor, top_k: int, ids_dtype: torch.dtype):
        T = router_logits.size(0)
        weights = torch.empty(T, top_k, dtype=router_logits.dtype, device=router_logits.device)
        ids = torch.empty(T, top_k, dtype=ids_dtype, device=router_logits.device)
        ops.router_topk_rocm(router_logits, weights, ids)
        ctx.save_for_backward(router_logits, ids)
        ctx.mark_non_differentiable(ids)
        ctx.set_materialize_grads(False)  # no zero fill for the gradient of the ids, which nothing reads
        return weights, ids

    @staticmethod
    def backward(ctx, d_weights: torch.Tensor | None, _d_ids):
        if d_weights is None:  # nothing downstream depends on the router weights
            return None, None, None
        router_logits, ids = ctx.saved_tensors
        d_logits = torch.empty_like(router_logits, memory_format=torch.contiguous_format)
        ops.router_topk_bwd_rocm(router_logits, ids, d_weights.contiguous(), d_logits)
        return d_logits, None, None


class _RouterGateTopK(torch.autograd.Function):
    """gate projection + top-k + fp32 softmax + cast + int32 expert ids in one kernel (fp32: the stock product, then the router's
    kernel, int64 ids); backward: the router's d_logits kernel, then the two skinny products of the linear layer (d_x = d_logits @ Wg,
    d_Wg = d_logits^T @ x) from the k values of a row of d_logits that are not zero, or, where a loss hangs on the logits themselves, on the
    stock GEMM.  Counterpart of gate(x) and xma/layers/moe/__init__.py:186-193, 256-262."""

    @staticmethod
    def forward(ctx, x: torch.Tensor, gate_weight: torch.Tensor, top_k: int):
        T, E = x.size(0), gate_weight.size(0)
        weights = torch.empty(T, top_k, dtype=x.dtype, device=x.device)
        if x.dtype == torch.float32:
            logits = torch.nn.functional.linear(x, gate_weight)
            ids = torch.empty(T, top_k, dtype=torch.int64, device=x.device)
            ops.router_topk_rocm(logits, weights, ids)
        else:
            logits = torch.empty(T, E, dtype=x.dtype, device=x.device)
            ids = torch.empty(T, top_k, dtype=torch.int32, device=x.device)
            ops.router_gate_topk_rocm(x, gate_weight, logits, weights, ids)
        ctx.save_for_backward(x, gate_weight, logits, ids)
        ctx.mark_non_differentiable(ids)
        ctx.set_materialize_grads(False)  # an output nothing depends on arrives as None in backward, not as zeros
        return logits, weights, ids

    @staticmethod
    def backward(ctx, d_logits_out, d_weights, _d_ids):
        x, gate_weight, logits, ids = ctx.saved_tensors
        if d_weights is None and d_logits_out is None:
            return None, None, None
        if d_weights is None:
            d_logits = d_logits_out
        else:
            d_logits = torch.empty_like(logits)
            ops.router_topk_bwd_rocm(logits, ids, d_weights.contiguous(), d_logits)
            if d_logits_out is None and _gate_bwd(x, gate_weight.size(0), ids.size(1)):
                need_x, need_gate = ctx.needs_input_grad[:2]
                d_x = torch.empty(x.shape, dtype=x.dtype, device=x.device) if need_x else None
                d_w = torch.empty_like(gate_weight, memory_format=torch.contiguous_format) if need_gate else None
                if need_x or need_gate:
                    ops.gate_bwd_rocm(x, gate_weight, d_logits.gather(1, ids.long()), ids.int(), d_x, d_w)
                return d_x, d_w, None
            if d_logits_out is not None:  # the caller also used the returned router logits (an auxiliary loss)
                d_logits = d_logits + d_logits_out
        d_x = d_logits @ gate_weight if ctx.needs_input_grad[0] else None
        d_w = _gate_weight_grad(d_logits, x) if ctx.needs_input_grad[1] else None
        return d_x, d_w, None


def _gate_bwd(x: torch.Tensor, num_experts: int, top_k: int) -> bool:
    """whether the gate's gradients come from the library's kernels, which take a row of d_logits as its k values: everywhere but in a
    backward that is itself recorded (create_graph), where the products have to be torch's"""
    return x.size(0) > 0 and not torch.is_grad_enabled() and ops.gate_bwd_supported(x.size(1), num_experts, top_k, x.dtype)


def _gate_weight_grad(d_logits: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    """d_Wg = d_logits^T @ x, (E, T) x (T, H): an output of E x H elements with a reduction over all tokens, for which the
    stock GEMM launches few workgroups.  From 32 experts and 8192 tokens on the tokens are cut into 32 slices whose
    products run as one batched GEMM and are added in fp32 (measured 158 -> 51 us at T = 32768, E = 128, H = 2048;
    104 -> 38 us at T = 16384, E = 64; with 8 experts the single GEMM is faster)."""
    T, E = d_logits.shape
    slices = 32
    if E >= 32 and T >= 8192 and T % slices == 0 and x.is_contiguous() and d_logits.is_contiguous():
        partial = torch.bmm(d_logits.view(slices, T // slices, E).transpose(1, 2), x.view(slices, T // slices, x.size(1)))
        return partial.sum(0, dtype=torch.float32).to(x.dtype)
    return d_logits.t() @ x


def router_gate_topk(x: torch.Tensor, gate_weight: torch.Tensor, top_k: int):
    """(router logits (T, E), router weights (T, k), selected experts int32 (T, k)) from the activations and the gate's
    weight (E, H); differentiable in both."""
    return _RouterGateTopK.apply(x, gate_weight, top_k)


def router_gate_topk_supported(x: torch.Tensor, gate_weight: torch.Tensor, top_k: int) -> bool:
    """Whether the fused kernel takes these tensors; anything else (mixed dtypes, tensors on different devices, a row
    pitch that is no multiple of 16 bytes, a shape outside the kernel's range) goes through gate(x) + router_topk.  Only
    properties a traced caller can evaluate are looked at; a tensor that starts off a 16-byte boundary is copied inside
    the op.  Note that the fused path returns int32 expert ids, the fallback int64 like torch.topk: `route` reads either."""
    return x.is_cuda and x.dim() == 2 and x.stride(1) == 1 and x.stride(0) % 8 == 0 and gate_weight.is_contiguous() and \
        gate_weight.dtype == x.dtype and gate_weight.device == x.device and gate_weight.dim() == 2 and \
        ops.router_gate_topk_supported(x.size(1), gate_weight.size(0), top_k, x.dtype)


def gate_without_autograd(gate: torch.nn.Module, x: torch.Tensor, top_k: int) -> bool:
    """Whether an fp32 layer takes gate(x) as `router_gate_topk` does: the stock product, but the gate's gradients by the library.  A plain
    linear layer that nothing hooks into, outside autocast, of a shape that the gradients' kernels cover."""
    weight = gate.weight if type(gate) is torch.nn.Linear and gate.bias is None else None
    return (
        type(weight) is torch.nn.Parameter and weight.dtype == x.dtype == torch.float32 and x.is_cuda and weight.device == x.device
        and x.dim() == 2 and x.stride(1) == 1 and weight.is_contiguous() and weight.shape[1] == x.shape[1]
        and ops.gate_bwd_supported(x.size(1), weight.size(0), top_k, x.dtype) and not torch.is_autocast_enabled("cuda") and not _hooked(gate)
    )


def _hooked(module: torch.nn.Module) -> bool:
    return bool(module._forward_hooks or module._forward_pre_hooks or module._backward_hooks or module._backward_pre_hooks
                or "forward" in module.__dict__ or torch.nn.modules.module._has_any_global_hook())


def router_topk(router_logits: torch.Tensor, top_k: int, ids_dtype: torch.dtype = torch.int64):
    """(router weights (T, k) in the logits' dtype, selected experts (T, k), int64 as torch.topk gives them or int32 for
    the routing kernel); differentiable in the logits."""
    return _RouterTopK.apply(router_logits, top_k, ids_dtype)


# ----------------------------------------------------------------------------------------- op mirrors
def scatter2scatter(
    X: torch.Tensor,
    W: torch.Tensor,
    sorted_expert_idxs: torch.Tensor,
    sorted_scattered_idxs: torch.Tensor,
    out: torch.Tensor,
    FAN_OUT: int,
    x_grouped: bool = False,
    y_grouped: bool = False,
    expert_offsets: torch.Tensor | None = None,
    row_scale: torch.Tensor | None = None,
) -> None:
    """Signature of the reference op (scatter_kernel.py:137-147) plus the inclusive ``expert_offsets`` the
    expert-major tile schedule is derived from (computed from ``sorted_expert_idxs`` when not given)."""
    assert sorted_scattered_idxs.size(0) == sorted_expert_idxs.size(0)
    assert sorted_scattered_idxs.size(0) == X.size(0) * (1 if x_grouped else FAN_OUT)
    assert out.size(0) == sorted_expert_idxs.size(0) and out.size(1) == W.size(-1)
    if expert_offsets is None:
        expert_offsets = torch.bincount(sorted_expert_idxs, minlength=W.size(0)).cumsum(-1)
    ops.scatter2scatter_rocm(X, W, sorted_scattered_idxs, expert_offsets, out, row_scale, FAN_OUT, x_grouped, y_grouped)


def group(
    A: torch.Tensor,
    sorted_expert_idxs: torch.Tensor,
    out: torch.Tensor,
    coeff: torch.Tensor | None = None,
    fan_out: int = 1,
) -> None:
    """Signature of the reference op (group_kernel.py:69-76)."""
    ops.group_rocm(A, sorted_expert_idxs, out, coeff, fan_out)


def group_bwd_W(DY: torch.Tensor, X: torch.Tensor, expert_offsets: torch.Tensor, DW: torch.Tensor, E: int) -> None:
    """Signature of the reference op (group_backward_kernel.py:102-103): both operands already grouped."""
    assert DW.size(0) == E
    idx = torch.empty(0, dtype=torch.int64, device=DY.device)
    ops.group_bwd_W_rocm(DY, X, idx, expert_offsets, DW, None, 0, 0)


def _empty_dw_like(expert_weights: torch.Tensor) -> torch.Tensor:
    """Uninitialised gradient with the shape and strides of ``expert_weights`` ((E, in, out) view of
    (E, out, in) storage); the dW kernel writes every element, so no zero fill is needed."""
    return torch.empty_like(expert_weights)


def _scaled_grouped_dy(grad_out: torch.Tensor, sorted_scattered_idxs: torch.Tensor, flat_w: torch.Tensor, top_k: int):
    """grouped_dy[n] = dy[idx[n] // k] * w[idx[n]] (the reference's grouped_grad_out, triton_implementation/__init__.py:134-140).
    The scale sits on the reduction index of dW2, so it has to be on an operand; one HBM-bound pass over (T*k, H) is
    cheaper than rescaling fragments inside the MFMA loop.  dX2 does not read this copy: it gathers dy through the index
    and scales in its epilogue."""
    out = torch.empty(sorted_scattered_idxs.numel(), grad_out.size(1), dtype=grad_out.dtype, device=grad_out.device)
    ops.group_rocm(grad_out, sorted_scattered_idxs, out, flat_w, top_k)
    return out


def _scale_activations_for_dw2(top_k: int, grad_out: torch.Tensor) -> bool:
    """Whether the fused SwiGLU backward scales h (in the dX2 epilogue) rather than dy (with `group`) for dW2.  The scaled
    grouped copy of dy is top_k times the size of dy and goes through HBM twice; from four experts per token on that
    costs more than the extra output of the epilogue (measured on the whole forward + backward step, two boxes: -2.4 / -3.1 % at
    top-8 with H = 2048, I = 768; -1.0 / -1.4 % at top-6 with I = 1408; +0.7 / +1.0 % at top-2 with H = 4096, I = 14336).  h then is not kept for
    the backward.  16-bit only: the fp32 kernels have no such epilogue."""
    return _scale_by_top_k(top_k) and grad_out.dtype in (torch.bfloat16, torch.float16)


def _scale_by_top_k(top_k: int) -> bool:
    return top_k >= 4


# ----------------------------------------------------------------------------------------- autograd
def _bias_grad(A, sorted_scattered_idxs, expert_offsets, bias, row_scale=None, fan_out=1):
    """d_bias (E, out) = per-expert column sums of the grouped (or gathered and scaled) gradient rows"""
    d_bias = torch.empty_like(bias, memory_format=torch.contiguous_format)
    ops.expert_column_sums_rocm(A, sorted_scattered_idxs, expert_offsets, d_bias, row_scale, fan_out)
    return d_bias


class _UpProjectionExperts(torch.autograd.Function):
    """x (T, H) -> grouped (T*k, out); counterpart of triton_implementation/__init__.py:12-72, plus the experts' bias
    that the reference has on its torch path only (moe/__init__.py:96-100)."""

    @staticmethod
    def forward(ctx, x, expert_weights, k, sorted_expert_idxs, sorted_scattered_idxs, expert_offsets, bias=None):
        output = torch.empty(sorted_expert_idxs.size(0), expert_weights.size(-1), device=x.device, dtype=x.dtype)
        ops.scatter2scatter_rocm(x, expert_weights, sorted_scattered_idxs, expert_offsets, output, None, k, False, True, bias)
        ctx.save_for_backward(x, expert_weights, sorted_scattered_idxs, expert_offsets, bias)
        ctx.k = k
        return output

    @staticmethod
    def backward(ctx, grad_out):
        x, expert_weights, sorted_scattered_idxs, expert_offsets, bias = ctx.saved_tensors
        k = ctx.k
        grad_out = grad_out.contiguous()

        d_weights = _empty_dw_like(expert_weights)
        ops.group_bwd_W_rocm(grad_out, x, sorted_scattered_idxs, expert_offsets, d_weights, None, 0, k)
        d_bias = None if bias is None else _bias_grad(grad_out, None, expert_offsets, bias)

        scattered = torch.empty(sorted_scattered_idxs.size(0), x.size(1), dtype=x.dtype, device=x.device)
        ops.scatter2scatter_rocm(
            grad_out, expert_weights.permute(0, 2, 1), sorted_scattered_idxs, expert_offsets, scattered, None, 1, True, False
        )
        d_input = torch.empty_like(x)
        ops.combine_rocm(scattered, None, d_input, k)
        return d_input, d_weights, None, None, None, None, d_bias


class _DownProjectionExperts(torch.autograd.Function):
    """grouped h (T*k, I) -> y (T, H) = sum_j w[t, j] * expert_out[t*k + j]; counterpart of
    triton_implementation/__init__.py:75-162 (there called with k = 1 and router_weights (T, top_k))."""

    @staticmethod
    def forward(ctx, x, expert_weights, k, sorted_expert_idxs, sorted_scattered_idxs, expert_offsets, router_weights, bias=None):
        assert k == 1
        T, top_k = router_weights.shape
        expert_out = torch.empty(sorted_expert_idxs.size(0), expert_weights.size(-1), device=x.device, dtype=x.dtype)
        ops.scatter2scatter_rocm(x, expert_weights, sorted_scattered_idxs, expert_offsets, expert_out, None, 1, True, False, bias)
        router_weights = router_weights.contiguous()
        y = torch.empty(T, expert_out.size(1), device=x.device, dtype=x.dtype)
        ops.combine_rocm(expert_out, router_weights, y, top_k)
        ctx.save_for_backward(x, expert_weights, sorted_scattered_idxs, expert_offsets, router_weights, expert_out, bias)
        return y

    @staticmethod
    def backward(ctx, grad_out):
        x, expert_weights, sorted_scattered_idxs, expert_offsets, router_weights, expert_out, bias = ctx.saved_tensors
        top_k = router_weights.size(1)
        grad_out = grad_out.contiguous()

        d_router_weights = torch.empty_like(router_weights)
        ops.combine_bwd_rocm(expert_out, grad_out, d_router_weights)

        flat_w = router_weights.view(-1)
        d_weights = _empty_dw_like(expert_weights)
        grouped_dy = _scaled_grouped_dy(grad_out, sorted_scattered_idxs, flat_w, top_k)
        ops.group_bwd_W_rocm(grouped_dy, x, sorted_scattered_idxs, expert_offsets, d_weights, None, 0, 0)
        d_bias = None if bias is None else _bias_grad(grouped_dy, None, expert_offsets, bias)

        d_input = torch.empty_like(x)
        ops.scatter2scatter_rocm(
            grad_out, expert_weights.permute(0, 2, 1), sorted_scattered_idxs, expert_offsets, d_input, flat_w, top_k, False, True
        )
        return d_input, d_weights, None, None, None, None, d_router_weights, d_bias


class _FusedSwiGLUExperts(torch.autograd.Function):
    """Whole expert computation with packed SwiGLU in the GEMM epilogues:
    forward  up-projection (+ bias, SwiGLU) -> down-projection (+ bias, scattered) -> combine
    backward combine' -> dX2 (+ SwiGLU') -> dW2, dW1 (and the bias gradients) -> dX1 (scattered) -> k-way sum.
    save_activations = False keeps x and the pre-activations z only: the backward then recomputes what it reads of h = swiglu_packed(z)
    and the expert outputs (one more down-projection GEMM, except where dX2 leaves the router weights' gradient), as the reference's
    backward recomputes its expert outputs (triton_implementation/__init__.py:117-128)."""

    @staticmethod
    def forward(ctx, x, w_fc, w_proj, router_weights, sorted_scattered_idxs, expert_offsets, b_fc=None, b_proj=None,
                save_activations=True):
        # w_fc: (E, H, 2I) view, w_proj: (E, I, H) view (both permuted views of the parameters)
        T, top_k = router_weights.shape
        M = sorted_scattered_idxs.numel()
        z = torch.empty(M, w_fc.size(-1), device=x.device, dtype=x.dtype)
        h = torch.empty(M, w_fc.size(-1) // 2, device=x.device, dtype=x.dtype)
        ops.up_projection_swiglu_rocm(x, w_fc, sorted_scattered_idxs, expert_offsets, z, h, top_k, b_fc)
        expert_out = torch.empty(M, w_proj.size(-1), device=x.device, dtype=x.dtype)
        ops.scatter2scatter_rocm(h, w_proj, sorted_scattered_idxs, expert_offsets, expert_out, None, 1, True, False, b_proj)
        router_weights = router_weights.contiguous()
        y = torch.empty(T, expert_out.size(1), device=x.device, dtype=x.dtype)
        ops.combine_rocm(expert_out, router_weights, y, top_k)
        # h is an operand of dW2 only where dW2 takes the scaled grouped copy of dy; otherwise the backward rebuilds it,
        # scaled, from z in the dX2 epilogue and h lives until the end of this forward only
        kept_h = h if save_activations and not _scale_activations_for_dw2(top_k, x) else h.new_empty(0)
        kept_out = expert_out if save_activations else expert_out.new_empty(0)
        ctx.save_for_backward(x, w_fc, w_proj, router_weights, sorted_scattered_idxs, expert_offsets, z, kept_h, kept_out,
                              b_fc, b_proj)
        return y

    @staticmethod
    def backward(ctx, grad_out):
        (x, w_fc, w_proj, router_weights, sorted_scattered_idxs, expert_offsets, z, h, expert_out, b_fc,
         b_proj) = ctx.saved_tensors
        top_k = router_weights.size(1)
        grad_out = grad_out.contiguous()
        flat_w = router_weights.view(-1)
        scaled_act_path = _scale_activations_for_dw2(top_k, grad_out)

        recomputed = expert_out.numel() == 0 and z.numel() != 0  # from z: what reads them, and the op below may not
        if recomputed and h.numel() == 0 and (b_proj is not None or not scaled_act_path):
            h = torch.empty(z.size(0), z.size(1) // 2, dtype=z.dtype, device=z.device)
            ops.swiglu_packed_forward_rocm(z, h)
        if recomputed and b_proj is not None:
            expert_out = torch.empty(z.size(0), w_proj.size(-1), device=z.device, dtype=z.dtype)
            ops.scatter2scatter_rocm(h, w_proj, sorted_scattered_idxs, expert_offsets, expert_out, None, 1, True, False, b_proj)
        d_router_weights = torch.empty_like(router_weights)
        if b_proj is not None:  # <dy, bias> is part of the gradient: it comes from the expert outputs
            ops.combine_bwd_rocm(expert_out, grad_out, d_router_weights)

        dz = torch.empty_like(z)
        d_w_proj = _empty_dw_like(w_proj)
        d_b_proj = None
        if scaled_act_path and z.numel() != 0:
            # dW2 = sum_n (w_n dy_n)^T h_n = sum_n dy_n^T (w_n h_n): the dX2 epilogue, which has z and w_n at hand, writes
            # w_n h_n (T*k, I), and dW2 takes dy unscaled through the index - instead of a scaled, grouped copy of dy
            # (T*k, H) written by `group` and read back by the GEMM
            scaled_h = torch.empty(z.size(0), z.size(1) // 2, dtype=z.dtype, device=z.device)
            if b_proj is None:
                ops.down_projection_dx_swiglu_router_rocm(
                    grad_out, w_proj.permute(0, 2, 1), sorted_scattered_idxs, expert_offsets, z, dz, scaled_h, flat_w, expert_out,
                    d_router_weights, top_k
                )
            else:
                ops.down_projection_dx_swiglu_scaled_act_rocm(
                    grad_out, w_proj.permute(0, 2, 1), sorted_scattered_idxs, expert_offsets, z, dz, scaled_h, flat_w, top_k
                )
            ops.group_bwd_W_rocm(grad_out, scaled_h, sorted_scattered_idxs, expert_offsets, d_w_proj, None, top_k, 0)
            if b_proj is not None:
                d_b_proj = _bias_grad(grad_out, sorted_scattered_idxs, expert_offsets, b_proj, flat_w, top_k)
        else:
            if b_proj is None:
                ops.down_projection_dx_swiglu_router_rocm(
                    grad_out, w_proj.permute(0, 2, 1), sorted_scattered_idxs, expert_offsets, z, dz, None, flat_w, expert_out,
                    d_router_weights, top_k, h
                )
            else:
                ops.down_projection_dx_swiglu_rocm(
                    grad_out, w_proj.permute(0, 2, 1), sorted_scattered_idxs, expert_offsets, z, dz, flat_w, top_k
                )
            if b_proj is None and ops._dw_loader_scales(z.size(0), w_proj.size(0), z.dtype, w_proj.size(2), w_proj.size(1)):
                # a handful of rows per expert: the weight gradient's loader gathers and scales the rows of dy itself (and
                # rounds them like the copy would), one launch less
                ops.group_bwd_W_rocm(grad_out, h, sorted_scattered_idxs, expert_offsets, d_w_proj, flat_w, top_k, 0)
            else:
                grouped_dy = _scaled_grouped_dy(grad_out, sorted_scattered_idxs, flat_w, top_k)
                ops.group_bwd_W_rocm(grouped_dy, h, sorted_scattered_idxs, expert_offsets, d_w_proj, None, 0, 0)
                if b_proj is not None:
                    d_b_proj = _bias_grad(grouped_dy, None, expert_offsets, b_proj)
        d_w_fc = _empty_dw_like(w_fc)
        ops.group_bwd_W_rocm(dz, x, sorted_scattered_idxs, expert_offsets, d_w_fc, None, 0, top_k)
        d_b_fc = None if b_fc is None else _bias_grad(dz, None, expert_offsets, b_fc)

        scattered = torch.empty(z.size(0), x.size(1), dtype=x.dtype, device=x.device)
        ops.scatter2scatter_rocm(dz, w_fc.permute(0, 2, 1), sorted_scattered_idxs, expert_offsets, scattered, None, 1, True, False)
        d_x = torch.empty_like(x)
        ops.combine_rocm(scattered, None, d_x, top_k)
        return d_x, d_w_fc, d_w_proj, d_router_weights, None, None, d_b_fc, d_b_proj, None


def up_projection_experts(x, expert_weights, k, sorted_expert_idxs, sorted_scattered_idxs, expert_offsets, bias=None):
    return _UpProjectionExperts.apply(x, expert_weights, k, sorted_expert_idxs, sorted_scattered_idxs, expert_offsets, bias)


def down_projection_experts(x, expert_weights, k, sorted_expert_idxs, sorted_scattered_idxs, expert_offsets, router_weights,
                            bias=None):
    return _DownProjectionExperts.apply(
        x, expert_weights, k, sorted_expert_idxs, sorted_scattered_idxs, expert_offsets, router_weights, bias
    )


def fused_swiglu_experts(x, w_fc, w_proj, router_weights, sorted_scattered_idxs, expert_offsets, b_fc=None, b_proj=None,
                         save_activations=True):
    """save_activations = False: the backward recomputes h and the expert outputs instead of keeping them, which frees
    T k (H + I) elements per layer between forward and backward (Mixtral-shaped layer: 604 MB of 1.5 GB) for h again and, unless
    the 256 x 256 tiles take dX2 of a layer without a down-projection bias, one more down-projection GEMM."""
    return _FusedSwiGLUExperts.apply(x, w_fc, w_proj, router_weights, sorted_scattered_idxs, expert_offsets, b_fc, b_proj,
                                     save_activations)


# ----------------------------------------------------------------------------------------- the layer as one call
# A pass of a handful of tokens is as long as its host work, so the layer with packed SwiGLU or GELU runs as one autograd node, whose
# forward and backward are one library call each (and the last sum another behind gate products of torch's), on scratch that is laid out once per shape:
# the same launches as the ops above, bit for bit.  Everything else (other activations, tracing, transforms, tensors that the
# entry point does not describe) goes through the ops.
_BLOCK_POINTERS = struct.Struct("29Q")
_BLOCK_SIZES = struct.Struct("17q")


class _Plan:
    """sizes, choices and scratch layout of a layer call; a function of the shape, the options and the dispatch limits only"""

    __slots__ = ("sizes_forward", "sizes_backward", "keep", "temp", "back", "keep_bytes", "temp_bytes", "back_bytes", "saved_shapes", "top_k")


def _layout(sizes: dict[str, int]) -> tuple[dict[str, int], int]:
    offsets, end = {}, 0
    for name, size in sizes.items():
        offsets[name] = end
        end += (size + 255) // 256 * 256
    return offsets, max(end, 256)


@lru_cache(maxsize=4096)
def _plan(T: int, H: int, I: int, E: int, k: int, dtype: torch.dtype, act: str, b_proj: bool, save: bool, device_index: int, _limits) -> _Plan:
    M, s = T * k, dtype.itemsize
    glu = act == "swiglu_packed"
    U = 2 * I if glu else I  # width of the up-projection
    epi_fwd, epi_bwd = (ops.EPI_SWIGLU, ops.EPI_SWIGLU_BWD) if glu else ops.EPI_GELU[act]
    few16 = dtype != torch.float32

    def gemm(N, K, w_is_kn, ldw, x_span, epilogue):
        """(which entry point, bytes of its workspace)"""
        if few16 and ops._few_rows_fwd(M, N, K, E, w_is_kn, ldw, x_span, dtype, epilogue):
            return 1, ops._few_rows_workspace_bytes(M, N, K, E, w_is_kn, epilogue)
        return 0, ops.scatter2scatter_workspace_bytes(M, N, K, E, device_index)

    def dw(N_out, K_in, span, scaled):
        return int(ops._dw_few(M, N_out, K_in, E, dtype, span, scaled, False))

    up, down = gemm(U, H, 0, H, T * H, epi_fwd), gemm(H, I, 0, I, M * I, ops.EPI_STORE)
    dx2, dx1 = gemm(I, H, 1, I, T * H, epi_bwd), gemm(H, U, 1, H, M * U, ops.EPI_STORE)
    # the operand of dW2: see xma_rocm_moe in the library's header
    if few16 and glu and _scale_by_top_k(k):
        dw2_form, dw2_operand = 1, M * I * s
    elif not b_proj and ops._dw_loader_scales(M, E, dtype, H, I):
        dw2_form, dw2_operand = 0, 0
    else:
        dw2_form, dw2_operand = 2, M * H * s
    keep_h = save and dw2_form != 1
    sizes = dict(weights=M * s, ids=M * 4, offsets=E * 8, idx=M * 8, z=M * U * s)
    temp = dict(counts=E * 4, workspace=max(ops.route_workspace_elements(M, E) * 4, up[1], down[1]))
    (sizes if keep_h else temp)["h"] = M * I * s
    (sizes if save else temp)["out"] = M * H * s
    # the scattered rows of dX1 take the place of dW2's operand
    gate_sums = get_library().xma_rocm_gate_bwd_workspace_bytes(T, H, E) if ops.gate_bwd_supported(H, E, k, dtype) else 0
    # dX2 by the 256 x 256 kernels leaves the router weights' gradient behind its K slices
    dots = ops.router_gradient_workspace_bytes(M, I, dx2[1]) if glu and not b_proj and ops.dx2_leaves_router_gradient(dx2[0], M, I, k, dtype) else 0
    back = dict(d_weights=M * s, dz=M * U * s, scattered=max(M * H * s, dw2_operand), workspace=max(down[1], dx2[1], dx1[1], gate_sums, dots, 256))
    if not save:
        back |= dict(h=M * I * s, out=M * H * s)
    p = _Plan()
    p.keep, p.keep_bytes = _layout(sizes)
    p.temp, p.temp_bytes = _layout(temp)
    p.back, p.back_bytes = _layout(back)
    p.top_k = k
    p.saved_shapes = ((T, H), (E, H), (T, E), (E, U, H), (E, H, I), (E, U), (E, H), (p.keep_bytes,))
    few = (up[0], down[0], dx2[0], dw(H, I, max((M if dw2_form == 2 else T) * H, M * I), dw2_form == 0), dw(U, H, max(M * U, T * H), False), dx1[0], dw2_form, int(not save))
    head = (_BLOCK_SIZES.size + _BLOCK_POINTERS.size, T, H, I, E, k, ops._DTYPE_CODE[dtype], ("swiglu_packed", "tanh", "none").index(act), *few)
    p.sizes_forward = _BLOCK_SIZES.pack(*head, temp["workspace"])
    p.sizes_backward = _BLOCK_SIZES.pack(*head, back["workspace"])
    return p


def _layer_forward(x, gate_weight, logits, w_fc, w_proj, b_fc, b_proj, k, act, save, grad):
    """(y, logits, kept buffer, plan); gate_weight None: the logits are given"""
    T, H = x.shape
    E, I = w_proj.size(0), w_proj.size(2)
    device = x.device
    p = _plan(T, H, I, E, k, x.dtype, act, b_proj is not None, save, device.index, ops.dispatch_limits())
    y = torch.empty_like(x)
    if gate_weight is not None and x.dtype == torch.float32:
        logits, gate_weight = torch.nn.functional.linear(x, gate_weight), None
    elif gate_weight is not None:
        logits = torch.empty(T, E, dtype=x.dtype, device=device)
    if grad:
        kept = torch.empty(p.keep_bytes, dtype=torch.uint8, device=device)
        scratch = torch.empty(p.temp_bytes, dtype=torch.uint8, device=device)
        a, b = kept.data_ptr(), scratch.data_ptr()
    else:
        kept = torch.empty(p.keep_bytes + p.temp_bytes, dtype=torch.uint8, device=device)
        a = kept.data_ptr()
        b = a + p.keep_bytes
    keep, temp = p.keep, p.temp
    check(
        get_library().xma_rocm_moe_forward(p.sizes_forward + _BLOCK_POINTERS.pack(
            x.data_ptr(), 0 if gate_weight is None else gate_weight.data_ptr(), w_fc.data_ptr(), w_proj.data_ptr(),
            0 if b_fc is None else b_fc.data_ptr(), 0 if b_proj is None else b_proj.data_ptr(), logits.data_ptr(),
            a + keep["weights"], a + keep["ids"], b + temp["counts"], a + keep["offsets"], a + keep["idx"], a + keep["z"],
            a + keep["h"] if "h" in keep else b + temp["h"], a + keep["out"] if "out" in keep else b + temp["out"], y.data_ptr(),
            b + temp["workspace"], 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0,
        ), ops._stream(x)),
        "xma_rocm_moe_forward",
    )
    return y, logits, kept, p


def _unpacked(saved, shapes, like: torch.Tensor) -> list[torch.Tensor | None]:
    """The saved tensors of `_Layer` as the library takes them.  Saved-tensor hooks may hand back a copy of another layout, which is
    laid out again; one of another shape, dtype or device is refused, as the ops refuse it."""
    out = []
    for t, shape in zip(saved, shapes):
        if t is not None:
            assert t.shape == shape and t.device == like.device and (t.dtype == like.dtype or len(shape) == 1 and t.dtype == torch.uint8), \
                "a saved tensor came back with another shape, device or dtype"
            if not t.is_contiguous() or t.data_ptr() % 16:
                t = t.clone(memory_format=torch.contiguous_format)
        out.append(t)
    return out


def _check_backward(rc: int, entry: str) -> None:
    """raises what the entry refused; the message of a rule that it shares with another entry begins with both names"""
    if rc:
        part = get_library().xma_rocm_last_error().decode(errors="replace").partition(":")[0].partition(", as ")[2]
        check(rc, entry + (", as xma_rocm_" + part if part else ""))


class _Layer(torch.autograd.Function):
    """the whole layer: with gate_weight (logits None) -> (y, logits), with given logits -> y"""

    @staticmethod
    def forward(ctx, x, gate_weight, logits, w_fc, w_proj, b_fc, b_proj, k, act, save):
        y, logits, kept, ctx.plan = _layer_forward(x, gate_weight, logits, w_fc, w_proj, b_fc, b_proj, k, act, save, True)
        ctx.save_for_backward(x, gate_weight, logits, w_fc, w_proj, b_fc, b_proj, kept)
        ctx.set_materialize_grads(False)
        return y if gate_weight is None else (y, logits)

    @staticmethod
    def backward(ctx, dy, d_logits_out=None):
        need_x, need_gate, need_logits = ctx.needs_input_grad[:3]
        if dy is None:  # nothing but the logits was used
            if d_logits_out is None:
                return (None,) * 10
            x, gate_weight = ctx.saved_tensors[:2]
            d_x = d_logits_out @ gate_weight if need_x else None
            return d_x, _gate_weight_grad(d_logits_out, x) if need_gate else None, *(None,) * 8
        dy = dy.contiguous()
        p = ctx.plan
        x, gate_weight, logits, w_fc, w_proj, b_fc, b_proj, kept = _unpacked(ctx.saved_tensors, p.saved_shapes, dy)
        scratch = torch.empty(p.back_bytes, dtype=torch.uint8, device=x.device)
        gated = gate_weight is not None and d_logits_out is None and _gate_bwd(x, gate_weight.size(0), p.top_k)
        d_logits = None if gated else torch.empty_like(logits, memory_format=torch.contiguous_format)
        d_x, d_w_fc, d_w_proj = torch.empty_like(x), torch.empty_like(w_fc), torch.empty_like(w_proj)
        d_b_fc, d_b_proj = (None if b is None else torch.empty_like(b) for b in (b_fc, b_proj))
        a, b, keep, back = kept.data_ptr(), scratch.data_ptr(), p.keep, p.back
        pointers = (
            x.data_ptr(), gate_weight.data_ptr() if gated else 0, w_fc.data_ptr(), w_proj.data_ptr(), 0 if b_fc is None else b_fc.data_ptr(),
            0 if b_proj is None else b_proj.data_ptr(), logits.data_ptr(), a + keep["weights"], a + keep["ids"], 0, a + keep["offsets"],
            a + keep["idx"], a + keep["z"], b + back["h"] if "h" in back else a + keep["h"] if "h" in keep else 0,
            b + back["out"] if "out" in back else a + keep["out"], 0, b + back["workspace"], dy.data_ptr(), b + back["d_weights"],
            0 if gated else d_logits.data_ptr(), b + back["dz"], b + back["scattered"], b + back["scattered"], d_w_fc.data_ptr(), d_w_proj.data_ptr(),
            0 if d_b_fc is None else d_b_fc.data_ptr(), 0 if d_b_proj is None else d_b_proj.data_ptr(), d_x.data_ptr(),
        )
        lib, stream = get_library(), ops._stream(x)
        if gated:
            d_gate = torch.empty_like(gate_weight) if need_gate else None
            _check_backward(lib.xma_rocm_moe_backward_gated(p.sizes_backward + _BLOCK_POINTERS.pack(*pointers, 0),
                                                            None if d_gate is None else d_gate.data_ptr(), stream), "xma_rocm_moe_backward_gated")
            return d_x, d_gate, None, d_w_fc, d_w_proj, d_b_fc, d_b_proj, None, None, None
        _check_backward(lib.xma_rocm_moe_backward_logits(p.sizes_backward + _BLOCK_POINTERS.pack(*pointers, 0), stream), "xma_rocm_moe_backward_logits")
        d_gate = d_x_gate = None
        if gate_weight is not None:
            if d_logits_out is not None:  # the caller also used the returned router logits (an auxiliary loss)
                d_logits = d_logits + d_logits_out
            if need_x:
                d_x_gate = (d_logits @ gate_weight).to(x.dtype)  # in an autocast region the product has another dtype
            if need_gate:
                d_gate = _gate_weight_grad(d_logits, x)
        recorded = d_x_gate is not None and d_x_gate.requires_grad  # create_graph: the sum is torch's as well
        T, H = x.shape
        check(lib.xma_rocm_combine_add(b + back["scattered"], H, None, None if d_x_gate is None or recorded else d_x_gate.data_ptr(), H,
                                       d_x.data_ptr(), H, T, p.top_k, H, ops._DTYPE_CODE[x.dtype], stream), "xma_rocm_combine_add")
        if recorded:
            d_x = d_x + d_x_gate
        return d_x, d_gate, d_logits if need_logits else None, d_w_fc, d_w_proj, d_b_fc, d_b_proj, None, None, None


def _activation(moe) -> str | None:
    """the layer's activation where the library has it: packed SwiGLU, or GELU in either form as a module that nothing hooks into"""
    act = moe.act
    if moe.is_glu:
        return "swiglu_packed" if getattr(act, "_xma_fused_activation", None) == "swiglu_packed" else None
    if type(act) is not torch.nn.GELU or act.approximate not in ops.EPI_GELU or _hooked(act):
        return None
    return act.approximate


def _plain(t: torch.Tensor, like: torch.Tensor) -> bool:
    return t.dtype == like.dtype and t.device == like.device and t.is_contiguous() and t.data_ptr() % 16 == 0 and \
        type(t) in (torch.nn.Parameter, torch.Tensor)


def layer(moe, x: torch.Tensor):
    """(y, router logits) of a layer with packed SwiGLU or GELU whose tensors the library's layer entry point describes: contiguous, one
    dtype and device, aligned; None for anything else, and under function transforms and forward-mode differentiation"""
    w_fc, w_proj, b_fc, b_proj = moe.c_fc.weight, moe.c_proj.weight, moe.c_fc.bias, moe.c_proj.bias
    gate, k = moe.gate, moe.top_k
    T, H = x.shape
    act = _activation(moe)
    if act is None:
        return None
    if T == 0 or x.dtype not in ops._DTYPE_CODE or type(x) not in (torch.Tensor, torch.nn.Parameter) or x.data_ptr() % 16 or not x.is_contiguous():
        return None
    if not (_plain(w_fc, x) and _plain(w_proj, x)) or (b_fc is not None and not _plain(b_fc, x)) or (b_proj is not None and not _plain(b_proj, x)):
        return None
    E, U, _ = w_fc.shape
    I = U // 2 if act == "swiglu_packed" else U
    if H % 8 or I % 8 or (act == "swiglu_packed" and U % 2) or w_fc.size(2) != H or w_proj.shape != (E, H, I) or E > 16384 or T * k >= 1 << 31:
        return None
    # the entry point has one E, H and I for all its tensors: the ops answer a gate over fewer experts and refuse the rest
    if moe.num_experts != E or (b_fc is not None and b_fc.shape != (E, U)) or (b_proj is not None and b_proj.shape != (E, H)):
        return None
    if torch._C._are_functorch_transforms_active() or torch.autograd.forward_ad._current_level >= 0:
        return None
    gate_weight, logits = gate.weight, None
    if gate.bias is None and router_gate_topk_supported(x, gate_weight, k):
        if gate_weight.shape != (E, H) or not _plain(gate_weight, x):  # the op copies a weight that starts off a 16-byte boundary
            return None
        tensors = (x, gate_weight, w_fc, w_proj, b_fc, b_proj)
    elif gate_without_autograd(gate, x, k) and gate_weight.shape == (E, H) and _plain(gate_weight, x):
        tensors = (x, gate_weight, w_fc, w_proj, b_fc, b_proj)
    else:
        gate_weight, logits = None, gate(x)
        if logits.shape != (T, E) or not _plain(logits, x):  # a gate that casts, for one
            return moe._compute_experts(x, *router_topk(logits, k)), logits
        tensors = (x, logits, w_fc, w_proj, b_fc, b_proj)
    save = bool(moe.save_activations) or act != "swiglu_packed"
    if torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in tensors):
        out = _Layer.apply(x, gate_weight, logits, w_fc, w_proj, b_fc, b_proj, k, act, save)
        return out if logits is None else (out, logits)
    return _layer_forward(x, gate_weight, logits, w_fc, w_proj, b_fc, b_proj, k, act, True, False)[:2]
