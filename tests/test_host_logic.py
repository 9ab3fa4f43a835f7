"""Host logic that needs no GPU: the C-ABI library loads and exports every symbol include/xma_rocm.h declares,
backend selection and error behaviour mirror the reference, module layout matches its state-dict."""

import ctypes
import os
import re

import pytest
import torch
import torch.nn as nn

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "xma_rocm.h")).read()
    return sorted(set(re.findall(r"\b(xma_rocm_[a-zA-Z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from xma.rocm import LIBRARY_PATH, get_library
    from xma.rocm.loader import SIGNATURES

    assert os.path.isfile(LIBRARY_PATH), "build the library first: python __graft_entry__.py"
    lib = ctypes.CDLL(LIBRARY_PATH)
    declared = _declared_symbols()
    assert len(declared) >= 13
    for name in declared:
        assert hasattr(lib, name), f"{name} declared in include/xma_rocm.h but not exported"
    assert sorted(SIGNATURES) == declared  # the ctypes table covers exactly the header
    lib = get_library()
    assert lib.xma_rocm_abi_version() == 1
    # host-only entry points (no GPU work)
    assert lib.xma_rocm_route_workspace_bytes(4 * 1024 * 1024, 64) == (4 * 1024 * 1024 // 4096) * 64 * 4
    assert lib.xma_rocm_continuous_count_workspace_bytes(4 * 1024 * 1024, 64) == 1024 * 64 * 4
    assert lib.xma_rocm_continuous_count_workspace_bytes(1000, 64) == 0
    assert lib.xma_rocm_route_workspace_bytes(0, 8) == 8 * 4
    assert lib.xma_rocm_route_workspace_bytes(-1, 8) == 0


def test_argument_errors_are_reported_before_any_launch():
    from xma.rocm import get_library

    lib = get_library()
    # bins < 1, E out of range, unsupported dtype, misaligned sizes: all rejected on the host
    assert lib.xma_rocm_continuous_count(None, 0, 10, None, 0, None, 0, None) == -1
    assert b"continuous_count" in lib.xma_rocm_last_error()
    assert lib.xma_rocm_route(None, 0, 10, 100000, None, None, None, None, None, None, 0, None) == -1
    # the entry point with static scratch refuses what does not fit its array, before touching the device
    assert lib.xma_rocm_route_static_max_units_times_experts() == 1 << 18
    big = ctypes.c_void_p(256)
    assert lib.xma_rocm_route_static(big, 0, 4096 * 129, 2048, big, big, None, None, big, None) == -3
    assert b"static scratch" in lib.xma_rocm_last_error()
    assert lib.xma_rocm_route_static(None, 0, 10, 100000, None, None, None, None, None, None) == -1
    assert lib.xma_rocm_combine(None, 8, None, None, 8, 4, 2, 12, 0, None) == -1  # H % 8 != 0
    assert lib.xma_rocm_combine(None, 8, None, None, 8, 4, 2, 16, 7, None) == -2  # dtype
    rc = lib.xma_rocm_scatter2scatter(None, 64, None, 64 * 64, 64, 0, None, None, None, 64, None, 0, None, 16, 60, 64, 2, 1, 1, 1,
                                      0, 0, None, 0, None)
    assert rc == -2 and b"multiples of 8" in lib.xma_rocm_last_error()
    # router: k > E, E and k beyond what a wave holds, row stride shorter than a row, dtype
    assert lib.xma_rocm_router_topk(None, 8, 4, 8, 9, 0, None, None, 1, None) == -1 and b"k <= E" in lib.xma_rocm_last_error()
    assert lib.xma_rocm_router_topk(None, 4096, 4, 4096, 2, 0, None, None, 1, None) == -2
    assert lib.xma_rocm_router_topk(None, 128, 4, 128, 65, 0, None, None, 1, None) == -2
    assert lib.xma_rocm_router_topk(None, 4, 4, 8, 2, 0, None, None, 1, None) == -1
    assert lib.xma_rocm_router_topk(None, 8, 4, 8, 2, 5, None, None, 1, None) == -2
    assert lib.xma_rocm_router_topk(None, 8, 4, 8, 2, 0, None, None, 1, None) == -1  # null pointers with T > 0
    assert lib.xma_rocm_router_topk_bwd(None, 8, 4, 8, 2, 0, None, 1, None, None, 4, None) == -1  # ldd < E
    assert lib.xma_rocm_router_topk(None, 8, 0, 8, 2, 0, None, None, 1, None) == 0
    # the few-token entry points: dtype (no fp32), M beyond the epilogue's grid, a missing workspace where sums go through
    # one (few column blocks and a long K: the launch is cut along K), none needed for W as (N, K) with a plain store (fails later, on the null operands), dW shapes
    p = ctypes.c_void_p(256)
    few = lib.xma_rocm_scatter2scatter_few_rows
    assert few(p, 64, p, 64 * 64, 64, 0, p, p, p, 64, None, 0, None, 0, None, None, 0, 4, 64, 64, 2, 1, 1, 1, 0, 2, None, 0, None) == -2
    assert few(p, 64, p, 64 * 64, 64, 0, p, p, p, 64, None, 0, None, 0, None, None, 0, 70000, 64, 64, 2, 1, 1, 1, 0, 0, None, 0, None) == -1
    assert few(p, 16384, p, 16384 * 64, 64, 1, p, p, p, 64, None, 0, None, 0, None, None, 0, 4, 64, 16384, 2, 1, 1, 1, 0, 0, None, 0, None) == -3
    assert b"workspace" in lib.xma_rocm_last_error()
    assert few(None, 64, None, 64 * 64, 64, 0, p, p, p, 64, None, 0, None, 0, None, None, 0, 4, 64, 64, 2, 1, 1, 1, 0, 0, None, 0, None) == -1
    assert b"null or misaligned" in lib.xma_rocm_last_error()
    # W as (N, K) is addressed with 32-bit byte offsets inside an expert
    assert few(p, 64, p, 64 << 26, 1 << 26, 0, p, p, p, 64, None, 0, None, 0, None, None, 0, 4, 64, 64, 2, 1, 1, 1, 0, 0, None, 0, None) == -2
    assert b"N * ldw" in lib.xma_rocm_last_error()
    ws = lib.xma_rocm_scatter2scatter_few_rows_workspace_bytes  # (M, N, K, E, w_is_kn, epilogue)
    assert ws(4, 64, 2048, 2, 0, 0) == 0 and ws(4, 64, 2048, 2, 0, 1) == 0  # the vector kernel finishes the job itself (2 rows per expert)
    assert ws(4, 64, 2048, 2, 0, 2) == 4 * 64 * 4  # SwiGLU backward: through the epilogue kernel
    assert ws(4, 64, 64, 2, 0, 2) == 0  # short rows of W: the small tile, one K range, epilogue in the kernel
    assert ws(4, 64, 16384, 2, 1, 0) == 32 * 4 * 64 * 4  # W as (K, N): the small tile at any number of rows, 32 ranges of K
    assert ws(64, 2048, 16384, 8, 1, 0) == 4 * 64 * 2048 * 4 and ws(64, 8192, 2048, 8, 1, 2) == 0  # small tile: 4 ranges of K; none
    assert ws(64, 16384, 2048, 8, 0, 1) == 0  # small MFMA tile, enough workgroups from N alone
    assert ws(64, 2048, 8192, 8, 0, 0) == 4 * 64 * 2048 * 4  # small MFMA tile cut into 4 ranges of K
    assert ws(0, 64, 64, 2, 1, 0) == 0
    # beyond 24 rows per expert what the 128 x 256 tiles ask for, not the small tile's sums, which grow with M
    assert ws(32000, 512, 2048, 8, 1, 0) == 0 and ws(2048, 8192, 1024, 4, 1, 2) == 0
    assert ws(8198, 1024, 4096, 4, 0, 1) == 0 and ws(8198, 4096, 1024, 4, 1, 0) == 0 and ws(8000, 8192, 1024, 4, 1, 2) == 0
    assert ws(8000, 1024, 16384, 4, 1, 0) == 2 * 8000 * 1024 * 4 and ws(258, 136, 8456, 2, 0, 0) == 8 * 258 * 136 * 4  # few tiles, long K
    assert ws(300, 64, 16384, 2, 0, 5) == 32 * 300 * 64 * 4  # a layout that they do not have: the small tile
    dw = lib.xma_rocm_group_bwd_W_few_rows
    assert dw(p, 64, 1, 1, None, p, 64, 1, 1, p, p, p, 64 * 64, 64, 64, 64, 2, 4, 2, None) == -2  # fp32
    assert dw(p, 64, 1, 1, None, p, 60, 1, 1, p, p, p, 64 * 64, 64, 64, 64, 2, 4, 0, None) == -2  # ldx % 8
    assert dw(p, 60, 1, 1, None, p, 64, 1, 1, p, p, p, 64 * 64, 64, 64, 64, 2, 4, 0, None) == -2  # lddy % 8
    assert dw(None, 64, 1, 1, None, p, 64, 1, 1, p, p, p, 64 * 64, 64, 64, 64, 2, 4, 0, None) == -1
    # empty problems are accepted without touching a pointer
    assert few(None, 64, None, 64 * 64, 64, 0, None, None, None, 64, None, 0, None, 0, None, None, 0, 0, 64, 64, 2, 1, 1, 1, 0, 0, None, 0, None) == 0
    assert lib.xma_rocm_combine(None, 8, None, None, 8, 0, 2, 16, 0, None) == 0
    assert lib.xma_rocm_continuous_count(None, 0, 0, ctypes.c_void_p(16), 4, None, 0, None) == 0


def test_router_gradient_entry_point_arguments():
    """xma_rocm_down_projection_dx_swiglu_router knows slots and rows, not how many experts there are: more slots than experts (ids that
    repeat) and more experts than route counts are taken; the rest is refused before any launch"""
    from xma.rocm import get_library, ops

    lib, p = get_library(), ctypes.c_void_p(1 << 20)

    def call(M=8, N=64, K=64, E=4, k=2, dtype=0, d_w=p, scale=p, space=p, short=0):
        need = lib.xma_rocm_down_projection_dx_swiglu_router_workspace_bytes(M, N, K, E)
        return lib.xma_rocm_down_projection_dx_swiglu_router(p, K, p, K * N, N, p, p, p, 2 * N, p, 2 * N, None, 0, scale, d_w, M, N, K, E, k,
                                                             dtype, space, need - short, None)

    assert call(M=0, E=2, k=4) == 0 and call(M=0, E=4096) == 0 and call(M=0, k=32, d_w=None) == 0
    for bad in (dict(k=0), dict(k=33, M=66), dict(M=7), dict(M=-2), dict(d_w=None), dict(scale=None), dict(dtype=2)):
        assert call(**bad) == -1, bad
    assert call(short=1) == -3 and call(space=None) == -3 and call(space=ctypes.c_void_p((1 << 20) + 8)) == -3
    assert call(M=1 << 24, N=1 << 13, space=p) == -2  # products beyond 32-bit offsets
    # what Python restates
    for M, N, K, E in ((8, 64, 64, 4), (1000, 1032, 256, 8), (4096, 768, 2048, 128), (20000, 16, 64, 4096)):
        slices = lib.xma_rocm_scatter2scatter_workspace_bytes(M, N, K, E)
        assert ops.router_gradient_workspace_bytes(M, N, slices) == lib.xma_rocm_down_projection_dx_swiglu_router_workspace_bytes(M, N, K, E)
    takes = ops.dx2_leaves_router_gradient
    assert takes(0, 8, 64, 32, torch.bfloat16) and takes(0, 8, 64, 2, torch.float16)
    assert not takes(1, 8, 64, 2, torch.bfloat16) and not takes(0, 8, 64, 33, torch.bfloat16) and not takes(0, 8, 64, 2, torch.float32)
    assert takes(0, (1 << 30) - 5, 128, 1, torch.bfloat16) and not takes(0, (1 << 30) - 4, 128, 1, torch.bfloat16)
    for H, E, k, dtype in ((8, 1, 1, 0), (64, 128, 32, 2), (64, 128, 33, 0), (64, 129, 2, 0), (12, 8, 2, 0), (64, 8, 9, 1), (0, 8, 2, 0), (64, 8, 0, 2)):
        name = (torch.bfloat16, torch.float16, torch.float32)[dtype]
        assert ops.gate_bwd_supported(H, E, k, name) == bool(lib.xma_rocm_gate_bwd_supported(H, E, k, dtype)), (H, E, k, dtype)


def test_layer_entry_points_refuse_what_they_cannot_run():
    """xma_rocm_moe_*: every argument that has a rule of its own, before any launch"""
    import struct

    from xma.rocm import get_library

    lib = get_library()
    sizes = ("size T H I E k dtype activation few_up few_down few_dx2 few_dw2 few_dw1 few_dx1 dw2_form recompute workspace_bytes").split()
    pointers = ("x gate_weight w_fc w_proj b_fc b_proj logits router_weights expert_ids counts expert_offsets sorted_scattered_idxs z h "
                "expert_out y workspace dy d_router_weights d_logits dz dw2_operand scattered d_w_fc d_w_proj d_b_fc d_b_proj d_x "
                "d_x_addend").split()
    text = open(os.path.join(ROOT, "include", "xma_rocm.h")).read()
    block = re.sub(r"/\*.*?\*/", "", text[text.index("typedef struct xma_rocm_moe {") : text.index("} xma_rocm_moe;")], flags=re.S)
    assert re.findall(r"\b(\w+)[,;]", block) == sizes + pointers  # the block's fields, in order

    def refused(entry, code, message, **change):
        v = dict.fromkeys(pointers, 256) | dict(T=4, H=64, I=32, E=8, k=2, dtype=0, activation=0, dw2_form=2, recompute=0, workspace_bytes=1 << 30)
        v |= dict(size=8 * len(sizes + pointers)) | dict.fromkeys((s for s in sizes if s.startswith("few_")), 1)
        v |= dict(d_b_fc=0, d_b_proj=0, b_fc=0, b_proj=0) | change
        rc = getattr(lib, "xma_rocm_moe_" + entry)(struct.pack(f"{len(sizes)}q{len(pointers)}Q", *(v[n] for n in sizes + pointers)), None)
        assert rc == code and message in lib.xma_rocm_last_error().decode(), (entry, change, rc, lib.xma_rocm_last_error())

    for entry in ("forward", "backward_router", "backward"):
        refused(entry, -1, "another size", size=8)
        for bad in (dict(T=0), dict(T=1 << 62, k=4), dict(H=0), dict(I=0), dict(E=0), dict(E=16385), dict(k=0), dict(k=9), dict(T=1 << 30, k=4)):
            refused(entry, -1, "T=", **bad)
        refused(entry, -1, "workspace of -1", workspace_bytes=-1)
        for name in ("x", "w_fc", "w_proj", "router_weights", "expert_ids", "expert_offsets", "sorted_scattered_idxs", "z", "expert_out"):
            refused(entry, -1, "null buffer", **{name: 0})
        for bad in (dict(activation=3), dict(activation=-1), dict(activation=1, recompute=1), dict(activation=2, dw2_form=1)):
            refused(entry, -1, "activation", **bad)
    for name in ("logits", "h", "y", "counts"):
        refused("forward", -1, "null buffer", **{name: 0})
    for name in ("logits", "dy", "d_router_weights", "d_logits"):
        refused("backward_router", -1, "null buffer", **{name: 0})
    refused("backward_router", -1, "null buffer", recompute=1, h=0)
    for name in ("dy", "dz", "d_w_fc", "d_w_proj", "scattered", "d_x", "h", "dw2_operand"):
        refused("backward", -1, "null buffer", **{name: 0})
    refused("backward", -1, "null buffer", d_b_fc=256)  # a bias gradient without the bias
    refused("backward", -1, "null buffer", d_b_proj=256)
    refused("backward", -1, "dw2_form 0 with d_b_proj", dw2_form=0, b_proj=256, d_b_proj=256)
    refused("backward", -1, "dw2_form 3", dw2_form=3)
    # what the single calls refuse: a workspace too small for route, or for the K ranges of a few-row launch
    refused("forward", -2, "dtype 5", dtype=5)
    refused("backward", -3, "scatter2scatter_few_rows: workspace", I=64, H=16384, workspace_bytes=16)


def test_whole_backward_refuses_before_any_launch():
    """xma_rocm_moe_backward_gated and _logits: every argument that has a rule of its own, under its own name; what its parts share with the other two
    entries under both (the K slices of its GEMMs take a device to be counted: tests/test_gpu_layer.py)"""
    import struct

    from xma.rocm import get_library

    lib = get_library()
    text = open(os.path.join(ROOT, "include", "xma_rocm.h")).read()
    block = re.sub(r"/\*.*?\*/", "", text[text.index("typedef struct xma_rocm_moe {") : text.index("} xma_rocm_moe;")], flags=re.S)
    names = re.findall(r"\b(\w+)[,;]", block)
    sizes = names[: names.index("x")]
    base = dict.fromkeys(names, 256) | dict(size=8 * len(names), T=4, H=64, I=32, E=8, k=2, dtype=0, activation=0, dw2_form=2, recompute=0)
    base |= dict(workspace_bytes=1 << 30, d_b_fc=0, d_b_proj=0, b_fc=0, b_proj=0) | dict.fromkeys((s for s in sizes if s.startswith("few_")), 1)

    def refused(code, message, d_gate=256, **change):
        v = base | change
        block = struct.pack(f"{len(sizes)}q{len(names) - len(sizes)}Q", *(v[n] for n in names))
        rc = lib.xma_rocm_moe_backward_gated(block, d_gate, None) if gated else lib.xma_rocm_moe_backward_logits(block, None)
        assert rc == code and lib.xma_rocm_last_error().decode().startswith(message), (change, rc, lib.xma_rocm_last_error())

    for gated in (False, True):
        entry = "moe_backward_" + ("gated" if gated else "logits")
        own, experts = entry + ": ", entry + ", as moe_backward: "
        refused(-1, own + "argument block", size=8)
        for bad in (dict(T=0), dict(H=0), dict(E=16385), dict(k=9)):
            refused(-1, own + "T=", **bad)
        refused(-1, own + "workspace of -1", workspace_bytes=-1)
        for name in ("x", "z", "expert_out", "logits", "dy", "d_router_weights", *(("gate_weight", "d_x", "scattered") if gated else ("d_logits",))):
            refused(-1, own + "null buffer", **{name: 0})
        refused(-1, own + "null buffer", recompute=1, h=0)
        refused(-1, own + "activation", activation=3)
        for name in ("dz", "d_w_fc", "d_w_proj", "h", "dw2_operand", *(() if gated else ("d_x", "scattered"))):
            refused(-1, experts + "null buffer", **{name: 0})
        refused(-1, experts + "null buffer", d_b_fc=256)
        refused(-1, experts + "dw2_form 3", dw2_form=3)
        refused(-1, experts + "dw2_form 0 with d_b_proj", dw2_form=0, b_proj=256, d_b_proj=256)
    for bad in (dict(H=68), dict(E=129), dict(k=33, E=64), dict(dtype=5)):
        refused(-2, own + "H=", **bad)
    refused(-1, own + "null or misaligned", workspace=0)
    for bad in (dict(x=264), dict(gate_weight=264), dict(d_x=264), dict(scattered=264), dict(workspace=264), dict(d_gate=264)):
        refused(-1, own + "null or misaligned", **bad)
    need = lib.xma_rocm_gate_bwd_workspace_bytes(4, 64, 8)
    refused(-3, own + f"workspace of {need - 1} bytes, {need} needed", workspace_bytes=need - 1)


def test_few_token_dispatch_rule():
    """which grouped GEMM forms take the kernels of the few-token regime: by rows per expert on average, per form, with a
    cap on the rows in all; fp32 never"""
    from xma.rocm import ops

    bf = torch.bfloat16
    assert ops._few_rows(14, 8, bf, "x @ W^T") and ops._few_rows(768, 8, bf, "x @ W^T") and not ops._few_rows(769, 8, bf, "x @ W^T")
    assert ops._few_rows(3072, 128, bf, "dy @ W") and not ops._few_rows(16385, 1024, bf, "x @ W^T")  # the cap on the rows
    assert ops._few_rows(768, 8, bf, "dy @ W") and not ops._few_rows(769, 8, bf, "dy @ W")
    assert ops._few_rows(1024, 8, bf, "dW") and not ops._few_rows(1025, 8, bf, "dW")
    assert ops._few_rows(16384, 128, bf, "dW") and not ops._few_rows(16385, 128, bf, "dW")
    assert not ops._few_rows(0, 8, bf, "dW") and not ops._few_rows(14, 8, torch.float32, "dW")
    assert ops._few_rows(14, 8, torch.float16, "dy @ W")


def test_which_few_row_launches_are_cut_along_k():
    """the kernel with four K steps in flight cuts nothing, so the workspace says which launches of x @ W^T it takes among those that the
    small tile would cut: not where that makes three or four K ranges, nor of two where one expert may have several times 32 rows (measured
    45 -> 82 us), nor with an activation behind fewer than 32 workgroups"""
    from xma.rocm import get_library

    need = lambda M, N, K, E, epi=0: get_library().xma_rocm_scatter2scatter_few_rows_workspace_bytes(M, N, K, E, 0, epi)
    for epi in (0, 1):
        assert need(64, 512, 2048, 4, epi) == 4 * 64 * 512 * 4 and need(16, 512, 1536, 4, epi) == 3 * 16 * 512 * 4
        assert need(16, 4096, 2048, 4, epi) == 4 * 16 * 4096 * 4 and need(1008, 320, 2000, 45, epi) == 4 * 1008 * 320 * 4
        # two ranges: up to eight rows per expert
        assert need(64, 1024, 1024, 8, epi) == 0 and need(65, 1024, 1024, 8, epi) == 2 * 65 * 1024 * 4
        assert need(32, 512, 1408, 4, epi) == epi * 2 * 32 * 512 * 4
        # four waves with rows for most experts: only K between 512 and 1024, which the small tile would not cut either
        assert need(128, 1024, 1024, 32, epi) == 2 * 128 * 1024 * 4 and need(128, 1024, 1016, 32, epi) == 0
    assert need(64, 512, 8192, 8) and need(12, 2816, 2048, 64) == 0  # K beyond; the vector kernel


def test_mid_rows_dispatch_rule():
    """which launches beyond the few-token limits take the few-row entry points for their 128 x 256 tiles"""
    from xma.rocm import ops

    bf, store, glu, bwd = torch.bfloat16, ops.EPI_STORE, ops.EPI_SWIGLU, ops.EPI_SWIGLU_BWD
    fwd = lambda M, N, K, E, kn=0, ldw=4096, span=1 << 20, dt=bf, epi=store: ops._mid_rows_fwd(M, N, K, E, kn, ldw, span, dt, epi)
    assert fwd(256 * 64, 2816, 2048, 64) and not fwd(1000 * 64, 2816, 2048, 64)  # many rounds: by the rows per expert
    assert fwd(1024 * 16, 2048, 2048, 16) and not fwd(4000 * 16, 2048, 2048, 16)  # few rounds, the last one nearly empty
    assert fwd(100 * 8, 4096, 28672, 8) and not fwd(176 * 8, 4096, 28672, 8)  # long K
    # many rounds, and an epilogue that writes a second tensor: measured 25 and 15 % slower with the smaller tiles
    assert not fwd(43320, 5328, 520, 6, epi=glu) and not fwd(3950, 15200, 2560, 25, epi=glu)
    # long K, experts of two of the smaller tiles and one of the larger: measured 484 against 575, 333 against 379 and 450 against 573 us
    assert not fwd(125 * 64, 2944, 6272, 64) and not fwd(134 * 128, 1344, 4096, 128) and not fwd(143 * 32, 5792, 4264, 32, epi=glu)
    assert fwd(134 * 128, 1344, 2048, 128) and fwd(300 * 16, 1024, 4096, 16)
    assert fwd(2048, 16384, 2048, 8, epi=glu) and fwd(8198, 4096, 1024, 16, epi=4) and not fwd(32000, 4096, 1024, 16, epi=4)
    assert not fwd(65536, 512, 64, 1024) and not fwd(2000, 64, 64, 1025) and not fwd(0, 64, 64, 8)
    assert fwd(999, 64, 64, 8, kn=0, epi=glu) and not fwd(999, 64, 64, 8, kn=1, epi=glu)
    assert fwd(999, 64, 64, 8, kn=1, epi=bwd) and not fwd(999, 64, 64, 8, kn=0, epi=bwd)
    assert not fwd(999, 64, 64, 8, span=1 << 31) and not fwd(999, 64, 64, 8, ldw=1 << 23) and not fwd(999, 64, 64, 8, dt=torch.float32)
    dw = ops._mid_rows_dw
    assert dw(640 * 64, 4096, 4096, 64, bf) and not dw(640 * 64 + 1, 4096, 4096, 64, bf)
    assert dw(1 << 20, 1024, 512, 8, bf) and not dw(1 << 20, 4096, 4096, 8, bf)
    assert dw(8192 * 8, 1024, 1024, 8, bf) and not dw(1024 * 8, 1024 + 8, 1024, 8, bf)  # at most one of the smaller tiles per compute unit
    assert not dw(999, 64, 64, 65536, bf) and not dw(999, 64, 64, 8, torch.float32)
    assert dw(128 * 16, 4096, 4096 + 8, 16, bf) and not dw(129 * 16, 4096, 4096 + 8, 16, bf)  # rows off 64-byte boundaries, many rounds
    assert dw(129 * 16, 4096, 768 + 8, 16, bf) and dw(129 * 16, 4096, 4096 + 32, 16, bf)
    loader = ops._dw_loader_scales  # a handful of tiles: up to 128 rows per expert; a round or two of them: 96 or 64
    assert loader(128 * 10, 10, bf, 608, 536) and not loader(129 * 10, 10, bf, 608, 536)
    assert loader(96 * 20, 20, bf, 1608, 736) and not loader(97 * 20, 20, bf, 1608, 736) and not loader(65 * 20, 20, bf, 1608, 744)
    # launches that the library prefers, whose sums would not fit if the small tile made them
    assert ops._few_rows_fwd(8198, 1024, 4096, 4, 0, 4096, 4099 * 4096, bf, glu) and ops._few_rows_fwd(8198, 4096, 1024, 4, 1, 4096, 8198 * 1024, bf, store)
    assert ops._few_rows_fwd(8000, 8192, 1024, 4, 1, 8192, 2000 * 1024, bf, bwd) and ops._few_rows_fwd(8000, 1024, 16384, 4, 1, 1024, 8000 * 16384, bf, store)
    assert ops._dw_loader_scales(64 * 8, 8, bf) and not ops._dw_loader_scales(64 * 8 + 1, 8, bf)


def test_layer_plan_makes_the_choices_of_the_ops(monkeypatch):
    """which entry point each GEMM of the layer's call takes, against what the single ops would do with their operands; and a plan that was
    laid out under other dispatch limits is not used again"""
    import random

    from xma.layers.moe import rocm_implementation as R
    from xma.rocm import ops

    monkeypatch.setattr(ops, "scatter2scatter_workspace_bytes", lambda *a: 0)
    calls = {}
    for name in ("xma_rocm_scatter2scatter_few_rows", "xma_rocm_scatter2scatter_bias", "xma_rocm_down_projection_dx_swiglu",
                 "xma_rocm_group_bwd_W_few_rows", "xma_rocm_group_bwd_W", "xma_rocm_group"):
        calls[name] = lambda *a, n=name: taken.append(n) or 0
    calls["xma_rocm_scatter2scatter_few_rows_workspace_bytes"] = lambda *a: 0
    lib = ops.get_library()

    class Library:
        def __getattr__(self, name):
            return calls.get(name) or getattr(lib, name)

    class Device(torch.Tensor):  # a tensor without memory that passes for one on the GPU
        is_cuda = property(lambda self: True)

    new = lambda *shape, dtype: torch.empty(shape, dtype=dtype, device="meta").as_subclass(Device)
    rng, seen = random.Random(5), set()
    for _ in range(150):
        E, H, I = rng.choice([2, 8, 64, 1200]), 8 * rng.randint(1, 600), 16 * rng.randint(1, 300)
        k, dtype, act = rng.randint(1, min(E, 6)), rng.choice([torch.bfloat16, torch.bfloat16, torch.float32]), rng.choice(["swiglu_packed", "swiglu_packed", "tanh"])
        T = max(1, int(E * 2 ** rng.uniform(0, 13)) // k)
        M, U = T * k, 2 * I if act == "swiglu_packed" else I
        plan = R._plan(T, H, I, E, k, dtype, act, False, True, 0, ops.dispatch_limits())
        few = dict(zip(("up", "down", "dx2", "dw2", "dw1", "dx1", "form"), R._BLOCK_SIZES.unpack(plan.sizes_forward)[8:15]))
        x, dy, z, h, out = new(T, H, dtype=dtype), new(T, H, dtype=dtype), new(M, U, dtype=dtype), new(M, I, dtype=dtype), new(M, H, dtype=dtype)
        w_fc, w_proj = new(E, U, H, dtype=dtype), new(E, H, I, dtype=dtype)
        idx, offs, w = new(M, dtype=torch.int64), new(E, dtype=torch.int64), new(M, dtype=dtype)
        with monkeypatch.context() as m:
            m.setattr(ops, "get_library", Library)
            m.setattr(ops, "_stream", lambda t: 0)
            m.setattr(ops, "_ptr", lambda t: None if t is None else 256)
            m.setattr(ops, "_few_rows_workspace_bytes", lambda *a: lib.xma_rocm_scatter2scatter_few_rows_workspace_bytes(*a))
            m.setattr(torch, "empty", lambda *a, **kw: None)
            want = {}
            for key, call in dict(
                up=(lambda: ops.up_projection_swiglu_rocm(x, w_fc.permute(0, 2, 1), idx, offs, z, h, k)) if act == "swiglu_packed" else None,
                down=lambda: ops.scatter2scatter_rocm(h, w_proj.permute(0, 2, 1), idx, offs, out, None, 1, True, False),
                dx2=(lambda: ops.down_projection_dx_swiglu_rocm(dy, w_proj, idx, offs, z, z, w, k)) if act == "swiglu_packed" else None,
                dw2={0: lambda: ops.group_bwd_W_rocm(dy, h, idx, offs, w_proj.permute(0, 2, 1), w, k, 0),
                     1: lambda: ops.group_bwd_W_rocm(dy, h, idx, offs, w_proj.permute(0, 2, 1), None, k, 0),
                     2: lambda: ops.group_bwd_W_rocm(out, h, idx, offs, w_proj.permute(0, 2, 1), None, 0, 0)}[few["form"]],
                dw1=lambda: ops.group_bwd_W_rocm(z, x, idx, offs, w_fc.permute(0, 2, 1), None, 0, k),
                dx1=lambda: ops.scatter2scatter_rocm(z, w_fc, idx, offs, out, None, 1, True, False),
            ).items():
                if call is None:
                    continue
                taken = []
                call()
                want[key] = int(taken[-1].endswith("few_rows"))
        assert want == {key: few[key] for key in want}, (T, H, I, E, k, dtype, act)
        seen |= {(key, v) for key, v in want.items()}
    assert len(seen) == 12  # both choices of all six

    R._plan.cache_clear()
    limits = [n for n in vars(ops) if re.match(r"(FEW|MID)_ROWS_[A-Z_]+$", n)]
    before = ops.dispatch_limits()
    for name in limits:
        with monkeypatch.context() as m:
            value = getattr(ops, name)
            m.setattr(ops, name, dict.fromkeys(value, 1) if isinstance(value, dict) else value + 1)
            assert ops.dispatch_limits() != before, name


def test_layer_call_leaves_other_shapes_to_the_ops(monkeypatch):
    """the layer's library call reads all its tensors by one E, H and I, so whatever has others goes through the ops (None here),
    which check each tensor"""
    from xma.functional import swiglu_packed
    from xma.layers import MoE
    from xma.layers.moe import rocm_implementation as R

    monkeypatch.setattr(R, "router_gate_topk_supported", lambda x, w, k: w.dtype == torch.bfloat16)  # as on the GPU
    reached = []
    monkeypatch.setattr(R, "_layer_forward", lambda *a: reached.append(a) or (a[0], a[0], None, None))

    def taken(**change):
        moe = MoE(8, 2, 64, 32, swiglu_packed, True, add_bias=True, std=0.02).bfloat16()
        for name, value in change.items():
            part, _, field = name.partition("__")
            setattr(getattr(moe, part) if field else moe, field or part, value)
        n = len(reached)
        with torch.no_grad():
            out = R.layer(moe, torch.randn(5, 64).bfloat16())
        assert (out is None) == (len(reached) == n)
        return out is not None

    param = lambda *shape: nn.Parameter(torch.zeros(*shape, dtype=torch.bfloat16))
    assert taken()
    assert not taken(gate__weight=param(6, 64)) and not taken(gate__weight=param(9, 64)) and not taken(gate__weight=param(8, 72))
    assert not taken(c_fc__bias=param(8, 32)) and not taken(c_fc__bias=param(7, 64)) and not taken(c_proj__bias=param(8, 32))
    assert not taken(gate__weight=nn.Parameter(torch.zeros(8 * 64 + 1, dtype=torch.bfloat16)[1:].view(8, 64)))  # off a 16-byte boundary
    assert not taken(num_experts=9) and not taken(c_proj__weight=param(7, 64, 32)) and not taken(c_fc__weight=param(8, 64, 72))


def test_layer_backward_looks_at_what_saved_tensor_hooks_return():
    """the library reads the saved tensors by address: another layout is laid out again, another kind is refused"""
    from xma.layers.moe import rocm_implementation as R

    bf = torch.bfloat16
    like = torch.zeros(4, 8, dtype=bf)
    x, kept = torch.randn(4, 8).to(bf), torch.arange(64, dtype=torch.uint8)
    wide = torch.zeros(4, 16, dtype=bf)[:, :8].copy_(x)
    off = torch.zeros(65, dtype=torch.uint8)[1:].copy_(kept)
    shapes = ((4, 8), (3, 8), (64,))
    assert all(a is b for a, b in zip(R._unpacked((x, None, kept), shapes, like), (x, None, kept)))
    for got, want in zip(R._unpacked((wide, None, off), shapes, like), (x, None, kept)):
        assert got is want or (torch.equal(got, want) and got.is_contiguous() and got.data_ptr() % 16 == 0)
    for bad in ((x.float(), None, kept), (x[:3], None, kept), (x, None, kept.to(bf)[:32]), (x, None, kept.int()), (x.to("meta"), None, kept),
                (x.to(torch.uint8), None, kept), (x.half(), None, kept)):
        with pytest.raises(AssertionError):
            R._unpacked(bad, shapes, like)


def test_fused_router_shape_rule_matches_the_library():
    """the Python restatement of the fused gate + router kernel's coverage (evaluated under torch.compile, where a ctypes
    call cannot be traced) against the library's own answer"""
    from xma.rocm import get_library
    from xma.rocm.ops import router_gate_topk_supported

    lib = get_library()
    codes = {torch.bfloat16: 0, torch.float16: 1, torch.float32: 2}
    for dtype, code in codes.items():
        for H in (0, 4, 8, 12, 64, 4096):
            for E in (0, 1, 8, 32, 33, 128, 129, 2048):
                for k in (0, 1, 2, 8, 32, 33, 128):
                    assert router_gate_topk_supported(H, E, k, dtype) == bool(
                        lib.xma_rocm_router_gate_topk_supported(H, E, k, code)), (dtype, H, E, k)


def test_backend_selection_and_errors():
    from xma import Accelerator, KernelBackend
    from xma.functional import continuous_count, swiglu_packed
    from xma.layers import MoE

    assert KernelBackend.torch.verify_accelerator()
    if not torch.cuda.is_available():
        assert Accelerator.get_accelerator() == Accelerator.cpu
        assert Accelerator.get_kernel_backend() == KernelBackend.torch
        assert not KernelBackend.rocm.verify_accelerator()
        with pytest.raises(AssertionError):  # explicit backend on the wrong accelerator (moe/__init__.py:205-208)
            continuous_count(torch.zeros(4, dtype=torch.int32), 4, kernel_backend=KernelBackend.rocm)
    x = torch.randint(0, 5, (100,))
    assert continuous_count(x, 1).tolist() == [100]
    assert continuous_count(x, 5, kernel_backend=KernelBackend.torch).dtype == torch.uint32
    with pytest.raises(AssertionError):
        continuous_count(x.view(10, 10), 5, kernel_backend=KernelBackend.torch)
    with pytest.raises(AssertionError):
        continuous_count(x.float(), 5, kernel_backend=KernelBackend.torch)
    moe = MoE(4, 2, 16, 24, swiglu_packed, True, add_bias=False, std=0.02)
    with pytest.raises((ValueError, AssertionError)):  # a backend this build does not have (moe/__init__.py:251-252)
        moe(torch.randn(3, 16), kernel_backend=KernelBackend.triton)


def test_module_layout_matches_reference_state_dict():
    from xma.layers import MoE
    from xma.layers.moe import Experts

    moe = MoE(6, 2, 32, 48, nn.GLU(), True, add_bias=True, std=0.02)
    sd = moe.state_dict()
    assert {k: tuple(v.shape) for k, v in sd.items()} == {
        "gate.weight": (6, 32),
        "c_fc.weight": (6, 96, 32), "c_fc.bias": (6, 96), "c_fc.N_array": (6,), "c_fc.K_array": (6,),
        "c_proj.weight": (6, 32, 48), "c_proj.bias": (6, 32), "c_proj.N_array": (6,), "c_proj.K_array": (6,),
    }
    assert sd["c_fc.N_array"].dtype == torch.uint32 and sd["c_fc.N_array"].view(torch.int32).tolist() == [96] * 6
    assert sd["c_proj.K_array"].view(torch.int32).tolist() == [48] * 6
    assert (sd["c_fc.bias"] == 0).all()
    y, logits = moe(torch.randn(2, 5, 32))
    assert y.shape == (2, 5, 32) and logits.shape == (10, 6)
    e = Experts(3, 4, 5, add_bias=False, std=0.1)
    assert e.bias is None and "in_features=4" in e.extra_repr()
    moe1 = MoE(4, 1, 16, 8, nn.GELU(approximate="tanh"), False, add_bias=False, std=0.02)  # top-1 uses max
    assert moe1(torch.randn(7, 16))[0].shape == (7, 16)


def test_torch_backend_matches_oracle_in_bf16():
    from oracle import moe as oracle
    from xma import KernelBackend, set_seed
    from xma.functional import swiglu_packed
    from xma.layers import MoE

    set_seed(3)
    moe = MoE(8, 2, 64, 96, swiglu_packed, True, add_bias=False, std=0.02).to(torch.bfloat16)
    x = torch.randn(50, 64).bfloat16()
    rw, sel = oracle.routing_weights(torch.randn(50, 8), 2, torch.bfloat16)
    y = moe._compute_experts(x, rw, sel, kernel_backend=KernelBackend.torch)
    want = oracle.experts_forward(x, rw, sel, moe.c_fc.weight.data, moe.c_proj.weight.data, oracle.swiglu_packed)
    assert torch.equal(y, want)


def test_rocm_ops_fail_loudly_without_the_library(monkeypatch):
    from xma.rocm import loader

    monkeypatch.setattr(loader, "_lib", None)
    monkeypatch.setattr(loader, "LIBRARY_PATH", "/nonexistent/libxma_rocm.so")
    with pytest.raises(loader.RocmLibraryError):
        loader.get_library()
