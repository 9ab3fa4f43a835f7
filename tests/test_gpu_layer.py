"""The layer as one autograd node against the same layer through the single ops: same launches, so bit for bit."""

import contextlib

import pytest
import torch
import torch.nn as nn

from xma.functional import swiglu_packed
from xma.layers import MoE

from .test_gpu_ops import _few_rows_limit, _tol
from .utils import nerr


pytestmark = pytest.mark.gpu


class _ThroughOps(MoE):
    def _compute_experts(self, *args, **kwargs):  # overridden: the layer does not run as one call
        return super()._compute_experts(*args, **kwargs)


def _layers(T, E, k, H, I, dtype, bias=False, save=True, seed=3, act=swiglu_packed):
    torch.manual_seed(seed)
    glu = act is swiglu_packed
    one = MoE(E, k, H, I, act, glu, add_bias=bias, std=0.05)
    if bias:
        nn.init.normal_(one.c_fc.bias)
        nn.init.normal_(one.c_proj.bias)
    ops = _ThroughOps(E, k, H, I, act, glu, add_bias=bias, std=0.05)
    ops.load_state_dict(one.state_dict())
    one, ops = one.to("cuda", dtype), ops.to("cuda", dtype)
    one.save_activations = ops.save_activations = save
    return one, ops, torch.randn(T, H, device="cuda", dtype=dtype), torch.randn(T, H, device="cuda", dtype=dtype)


def _step(moe, x, dy, aux=0.0, use_y=True):
    x = x.clone().requires_grad_()
    y, logits = moe(x)
    loss = (y * dy).sum() if use_y else 0.0
    if aux:
        loss = loss + aux * (logits.float() ** 2).sum()
    grads = torch.autograd.grad(loss, [x, *moe.parameters()], allow_unused=True)
    return [y, logits, *grads]


def _same(a, b):
    assert len(a) == len(b)
    for u, v in zip(a, b):
        assert (u is None) == (v is None)
        assert u is None or (u.shape == v.shape and u.dtype == v.dtype and torch.equal(u, v))


CASES = [
    # T, E, k, H, I: vector kernel, small tile, 128 x 256 tiles (both forms of dW2's operand), 256 x 256 tiles
    (1, 8, 2, 2048, 64),
    (7, 16, 8, 64, 24),
    (33, 8, 2, 64, 40),
    (300, 8, 2, 136, 72),
    (500, 8, 5, 128, 64),
    (3100, 4, 2, 128, 2816),
]


@pytest.mark.parametrize("bias,save", [(False, True), (True, True), (False, False), (True, False)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("case", CASES)
def test_one_call_matches_the_ops(case, dtype, bias, save):
    T, E, k, H, I = case
    one, ops, x, dy = _layers(T, E, k, H, I, dtype, bias, save)
    with torch.no_grad():
        _same(one(x), ops(x))
    _same(_step(one, x, dy), _step(ops, x, dy))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_which_gradients_are_asked_for(dtype):
    """an auxiliary loss on the logits, alone and beside the output; frozen gate; frozen experts; no gradient of x"""
    one, ops, x, dy = _layers(65, 8, 2, 64, 32, dtype)
    _same(_step(one, x, dy, aux=0.1), _step(ops, x, dy, aux=0.1))
    _same(_step(one, x, dy, aux=0.1, use_y=False), _step(ops, x, dy, aux=0.1, use_y=False))
    for frozen in (["gate.weight"], ["c_fc.weight", "c_proj.weight"], ["gate.weight", "c_fc.weight", "c_proj.weight"]):
        got = []
        for moe in (one, ops):
            for n, p in moe.named_parameters():
                p.requires_grad_(n not in frozen)
                p.grad = None
            xx = x.clone().requires_grad_(len(frozen) == 3)
            moe(xx)[0].backward(dy)
            got.append([xx.grad, *(p.grad for p in moe.parameters())])
        _same(*got)


def test_what_goes_through_the_ops():
    """forms the layer entry point does not describe are accepted as before, with the same results"""
    from xma.layers.moe import rocm_implementation as R

    one, ops, x, dy = _layers(40, 8, 2, 64, 32, torch.bfloat16)
    assert R.layer(one, x) is not None
    wide = torch.randn(40, 80, device="cuda", dtype=torch.bfloat16)
    assert R.layer(one, wide[:, 8:72]) is None and R.layer(one, x[:0]) is None
    flat = torch.randn(40 * 64 + 1, device="cuda", dtype=torch.bfloat16)[1:].view(40, 64)  # starts off a 16-byte boundary
    assert R.layer(one, flat) is None
    held = one.c_fc.weight
    one.c_fc.weight = nn.Parameter(held.detach().transpose(1, 2).contiguous().transpose(1, 2))  # same values, (E, in, out) storage
    assert R.layer(one, x) is None
    one.c_fc.weight = held
    with torch.autograd.forward_ad.dual_level():
        assert R.layer(one, x) is None
    y, logits = one(x.view(5, 8, 64))
    assert y.shape == (5, 8, 64) and logits.shape == (40, 8)
    torch.manual_seed(0)
    with torch.autograd.graph.save_on_cpu():
        a = _step(one, x, dy)
    _same(a, _step(ops, x, dy))


def test_workspace_too_small_is_refused(monkeypatch):
    """a workspace that holds less than the K slices of the 256 x 256 kernels: each of the three entries refuses it before any launch"""
    from xma.layers.moe import rocm_implementation as R
    from xma.rocm import ops
    from xma.rocm.loader import RocmLibraryError, get_library

    T, E, k, H, I = 300, 4, 2, 2048, 1024
    one, _, x, dy = _layers(T, E, k, H, I, torch.bfloat16, save=False)
    plan = R._plan
    short = ops.route_workspace_elements(T * k, E) * 4
    assert get_library().xma_rocm_scatter2scatter_workspace_bytes(T * k, 2 * I, H, E) > short
    cut = set()

    def cut_plan(*args):
        p = plan.__wrapped__(*args)
        for name in cut:
            setattr(p, name, getattr(p, name)[:-8] + short.to_bytes(8, "little"))
        return p

    monkeypatch.setattr(R, "_plan", cut_plan)
    with _few_rows_limit(0):
        cut = {"sizes_forward"}
        with torch.no_grad(), pytest.raises(RocmLibraryError, match="xma_rocm_moe_forward failed with code -3"):
            one(x)
        cut = {"sizes_backward"}
        for save, entry in ((False, "xma_rocm_moe_backward_router"), (True, "xma_rocm_moe_backward")):
            one.save_activations = save
            y = one(x.clone().requires_grad_())[0]
            with pytest.raises(RocmLibraryError, match=f"{entry} failed with code -3"):
                y.backward(dy)
    torch.cuda.synchronize()


@pytest.mark.parametrize("autocast", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_backward_in_an_autocast_region(dtype, autocast):
    """the gate's product there comes in the region's dtype; what the layer adds to d_x is its value, not its bytes"""
    one, ops, x, dy = _layers(40, 8, 2, 64, 32, dtype)
    with torch.autocast("cuda", dtype=autocast):
        _same(_step(one, x, dy), _step(ops, x, dy))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_saved_tensor_hooks(dtype):
    """what hooks hand back for the saved tensors: other strides and starts give the same gradients, another dtype or device an error"""

    def moved(t):  # the same values in rows further apart, or off a 16-byte boundary
        if t.dim() == 1:
            return torch.empty(t.numel() + 1, device=t.device, dtype=t.dtype)[1:].copy_(t)
        return t.new_empty(*t.shape[:-1], t.shape[-1] + 8)[..., : t.shape[-1]].copy_(t)

    one, _, x, dy = _layers(40, 8, 2, 64, 32, dtype, bias=True)
    want = _step(one, x, dy)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: moved(t) if t.dtype in (dtype, torch.uint8) else t):
        _same(_step(one, x, dy), want)
    for wrong in (lambda t: t.cpu(), lambda t: t.double()):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, wrong):
            y = one(x.clone().requires_grad_())[0]
        with pytest.raises(AssertionError):
            y.backward(dy)


@pytest.mark.parametrize("T", [40, 5000])
def test_gates_the_entry_point_does_not_describe(T):
    """a gate weight off a 16-byte boundary takes the router's kernel as a copy, as the ops do, and a gate over fewer experts than the
    layer has is answered: bit for bit what the ops give"""
    one, ops, x, dy = _layers(T, 8, 2, 64, 32, torch.bfloat16)
    shifted = torch.empty(8 * 64 + 1, device="cuda", dtype=torch.bfloat16)[1:].view(8, 64)
    for weight in (shifted.copy_(one.gate.weight.detach()), one.gate.weight.detach()[:6].clone()):
        one.gate.weight, ops.gate.weight = nn.Parameter(weight), nn.Parameter(weight)
        _same(_step(one, x, dy), _step(ops, x, dy))


def test_two_passes_before_the_backward():
    """each pass keeps its own buffers"""
    one, ops, x, dy = _layers(50, 8, 2, 64, 32, torch.bfloat16)
    got = []
    for moe in (one, ops):
        x1, x2 = x.clone().requires_grad_(), (x * 0.5).requires_grad_()
        y1, y2 = moe(x1)[0], moe(x2)[0]
        y1.backward(dy, retain_graph=True)
        y2.backward(dy)
        y1.backward(dy)
        got.append([x1.grad, x2.grad, *(p.grad for p in moe.parameters())])
    _same(*got)


@pytest.mark.parametrize("form,bias", [("tanh", False), ("tanh", True), ("none", True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("case", [*CASES, (5, 8, 2, 64, 2048), (700, 4, 2, 1024, 264)])
def test_gelu_matches_the_ops(case, dtype, form, bias):
    """GELU in the epilogues (or passes) of the library against the ops with torch's GELU between them; the gradient of the
    pre-activations is not rounded in between here, hence agreement within the bar of the ops"""
    from xma.layers.moe import rocm_implementation as R

    T, E, k, H, I = case
    one, ops, x, dy = _layers(T, E, k, H, I, dtype, bias, act=nn.GELU(approximate=form))
    with torch.no_grad():
        got = R.layer(one, x)
        assert got is not None and R._activation(ops) == form
        for a, b in zip(got, ops(x)):
            assert torch.isfinite(a).all() and nerr(a, b) <= _tol(dtype)
    for a, b in zip(_step(one, x, dy), _step(ops, x, dy)):
        assert torch.isfinite(a).all() and nerr(a, b) <= _tol(dtype)


def test_hooked_activation_is_called():
    one, _, x, _ = _layers(9, 8, 2, 64, 32, torch.bfloat16, act=nn.GELU(approximate="tanh"))
    calls = []
    one.act.register_forward_hook(lambda *a: calls.append(1))
    one(x)
    assert calls


@pytest.mark.parametrize("T,E,k", [(1, 8, 2), (2, 1, 1), (5, 33, 3), (16, 128, 8), (16, 40, 32), (16, 96, 1), (17, 128, 8)])
def test_routing_behind_the_gate(T, E, k):
    """up to 16 tokens the router's kernel routes as well: bit-identical to route's own kernel, also where equal logits tie"""
    one, ops, x, dy = _layers(T, E, k, 136, 64, torch.bfloat16)
    with torch.no_grad():
        for m in (one, ops):
            m.gate.weight[E // 2 :] = m.gate.weight[E // 2].clone()
    _same(_step(one, x, dy), _step(ops, x, dy))


@pytest.mark.parametrize("act", [swiglu_packed, nn.GELU(approximate="tanh")], ids=["swiglu", "gelu"])
@pytest.mark.parametrize("T,k", [(7, 2), (300, 2), (300, 4)])  # routing inside the router's kernel; 128 x 256 tiles, both operands of dW2
def test_side_stream_capture_and_replay(T, k, act):
    """forward and backward of the layer as one call on another stream, and captured once and replayed on new inputs (new routing
    included) with eager passes and synchronisations in between"""
    from xma.layers.moe import rocm_implementation as R

    one, _, sx, sdy = _layers(T, 8, k, 256, 512, torch.bfloat16, act=act)
    assert R.layer(one, sx) is not None

    def step(x, dy):
        x = x.detach().requires_grad_()
        for p in one.parameters():
            p.grad = None
        y, logits = one(x)
        y.backward(dy)
        return [y.detach(), logits.detach(), x.grad, *(p.grad for p in one.parameters())]

    want = step(sx, sdy)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(3):
            got = step(sx, sdy)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    _same(got, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = step(sx, sdy)
    for seed in range(4):
        g = torch.Generator(device="cuda").manual_seed(seed)
        x, dy = (torch.randn(t.shape, device="cuda", generator=g).bfloat16() for t in (sx, sdy))
        sx.copy_(x), sdy.copy_(dy)
        graph.replay()
        torch.cuda.synchronize()
        got = [o.clone() for o in outs]
        _same(got, step(x, dy))
        torch.cuda.synchronize()


def _biased_gate(moe, bias):
    gate = nn.Linear(moe.gate.in_features, moe.gate.out_features).to("cuda", moe.gate.weight.dtype)
    with torch.no_grad():
        gate.weight.copy_(moe.gate.weight)
        gate.bias.copy_(bias)
    moe.gate = gate


LARGE_TILES = [  # T, E, k, H, I through the 256 x 256 tiles: both forms of dW2's operand, parts of a row's products that end anywhere
    (33, 8, 2, 64, 40),
    (300, 8, 2, 136, 72),
    (500, 8, 5, 128, 264),
    (300, 160, 2, 64, 136),  # more experts than the gate's kernels take
    (40, 8, 8, 64, 128),
]


def _takes_large_tiles(moe, T, dtype):
    from xma.layers.moe import rocm_implementation as R
    from xma.rocm import ops

    E, H, I = moe.c_proj.weight.shape
    sizes = R._plan(T, H, I, E, moe.top_k, dtype, "swiglu_packed", moe.c_proj.bias is not None, bool(moe.save_activations), 0, ops.dispatch_limits())
    return R._BLOCK_SIZES.unpack(sizes.sizes_backward)[10] == 0


@pytest.mark.parametrize("bias,save", [(False, True), (False, False), (True, True), (True, False)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", [*LARGE_TILES, (32768, 8, 2, 256, 768)])  # the last by the dispatch's own rule
def test_one_call_matches_the_ops_by_large_tiles(case, dtype, bias, save):
    """there dX2 leaves the gradient of the router weights, whatever else hangs on the logits: with and without an auxiliary loss, a gate
    with a bias, biases of the experts (whose gradient comes from the expert outputs)"""
    T, E, k, H, I = case
    print(f"layer by large tiles {case} {dtype} bias={bias} save={save}", flush=True)
    one, ops, x, dy = _layers(T, E, k, H, I, dtype, bias, save)
    with _few_rows_limit(0) if T < 1000 else contextlib.nullcontext():
        assert _takes_large_tiles(one, T, dtype)
        for aux in (0.0, 0.1):
            _same(_step(one, x, dy, aux), _step(ops, x, dy, aux))
        gate_bias = torch.randn(E, device="cuda").to(dtype)
        for moe in (one, ops):
            _biased_gate(moe, gate_bias)
        _same(_step(one, x, dy, 0.1), _step(ops, x, dy, 0.1))


@pytest.mark.parametrize("aux", [0.0, 0.1])
@pytest.mark.parametrize("save", [True, False])
@pytest.mark.parametrize("k", [2, 4])
def test_large_tiles_capture_and_replay(k, save, aux):
    """the same backward captured once and replayed on new inputs, with eager passes and synchronisations in between"""
    one, _, sx, sdy = _layers(300, 8, k, 136, 264, torch.bfloat16, save=save)

    def step(x, dy):
        x = x.detach().requires_grad_()
        y, logits = one(x)
        outs, grads = ([y, logits], [dy, aux * logits.detach()]) if aux else ([y], [dy])
        return [t.detach() for t in (y, logits, *torch.autograd.grad(outs, [x, *one.parameters()], grads))]

    print(f"large tiles captured k={k} save={save} aux={aux}", flush=True)
    with _few_rows_limit(0):
        assert _takes_large_tiles(one, 300, torch.bfloat16)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(3):
                step(sx, sdy)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            outs = step(sx, sdy)
        for seed in range(4):
            g = torch.Generator(device="cuda").manual_seed(seed)
            x, dy = (torch.randn(t.shape, device="cuda", generator=g).bfloat16() for t in (sx, sdy))
            sx.copy_(x), sdy.copy_(dy)
            graph.replay()
            torch.cuda.synchronize()
            got = [o.clone() for o in outs]
            _same(got, step(x, dy))
            torch.cuda.synchronize()


@pytest.mark.parametrize("k,bias,large,again", [(2, False, True, 0), (5, False, True, 0), (2, True, True, 1), (2, False, False, 1), (5, False, False, 1)])
def test_what_the_ops_compute_again(monkeypatch, k, bias, large, again):
    """save_activations = False: the down-projection is repeated only where something reads the expert outputs (a bias there, few-row
    launches), with the gradients of a layer that keeps them either way"""
    from xma.rocm import ops as rocm_ops

    _, ops, x, dy = _layers(300, 8, k, 136, 72, torch.bfloat16, bias, save=False)
    calls, one = [], rocm_ops.scatter2scatter_rocm
    monkeypatch.setattr(rocm_ops, "scatter2scatter_rocm", lambda *a: calls.append(1) or one(*a))
    with _few_rows_limit(0) if large else contextlib.nullcontext():
        got = _step(ops, x, dy)
        assert len(calls) == 2 + again  # the down-projection, dX1
        ops.save_activations = True
        _same(got, _step(ops, x, dy))
