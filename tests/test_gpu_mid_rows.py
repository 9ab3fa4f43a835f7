"""The 128 x 256 tiles that the few-row entry points take beyond 24 (forward-type) and 40 (dW) rows per expert, at the edges of
their tiles, K steps and ranges, each against the CPU oracle and the 256 x 256 kernels on the same operands."""

import pytest
import torch

from oracle import moe as oracle

from .test_gpu_ops import _few_rows_limit, _tol
from .utils import nerr


pytestmark = pytest.mark.gpu

# rows per expert, K, N: one tile and one row more, 32- and 64-row blocks of the waves, empty experts, a K step and its tail, K ranges
# (few tiles, long K), one and several column tiles with clamped columns, more experts than lanes, and more than two chunks of them
CASES = [
    ([25], 8, 8),
    ([128, 129, 0, 32, 33, 127], 72, 264),
    ([64, 65, 0, 97], 64, 256),
    ([300, 0, 1], 200, 136),
    ([260] * 8, 1024, 512),
    ([90, 31], 4096, 256),
    ([258, 131], 8456, 136),
    ([40 + e for e in range(70)], 136, 24),
    ([e % 37 * 7 for e in range(140)], 192, 256),
]


def _both(fn, outs):
    """fn() with the 256 x 256 kernels and through the few-row entry points, all outputs poisoned in between"""
    res = []
    for limit in (0, 65535):
        for o in outs:
            o.fill_(float("nan"))
        with _few_rows_limit(limit):
            fn()
        torch.cuda.synchronize()
        res.append([o.clone() for o in outs])
    return zip(*res)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"E{len(c[0])}-M{sum(c[0])}-K{c[1]}-N{c[2]}")
def test_mid_rows_tiles(dtype, case):
    from xma.rocm import ops

    rows, K, N = case
    E, M = len(rows), sum(rows)
    assert M > 24 * E
    g = torch.Generator().manual_seed(M + K)
    se = torch.repeat_interleave(torch.arange(E), torch.tensor(rows))
    ss = torch.randperm(M, generator=g)
    offs = torch.tensor(rows).cumsum(0).cuda()
    idx = ss.cuda()
    wide = torch.randn(M, K + 16, generator=g).to(dtype)
    x = wide[:, 8 : 8 + K]  # rows further apart than they are long
    Wn = (torch.randn(E, N, K, generator=g) * K**-0.5).to(dtype)
    Wk = (torch.randn(E, K, N, generator=g) * K**-0.5).to(dtype)
    bias = torch.randn(E, N, generator=g).to(dtype)
    w = torch.rand(M, generator=g).to(dtype)
    z = torch.randn(M, 2 * N, generator=g).to(dtype)
    dy = torch.randn(M, N, generator=g).to(dtype)
    xd, Wnd, Wkd, bd, wd, zd, dyd = wide.cuda()[:, 8 : 8 + K], Wn.cuda(), Wk.cuda(), bias.cuda(), w.cuda(), z.cuda(), dy.cuda()
    out, h, dz, dW = (torch.empty(s, dtype=dtype, device="cuda") for s in ((M, N), (M, N // 2), (M, 2 * N), (E, N, K)))
    tol = _tol(dtype)

    def agree(fn, outs, want):
        for (tiles256, got), ref in zip(_both(fn, outs), want):
            assert torch.isfinite(got).all()
            assert nerr(got, ref) <= tol and nerr(got, tiles256) <= tol

    for x_grouped in (False, True):
        for y_grouped in (False, True):
            for scale in (None, w):
                sd = None if scale is None else wd
                args = (se, ss, 1, x_grouped, y_grouped)
                agree(lambda: ops.scatter2scatter_rocm(xd, Wnd.permute(0, 2, 1), idx, offs, out, sd, 1, x_grouped, y_grouped, bd), [out],
                      [oracle.scatter2scatter(x, Wn.permute(0, 2, 1), *args, scale, bias=bias)])
                agree(lambda: ops.scatter2scatter_rocm(xd, Wkd, idx, offs, out, sd, 1, x_grouped, y_grouped), [out],
                      [oracle.scatter2scatter(x, Wk, *args, scale)])
    if N % 16 == 0:
        want = oracle.scatter2scatter(x, Wn.permute(0, 2, 1), se, ss, 1, False, True, None, bias=bias)
        agree(lambda: ops.up_projection_swiglu_rocm(xd, Wnd.permute(0, 2, 1), idx, offs, out, h, 1, bd), [out, h],
              [want, oracle.swiglu_packed(want)])
    # SwiGLU backward, its second output, and the three forms of dW: agreement with the 256 x 256 kernels, which other tests hold
    # against the oracle
    def same(fn, outs):
        for tiles256, got in _both(fn, outs):
            assert torch.isfinite(got).all() and nerr(got, tiles256) <= tol

    same(lambda: ops.down_projection_dx_swiglu_rocm(xd, Wkd, idx, offs, zd, dz, wd, 1), [dz])
    same(lambda: ops.down_projection_dx_swiglu_scaled_act_rocm(xd, Wkd, idx, offs, zd, dz, out, wd, 1), [dz, out])
    for dy_fan, x_fan in ((0, 0), (1, 0), (0, 1)):
        same(lambda: ops.group_bwd_W_rocm(dyd, xd, idx, offs, dW.permute(0, 2, 1), None, dy_fan, x_fan), [dW])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", [c for c in CASES if c[2] % 16 == 0], ids=lambda c: f"E{len(c[0])}-M{sum(c[0])}-K{c[1]}-N{c[2]}")
def test_swiglu_of_transposed_weights(dtype, case):
    """SwiGLU with W stored as (K, N) and its backward with W stored as (N, K), with and without the second output (which the ops
    take in the other layout only)"""
    from xma.rocm import ops
    from xma.rocm.loader import check, get_library

    rows, K, N = case
    E, M = len(rows), sum(rows)
    g = torch.Generator().manual_seed(M + N)
    se = torch.repeat_interleave(torch.arange(E), torch.tensor(rows))
    ss = torch.randperm(M, generator=g)
    idx, offs = ss.cuda(), torch.tensor(rows).cumsum(0).cuda()
    x = torch.randn(M, K, generator=g).to(dtype)
    Wk = (torch.randn(E, K, N, generator=g) * K**-0.5).to(dtype)
    bias, w, z = (t.to(dtype) for t in (torch.randn(E, N, generator=g), torch.rand(M, generator=g), torch.randn(M, 2 * N, generator=g)))
    xd, Wkd, bd, wd, zd = x.cuda(), Wk.cuda(), bias.cuda(), w.cuda(), z.cuda()
    Wnd = Wkd.transpose(1, 2).contiguous()
    out, h, dz, dz2, act = (torch.empty(s, dtype=dtype, device="cuda") for s in ((M, N), (M, N // 2), (M, 2 * N), (M, 2 * N), (M, N)))
    tol = _tol(dtype)
    want = oracle.scatter2scatter(x, Wk, se, ss, 1, False, True, None, bias=bias)
    for (tiles256, got), ref in zip(_both(lambda: ops.up_projection_swiglu_rocm(xd, Wkd, idx, offs, out, h, 1, bd), [out, h]),
                                    (want, oracle.swiglu_packed(want))):
        assert torch.isfinite(got).all() and nerr(got, ref) <= tol and nerr(got, tiles256) <= tol
    z32 = z.float().requires_grad_()
    h32 = oracle.swiglu_packed(z32)
    h32.backward(oracle.scatter2scatter(x, Wk, se, ss, 1, False, True, w, compute_dtype=torch.float32).float())
    ((tiles256, got),) = _both(lambda: ops.down_projection_dx_swiglu_rocm(xd, Wnd.permute(0, 2, 1), idx, offs, zd, dz, wd, 1), [dz])
    assert torch.isfinite(got).all() and nerr(got, z32.grad) <= tol and nerr(got, tiles256) <= tol
    need = get_library().xma_rocm_scatter2scatter_few_rows_workspace_bytes(M, N, K, E, 0, ops.EPI_SWIGLU_BWD)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    check(get_library().xma_rocm_scatter2scatter_few_rows(
        xd.data_ptr(), K, Wnd.data_ptr(), N * K, K, 0, idx.data_ptr(), offs.data_ptr(), dz2.data_ptr(), 2 * N, zd.data_ptr(), 2 * N,
        act.data_ptr(), N, wd.data_ptr(), None, 0, M, N, K, E, 1, 0, 1, ops.EPI_SWIGLU_BWD, ops._code(xd), ws.data_ptr(), need, ops._stream(xd),
    ), "xma_rocm_scatter2scatter_few_rows")
    assert torch.equal(dz2, got) and nerr(act, h32.detach() * w.float()[ss][:, None]) <= tol


def test_rows_beyond_32_bit_offsets():
    """an operand that the 128 x 256 tiles cannot address goes through the small tile, uncut: the workspace is theirs"""
    from xma.rocm import ops

    E, M, K, N = 2, 52, 8192, 64
    far = torch.empty(M, (1 << 32) // (2 * M) // 8 * 8 + 8, dtype=torch.bfloat16, device="cuda")[:, :K]
    g = torch.Generator().manual_seed(4)
    x = torch.randn(M, K, generator=g).bfloat16()
    W = (torch.randn(E, N, K, generator=g) * K**-0.5).bfloat16()
    assert M > 24 * E and M * far.stride(0) * 2 >= 1 << 32 and ops._few_rows_workspace_bytes(M, N, K, E, 0, 0) < 16 * M * N * 4
    far.copy_(x)
    offs, idx = torch.tensor([30, M]).cuda(), torch.randperm(M, generator=g).cuda()
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    ops.scatter2scatter_rocm(far, W.cuda().permute(0, 2, 1), idx, offs, out, None, 1, False, True)
    rows = x[idx.cpu()].float()
    want = torch.cat([rows[:30] @ W[0].float().t(), rows[30:] @ W[1].float().t()])
    assert nerr(out, want) <= _tol(torch.bfloat16)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,N,K", [
    ((300, 0, 64, 65, 129, 200), 1288, 2056),  # 594 tiles, rows of dW off 64-byte boundaries
    ((0, 300, 63, 1, 128, 300), 1288, 2080),  # on them
    (tuple(7 * e % 150 * (e % 9 != 4) for e in range(69)), 520, 776),  # 1380 tiles, more experts than a wave has lanes
    (tuple(11 * e % 170 * (e % 7 != 2) for e in range(61)), 776, 800),  # 1708 tiles, ranked by their rows
], ids=lambda v: str(len(v)) if isinstance(v, tuple) else str(v))
def test_dw_walk(dtype, counts, N, K):
    """launches of more than 512 tiles: a workgroup goes on to a second and third one, whose first items it loads while the one before
    leaves through the ring's free place, also past experts without rows; every expert on its own against an fp32 product"""
    from xma.rocm import ops

    E, M = len(counts), sum(counts)
    tiles = E * -(-N // 128) * -(-K // 256)
    assert tiles > 512 and tiles % 8 and 640 * E >= M > (40 if tiles >= 1024 else 96) * E and 0 in counts
    g = torch.Generator(device="cuda").manual_seed(N + K)
    offs = torch.tensor(counts).cumsum(0).cuda()
    idx = torch.randperm(M, generator=g, device="cuda")
    x, dy = (torch.randn(M, n, generator=g, device="cuda").to(dtype) for n in (K, N))
    for dy_fan, x_fan in ((0, 0), (1, 0), (0, 1)):
        dW = torch.full((E, N, K), float("nan"), dtype=dtype, device="cuda")
        ops.group_bwd_W_rocm(dy, x, idx, offs, dW.permute(0, 2, 1), None, dy_fan, x_fan)
        gx, gdy = (x[idx] if x_fan else x), (dy[idx] if dy_fan else dy)
        row = 0
        for e, c in enumerate(counts):
            want = gdy[row : row + c].float().t() @ gx[row : row + c].float()
            err = (dW[e].float() - want).abs().max()
            assert err <= 2.0**-8 * want.abs().max(), (e, c)  # rounding to bf16: 2^-9 of the value; fp16 is closer
            row += c
