"""GPU parity of the MoE ops (grouped GEMMs, dW, group, combine) through the C ABI against the
op-level oracle.  Tolerance: max-abs-normalised error <= 1e-2 for bf16/fp16 results with fp32
accumulation (the bar of the north star), <= 2e-5 for the fp32 kernels; operands are bit-identical on both sides."""

import pytest
import torch

from oracle import moe as oracle
from tests.utils import nerr

pytestmark = pytest.mark.gpu

TOL = 1e-2
TOL_F32 = 2e-5  # fp32 kernels: fp32 operands and accumulators, only the summation order differs from the oracle's


def _tol(dtype):
    return TOL_F32 if dtype == torch.float32 else TOL


def _routing(T, E, k, seed, skew=0.0, empty=()):
    g = torch.Generator().manual_seed(seed)
    logits = torch.randn(T, E, generator=g) + skew * torch.randn(E, generator=g)
    for e in empty:
        logits[:, e] = -1e9
    sel = logits.topk(k, dim=-1).indices
    se, ss = sel.flatten().sort(stable=True)
    offs = torch.bincount(se, minlength=E).cumsum(0)
    return sel, se, ss, offs


class _few_rows_limit:
    """the number of rows up to which the ops take the few-token entry points, whatever the number of experts, set for the
    length of a with block (0: never)"""

    def __init__(self, limit):
        self.limit = limit

    def __enter__(self):
        from xma.rocm import ops

        self.saved = (ops.FEW_ROWS_MAX, ops.FEW_ROWS_PER_EXPERT)
        ops.FEW_ROWS_MAX, ops.FEW_ROWS_PER_EXPERT = self.limit, dict.fromkeys(ops.FEW_ROWS_PER_EXPERT, 1 << 30)

    def __exit__(self, *exc):
        from xma.rocm import ops

        ops.FEW_ROWS_MAX, ops.FEW_ROWS_PER_EXPERT = self.saved


def _limits(rows):
    """both code paths where the number of rows would pick the few-token one, else the only one there is"""
    from xma.rocm import ops

    return (0, ops.FEW_ROWS_MAX) if rows <= ops.FEW_ROWS_MAX else (ops.FEW_ROWS_MAX,)


CASES = [
    # T, E, k, K, N, skew, empty experts
    (7, 4, 2, 64, 64, 0.0, ()),
    (7, 8, 4, 128, 72, 0.0, ()),
    (300, 3, 2, 192, 320, 0.0, ()),
    (700, 8, 2, 256, 512, 1.5, (3,)),
    (1024, 2, 1, 64, 264, 0.0, ()),
    (513, 6, 4, 72, 40, 2.0, (0, 5)),
    (100, 2, 1, 96, 136, 0.0, ()),  # about 50 rows per expert: two of a wave's four row blocks are computed
    (300, 3, 2, 1096, 320, 0.0, ()),  # few tiles, long K (with a tail): tiles are split into K slices
    (400, 100, 3, 128, 264, 1.0, (7, 99)),  # more experts than lanes of a wave: the schedule is scanned through LDS
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("w_kn", [False, True])
@pytest.mark.parametrize("x_grouped,y_grouped", [(False, True), (True, False), (True, True), (False, False)])
def test_scatter2scatter(dtype, case, w_kn, x_grouped, y_grouped):
    from xma.layers.moe import rocm_implementation as R

    T, E, k, K, N, skew, empty = case
    print(f"case T={T} E={E} k={k} K={K} N={N} w_kn={w_kn} xg={x_grouped} yg={y_grouped} {dtype}", flush=True)
    sel, se, ss, offs = _routing(T, E, k, 0, skew, empty)
    g = torch.Generator().manual_seed(1)
    M = T * k
    X = torch.randn(M if x_grouped else T, K, generator=g).to(dtype)
    if w_kn:
        W = (torch.randn(E, K, N, generator=g) * 0.1).to(dtype)  # contiguous (E, K, N)
    else:
        W = (torch.randn(E, N, K, generator=g) * 0.1).to(dtype).permute(0, 2, 1)  # view of (E, N, K)
    scale = torch.rand(M, generator=g).to(dtype)
    for rs in (None, scale):
        want = oracle.scatter2scatter(X, W, se, ss, k, x_grouped, y_grouped, rs)
        Wd = W.cuda() if w_kn else W.permute(0, 2, 1).contiguous().cuda().permute(0, 2, 1)
        for limit in _limits(M):
            out = torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
            with _few_rows_limit(limit):
                R.scatter2scatter(X.cuda(), Wd, se.cuda(), ss.cuda(), out, k, x_grouped, y_grouped, offs.cuda(),
                                  None if rs is None else rs.cuda())
            torch.cuda.synchronize()
            assert torch.isfinite(out).all()
            assert nerr(out, want) <= _tol(dtype), limit


@pytest.mark.usefixtures("either_tile")
def test_scatter2scatter_launches_outside_the_persistent_kernel():
    """Three launches that the layer itself never makes and that take the one-workgroup-per-tile kernel instead of the
    persistent one: more experts than its schedule tables hold (E = 1100, most of them empty), a row scale that starts
    off a 4-byte boundary (the persistent kernel fetches the aligned dword around a 16-bit scale), and dy @ W (W as
    (K, N)) with the SwiGLU forward epilogue, reachable through the C ABI only."""
    from xma.layers.moe import rocm_implementation as R
    from xma.rocm.loader import get_library

    dtype = torch.bfloat16
    g = torch.Generator().manual_seed(31)
    # (1) E = 1100
    T, E, k, K, N = 700, 1100, 2, 136, 264
    sel, se, ss, offs = _routing(T, E, k, 5, skew=2.0)
    M = T * k
    X = torch.randn(T, K, generator=g).to(dtype)
    W = (torch.randn(E, N, K, generator=g) * 0.1).to(dtype)
    want = oracle.scatter2scatter(X, W.permute(0, 2, 1), se, ss, k, False, True, None)
    out = torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
    R.scatter2scatter(X.cuda(), W.cuda().permute(0, 2, 1), se.cuda(), ss.cuda(), out, k, False, True, offs.cuda(), None)
    torch.cuda.synchronize()
    assert torch.isfinite(out).all() and nerr(out, want) <= TOL
    # (2) a row scale at an odd element offset, grouped rows in, scattered rows out
    T, E, k, K, N = 300, 3, 2, 192, 320
    sel, se, ss, offs = _routing(T, E, k, 6)
    M = T * k
    X = torch.randn(M, K, generator=g).to(dtype)
    W = (torch.randn(E, N, K, generator=g) * 0.1).to(dtype)
    scale_buf = torch.rand(M + 1, generator=g).to(dtype)
    want = oracle.scatter2scatter(X, W.permute(0, 2, 1), se, ss, k, True, False, scale_buf[1:])
    sd = scale_buf.cuda()[1:]
    assert sd.data_ptr() % 4 == 2
    out = torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
    R.scatter2scatter(X.cuda(), W.cuda().permute(0, 2, 1), se.cuda(), ss.cuda(), out, k, True, False, offs.cuda(), sd)
    torch.cuda.synchronize()
    assert torch.isfinite(out).all() and nerr(out, want) <= TOL
    # (3) W[e] as (K, N) with the SwiGLU forward epilogue: z and h = swiglu_packed(z), straight through the C ABI
    lib = get_library()
    K, N = 200, 272
    X = torch.randn(T, K, generator=g).to(dtype)
    Wkn = (torch.randn(E, K, N, generator=g) * 0.1).to(dtype)
    want_z = oracle.scatter2scatter(X, Wkn, se, ss, k, False, True, None)
    want_h = oracle.swiglu_packed(want_z.float())
    Xd, Wd, ssd, offsd = X.cuda(), Wkn.cuda(), ss.cuda(), offs.cuda()
    z = torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
    h = torch.full((M, N // 2), float("nan"), dtype=dtype, device="cuda")
    rc = lib.xma_rocm_scatter2scatter(Xd.data_ptr(), K, Wd.data_ptr(), K * N, N, 1, ssd.data_ptr(), offsd.data_ptr(),
                                      z.data_ptr(), N, h.data_ptr(), N // 2, None, M, N, K, E, k, 0, 1, 1, 0, None, 0,
                                      torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert rc == 0, lib.xma_rocm_last_error()
    assert torch.isfinite(z).all() and torch.isfinite(h).all()
    assert nerr(z, want_z) <= TOL and nerr(h, want_h) <= TOL


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.usefixtures("either_tile")
def test_scatter2scatter_bias_and_expert_column_sums(dtype):
    """The experts' bias as the first term of the grouped GEMM's sums (plain store and SwiGLU epilogues, both weight
    layouts, with and without a row scale, a tile split along K), and its gradient, the per-expert column sums of grouped
    rows or of gathered and scaled rows; experts without rows give zero sums."""
    from xma.rocm import ops

    for T, E, k, K, N, skew, empty in [(300, 3, 2, 192, 320, 0.0, ()), (513, 6, 4, 72, 40, 2.0, (0, 5)), (300, 3, 2, 1096, 320, 0.0, ())]:
        print(f"bias case T={T} E={E} k={k} K={K} N={N} {dtype}", flush=True)
        sel, se, ss, offs = _routing(T, E, k, 3, skew, empty)
        g = torch.Generator().manual_seed(4)
        M = T * k
        X = torch.randn(T, K, generator=g).to(dtype)
        bias = torch.randn(E, N, generator=g).to(dtype)
        scale = torch.rand(M, generator=g).to(dtype)
        for w_kn in (False, True):
            W = (torch.randn(E, K, N, generator=g) * 0.1).to(dtype)
            Wd = W.cuda() if w_kn else W.permute(0, 2, 1).contiguous().cuda().permute(0, 2, 1)
            for rs in (None, scale):
                want = oracle.scatter2scatter(X, W, se, ss, k, False, True, rs, bias=bias)
                out = torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
                ops.scatter2scatter_rocm(X.cuda(), Wd, ss.cuda(), offs.cuda(), out, None if rs is None else rs.cuda(), k, False,
                                         True, bias.cuda())
                torch.cuda.synchronize()
                assert torch.isfinite(out).all() and nerr(out, want) <= _tol(dtype), (w_kn, rs is None)
            if not w_kn and N % 16 == 0:
                want_z = oracle.scatter2scatter(X, W, se, ss, k, False, True, None, bias=bias)
                z = torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
                h = torch.full((M, N // 2), float("nan"), dtype=dtype, device="cuda")
                ops.up_projection_swiglu_rocm(X.cuda(), Wd, ss.cuda(), offs.cuda(), z, h, k, bias.cuda())
                torch.cuda.synchronize()
                assert nerr(z, want_z) <= _tol(dtype) and nerr(h, oracle.swiglu_packed(want_z)) <= _tol(dtype)
        # column sums: grouped rows; gathered rows times a scale
        A = torch.randn(M, N, generator=g).to(dtype)
        counts = torch.bincount(se, minlength=E).tolist()
        want = torch.stack([a.float().sum(0) for a in A.split(counts)])
        got = torch.full((E, N), float("nan"), dtype=dtype, device="cuda")
        ops.expert_column_sums_rocm(A.cuda(), None, offs.cuda(), got, None, 1)
        B = torch.randn(T, N, generator=g).to(dtype)
        rows = B.float()[ss // k] * scale.float()[ss][:, None]
        want2 = torch.stack([a.sum(0) for a in rows.split(counts)])
        got2 = torch.full((E, N), float("nan"), dtype=dtype, device="cuda")
        ops.expert_column_sums_rocm(B.cuda(), ss.cuda(), offs.cuda(), got2, scale.cuda(), k)
        torch.cuda.synchronize()
        assert nerr(got, want) <= _tol(dtype) and nerr(got2, want2) <= _tol(dtype)
        for e in empty:
            assert torch.count_nonzero(got[e]) == 0 and torch.count_nonzero(got2[e]) == 0


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("counts,N", [((0, 1, 127, 128, 129, 700), 130), ((15, 17, 63, 0, 64, 65), 258), ((3,) * 511 + (40,), 256), ((3,) * 512, 254)])
def test_expert_column_sums_block_sizes(dtype, counts, N):
    """both workgroup sizes (below and from 1024 workgroups on), experts around the rows of one step, a partial column block"""
    from xma.rocm import ops

    print(f"column sums E={len(counts)} N={N} {dtype}", flush=True)
    A = torch.randn(sum(counts), N, generator=torch.Generator().manual_seed(5)).to(dtype)
    got = torch.full((len(counts), N), float("nan"), dtype=dtype, device="cuda")
    ops.expert_column_sums_rocm(A.cuda(), None, torch.tensor(counts).cumsum(0).cuda(), got, None, 1)
    want = torch.stack([a.double().sum(0) for a in A.split(counts)])
    assert nerr(got, want) <= _tol(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("counts,N", [((0, 1, 255, 256, 257, 1025), 136), ((15, 17, 63, 0, 64, 65), 264), ((4,) * 511 + (40,), 256), ((5, 3), 8)])
def test_expert_column_sums_whole_pieces(dtype, counts, N):
    """rows of whole 16-byte pieces: grouped, further apart than they are long, and gathered and scaled; a start off 16 bytes takes the
    other kernel.  Against 64 bits: fp32 sums of the rows and one rounding"""
    from xma.rocm import ops

    print(f"column sums of pieces E={len(counts)} N={N} {dtype}", flush=True)
    _, _, ss, offs = _routing_with_counts(counts, 2, 3)
    g, M = torch.Generator().manual_seed(5), sum(counts)
    wide, scale = torch.randn(M, N + 24, generator=g).to(dtype).cuda(), torch.rand(M, generator=g).to(dtype).cuda()
    ss, offs = ss.cuda(), offs.cuda()
    unit, smallest = {torch.bfloat16: (2.0**-8, 0.0), torch.float16: (2.0**-11, 2.0**-24), torch.float32: (2.0**-24, 0.0)}[dtype]
    for A in (wide[:, :N].contiguous(), wide[:, 16 : 16 + N], wide[:, 4 : 4 + N]):
        for gathered in (False, True):
            got = torch.full((len(counts), N), float("nan"), dtype=dtype, device="cuda")
            src = A[: M // 2] if gathered else A
            ops.expert_column_sums_rocm(src, ss if gathered else None, offs, got, scale if gathered else None, 2 if gathered else 1)
            rows = src.double()[ss // 2] * scale.double()[ss][:, None] if gathered else src.double()
            want = torch.stack([a.sum(0) for a in rows.split(counts)])
            size = torch.stack([a.abs().sum(0) for a in rows.split(counts)])
            assert ((got.double() - want).abs() <= unit * want.abs() + (max(counts) + 1) * 2.0**-24 * size + smallest).all()


@pytest.mark.parametrize("E,N", [(3, 72), (64, 1024)])  # small and large tiles
@pytest.mark.parametrize("K", [8, 16, 24, 32, 40, 72, 136])
def test_fp32_k_steps(E, N, K):
    """fp32 GEMMs whose K, and for dW whose rows per expert (none, one, around the steps of 16 and 32), make none to several K steps with and
    without a remainder, rows gathered and grouped: against 64 bits, fp32 sums of K (rows) products"""
    from xma.rocm import ops

    print(f"fp32 K steps E={E} N={N} K={K}", flush=True)
    edges = (0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 97)
    counts = [90 + (i % 5) for i in range(E)] if E == 64 else [33, 0, 65]
    if E == 64:
        counts[: len(edges)] = edges
        counts[20] += 90 * 64 - sum(counts)
    counts[-1] += sum(counts) % 2
    _, _, ss, offs = _routing_with_counts(tuple(counts), 2, 7)
    g, M = torch.Generator().manual_seed(9), sum(counts)
    X, Xt, DY, W, w = (torch.randn(*n, generator=g).cuda() for n in ((M, K), (M // 2, K), (M, N), (E, N, K), (M,)))
    ss, offs, nan = ss.cuda(), offs.cuda(), lambda *n: torch.full(n, float("nan"), device="cuda")
    starts = [0, *offs.tolist()]
    for gathered in (False, True):
        rows = Xt.double()[ss // 2] if gathered else X.double()
        src, fan = (Xt, 2) if gathered else (X, 1)
        for weight in (W.permute(0, 2, 1), W.permute(0, 2, 1).contiguous()):
            out, want, size = nan(M, N), torch.empty(M, N, dtype=torch.float64, device="cuda"), torch.empty(M, N, dtype=torch.float64, device="cuda")
            ops.scatter2scatter_rocm(src, weight, ss, offs, out, None, fan, not gathered, True)
            for e in range(E):
                part = slice(starts[e], starts[e + 1])
                want[part], size[part] = rows[part] @ W[e].double().t(), rows[part].abs() @ W[e].double().t().abs()
            assert ((out.double() - want).abs() <= (K + 1) * 2.0**-24 * size).all()
        for scale in (None, w):
            dw = nan(E, N, K)
            ops.group_bwd_W_rocm(DY, src, ss, offs, dw.permute(0, 2, 1), scale, 0, fan if gathered else 0)
            dy = DY.double() if scale is None else (DY * w[ss][:, None]).double()  # rounded to fp32, as the loader does
            for e in range(E):
                part = slice(starts[e], starts[e + 1])
                want, size = dy[part].t() @ rows[part], dy[part].t().abs() @ rows[part].abs()
                assert ((dw[e].double() - want).abs() <= (counts[e] + 1) * 2.0**-24 * size).all(), e


def _routing_with_counts(counts, k, seed):
    """a routing whose experts own exactly `counts` rows (sum divisible by k): the slots are dealt out at random"""
    g = torch.Generator().manual_seed(seed)
    E, M = len(counts), sum(counts)
    assert M % k == 0
    flat = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(M, generator=g)]
    sel = flat.view(M // k, k)
    se, ss = flat.sort(stable=True)
    offs = torch.bincount(se, minlength=E).cumsum(0)
    assert torch.bincount(se, minlength=E).tolist() == list(counts)
    return sel, se, ss, offs


# rows per expert around the 32-row blocks and 256-row tiles of the kernels (an empty expert, single rows, one row more or
# less than a block, a tile and two tiles), with K = 4 or 6 steps of 64 (complete and with a tail) and one odd step count:
# tiles of more than 192 rows and an even number of at least four K steps fetch the next tile's operands inside their
# last K step, all others behind it
ROW_COUNT_CASES = [
    # counts, k, K, N
    ((1, 31, 33, 65, 129, 257, 0, 512), 2, 256, 264),
    ((257, 1, 193, 192, 511, 513, 224, 3), 2, 232, 520),
    ((300, 260, 1, 255), 1, 384, 72),
    ((256, 200, 700, 4), 4, 328, 512),
    ((193, 250, 256, 257), 1, 320, 264),  # five K steps: odd
    ((3333, 259, 4000), 2, 256, 520),  # 14 and 16 row tiles: the tiles of such an expert are walked in bands of row tiles
    ((3100, 7), 1, 64, 776),  # 13 row tiles in bands of 5, 5 and 3
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("case", ROW_COUNT_CASES)
@pytest.mark.parametrize("w_kn", [False, True])
@pytest.mark.usefixtures("either_tile")
def test_scatter2scatter_expert_row_counts(dtype, case, w_kn):
    from xma.layers.moe import rocm_implementation as R

    counts, k, K, N = case
    print(f"case counts={counts} k={k} K={K} N={N} w_kn={w_kn} {dtype}", flush=True)
    sel, se, ss, offs = _routing_with_counts(counts, k, 11)
    E, M = len(counts), sum(counts)
    T = M // k
    g = torch.Generator().manual_seed(12)
    scale = torch.rand(M, generator=g).to(dtype)
    if w_kn:
        W = (torch.randn(E, K, N, generator=g) * 0.1).to(dtype)
        Wd = W.cuda()
    else:
        W = (torch.randn(E, N, K, generator=g) * 0.1).to(dtype).permute(0, 2, 1)
        Wd = W.permute(0, 2, 1).contiguous().cuda().permute(0, 2, 1)
    for x_grouped, y_grouped, rs in [(False, True, None), (True, False, scale), (True, True, None), (False, False, scale)]:
        X = torch.randn(M if x_grouped else T, K, generator=g).to(dtype)
        want = oracle.scatter2scatter(X, W, se, ss, k, x_grouped, y_grouped, rs)
        out = torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
        R.scatter2scatter(X.cuda(), Wd, se.cuda(), ss.cuda(), out, k, x_grouped, y_grouped, offs.cuda(),
                          None if rs is None else rs.cuda())
        torch.cuda.synchronize()
        assert torch.isfinite(out).all()
        assert nerr(out, want) <= _tol(dtype)
        # every row against its own magnitude: a wrong row of a small expert does not hide behind the large ones
        row_err = (out.cpu().float() - want.float()).abs().amax(dim=1) / want.float().abs().amax(dim=1).clamp_min(1e-6)
        assert row_err.max() <= 4 * _tol(dtype), int(row_err.argmax())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("case", ROW_COUNT_CASES)
def test_group_bwd_W_expert_row_counts(dtype, case):
    from xma.rocm import ops

    counts, k, K, N = case
    print(f"case counts={counts} k={k} K={K} N={N} {dtype}", flush=True)
    sel, se, ss, offs = _routing_with_counts(counts, k, 13)
    E, M = len(counts), sum(counts)
    T = M // k
    g = torch.Generator().manual_seed(14)
    x_tok = torch.randn(T, K, generator=g).to(dtype)
    dy_grp = torch.randn(M, N, generator=g).to(dtype)
    x_grp = torch.randn(M, K, generator=g).to(dtype)
    for X, x_fan, want in [(x_grp, 0, oracle.group_bwd_W(dy_grp, x_grp, offs, E)),
                           (x_tok, k, oracle.group_bwd_W(dy_grp, oracle.group(x_tok, ss, None, k), offs, E))]:
        for limit in _limits(M):
            DW = torch.full((E, N, K), float("nan"), dtype=dtype, device="cuda").permute(0, 2, 1)
            with _few_rows_limit(limit):
                ops.group_bwd_W_rocm(dy_grp.cuda(), X.cuda(), ss.cuda(), offs.cuda(), DW, None, 0, x_fan)
            torch.cuda.synchronize()
            assert torch.isfinite(DW).all()
            for e in range(E):  # every expert's slice against its own magnitude
                if counts[e] == 0:
                    assert (DW[e] == 0).all()
                else:
                    assert nerr(DW[e], want[e]) <= _tol(dtype), (e, limit)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("case", CASES)
def test_group_bwd_W(dtype, case):
    from xma.rocm import ops

    T, E, k, K, N, skew, empty = case
    print(f"case T={T} E={E} k={k} K={K} N={N} {dtype}", flush=True)
    sel, se, ss, offs = _routing(T, E, k, 2, skew, empty)
    g = torch.Generator().manual_seed(3)
    M = T * k
    x_tok = torch.randn(T, K, generator=g).to(dtype)
    dy_tok = torch.randn(T, N, generator=g).to(dtype)
    dy_grp = torch.randn(M, N, generator=g).to(dtype)
    x_grp = torch.randn(M, K, generator=g).to(dtype)
    scale = torch.rand(M, generator=g).to(dtype)

    def run(DY, X, dy_scale, dy_fan, x_fan):
        DW = torch.full((E, N, K), float("nan"), dtype=dtype, device="cuda").permute(0, 2, 1)
        ops.group_bwd_W_rocm(DY.cuda(), X.cuda(), ss.cuda(), offs.cuda(), DW, None if dy_scale is None else dy_scale.cuda(),
                             dy_fan, x_fan)
        torch.cuda.synchronize()
        assert torch.isfinite(DW).all()
        return DW

    for limit in _limits(M):
        with _few_rows_limit(limit):
            # both grouped (the reference op), x gathered (dW1), dy gathered and scaled (dW2)
            want = oracle.group_bwd_W(dy_grp, x_grp, offs, E)
            assert nerr(run(dy_grp, x_grp, None, 0, 0), want) <= _tol(dtype)
            want = oracle.group_bwd_W(dy_grp, oracle.group(x_tok, ss, None, k), offs, E)
            assert nerr(run(dy_grp, x_tok, None, 0, k), want) <= _tol(dtype)
            want = oracle.group_bwd_W(oracle.group(dy_tok, ss, scale, k), x_grp, offs, E)
            assert nerr(run(dy_tok, x_grp, scale, k, 0), want) <= _tol(dtype)
            # experts without rows get an all-zero slice
            got = run(dy_grp, x_grp, None, 0, 0)
            for e in empty:
                assert (got[e] == 0).all()


FEW_ROWS_CASES = [
    # T, E, k, H, I, empty experts
    (7, 8, 2, 264, 136, ()),
    (3, 128, 8, 576, 256, ()),  # more experts than rows
    (16, 4, 4, 2048, 72, (2,)),  # about twenty rows per expert: several passes of 4 or 8 rows over the weights
    (1, 8, 1, 64, 8, ()),
    (9, 5, 3, 4104, 24, (0, 4)),  # a row of W as (N, K) is 513 pieces of 16 bytes: two passes of a wave and one lane more
    (7, 8, 2, 512, 8192, ()),  # long K for the down-projection and dX1: both cut into ranges of K
    (5, 2, 2, 64, 3200, ()),  # down-projection: 25 K steps in 6 ranges of 5, of which only 5 hold a step
    (5, 8, 2, 2056, 40, (3,)),  # one or two rows per expert and rows of W longer than 4 KB: the vector kernel for the up-projection
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", FEW_ROWS_CASES)
def test_forward_type_gemms_few_rows(dtype, case):
    """The six operand forms of the layer's forward-type GEMMs through the kernels written for a handful of rows (weights
    streamed once per 32 rows of an expert; vector FMAs or a small MFMA tile, sums through a workspace and one small
    epilogue kernel where K is cut), each against the oracle and against the 256 x 256 kernels on the same operands: up-projection + SwiGLU with a bias (z and h), up-projection with a plain store,
    down-projection with a bias, a row scale and scattered rows, dX1 (dz @ W1, scattered), dX2 + SwiGLU backward with and
    without the scaled activations."""
    from xma.rocm import ops

    T, E, k, H, I, empty = case
    print(f"case T={T} E={E} k={k} H={H} I={I} {dtype}", flush=True)
    sel, se, ss, offs = _routing(T, E, k, 41, 0.0, empty)
    M = T * k
    assert M <= ops.FEW_ROWS_MAX
    g = torch.Generator().manual_seed(42)
    x = torch.randn(T, H, generator=g).to(dtype)
    W1 = (torch.randn(E, 2 * I, H, generator=g) * 0.05).to(dtype)  # c_fc.weight (E, out, in)
    W2 = (torch.randn(E, H, I, generator=g) * 0.05).to(dtype)  # c_proj.weight
    b1 = torch.randn(E, 2 * I, generator=g).to(dtype)
    b2 = torch.randn(E, H, generator=g).to(dtype)
    w = torch.rand(M, generator=g).to(dtype)
    dy = torch.randn(T, H, generator=g).to(dtype)
    dzg = torch.randn(M, 2 * I, generator=g).to(dtype)
    xd, W1d, W2d, b1d, b2d, wd, dyd, dzd, ssd, offsd = (t.cuda() for t in (x, W1, W2, b1, b2, w, dy, dzg, ss, offs))
    tol = _tol(dtype)

    def both(fn):
        """fn() -> tuple of device outputs; run with the MFMA kernels and with the few-row kernels"""
        res = {}
        for limit in (0, ops.FEW_ROWS_MAX):
            with _few_rows_limit(limit):
                res[limit] = fn()
            torch.cuda.synchronize()
        return res[ops.FEW_ROWS_MAX], res[0]

    def new(*shape):
        return torch.full(shape, float("nan"), dtype=dtype, device="cuda")

    # up-projection + SwiGLU, bias
    def up():
        z, h = new(M, 2 * I), new(M, I)
        ops.up_projection_swiglu_rocm(xd, W1d.permute(0, 2, 1), ssd, offsd, z, h, k, b1d)
        return z, h

    want_z = oracle.scatter2scatter(x, W1.permute(0, 2, 1), se, ss, k, False, True, None, bias=b1)
    (z_f, h_f), (z_m, h_m) = both(up)
    assert torch.isfinite(z_f).all() and torch.isfinite(h_f).all()
    assert nerr(z_f, want_z) <= tol and nerr(z_f, z_m) <= tol
    assert nerr(h_f, oracle.swiglu_packed(want_z)) <= tol and nerr(h_f, h_m) <= tol

    # up-projection, plain store, no bias
    def up_store():
        z = new(M, 2 * I)
        ops.scatter2scatter_rocm(xd, W1d.permute(0, 2, 1), ssd, offsd, z, None, k, False, True)
        return (z,)

    (z_f,), (z_m,) = both(up_store)
    assert nerr(z_f, oracle.scatter2scatter(x, W1.permute(0, 2, 1), se, ss, k, False, True, None)) <= tol and nerr(z_f, z_m) <= tol

    # down-projection: grouped rows in, scattered rows out, bias and row scale
    hg = torch.randn(M, I, generator=g).to(dtype)
    hgd = hg.cuda()

    def down():
        out = new(M, H)
        ops.scatter2scatter_rocm(hgd, W2d.permute(0, 2, 1), ssd, offsd, out, wd, 1, True, False, b2d)
        return (out,)

    (o_f,), (o_m,) = both(down)
    want = oracle.scatter2scatter(hg, W2.permute(0, 2, 1), se, ss, 1, True, False, w, bias=b2)
    assert torch.isfinite(o_f).all() and nerr(o_f, want) <= tol and nerr(o_f, o_m) <= tol

    # dX1: dz @ W1 (W as (K, N) = the parameter as stored), scattered rows out
    def dx1():
        out = new(M, H)
        ops.scatter2scatter_rocm(dzd, W1d, ssd, offsd, out, None, 1, True, False)
        return (out,)

    (o_f,), (o_m,) = both(dx1)
    want = oracle.scatter2scatter(dzg, W1, se, ss, 1, True, False, None)
    assert torch.isfinite(o_f).all() and nerr(o_f, want) <= tol and nerr(o_f, o_m) <= tol

    # dX2 + SwiGLU backward, without and with the scaled activations
    zg = torch.randn(M, 2 * I, generator=g).to(dtype)
    zgd = zg.cuda()

    def dx2():
        dz = new(M, 2 * I)
        ops.down_projection_dx_swiglu_rocm(dyd, W2d, ssd, offsd, zgd, dz, wd, k)
        return (dz,)

    def dx2_act():
        dz, act = new(M, 2 * I), new(M, I)
        ops.down_projection_dx_swiglu_scaled_act_rocm(dyd, W2d, ssd, offsd, zgd, dz, act, wd, k)
        return dz, act

    z32 = zg.float().requires_grad_()
    h32 = oracle.swiglu_packed(z32)
    dh = torch.stack([(dy.float()[ss[n] // k] * w.float()[ss[n]]) @ W2.float()[se[n]] for n in range(M)])
    h32.backward(dh)
    (dz_f,), (dz_m,) = both(dx2)
    assert torch.isfinite(dz_f).all() and nerr(dz_f, z32.grad) <= tol and nerr(dz_f, dz_m) <= tol
    (dz_a, act_f), (_, act_m) = both(dx2_act)
    assert torch.equal(dz_a, dz_f)
    assert nerr(act_f, h32.detach() * w.float()[ss][:, None]) <= tol and nerr(act_f, act_m) <= tol


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", [(7, 8, 2, 264, 136, ()), (3, 128, 8, 576, 512, ()), (16, 4, 4, 2048, 72, (2,)), (1, 8, 1, 64, 8, ()),
                                  (9, 5, 3, 4104, 24, (0, 4)), (100, 3, 2, 200, 328, ())])
def test_group_bwd_W_few_rows(dtype, case):
    """The weight gradient written for a handful of rows (a 128 x 128 tile of dW per workgroup, the expert's rows as the K
    dimension of the MFMAs, 32 at a time, streamed stores) against the oracle and against the 256 x 256 kernel on the same
    operands: every operand form of the layer, tiles partly outside dW in both directions, experts without rows (zeros),
    more experts than rows, about 67 rows per expert (two full passes and a partial one)."""
    from xma.rocm import ops

    T, E, k, K, N, empty = case
    print(f"case T={T} E={E} k={k} K={K} N={N} {dtype}", flush=True)
    sel, se, ss, offs = _routing(T, E, k, 21, 0.0, empty)
    M = T * k
    assert M <= ops.FEW_ROWS_MAX
    g = torch.Generator().manual_seed(22)
    x_tok = torch.randn(T, K, generator=g).to(dtype)
    dy_tok = torch.randn(T, N, generator=g).to(dtype)
    dy_grp = torch.randn(M, N, generator=g).to(dtype)
    x_grp = torch.randn(M, K, generator=g).to(dtype)
    scale = torch.rand(M, generator=g).to(dtype)
    forms = [(dy_grp, x_grp, None, 0, 0, oracle.group_bwd_W(dy_grp, x_grp, offs, E)),
             (dy_grp, x_tok, None, 0, k, oracle.group_bwd_W(dy_grp, oracle.group(x_tok, ss, None, k), offs, E)),
             (dy_tok, x_grp, scale, k, 0, oracle.group_bwd_W(oracle.group(dy_tok, ss, scale, k), x_grp, offs, E)),
             (dy_tok, x_grp, None, k, 0, oracle.group_bwd_W(oracle.group(dy_tok, ss, None, k), x_grp, offs, E))]
    counts = torch.bincount(se, minlength=E)
    for DY, X, sc, dy_fan, x_fan, want in forms:
        got = {}
        for limit in (0, ops.FEW_ROWS_MAX):
            DW = torch.full((E, N, K), float("nan"), dtype=dtype, device="cuda").permute(0, 2, 1)
            with _few_rows_limit(limit):
                ops.group_bwd_W_rocm(DY.cuda(), X.cuda(), ss.cuda(), offs.cuda(), DW, None if sc is None else sc.cuda(), dy_fan, x_fan)
            torch.cuda.synchronize()
            assert torch.isfinite(DW).all()
            got[limit] = DW
        few, mfma = got[ops.FEW_ROWS_MAX], got[0]
        assert nerr(few, want) <= _tol(dtype)
        assert nerr(few, mfma) <= _tol(dtype)
        for e in range(E):
            if counts[e] == 0:
                assert (few[e] == 0).all()
            else:
                assert nerr(few[e], want[e]) <= _tol(dtype), e


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_group_and_combine(dtype):
    from xma.layers.moe import rocm_implementation as R
    from xma.rocm import ops

    g = torch.Generator().manual_seed(5)
    for T, k, H in [(7, 2, 64), (33, 4, 136), (1000, 8, 2048), (513, 1, 72)]:
        E = 8
        sel, se, ss, offs = _routing(T, E, k, 6)
        A = torch.randn(T, H, generator=g).to(dtype)
        coeff = torch.rand(T * k, generator=g).to(dtype)
        for c in (None, coeff):
            out = torch.empty(T * k, H, dtype=dtype, device="cuda")
            R.group(A.cuda(), ss.cuda(), out, None if c is None else c.cuda(), k)
            assert torch.equal(out.cpu(), oracle.group(A, ss, c, k))  # one rounding of an fp32 product: exact match
        eo = torch.randn(T * k, H, generator=g).to(dtype)
        w = torch.rand(T, k, generator=g).to(dtype)
        dy = torch.randn(T, H, generator=g).to(dtype)
        for ww in (None, w):
            y = torch.empty(T, H, dtype=dtype, device="cuda")
            ops.combine_rocm(eo.cuda(), None if ww is None else ww.cuda(), y, k)
            assert nerr(y, oracle.combine(eo, ww, k)) <= _tol(dtype)
        d_w = torch.empty(T, k, dtype=dtype, device="cuda")
        ops.combine_bwd_rocm(eo.cuda(), dy.cuda(), d_w)
        assert nerr(d_w, oracle.combine_bwd(eo, dy, k)) <= _tol(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_swiglu_packed_standalone(dtype):
    from xma import KernelBackend
    from xma.functional import swiglu_packed

    g = torch.Generator().manual_seed(7)
    for rows, cols in [(1, 8), (7, 64), (300, 1408), (65, 4096)]:
        x = (torch.randn(rows, 2 * cols, generator=g) * 2).to(dtype)
        dy = torch.randn(rows, cols, generator=g).to(dtype)
        xd = x.cuda().requires_grad_()
        y = swiglu_packed(xd, kernel_backend=KernelBackend.rocm)
        y.backward(dy.cuda())
        assert nerr(y, oracle.swiglu_packed(x.float())) <= _tol(dtype)
        dg, du = oracle.swiglu_backward(x[..., 0::2].float(), x[..., 1::2].float(), dy.float())
        want = torch.stack([dg, du], dim=-1).flatten(-2)
        assert nerr(xd.grad, want) <= _tol(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,cols", [(1, 1024), (1, 2048), (1, 2056), (3, 1000), (33, 1003), (11003, 4104)])
def test_swiglu_packed_pieces(dtype, rows, cols):
    """Edges of the 16-byte kernels (a workgroup takes 2048 outputs; columns that no 16-byte piece divides; a launch above 256
    MB, non-temporal): bit-identical to the same rows one by one or in parts, and the first rows against the oracle."""
    from xma import KernelBackend
    from xma.functional import swiglu_packed

    print(f"swiglu_packed {rows}x{cols} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(rows + cols)
    x = torch.randn(rows, 2 * cols, generator=g, device="cuda").to(dtype).requires_grad_()
    dy = torch.randn(rows, cols, generator=g, device="cuda").to(dtype)
    y = swiglu_packed(x, kernel_backend=KernelBackend.rocm)
    y.backward(dy)
    for part in torch.arange(rows).chunk(3):
        lo, hi = int(part[0]), int(part[-1]) + 1
        xp = x.detach()[lo:hi].clone().requires_grad_()
        yp = swiglu_packed(xp, kernel_backend=KernelBackend.rocm)
        yp.backward(dy[lo:hi].clone())
        assert torch.equal(yp, y[lo:hi]) and torch.equal(xp.grad, x.grad[lo:hi])
    n = min(rows, 40)
    x32, dy32 = x.detach()[:n].float().cpu(), dy[:n].float().cpu()
    assert nerr(y[:n], oracle.swiglu_packed(x32)) <= _tol(dtype)
    dg, du = oracle.swiglu_backward(x32[..., 0::2], x32[..., 1::2], dy32)
    assert nerr(x.grad[:n], torch.stack([dg, du], dim=-1).flatten(-2)) <= _tol(dtype)


def _2d_sizes():
    """the reference's 2-D size rule (tests/utils.py:31-42: squares 2^i + j, and ragged sizes around 3000), thinned so
    that the CPU oracle stays within seconds"""
    import random

    rng = random.Random(0)
    sizes = [(2**i + j, 2**i + j) for i in range(11) for j in (0, 1, 3, 7, 9)]
    ragged = [(3000 + rng.randint(-1000, 1000), 3000 + rng.randint(-1000, 1000)) for _ in range(50)]
    return sizes + ragged[:8]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_swiglu_two_operands(dtype):
    """swiglu(gate, up) on separate operands, forward and backward, over the reference's 2-D size grid
    (tests/functional/swiglu_test.py:62-95: integer-valued inputs in [-8, 8), fp32 atol 7e-5 / 4.6e-5) - odd widths,
    widths below one 16-byte access, rows that are not 16-byte aligned - against the oracle's closed forms."""
    from xma import KernelBackend
    from xma.functional import swiglu

    g = torch.Generator().manual_seed(11)
    for rows, cols in _2d_sizes():
        print(f"swiglu case {rows}x{cols} {dtype}", flush=True)
        gate = torch.randint(-8, 8, (rows, cols), generator=g).to(dtype)
        up = torch.randint(-8, 8, (rows, cols), generator=g).to(dtype)
        dy = torch.randn(rows, cols, generator=g).to(dtype)
        gd, ud = gate.cuda().requires_grad_(), up.cuda().requires_grad_()
        y = swiglu(gd, ud, kernel_backend=KernelBackend.rocm)
        y.backward(dy.cuda())
        want = oracle.swiglu(gate.float(), up.float())
        dg, du = oracle.swiglu_backward(gate.float(), up.float(), dy.float())
        assert y.dtype == dtype and y.shape == (rows, cols)
        assert nerr(y, want) <= _tol(dtype), (rows, cols)
        assert nerr(gd.grad, dg) <= _tol(dtype) and nerr(ud.grad, du) <= _tol(dtype), (rows, cols)
        if dtype == torch.float32:
            assert (y.cpu() - want).abs().max() <= 7e-5
            assert (gd.grad.cpu() - dg).abs().max() <= 4.6e-5 * dy.abs().max() * 4


def test_swiglu_views_and_shapes():
    """3-D inputs, operands that are column slices of one wider tensor (row pitch larger than the width, starts not
    16-byte aligned), empty input; and the packed form at widths that are not multiples of 8."""
    from xma import KernelBackend
    from xma.functional import swiglu, swiglu_packed

    g = torch.Generator().manual_seed(12)
    for dtype in (torch.bfloat16, torch.float32):
        x = (torch.randn(3, 37, 2 * 203, generator=g) * 2).to(dtype)
        xd = x.cuda()
        for lo in (0, 1, 8):  # chunk-style halves of one tensor; lo shifts the alignment of the row starts
            gate, up = x[..., lo:203], x[..., 203 + lo :]
            y = swiglu(xd[..., lo:203], xd[..., 203 + lo :], kernel_backend=KernelBackend.rocm)
            assert y.shape == gate.shape
            assert nerr(y, oracle.swiglu(gate.float(), up.float())) <= _tol(dtype)
        for cols in (1, 3, 12, 203, 1001):
            xp = (torch.randn(5, 29, 2 * cols, generator=g) * 2).to(dtype)
            dy = torch.randn(5, 29, cols, generator=g).to(dtype)
            xpd = xp.cuda().requires_grad_()
            y = swiglu_packed(xpd, kernel_backend=KernelBackend.rocm)
            y.backward(dy.cuda())
            assert nerr(y, oracle.swiglu_packed(xp.float())) <= _tol(dtype), cols
            dg, du = oracle.swiglu_backward(xp[..., 0::2].float(), xp[..., 1::2].float(), dy.float())
            assert nerr(xpd.grad, torch.stack([dg, du], dim=-1).flatten(-2)) <= _tol(dtype), cols
        empty = torch.empty(0, 16, dtype=dtype, device="cuda")
        assert swiglu(empty, empty, kernel_backend=KernelBackend.rocm).shape == (0, 16)


def test_swiglu_broadcast_operands_and_gradients():
    """Operands and upstream gradients whose rows overlap in memory: the gradient autograd hands back for ``y.sum(0)``
    has strides (0, 1), an ``expand``-ed operand too.  The rocm path copies them (the kernels want rows that do not
    overlap); results against the oracle's closed forms."""
    from xma import KernelBackend
    from xma.functional import swiglu, swiglu_packed

    g = torch.Generator().manual_seed(13)
    for dtype in (torch.bfloat16, torch.float32):
        rows, cols = 37, 203
        gate = (torch.randn(rows, cols, generator=g) * 2).to(dtype)
        up = (torch.randn(rows, cols, generator=g) * 2).to(dtype)
        v = torch.randn(cols, generator=g).to(dtype)
        gd, ud, vd = gate.cuda().requires_grad_(), up.cuda().requires_grad_(), v.cuda()
        (swiglu(gd, ud, kernel_backend=KernelBackend.rocm).sum(0) * vd).sum().backward()
        dy = v.float().expand(rows, cols)  # what the sum over the rows hands back, up to the rounding of y.sum(0)
        dg, du = oracle.swiglu_backward(gate.float(), up.float(), dy)
        assert nerr(gd.grad, dg) <= _tol(dtype) and nerr(ud.grad, du) <= _tol(dtype)
        # one row of `up` for all rows of `gate`, forward and backward
        u1 = (torch.randn(1, cols, generator=g) * 2).to(dtype)
        gd, u1d = gate.cuda().requires_grad_(), u1.cuda().requires_grad_()
        y = swiglu(gd, u1d.expand(rows, cols), kernel_backend=KernelBackend.rocm)
        y.backward(torch.ones_like(y))
        assert nerr(y, oracle.swiglu(gate.float(), u1.float().expand(rows, cols))) <= _tol(dtype)
        dg, du = oracle.swiglu_backward(gate.float(), u1.float().expand(rows, cols), torch.ones(rows, cols))
        assert nerr(gd.grad, dg) <= _tol(dtype) and nerr(u1d.grad, du.sum(0, keepdim=True)) <= 2 * _tol(dtype)
        # the packed form with the same kind of gradient
        xp = (torch.randn(rows, 2 * cols, generator=g) * 2).to(dtype)
        xpd = xp.cuda().requires_grad_()
        (swiglu_packed(xpd, kernel_backend=KernelBackend.rocm).sum(0) * vd).sum().backward()
        dg, du = oracle.swiglu_backward(xp[..., 0::2].float(), xp[..., 1::2].float(), dy)
        assert nerr(xpd.grad, torch.stack([dg, du], dim=-1).flatten(-2)) <= _tol(dtype)


SCALED_ACT_CASES = [
    # counts, k, H (= K of dX2), I (= N)
    ((1, 31, 33, 65, 129, 257, 0, 512), 2, 256, 264),
    ((256, 200, 700, 4), 4, 328, 512),
    ((300, 260, 1, 255), 1, 1096, 72),  # few tiles and a long K with a tail: the tiles are split into K slices
    ((3333, 259, 4000), 2, 64, 136),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", SCALED_ACT_CASES)
@pytest.mark.usefixtures("either_tile")
def test_down_projection_dx_swiglu_scaled_act(dtype, case):
    """dX2 + SwiGLU backward with the second output of its epilogue (xma_rocm_down_projection_dx_swiglu): dz bit-identical
    to the launch without it; scaled_act[n] = swiglu_packed(z[n]) * w[idx[n]] against the oracle's activation in fp32
    (one rounding); and dW2 from it, sum_n dy[idx[n] // k]^T scaled_act[n], against the oracle's weight gradient of the
    scaled grouped dy, sum_n (w dy)[n]^T h[n], per expert."""
    from xma.rocm import ops

    counts, k, H, I = case
    print(f"case counts={counts} k={k} H={H} I={I} {dtype}", flush=True)
    sel, se, ss, offs = _routing_with_counts(counts, k, 21)
    E, M = len(counts), sum(counts)
    T = M // k
    g = torch.Generator().manual_seed(22)
    dy = torch.randn(T, H, generator=g).to(dtype)
    W2 = (torch.randn(E, H, I, generator=g) * 0.1).to(dtype)  # c_proj.weight: (E, out = H, in = I)
    z = torch.randn(M, 2 * I, generator=g).to(dtype)
    w = torch.rand(M, generator=g).to(dtype)
    dyd, W2d, zd, wd, ssd, offsd = dy.cuda(), W2.cuda(), z.cuda(), w.cuda(), ss.cuda(), offs.cuda()
    dz0 = torch.full((M, 2 * I), float("nan"), dtype=dtype, device="cuda")
    ops.down_projection_dx_swiglu_rocm(dyd, W2d, ssd, offsd, zd, dz0, wd, k)  # W logically (E, K = H, N = I)
    dz1 = torch.full_like(dz0, float("nan"))
    hs = torch.full((M, I), float("nan"), dtype=dtype, device="cuda")
    ops.down_projection_dx_swiglu_scaled_act_rocm(dyd, W2d, ssd, offsd, zd, dz1, hs, wd, k)
    torch.cuda.synchronize()
    assert torch.equal(dz0, dz1) and torch.isfinite(dz1).all()
    h32 = oracle.swiglu_packed(z.float())
    want_hs = h32 * w.float()[ss][:, None]
    assert torch.isfinite(hs).all()
    assert nerr(hs, want_hs) <= _tol(dtype)
    row_err = (hs.cpu().float() - want_hs).abs().amax(dim=1) / want_hs.abs().amax(dim=1).clamp_min(1e-6)
    assert row_err.max() <= 4 * _tol(dtype), int(row_err.argmax())
    # dW2 both ways against the oracle (grouped scaled dy, unscaled h)
    gdy = (dy.float()[ss // k] * w.float()[ss][:, None]).to(dtype)
    want_dw = oracle.group_bwd_W(gdy, h32.to(dtype), offs, E)  # (E, I, H)
    dw = torch.full((E, H, I), float("nan"), dtype=dtype, device="cuda").permute(0, 2, 1)
    ops.group_bwd_W_rocm(dyd, hs, ssd, offsd, dw, None, k, 0)
    torch.cuda.synchronize()
    assert torch.isfinite(dw).all()
    for e in range(E):
        if counts[e] == 0:
            assert torch.count_nonzero(dw[e]) == 0
        else:
            assert nerr(dw[e], want_dw[e]) <= 2 * _tol(dtype), e  # two roundings (w h, then the sum) against (w dy, h)


@pytest.mark.parametrize("scaled_act", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", [*SCALED_ACT_CASES, ((40, 0, 33, 3), 4, 64, 8), ((700, 1, 257, 66), 32, 128, 264)])
def test_router_gradient_from_dx2(dtype, case, scaled_act):
    """d_w[t, j] = <dy[t] @ W2[e], swiglu_packed(z)> by the 256 x 256 kernels, which do not read the expert outputs, against 64 bits: fp32
    sums of H and of I products, an activation of a few 2^-21, one rounding; the other outputs as without it"""
    from xma.rocm import ops

    counts, k, H, I = case
    E = max(len(counts), k)
    counts = (*counts, *[0] * (E - len(counts)))
    counts = (counts[0] - sum(counts) % k + k, *counts[1:])
    print(f"router gradient counts={counts} k={k} H={H} I={I} {dtype} scaled_act={scaled_act}", flush=True)
    _, _, ss, offs = _routing_with_counts(counts, k, 21)
    M = sum(counts)
    g = torch.Generator().manual_seed(22)
    new = lambda *s: torch.randn(*s, generator=g).to(dtype).cuda()
    dy, W2, z, w, ss, offs = new(M // k, H), new(E, H, I), new(M, 2 * I), torch.rand(M, generator=g).to(dtype).cuda(), ss.cuda(), offs.cuda()
    nan = lambda *s: torch.full(s, float("nan"), dtype=dtype, device="cuda")
    dz, dz0, act, act0, d_w = nan(M, 2 * I), nan(M, 2 * I), nan(M, I), nan(M, I), nan(M // k, k)
    with _few_rows_limit(0):
        ops.down_projection_dx_swiglu_router_rocm(dy, W2, ss, offs, z, dz, act if scaled_act else None, w, nan(M, H), d_w, k)
        if scaled_act:
            ops.down_projection_dx_swiglu_scaled_act_rocm(dy, W2, ss, offs, z, dz0, act0, w, k)
            assert torch.equal(act, act0)
        else:
            ops.down_projection_dx_swiglu_rocm(dy, W2, ss, offs, z, dz0, w, k)
    assert torch.equal(dz, dz0)
    expert = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).tolist()
    gate, up = z.double()[:, ::2], z.double()[:, 1::2]
    h = up * gate * torch.sigmoid(gate)
    want, size = torch.empty(M, dtype=torch.float64, device="cuda"), torch.empty(M, dtype=torch.float64, device="cuda")
    for e in set(expert):
        rows = torch.tensor([i for i, x in enumerate(expert) if x == e], device="cuda")
        a, b = dy.double()[ss[rows] // k], W2[e].double()
        want[ss[rows]] = ((a @ b) * h[rows]).sum(1)
        size[ss[rows]] = ((a.abs() @ b.abs()) * h[rows].abs()).sum(1)
    unit, smallest = (2.0**-8, 2.0**-133) if dtype == torch.bfloat16 else (2.0**-11, 2.0**-24)
    bound = unit * want.abs() + ((H + I + 8) * 2.0**-24 + 2.0**-18) * size + smallest
    assert ((d_w.view(-1).double() - want).abs() <= bound).all()


@pytest.mark.parametrize("E,k,M,H,I", [(2, 5, 600, 64, 136), (4096, 2, 20000, 64, 16)])  # more slots than experts; more experts than route counts
def test_router_gradient_knows_no_number_of_experts(E, k, M, H, I):
    """the ids of a caller's own, in the same bounds as above; the pass over the expert outputs that it replaces takes them as well"""
    from xma.rocm import ops

    print(f"router gradient E={E} k={k} M={M}", flush=True)
    g = torch.Generator().manual_seed(23)
    expert, ss = torch.randint(0, E, (M,), generator=g).sort().values.cuda(), torch.randperm(M, generator=g).cuda()
    offs = torch.bincount(expert, minlength=E).cumsum(0)
    new = lambda *s: torch.randn(*s, generator=g).bfloat16().cuda()
    dy, W2, z, w = new(M // k, H), new(E, H, I), new(M, 2 * I), torch.rand(M, generator=g).bfloat16().cuda()
    dz, d_w = torch.empty_like(z), torch.full((M // k, k), float("nan"), dtype=torch.bfloat16, device="cuda")
    with _few_rows_limit(0):
        ops.down_projection_dx_swiglu_router_rocm(dy, W2, ss, offs, z, dz, None, w, new(M, H), d_w, k)
    gate, up = z.double()[:, ::2], z.double()[:, 1::2]
    h, a, b = up * gate * torch.sigmoid(gate), dy.double()[ss // k][:, :, None], W2.double()[expert]
    want, size = torch.empty(2, M, dtype=torch.float64, device="cuda")
    want[ss], size[ss] = ((a * b).sum(1) * h).sum(1), ((a.abs() * b.abs()).sum(1) * h.abs()).sum(1)
    bound = 2.0**-8 * want.abs() + ((H + I + 8) * 2.0**-24 + 2.0**-18) * size + 2.0**-133
    assert ((d_w.view(-1).double() - want).abs() <= bound).all()


def test_scatter2scatter_with_and_without_workspace():
    """The same launch through the C ABI with the scratch for splitting the last round of tiles along K and without
    it (every tile by one workgroup): both within tolerance of the oracle; the workspace query and its error code."""
    from xma.rocm.loader import get_library

    lib = get_library()
    T, E, k, K, N = 300, 3, 2, 2048, 320
    dtype = torch.bfloat16
    sel, se, ss, offs = _routing(T, E, k, 0)
    g = torch.Generator().manual_seed(3)
    M = T * k
    X = torch.randn(M, K, generator=g).to(dtype)
    W = (torch.randn(E, N, K, generator=g) * 0.1).to(dtype)
    want = oracle.scatter2scatter(X, W.permute(0, 2, 1), se, ss, k, True, True, None)
    Xd, Wd, ssd, offsd = X.cuda(), W.cuda(), ss.cuda(), offs.cuda()
    st = torch.cuda.current_stream().cuda_stream
    need = lib.xma_rocm_scatter2scatter_workspace_bytes(M, N, K, E)
    assert need > 0  # a handful of tiles: a last (and only) round that can be split
    ws = torch.empty(need // 4, dtype=torch.float32, device="cuda")

    def run(wptr, wbytes):
        out = torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
        rc = lib.xma_rocm_scatter2scatter(Xd.data_ptr(), K, Wd.data_ptr(), N * K, K, 0, ssd.data_ptr(), offsd.data_ptr(),
                                          out.data_ptr(), N, None, 0, None, M, N, K, E, k, 1, 1, 0, 0, wptr, wbytes, st)
        torch.cuda.synchronize()
        return rc, out

    rc, split = run(ws.data_ptr(), need)
    assert rc == 0 and nerr(split, want) <= TOL
    rc, whole = run(None, 0)
    assert rc == 0 and nerr(whole, want) <= TOL
    assert nerr(split, whole) <= 2e-3  # the two differ only in the order of the fp32 summation over K
    rc, _ = run(ws.data_ptr(), need - 16)
    assert rc == -3 and b"workspace" in lib.xma_rocm_last_error()
    # launches of many rounds of tiles never split: no scratch asked for
    assert lib.xma_rocm_scatter2scatter_workspace_bytes(16384, 28672, 4096, 8) == 0


@pytest.mark.parametrize("counts,K,N", [
    ((63, 0, 64, 65, 129, 1), 40, 72),  # 64 x 64 tiles, dW 64 x 64: edges of both, K and N with remainders
    ((1, 3, 0, 2), 1032, 136),  # few rows, long K: an odd and an even number of K steps in flight
    ((2047, 127, 0, 1), 40, 15368),  # 128 x 128 tiles; dW by 64 x 64
    ((70, 0, 17, 128, 5, 64, 33, 300), 1000, 1032),  # dW from 512 tiles of 128 x 128 on
])
def test_fp32_tiles(counts, K, N):
    """Both output tiles of the fp32 GEMMs, in the three forms, with rows in scattered and in grouped order; the bound is
    that of the other fp32 tests (operands and sums in fp32, only the order of a sum differs from the oracle's)."""
    from xma.rocm import ops

    g = torch.Generator().manual_seed(17)
    E, M = len(counts), sum(counts)
    se = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    ss = torch.randperm(M, generator=g)
    offs = torch.tensor(counts).cumsum(0)
    X, DY = torch.randn(M, K, generator=g), torch.randn(M, N, generator=g)
    W = torch.randn(E, N, K, generator=g) * 0.1
    Wd, ssd, offsd = W.cuda(), ss.cuda(), offs.cuda()
    print(f"case counts={counts} K={K} N={N}", flush=True)
    for x_grouped, y_grouped in ((False, True), (True, False)):
        out = torch.full((M, N), float("nan"), device="cuda")
        ops.scatter2scatter_rocm(X.cuda(), Wd.permute(0, 2, 1), ssd, offsd, out, None, 1, x_grouped, y_grouped)
        assert nerr(out, oracle.scatter2scatter(X, W.permute(0, 2, 1), se, ss, 1, x_grouped, y_grouped, None)) <= TOL_F32
        out = torch.full((M, K), float("nan"), device="cuda")
        ops.scatter2scatter_rocm(DY.cuda(), Wd, ssd, offsd, out, None, 1, x_grouped, y_grouped)
        assert nerr(out, oracle.scatter2scatter(DY, W, se, ss, 1, x_grouped, y_grouped, None)) <= TOL_F32
    dw = torch.full((E, N, K), float("nan"), device="cuda")
    ops.group_bwd_W_rocm(DY.cuda(), X.cuda(), ssd, offsd, dw.permute(0, 2, 1), None, 0, 1)
    assert nerr(dw.permute(0, 2, 1), oracle.group_bwd_W(DY, X[ss], offs, E)) <= TOL_F32


@pytest.mark.parametrize("K", [200, 232, 328, 456, 1000])
@pytest.mark.parametrize("w_kn", [False, True])
@pytest.mark.usefixtures("either_tile")
def test_scatter2scatter_k_tail_of_overlapping_tiles(K, w_kn):
    """Four to sixteen K steps with a partial last one, tiles of more than 192 rows one after another on a workgroup (which load
    the next tile's first step inside their last one) and a smaller one among them: whatever lies past K in memory is NaN."""
    from xma.rocm import ops

    counts, N, pad = (2300, 150, 2305, 2048), 2568, 64
    E, M = len(counts), sum(counts)
    print(f"K tail K={K} w_kn={w_kn}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(K)
    X = torch.full((M, K + pad), float("nan"), device="cuda", dtype=torch.bfloat16)
    X[:, :K] = torch.randn(M, K, generator=g, device="cuda")
    W = torch.full((E, K + pad, N) if w_kn else (E, N, K + pad), float("nan"), device="cuda", dtype=torch.bfloat16)
    Wv = W[:, :K] if w_kn else W[..., :K].permute(0, 2, 1)
    Wv.copy_(torch.randn(E, K, N, generator=g, device="cuda") * 0.1)
    out = torch.full((M, N), float("nan"), device="cuda", dtype=torch.bfloat16)
    idx = torch.randperm(M, generator=g, device="cuda")
    ops.scatter2scatter_rocm(X[:, :K], Wv, idx, torch.tensor(counts).cumsum(0).cuda(), out, None, 1, False, True)
    row = 0
    for e, c in enumerate(counts):
        want = X[idx[row : row + c], :K].float() @ Wv[e].float()
        err = (out[row : row + c].float() - want).abs().max() / want.abs().max()
        assert err <= 2.0**-8, e  # rounding to bf16: half a unit in the last place, 2^-9 of the value
        row += c


@pytest.mark.parametrize("counts", [(17,) * 1000, (0,) * 400 + (16990,) + (0,) * 598 + (10,)])
@pytest.mark.parametrize("w_kn", [False, True])
@pytest.mark.usefixtures("either_tile")
def test_scatter2scatter_walk_refills_its_table(counts, w_kn):
    """Launches of more than 256 candidate tiles for each of 256 workgroups, (M / 256 + E) column blocks in all: a workgroup
    looks for its tiles 256 candidates at a time, and the second table holds tiles (even counts) or none (two experts with
    rows).  bf16 products of 64 terms, so the result is the rounded fp32 sum."""
    from xma.rocm import ops

    E, M, K, N = len(counts), sum(counts), 64, 67 * 256 - 8
    assert (M // 256 + E) * 67 > 256 * 256 and M > ops.FEW_ROWS_MAX
    print(f"walk refill E={E} M={M} N={N} w_kn={w_kn}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    X = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    W = torch.randn(E, *((K, N) if w_kn else (N, K)), generator=g, device="cuda", dtype=torch.bfloat16)
    out = torch.full((M, N), float("nan"), device="cuda", dtype=torch.bfloat16)
    idx = torch.randperm(M, generator=g, device="cuda")
    Wv = W if w_kn else W.permute(0, 2, 1)
    ops.scatter2scatter_rocm(X, Wv, idx, torch.tensor(counts).cumsum(0).cuda(), out, None, 1, False, True)
    row = 0
    for e, c in enumerate(counts):
        if c:
            want = X[idx[row : row + c]].float() @ Wv[e].float()
            err = (out[row : row + c].float() - want).abs().max() / want.abs().max()
            assert err <= 2.0**-8, e  # rounding to bf16: half a unit in the last place, 2^-9 of the value
        row += c


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(
    "counts,K,N",
    [  # rows per expert: one step of K and one column block; K tails and N remainders; more steps than stages; second pass of rows
        ([1], 8, 16),
        ([0, 2, 0, 1], 136, 144),
        ([3, 0, 1, 1], 640, 272),
        ([33, 0, 65], 1032, 64),
        ([1, 32, 0, 2], 2048, 528),
        ([0] * 63 + [1, 2] + [0] * 62 + [1, 1] + [0] * 170 + [4], 264, 80),  # experts with rows at the ends of the lists that a wave reads
    ],
)
def test_forward_gemm_of_few_workgroups(dtype, counts, K, N):
    """x @ W^T where at most one workgroup per compute unit has work: store with bias, row scale and scattered rows, and SwiGLU with gathered
    rows, against the products in 64 bits"""
    from xma.rocm import ops

    print(f"counts={len(counts)} K={K} N={N} {dtype}", flush=True)
    E, M = len(counts), sum(counts)
    g = torch.Generator(device="cuda").manual_seed(K + N)
    new = lambda *s: torch.randn(*s, device="cuda", generator=g).to(dtype)
    nan = lambda *s: torch.full(s, float("nan"), device="cuda", dtype=dtype)
    offs = torch.tensor(counts, device="cuda").cumsum(0)
    idx = torch.randperm(M, device="cuda", generator=g)
    X, W, b, w = new(M, K), new(E, N, K), new(E, N), new(M)
    e = torch.repeat_interleave(torch.arange(E, device="cuda"), torch.tensor(counts, device="cuda"))
    unit = 2.0 ** {torch.bfloat16: -8, torch.float16: -11}[dtype]

    def close(got, rows, scale):
        """fp32 sums of K products and the bias, scaled, then one rounding"""
        product = lambda f: torch.stack([f(rows[i].double()) @ f(W[e[i]].double()).t() + f(b[e[i]].double()) for i in range(M)]) * f(scale)
        want, size = product(lambda t: t), product(torch.abs)
        assert ((got.double() - want).abs() <= unit * want.abs() + (K + 2) * 2.0**-24 * size + 2.0**-24).all()

    out = nan(M, N)
    ops.scatter2scatter_rocm(X, W.permute(0, 2, 1), idx, offs, out, w, 1, True, False, b)
    close(out[idx], X, w[idx].double()[:, None])
    z, h, x = nan(M, N), nan(M, N // 2), new(M, K)
    ops.up_projection_swiglu_rocm(x, W.permute(0, 2, 1), idx, offs, z, h, 1, b)
    close(z, x[idx], torch.ones(M, 1, device="cuda", dtype=torch.float64))
    gate, up = z.double()[:, ::2], z.double()[:, 1::2]
    want = up * gate * torch.sigmoid(gate)
    assert ((h.double() - want).abs() <= (unit + 2.0**-20) * want.abs() + 2.0**-24).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(
    "counts,K,N",
    [  # four waves, 128 columns: more steps than stages, K tails and N remainders; a second pass of rows
        ([1 if e % 5 == 0 else 0 for e in range(60)], 1032, 1424),
        ([0] * 20 + [33] + [0] * 20 + [1, 2, 34], 520, 720),
        ([3, 9, 1, 40, 5, 0, 2, 4], 776, 3600),  # rows for most experts
        ([1 if e % 11 == 5 else 0 for e in range(64)], 2048, 2832),  # 16 steps, in the place of the vector kernel
        # two waves, as many steps; a second pass of rows
        ([0] * 30 + [1, 1, 1] + [0] * 30 + [1], 2040, 4048),
        ([0] * 20 + [33] + [0] * 20 + [1, 2, 34], 776, 272),
    ],
)
def test_forward_gemm_of_four_k_steps_in_flight(dtype, counts, K, N):
    """the forms of that kernel which the launches above do not reach: rows gathered from tokens (fan_out 2) with SwiGLU, and both forms of
    GELU, against the products in 64 bits"""
    from xma.rocm import ops

    print(f"four steps in flight E={len(counts)} K={K} N={N} {dtype}", flush=True)
    counts = [*counts[:-1], counts[-1] + sum(counts) % 2]
    E, M = len(counts), sum(counts)
    assert ops._few_rows_fwd(M, N, K, E, 0, K, M * K, dtype, ops.EPI_SWIGLU) and ops._few_rows_workspace_bytes(M, N, K, E, 0, ops.EPI_SWIGLU) == 0
    g = torch.Generator(device="cuda").manual_seed(K + N)
    new = lambda *s: torch.randn(*s, device="cuda", generator=g).to(dtype)
    nan = lambda *s: torch.full(s, float("nan"), device="cuda", dtype=dtype)
    offs, idx = torch.tensor(counts, device="cuda").cumsum(0), torch.randperm(M, device="cuda", generator=g)
    X, W, b = new(M // 2, K), new(E, N, K) * 0.05, new(E, N)
    e = torch.repeat_interleave(torch.arange(E, device="cuda"), torch.tensor(counts, device="cuda")).tolist()
    unit = 2.0 ** {torch.bfloat16: -8, torch.float16: -11}[dtype]
    product = lambda f: torch.stack([f(X[idx[i] // 2].double()) @ f(W[e[i]].double()).t() + f(b[e[i]].double()) for i in range(M)])
    want, size = product(lambda t: t), product(torch.abs)

    def near(z):
        return ((z.double() - want).abs() <= unit * want.abs() + (K + 2) * 2.0**-24 * size + 2.0**-24).all()

    z, h = nan(M, N), nan(M, N // 2)
    ops.up_projection_swiglu_rocm(X, W.permute(0, 2, 1), idx, offs, z, h, 2, b)
    gate, up = z.double()[:, ::2], z.double()[:, 1::2]
    act = up * gate * torch.sigmoid(gate)
    assert near(z) and ((h.double() - act).abs() <= (unit + 2.0**-20) * act.abs() + 2.0**-24).all()
    for form, (epi, _) in ops.EPI_GELU.items():
        z, h = nan(M, N), nan(M, N)
        ops._scatter2scatter(X, W.permute(0, 2, 1), idx, offs, z, h, None, 2, False, True, epi, M, N, K, b)
        act = torch.nn.functional.gelu(z.double(), approximate=form)
        # a few units of fp32 of the argument, whose own size is that of z
        assert near(z) and ((h.double() - act).abs() <= unit * act.abs() + 2.0**-18 * (1 + z.double().abs())).all()


def test_few_rows_beyond_32_bit_offsets_leaves_the_workspace_alone():
    """rows of X that only the small tile's 64-bit addresses reach, in a shape whose usual kernel asks for no workspace: a workspace of
    another purpose stays as it is (the small tile would cut this K in two ranges and leave their sums there)"""
    from xma.rocm.loader import get_library

    lib, (M, N, K, E), ldx = get_library(), (5, 512, 1024, 4), 1 << 28
    assert lib.xma_rocm_scatter2scatter_few_rows_workspace_bytes(M, N, K, E, 0, 0) == 0
    print("few rows, X beyond 2 GiB", flush=True)
    g = torch.Generator(device="cuda").manual_seed(1)
    X = torch.empty((M - 1) * ldx + K, dtype=torch.bfloat16, device="cuda").as_strided((M, K), (ldx, 1))
    X.copy_(torch.randn(M, K, device="cuda", generator=g))
    W = torch.randn(E, N, K, device="cuda", generator=g).bfloat16()
    counts, out = torch.tensor([2, 0, 2, 1]), torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    offs, space = counts.cumsum(0).cuda(), torch.full((1 << 20,), 171, dtype=torch.uint8, device="cuda")
    rc = lib.xma_rocm_scatter2scatter_few_rows(
        X.data_ptr(), ldx, W.data_ptr(), N * K, K, 0, None, offs.data_ptr(), out.data_ptr(), N, None, 0, None, 0, None, None, 0, M, N, K, E, 1, 1, 1,
        0, 0, space.data_ptr(), 16, torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and (space == 171).all()
    w = W[torch.repeat_interleave(torch.arange(E), counts).cuda()].double()
    want, size = (w * X.double()[:, None]).sum(2), (w.abs() * X.double().abs()[:, None]).sum(2)
    assert ((out.double() - want).abs() <= 2.0**-8 * want.abs() + (K + 1) * 2.0**-24 * size).all()  # fp32 sums of K products, one rounding


@pytest.mark.parametrize("rows,N", [(1, 8), (800, 128)])  # small and large tiles
@pytest.mark.parametrize("E", [7677, 7678, 8192])  # around the table's size from which a workgroup asks for more than 64 KB of LDS; the most
def test_fp32_gemm_of_many_experts(E, rows, N):
    """both orders of the weights, as many experts as the fp32 kernels take; every 97th expert and the last against 64 bits"""
    from xma.rocm import ops

    print(f"fp32 E={E} rows={rows} N={N}", flush=True)
    K, M = 8, E * rows
    g = torch.Generator(device="cuda").manual_seed(E)
    X, W = torch.randn(M, K, device="cuda", generator=g), torch.randn(E, N, K, device="cuda", generator=g)
    offs = torch.arange(1, E + 1, device="cuda") * rows
    idx = torch.arange(M, device="cuda")
    for weight in (W.permute(0, 2, 1), W.permute(0, 2, 1).contiguous()):
        out = torch.full((M, N), float("nan"), device="cuda")
        ops.scatter2scatter_rocm(X, weight, idx, offs, out, None, 1, True, True)
        assert torch.isfinite(out).all()
        for e in [*range(0, E, 97), E - 1]:
            x, w = X[e * rows : (e + 1) * rows].double(), W[e].double().t()
            assert ((out[e * rows : (e + 1) * rows].double() - x @ w).abs() <= (K + 1) * 2.0**-24 * (x.abs() @ w.abs())).all(), e
