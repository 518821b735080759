"""The eight-wavefront tiles (block-scaled e4m3, bf16) at the edges of their
tiles, stages and token groups: block-scaled results against the
four-wavefront tiles (the same block sums, scaled and added in the same
order: bit-identical with tile scales), and both kinds against float64 products of the decoded operands."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
F8 = torch.float8_e4m3fn


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _codes(shape, g):
    return (torch.randn(shape, device="cuda", generator=g) * 40).clamp(-448, 448).to(F8)


def _scales(shape, g):
    return torch.rand(shape, device="cuda", generator=g) * 0.01 + 0.001


def _check(got, ref, mag):
    """One bf16 rounding (2^-9 of the value) of a float32 sum of magnitude `mag`."""
    err = (got.double() - ref).abs()
    bound = ref.abs() * 2.0 ** -8 + mag * 2.0 ** -14 + 1e-30
    assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.parametrize("bm", ["128", "256"])
@pytest.mark.parametrize("M,N,K", [(1, 128, 128), (33, 384, 256), (128, 640, 384), (129, 256, 1152), (300, 1280, 512)])
def test_dense_tiles(monkeypatch, bm, M, N, K):
    from qmoe import _capi, ops

    g = _gen(M + N + K)
    x, w = _codes((M, K), g), _codes((N, K), g)
    xs, ws = _scales((M, K // 128), g), _scales((N // 128, K // 128), g)
    args = (_capi.W8A8_BLK, x.view(torch.uint8), w.view(torch.uint8))
    kw = dict(a_scale=xs, w_scale=ws, ws_bn=128)
    monkeypatch.setenv("QMOE_SKINNY_MAX_ROWS", "0")
    monkeypatch.setenv("QMOE_T8_BM", bm)
    with ops.record_plans() as plans:
        got = ops.gemm(*args, **kw)
    assert plans[0][4] == "tiled_8w"
    monkeypatch.setenv("QMOE_F8_KSPLIT", "1")
    xd = x.double() * xs.double().repeat_interleave(128, 1)
    wd = w.double() * ws.double().repeat_interleave(128, 0).repeat_interleave(128, 1)
    _check(got, xd @ wd.t(), xd.abs() @ wd.abs().t())
    monkeypatch.setenv("QMOE_T8_BM", "0")
    base = ops.gemm(*args, **kw)
    if K % 256 == 0:  # the four-wavefront tiles' granule
        assert torch.equal(got, base)


@pytest.mark.parametrize("bm", ["128", "256"])
@pytest.mark.parametrize("recipe,N,K,act", [("tiles", 512, 384, "silu"), ("tiles", 384, 256, None),
                                            ("channel", 200, 640, None), ("channel", 1026, 512, "silu"),
                                            ("e5m2", 1026, 640, "silu"), ("e5m2", 512, 512, None)])
def test_grouped(monkeypatch, bm, recipe, N, K, act):
    """Experts of 0 to 260 rows, gathered tokens, scattered rows, routing weights and bias."""
    from qmoe import _capi, ops

    g = _gen(N + K)
    counts = [0, 1, 31, 33, 64, 65, 127, 129, 200, 260]
    E, M, T = len(counts), sum(counts), 150
    x, w = _codes((T, K), g), _codes((E, N, K), g)
    tiles = recipe == "tiles"
    if recipe == "e5m2":
        w = w.float().to(torch.float8_e5m2)
    nb = (K + 511) // 512
    xs = _scales((T, K // 128 if tiles else nb), g)
    ws = _scales((E, N // 128, K // 128) if tiles else (E, N), g)
    i32 = dict(dtype=torch.int32, device="cuda")
    offs = torch.tensor(np.concatenate([[0], np.cumsum(counts)]), **i32)
    rows = torch.randint(0, T, (M,), generator=g, **i32)
    perm = torch.randperm(M, generator=torch.Generator().manual_seed(2)).to(**i32)
    rw = torch.rand(M, device="cuda", generator=g).to(torch.bfloat16)
    bias = torch.randn((E, N), device="cuda", generator=g)

    def run(v):
        monkeypatch.setenv("QMOE_T8_BM", v)
        out = torch.empty((M, N // 2 if act else N), dtype=torch.bfloat16, device="cuda")
        return ops.gemm(_capi.W8A8_BLK if tiles else _capi.W8A8_GMM, x.view(torch.uint8), w.view(torch.uint8),
                        a_scale=xs, w_scale=ws, ws_bn=128 if tiles else 1, wfmt=2 if recipe == "e5m2" else 0,
                        bias=bias, group_offs=offs,
                        active=torch.arange(E, **i32), num_active=torch.tensor([E], **i32), slots=E, max_rows=T, M=M,
                        a_rows=rows, activation=act, row_weight=rw, y_rows=perm, out=out)

    monkeypatch.setenv("QMOE_SKINNY_MAX_ROWS", "0")
    with ops.record_plans() as plans:
        got = run(bm)
    assert tuple(plans[0][4:]) == ("tiled_8w", int(bm), 1)
    if K % 256 == 0:
        base = run("0")
        if tiles:
            assert torch.equal(got, base)
        else:
            # the channel scale and the bias may be one fma here and two
            # roundings there: 2^-24 of the float32 values, which the activation
            # magnifies at most a few hundred times near its zeros, then at most
            # one bf16 step (2^-7 of the value at the lower end of a binade)
            d = (got.double() - base.double()).abs()
            assert bool((d <= base.double().abs() * 2.0 ** -7 + 2.0 ** -14).all())
    xd = x.double() * xs.double().repeat_interleave(128 if tiles else 512, 1)[:, :K]
    g0 = 0
    for e, c in enumerate(counts):
        r = slice(g0, g0 + c)
        g0 += c
        s = ws[e].double()
        wd = w[e].double() * (s.repeat_interleave(128, 0).repeat_interleave(128, 1) if tiles else s[:, None])
        xr = xd[rows[r].long()]
        h, mag = xr @ wd.t() + bias[e].double(), xr.abs() @ wd.abs().t() + bias[e].double().abs()
        if act:
            a, u = h[:, :N // 2], h[:, N // 2:]
            mag = 4 * ((u.abs() + 1) * mag[:, :N // 2] + (a.abs() + 1) * mag[:, N // 2:])
            h = a * torch.sigmoid(a) * u
        wt = rw[r].double()[:, None]
        _check(got[perm[r].long()], h * wt, mag * wt)


@pytest.mark.parametrize("bm", ["128", "256"])
@pytest.mark.parametrize("M,N,K", [(1, 1, 64), (65, 255, 128), (129, 257, 192), (300, 600, 448), (70, 520, 2880)])
def test_bf16(monkeypatch, bm, M, N, K):
    from qmoe import _capi, ops

    g = _gen(M + N + K)
    x = torch.randn((M, K), device="cuda", generator=g).to(torch.bfloat16)
    w = torch.randn((N, K + 8), device="cuda", generator=g).to(torch.bfloat16)[:, :K]  # padded rows
    bias = torch.randn((1, N), device="cuda", generator=g)
    monkeypatch.setenv("QMOE_SKINNY_MAX_ROWS", "0")
    monkeypatch.setenv("QMOE_T8_BM", bm)
    with ops.record_plans() as plans:
        got = ops.gemm(_capi.W16A16, x, w, bias=bias)
    assert plans[0][4] == "tiled_8w"
    _check(got, x.double() @ w.double().t() + bias.double(), x.double().abs() @ w.double().abs().t() + bias.double().abs())


def _tall_tiles(M, N):
    """256-token tiles ahead of a dense problem's 128-token ones: the fewest
    weighted rounds over 256 CUs (256-token tiles 168, 128-token ones 100, a
    second launch 10), tall rounds whole but for the last or the last two."""
    nt = -(-N // 256)
    m256 = -(-M // 256)
    rounds = -(-m256 * nt // 256)
    tall = [0, m256] + [r * 256 // nt for r in range(rounds - 1, 0, -1) if r >= rounds - 2]

    def cost(t):
        rest = max(M - 256 * t, 0)
        return -(-t * nt // 256) * 168 + -(-(-(-rest // 128) * nt) // 256) * 100 + (10 if t and rest else 0)

    return min(tall, key=cost)


@pytest.mark.parametrize("kind", ["fp8", "bf16"])
@pytest.mark.parametrize("M,N,K,two", [(1024, 18432, 256, True), (2047, 18432, 1152, True), (1500, 14300, 256, True),
                                       (769, 18300, 256, False)])
def test_dense_rounds_of_two_heights(monkeypatch, kind, M, N, K, two):
    """Problems whose last, partly filled round of 256-token tiles runs as
    128-token tiles (the last of the four: all in one height): the same sums
    in the same order as 128-token tiles throughout, also from padded and
    gathered activation rows."""
    from qmoe import _capi, ops

    g = _gen(M + N)
    rw = torch.rand(M, device="cuda", generator=g).to(torch.bfloat16)
    perm = torch.randperm(M, generator=torch.Generator().manual_seed(3)).to(dtype=torch.int32, device="cuda")
    rows = torch.randint(0, M, (M,), generator=g, dtype=torch.int32, device="cuda")
    if kind == "fp8":
        N = (N + 127) // 128 * 128
        x, w = _codes((M, K + 16), g)[:, :K], _codes((N, K), g)
        xs, ws = _scales((M, K // 128 + 3), g)[:, :K // 128], _scales((N // 128, K // 128), g)
        call = lambda **kw: ops.gemm(_capi.W8A8_BLK, x.view(torch.uint8), w.view(torch.uint8), a_scale=xs,  # noqa: E731
                                     w_scale=ws, ws_bn=128, **kw)
        xd = x.double() * xs.double().repeat_interleave(128, 1)
        wd = w.double() * ws.double().repeat_interleave(128, 0).repeat_interleave(128, 1)
    else:
        x = torch.randn((M, K + 8), device="cuda", generator=g).to(torch.bfloat16)[:, :K]
        w = torch.randn((N, K), device="cuda", generator=g).to(torch.bfloat16)
        call = lambda **kw: ops.gemm(_capi.W16A16, x, w, **kw)  # noqa: E731
        xd, wd = x.double(), w.double()
    assert (0 < 256 * _tall_tiles(M, N) < M) == two
    ref, mag = xd @ wd.t(), xd.abs() @ wd.abs().t()
    for kw in ({}, dict(row_weight=rw, y_rows=perm), dict(a_rows=rows)):
        monkeypatch.delenv("QMOE_T8_BM", raising=False)
        with ops.record_plans() as plans:
            got = call(**kw)
        assert tuple(plans[0][4:6]) == ("tiled_8w", 256 if _tall_tiles(M, N) else 128)
        monkeypatch.setenv("QMOE_T8_BM", "128")
        assert torch.equal(got, call(**kw))
        if "y_rows" in kw:
            wt = rw.double()[:, None]
            _check(got[perm.long()], ref * wt, mag * wt)
        elif kw:
            _check(got, ref[rows.long()], mag[rows.long()])
        else:
            _check(got, ref, mag)
