"""The bf16 x 4-bit tiles at the sizes where their code lines can go wrong:
row strides that start rows at every 16-byte place of a 128-byte line, K of
one to five stages and around whole lines, ragged channel and token tiles, K
slices that begin inside a line, and experts with few rows. Results against
float64 products of the exactly dequantized weights."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

FP4 = [0.0, 0.5, 1, 1.5, 2, 3, 4, 6, -0.0, -0.5, -1, -1.5, -2, -3, -4, -6]


def _weights(fmt, rows, K, pad, gen):
    """Codes [rows, K/2] (row stride padded by `pad` bytes), scales, f64 values."""
    kb = K // 2
    buf = torch.randint(0, 256, (rows, kb + pad), device="cuda", dtype=torch.uint8, generator=gen)
    codes = buf[:, :kb]
    nib = torch.stack([codes & 15, codes >> 4], -1).flatten(-2).long()
    if fmt == "mx":
        s = torch.randint(119, 128, (rows, K // 32), device="cuda", generator=gen).to(torch.uint8)
        lut = torch.tensor(FP4, device="cuda", dtype=torch.float64)
        val = lut[nib] * torch.exp2(s.double() - 127).repeat_interleave(32, 1)
    else:
        g = 16 if fmt == "nv" else 32
        s = (torch.rand((rows, K // g), device="cuda", generator=gen) * 0.02 + 0.001).to(torch.bfloat16)
        lut = torch.tensor(FP4 if fmt == "nv" else [v - 8.0 for v in range(16)], device="cuda", dtype=torch.float64)
        val = (lut[nib] * s.double().repeat_interleave(g, 1)).to(torch.bfloat16).double()
    return codes, s, val


def _kind(fmt):
    from qmoe import _capi

    return {"mx": _capi.W4A16_MX, "nv": _capi.W4A16_NV, "i4": _capi.W4A16_I4}[fmt]


def _check(got, ref, mag):
    """One bf16 rounding (2^-9 of the value) of a float32 sum: K terms whose
    partial sums err by at most K * 2^-24 of the sum of magnitudes `mag`."""
    err = (got.double() - ref).abs()
    bound = ref.abs() * 2.0 ** -8 + mag * 2.0 ** -12 + 1e-30
    assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.parametrize("fmt", ["mx", "nv", "i4"])
@pytest.mark.parametrize("K,pad", [(64, 0), (128, 16), (192, 0), (320, 48), (576, 32), (1088, 0), (2880, 0), (2816, 80)])
@pytest.mark.parametrize("M,N", [(33, 255), (70, 600), (129, 257), (300, 1)])
def test_dense(monkeypatch, fmt, K, pad, M, N):
    from qmoe import ops

    gen = torch.Generator(device="cuda").manual_seed(K * 7 + M + N)
    codes, s, val = _weights(fmt, N, K, pad, gen)
    x = torch.randn((M, K), device="cuda", generator=gen).to(torch.bfloat16)
    ref, mag = x.double() @ val.t(), x.double().abs() @ val.abs().t()
    monkeypatch.setenv("QMOE_SKINNY_MAX_ROWS", "0")
    monkeypatch.setenv("QMOE_SKINNY_ROW_SPLIT", "0")
    _check(ops.gemm(_kind(fmt), x, codes, w_scale=s), ref, mag)
    for bm in ("32", "64", "128"):
        for ks in ("1", "3"):
            monkeypatch.setenv("QMOE_W4_BM", bm)
            monkeypatch.setenv("QMOE_W4_KSPLIT", ks)
            _check(ops.gemm(_kind(fmt), x, codes, w_scale=s), ref, mag)


@pytest.mark.parametrize("fmt", ["mx", "nv", "i4"])
@pytest.mark.parametrize("bm,M,N,K,act", [
    (32, 257, 700, 576, None), (64, 300, 700, 1088, None), (128, 400, 515, 320, None),  # two K groups
    (64, 1100, 4000, 128, None), (128, 2049, 4000, 192, None),  # 288 and 272 tiles: one K group
    (32, 70, 1000, 320, "silu"), (64, 129, 1000, 576, "swigluoai"), (128, 300, 514, 192, "silu"),
    (128, 2049, 4000, 128, "silu"),  # 17 x 16 tiles of gate and up rows
])
def test_dense_line_tiles(monkeypatch, fmt, bm, M, N, K, act):
    """Every instance of the line pipeline in dense problems: tile heights,
    one and two K groups, fused activations, ragged channels and tokens."""
    from qmoe import ops

    gen = torch.Generator(device="cuda").manual_seed(K + M + N)
    codes, s, val = _weights(fmt, N, K, 0, gen)
    x = torch.randn((M, K), device="cuda", generator=gen).to(torch.bfloat16)
    h, mag = x.double() @ val.t(), x.double().abs() @ val.abs().t()
    if act:
        g, u = h[:, :N // 2], h[:, N // 2:]
        # |d act| <= 2 |u| dg + 2 |g| du near these sizes
        mag = 2 * ((u.abs() + 1) * mag[:, :N // 2] + (g.abs() + 1) * mag[:, N // 2:]) + 1
        if act == "silu":
            h = g * torch.sigmoid(g) * u
        else:
            g, u = g.clamp(max=7.0), u.clamp(-7.0, 7.0)
            h = (u + 1) * g * torch.sigmoid(1.702 * g)
    monkeypatch.setenv("QMOE_SKINNY_MAX_ROWS", "0")
    monkeypatch.setenv("QMOE_SKINNY_ROW_SPLIT", "0")
    monkeypatch.setenv("QMOE_W4_BM", str(bm))
    for ks in (1, 2) if K >= 320 else (1,):
        monkeypatch.setenv("QMOE_W4_KSPLIT", str(ks))
        with ops.record_plans() as plans:
            got = ops.gemm(_kind(fmt), x, codes, w_scale=s, activation=act)
        assert tuple(plans[0][4:]) == ("tiled_4b", bm, ks)
        _check(got, h, mag)


@pytest.mark.parametrize("fmt", ["mx", "nv", "i4"])
@pytest.mark.parametrize("bm", ["64", "128"])
@pytest.mark.parametrize("K,N,act", [(320, 64, None), (576, 520, "silu"), (1088, 514, "swigluoai"), (2880, 256, None)])
def test_grouped(monkeypatch, fmt, bm, K, N, act):
    """Experts of 0, 1, 31, 33, 65, 96, 97 and 140 rows, gathered tokens, scattered rows, weights and bias."""
    from qmoe import ops

    gen = torch.Generator(device="cuda").manual_seed(K + N)
    counts = [0, 1, 31, 33, 65, 96, 97, 140]
    E, M, T = len(counts), sum(counts), 90
    codes, s, val = _weights(fmt, E * N, K, 0, gen)
    codes, s, val = codes.view(E, N, -1), s.view(E, N, -1), val.view(E, N, K)
    x = torch.randn((T, K), device="cuda", generator=gen).to(torch.bfloat16)
    i32 = dict(dtype=torch.int32, device="cuda")
    offs = torch.tensor(np.concatenate([[0], np.cumsum(counts)]), **i32)
    rows = torch.randint(0, T, (M,), generator=gen, **i32)
    perm = torch.randperm(M, generator=torch.Generator().manual_seed(1)).to(**i32)
    rw = torch.rand(M, device="cuda", generator=gen).to(torch.bfloat16)
    bias = torch.randn((E, N), device="cuda", generator=gen)
    active = torch.arange(E, **i32)
    monkeypatch.setenv("QMOE_SKINNY_MAX_ROWS", "0")
    monkeypatch.setenv("QMOE_W4_BM", bm)
    out = torch.empty((M, N // 2 if act else N), dtype=torch.bfloat16, device="cuda")
    ops.gemm(_kind(fmt), x, codes, w_scale=s, bias=bias, group_offs=offs, active=active,
             num_active=torch.tensor([E], **i32), slots=E, max_rows=T, M=M, a_rows=rows, activation=act, row_weight=rw,
             y_rows=perm, out=out)
    g0 = 0
    for e, c in enumerate(counts):
        r = slice(g0, g0 + c)
        g0 += c
        xs = x[rows[r].long()].double()
        h, mag = xs @ val[e].t() + bias[e].double(), xs.abs() @ val[e].abs().t() + bias[e].double().abs()
        if act:
            I = N // 2
            g, u = h[:, :I], h[:, I:]
            # |d act| <= 2 |u| dg + 2 |g| du near these sizes
            mag = 2 * ((u.abs() + 1) * mag[:, :I] + (g.abs() + 1) * mag[:, I:]) + 1
            if act == "silu":
                h = g * torch.sigmoid(g) * u
            else:
                g, u = g.clamp(max=7.0), u.clamp(-7.0, 7.0)
                h = (u + 1) * g * torch.sigmoid(1.702 * g)
        w = rw[r].double()[:, None]
        _check(out[perm[r].long()], h * w, mag * w)


@pytest.mark.parametrize("K,ks", [(2496, None), (2560, None), (2624, "1"), (2624, "3"), (64, "1"), (384, None)])
@pytest.mark.parametrize("M", [33, 129])
def test_ring_fused_activation(monkeypatch, K, ks, M):
    """The NVFP4 ring below and above the K from which two K groups share a
    workgroup, halves of equal and unequal stages, gate and up rows."""
    from qmoe import ops

    I = 257
    gen = torch.Generator(device="cuda").manual_seed(K + M)
    codes, s, val = _weights("nv", 2 * I, K, 0, gen)
    x = torch.randn((M, K), device="cuda", generator=gen).to(torch.bfloat16)
    monkeypatch.setenv("QMOE_SKINNY_MAX_ROWS", "0")
    monkeypatch.setenv("QMOE_SKINNY_ROW_SPLIT", "0")
    if ks:
        monkeypatch.setenv("QMOE_W4_KSPLIT", ks)
    got = ops.gemm(_kind("nv"), x, codes, w_scale=s, activation="silu")
    h, mag = x.double() @ val.t(), x.double().abs() @ val.abs().t()
    g, u = h[:, :I], h[:, I:]
    mag = 2 * ((u.abs() + 1) * mag[:, :I] + (g.abs() + 1) * mag[:, I:]) + 1
    _check(got, g * torch.sigmoid(g) * u, mag)
