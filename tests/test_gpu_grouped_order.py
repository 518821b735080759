"""Grouped tiles whose workgroups find their tile by a scan of the group sizes
(bf16 x 4-bit and eight-wavefront FP8 tiles): every (m-tile, weight tile) pair
runs once, for fewer m-tiles than XCDs, for whole multiples of 8 and a few
more, and for more groups than one pass of the scan holds."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _counts(name):
    if name == "one":
        return [0, 0, 5]
    if name == "four":
        return [130, 0, 200, 1]  # 5 m-tiles of 128 rows
    if name == "sixteen":
        return [1] * 8 + [128] * 8
    if name == "seventeen":
        return [3] * 17
    if name == "ends":
        return [70] + [0] * 298 + [129]  # 300 groups: the first and the last
    return [1 if i % 3 else 0 for i in range(257)]  # one group past a pass


@pytest.mark.parametrize("kind", ["mxfp4", "fp8"])
@pytest.mark.parametrize("name", ["one", "four", "sixteen", "seventeen", "ends", "past"])
def test_every_pair_runs_once(monkeypatch, kind, name):
    from qmoe import _capi, ops

    counts = _counts(name)
    E, M, K, N = len(counts), sum(counts), 128, 600  # 3 weight tiles
    g = torch.Generator(device="cuda").manual_seed(E + M)
    i32 = dict(dtype=torch.int32, device="cuda")
    offs = torch.tensor([sum(counts[:e]) for e in range(E + 1)], **i32)
    kw = dict(group_offs=offs, active=torch.arange(E, **i32), num_active=torch.tensor([E], **i32), slots=E, max_rows=M,
              M=M, out=torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda"))
    monkeypatch.setenv("QMOE_SKINNY_MAX_ROWS", "0")
    with ops.record_plans() as plans:
        if kind == "mxfp4":
            codes = torch.randint(0, 256, (E, N, K // 2), dtype=torch.uint8, device="cuda", generator=g)
            s = torch.randint(120, 128, (E, N, K // 32), device="cuda", generator=g).to(torch.uint8)
            lut = torch.tensor([0.0, 0.5, 1, 1.5, 2, 3, 4, 6], device="cuda", dtype=torch.float64)
            nib = torch.stack([codes & 15, codes >> 4], -1).flatten(-2).long()
            w = lut[nib & 7] * (1 - 2 * (nib >> 3)) * torch.exp2(s.double() - 127).repeat_interleave(32, -1)
            x = torch.randn((M, K), device="cuda", generator=g).to(torch.bfloat16)
            xd = x.double()
            got = ops.gemm(_capi.W4A16_MX, x, codes, w_scale=s, **kw)
        else:
            f8 = torch.float8_e4m3fn
            x8 = (torch.randn((M, K), device="cuda", generator=g) * 40).clamp(-448, 448).to(f8)
            w8 = (torch.randn((E, N, K), device="cuda", generator=g) * 40).clamp(-448, 448).to(f8)
            xs = torch.rand((M, 1), device="cuda", generator=g) * 0.01 + 0.001
            ws = torch.rand((E, N), device="cuda", generator=g) * 0.01 + 0.001
            xd, w = x8.double() * xs.double(), w8.double() * ws.double()[..., None]
            monkeypatch.setenv("QMOE_T8_BM", "128")
            got = ops.gemm(_capi.W8A8_GMM, x8.view(torch.uint8), w8.view(torch.uint8), a_scale=xs, w_scale=ws, ws_bn=1,
                           **kw)
    assert plans[0][4] == ("tiled_4b" if kind == "mxfp4" else "tiled_8w")
    for e, c in enumerate(counts):
        if c:
            r = slice(int(offs[e]), int(offs[e]) + c)
            ref, mag = xd[r] @ w[e].t(), xd[r].abs() @ w[e].abs().t()
            # one bf16 rounding of a float32 sum of K terms
            assert bool(((got[r].double() - ref).abs() <= ref.abs() * 2.0 ** -8 + mag * 2.0 ** -14).all()), e
