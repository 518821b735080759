"""Which kernel, tile and K split a problem gets (no GPU: the plans read no
memory), on both sides of the rules' lines."""

import ctypes

import pytest


def _plan(kind, M, N, K, **kw):
    from qmoe import _capi, ops

    if kind == "W4A16_I4":
        kw["wq_group"] = 32
    return ops.plan_for_shape(getattr(_capi, kind), M, N, K, **kw)[4:]


@pytest.mark.parametrize("kind,M,N,K,tile,ks", [
    # one round of 64-token tiles, two workgroups per CU, before 128-token tiles on half of the CUs
    ("W4A16_MX", 700, 5760, 2880, 64, 1),
    ("W4A16_NV", 700, 5760, 2880, 64, 1),
    ("W4A16_I4", 700, 5760, 2880, 64, 1),
    ("W4A16_MX", 4096, 5760, 2880, 128, 1),  # more than a round of them
    ("W4A16_MX", 512, 32768, 512, 128, 1),
    # few tiles over a long K: more than four slices
    ("W4A16_MX", 128, 256, 7168, 32, 12),
    ("W4A16_NV", 128, 256, 7168, 32, 12),
    ("W4A16_I4", 128, 256, 7168, 32, 12),
    ("W4A16_I4", 1024, 128, 2880, 32, 8),
    ("W4A16_NV", 203, 5760, 2880, 32, 1),
    # tiles in multiples of the XCDs: 84 tiles in 3 slices would be 264 workgroups
    ("W4A16_MX", 65, 7168, 2048, 32, 2),
    ("W4A16_MX", 33, 256, 64, 32, 1),  # a single stage
])
def test_dense_4bit_plans(monkeypatch, kind, M, N, K, tile, ks):
    monkeypatch.setenv("QMOE_SKINNY_ROW_SPLIT", "0")
    monkeypatch.setenv("QMOE_SKINNY_MAX_ROWS", "0")
    assert _plan(kind, M, N, K) == ("tiled_4b", tile, ks)


@pytest.mark.parametrize("kind", ["W4A16_MX", "W4A16_NV", "W4A16_I4"])
@pytest.mark.parametrize("M", [33, 100, 256, 257, 2000, 8192])
@pytest.mark.parametrize("N", [1, 255, 1000, 5760])
def test_dense_4bit_workspace_is_bounded(monkeypatch, kind, M, N):
    """A split is one workgroup per CU: its f32 slices are at most 256 tiles."""
    from qmoe import _capi

    monkeypatch.setenv("QMOE_SKINNY_MAX_ROWS", "0")
    monkeypatch.setenv("QMOE_SKINNY_ROW_SPLIT", "0")
    for K in (64, 320, 2880, 16384):
        path, tile, ks = _plan(kind, M, N, K)
        assert path == "tiled_4b" and ks >= 1 and (ks == 1 or K // 64 // ks >= 4)
        if ks > 1:
            tiles = -(-M // tile) * -(-N // 256)
            assert tiles * ks <= 256 and ks * M * N * 4 <= 256 * tile * 256 * 4 <= 64 << 20
        d = _capi.GemmDesc()
        d.kind, d.a, d.w, d.y, d.w_scale = getattr(_capi, kind), 1 << 24, 1 << 24, 1 << 24, 1 << 24
        d.lda, d.ldw, d.ldy, d.ldws = K, K // 2, N, K // (16 if kind == "W4A16_NV" else 32)
        d.M, d.N, d.K, d.slots, d.max_rows, d.wq_group = M, N, K, 1, M, 32 if kind == "W4A16_I4" else 0
        n = ctypes.c_int64(0)
        assert _capi.lib.qmoe_gemm_workspace_size(ctypes.byref(d), ctypes.byref(n)) == 0
        assert n.value == (ks * M * N * 4 if ks > 1 else 0)


@pytest.mark.parametrize("bm", [32, 64, 128])
@pytest.mark.parametrize("kind,M", [("W4A16_MX", 129), ("W4A16_NV", 129), ("W4A16_I4", 100), ("W4A16_NV", 700)])
def test_forced_4bit_tile_height(monkeypatch, bm, kind, M):
    monkeypatch.setenv("QMOE_SKINNY_MAX_ROWS", "0")
    monkeypatch.setenv("QMOE_W4_BM", str(bm))
    assert _plan(kind, M, 5760, 2880) == ("tiled_4b", bm, 1)
    monkeypatch.setenv("QMOE_W4_KSPLIT", "3")
    assert _plan(kind, M, 5760, 2880) == ("tiled_4b", bm, 3)


@pytest.mark.parametrize("kind,E,M,N,K,act,tile", [
    # weight tiles on one workgroup per CU, or one round of two per CU, in 64-token tiles
    ("W4A16_MX", 4, 512, 5760, 2880, "silu", 64),
    ("W4A16_MX", 8, 1024, 2880, 2880, None, 64),
    ("W4A16_NV", 8, 1024, 5760, 2880, "silu", 64),
    ("W4A16_MX", 4, 1200, 5760, 2880, "silu", 64),  # 276 128-token tiles of equal experts
    ("W4A16_MX", 16, 1024, 2880, 2880, None, 128),  # 288 64-token tiles, 192 of 128
    ("W4A16_I4", 128, 128 * 64, 5760, 2880, "silu", 128),
    ("W4A16_MX", 128, 128 * 40, 5760, 2880, "silu", 64),
])
def test_grouped_4bit_tile_heights(monkeypatch, kind, E, M, N, K, act, tile):
    monkeypatch.setenv("QMOE_SKINNY_MAX_ROWS", "0")
    assert _plan(kind, M, N, K, activation=act, experts=E) == ("tiled_4b", tile, 1)


@pytest.mark.parametrize("kind,E,M,N,K,act,path", [
    ("W4A16_MX", 8, 8, 2880, 2880, None, "stream"),  # 96 weight tiles
    ("W4A16_MX", 8, 64, 5760, 2880, "silu", "stream"),
    ("W4A16_MX", 32, 127, 2880, 2880, None, "stream"),  # 384, 3 rows each
    ("W4A16_MX", 32, 128, 2880, 2880, None, "tiled_4b"),
    ("W4A16_MX", 32, 32, 5760, 2880, "silu", "stream"),
    ("W4A16_MX", 128, 127, 5760, 2880, "silu", "stream"),
    ("W4A16_MX", 128, 128, 5760, 2880, "silu", "tiled_4b"),
    ("W4A16_MX", 128, 128, 2880, 2880, None, "tiled_4b"),
    ("W4A16_NV", 16, 128, 5760, 2880, "silu", "stream"),
    ("W4A16_NV", 32, 160, 5760, 2880, "silu", "stream"),
    ("W4A16_NV", 32, 192, 5760, 2880, "silu", "tiled_4b"),
    ("W4A16_NV", 128, 1024, 1536, 2048, "silu", "stream"),
    ("W4A16_NV", 128, 128, 2880, 2880, None, "tiled_4b"),
    ("W4A16_I4", 128, 1024, 5760, 2880, "silu", "stream"),
    ("W4A16_MX", 8, 128, 2880, 2880, None, "tiled_4b"),  # beyond the streaming kernel's rows
])
def test_grouped_4bit_streaming_limit(kind, E, M, N, K, act, path):
    assert _plan(kind, M, N, K, activation=act, experts=E)[0] == path


def test_grouped_4bit_operands_that_the_tiles_decline():
    """Rows of scales of an odd length: streaming, sized by the rows per expert."""
    from qmoe import _capi

    d = _capi.GemmDesc()
    d.kind, d.a, d.w, d.y, d.w_scale = _capi.W4A16_MX, 1 << 24, 1 << 24, 1 << 24, 1 << 24
    d.lda, d.ldw, d.ldy, d.w_gstride = 2880, 1440, 2880, 1440 * 2880
    d.group_offs = d.active = d.num_active = 1 << 24
    d.M = d.max_rows = d.slots = 128
    d.N = d.K = 2880
    path, tile, ks = (ctypes.c_int32() for _ in range(3))
    for ldws, want in ((90, 2), (91, 0)):
        d.ldws, d.ws_gstride = ldws, ldws * 2880
        assert _capi.lib.qmoe_gemm_plan(ctypes.byref(d), ctypes.byref(path), ctypes.byref(tile), ctypes.byref(ks)) == 0
        assert path.value == want


@pytest.mark.parametrize("kind,E,rows,N,K,act,want", [
    # fewer than 200 tiles of 128 tokens: the four-wavefront tiles
    ("W8A8_GMM", 8, 64, 4096, 7168, "silu", ("tiled_1b", 64)),
    ("W8A8_BLK", 8, 96, 4096, 14336, None, ("tiled_1b_n128", 64)),
    ("W8A8_GMM", 4, 200, 4096, 7168, "silu", ("tiled_1b", 128)),
    ("W8A8_GMM", 8, 64, 7168, 2048, None, ("tiled_8w", 128)),
    # tile-scaled, few rows, no activation: their 128-row weight tiles
    ("W8A8_BLK", 32, 8, 7168, 2048, None, ("tiled_1b_n128", 32)),
    ("W8A8_BLK", 32, 48, 7168, 2048, None, ("tiled_1b_n128", 64)),
    ("W8A8_BLK", 32, 64, 7168, 2048, None, ("tiled_8w", 128)),
    ("W8A8_BLK", 256, 48, 7168, 2048, None, ("tiled_8w", 128)),
    ("W8A8_GMM", 32, 8, 7168, 2048, None, ("tiled_8w", 128)),
    # tile heights by the rounds of tiles
    ("W8A8_GMM", 64, 96, 4096, 7168, "silu", ("tiled_8w", 128)),
    ("W8A8_GMM", 64, 128, 4096, 7168, "silu", ("tiled_8w", 256)),
    ("W8A8_GMM", 64, 200, 4096, 7168, "silu", ("tiled_8w", 256)),
    ("W8A8_GMM", 64, 300, 4096, 7168, "silu", ("tiled_8w", 128)),
    ("W8A8_GMM", 256, 64, 4096, 7168, "silu", ("tiled_8w", 128)),
    ("W8A8_GMM", 8, 64, 4096, 7168 + 128, "silu", ("tiled_8w", 128)),  # K outside the other tiles' granule
])
def test_grouped_fp8_plans(kind, E, rows, N, K, act, want):
    assert _plan(kind, E * rows, N, K, activation=act, experts=E, ws_bn=128 if kind == "W8A8_BLK" else 1)[:2] == want


@pytest.mark.parametrize("N,path", [(1, "tiled_generic"), (64, "tiled_generic"), (128, "tiled_generic"),
                                    (129, "tiled_8w"), (256, "tiled_8w"), (257, "tiled_generic"),
                                    (320, "tiled_generic"), (385, "tiled_8w"), (576, "tiled_8w"), (640, "tiled_8w")])
def test_bf16_width_that_256_row_tiles_pad(N, path):
    assert _plan("W16A16", 40000, N, 2880)[0] == path


@pytest.mark.parametrize("M,N,K,want", [
    (256, 24576, 1536, ("tiled_8w", 128)), (257, 24576, 1536, ("tiled_1b_n128", 64)),
    (320, 24576, 7168, ("tiled_1b_n128", 64)), (321, 24576, 7168, ("tiled_8w", 256)),
    (300, 18432, 7168, ("tiled_8w", 128)),  # 216 tiles: one round
    (300, 24576, 7168 + 128, ("tiled_8w", 256)),  # K outside the other tiles' granule
])
def test_block_fp8_of_257_to_320_tokens(M, N, K, want):
    assert _plan("W8A8_BLK", M, N, K, ws_bn=128)[:2] == want
