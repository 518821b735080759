"""Measured cases: the quantized linears and fused MoE layers of the decoder
layers this framework serves, through its public entry points.

Every case is one call that a serving step makes: a linear
(`quantized_matmul`, `quantized_matmul_fp4`, `UnquantizedLinearMethod.apply`),
a whole MoE layer (`Mxfp4MoEMethod.apply_monolithic`, or `select_experts` +
`fused_moe_gmm`) or the fused decode layer (`ops.moe_decode_routed`). Cases
with ``graph`` replay the call as a HIP graph captured once, as a serving
engine does for its decode batch sizes.
"""

import math
import os
import sys
from types import SimpleNamespace

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vllm-torchtpu_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DEV = "cuda"
F8 = torch.float8_e4m3fn


def listed():
    return [
        # one user's token through Llama-3-8B's up projection, launched from Python: latency
        dict(name="fp8_up_1", kind="linear", fmt="fp8", M=1, K=4096, N=14336, graph=False),
        # a decode batch of 16 through a GPT-OSS-shaped MXFP4 linear
        dict(name="mxfp4_16", kind="linear", fmt="mxfp4", M=16, K=2880, N=5760, graph=True),
        # a mixed prefill / decode batch of ragged size, INT8 recipe, Llama-3-8B's qkv
        dict(name="int8_qkv_777", kind="linear", fmt="int8", M=777, K=4096, N=6144, graph=False),
        # a full prefill chunk through Llama-3-8B's down projection
        dict(name="fp8_down_4096", kind="linear", fmt="fp8", M=4096, K=14336, N=4096, graph=False),
        # a prefill chunk through DeepSeek-V3's dense gate_up, native 128 x 128 tiles
        dict(name="fp8_blocks_2048", kind="linear", fmt="fp8_blocks", M=2048, K=7168, N=18432, graph=False),
        # a prefill chunk through the MXFP4 linear
        dict(name="mxfp4_4096", kind="linear", fmt="mxfp4", M=4096, K=2880, N=5760, graph=False),
        # a short prompt (odd length) through an NVFP4 linear
        dict(name="nvfp4_203", kind="linear", fmt="nvfp4", M=203, K=2880, N=5760, graph=False),
        # an unquantized attention projection (the linears of an MXFP4 checkpoint stay bf16)
        dict(name="bf16_1024", kind="linear", fmt="bf16", M=1024, K=4096, N=6144, graph=False),
        # GPT-OSS MoE layer, decode batch of 16
        dict(name="gptoss_moe_16", kind="moe_mxfp4", E=128, k=4, H=2880, I=2880, T=16, graph=True),
        # the same layer, a prefill chunk
        dict(name="gptoss_moe_2048", kind="moe_mxfp4", E=128, k=4, H=2880, I=2880, T=2048, graph=False),
        # DeepSeek-V3 MoE layer (shared + routed experts), decode batch of 8
        dict(name="dsv3_decode_8", kind="decode_op", E=256, k=8, H=7168, I=2048, T=8, graph=True),
        # DeepSeek-V3 routed experts (default per-channel recipe), a prefill chunk
        dict(name="dsv3_moe_2048", kind="moe_fp8", fmt="fp8", E=256, k=8, H=7168, I=2048, T=2048, graph=False),
    ]


# (K, N) of the linears of Llama-3-8B, DeepSeek-V3 and GPT-OSS decoder layers
_SHAPES = [(4096, 14336), (14336, 4096), (4096, 6144), (4096, 4096), (7168, 1536), (7168, 576), (1536, 24576),
           (512, 32768), (2048, 7168), (2880, 5760), (7168, 256)]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear"] * 7 + ["moe_mxfp4", "moe_fp8", "decode_op"])
    if kind == "linear":
        fmt = rng.choice(["fp8", "int8", "fp8_blocks", "mxfp4", "nvfp4", "bf16"])
        if rng.random() < 0.5:
            K, N = rng.choice(_SHAPES)
        else:
            K, N = 128 * _log_int(rng, 4, 112), _log_int(rng, 200, 20000)
        if fmt == "fp8_blocks":
            K, N = (K + 127) // 128 * 128, (N + 127) // 128 * 128
        M = _log_int(rng, 1, min(4096, int(5.4e11 / (2.0 * K * N))))
        return dict(kind=kind, fmt=fmt, M=M, K=K, N=N, graph=M <= 16 and rng.random() < 0.5)
    if kind == "moe_mxfp4":
        return dict(kind=kind, E=rng.choice([32, 64, 128]), k=4, H=2880, I=2880, T=_log_int(rng, 1, 2048), graph=False)
    if kind == "moe_fp8":
        return dict(kind=kind, fmt=rng.choice(["fp8", "fp8_block"]), E=rng.choice([32, 64, 128]), k=8, H=7168, I=2048,
                    T=_log_int(rng, 1, 2048), graph=False)
    return dict(kind=kind, E=rng.choice([64, 128, 256]), k=8, H=7168, I=2048, T=rng.randint(1, 16), graph=True)


# ---------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _normal(shape, g, std=1.0):
    return torch.empty(shape, device=DEV, dtype=torch.float32).normal_(0.0, std, generator=g)


def _acts(rows, cols, g):
    """Post-norm hidden states: unit variance, a few columns ten times larger."""
    x = _normal((rows, cols), g)
    x[:, torch.randint(0, cols, (max(1, cols // 512),), generator=g, device=DEV)] *= 10.0
    return x.to(torch.bfloat16)


def _channel_codes(shape, g, int8=False):
    """Gaussian weights [.., N, K] as per-channel e4m3 / int8 codes and f32 scales."""
    w = _normal(shape, g, 0.02)
    s = w.abs().amax(-1) / (127.0 if int8 else 448.0)
    v = w / s[..., None]
    return (v.round().clamp(-127, 127).to(torch.int8) if int8 else v.clamp(-448, 448).to(F8)), s


def _tile_codes(shape, g):
    """Gaussian weights [N, K] as e4m3 codes with one f32 scale per 128 x 128 tile."""
    n, k = shape
    t = _normal((n // 128, 128, k // 128, 128), g, 0.02)
    s = t.abs().amax(dim=(1, 3)) / 448.0
    return (t / s[:, None, :, None]).clamp(-448, 448).to(F8).view(n, k), s.contiguous()


def _fp4_codes(v):
    """Nearest e2m1 codes of v [.., K], two per byte (low nibble = even column)."""
    edges = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=v.device)
    c = torch.bucketize(v.abs(), edges).to(torch.uint8) | ((v < 0).to(torch.uint8) << 3)
    return (c[..., 0::2] | (c[..., 1::2] << 4)).contiguous()


def _mxfp4_weights(n, k, g):
    w = _normal((n, k // 32, 32), g, 0.02)
    e = torch.floor(torch.log2(w.abs().amax(-1).clamp_min(1e-20))) - 2.0
    return _fp4_codes((w * torch.exp2(-e)[..., None]).view(n, k)), (e + 127.0).to(torch.uint8)


def _nvfp4_weights(n, k, g):
    """Codes and the fused bf16 block scales (e4m3 block scale x f32 global scale)."""
    w = _normal((n, k // 16, 16), g, 0.02)
    glob = 0.1 / (448.0 * 6.0)
    blk = (w.abs().amax(-1) / (6.0 * glob)).clamp(2.0 ** -6, 448.0).to(F8).float()
    s = (blk * glob).to(torch.bfloat16)
    return _fp4_codes((w / s.float()[..., None]).view(n, k)), s


def _linear_inputs(c, seed):
    g = _gen(seed)
    M, K, N, fmt = c["M"], c["K"], c["N"], c["fmt"]
    if fmt in ("fp8", "int8"):
        w, s = _channel_codes((N, K), g, fmt == "int8")
    elif fmt == "fp8_blocks":
        w, s = _tile_codes((N, K), g)
    elif fmt == "mxfp4":
        w, s = _mxfp4_weights(N, K, g)
    elif fmt == "nvfp4":
        w, s = _nvfp4_weights(N, K, g)
    else:
        w, s = _normal((N, K), g, 0.02).to(torch.bfloat16), None
    return dict(x=_acts(M, K, g), w=w, s=s)


def _moe_inputs(c, seed):
    g = _gen(seed)
    E, H, I, T, kind = c["E"], c["H"], c["I"], c["T"], c["kind"]
    d = dict(x=_acts(T, H, g))
    if kind == "moe_mxfp4":
        parts = [(_mxfp4_weights(2 * I, H, g), _mxfp4_weights(H, I, g)) for _ in range(E)]
        d["w13"], d["s13"] = (torch.stack([p[0][i] for p in parts]) for i in (0, 1))
        d["w2"], d["s2"] = (torch.stack([p[1][i] for p in parts]) for i in (0, 1))
        d["b13"], d["b2"] = _normal((E, 2 * I), g, 0.1).to(torch.bfloat16), _normal((E, H), g, 0.1).to(torch.bfloat16)
        d["logits"] = _normal((T, E), g).to(torch.bfloat16)
        return d
    tiles = kind == "decode_op" or c["fmt"] == "fp8_block"
    make = _tile_codes if tiles else _channel_codes
    d["w13"] = torch.empty((E, 2 * I, H), device=DEV, dtype=F8)
    d["w2"] = torch.empty((E, H, I), device=DEV, dtype=F8)
    s13, s2 = [], []
    for e in range(E):
        d["w13"][e], s = make((2 * I, H), g)
        s13.append(s)
        d["w2"][e], s = make((H, I), g)
        s2.append(s)
    d["s13"], d["s2"] = torch.stack(s13), torch.stack(s2)
    if kind == "decode_op":
        d["sh13"], d["ss13"] = make((2 * I, H), g)
        d["sh2"], d["ss2"] = make((H, I), g)
    d["logits"] = _normal((T, E), g).to(torch.bfloat16)
    d["bias"] = _normal((E,), g, 0.1)
    return d


def _grouped_layer(bias):
    """The routing attributes of a DeepSeek-V3 layer (8 groups, 4 kept)."""
    return SimpleNamespace(e_score_correction_bias=bias, routed_scaling_factor=2.5, use_grouped_topk=True,
                           num_expert_group=8, topk_group=4, hash_indices_table=None)


def _call(c, d):
    """The call of one case as a function of no arguments."""
    from qmoe import ops
    from qmoe.layers.fused_moe import fused_moe_gmm
    from qmoe.layers.linear_common import quantized_matmul, quantized_matmul_fp4
    from qmoe.layers.moe_routing import select_experts
    from qmoe.layers.quantization.mxfp4 import Mxfp4MoEMethod
    from qmoe.layers.quantization.unquantized import UnquantizedLinearMethod

    x = d["x"]
    if c["kind"] == "linear":
        w, s = d["w"], d["s"]
        if c["fmt"] in ("mxfp4", "nvfp4"):
            return lambda: quantized_matmul_fp4(x, w, s)
        if c["fmt"] == "bf16":
            layer = torch.nn.Module()
            layer.weight = torch.nn.Parameter(w, requires_grad=False)
            method = UnquantizedLinearMethod()
            method.process_weights_after_loading(layer)
            return lambda: method.apply(layer, x)
        return lambda: quantized_matmul(x, w.t(), s)
    if c["kind"] == "moe_mxfp4":
        layer = torch.nn.Module()
        for name, t in (("w13_weight", d["w13"]), ("w13_weight_scale", d["s13"]), ("w2_weight", d["w2"]),
                        ("w2_weight_scale", d["s2"]), ("w13_bias", d["b13"]), ("w2_bias", d["b2"])):
            setattr(layer, name, torch.nn.Parameter(t, requires_grad=False))
        layer.moe_config = SimpleNamespace(experts_per_token=c["k"], has_bias=True)
        layer.activation, layer.scoring_func, layer.renormalize = "swigluoai", "softmax", True
        method = Mxfp4MoEMethod(layer.moe_config, mx_activations=False)
        method.process_weights_after_loading(layer)
        d["w13"] = d["s13"] = d["b13"] = None  # de-interleaved copies are the layer's
        logits = d["logits"]
        return lambda: method.apply_monolithic(layer, x, logits)
    if c["kind"] == "moe_fp8":
        layer = _grouped_layer(d["bias"])

        def moe():
            tw, ids = select_experts(x, d["logits"], topk=c["k"], renormalize=True, scoring_fn="sigmoid", layer=layer)
            return fused_moe_gmm(x, d["w13"], d["w2"], d["s13"], d["s2"], None, None, tw, ids, None, c["k"], "silu",
                                 weight_format=c["fmt"])

        return moe
    return lambda: ops.moe_decode_routed(
        x, d["logits"], c["k"], d["w13"], d["w2"], d["s13"], d["s2"], d["sh13"], d["ss13"], d["sh2"], d["ss2"], None,
        scoring_func="sigmoid", renormalize=True, bias=d["bias"], num_expert_group=8, topk_group=4, routed_scale=2.5,
        weight_blocks=128)[0]


def prepare(case, seed):
    d = _linear_inputs(case, seed) if case["kind"] == "linear" else _moe_inputs(case, seed)
    state = dict(call=_call(case, d))
    if case["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            state["call"]()
            torch.cuda.synchronize()
            state["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(state["graph"], stream=side):
                state["out"] = state["call"]()
        torch.cuda.current_stream().wait_stream(side)
    return state


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return state["call"]()


# ---------------------------------------------------------------- work and tolerance


def work(case):
    c = case
    if c["kind"] == "linear":
        M, K, N, fmt = c["M"], c["K"], c["N"], c["fmt"]
        weight = {"fp8": N * K + 4 * N, "int8": N * K + 4 * N, "fp8_blocks": N * K + 4 * (N // 128) * (K // 128),
                  "mxfp4": N * K // 2 + N * K // 32, "nvfp4": N * K // 2 + 2 * N * K // 16, "bf16": 2 * N * K}[fmt]
        return {"bytes": weight + 2 * M * K + 2 * M * N, "flops": 2.0 * M * N * K}
    E, k, H, I, T = c["E"], c["k"], c["H"], c["I"], c["T"]
    expert = 3 * H * I
    expert = expert // 2 + expert // 32 + 4 * (2 * I + H) if c["kind"] == "moe_mxfp4" else expert + 4 * (2 * I + H)
    touched = E * (1.0 - (1.0 - k / E) ** T)  # distinct experts of T tokens, expected
    routes = T * k
    if c["kind"] == "decode_op":
        touched, routes = touched + 1, routes + T
    return {"bytes": touched * expert + 4.0 * T * H + 2.0 * T * E, "flops": 6.0 * routes * H * I}


def tolerance(case):
    """bf16 results of float32 sums taken in another order (other kernels and K
    splits of this framework, the listed cases, measured on MI355X): linears
    move by at most 4e-5 (one bf16 step of a few values in ten thousand, at
    most 0.008 of a value), MoE layers, which round an intermediate to bf16 on
    the way, by 1.4e-4 and 0.012, with an e4m3 intermediate by 2.6e-4 and
    0.017. About four times that is allowed."""
    if case["kind"] == "linear":
        return {"rel": 2e-4, "max": 3.2e-2}
    return {"rel": 6e-4, "max": 5e-2} if case["kind"] == "moe_mxfp4" else {"rel": 1.2e-3, "max": 8e-2}


# ---------------------------------------------------------------- float64 results


def _over(a, b):
    """a / b in float32 with a tensor divisor (a true division)."""
    return a / torch.full_like(a, b)


def _rows_fp8(x, block, guard=True):
    """e4m3 codes per (row, block) of float32 values, decoded: float64 [M, K]."""
    M, K = x.shape
    out = torch.empty((M, K), dtype=torch.float64, device=x.device)
    for b in range(0, K, block):
        v = x[:, b:b + block].float()
        s = _over(v.abs().amax(1, keepdim=True), 448.0)
        if guard:  # runtime linear recipe: divide, a zero scale counts as one
            s = torch.where(s == 0, torch.ones_like(s), s)
            q = (v / s).clamp(-448, 448)
        else:  # fused decode recipe: multiply by the reciprocal, zero rows stay zero
            q = v * torch.where(s == 0, torch.zeros_like(s), torch.ones_like(s) / s)
            q = q.clamp(-448, 448)
        out[:, b:b + block] = q.to(F8).double() * s.double()
    return out


def _rows_int8(x):
    """int8 codes per row in bf16 arithmetic, decoded."""
    s = _over(x.float().abs().amax(1, keepdim=True), 127.0).bfloat16().float()
    s = torch.where(s == 0, torch.ones_like(s), s)
    q = (x.float() / s).bfloat16().float().round().clamp(-128, 127)
    return q.double() * s.double()


def _rows_grouped(x):
    """The grouped matmul's codes: per (row, 512 columns), bf16 arithmetic, decoded."""
    M, K = x.shape
    out = torch.empty((M, K), dtype=torch.float64, device=x.device)
    for b in range(0, K, 512):
        v = x[:, b:b + 512].float()
        s = _over(v.abs().amax(1, keepdim=True), 448.0).bfloat16().float()
        inv = torch.where(s == 0, torch.zeros_like(s), (torch.ones_like(s) / s).bfloat16().float())
        out[:, b:b + 512] = (v * inv).bfloat16().float().to(F8).double() * s.double()
    return out


def _fp4_values(codes):
    lut = torch.tensor([0.0, 0.5, 1, 1.5, 2, 3, 4, 6, -0.0, -0.5, -1, -1.5, -2, -3, -4, -6], device=codes.device,
                       dtype=torch.float64)
    return torch.stack([lut[(codes & 15).long()], lut[(codes >> 4).long()]], -1).flatten(-2)


def _mxfp4_values(codes, s):
    return _fp4_values(codes) * torch.exp2(s.double() - 127.0).repeat_interleave(32, -1)


def _tile_values(codes, s):
    return codes.double() * s.double().repeat_interleave(128, 0).repeat_interleave(128, 1)


def _scores(logits, fn):
    x = logits.double()
    return (torch.softmax(x, -1) if fn == "softmax" else torch.sigmoid(x)).float()


def _top(scores, k):
    """The k best columns, ties to the lowest."""
    return torch.sort(scores, dim=-1, descending=True, stable=True)[1][:, :k]


def _route(c, d):
    """(bf16-valued routing weights, expert ids) of a MoE case."""
    k = c["k"]
    if c["kind"] == "moe_mxfp4":
        s = _scores(d["logits"], "softmax")
        ids = _top(s, k)
        scale = 1.0
    else:
        s = _scores(d["logits"], "sigmoid")
        pick = s + d["bias"][None, :]
        T, E = s.shape
        g = pick.view(T, 8, E // 8)
        best = _top(torch.sort(g, -1, descending=True)[0][..., :2].sum(-1), 4)
        keep = torch.zeros((T, 8), dtype=torch.bool, device=s.device).scatter_(1, best, True)
        ids = _top(torch.where(keep.repeat_interleave(E // 8, 1), pick, torch.full_like(pick, -math.inf)), k)
        scale = 2.5 if c["kind"] == "moe_fp8" else 1.0
    w = s.gather(1, ids)
    w = w / w.sum(-1, keepdim=True).clamp_min(1e-20)
    return (w * scale).bfloat16().double(), ids


def _exact_linear(c, d):
    x, w, s, fmt = d["x"], d["w"], d["s"], c["fmt"]
    if fmt == "fp8":
        return _rows_fp8(x, c["K"]) @ (w.double() * s.double()[:, None]).t()
    if fmt == "int8":
        return _rows_int8(x) @ (w.double() * s.double()[:, None]).t()
    if fmt == "fp8_blocks":
        return _rows_fp8(x, 128) @ _tile_values(w, s).t()
    if fmt == "mxfp4":
        return x.double() @ _mxfp4_values(w, s).t()
    if fmt == "nvfp4":
        return x.double() @ (_fp4_values(w) * s.double().repeat_interleave(16, -1)).bfloat16().double().t()
    return x.double() @ w.double().t()


def _exact_moe(c, d):
    kind, I = c["kind"], c["I"]
    tw, ids = _route(c, d)
    x = d["x"]
    tiles = kind == "decode_op" or c.get("fmt") == "fp8_block"
    if kind == "moe_mxfp4":
        quant = lambda t: t.double()  # noqa: E731
        value = _mxfp4_values
    elif tiles:
        quant = lambda t: _rows_fp8(t, 128, guard=kind != "decode_op")  # noqa: E731
        value = _tile_values
    else:
        quant = _rows_grouped
        value = lambda q, s: q.double() * s.double()[:, None]  # noqa: E731
    xq = quant(x)
    out = torch.zeros((c["T"], c["H"]), dtype=torch.float64, device=x.device)

    def expert(rows, w13, s13, w2, s2, coeff, b13=None, b2=None):
        w1 = value(w13, s13)
        if kind == "moe_mxfp4":
            h = xq[rows] @ w1.t() + b13.double()
            gate, up = h[:, 0::2].clamp(max=7.0), h[:, 1::2].clamp(-7.0, 7.0)
            mid = (up + 1.0) * gate * torch.sigmoid(1.702 * gate)
        else:
            h = xq[rows] @ w1.t()
            mid = torch.nn.functional.silu(h[:, :I]) * h[:, I:]
        if kind == "decode_op":  # the coefficient goes in before the float32 intermediate is quantized
            return quant((mid * coeff).float()) @ value(w2, s2).t()
        y = quant(mid.bfloat16()) @ value(w2, s2).t()
        return (y if b2 is None else y + b2.double()) * coeff

    for e in range(c["E"]):
        rows, slot = (ids == e).nonzero(as_tuple=True)
        if not rows.numel():
            continue
        coeff = tw[rows, slot][:, None] * (2.5 if kind == "decode_op" else 1.0)
        b = (d["b13"][e], d["b2"][e]) if kind == "moe_mxfp4" else ()
        out.index_add_(0, rows, expert(rows, d["w13"][e], d["s13"][e], d["w2"][e], d["s2"][e], coeff, *b))
    if kind == "decode_op":
        rows = torch.arange(c["T"], device=x.device)
        out += expert(rows, d["sh13"], d["ss13"], d["sh2"], d["ss2"], torch.ones((c["T"], 1), device=x.device).double())
    return out


def exact(case, seed):
    if case["kind"] == "linear":
        return _exact_linear(case, _linear_inputs(case, seed))
    return _exact_moe(case, _moe_inputs(case, seed))
