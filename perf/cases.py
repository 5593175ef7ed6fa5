"""The work that a program built on wdl has the library do, one case at a time, through its public entry points.

A case is a dict of plain values. Sizes are those of the quantized Wan block (dim 3072, 24 heads of 128, feed-forward
14336, a 512-token prompt) at 512x928 (464 tokens per latent frame, chunks of 3 frames, a 21-frame window) and
704x1280 (880 tokens per frame), and of a block of half that width; `draw` spreads them over the ranges between.
"""

from __future__ import annotations

import math
import random
import sys
from pathlib import Path

import torch

_PACKAGE = str(Path(__file__).resolve().parents[1] / "wan-dit-lab_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

DEVICE = "cuda"
BF, FP8 = torch.bfloat16, torch.float8_e4m3fn
HEAD, GROUP, RANK, POSITIONS = 128, 64, 32, 1024
GELU_SHIFT = 0.171875
EPS = 1e-6


def listed():
    return [
        # a short prompt's key projection: the smallest W4A4 call, once per prompt and block
        dict(name="linear_prompt", op="linear", tokens=77, inner=3072, outer=3072),
        # the fused Q, K, V projection of a 3-frame chunk at 512x928
        dict(name="linear_qkv_chunk", op="linear", tokens=1392, inner=3072, outer=9216),
        # the feed-forward of one latent frame at 512x928 (frame by frame streaming)
        dict(name="mlp_frame", op="mlp", tokens=464, dim=3072, hidden=14336),
        # the feed-forward of a 3-frame chunk at 704x1280
        dict(name="mlp_hd_chunk", op="mlp", tokens=2640, dim=3072, hidden=14336),
        # one frame over two cached frames: a stream's first seconds
        dict(name="attend_frame", op="attend", tokens=464, cached=928, heads=24, frame=0),
        # a chunk over the full window at 512x928: the steady state of a stream
        dict(name="attend_window", op="attend", tokens=1392, cached=8352, heads=24, frame=0),
        # a chunk over the full window at 704x1280, block-causal per latent frame
        dict(name="attend_hd_framed", op="attend", tokens=2640, cached=15840, heads=24, frame=880),
        # a chunk over the prompt
        dict(name="cross_chunk", op="cross", tokens=1392, keys=512, heads=24),
        # the second feed-forward layer as an FP8 (W8A8) linear
        dict(name="fp8_ffn_down", op="fp8", tokens=1392, inner=14336, outer=3072, rows=False),
        # the mixed-precision model's fused Q, K, V projection at 704x1280: FP8 weights, bf16 activations
        dict(name="fp8_weight_qkv_hd", op="fp8_weight", tokens=2640, inner=3072, outer=9216),
        # the rotation alone with its gradient (a model in training takes it as an operator of its own)
        dict(name="rope_gradient", op="rope", tokens=1392, heads=24, grid="3,16,28", start=5, dtype="float32"),
        # a whole block over a full window, as every denoising step runs it 30 times
        dict(name="block_chunk", op="block", grid="3,16,29", cached=8352, dim=3072, hidden=14336, prompt=512,
             mixed=False),
    ]


def _spread(rng, low, high):
    """A whole number between low and high, even over the logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng: random.Random):
    op = rng.choice(("linear", "linear", "mlp", "mlp", "attend", "attend", "cross", "fp8", "fp8_weight", "rope",
                     "block"))
    dim = rng.choice((1536, 3072, 3072))
    hidden = {1536: 8960, 3072: 14336}[dim]
    if op in ("linear", "fp8", "fp8_weight"):
        inner, outer = rng.choice(((dim, dim), (dim, 3 * dim), (hidden, dim)) if op != "fp8_weight" else
                                  ((dim, dim), (dim, 3 * dim)))
        case = dict(op=op, tokens=_spread(rng, 16, 2640), inner=inner, outer=outer)
        if op == "fp8":
            case["rows"] = rng.random() < 0.5
        return case
    if op == "mlp":
        return dict(op=op, tokens=_spread(rng, 16, 2640), dim=dim, hidden=hidden)
    if op == "attend":
        frames, per_frame = rng.randint(1, 3), _spread(rng, 64, 880)
        cached = 0 if rng.random() < 0.15 else _spread(rng, per_frame, min(15000, 18 * per_frame))
        return dict(op=op, tokens=frames * per_frame, cached=cached, heads=dim // HEAD,
                    frame=per_frame if rng.random() < 0.3 else 0)
    if op == "cross":
        return dict(op=op, tokens=_spread(rng, 64, 2640), keys=_spread(rng, 32, 512), heads=dim // HEAD)
    if op == "rope":
        f, h, w = rng.randint(1, 3), rng.randint(8, 22), rng.randint(8, 40)
        return dict(op=op, tokens=f * h * w + rng.randint(0, 40), heads=dim // HEAD, grid=f"{f},{h},{w}",
                    start=rng.randint(0, 200), dtype=rng.choice(("bfloat16", "float16", "float32")))
    f, h, w = rng.randint(1, 3), rng.randint(8, 16), rng.randint(12, 28)
    return dict(op="block", grid=f"{f},{h},{w}", cached=rng.randint(0, 6) * 3 * h * w, dim=dim, hidden=hidden,
                prompt=_spread(rng, 64, 512), mixed=rng.random() < 0.25)


# ------------------------------------------------------------------------------------------------ inputs

def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _activations(g, tokens, width):
    """Rows of N(0, 1) with one channel in a hundred twenty times as large, as a transformer's residual has them."""
    loud = torch.rand(width, device=DEVICE, generator=g) < 0.01
    x = torch.randn(tokens, width, device=DEVICE, generator=g)
    return torch.where(loud, x * 20, x).to(BF)


def _w4a4(g, outer, inner, shift=0.0):
    """A W4A4 layer in logical form: int4 weights with group scales of an N(0, 0.02^2) weight, low-rank factors,
    per-channel smoothing. shift: the layer after GELU takes its shifted input off the bias."""
    q = torch.randn(outer, inner, device=DEVICE, generator=g).mul_(7 / 3).round_().clamp_(-8, 7).to(torch.int32)
    scales = ((torch.rand(outer, inner // GROUP, device=DEVICE, generator=g) * 0.5 + 0.75) * (0.06 / 7)).to(BF)
    smooth = (torch.rand(inner, device=DEVICE, generator=g) * 1.5 + 0.5).to(BF)
    bias = torch.randn(outer, device=DEVICE, generator=g) * 0.02
    if shift:
        bias -= shift * ((q.view(outer, -1, GROUP) * scales.float()[..., None]).view(outer, inner)
                         / smooth.float()).sum(1)
    return dict(q=q, wscales=scales, smooth=smooth, bias=bias.to(BF),
                proj_down=(torch.randn(inner, RANK, device=DEVICE, generator=g) / inner ** 0.5).to(BF),
                proj_up=(torch.randn(outer, RANK, device=DEVICE, generator=g) * 0.02).to(BF))


def _linear(g, outer, inner):
    layer = torch.nn.Linear(inner, outer, device=DEVICE, dtype=BF)
    with torch.no_grad():
        layer.weight.copy_(torch.randn(outer, inner, device=DEVICE, generator=g) * 0.02)
        layer.bias.copy_(torch.randn(outer, device=DEVICE, generator=g) * 0.02)
    return layer


def _qkv(g, tokens, heads):
    """Q, K, V as views of a fused projection's output, K with the per-channel offset that real keys have."""
    x = torch.randn(3, tokens, heads, HEAD, device=DEVICE, generator=g)
    x[1] += 3 * torch.randn(heads, HEAD, device=DEVICE, generator=g)
    x = x.permute(1, 0, 2, 3).reshape(tokens, 3, heads, HEAD).to(BF)
    return x


def _cache_rows(g, cached, heads):
    rows = _qkv(g, cached, heads)
    return rows[None, :, 1], rows[None, :, 2]


def _table():
    """cos and sin of position x 10000^(-2i/d) for the 22 time, 21 height and 21 width pairs of a head, fp64."""
    parts = []
    for pairs in (22, 21, 21):
        angle = torch.arange(POSITIONS, dtype=torch.float64)[:, None] * \
            10000 ** (-torch.arange(pairs, dtype=torch.float64) / pairs)
        parts.append(torch.stack((torch.cos(angle), torch.sin(angle))))
    return torch.cat(parts, -1).to(DEVICE)


def _grid(case):
    return tuple(int(v) for v in case["grid"].split(","))


BLOCK_LINEARS = ("qkv", "o", "cq", "ck", "cv", "co")


def _block_inputs(case, seed):
    g = _generator(seed)
    dim, hidden, heads = case["dim"], case["hidden"], case["dim"] // HEAD
    f, h, w = _grid(case)
    tokens, cached = f * h * w, case["cached"]
    parts = {}
    for name in BLOCK_LINEARS:
        outer = 3 * dim if name == "qkv" else dim
        if case["mixed"]:
            weight = torch.randn(outer, dim, device=DEVICE, generator=g) * 0.02
            scale = weight.abs().amax(1, keepdim=True) / 448
            parts[name] = dict(fp8=(weight / scale).to(FP8), fp8_scale=scale,
                               bias=(torch.randn(outer, device=DEVICE, generator=g) * 0.02).to(BF))
        else:
            parts[name] = _w4a4(g, outer, dim)
    parts["ffn1"], parts["ffn2"] = _w4a4(g, hidden, dim), _w4a4(g, dim, hidden, GELU_SHIFT)
    for name in ("wq", "wk", "cwq", "cwk"):
        parts[name] = (torch.rand(dim, device=DEVICE, generator=g) * 0.5 + 0.75).to(BF)
    parts["n3w"] = torch.rand(dim, device=DEVICE, generator=g) * 0.5 + 0.75
    parts["n3b"] = torch.randn(dim, device=DEVICE, generator=g) * 0.02
    parts["modulation"] = torch.randn(6, dim, device=DEVICE, generator=g) / dim ** 0.5
    time = torch.randn(6, dim, device=DEVICE, generator=g) * 0.1 + parts["modulation"]
    history = _cache_rows(g, cached, heads) if cached else None
    return dict(parts=parts, e=time, x=_activations(g, tokens, dim), history=history, heads=heads, tokens=tokens,
                prompt=torch.randn(case["prompt"], dim, device=DEVICE, generator=g).to(BF),
                start=cached // (h * w))


def _filled_cache(history, cached, tokens, heads):
    from wdl.kvcache import KVCache

    cache = KVCache(cached, 0, chunk=1)
    cache.allocate(torch.empty(1, tokens, heads, HEAD, device=DEVICE, dtype=BF))
    if cached:
        cache.store(0, *history)
    cache.saved = cached
    return cache


def prepare(case, seed):
    op = case["op"]
    g = _generator(seed)
    if op == "linear":
        from wdl.w4a4 import PackedW4A4Linear, pack_parts

        layer = PackedW4A4Linear(**pack_parts(_w4a4(g, case["outer"], case["inner"]), DEVICE))
        return dict(op=op, layer=layer, x=_activations(g, case["tokens"], case["inner"]))
    if op == "mlp":
        from wdl.w4a4 import PackedW4A4GeluMLP, pack_parts

        first, second = _w4a4(g, case["hidden"], case["dim"]), _w4a4(g, case["dim"], case["hidden"], GELU_SHIFT)
        layer = PackedW4A4GeluMLP(pack_parts(first, DEVICE), pack_parts(second, DEVICE))
        return dict(op=op, layer=layer, x=_activations(g, case["tokens"], case["dim"]))
    if op == "attend":
        tokens, cached, heads = case["tokens"], case["cached"], case["heads"]
        qkv = _qkv(g, tokens, heads)
        history = _cache_rows(g, cached, heads) if cached else None
        return dict(op=op, cache=_filled_cache(history, cached, tokens, heads), frame=case["frame"], tokens=tokens,
                    q=qkv[None, :, 0].contiguous(), k=qkv[None, :, 1].contiguous(), v=qkv[None, :, 2])
    if op == "cross":
        from wdl.ops import attn_bf16_prep_launch

        width = case["heads"] * HEAD
        k, v = (torch.randn(case["keys"], width, device=DEVICE, generator=g).to(BF) for _ in range(2))
        return dict(op=op, q=torch.randn(case["tokens"], width, device=DEVICE, generator=g).to(BF),
                    keys=attn_bf16_prep_launch(k, v))
    if op in ("fp8", "fp8_weight"):
        from wdl.fp8 import DynamicFp8Linear, Fp8Linear, Fp8WeightOnlyLinear

        plain = _linear(g, case["outer"], case["inner"])
        layer = Fp8WeightOnlyLinear(plain) if op == "fp8_weight" else \
            DynamicFp8Linear(plain, rows=True) if case["rows"] else Fp8Linear(plain)
        return dict(op=op, layer=layer, x=_activations(g, case["tokens"], case["inner"]))
    if op == "rope":
        dtype = getattr(torch, case["dtype"])
        shape = (1, case["tokens"], case["heads"], HEAD)
        x, dy = (torch.randn(shape, device=DEVICE, generator=g).to(dtype) for _ in range(2))
        return dict(op=op, x=x.requires_grad_(), dy=dy, grid=[_grid(case)], start=case["start"],
                    table=_table().float())
    from wdl.block import QuantizedWanBlock
    from wdl.w4a4 import pack_parts

    t = _block_inputs(case, seed)
    parts = {name: pack_parts(p, DEVICE) if isinstance(p, dict) and "q" in p else
             dict(p, fp8_scale=p["fp8_scale"].reshape(-1)) if isinstance(p, dict) else p
             for name, p in t["parts"].items()}
    block = QuantizedWanBlock(parts, case["dim"], t["heads"])
    cache = _filled_cache(t["history"], case["cached"], t["tokens"], t["heads"])
    return dict(op=op, block=block, cache=cache, x=t["x"], e=t["e"], grid=_grid(case), table=_table().float(),
                start=t["start"], context=block.prepare_context(t["prompt"]), tokens=t["tokens"])


# ------------------------------------------------------------------------------------------------ one pass

def _written(cache, tokens):
    """The rows of the cache that a pass writes: values and scales of the chunk's keys and values."""
    at = cache.saved
    return [t[:, at:at + tokens] for t in (cache.k, cache.ks, cache.v, cache.vs)]


def run(state):
    op = state["op"]
    if op in ("linear", "mlp", "fp8", "fp8_weight"):
        with torch.no_grad():
            return state["layer"](state["x"])
    if op == "attend":
        cache = state["cache"]
        if not state["frame"]:
            return [cache.attend(state["q"], state["k"], state["v"]), *_written(cache, state["tokens"])]
        from wdl import sage_kv

        # the frame-by-frame mask: the chunk goes into the cache, then attends over the rows before it and itself
        cache.store(cache.saved, state["k"], state["v"])
        out = sage_kv.attend(state["q"], cache.k, cache.ks, cache.v, cache.vs, cache.saved, state["k"], state["v"],
                             frame_tokens=state["frame"])
        return [out, *_written(cache, state["tokens"])]
    if op == "cross":
        from wdl.ops import attn_bf16_launch

        return attn_bf16_launch(state["q"], state["keys"], HEAD ** -0.5)
    if op == "rope":
        from wdl.rope import rope_apply

        y = rope_apply(state["x"], state["grid"], state["table"], state["start"])
        return [y.detach(), torch.autograd.grad(y, state["x"], state["dy"])[0]]
    # the block updates its residual stream in place: each pass starts from the chunk's own
    y = state["block"].forward(state["x"].clone(), state["e"], state["grid"], state["table"], state["start"],
                               state["cache"], state["context"])
    return [y, *_written(state["cache"], state["tokens"])]


# ------------------------------------------------------------------------------------------------ what it takes

def _linear_work(tokens, inner, outer, weight_bits=4):
    low_rank = weight_bits == 4
    return dict(bytes=2 * tokens * (inner + outer) + inner * outer * weight_bits / 8 + 2 * outer +
                (2 * inner * outer / GROUP + 2 * RANK * (inner + outer) + 2 * inner if low_rank else 0),
                flops=2 * tokens * inner * outer + (2 * RANK * tokens * (inner + outer) if low_rank else 0))


def _attend_work(tokens, cached, heads, frame):
    width = heads * HEAD
    seen = tokens * (cached + tokens) if not frame else \
        sum(min(frame, tokens - i) * min(cached + tokens, cached + i + frame) for i in range(0, tokens, frame))
    return dict(bytes=4 * 2 * tokens * width + 2 * (cached + tokens) * heads * (HEAD + 4), flops=4 * seen * width)


def _sum(*works):
    return {key: float(sum(w[key] for w in works)) for key in ("bytes", "flops")}


def work(case):
    op = case["op"]
    if op == "linear":
        return _sum(_linear_work(case["tokens"], case["inner"], case["outer"]))
    if op == "mlp":
        n, d, h = case["tokens"], case["dim"], case["hidden"]
        both = _sum(_linear_work(n, d, h), _linear_work(n, h, d))
        return dict(both, bytes=both["bytes"] - 4 * n * h)  # the hidden layer need not reach memory
    if op == "attend":
        return _sum(_attend_work(case["tokens"], case["cached"], case["heads"], case["frame"]))
    if op == "cross":
        n, keys, width = case["tokens"], case["keys"], case["heads"] * HEAD
        return dict(bytes=4.0 * (n + keys) * width, flops=4.0 * n * keys * width)
    if op in ("fp8", "fp8_weight"):
        bits = 16 if case.get("rows") else 8  # with one scale per row the bf16 weight is quantized on each call
        return _sum(_linear_work(case["tokens"], case["inner"], case["outer"], bits))
    if op == "rope":
        size = 4 if case["dtype"] == "float32" else 2
        values = case["tokens"] * case["heads"] * HEAD
        return dict(bytes=4.0 * size * values, flops=2 * 3.0 * values)
    f, h, w = _grid(case)
    n, d, hidden = f * h * w, case["dim"], case["hidden"]
    bits = 8 if case["mixed"] else 4
    inner = [_linear_work(n, d, o, bits) for o in (3 * d, d, d, d)] + [_linear_work(n, d, hidden),
                                                                      _linear_work(n, hidden, d)]
    weights = sum(v["bytes"] for v in inner) - sum(2 * n * (d + o) for o in (3 * d, d, d, d, hidden, hidden))
    attend, keys = _attend_work(n, case["cached"], d // HEAD, 0), case["prompt"]
    # activations between the layers need not reach memory: the chunk in and out, the weights, the cached rows and
    # the prompt's keys and values do
    return dict(bytes=float(weights + 2 * 2 * n * d + attend["bytes"] - 8 * n * d + 4 * keys * d),
                flops=float(sum(v["flops"] for v in inner) + attend["flops"] + 4 * n * keys * d))


def tolerance(case):
    """About four times what another order of the sums was seen to change (K split over the CUs or not, 5 or 16
    partial sums of the key mean), and room for the 16-bit roundings that such an order turns over by one step."""
    op = case["op"]
    if op == "attend":  # int8 keys: another order of the key mean's sum turns codes over; seen 2.2e-3, at most 0.21
        return {"rel": 1e-2, "max": 0.8}
    if op == "block":   # as attend, through three more layers' int4 codes; seen 6.1e-3, at most 0.1
        return {"rel": 2e-2, "max": 0.4}
    if op == "cross":   # the softmax weights are rounded to bf16 at another reference value
        return {"rel": 4e-3, "max": 5e-2}
    if op == "rope":
        return {"rel": 1e-6, "max": 1e-5} if case["dtype"] == "float32" else {"rel": 2e-3, "max": 2e-2}
    return {"rel": 1e-3, "max": 4e-2}  # bf16 results of fp32 sums: seen 3e-5, one bf16 step at the most


# ------------------------------------------------------------------------------------------------ in 64 bits

def _quantized(x, smooth, shift=0.0):
    """The int4 activations of a layer, in 64 bits: per 64 values one scale, largest / 7 (after GELU: shifted,
    largest / 15) rounded to bf16."""
    v = (x + shift) / smooth.double()
    g = v.view(v.shape[0], -1, GROUP)
    low, high = (0, 15) if shift else (-8, 7)
    scale = (g.abs().amax(-1, keepdim=True) / high).to(BF).double()
    return (torch.round(g / torch.where(scale > 0, scale, 1)).clamp(low, high) * scale).view_as(v)


def _exact_w4a4(x, t, shift=0.0):
    weight = (t["q"].view(t["q"].shape[0], -1, GROUP) * t["wscales"].double()[..., None]).view(t["q"].shape)
    return _quantized(x, t["smooth"], shift) @ weight.t() + \
        (x @ t["proj_down"].double()) @ t["proj_up"].double().t() + t["bias"].double()


def _exact_mlp(x, first, second):
    h = torch.nn.functional.gelu(_exact_w4a4(x, first), approximate="tanh")
    return _exact_w4a4(h, second, GELU_SHIFT)


def _to_fp8(x, **side):
    """(e4m3 values, scale) with the largest magnitude at 448: the scale and the quotients rounded to fp32 once. With
    one scale for the whole tensor the quotients have x's type, as torch's x / scale does."""
    scale = (x.double().abs().amax(**side).clamp(min=1e-12) / 448).float()
    y = (x.double() / scale.double()).float()
    return (y if side else y.to(x.dtype)).to(FP8), scale


def _exact_rows(x):
    """FP8 rows as a cache keeps them."""
    return _to_fp8(x, dim=-1, keepdim=True)


def _exact_attention(q, k, v, frame=0, cached=0):
    """q [n, heads, 128] over k, v [L, heads, 128], all fp64; frame: query i sees the keys before its frame's end."""
    n, heads, _ = q.shape
    hidden = None
    if frame:
        end = cached + (torch.arange(n, device=q.device) // frame + 1) * frame
        hidden = torch.arange(k.shape[0], device=q.device)[None, :] >= end[:, None]
    out = torch.empty_like(q)
    for h in range(heads):
        s = q[:, h] @ k[:, h].t() * HEAD ** -0.5
        if hidden is not None:
            s.masked_fill_(hidden, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, h]
    return out


def _with_history(history, k, v):
    """Keys and values of a chunk behind the cached rows, which hold FP8."""
    if history is None:
        return k, v
    rows = []
    for old in history:
        codes, scale = _exact_rows(old[0])
        rows.append(codes.double() * scale.double())
    return torch.cat([rows[0], k]), torch.cat([rows[1], v])


def _exact_rope(x, grid, start, table, inverse=False):
    """x [tokens, heads, 128] fp64; the rows past the grid are copied."""
    f, h, w = grid
    i = torch.arange(f * h * w, device=x.device)
    at = torch.stack((start + i // (h * w), i // w % h, i % w))
    which = torch.tensor([0] * 22 + [1] * 21 + [2] * 21, device=x.device)
    cos, sin = table.double()[:, at[which].t(), torch.arange(64, device=x.device)][:, :, None]
    sin = -sin if inverse else sin
    even, odd = x[:len(i), :, ::2], x[:len(i), :, 1::2]
    turned = torch.stack((even * cos - odd * sin, odd * cos + even * sin), -1).flatten(-2)
    return torch.cat((turned, x[len(i):]))


def _exact_fp8(x, layer, rows, weight_only):
    side = dict(dim=1, keepdim=True) if rows else {}
    dense = lambda t: torch.mul(*(v.double() for v in _to_fp8(t, **side)))  # noqa: E731
    x = x.double() if weight_only else dense(x)
    return x @ dense(layer.weight.detach()).t() + layer.bias.detach().double()


def _norm(x):
    return torch.nn.functional.layer_norm(x, (x.shape[1],), eps=EPS)


def _rms(x, weight):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * weight.double()


def _exact_block(case, seed):
    t = _block_inputs(case, seed)
    p, heads, table = t["parts"], t["heads"], _table().float()
    shift_a, scale_a, gate_a, shift_f, scale_f, gate_f = t["e"].double()

    def linear(x, name):
        part = p[name]
        if "fp8" not in part:
            return _exact_w4a4(x, part)
        return x @ (part["fp8"].double() * part["fp8_scale"].double()).t() + part["bias"].double()

    split = lambda x: x.view(x.shape[0], heads, HEAD)  # noqa: E731
    x = t["x"].double()
    q, k, v = linear(_norm(x) * (1 + scale_a) + shift_a, "qkv").chunk(3, 1)
    q, k = (_exact_rope(split(_rms(y, p[w])), _grid(case), t["start"], table) for y, w in ((q, "wq"), (k, "wk")))
    v = split(v)
    rows = []
    for y in (k, v):
        scale = y.abs().amax(-1, keepdim=True) / 448
        rows += [(y / scale).float().to(FP8).double()[None], scale[None]]
    x = x + linear(_exact_attention(q, *_with_history(t["history"], k, v)).flatten(1), "o") * gate_a
    context = t["prompt"].double()
    ck, cv = _rms(linear(context, "ck"), p["cwk"]), linear(context, "cv")
    cq = _rms(linear(_norm(x) * p["n3w"].double() + p["n3b"].double(), "cq"), p["cwq"])
    x = x + linear(_exact_attention(split(cq), split(ck), split(cv)).flatten(1), "co")
    return [x + _exact_mlp(_norm(x) * (1 + scale_f) + shift_f, p["ffn1"], p["ffn2"]) * gate_f, *rows]


@torch.no_grad()
def exact(case, seed):
    op = case["op"]
    g = _generator(seed)
    if op == "linear":
        t = _w4a4(g, case["outer"], case["inner"])
        return _exact_w4a4(_activations(g, case["tokens"], case["inner"]).double(), t)
    if op == "mlp":
        first, second = _w4a4(g, case["hidden"], case["dim"]), _w4a4(g, case["dim"], case["hidden"], GELU_SHIFT)
        return _exact_mlp(_activations(g, case["tokens"], case["dim"]).double(), first, second)
    if op == "attend":
        qkv = _qkv(g, case["tokens"], case["heads"])
        history = _cache_rows(g, case["cached"], case["heads"]) if case["cached"] else None
        q, k, v = qkv.double().unbind(1)
        out = _exact_attention(q, *_with_history(history, k, v), case["frame"], case["cached"])
        (kc, ks), (vc, vs) = _exact_rows(qkv[None, :, 1]), _exact_rows(qkv[None, :, 2])
        return [out[None], kc.double(), ks.double(), vc.double(), vs.double()]
    if op == "cross":
        width = case["heads"] * HEAD
        k, v = (torch.randn(case["keys"], width, device=DEVICE, generator=g).to(BF) for _ in range(2))
        q = torch.randn(case["tokens"], width, device=DEVICE, generator=g).to(BF)
        return _exact_attention(*(t.double().view(-1, case["heads"], HEAD) for t in (q, k, v))).flatten(1)
    if op in ("fp8", "fp8_weight"):
        layer = _linear(g, case["outer"], case["inner"])
        x = _activations(g, case["tokens"], case["inner"])
        return _exact_fp8(x, layer, op == "fp8_weight" or case["rows"], op == "fp8_weight")
    if op == "rope":
        dtype = getattr(torch, case["dtype"])
        shape = (1, case["tokens"], case["heads"], HEAD)
        x, dy = (torch.randn(shape, device=DEVICE, generator=g).to(dtype).double()[0] for _ in range(2))
        table = _table().float()
        return [_exact_rope(x, _grid(case), case["start"], table)[None],
                _exact_rope(dy, _grid(case), case["start"], table, inverse=True)[None]]
    return _exact_block(case, seed)
