"""Performance cases of the NF5 path: what a program built on ``axs.unified`` calls.

``listed()`` names fixed cases, ``draw()`` gives others of the same ranges,
``prepare()`` makes what a program holds before the call, ``run()`` is one pass
through the public entry points and ``exact()`` is the same result from plain
torch in 64 bits (the fake-quantized operands, which are exact 32-bit values,
contracted and summed in float64).

Kinds of work:
  fq     fake_quantize_unified forward and its straight-through backward
  codec  quantize_unified, then dequantize_unified (stored weights)
  wire   the 6.25-bit gradient buffer, packed and unpacked
  infer  the quantized linear without gradients (module or backend call)
  train  the quantized linear, forward and backward
  norm   AXSLayerNormUnified, forward and backward
  model  a decoder's training pass, forward, loss and backward, in a HIP graph
"""
from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn as nn
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "axs-6_amd"))

import axs.unified as axu  # noqa: E402
from axs.unified.distributed import pack_gradient_to_buffer, unpack_buffer_to_gradient  # noqa: E402

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
SIZE = {"f32": 4, "bf16": 2, "f16": 2}

# accelerated_linear keeps 16-bit operands' fake-quantized values in 32 bits up
# to this many outputs and rounds them to the operand's type above
FUSED_OUTPUTS = 128 * 1024


def listed() -> list[dict]:
    return [
        # the smallest call: a 256 x 256 layer's values, forward and backward; launches count
        dict(name="fq_256x256", kind="fq", rows=256, cols=256, dtype="f32", block=32, rounding="nearest"),
        # a large activation tensor with outliers, the benchmark's headline shape
        dict(name="fq_8192x4096", kind="fq", rows=8192, cols=4096, dtype="f32", block=32, rounding="nearest"),
        # stochastic rounding of 16-bit gradients whose rows end in a partial block
        dict(name="fq_stochastic_odd_bf16", kind="fq", rows=8192, cols=4095, dtype="bf16", block=32,
             rounding="stochastic"),
        # a feed-forward weight stored as exponents, codes and signs, and read back
        dict(name="codec_11008x4096", kind="codec", rows=11008, cols=4096, dtype="f32", block=32),
        # the same layer's gradient as it goes over the wire
        dict(name="wire_11008x4096", kind="wire", rows=11008, cols=4096, dtype="f32", block=32),
        # token-by-token generation through a converted model's layer
        dict(name="decode_1", kind="infer", via="module", M=1, K=4096, N=11008, dtype="f32", bias=True),
        # a batch of sequences generating at once, 16-bit weights
        dict(name="decode_32_bf16", kind="infer", via="backend", M=32, K=4096, N=4096, dtype="bf16", bias=False),
        # a short prompt through a 16-bit feed-forward layer
        dict(name="prefill_256_bf16", kind="infer", via="module", M=256, K=4096, N=11008, dtype="bf16", bias=True),
        # the linear's headline shape
        dict(name="forward_4096", kind="infer", via="backend", M=4096, K=4096, N=4096, dtype="f32", bias=True),
        # a feed-forward layer of a large model in training
        dict(name="train_8192x4096x11008", kind="train", M=8192, K=4096, N=11008, dtype="f32", block=32, bias=True),
        # the norm in front of such a layer
        dict(name="norm_8192x4096", kind="norm", rows=8192, cols=4096, dtype="f32"),
        # a small decoder's whole training pass (4 layers of width 256, 64 sequences of 128 tokens)
        dict(name="minigpt", kind="model", batch=64, context=128, width=256, heads=4, layers=4, ff=1024, vocab=256),
    ]


def _log(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo: int, hi: int) -> int:
    """A feature size: mostly whole blocks, sometimes any number."""
    v = _log(rng, lo, hi)
    return v if rng.random() < 0.25 else max(32, v // 32 * 32)


def draw(rng) -> dict:
    kind = rng.choice(["fq", "fq", "codec", "wire", "infer", "infer", "infer", "train", "train", "norm", "model"])
    dtype = rng.choice(["f32", "f32", "bf16", "bf16", "f16"])
    if kind in ("fq", "codec", "wire", "norm"):
        cols = _width(rng, 64, 16384)
        rows = _log(rng, 64, max(65, min(65536, (45 << 20) // cols)))
        case = dict(kind=kind, rows=rows, cols=cols, dtype=dtype)
        if kind != "norm":
            case["block"] = rng.choice([8, 16, 32, 32, 32])
        if kind == "fq":
            case["rounding"] = rng.choice(["nearest", "nearest", "stochastic"])
        return case
    if kind == "infer":
        M = _log(rng, 1, 64) if rng.random() < 0.5 else _log(rng, 64, 8192)
        return dict(kind="infer", via=rng.choice(["module", "backend"]), M=M, K=_width(rng, 256, 11008),
                    N=_width(rng, 256, 11008), dtype=dtype, bias=rng.random() < 0.5)
    if kind == "train":
        return dict(kind="train", M=_log(rng, 64, 8192), K=_width(rng, 256, 8192), N=_width(rng, 256, 5504),
                    dtype=dtype, block=rng.choice([16, 32, 32, 32]), bias=rng.random() < 0.5)
    width = 64 * rng.randint(2, 6)
    return dict(kind="model", batch=rng.randint(4, 64), context=_log(rng, 32, 128), width=width, heads=width // 64,
                layers=rng.randint(1, 4), ff=4 * width, vocab=rng.choice([256, 1000, 4096]))


# ---- the decoder ------------------------------------------------------------------


class Block(nn.Module):
    def __init__(self, width: int, heads: int, ff: int) -> None:
        super().__init__()
        self.heads = heads
        self.ln1, self.ln2 = nn.LayerNorm(width), nn.LayerNorm(width)
        self.qkv, self.out = nn.Linear(width, 3 * width), nn.Linear(width, width)
        self.up, self.down = nn.Linear(width, ff), nn.Linear(ff, width)

    def forward(self, x, mask):
        B, T, D = x.shape
        q, k, v = self.qkv(self.ln1(x)).reshape(B, T, 3, self.heads, -1).permute(2, 0, 3, 1, 4).contiguous()
        s = torch.matmul(q, k.transpose(-2, -1).contiguous()) * (D // self.heads) ** -0.5 + mask
        o = torch.matmul(F.softmax(s, dim=-1), v).transpose(1, 2).reshape(B, T, D)
        x = x + self.out(o)
        return x + self.down(F.gelu(self.up(self.ln2(x))))


class Decoder(nn.Module):
    def __init__(self, c: dict) -> None:
        super().__init__()
        self.embed = nn.Embedding(c["vocab"], c["width"])
        self.pos = nn.Parameter(torch.zeros(1, c["context"], c["width"]))
        self.blocks = nn.ModuleList(Block(c["width"], c["heads"], c["ff"]) for _ in range(c["layers"]))
        self.ln = nn.LayerNorm(c["width"])
        self.head = nn.Linear(c["width"], c["vocab"], bias=False)

    def forward(self, idx, mask):
        x = self.embed(idx) + self.pos
        for b in self.blocks:
            x = b(x, mask)
        return self.head(self.ln(x))


def _decoder(c: dict, seed: int) -> tuple[Decoder, torch.Tensor, torch.Tensor]:
    """A decoder with seeded weights on the GPU, its tokens and its causal mask."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    with torch.device("cuda"):
        model = Decoder(c)
    with torch.no_grad():
        for name, p in model.named_parameters():
            if p.dim() > 1:
                p.normal_(0.0, 0.02, generator=g)
            elif name.endswith("weight"):
                p.fill_(1.0)
            else:
                p.zero_()
    tokens = torch.randint(0, c["vocab"], (c["batch"], c["context"] + 1), generator=g, device="cuda")
    mask = torch.full((c["context"], c["context"]), float("-inf"), device="cuda").triu(1)
    return model, tokens, mask


def _pass(model, tokens, mask):
    logits = model(tokens[:, :-1], mask)
    loss = F.cross_entropy(logits.reshape(-1, logits.shape[-1]), tokens[:, 1:].reshape(-1))
    grads = torch.autograd.grad(loss, [model.pos, *(p for n, p in model.named_parameters() if n != "pos")])
    return logits, loss, grads


# ---- prepare and run --------------------------------------------------------------


def _normal(g, *shape, std=1.0, dtype="f32"):
    return (torch.randn(*shape, generator=g, device="cuda") * std).to(DTYPES[dtype])


def prepare(case: dict, seed: int) -> dict:
    g = torch.Generator(device="cuda").manual_seed(seed)
    k, s = case["kind"], {"case": case, "seed": seed}
    if k == "model":
        # recorded once, as a program with launch-bound steps does; the gradient is rounded to nearest, so that a
        # replay gives the same result again
        model, tokens, mask = _decoder(case, seed)
        model = axu.convert_to_axs_unified(model, quantize_grad=False, inplace=True)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _pass(model, tokens, mask)
        torch.cuda.current_stream().wait_stream(side)
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["out"] = _pass(model, tokens, mask)
        s["keep"] = (model, tokens, mask)
        return s
    d = case["dtype"]
    if k in ("fq", "codec", "wire", "norm"):
        r, c = case["rows"], case["cols"]
        if k == "fq":
            # activations with one value in a hundred scaled up, which spreads the block exponents
            x = torch.randn(r, c, generator=g, device="cuda")
            x.mul_(torch.where(torch.rand(r, c, generator=g, device="cuda") < 0.01, 100.0, 1.0))
            s.update(x=x.to(DTYPES[d]).requires_grad_(), dy=_normal(g, r, c, dtype=d))
        elif k == "norm":
            m = axu.AXSLayerNormUnified(c).to("cuda", DTYPES[d])
            with torch.no_grad():
                m.weight.copy_(1.0 + 0.1 * torch.randn(c, generator=g, device="cuda"))
                m.bias.copy_(0.1 * torch.randn(c, generator=g, device="cuda"))
            s.update(x=_normal(g, r, c, dtype=d).requires_grad_(), dy=_normal(g, r, c, dtype=d), module=m)
        else:
            s.update(x=_normal(g, r, c, std=0.02 if k == "codec" else 1e-3, dtype=d))
        return s
    M, K, N = case["M"], case["K"], case["N"]
    x, w = _normal(g, M, K, dtype=d), _normal(g, N, K, std=K ** -0.5, dtype=d)
    b = _normal(g, N, std=0.1, dtype=d) if case["bias"] else None
    if k == "train":
        s.update(x=x.requires_grad_(), w=w.requires_grad_(), b=None if b is None else b.requires_grad_(),
                 dy=_normal(g, M, N, dtype=d))
    elif case["via"] == "module":
        with torch.device("meta"):
            m = axu.AXSLinearUnified(K, N, bias=case["bias"])
        m.weight = nn.Parameter(w)
        if b is not None:
            m.bias = nn.Parameter(b)
        s.update(x=x, module=m.eval())
    else:
        s.update(x=x, w=w, b=b)
    return s


def run(s: dict):
    c = s["case"]
    k = c["kind"]
    if k == "model":
        s["graph"].replay()
        return s["out"]
    if k == "fq":
        if c["rounding"] == "stochastic":
            torch.default_generator.manual_seed(s["seed"])  # the draw's seed comes from torch's CPU generator
        y = axu.fake_quantize_unified(s["x"], c["block"], c["rounding"])
        return y, torch.autograd.grad(y, s["x"], s["dy"])[0]
    if k == "codec":
        q = axu.quantize_unified(s["x"], c["block"])
        return q.shared_exponents, q.signs, q.magnitudes, axu.dequantize_unified(q)
    if k == "wire":
        buf = pack_gradient_to_buffer(s["x"], c["block"])
        return buf, unpack_buffer_to_gradient(buf, s["x"].shape, c["block"])
    if k == "norm":
        m = s["module"]
        y = m(s["x"])
        return (y, *torch.autograd.grad(y, (s["x"], m.weight, m.bias), s["dy"]))
    if k == "infer":
        with torch.no_grad():
            return s["module"](s["x"]) if c["via"] == "module" else axu.accelerated_linear(s["x"], s["w"], s["b"])
    torch.default_generator.manual_seed(s["seed"])  # of the stochastic rounding of the output gradient
    y = axu.axs_linear_unified(s["x"], s["w"], s["b"], c["block"])
    wrt = (s["x"], s["w"]) + (() if s["b"] is None else (s["b"],))
    return (y, *torch.autograd.grad(y, wrt, s["dy"]))


def work(case: dict) -> dict:
    k = case["kind"]
    if k == "model":
        T, W, L = case["batch"] * case["context"], case["width"], case["layers"]
        lin = L * (4 * W * W + 2 * W * case["ff"]) + W * case["vocab"]
        par = lin + L * (9 * W + case["ff"]) + (case["vocab"] + case["context"] + 2) * W
        return {"flops": 6 * T * lin + 12 * L * T * case["context"] * W, "bytes": 8 * par + 4 * T * case["vocab"]}
    e = SIZE[case["dtype"]]
    if k in ("infer", "train"):
        M, K, N = case["M"], case["K"], case["N"]
        if k == "infer":
            return {"flops": 2 * M * N * K, "bytes": e * (M * K + N * K + M * N)}
        return {"flops": 6 * M * N * K, "bytes": 2 * e * (M * K + N * K + M * N)}
    n = case["rows"] * case["cols"]
    if k == "fq":
        return {"bytes": 2 * e * n}  # the backward hands its input on
    if k == "norm":
        return {"bytes": 5 * e * n}
    blocks = case["rows"] * -(-case["cols"] // case["block"])
    # written once and read back once
    stored = blocks * (1 + 2 * case["block"]) if k == "codec" else blocks * (1 + case["block"] * 3 // 4)
    return {"bytes": e * n + 2 * stored + 4 * n}


def tolerance(case: dict):
    k, d = case["kind"], case.get("dtype")
    if k in ("fq", "codec", "wire"):
        return "exact"  # every value is defined to the last bit
    if k == "model":
        # a rounding of one layer moves values over a quantization step of the next
        return {"rel": 0.03, "max": 0.9}
    if k == "norm":
        return {"rel": 4e-6} if d == "f32" else {"rel": 8e-3 if d == "bf16" else 1e-3}
    if d == "bf16":
        return {"rel": 8e-3}  # one rounding of the result: 1.7e-3
    if k == "infer" and case["via"] == "backend" and case["M"] * case["N"] <= FUSED_OUTPUTS:
        return {"rel": 4e-6 if d == "f32" else 1e-3}
    return {"rel": 1.4e-3}  # operands rounded to 11 bits: 3.2e-4


# ---- the same in 64 bits ------------------------------------------------------------

# the format's 32 levels (float32 bit patterns)
_LEVELS = (
    0x3C04B96E, 0x3CC7303E, 0x3D26292A, 0x3D68FC26, 0x3D96163B, 0x3DB7EB43, 0x3DDA0C14, 0x3DFC887B,
    0x3E0FB8B1, 0x3E216C8A, 0x3E3369C5, 0x3E45BB68, 0x3E586DBB, 0x3E6B8E8E, 0x3E7F2D9B, 0x3E89AE7A,
    0x3E9418D0, 0x3E9EE22E, 0x3EAA1958, 0x3EB5D02B, 0x3EC21CA7, 0x3ECF1A59, 0x3EDCEC91, 0x3EEBC1B0,
    0x3EFBD888, 0x3F06C4BE, 0x3F10AB83, 0x3F1C0741, 0x3F2988AE, 0x3F3A8BF4, 0x3F5273DC, 0x3F800000)


def _uniform(seed: int, n: int, device) -> torch.Tensor:
    """The n draws of a call whose seed torch's CPU generator gives after manual_seed(seed)."""
    word = 0xFFFFFFFFFFFFFFFF
    z = int(torch.randint(0, 2 ** 62, (1,), generator=torch.Generator().manual_seed(seed)))
    z = (z + 0x9E3779B97F4A7C15) & word
    z = ((z ^ z >> 30) * 0xBF58476D1CE4E5B9) & word
    z = ((z ^ z >> 27) * 0x94D049BB133111EB) & word
    z ^= z >> 31
    m = 0xFFFFFFFF
    h = torch.arange(n, dtype=torch.int64, device=device) ^ (z & m) ^ (z >> 32)
    h = h ^ h >> 16
    h = (h * 0x7FEB352D) & m
    h = h ^ h >> 15
    h = (h * 0x846CA68B) & m
    h = h ^ h >> 16
    return (h >> 8).float() * 2.0 ** -24


def _blocks(x, block: int, u=None):
    """(index into the 1024 steps, sign, block scale) of x's blocks."""
    x = x.detach().float()
    rows = x.reshape(-1, x.shape[-1])
    pad = -rows.shape[-1] % block
    v = F.pad(rows, (0, pad)).reshape(rows.shape[0], -1, block)
    amax = v.abs().amax(-1, keepdim=True)
    # the logarithm is rounded to float32 before its floor
    e = amax.double().clamp(min=1e-45).log2().float().floor().double() + 1.0
    scale = torch.where(amax == 0, 1.0, torch.exp2(e)).float()
    n = (v.abs() / scale).clamp(0.0, 1.0)
    if u is not None:
        # by a tensor: torch divides by a plain number with its reciprocal
        d = (u.reshape(rows.shape) - 0.5) / torch.full((), 1023.0, device=u.device)
        n = n + F.pad(d, (0, pad)).reshape(v.shape)
    return (n * 1023.0).int().clamp(0, 1023), v, scale


def _codes(device):
    levels = torch.tensor(_LEVELS, dtype=torch.int32).view(torch.float32)
    mid = (levels[:-1].double() + levels[1:].double()) / 2
    code = torch.bucketize(torch.linspace(0, 1, 1024, dtype=torch.float64), mid)
    return code.to(device), levels.to(device)


def _fq(x, block: int, u=None, keep: bool = False):
    """The fake-quantized x in float64, rounded to x's type unless `keep`."""
    i, v, scale = _blocks(x, block, u)
    code, levels = _codes(x.device)
    q = (v.sign() * levels[code[i.long()]] * scale).reshape(v.shape[0], -1)[:, : x.shape[-1]].reshape(x.shape)
    if not keep and x.dtype in (torch.bfloat16, torch.float16):
        q = q.to(x.dtype)
    return q.double()


class _ExactLinear(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w, b):
        xq, wq = _fq(x, 32), _fq(w, 32)
        ctx.save_for_backward(xq, wq)
        return F.linear(xq, wq, b)

    @staticmethod
    def backward(ctx, dy):
        xq, wq = ctx.saved_tensors
        d, x2 = dy.reshape(-1, dy.shape[-1]), xq.reshape(-1, xq.shape[-1])
        return dy @ wq, d.t() @ x2, d.sum(0) if ctx.needs_input_grad[2] else None


class _ExactEmbed(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        return _fq(x, 32)

    @staticmethod
    def backward(ctx, dy):
        return dy


def exact(case: dict, seed: int):
    k = case["kind"]
    if k == "model":
        model, tokens, mask = _decoder(case, seed)
        model, mask = model.double(), mask.double()
        for m in model.modules():
            if isinstance(m, nn.Linear):
                m.forward = lambda x, m=m: _ExactLinear.apply(x, m.weight, m.bias)
            elif isinstance(m, nn.Embedding):
                m.forward = lambda t, m=m: _ExactEmbed.apply(F.embedding(t, m.weight))
        logits, loss, grads = _pass(model, tokens, mask)
        return logits.detach(), loss.detach(), grads
    if k == "norm":
        s = prepare(case, seed)
        m = s["module"]
        x, w, b = (t.detach().double().requires_grad_() for t in (s["x"], m.weight, m.bias))
        y = F.layer_norm(x, (case["cols"],), w, b, m.eps)
        return (y.detach(), *torch.autograd.grad(y, (x, w, b), s["dy"].double()))
    s = prepare(case, seed)
    if k == "fq":
        u = _uniform(seed, s["x"].numel(), "cuda") if case["rounding"] == "stochastic" else None
        return _fq(s["x"], case["block"], u), s["dy"].double()
    if k in ("codec", "wire"):
        i, v, scale = _blocks(s["x"], case["block"])
        code, levels = _codes(v.device)
        # the stored form keeps the level of the value itself and an exponent of 8 bits
        y = (v.sign() + (v == 0)) * levels[code[i.long()]].double() * scale
        y = y.reshape(v.shape[0], -1)[:, : case["cols"]].reshape(s["x"].shape)
        return (None, None, None, y) if k == "codec" else (None, y)
    if k == "infer":
        m = s.get("module")
        w, b = (m.weight, m.bias) if m is not None else (s["w"], s["b"])
        # 16-bit operands: see FUSED_OUTPUTS
        keep = m is None and case["M"] * case["N"] <= FUSED_OUTPUTS
        return F.linear(_fq(s["x"], 32, keep=keep), _fq(w, 32, keep=keep),
                        None if b is None else b.detach().double()).detach()
    xq, wq = _fq(s["x"], case["block"]), _fq(s["w"], case["block"])
    dyq = _fq(s["dy"], case["block"], _uniform(seed, s["dy"].numel(), "cuda"))
    y = F.linear(xq, wq, None if s["b"] is None else s["b"].detach().double())
    return (y, dyq @ wq, dyq.t() @ xq) + (() if s["b"] is None else (dyq.sum(0),))
