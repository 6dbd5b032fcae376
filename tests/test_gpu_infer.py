"""The linear without gradients (``axs_linear_unified`` under ``no_grad`` and
``accelerated_linear``), which takes the library's inference forms where it has
one for the shape: FQ values in the operands' type, as the training forward.

Bars, rel-L2 against the fp64 product of the oracle's FQ operands rounded to
the operands' type: the output's rounding, at most its unit roundoff per value
(2^-9 bf16, 2^-11 f16), on top of the operands' -- none for 16-bit types, whose
FQ values the 16-bit operands hold exactly, and for f32 the 11-bit rounding of
both packed operands, 1e-3 (3.2e-4 measured)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
BAR = {torch.float32: 1e-3, torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -11}


def _inputs(m, K, N, dt, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(m, K, generator=g)
    x[torch.rand(m, K, generator=g) < 0.01] *= 100.0
    x[:, 5] = 0.0
    w = torch.randn(N, K, generator=g) * K ** -0.5
    w[:, 3] = 0.0
    return x.to(dt), w.to(dt), torch.randn(N, generator=g).to(dt)


def _exact(x, w, b):
    def q(t):
        return torch.from_numpy(oracle.fake_quantize(t.float().numpy(), 32)).to(t.dtype).double()

    y = q(x) @ q(w).t()
    return y if b is None else y + b.double()


def _infer(x, w, b):
    from axs.unified import functional_unified as fu

    with torch.no_grad():
        return fu.axs_linear_unified(x.to(DEV), w.to(DEV), None if b is None else b.to(DEV))


def _form(m, K, N, dt):
    from axs import _lib

    return _lib.lib().axs6_nf5_linear_infer_workspace(m, N, K, _lib.DTYPE_CODE[dt], 32) >= 0


# one and two rows: a row step's edges, K split over two waves (16+ steps, or
# 8+ with few rows), ragged last steps and row counts
@pytest.mark.parametrize("dt", list(BAR), ids=str)
@pytest.mark.parametrize("m,K,N", [(1, 32, 1), (2, 512, 7), (1, 544, 300), (2, 4096, 1030), (1, 8192, 257),
                                   (2, 4608, 2050)])
def test_infer_streamed_rows(m, K, N, dt):
    print(f"[infer {dt} m={m} K={K} N={N}]", flush=True)
    x, w, b = _inputs(m, K, N, dt, K + N + m)
    assert _form(m, K, N, dt)
    y = _infer(x, w, b)
    assert y.dtype == dt and y.shape == (m, N) and not y.requires_grad
    assert oracle.rel_l2(y.float().cpu().numpy(), _exact(x, w, b)) <= BAR[dt]


# the weight quantized inside the GEMM: every row tile (32, 64, 128, 256) at its
# edges, ragged column tiles, N off the 4-value store, K ending in half a step,
# K split over workgroups and (the last) not
@pytest.mark.parametrize("dt", list(BAR), ids=str)
@pytest.mark.parametrize("m,K,N", [(3, 1056, 4030), (32, 4096, 1024), (33, 2080, 2051), (64, 1024, 4224),
                                   (65, 4128, 2049), (128, 8192, 1027), (129, 2048, 4096), (256, 3104, 2710),
                                   (5, 1024, 65540), (1, 14336, 2050), (2, 11008, 1027), (2, 6176, 4096)])
def test_infer_gemm(m, K, N, dt):
    print(f"[infer gemm {dt} m={m} K={K} N={N}]", flush=True)
    x, w, b = _inputs(m, K, N, dt, K + N + m)
    assert _form(m, K, N, dt) or (dt == torch.float32 and m > 128)
    y = _infer(x, w, b)
    assert y.dtype == dt and y.shape == (m, N)
    assert oracle.rel_l2(y.float().cpu().numpy(), _exact(x, w, b)) <= BAR[dt]
    assert torch.equal(_infer(x, w, b), y)     # fixed summation order


@pytest.mark.parametrize("dt", list(BAR), ids=str)
def test_infer_gemm_raw_input(dt):
    from axs.unified import functional_unified as fu

    x, w, _ = _inputs(48, 1024, 4096, dt, 2)
    assert _form(48, 1024, 4096, dt)
    with torch.no_grad():
        y = fu.axs_linear_unified(x.to(DEV), w.to(DEV), None, 32, False)
    wq = torch.from_numpy(oracle.fake_quantize(w.float().numpy(), 32)).to(dt).double()
    assert oracle.rel_l2(y.float().cpu().numpy(), x.double() @ wq.t()) <= BAR[dt]


@pytest.mark.parametrize("dt", list(BAR), ids=str)
@pytest.mark.parametrize("m,N", [(2, 64), (20, 4160), (100, 8200)])
def test_infer_special_blocks(m, N, dt):
    """NaN, inf, tiny, huge and part-subnormal blocks of the weight."""
    K = 1024
    assert _form(m, K, N, dt)
    x, w, _ = _inputs(m, K, N, dt, 4)
    big, small, sub = (1e3, 1e-3, 1e-7) if dt == torch.float16 else (1e30, 1e-33, 1e-41)
    w = w.float()
    w[3, 100] = float("nan")
    w[4, 64:96] = w[4, 64:96].abs() + 0.1
    w[4, 70] = float("inf")
    w[5] *= small
    w[6] *= big
    w[7, 0:32] = sub
    w[7, 3] = 0.5
    w = w.to(dt)
    y = _infer(x, w, None).float().cpu().numpy()
    with np.errstate(invalid="ignore", over="ignore"):
        want = _exact(x, w, None).numpy()
    assert np.array_equal(np.isnan(y), np.isnan(want)) and np.array_equal(np.isinf(y), np.isinf(want))
    for c in (0, 5, 6, 7):       # each row against its own scale
        assert oracle.rel_l2(y[:, c], want[:, c]) <= 2 * BAR[dt], c


def test_infer_keeps_the_training_path_under_grad():
    """A recorded gradient takes the training forward, bit for bit."""
    from axs.unified import functional_unified as fu, hip_linear

    x, w, b = (t.to(DEV) for t in _inputs(2, 256, 96, torch.float32, 9))
    want = hip_linear.forward_train(x, w, b)[0]
    for needs in ((True, False, False), (False, True, False), (False, False, True)):
        a = [t.clone().requires_grad_(n) for t, n in zip((x, w, b), needs)]
        y = fu.axs_linear_unified(*a)
        assert y.requires_grad and torch.equal(y.detach(), want)
        y.sum().backward()
    assert not fu.axs_linear_unified(x, w, b).requires_grad


@pytest.mark.parametrize("m", [1, 40])
def test_infer_in_graph_replays(m):
    x, w, b = (t.to(DEV) for t in _inputs(m, 4096, 1030, torch.bfloat16, 11))
    eager = _infer(x, w, b)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _infer(x, w, b)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = _infer(x, w, b)
    for i in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, eager), i


# f32 weights whose block scales leave the window in which the GEMM form sums
# without a reference exponent: near the type's top under small inputs, in its
# subnormals under large ones, and rows that cross it inside the contraction
# (over the splits of K and inside one).  K split over workgroups and (the last) not.
@pytest.mark.parametrize("m,K,N", [(5, 1024, 4160), (33, 2080, 2051), (100, 1024, 8200), (5, 1024, 65540)])
def test_infer_gemm_weight_range(m, K, N):
    from axs.unified import hip_linear

    print(f"[infer range m={m} K={K} N={N}]", flush=True)
    assert _form(m, K, N, torch.float32)
    g = torch.Generator().manual_seed(K + N + m)
    x = torch.randn(m, K, generator=g)
    w = torch.randn(N, K, generator=g).clamp_(-4.0, 4.0)   # 4 x 3e37: no block scales to inf
    w[:, :32].abs_()
    h = K // 2
    for xs, ws in ((1e-3, 3e37), (1e-6, 3e37), (1e10, 1e-43), (1e10, 1e-36), (1.0, 1.0)):
        xv, wv = x * xs, w * ws
        if ws == 1.0:   # rows of other scales in a tile of ordinary ones
            wv[1] *= 2.0 ** 112
            wv[2] *= 2.0 ** -138
            wv[3, :h] = 0.0          # nothing, then tiny
            wv[3, h:] *= 2.0 ** -135
            wv[4, :h] *= 2.0 ** -120   # tiny, then huge
            wv[4, h:] *= 2.0 ** 112
            wv[5, h:] *= 2.0 ** -100   # ordinary, then tiny
            wv[6] = 0.0
            wv[7, 32:] *= 2.0 ** -140  # one ordinary block
            xv[:, 64:96] = 0.0
        y = _infer(xv, wv, None).cpu().double()
        # the training forward packs every row relative to its largest block
        # from the same operand values: only the summation orders differ
        t = hip_linear.forward_train(xv.to(DEV), wv.to(DEV), None)[0].cpu().double()
        assert bool(torch.isfinite(y).all()), (xs, ws, int((~torch.isfinite(y)).sum()))
        scale = t.norm(dim=0).clamp_min(1e-300)
        err = ((y - t).norm(dim=0) / scale).amax()
        assert err <= 1e-5, (xs, ws, float(err), int(((y - t).norm(dim=0) / scale).argmax()))
        if ws > 1e-38:   # FQ values of subnormal blocks are rounded once more in the oracle
            n = 64
            want = _exact(xv, wv[:n], None)
            err = ((y[:, :n] - want).norm(dim=0) / want.norm(dim=0).clamp_min(1e-300))
            ok = torch.ones(n, dtype=torch.bool)
            if ws == 1.0:
                ok[[2, 3, 6]] = False
            assert float(err[ok].amax()) <= 2 * BAR[torch.float32], (xs, ws)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("m", [1, 2, 40])
def test_infer_subnormal_values_round_once(m, dt):
    """FQ values that are subnormal in the operands' type, rounded to it once
    from the table's own value: one product per output, so every bit is defined
    (the f32 product of the rounded values, rounded to the type)."""
    from axs.unified import functional_unified as fu

    K, N = 1024, 4160
    assert _form(m, K, N, dt)
    lo = -24 if dt == torch.float16 else -133        # the type's smallest power of two
    top = 0 if dt == torch.float16 else -110
    g = torch.Generator().manual_seed(21)
    w = torch.randn(N, K, generator=g) * torch.exp2(torch.randint(lo + 4, top, (N, 1), generator=g).float())
    w = w.to(dt)
    one = 1.0 if dt == torch.float16 else 2.0 ** 60
    x = torch.zeros(m, K)
    for i in range(m):
        x[i, 25 * i + 5] = one
    x = x.to(dt)
    with torch.no_grad():
        y = fu.axs_linear_unified(x.to(DEV), w.to(DEV), None, 32, False).cpu()
    wq = torch.from_numpy(oracle.fake_quantize(w.float().numpy(), 32)).to(dt)
    pick = x.float().argmax(1)
    assert torch.equal(y, (wq[:, pick].t().double() * one).to(dt))
    # the same values as the input, one weight per output row
    v = w[:m]
    d = torch.zeros(N, K)
    d[torch.arange(N), torch.arange(N) % K] = one
    d = d.to(dt)
    y = _infer(v, d, None).cpu()
    vq = torch.from_numpy(oracle.fake_quantize(v.float().numpy(), 32)).to(dt)
    dq = torch.from_numpy(oracle.fake_quantize(d.float().numpy(), 32)).to(dt)
    k = torch.arange(N) % K
    want = (vq[:, k].float() * dq[torch.arange(N), k].float()).to(dt)
    assert torch.equal(y, want)


@pytest.mark.parametrize("m", [1, 40])
@pytest.mark.parametrize("dt,bt", [(torch.bfloat16, torch.float32), (torch.float16, torch.float64),
                                   (torch.float32, torch.bfloat16), (torch.float32, torch.float64)], ids=str)
def test_infer_bias_of_another_type(m, dt, bt):
    """A bias of another floating type is added in its own value (float64: as
    float32), and broadcasts as F.linear's."""
    x, w, _ = _inputs(m, 1024, 4100, dt, 31)
    assert _form(m, 1024, 4100, dt)
    b = (torch.randn(4100, generator=torch.Generator().manual_seed(32)) * 3.0).to(bt)
    want = _exact(x, w, b)
    y = _infer(x, w, b)
    assert y.dtype == dt
    assert oracle.rel_l2(y.float().cpu().numpy(), want) <= BAR[dt]
    y = _infer(x, w, b[:1])
    assert oracle.rel_l2(y.float().cpu().numpy(), _exact(x, w, b[:1])) <= BAR[dt]
    with pytest.raises(RuntimeError, match="broadcast"):
        _infer(x, w, b[:7])


def test_infer_float64_is_computed_in_float32():
    x, w, b = _inputs(40, 1024, 4100, torch.float32, 33)
    y = _infer(x.double(), w.double(), b.double())
    assert y.dtype == torch.float64 and torch.equal(y, _infer(x, w, b).double())
