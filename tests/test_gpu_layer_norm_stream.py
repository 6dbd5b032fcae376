"""The LayerNorm vector kernels' streaming instances (tensors of 128 MiB and
more: nontemporal stores and last-use loads) and the backward's next-row
prefetch, at the edges: just below and at 128 MiB, row counts that leave a
partial chunk or fewer rows than workgroups, and rows whose last vector group
is partial; and the ragged instances (rows of no whole number of vectors).
Against float64 F.layer_norm; the bars are those of the kernels' other test
(f32: rounding of sums of up to 16K terms; 16-bit: one rounding of the result)."""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TOL = {torch.float32: 2e-6, torch.bfloat16: 8e-3, torch.float16: 1e-3}


# (rows, cols, dtype)
CASES = [
    (32768, 1024, torch.float32),    # 128 MiB, a wave per row
    (32767, 1024, torch.float32),    # one row less: not streamed
    (131075, 260, torch.float32),    # streamed, last group of one vector
    (8209, 4100, torch.float32),     # streamed, a workgroup per row
    (4099, 8188, torch.float32),     # streamed, prefetch in f32, last group short
    (16387, 4104, torch.bfloat16),   # streamed, prefetch
    (8193, 8192, torch.float16),
    (65539, 1032, torch.bfloat16),
    (262145, 264, torch.float16),
    (16400, 4097, torch.bfloat16),   # streamed, ragged
    (65600, 515, torch.float32),     # streamed, ragged, a wave per row
    # ragged rows on both sides of the row counts from which the backward takes the vector form
    (511, 1001, torch.float32),
    (512, 1001, torch.float32),
    (513, 257, torch.float32),
    (2047, 1027, torch.float32),
    (2048, 1027, torch.float32),
    (2048, 8191, torch.float32),
    (2050, 2047, torch.float16),
    (2048, 8191, torch.bfloat16),
    (530, 515, torch.bfloat16),
    # the streamed forms below their size
    (8192, 1024, torch.float32),
    (8191, 1024, torch.float32),
    (32771, 260, torch.float32),     # a wave per row, last group of one vector
    (2053, 4100, torch.float32),     # a workgroup per row, last group of one vector
    (1025, 8188, torch.float32),     # prefetch in f32, last group short
    (4099, 4104, torch.bfloat16),    # prefetch, last group of one vector
    (2049, 8192, torch.float16),
    (16387, 1032, torch.bfloat16),
    (65537, 264, torch.float16),     # a wave per row, 16-bit
    (1, 2056, torch.bfloat16),       # prefetch past the only row
    (17, 8192, torch.float32),
    (5, 520, torch.float16),
    # ragged rows: unaligned vectors, the last one overlapping its neighbour
    (300, 5, torch.float32),         # two vectors sharing three values
    (300, 9, torch.bfloat16),
    (301, 15, torch.float16),        # sharing one value
    (70, 257, torch.float32),
    (33, 1027, torch.float32),       # a workgroup per row
    (9, 8191, torch.float32),        # the longest ragged vector row
    (31, 2047, torch.float16),
    (9, 8191, torch.bfloat16),
    (4100, 4097, torch.bfloat16),
    (16400, 515, torch.float32),     # a wave per row
]


@pytest.mark.parametrize("rows,cols,dtype", CASES, ids=str)
def test_layer_norm_streaming_edges(rows, cols, dtype):
    from axs.unified import AXSLayerNormUnified

    print(f"[layer_norm {rows} x {cols} {dtype}]", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(rows + cols)
    x = (torch.randn(rows, cols, generator=gen, device=DEV) * 3.0 + 0.7).to(dtype).requires_grad_(True)
    dy = torch.randn(rows, cols, generator=gen, device=DEV).to(dtype)
    m = AXSLayerNormUnified(cols).to(DEV, dtype)
    with torch.no_grad():
        m.weight.copy_(1.0 + 0.5 * torch.randn(cols, generator=gen, device=DEV))
        m.bias.copy_(0.3 * torch.randn(cols, generator=gen, device=DEV))
    y = m(x)
    y.backward(dy)
    xd = x.detach().double().requires_grad_(True)
    wd = m.weight.detach().double().requires_grad_(True)
    bd = m.bias.detach().double().requires_grad_(True)
    yd = F.layer_norm(xd, (cols,), wd, bd, m.eps)
    yd.backward(dy.double())
    for name, a, b in (("y", y, yd), ("dx", x.grad, xd.grad), ("dgamma", m.weight.grad, wd.grad),
                       ("dbeta", m.bias.grad, bd.grad)):
        a, b = a.detach().double(), b.detach()
        err = float(torch.linalg.vector_norm(a - b) / torch.linalg.vector_norm(b))
        assert err <= TOL[dtype], (name, err)
        assert float((a - b).abs().amax()) <= 50 * TOL[dtype] * float(b.abs().amax()), name
