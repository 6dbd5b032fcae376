"""Fake-quantize of rows that do not tile into 16-byte vectors of whole blocks
(``fq_rows_kernel``: unaligned 16-byte groups, rows padded to whole blocks of
lanes), bit for bit against the oracle: every length of a cut group, rows of
fewer and more groups than a workgroup steps by (256), rows shorter and longer
than a workgroup's share, and a tensor whose last group is its last bytes."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
SEED = 11

# cut groups of 1 .. 7 values; 1017 and 1033: 128 (f32: 256) groups and one more
# block; 2041 and 2049: 256 (f32: 512) and more; 9001: several workgroups a row
COLS = [65, 66, 67, 68, 69, 70, 71, 127, 257, 1017, 1033, 2041, 2049, 4095, 9001]


def _bits(t):
    return t.view(torch.int32 if t.dtype == torch.float32 else torch.int16)


def _want(x, bs, u=None):
    return torch.from_numpy(oracle.fake_quantize(x.float().numpy(), bs, u)).to(x.dtype)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("cols", COLS)
def test_fq_ragged_rows(cols, dt):
    from axs.unified.hip_kernels import hip_fused_fake_quantize

    g = torch.Generator().manual_seed(cols)
    for rows, bs in ((1, 32), (3, 8), (37, 32), (50, 16)):
        x = (torch.randn(rows, cols, generator=g) * torch.exp2(torch.randint(-8, 8, (rows, 1), generator=g))).to(dt)
        x[0, : min(40, cols)] = 0.0
        # one element into a buffer that ends with the tensor
        buf = torch.empty(rows * cols + 1, dtype=dt, device=DEV)
        xd = buf[1:].view(rows, cols).copy_(x)
        for v in (x.to(DEV), xd):
            got = hip_fused_fake_quantize(v, bs).cpu()
            assert torch.equal(_bits(got), _bits(_want(x, bs))), (rows, bs)
        u = oracle.uniform(SEED, 0, x.numel())
        got = hip_fused_fake_quantize(xd, bs, "stochastic", seed=SEED).cpu()
        assert torch.equal(_bits(got), _bits(_want(x, bs, u))), (rows, bs)


# the tensors' sizes at which a lane takes 16 bytes instead of one value, and a
# thread three groups instead of one: on both sides, with every cut group
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("cols", [65, 66, 67, 68, 69, 70, 71, 76, 1017, 4095])
def test_fq_ragged_rows_sizes(cols, dt):
    from axs.unified.hip_kernels import hip_fused_fake_quantize

    per = 4 if dt == torch.float32 else 8
    many = -(-(3 << 18) // -(-cols // per))
    one = -(-(1 << 18) // cols)
    g = torch.Generator().manual_seed(cols)
    for rows in (one - 1, one, many - 1, many):
        x = torch.randn(rows, cols, generator=g).to(dt)
        x[rows // 2] *= 0.01
        x[-1, -5:] = 0.0
        buf = torch.empty(rows * cols + 1, dtype=dt, device=DEV)
        xd = buf[1:].view(rows, cols).copy_(x)
        got = hip_fused_fake_quantize(xd, 32).cpu()
        assert torch.equal(_bits(got), _bits(_want(x, 32))), rows
        if rows in (one, many):
            u = oracle.uniform(SEED, 0, x.numel())
            got = hip_fused_fake_quantize(x.to(DEV), 16, "stochastic", seed=SEED).cpu()
            assert torch.equal(_bits(got), _bits(_want(x, 16, u))), rows


def test_fq_ragged_rows_past_one_grid_dimension():
    """More groups than the threads of one grid dimension (2^32, three groups a
    thread): 140 GB of rows of 65 values, in place; rows around the border of a
    dimension's share, at the 2^32 threads and at the end."""
    from axs import _lib

    cols, per_row = 65, 12                       # bf16, block 32: 12 groups of 8 values
    rows = 3 * 2 ** 32 // per_row + 1000
    free, _ = torch.cuda.mem_get_info()
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < rows * cols * 2 + (2 << 30):
        pytest.skip(f"needs 142 GB of device memory, {free >> 30} GiB are free")
    x = torch.zeros(rows, cols, dtype=torch.bfloat16, device=DEV)
    g = torch.Generator().manual_seed(3)
    share = 3 * 256 * 2 ** 22 // per_row         # rows of one step along y
    spots = [0, share - 4, 2 * share - 4, 3 * 2 ** 32 // per_row - 4, rows - 8]
    want = []
    for r in spots:
        v = torch.randn(8, cols, generator=g).bfloat16()
        x[r : r + 8].copy_(v)
        want.append(_want(v, 32))
    _lib.call("axs6_nf5_fake_quantize", x.data_ptr(), x.data_ptr(), _lib.DTYPE_CODE[x.dtype], rows, cols, 32, 0, 0, 0,
              None, _lib.stream_of(x))
    for r, w in zip(spots, want):
        assert torch.equal(_bits(x[r : r + 8].cpu()), _bits(w)), r
    del x
    torch.cuda.empty_cache()
