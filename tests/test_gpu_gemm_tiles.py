"""The GEMM's choice between 128x128 and 256x256 tiles: at 512 small tiles (two
per CU) and just over, with whole and ragged edges, short and long contractions
and every output type, and a remainder of one row or column.  Small integers
are exact in fp16 and their sums in fp32, so every output is exact (16-bit
ones: the rounded sum)."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("M,N,Kp", [
    (2048, 4096, 128),    # 512 small tiles: stays
    (2048, 4097, 128),    # one column more: 8 x 17 large tiles
    (2049, 4096, 1088),   # one row more, a long contraction
    (129, 33000, 64),     # a large tile's second half with one row
    (66000, 100, 192),    # half of the only column of tiles
    (3583, 4095, 1024),   # ragged in both, the longest short contraction
], ids=str)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_gemm_tile_choice_exact(M, N, Kp, dtype):
    from axs import _lib

    print(f"[gemm {M} x {N} x {Kp} {dtype}]", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M + N)
    a = torch.randint(-8, 9, (M, Kp), generator=g, device=DEV).float()
    b = torch.randint(-8, 9, (N, Kp), generator=g, device=DEV).float()
    bias = torch.randint(-4, 5, (N,), generator=g, device=DEV).float()
    a16, b16 = a.half(), b.half()
    out = torch.full((M + 1, N), -1.0, dtype=dtype, device=DEV)
    _lib.call("axs6_gemm_f16_nt", a16.data_ptr(), Kp, b16.data_ptr(), Kp, M, N, Kp, None, None, bias.data_ptr(),
              out.data_ptr(), N, _lib.DTYPE_CODE[dtype], _lib.stream_of(a16))
    want = a.double() @ b.double().t() + bias.double()
    assert torch.equal(out[:M].double(), want.float().to(dtype).double())
    assert bool((out[M] == -1.0).all())
