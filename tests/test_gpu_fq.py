"""GPU parity of the NF5 fake-quantize / quantize / dequantize kernels
against the CPU oracle and the golden vectors: bit-exact (NaN matched by
position), per BASELINE configs 1-2 and the reference's own test cases
(tests/test_triton_kernels.py:78-259 of the reference)."""
from __future__ import annotations

import hashlib

import numpy as np
import pytest
import torch

import oracle
from conftest import bits_equal, first_mismatch, load_golden

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _fq(x: torch.Tensor, bs=32, rounding="nearest", seed=None) -> torch.Tensor:
    from axs.unified.hip_kernels import hip_fused_fake_quantize

    return hip_fused_fake_quantize(x, bs, rounding, seed=seed)


def config2_input(shape, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(*shape, generator=g)
    m = torch.rand(*shape, generator=g) < 0.01
    x[m] *= 100.0
    return x


@pytest.mark.parametrize("shape,seed", [((256, 256), 1), ((4096, 4096), 2), ((8192, 4096), 3)],
                         ids=["256x256", "4096x4096", "8192x4096"])
def test_config2_fake_quantize_bitexact(shape, seed):
    print(f"[fq config2 {shape}]", flush=True)
    x = config2_input(shape, seed)
    got = _fq(x.to(DEV)).cpu().numpy()
    want = oracle.fake_quantize(x.numpy(), 32)
    assert bits_equal(got, want), first_mismatch(got, want)


@pytest.mark.parametrize("bs", [8, 16, 32])
def test_block_sizes_bitexact(bs):
    x = config2_input((512, 512), 10 + bs)
    got = _fq(x.to(DEV), bs).cpu().numpy()
    assert bits_equal(got, oracle.fake_quantize(x.numpy(), bs))


@pytest.mark.parametrize("bs", [8, 16, 32])
@pytest.mark.parametrize("unaligned", [False, True], ids=["vector", "general"])
def test_edge_golden(bs, unaligned):
    g = load_golden("edge_cases.npz")
    x = torch.from_numpy(g["x"])
    if unaligned:
        # a view one element into a buffer forces the general (scalar) kernel
        buf = torch.zeros(x.numel() + 1, dtype=torch.float32, device=DEV)
        buf[1:] = x.reshape(-1).to(DEV)
        xd = buf[1:].view(x.shape)
        assert xd.data_ptr() % 16 != 0
    else:
        xd = x.to(DEV)
    got = _fq(xd, bs).cpu().numpy()
    want = g[f"fq_bs{bs}"]
    assert bits_equal(got, want), first_mismatch(got, want)


def test_ragged_golden_all_dtypes():
    g = load_golden("ragged.npz")
    for i in range(8):
        x = torch.from_numpy(g[f"x{i}"])
        for bs in (8, 16, 32):
            got = _fq(x.to(DEV), bs).cpu().numpy()
            assert bits_equal(got, g[f"x{i}_fq_bs{bs}"]), (i, bs, first_mismatch(got, g[f"x{i}_fq_bs{bs}"]))
        for tag, dt in (("bf16", torch.bfloat16), ("f16", torch.float16)):
            xin = torch.from_numpy(g[f"x{i}_in_{tag}"]).view(dt)
            y = _fq(xin.to(DEV), 32)
            assert y.dtype == dt and y.shape == xin.shape
            assert np.array_equal(y.cpu().view(torch.int16).numpy(), g[f"x{i}_fq_{tag}"]), (i, tag)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("bs", [8, 16, 32])
def test_half_dtypes_vs_oracle(dt, bs):
    x = config2_input((1024, 2048), 20 + bs).to(dt)
    got = _fq(x.to(DEV), bs).cpu()
    want = torch.from_numpy(oracle.fake_quantize(x.float().numpy(), bs)).to(dt)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


def test_bf16_nan_and_rounding_bits():
    """bf16 outputs are rounded to nearest even from the f32 FQ value, and a
    NaN block is written as 0x7FC0 (torch's bf16 NaN)."""
    x = config2_input((64, 512), 77)
    x[3, 7] = float("nan")
    xb = x.to(torch.bfloat16)
    got = _fq(xb.to(DEV), 32).cpu().view(torch.int16)
    want = torch.from_numpy(oracle.fake_quantize(xb.float().numpy(), 32)).to(torch.bfloat16).view(torch.int16)
    nan = (got[3, :32] & 0x7FFF) > 0x7F80
    assert bool(nan.all()) and bool(((got[3, :32] & 0xFFFF) == 0x7FC0).all())
    mask = torch.ones_like(got, dtype=torch.bool)
    mask[3, :32] = False
    assert torch.equal(got[mask], want[mask])


def test_exponent_range_and_bands():
    # blocks spanning the whole float32 range, incl. subnormals and overflow
    rng = np.random.default_rng(5)
    rows = []
    for e in range(-160, 130, 2):
        rows.append((rng.standard_normal(32) * 2.0 ** e).astype(np.float32))
    for k in range(-148, 129):
        top = (k + 127) << 23 if k >= -126 else 1 << (k + 149)
        for d in (1, 2, 11, 22, 44, 45):
            if d >= top:
                continue
            v = np.array([top - d], np.uint32).view(np.float32)[0]
            if not np.isfinite(v):
                continue
            r = (rng.uniform(-1, 1, 32) * v).astype(np.float32)
            r[rng.integers(32)] = -v if d % 2 else v
            rows.append(r)
    x = np.stack(rows)
    for bs in (8, 16, 32):
        got = _fq(torch.from_numpy(x).to(DEV), bs).cpu().numpy()
        want = oracle.fake_quantize(x, bs)
        assert bits_equal(got, want), (bs, first_mismatch(got, want))


@pytest.mark.parametrize("shape", [(1024, 4096), (37, 100)], ids=["vector", "general"])
@pytest.mark.parametrize("bs", [8, 32])
def test_stochastic_bitexact_given_stream(shape, bs):
    x = config2_input(shape, 40)
    seed = 0x1234ABCD5678
    got = _fq(x.to(DEV), bs, "stochastic", seed=seed).cpu().numpy()
    want = oracle.fake_quantize(x.numpy(), bs, oracle.uniform(seed, 0, x.numel()))
    assert bits_equal(got, want), first_mismatch(got, want)


def test_stochastic_statistics():
    torch.manual_seed(0)
    x = torch.randn(1024, 1024, device=DEV)
    nearest = _fq(x)
    sto = _fq(x, rounding="stochastic")
    assert not torch.equal(nearest, sto)
    ratio = ((x - sto).pow(2).mean() / (x - nearest).pow(2).mean()).item()
    assert 0.5 < ratio < 2.0, ratio
    xs = torch.randn(256, 256, device=DEV)
    errs = [(xs - _fq(xs, rounding="stochastic")).mean().item() for _ in range(20)]
    assert abs(sum(errs) / len(errs)) < 0.01
    # same seed reproduces, different seeds differ
    assert torch.equal(_fq(x, rounding="stochastic", seed=7), _fq(x, rounding="stochastic", seed=7))
    assert not torch.equal(_fq(x, rounding="stochastic", seed=7), _fq(x, rounding="stochastic", seed=8))


@pytest.mark.parametrize("shape", [(64,), (32, 64), (4, 8, 16), (2, 3, 4, 32), (7, 13), (3, 100, 17)])
def test_shape_dtype_device_preserved(shape):
    x = torch.randn(*shape, device=DEV)
    y = _fq(x)
    assert y.shape == x.shape and y.dtype == x.dtype and y.device == x.device
    assert bits_equal(y.cpu().numpy(), oracle.fake_quantize(x.cpu().numpy(), 32))


def test_non_contiguous_and_float64():
    x = torch.randn(96, 64, device=DEV).t()
    assert not x.is_contiguous()
    assert bits_equal(_fq(x).cpu().numpy(), oracle.fake_quantize(x.cpu().contiguous().numpy(), 32))
    xd = torch.randn(16, 64, dtype=torch.float64, device=DEV)
    y = _fq(xd)
    assert y.dtype == torch.float64
    want = oracle.fake_quantize(xd.float().cpu().numpy(), 32).astype(np.float64)
    assert bits_equal(y.cpu().numpy(), want)


def test_zero_and_empty():
    z = torch.zeros(128, 128, device=DEV)
    assert (_fq(z) == 0).all()
    e = torch.zeros(0, 32, device=DEV)
    assert _fq(e).shape == (0, 32)


# ------------------------------------------------------------- quantize --

def _quant(x: torch.Tensor, bs=32, rounding="nearest", seed=None):
    from axs.unified.hip_kernels import hip_quantize

    e, c, s, fq = hip_quantize(x, bs, rounding, with_fake_quantized=True, seed=seed)
    return e.cpu().numpy(), c.cpu().numpy(), s.cpu().numpy(), fq.cpu().numpy()


@pytest.mark.parametrize("bs", [8, 16, 32])
def test_quantize_edge_golden(bs):
    g = load_golden("edge_cases.npz")
    e, c, s, fq = _quant(torch.from_numpy(g["x"]).to(DEV), bs)
    assert np.array_equal(e, g[f"exp_bs{bs}"]), first_mismatch(e, g[f"exp_bs{bs}"])
    assert np.array_equal(c, g[f"code_bs{bs}"])
    assert np.array_equal(s, g[f"sign_bs{bs}"])
    assert bits_equal(fq, g[f"fq_bs{bs}"])


@pytest.mark.parametrize("bs", [8, 16, 32])
@pytest.mark.parametrize("shape", [(300, 256), (37, 100)])
def test_quantize_vs_oracle(bs, shape):
    x = config2_input(shape, 60 + bs)
    x[0, :5] = torch.tensor([float("nan"), 0.0, -0.0, 1e-40, -3e38])
    for rounding, seed in (("nearest", None), ("stochastic", 99)):
        e, c, s, fq = _quant(x.to(DEV), bs, rounding, seed)
        u = oracle.uniform(seed, 0, x.numel()) if seed else None
        oe, oc, os_ = oracle.quantize(x.numpy(), bs, u)
        assert np.array_equal(e, oe) and np.array_equal(c, oc) and np.array_equal(s, os_)
        assert bits_equal(fq, oracle.fake_quantize(x.numpy(), bs, u))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("bs", [8, 16, 32])
def test_quantize_16bit_vs_oracle(dt, bs):
    """16-bit inputs on the vector kernel (8 values per lane): codes, signs,
    exponents and the FQ output, nearest and stochastic."""
    x = config2_input((64, 256), 90 + bs).to(dt)
    x[0, :5] = torch.tensor([float("nan"), 0.0, -0.0, 1e-40, -3e38]).to(dt)
    xf = x.float().numpy()
    from axs.unified.hip_kernels import hip_quantize

    for rounding, seed in (("nearest", None), ("stochastic", 7)):
        e, c, s, fq = hip_quantize(x.to(DEV), bs, rounding, with_fake_quantized=True, seed=seed)
        u = oracle.uniform(seed, 0, x.numel()) if seed else None
        oe, oc, os_ = oracle.quantize(xf, bs, u)
        assert np.array_equal(e.cpu().numpy(), oe) and np.array_equal(c.cpu().numpy(), oc)
        assert np.array_equal(s.cpu().numpy(), os_)
        want = torch.from_numpy(oracle.fake_quantize(xf, bs, u)).to(dt)
        got = fq.cpu()
        nan = torch.isnan(want)                 # NaN payloads differ between conversions: positions only
        assert torch.equal(torch.isnan(got), nan)
        assert torch.equal(got.view(torch.int16)[~nan], want.view(torch.int16)[~nan])


@pytest.mark.parametrize("bs", [8, 16, 32])
def test_quantize_without_optional_outputs(bs):
    """No signs and no FQ output (null pointers) on the vector kernel."""
    from axs import _lib

    x = config2_input((40, 192), 70 + bs).to(DEV)
    nblk = 192 // bs
    e = torch.empty((40, nblk), dtype=torch.uint8, device=DEV)
    c = torch.empty((40, 192), dtype=torch.uint8, device=DEV)
    _lib.call("axs6_nf5_quantize", x.data_ptr(), _lib.F32, 40, 192, bs, 0, 0, 0, e.data_ptr(), c.data_ptr(),
              None, None, None, _lib.stream_of(x))
    torch.cuda.synchronize()
    oe, oc, _ = oracle.quantize(x.cpu().numpy(), bs)
    assert np.array_equal(e.cpu().numpy(), oe) and np.array_equal(c.cpu().numpy().reshape(oc.shape), oc)


def test_config1_golden():
    g = load_golden("config1.npz")
    gen = torch.Generator().manual_seed(0)
    x = torch.randn(1024, 1024, generator=gen) * 0.02
    sha = lambda a: hashlib.sha256(np.ascontiguousarray(a).tobytes()).hexdigest()  # noqa: E731
    e, c, s, fq = _quant(x.to(DEV), 32)
    oe, oc, os_ = oracle.quantize(x.numpy(), 32)
    assert np.array_equal(e, oe) and np.array_equal(c, oc) and np.array_equal(s, os_)
    assert bits_equal(fq, oracle.fake_quantize(x.numpy(), 32))
    # the fixture's hashes hold for the reference's own input: torch's CPU
    # randn stream must reproduce it (it does for this torch build; a
    # different stream is a test-environment error, not a skip)
    assert sha(x.numpy()) == str(g["input_sha"]), "torch.randn(seed 0) no longer gives the config-1 input"
    assert np.array_equal(e, g["exps"])
    assert sha(c) == str(g["codes_sha"]) and sha(s) == str(g["signs_sha"])
    assert sha(fq) == str(g["fq_sha"])


# 101 columns: ragged rows (general kernel); 128: whole blocks (vector kernel)
@pytest.mark.parametrize("cols", [101, 128])
@pytest.mark.parametrize("bs", [8, 16, 32])
def test_dequantize_vs_oracle(bs, cols):
    from axs.unified.quantize_unified import dequantize_unified, quantize_unified

    x = config2_input((200, cols), 80 + bs)
    q = quantize_unified(x.to(DEV), bs)
    d = dequantize_unified(q).cpu().numpy()
    oe, oc, os_ = oracle.quantize(x.numpy(), bs)
    want = oracle.dequantize(oe, oc, os_, x.shape[1], bs)
    assert bits_equal(d, want), first_mismatch(d, want)
    g = load_golden("edge_cases.npz")
    q = quantize_unified(torch.from_numpy(g["x"]).to(DEV), bs)
    assert bits_equal(dequantize_unified(q).cpu().numpy(), g[f"deq_bs{bs}"])


# Whole blocks in runs of two vectors per lane: less than a wave, a run cut in
# its second half, the first size that dequantizes two groups per lane (and not
# a multiple of its run), the first that quantizes two runs per workgroup.
@pytest.mark.parametrize("shape", [(3, 8), (129, 24), (1281, 1032), (8201, 1032)], ids=str)
def test_codec_vector_runs(shape):
    from axs.unified.quantize_unified import dequantize_unified, quantize_unified

    x = config2_input(shape, 83)
    q = quantize_unified(x.to(DEV), 8)
    oe, oc, os_ = oracle.quantize(x.numpy(), 8)
    assert np.array_equal(q.shared_exponents.cpu().numpy().reshape(oe.shape), oe)
    assert np.array_equal(q.magnitudes.cpu().numpy().reshape(oc.shape), oc)
    d = dequantize_unified(q).cpu().numpy()
    want = oracle.dequantize(oe, oc, os_, x.shape[1], 8)
    assert bits_equal(d, want), first_mismatch(d, want)
    e, c, s, fq = _quant(x.to(DEV), 8, "stochastic", 5)
    u = oracle.uniform(5, 0, x.numel())
    oe, oc, os_ = oracle.quantize(x.numpy(), 8, u)
    assert np.array_equal(c.reshape(oc.shape), oc) and np.array_equal(s.reshape(os_.shape), os_)
    assert bits_equal(fq, oracle.fake_quantize(x.numpy(), 8, u))


@pytest.mark.parametrize("rows", [16383, 16385])
def test_quantize_fq_output_vector_choice(rows):
    """f32 with the FQ output on both sides of the size from which it loads one
    vector ahead instead of two together (16384 rows of 1024)."""
    x = config2_input((rows, 1024), 84)
    e, c, s, fq = _quant(x.to(DEV), 32, "nearest", 0)
    oe, oc, os_ = oracle.quantize(x.numpy(), 32)
    assert np.array_equal(e.reshape(oe.shape), oe) and np.array_equal(c.reshape(oc.shape), oc)
    assert np.array_equal(s.reshape(os_.shape), os_)
    assert bits_equal(fq, oracle.fake_quantize(x.numpy(), 32))


# Ragged rows (fq_rows_kernel): rows of >= 64 values that do not tile into
# 16-byte vectors of whole blocks -- a ragged last block, or a view whose start
# is off 16-byte alignment.  A cut last group and none, rows of fewer and more
# groups than a workgroup steps by (256), a last workgroup partly past the
# tensor; every length of a cut group is in test_gpu_fq_ragged.py.
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("bs", [8, 16, 32])
@pytest.mark.parametrize("shape", [(300, 4100), (64, 1000), (129, 777), (5, 64), (33, 255)], ids=str)
def test_rows_kernel_bitexact(dt, bs, shape):
    print(f"[fq rows {dt} bs={bs} {shape}]", flush=True)
    x = config2_input(shape, 7 * bs + shape[1]).to(dt)
    got = _fq(x.to(DEV), bs).cpu()
    want = torch.from_numpy(oracle.fake_quantize(x.float().numpy(), bs)).to(dt)
    if dt == torch.float32:
        assert bits_equal(got.numpy(), want.numpy()), first_mismatch(got.numpy(), want.numpy())
    else:
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("bs", [8, 32])
def test_rows_kernel_unaligned_view(dt, bs):
    """Whole-block rows in a view one element into its buffer (the vector
    kernel needs 16-byte alignment): the ragged rows' kernel, same bits."""
    x = config2_input((256, 4096), 91 + bs).to(dt)
    buf = torch.zeros(x.numel() + 1, dtype=dt, device=DEV)
    buf[1:] = x.reshape(-1).to(DEV)
    xd = buf[1:].view(x.shape)
    assert xd.data_ptr() % 16 != 0
    bits = torch.int32 if dt == torch.float32 else torch.int16
    got = _fq(xd, bs).cpu().view(bits)
    assert torch.equal(got, _fq(x.to(DEV), bs).cpu().view(bits))


def test_rows_kernel_exponent_range():
    """Blocks across the whole float32 range (subnormal, tiny, huge, inf
    scale, NaN) through the ragged rows' kernel: rows of four such blocks plus
    a ragged block of seven values."""
    rng = np.random.default_rng(8)
    blocks = []
    for e in range(-160, 130, 2):
        blocks.append((rng.standard_normal(32) * 2.0 ** e).astype(np.float32))
    nan = rng.standard_normal(32).astype(np.float32)
    nan[5] = np.nan
    inf = rng.standard_normal(32).astype(np.float32)
    inf[9] = np.inf
    blocks += [nan, inf, np.zeros(32, np.float32), np.full(32, -0.0, np.float32)]
    while len(blocks) % 4:
        blocks.append(rng.standard_normal(32).astype(np.float32))
    wide = np.stack(blocks).reshape(-1, 128)
    # 7 extra values: one value per lane; 8: four per lane (rows of 136)
    for extra in (7, 8):
        x = np.concatenate([wide, rng.standard_normal((wide.shape[0], extra)).astype(np.float32)], axis=1)
        for bs in (8, 16, 32):
            got = _fq(torch.from_numpy(x).to(DEV), bs).cpu().numpy()
            want = oracle.fake_quantize(x, bs)
            assert bits_equal(got, want), (extra, bs, first_mismatch(got, want))


@pytest.mark.parametrize("bs", [8, 32])
@pytest.mark.parametrize("cols", [1030, 1032], ids=["one-per-lane", "four-per-lane"])
def test_rows_kernel_stochastic_given_stream(bs, cols):
    x = config2_input((200, cols), 55)
    seed = 0x5EED0F00D
    got = _fq(x.to(DEV), bs, "stochastic", seed=seed).cpu().numpy()
    want = oracle.fake_quantize(x.numpy(), bs, oracle.uniform(seed, 0, x.numel()))
    assert bits_equal(got, want), first_mismatch(got, want)


# Short rows (fq_short_kernel): rows of 1-63 values, or of whole 4-value
# groups under 256, that are not whole blocks or not 16-byte aligned --
# whole rows per wave step, one or four values per lane, block maxima by
# segmented shuffles; row counts that leave the last step partly empty, and
# NaN / inf / subnormal / zero values in the blocks.
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("bs", [8, 16, 32])
def test_short_rows_kernel_bitexact(dt, bs):
    specials = torch.tensor([float("nan"), float("inf"), -0.0, 0.0, 1e-40, -3e38, 2.0 ** -130])
    # 4, 40, 68 ... 252: whole 4-value groups, four values per lane
    for cols in (1, 3, 4, 7, 9, 17, 31, 33, 40, 63, 68, 100, 132, 200, 252, 99):
        for rows in (1, 5, 1000):
            print(f"[fq short {dt} bs={bs} {rows}x{cols}]", flush=True)
            x = config2_input((rows, cols), 13 * cols + rows + bs)
            if rows * cols > 64:
                x.view(-1)[7:7 + 7 * 9:9] = specials
            x = x.to(dt)
            got = _fq(x.to(DEV), bs).cpu()
            want = torch.from_numpy(oracle.fake_quantize(x.float().numpy(), bs)).to(dt)
            bits = torch.int32 if dt == torch.float32 else torch.int16
            nan = torch.isnan(want)
            assert torch.equal(torch.isnan(got), nan), (rows, cols)
            assert torch.equal(got.view(bits)[~nan], want.view(bits)[~nan]), (rows, cols)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("cols", [20, 100, 200])
def test_short_rows_kernel_unaligned_view(dt, cols):
    """Short rows of whole 4-value groups in a view one element into its
    buffer: one value per lane (or the ragged rows' kernel), same bits as the
    aligned tensor's four-per-lane form."""
    x = config2_input((999, cols), 5 + cols).to(dt)
    buf = torch.zeros(x.numel() + 1, dtype=dt, device=DEV)
    buf[1:] = x.reshape(-1).to(DEV)
    bits = torch.int32 if dt == torch.float32 else torch.int16
    for bs in (8, 16, 32):
        got = _fq(buf[1:].view(x.shape), bs).cpu().view(bits)
        assert torch.equal(got, _fq(x.to(DEV), bs).cpu().view(bits)), bs


@pytest.mark.parametrize("bs", [8, 32])
@pytest.mark.parametrize("cols", [3, 20, 45, 100])
def test_short_rows_kernel_stochastic_given_stream(bs, cols):
    x = config2_input((3001, cols), 71 + cols)
    seed = 0xD1CE
    got = _fq(x.to(DEV), bs, "stochastic", seed=seed).cpu().numpy()
    want = oracle.fake_quantize(x.numpy(), bs, oracle.uniform(seed, 0, x.numel()))
    assert bits_equal(got, want), first_mismatch(got, want)


# Quantize of padded rows under 192 positions (quantize_short_kernel): four
# positions per lane over the run of whole blocks, values read one by one.
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("bs", [8, 16, 32])
def test_quantize_short_rows_kernel(dt, bs):
    from axs.unified.hip_kernels import hip_dequantize, hip_quantize

    specials = torch.tensor([float("nan"), float("inf"), -0.0, 0.0, 1e-40, -3e38, 2.0 ** -130])
    for cols in (1, 3, 7, 9, 17, 31, 33, 40, 55, 68, 100, 131, 200, 225):
        if (cols + bs - 1) // bs * bs >= 192:      # longer padded rows: the row-segment kernel
            continue
        for rows in (1, 7, 1001):
            print(f"[quantize short {dt} bs={bs} {rows}x{cols}]", flush=True)
            x = config2_input((rows, cols), 31 * cols + rows + bs)
            if rows * cols > 64:
                x.view(-1)[5:5 + 7 * 8:8] = specials
            x = x.to(dt)
            xf = x.float().numpy()
            for rounding, seed in (("nearest", None), ("stochastic", 4321)):
                e, c, s, fq = hip_quantize(x.to(DEV), bs, rounding, with_fake_quantized=True, seed=seed)
                u = oracle.uniform(seed, 0, x.numel()) if seed else None
                oe, oc, os_ = oracle.quantize(xf, bs, u)
                assert np.array_equal(e.cpu().numpy(), oe), (rows, cols, rounding)
                assert np.array_equal(c.cpu().numpy(), oc), (rows, cols, rounding)
                assert np.array_equal(s.cpu().numpy(), os_), (rows, cols, rounding)
                want = torch.from_numpy(oracle.fake_quantize(xf, bs, u)).to(dt)
                nan = torch.isnan(want)
                bits = torch.int32 if dt == torch.float32 else torch.int16
                assert torch.equal(torch.isnan(fq.cpu()), nan)
                assert torch.equal(fq.cpu().view(bits)[~nan], want.view(bits)[~nan]), (rows, cols, rounding)
            d = hip_dequantize(e, c, s, rows, cols, bs).cpu().numpy()
            assert bits_equal(d, oracle.dequantize(oe, oc, os_, cols, bs)), (rows, cols)


# Row-segment quantize / dequantize (quantize_rows_kernel,
# dequantize_rows_kernel): ragged rows of >= 64 values, padded-layout codes.
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("bs", [8, 16, 32])
@pytest.mark.parametrize("shape", [(300, 4100), (129, 777), (16, 2049)], ids=str)
def test_quantize_rows_kernel(dt, bs, shape):
    from axs.unified.hip_kernels import hip_dequantize, hip_quantize

    print(f"[quantize rows {dt} bs={bs} {shape}]", flush=True)
    x = config2_input(shape, 3 * bs + shape[1]).to(dt)
    x[0, :5] = torch.tensor([float("nan"), 0.0, -0.0, 1e-40, -3e38]).to(dt)
    xf = x.float().numpy()
    for rounding, seed in (("nearest", None), ("stochastic", 1234)):
        e, c, s, fq = hip_quantize(x.to(DEV), bs, rounding, with_fake_quantized=True, seed=seed)
        u = oracle.uniform(seed, 0, x.numel()) if seed else None
        oe, oc, os_ = oracle.quantize(xf, bs, u)
        assert np.array_equal(e.cpu().numpy(), oe), (rounding, first_mismatch(e.cpu().numpy(), oe))
        assert np.array_equal(c.cpu().numpy(), oc) and np.array_equal(s.cpu().numpy(), os_)
        # without the FQ output (rows that are not whole aligned 4-value groups
        # then take the four-positions-per-lane run kernel)
        e2, c2, s2, _ = hip_quantize(x.to(DEV), bs, rounding, seed=seed)
        assert np.array_equal(e2.cpu().numpy(), oe) and np.array_equal(c2.cpu().numpy(), oc)
        assert np.array_equal(s2.cpu().numpy(), os_)
        want = torch.from_numpy(oracle.fake_quantize(xf, bs, u)).to(dt)
        got = fq.cpu()
        nan = torch.isnan(want)
        assert torch.equal(torch.isnan(got), nan)
        bits = torch.int32 if dt == torch.float32 else torch.int16
        assert torch.equal(got.view(bits)[~nan], want.view(bits)[~nan])
    e, c, s, _ = hip_quantize(x.to(DEV), bs, "nearest")
    d = hip_dequantize(e, c, s, shape[0], shape[1], bs).cpu().numpy()
    want = oracle.dequantize(*oracle.quantize(xf, bs), shape[1], bs)
    assert bits_equal(d, want), first_mismatch(d, want)


@pytest.mark.parametrize("cols", [1001, 1004, 13], ids=["one-per-lane", "four-per-lane", "short"])
def test_quantize_rows_kernel_without_optional_outputs(cols):
    """No signs and no FQ output on the row-segment kernel, and the dequantize
    without signs (all values positive)."""
    from axs import _lib

    rows, bs = 50, 32
    nblk = (cols + bs - 1) // bs
    x = config2_input((rows, cols), 17).abs().to(DEV)
    e = torch.empty((rows, nblk), dtype=torch.uint8, device=DEV)
    c = torch.empty((rows, nblk * bs), dtype=torch.uint8, device=DEV)
    st = _lib.stream_of(x)
    _lib.call("axs6_nf5_quantize", x.data_ptr(), _lib.F32, rows, cols, bs, 0, 0, 0, e.data_ptr(), c.data_ptr(),
              None, None, None, st)
    y = torch.empty((rows, cols), device=DEV)
    _lib.call("axs6_nf5_dequantize", e.data_ptr(), c.data_ptr(), None, y.data_ptr(), rows, cols, bs, st)
    torch.cuda.synchronize()
    oe, oc, os_ = oracle.quantize(x.cpu().numpy(), bs)
    assert np.array_equal(e.cpu().numpy(), oe) and np.array_equal(c.cpu().numpy().reshape(oc.shape), oc)
    assert bits_equal(y.cpu().numpy(), oracle.dequantize(oe, oc, os_, cols, bs))
