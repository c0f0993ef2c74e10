"""GPU parity of the row GEMV (`gemv_row_kernel`) at every row length it
serves: rows of 4, 8, 12, 16, 24, 28 and 32 slabs of 256 bytes (and 56 with
8-bit indices), i.e. K = 2048 .. 16384 with 4-bit indices and 1024 .. 14336
with 8-bit.  A wave owns whole rows: 1, 2 or 4 rows per wave and 3 to 14
loads per lane, activations staged by 1 or 2 chunks per thread; rows of 4, 8
and 16 slabs also take 2..4 activation rows per launch, which share each
load's table lookups.

Oracle: the C restatement of the reference Rust kernel (kernel/src/lib.rs:
36-151, oracle/rowdot.c).  Bar: max relative error 2e-3, normwise and per
element with an rms floor (bf16 / fp16 outputs add their own rounding).
"""
import numpy as np
import pytest
import torch

from epure import PackedWeight
from epure.kernels import _abi, cuda
from oracle import ref, rowdot

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
TOL = 2e-3


def rng(seed):
    return np.random.Generator(np.random.PCG64(seed))


def assert_close(y, r, tol=TOL):
    y = np.asarray(y, np.float64)
    r = np.asarray(r, np.float64)
    assert y.shape == r.shape
    assert np.isfinite(y).all()
    err = np.abs(y - r)
    scale = np.abs(r).max()
    assert err.max() <= tol * scale, f"normwise {err.max() / scale:.3e}"
    floor = np.sqrt(np.mean(r ** 2))
    rel = (err / np.maximum(np.abs(r), floor)).max()
    assert rel <= tol, f"per-element {rel:.3e}"


def case(n, k, levels, x_dtype, scale_f32, seed, out_dtype=torch.float32, accumulate=False):
    _, packed, scale, cb = ref.synth_linear(n, k, levels, 128, seed=seed)
    s = PackedWeight((n, k), packed, scale.astype(np.float32 if scale_f32 else np.float16),
                     cb.astype(np.float32), 128, levels).to(DEV)
    x32 = rng(seed + 1).standard_normal((1, k)).astype(np.float32)
    if x_dtype == torch.bfloat16:
        x32 = ref.round_bf16(x32)
    x = torch.from_numpy(x32).to(DEV).to(x_dtype)
    x_in = x.float().cpu().numpy()
    want = rowdot.dequant_matmul(x_in, ref.packed_2d(packed, n, k, levels), np.asarray(scale, np.float32),
                                 np.asarray(cb, np.float32), 128, levels <= 16)
    print(f"case: row GEMV N={n} K={k} levels={levels} x={x_dtype} f32 scales={scale_f32} "
          f"y={out_dtype} acc={accumulate}", flush=True)
    h = cuda._hot(s)
    out = torch.from_numpy(rng(seed + 2).standard_normal((1, n)).astype(np.float32)).to(DEV).to(out_dtype)
    start = out.float().cpu().numpy()
    y = cuda.forward(x, h, out=out, accumulate=accumulate)
    assert y is not None, f"declined: {_abi.last_error()}"
    torch.cuda.synchronize()
    tol = TOL if out_dtype == torch.float32 else TOL + 2.0 ** -8
    assert_close(out.float().cpu().numpy(), want + (start if accumulate else 0.0), tol)


# (levels, K): slabs of a row = K / 512 (4-bit) or K / 256 (8-bit)
ROWS = [(16, 2048), (16, 4096), (16, 6144), (16, 8192), (16, 12288), (16, 14336), (16, 16384),
        (256, 1024), (256, 3072), (256, 4096), (256, 6144), (256, 7168), (256, 8192), (256, 14336)]


@pytest.mark.parametrize("levels,k", ROWS)
@pytest.mark.parametrize("x_dtype", [torch.bfloat16, torch.float32])
def test_row_gemv_lengths(levels, k, x_dtype):
    """Every row length, a ragged N (not a multiple of any workgroup's rows),
    bf16 activations and f32 ones (hi and lo fp16 terms)."""
    case(300, k, levels, x_dtype, False, seed=k + levels)


@pytest.mark.parametrize("levels,k", [(16, 6144), (16, 14336), (256, 14336)])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_row_gemv_f32_scales_and_accumulate(levels, k, out_dtype):
    """f32 group scales (after make_trainable: one 32-bit load per scale) and
    accumulation into y, fp16 activations."""
    case(1000, k, levels, torch.float16, True, seed=3 * k + levels, out_dtype=out_dtype, accumulate=True)


def case_m(m, n, k, levels, x_dtype, seed, out_dtype=torch.float32, accumulate=False, ld_pad=0):
    _, packed, scale, cb = ref.synth_linear(n, k, levels, 128, seed=seed)
    s = PackedWeight((n, k), packed, scale.astype(np.float16), cb.astype(np.float32), 128, levels).to(DEV)
    x32 = rng(seed + 1).standard_normal((m, k + ld_pad)).astype(np.float32)
    if x_dtype == torch.bfloat16:
        x32 = ref.round_bf16(x32)
    wide = torch.from_numpy(x32).to(DEV).to(x_dtype)
    x = wide[:, :k]
    x_in = x.float().cpu().numpy()
    want = rowdot.dequant_matmul(np.ascontiguousarray(x_in), ref.packed_2d(packed, n, k, levels),
                                 np.asarray(scale, np.float32), np.asarray(cb, np.float32), 128, levels <= 16)
    print(f"case: row GEMV M={m} N={n} K={k} levels={levels} x={x_dtype} y={out_dtype} "
          f"acc={accumulate} ld={k + ld_pad}", flush=True)
    h = cuda._hot(s)
    out = torch.from_numpy(rng(seed + 2).standard_normal((m, n)).astype(np.float32)).to(DEV).to(out_dtype)
    start = out.float().cpu().numpy()
    y = cuda.forward(x, h, out=out, accumulate=accumulate)
    assert y is not None, f"declined: {_abi.last_error()}"
    torch.cuda.synchronize()
    tol = TOL if out_dtype == torch.float32 else TOL + 2.0 ** -8
    assert_close(out.float().cpu().numpy(), want + (start if accumulate else 0.0), tol)


# rows of 4, 8 and 16 slabs with 2..4 activation rows (the row kernel takes
# up to 4 with 4-bit indices, 2 with 4-bit rows of 16 slabs and with 8-bit
# indices; the other cases check the kernels that serve them instead)
@pytest.mark.parametrize("levels,k,m", [(16, 2048, 2), (16, 2048, 4), (16, 4096, 3), (16, 8192, 2),
                                        (256, 1024, 2), (256, 2048, 2), (256, 4096, 2), (256, 4096, 4)])
@pytest.mark.parametrize("x_dtype", [torch.bfloat16, torch.float16])
def test_row_gemv_several_rows(levels, k, m, x_dtype):
    """2, 3 (a zero-padded fourth row) and 4 activation rows share each
    load's table lookups; ragged N."""
    case_m(m, 300, k, levels, x_dtype, seed=7 * k + m + levels)


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_row_gemv_several_rows_strided_accumulate(out_dtype):
    """Activation rows further apart than K, results added into y."""
    case_m(4, 1000, 4096, 16, torch.bfloat16, seed=91, out_dtype=out_dtype, accumulate=True, ld_pad=96)
    case_m(2, 1000, 4096, 256, torch.bfloat16, seed=92, out_dtype=out_dtype, accumulate=True, ld_pad=96)


@pytest.mark.parametrize("levels,k,n", [
    (16, 2048, 28671), (16, 2048, 28673), (16, 4096, 14353), (16, 8192, 3585), (16, 8192, 8191),
    (16, 16384, 6145), (256, 1024, 28705), (256, 2048, 14337), (256, 4096, 7171), (256, 7168, 12289)])
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float16])
def test_row_gemv_streams_row_blocks(levels, k, n, xdt):
    """Layers of several rounds of workgroups, each streaming a share of the
    row blocks: counts of blocks that no share divides, shares of odd and
    even length, and a last block cut by N, against the f64 product of the
    operands (fp16 codebook values, f32 scales and sums: x is exact in both
    types)."""
    s = PackedWeight((n, k), *_random_store(n, k, levels), 128, levels).to(DEV)
    x = _random_x(k, xdt)
    y = cuda.forward(x, cuda._hot(s), out=torch.empty((1, n), device=DEV, dtype=torch.float32))
    assert y is not None, f"declined: {_abi.last_error()}"
    idx = s.packed.view(n, -1)
    if levels == 16:
        idx = torch.stack((idx & 15, idx >> 4), dim=-1).view(n, k)
    w = s.cb.double()[idx.long()] * s.scale.double().repeat_interleave(128, dim=1)
    want = (x.double() @ w.t())
    err = (y.double() - want).abs().max() / want.pow(2).mean().sqrt()
    # f32 sums of K products and an exact per-32 rescale of fp16-sized x:
    # K * 2^-24 = 1e-3 of the summed magnitudes at the longest row bounds it;
    # the sums' rounding is random and stays far below
    assert err < 1e-4, f"{float(err):.2e}"


def _random_store(n, k, levels):
    g = torch.Generator()
    g.manual_seed(n + k)
    packed = torch.randint(0, 256, (n * k // (2 if levels == 16 else 1),), generator=g, dtype=torch.uint8)
    cb = torch.sort(torch.randn(levels, generator=g)).values.half().float()
    scale = (torch.randn(n, k // 128, generator=g).abs() * 0.02 + 1e-3).half()
    return packed, scale, cb


def _random_x(k, xdt):
    g = torch.Generator()
    g.manual_seed(k)
    return torch.randn(1, k, generator=g).to(DEV).to(xdt)


@pytest.mark.parametrize("levels,k,n", [(16, 2048, 28673), (16, 6144, 7177), (16, 12288, 6149), (256, 3072, 7177),
                                        (256, 6144, 12293), (256, 14336, 6149)])
@pytest.mark.parametrize("scale_dt", [torch.float32, torch.bfloat16])
def test_row_gemv_streamed_blocks_of_other_scales(levels, k, n, scale_dt):
    """The streamed form with f32 and bf16 group scales (their own
    instantiation and conversion), rows of 12, 24 and 56 slabs, and results
    added to a 16-bit y: against the f64 product of the operands plus y, the
    sum rounded to y's type once."""
    packed, scale, cb = _random_store(n, k, levels)
    s = PackedWeight((n, k), packed, scale.to(scale_dt), cb, 128, levels).to(DEV)
    print(f"case: streamed row GEMV N={n} K={k} levels={levels} scales={scale_dt}", flush=True)
    x = _random_x(k, torch.float16)
    y0 = torch.randn(1, n, generator=torch.Generator(device=DEV).manual_seed(n), device=DEV).half()
    y = cuda.forward(x, cuda._hot(s), out=y0.clone(), accumulate=True)
    assert y is not None, f"declined: {_abi.last_error()}"
    idx = s.packed.view(n, -1)
    if levels == 16:
        idx = torch.stack((idx & 15, idx >> 4), dim=-1).view(n, k)
    w = s.cb.double()[idx.long()] * s.scale.double().repeat_interleave(128, dim=1)
    want = x.double() @ w.t() + y0.double()
    # y's own rounding, 2^-11 of it, beside the sums' 1e-4 of the rms
    err = (y.double() - want).abs() - 2.0 ** -11 * want.abs()
    assert err.max() <= 1e-4 * want.pow(2).mean().sqrt()
