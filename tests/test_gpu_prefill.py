"""GPU parity of the prefill path (more than 64 activation rows) through the C ABI.

Oracles: the C restatement of the reference Rust kernel (kernel/src/lib.rs,
oracle/rowdot.c) where it finishes in seconds, and the closed form
y = x . (cb[idx] * scale)^T in float64 on the GPU (the exact f32 tile of
container.py:70-88, oracle/decoder.py dense_tile) for the large shapes.
Bar: max relative error 2e-3, normwise and per element with an rms floor.
The cases cover both tile heights (64 and 128 rows), K split into several
partial sums, N past the last 256-row tile, every x and output dtype,
accumulation, group sizes, and rows of very different magnitude.
"""
import numpy as np
import pytest
import torch

from epure import PackedWeight
from epure.kernels import _abi, cuda
from oracle import ref, rowdot
from oracle.decoder import dense_tile

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
TOL = 2e-3
# A bf16 output adds its own rounding on top: bf16 keeps 8 significant bits,
# so round-to-nearest moves a value by at most 2^-8 of itself (half an ulp of
# 2^-7) -- hence TOL + 2^-8 for bf16 outputs (normwise, so |y| <= max|y|).


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


def make(n, k, levels=16, group=128, seed=0):
    idx, packed, scale, cb = ref.synth_linear(n, k, levels, group, seed=seed)
    s = PackedWeight((n, k), packed, scale, cb.astype(np.float32), group, levels).to(DEV)
    return idx, packed, scale, cb, s


def rust_ref(x32, packed, scale, cb, n, k, levels, group):
    return rowdot.dequant_matmul(x32, ref.packed_2d(packed, n, k, levels),
                                 np.asarray(scale, np.float32), np.asarray(cb, np.float32), group,
                                 levels <= 16)


def f64_ref(x, s):
    """x . W^T in float64 on the GPU, W the exact f32 dequantized tile."""
    w = dense_tile(s.packed, s.scale, s.cb, s.out_features, s.in_features, s.group, s.levels)
    return (x.double() @ w.double().t()).cpu().numpy()


def x_bf16(m, k, seed, scale=1.0):
    x32 = ref.round_bf16((rng(seed).standard_normal((m, k)) * scale).astype(np.float32))
    return x32, torch.from_numpy(x32).to(DEV).to(torch.bfloat16)


def run(s, x, out_dtype=torch.float32, accumulate=False, out=None):
    print(f"case: N={s.out_features} K={s.in_features} M={x.shape[0]} levels={s.levels} "
          f"group={s.group} x={x.dtype} y={out_dtype} acc={accumulate}", flush=True)
    h = cuda._hot(s)
    if out is None:
        out = torch.empty((x.shape[0], s.out_features), device=DEV, dtype=out_dtype)
    y = cuda.forward(x, h, out=out, accumulate=accumulate)
    assert y is not None, f"declined: {_abi.last_error()}"
    torch.cuda.synchronize()
    return y


@pytest.mark.parametrize("levels", [16, 256])
@pytest.mark.parametrize("m", [65, 100, 256])
def test_prefill_vs_rust_order(levels, m):
    n, k = 300, 1024
    _, packed, scale, cb, s = make(n, k, levels, seed=m + levels)
    x32, x = x_bf16(m, k, m)
    assert_close(run(s, x).cpu().numpy(), rust_ref(x32, packed, scale, cb, n, k, levels, 128))


@pytest.mark.parametrize("levels", [16, 256])
@pytest.mark.parametrize("m,n,k", [(1024, 1024, 4096), (1500, 520, 2048), (128, 256, 8192),
                                   (2048, 256, 14336)])
def test_prefill_large_and_split(levels, m, n, k):
    """128-row tiles (4-bit, M >= 1024), ragged M and N, and small grids
    whose K is split into partial sums."""
    _, _, _, _, s = make(n, k, levels, seed=n + k + m)
    _, x = x_bf16(m, k, k + m)
    assert_close(run(s, x).cpu().numpy(), f64_ref(x, s))


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,k", [(96, 512), (160, 8192)])
def test_prefill_accumulate_and_out_dtypes(out_dtype, m, k):
    """One split (accumulation in the epilogue) and several (through the
    ordered reduction)."""
    n = 384
    _, _, _, _, s = make(n, k, seed=k + 1)
    _, x = x_bf16(m, k, k + 2)
    want = f64_ref(x, s)
    out_tol = TOL if out_dtype == torch.float32 else TOL + 2.0 ** -8
    assert_close(run(s, x, out_dtype).float().cpu().numpy(), want, out_tol)
    base = torch.from_numpy(rng(k + 3).standard_normal((m, n)).astype(np.float32)).to(DEV)
    out = base.to(out_dtype)
    start = out.float().cpu().numpy()
    run(s, x, out_dtype, accumulate=True, out=out)
    assert_close(out.float().cpu().numpy(), want + start, out_tol)


@pytest.mark.parametrize("xdt", [torch.float16, torch.float32])
def test_prefill_x_dtypes(xdt):
    n, k, m = 512, 2048, 200
    _, packed, scale, cb, s = make(n, k, seed=31)
    x32 = rng(32).standard_normal((m, k)).astype(np.float32)
    x = torch.from_numpy(x32).to(DEV).to(xdt)
    assert_close(run(s, x).cpu().numpy(), f64_ref(x, s))


@pytest.mark.parametrize("m", [80, 300])
@pytest.mark.parametrize("group,levels", [(32, 16), (64, 16), (16, 256), (256, 256), (96, 16), (48, 256)])
def test_prefill_groups(group, levels, m):
    """Both tilings: 64 and 128 activation rows (from M = 160 at 4 bits, 128
    at 8), each x 32 weight rows per wave.  Groups that
    neither divide the 64-wide k step nor are 64 * 2^i (96, 48) are served by
    the generic MFMA path."""
    n, k = 300, 1024 if 1024 % group == 0 else 1152
    _, packed, scale, cb, s = make(n, k, levels, group=group, seed=group)
    x32, x = x_bf16(m, k, group)
    assert_close(run(s, x).cpu().numpy(), rust_ref(x32, packed, scale, cb, n, k, levels, group))


def test_prefill_levels_below_16_read_zero():
    n, k, m = 64, 512, 70
    idx = rng(3).integers(0, 16, (n, k), dtype=np.uint8)
    packed = ref.pack4(idx, 16)
    cb = np.sort(rng(4).standard_normal(10)).astype(np.float16)
    scale = (np.abs(rng(5).normal(0, 0.02, (n, 4))) + 1e-3).astype(np.float16)
    s = PackedWeight((n, k), packed, scale, cb.astype(np.float32), 128, 10).to(DEV)
    x32, x = x_bf16(m, k, 6)
    assert_close(run(s, x).cpu().numpy(), rust_ref(x32, packed, scale, cb, n, k, 10, 128))


def test_prefill_rows_of_very_different_magnitude():
    n, k, m = 256, 2048, 80
    _, _, _, _, s = make(n, k, seed=41)
    mags = np.ones(m, np.float32)
    mags[:4] = [3e5, 1e-12, 1e-30, 0.0]
    x32 = ref.round_bf16((rng(42).standard_normal((m, k)) * mags[:, None]).astype(np.float32))
    x = torch.from_numpy(x32).to(DEV).to(torch.bfloat16)
    y = run(s, x).cpu().numpy()
    want = f64_ref(x, s)
    for r in [0, 1, 2] + list(range(4, m)):
        assert_close(y[r:r + 1], want[r:r + 1])
    assert np.all(y[3] == 0.0)


def test_prefill_deterministic():
    n, k, m = 512, 8192, 128  # split K
    _, _, _, _, s = make(n, k, seed=51)
    _, x = x_bf16(m, k, 52)
    a = run(s, x).cpu().numpy()
    b = run(s, x).cpu().numpy()
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def test_batch1_8bit_long_k_stays_on_the_gemv():
    """Batch-1 8-bit at K = 14336 is served by the LUT GEMV (~22 us per
    4096 x 14336 launch); a shape-check slip once routed it to the MFMA tile
    path (~450 us).  The bar leaves 2.5x headroom over the GEMV's time."""
    n, k = 4096, 14336
    _, packed, scale, cb = ref.synth_linear(n, k, 256, 128, seed=77)
    s = PackedWeight((n, k), packed, scale, cb.astype(np.float32), 128, 256).to(DEV)
    x = torch.randn(1, k, device=DEV).to(torch.bfloat16)
    h = cuda._hot(s)
    for _ in range(3):
        cuda.forward(x, h)
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(20):
        cuda.forward(x, h)
    e1.record()
    torch.cuda.synchronize()
    us = e0.elapsed_time(e1) / 20 * 1e3
    assert us < 60.0, f"{us:.1f} us per launch"


@pytest.mark.parametrize("levels,group", [(16, 128), (16, 32), (256, 128), (256, 16)])
@pytest.mark.parametrize("m,n,k", [(5, 515, 1024), (32, 300, 512), (33, 257, 4096), (64, 256, 64),
                                   (65, 130, 2048), (161, 513, 1088), (1024, 300, 512),
                                   (32, 70, 832), (32, 70, 1024), (64, 70, 192), (64, 70, 256), (200, 70, 448),
                                   (200, 70, 640)])
def test_f32_scales_on_the_tiles(levels, group, m, n, k):
    """f32 group scales (a fine-tuned store's) on the tile kernel at the edges
    of its row tiles (32, 64, 128), with K split and whole, and on the generic
    one on either side of the shortest rows the tiles take, against the f64
    product of its operands: fp16(fp16(cb) * fp16(scale)) and x, exact in
    fp16.  What is left is the f32 sum of K <= 4096 products in some order,
    at most K * 2^-24 = 2.5e-4 of the sum of their magnitudes and far less of
    the result: held to 1e-4 of it."""
    _, packed, scale, cb, _ = make(n, k, levels, group, seed=m + n + k)
    f32 = (np.asarray(scale, np.float32) * np.float32(1.0003)).astype(np.float32)
    s = PackedWeight((n, k), packed, f32, cb.astype(np.float32), group, levels).to(DEV)
    assert s.scale.dtype == torch.float32
    _, x = x_bf16(m, k, m)
    want = (x.double() @ s.materialize(torch.float16).double().t()).cpu().numpy()
    assert_close(run(s, x).cpu().numpy(), want, 1e-4)


def graph_us(s, x, calls=20):
    """us a call of the packed linear's kernels, replayed as a graph."""
    h = cuda._hot(s)
    out = torch.empty((x.shape[0], s.out_features), device=DEV, dtype=x.dtype)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert cuda.forward(x, h, out=out) is not None
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for _ in range(calls):
            cuda.forward(x, h, out=out)
    best = float("inf")
    for _ in range(6):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        graph.replay()
        e0.record()
        graph.replay()
        e1.record()
        e1.synchronize()
        best = min(best, e0.elapsed_time(e1) * 1e3 / calls)
    return best


@pytest.mark.parametrize("levels,m,n,k", [(16, 1024, 8192, 1024), (16, 2048, 2048, 1024), (16, 32, 2048, 64),
                                          (256, 32, 512, 512), (256, 5, 8192, 256), (256, 2048, 512, 128)])
def test_f32_scales_no_slower_than_the_generic_tiles(levels, m, n, k):
    """Against the same layer with bf16 scales, which the generic MFMA kernel
    serves: within 15% where its plan, row count or row length made the tile
    kernel 1.2 to 2 times slower."""
    _, _, _, _, s = make(n, k, levels, 64, seed=m + n)
    _, x = x_bf16(m, k, m)
    stores = [PackedWeight((n, k), s.packed, s.scale.to(dt), s.cb, 64, levels)
              for dt in (torch.float32, torch.bfloat16)]
    f32, generic = (graph_us(t, x) for t in stores)
    assert f32 < 1.15 * generic, (f32, generic)


@pytest.mark.parametrize("m,n,k", [(1024, 8192, 128), (1024, 8193, 128), (1040, 7168, 192), (2048, 4096, 6144),
                                   (2048, 4096, 6208), (4096, 300, 512)])
def test_one_and_two_weight_tiles(m, n, k):
    """4-bit prompts of 1024 rows and more on both sides of the one-tile
    rule (one round of workgroups, rows of up to 6144 values), against the
    f64 product of the operands (fp16 x, fp16 weights).  What is left is the
    f32 sum of K products in some order: at most K * 2^-24 = 3.7e-4 of the
    sum of their magnitudes and far less of the result, held to 1e-4 of it."""
    _, _, _, _, s = make(n, k, 16, 64, seed=m + n + k)
    x = torch.randn(m, k, generator=torch.Generator(device=DEV).manual_seed(m), device=DEV).to(torch.float16)
    want = x.double() @ s.materialize(torch.float16).double().t()
    assert (run(s, x).double() - want).abs().max() <= 1e-4 * want.abs().max()


@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("k", [64, 512, 576, 1024, 1088, 2112, 4160, 8256, 16384, 16448])
def test_row_prep_row_lengths(k, xdt):
    """The row exponents and fp16 activations at row lengths on either side of
    every split of a row over threads (64 / 128 / 256 threads, 1 / 2 / 4 / 8
    pieces each, and pieces past 8), from a view with a longer row stride,
    each row's largest value in another place.  Against the f64 product of x
    and the fp16 weights: fp16 rounds each x to 2^-11 of itself at most,
    independently, so a row's sums move by about 2^-11 of their own rms (K
    terms on both sides), and their largest deviation of 128 by less than
    four times that, against the largest of the row."""
    m, n = 70, 128
    _, packed, scale, cb, s = make(n, k, 16, 64, seed=k)
    x32 = rng(k + 1).standard_normal((m, k + 8)).astype(np.float32)
    x32 *= np.exp2(rng(k + 2).integers(-12, 8, (m, 1))).astype(np.float32)
    x32[np.arange(m), (np.arange(m) * 977) % k] *= 64.0
    x = torch.from_numpy(x32).to(DEV).to(xdt)[:, :k]
    want = (x.double() @ s.materialize(torch.float16).double().t()).cpu().numpy()
    y = run(s, x).double().cpu().numpy()
    rows = np.abs(want).max(1, keepdims=True)
    assert (np.abs(y - want) / rows).max() <= 4 * 2.0 ** -11
