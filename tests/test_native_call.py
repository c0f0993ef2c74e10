"""The native call path from torch tensors (csrc/torch_call.cpp)."""
import os
import subprocess

import pytest
import torch
import torch.nn.utils.parametrize
import torch.utils._python_dispatch

from epure import PackedLinear, PackedWeight, make_trainable
from epure.kernels import _abi, cuda

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def host_store(n=16, k=128, group=32):
    g = torch.Generator().manual_seed(1)
    packed = torch.randint(0, 256, (n * k // 2,), generator=g, dtype=torch.uint8)
    scale = torch.rand(n, k // group, generator=g).half()
    return PackedWeight((n, k), packed, scale, torch.randn(16, generator=g), group, 16)


# ------------------------------------------------------------------ refusals (no GPU needed)
def test_host_tensors_are_refused():
    """The kernels would read host memory through the current device's
    stream: refused as torch.cuda.current_stream(x.device) does."""
    assert _abi._load() is not None, _abi.LOAD_ERROR
    h = cuda._hot(host_store())
    x = torch.zeros(8, h.K, dtype=torch.bfloat16)
    gy = torch.zeros(8, h.N, dtype=torch.bfloat16)
    with pytest.raises(ValueError):
        cuda.forward(x, h)
    with pytest.raises(ValueError):
        cuda.backward(gy, x, h)


class ModuleStore(torch.nn.Module):
    """A store of another class: sizes as properties, a group read from JSON."""

    def __init__(self, store):
        super().__init__()
        self.shape, self.levels, self.group = store.shape, store.levels, float(store.group)
        for name in ("packed", "scale", "cb"):
            self.register_buffer(name, getattr(store, name))

    @property
    def out_features(self):
        return self.shape[0]

    @property
    def in_features(self):
        return self.shape[1]


def test_store_sizes_need_not_be_instance_attributes(monkeypatch):
    """Sizes come from the store's attributes however they are defined; a
    host x is declined after them."""
    monkeypatch.setattr(cuda, "_AVAILABLE", True)
    s = ModuleStore(host_store())
    assert cuda.linear(torch.zeros(1, 128, dtype=torch.bfloat16), s) is None


def test_extension_is_rebuilt_with_the_c_header():
    """It calls the library through the header's function types: a changed
    signature has to reach it."""
    csrc = os.path.join(ROOT, "epure-runtime_amd", "csrc")
    out = os.path.abspath(_abi.TORCH_PATH)
    # -o: the other prerequisites count as old
    r = subprocess.run(["make", "-n", "-C", csrc, "-o", "torch_call.cpp", "-o",
                        os.path.join(ROOT, "epure-runtime_amd", "_build", "torch_id"),
                        "-W", os.path.join(ROOT, "include", "epure_hip.h"), out],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "torch_call.cpp" in r.stdout, r.stdout + r.stderr


# ------------------------------------------------------------------ without the extension
def test_library_serves_without_the_extension(monkeypatch):
    """An extension that is absent, or was built for another torch, costs the
    native call path only: the library stays loaded and is called by ctypes."""
    def broken(handle):
        raise ImportError("undefined symbol")
    for name in ("lib", "call", "LOAD_ERROR", "CALL_ERROR"):
        monkeypatch.setattr(_abi, name, None)
    monkeypatch.setattr(_abi, "_load_call", broken)
    assert _abi._load() is not None and _abi.LOAD_ERROR is None
    assert _abi.call is None and isinstance(_abi.CALL_ERROR, ImportError)
    h = cuda._hot(host_store())
    with pytest.raises((ValueError, RuntimeError)):     # the stream of a host tensor
        cuda.forward(torch.zeros(8, h.K, dtype=torch.bfloat16), h)


@pytest.mark.gpu
def test_calls_without_the_extension_are_the_same(monkeypatch):
    dev = torch.device("cuda:0")
    lin = PackedLinear(host_store(144, 256).to(dev))
    h = cuda._hot(lin.store)
    x = torch.randn(2, 12, 256, device=dev).to(torch.bfloat16)
    x2, gy = x.view(24, 256), torch.randn(24, 144, device=dev).to(torch.bfloat16)

    def results():
        acc = torch.ones(24, 144, device=dev)
        with torch.no_grad():
            y = lin(x)
        return [y, cuda.forward(x2, h), cuda.forward(x2, h, out=acc, accumulate=True),
                *cuda.backward(gy, x2, h), cuda.backward(gy, x2, h, need_cb=False, need_scale=False,
                                                         gx_dtype=torch.float32)[0]]
    native = results()
    assert _abi.call is not None, _abi.CALL_ERROR
    monkeypatch.setattr(_abi, "call", None)
    for a, b in zip(results(), native):
        assert a.dtype == b.dtype and torch.equal(a, b)
    assert cuda.backward(gy.float(), x2, h) is None          # declined on both


# ------------------------------------------------------------------ linear, on the GPU
DEV = torch.device("cuda:0")


def gpu_linear(levels=16, n=144, k=256, group=32):
    g = torch.Generator().manual_seed(levels + k)
    packed = torch.randint(0, 256, (n * k // (1 if levels > 16 else 2),), generator=g, dtype=torch.uint8)
    scale = (torch.rand(n, k // group, generator=g) + 0.1).half()
    return PackedLinear(PackedWeight((n, k), packed, scale, torch.randn(levels, generator=g), group, levels)).to(DEV)


def rows(m, k, dtype, seed=3):
    return torch.randn(m, k, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV).to(dtype)


def direct(lin, x):
    """What the kernels give for the contiguous rows of x."""
    y = cuda.forward(x.reshape(-1, x.shape[-1]).contiguous(), cuda._hot(lin.store))
    return y.view(*x.shape[:-1], -1)


def call(x, s):
    return _abi.call.linear(x, s.packed, s.scale, s.cb, s.out_features, s.in_features, s.levels, s.group,
                            cuda.SERVE_F32)


@pytest.mark.gpu
@pytest.mark.parametrize("levels", [16, 256])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_linear_takes_every_layout(levels, dtype):
    """1-D to 4-D x, a transposed one, every second column, rows further
    apart than K, a slice at an offset: the kernels' result for the same rows
    (bit for bit; with rows apart the same kernels run), in x's shape."""
    lin = gpu_linear(levels)
    k = lin.store.in_features
    x = rows(24, k, dtype)
    wide = rows(24, k + 8, dtype, 4)
    for v in (x[0], x[:1], x, x.view(2, 12, k), x.view(2, 3, 4, k), rows(k, 24, dtype, 5).t(),
              rows(24, 2 * k, dtype, 6)[:, ::2], wide[:, :k], wide[:, 8:], x[8:20], x.view(2, 12, k)[:, :5]):
        with torch.no_grad():
            y = lin(v)
        assert y.shape == (*v.shape[:-1], 144) and y.dtype == dtype and not y.requires_grad
        assert torch.equal(y, direct(lin, v)), (v.shape, v.stride())


@pytest.mark.gpu
def test_linear_serves_f32_only_when_asked(monkeypatch):
    lin = gpu_linear()
    x = rows(5, 256, torch.float32)
    with torch.no_grad():
        assert cuda.linear(x, lin.store) is None
        assert cuda.linear(x.to(torch.float64), lin.store) is None
        monkeypatch.setattr(cuda, "SERVE_F32", True)
        assert torch.equal(cuda.linear(x, lin.store), direct(lin, x))


@pytest.mark.gpu
def test_linear_runs_on_the_current_stream():
    lin = gpu_linear()
    x = rows(40, 256, torch.bfloat16)
    want = direct(lin, x)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.no_grad(), torch.cuda.stream(side):
        v = torch.zeros_like(x)
        for _ in range(50):      # the product is behind these on its stream, or reads zeros
            v.copy_(torch.zeros_like(x))
        v.copy_(x)
        y = lin(v)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    assert torch.equal(y, want)


@pytest.mark.gpu
def test_linear_reports_the_library_error():
    """Rows that overlap: refused by the library, as an exception."""
    lin = gpu_linear()
    x = rows(1, 256, torch.bfloat16).expand(8, 256)
    with torch.no_grad(), pytest.raises(RuntimeError, match="ep_dequant_matmul failed.*row length"):
        lin(x)


class Wrapped(torch.Tensor):
    pass


class FunctionMode(torch.overrides.TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class DispatchMode(torch.utils._python_dispatch.TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@pytest.mark.gpu
def test_linear_hands_back_what_torch_wants_to_see():
    """A tensor subclass, function and dispatch modes, a wrong or empty row
    and autograd take the path through torch's operators."""
    lin = gpu_linear()
    s, x = lin.store, rows(6, 256, torch.bfloat16)
    want = direct(lin, x)
    with torch.no_grad():
        assert torch.equal(call(x, s), want)
        assert call(x.as_subclass(Wrapped), s) is NotImplemented
        assert call(x[:, :128], s) is NotImplemented
        assert call(x[:0], s) is NotImplemented and lin(x[:0]).shape == (0, 144)
        for mode in (FunctionMode(), DispatchMode()):
            with mode:
                assert call(x, s) is NotImplemented
                y = lin(x)
            assert torch.equal(y, want)
        assert torch.equal(lin(x.as_subclass(Wrapped)).as_subclass(torch.Tensor), want)
    seen = []
    with torch.no_grad():
        torch.vmap(lambda v: seen.append(call(v, s)) or v)(x.view(2, 3, 256))
    assert seen == [NotImplemented]
    assert torch.equal(call(x, s), want)                  # grad mode, nothing requires grad
    assert call(x.clone().requires_grad_(True), s) is NotImplemented


@pytest.mark.gpu
def test_linear_of_a_trainable_store():
    """Without grad mode the native call; with it the autograd function."""
    lin = gpu_linear()
    make_trainable(torch.nn.Sequential(lin), "both", verbose=False)
    x = rows(6, 256, torch.bfloat16)
    with torch.no_grad():
        y = lin(x)
        assert call(x, lin.store) is not NotImplemented
    assert call(x, lin.store) is NotImplemented
    z = lin(x)
    assert z.requires_grad and torch.equal(z.detach(), y)
    z.float().sum().backward()
    assert lin.store.scale.grad is not None and lin.store.cb.grad is not None


class Doubled(torch.nn.Module):
    def forward(self, t):
        return 2 * t


@pytest.mark.gpu
def test_linear_of_a_parametrized_store():
    """A store whose scale is computed: its value, not a kept tensor."""
    lin = gpu_linear()
    x = rows(6, 256, torch.bfloat16)
    with torch.no_grad():
        y = lin(x)
        torch.nn.utils.parametrize.register_parametrization(lin.store, "scale", Doubled())
        assert torch.equal(lin(x), 2 * y)
