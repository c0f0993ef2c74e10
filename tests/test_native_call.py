"""The native call path from torch tensors (csrc/torch_call.cpp)."""
import os
import subprocess

import pytest
import torch

from epure import PackedLinear, PackedWeight
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
