"""Which products go to the large tiles, and what the host does on the way, without a GPU."""

import pytest
import torch

from fastgen_amd.kernels import KernelArgumentError, _lib, linear, ops


class OnGpu(torch.Tensor):
    """A tensor that says that it is on a GPU."""

    is_cuda = True


def on_gpu(*shape, dtype=torch.bfloat16, device="cpu"):
    return torch.zeros(*shape, dtype=dtype, device=device).as_subclass(OnGpu)


@pytest.fixture
def calls(monkeypatch):
    """What reaches the kernels' libraries: (entry, arguments)."""
    seen = []

    class Library:
        def __getattr__(self, entry):
            return lambda *a: seen.append((entry, a)) or 0

    monkeypatch.setattr(_lib, "load", lambda name: Library())
    monkeypatch.setattr(ops, "_stream", lambda t: None)
    monkeypatch.setattr(ops, "_n_cus", 256)
    monkeypatch.setattr(linear, "force", None)
    monkeypatch.setattr(linear, "choices", {})
    return seen


def packed(n, k, device="cpu"):
    return ops.PackedWeight(on_gpu(-(-n // 16), -(-k // 32), 64, 8, device=device), n, k)


def test_operands_on_different_devices_are_refused(calls):
    for x, w in (("cpu", "meta"), ("meta", "cpu")):
        with pytest.raises(KernelArgumentError, match="different devices"):
            ops.gemm_large(on_gpu(20, 128, device=x), packed(32, 128, device=w))
    assert not calls
    ops.gemm_large(on_gpu(20, 128), packed(32, 128))
    assert [c[0] for c in calls] == ["fg_gemm_large"]
