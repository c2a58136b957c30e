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


def names(calls):
    return {entry for entry, _ in calls}


@pytest.mark.parametrize("rows", [100, 300])
def test_a_forced_kernel_is_the_one_of_that_name(calls, monkeypatch, rows):
    """"tiled" is the tiled kernel also where the large tiles can take the matrix; "large" are those, where they can, also in
    products that their rule leaves to others."""
    x, w = on_gpu(rows, 128), linear.StreamedMatrix(on_gpu(512, 128), packed(512, 128))
    monkeypatch.setattr(linear, "force", "tiled")
    linear.linear(x, w, partials_ok=True)
    monkeypatch.setattr(linear, "force", "tiled256")
    linear.linear(x, w, epilogue="silu_mul")
    assert names(calls) == {"fg_gemm_tiled"}
    calls.clear()
    monkeypatch.setattr(linear, "force", "large")
    for more in ({}, {"partials_ok": True}, {"epilogue": "silu_mul"}, {"out_dtype": torch.float32}):
        linear.linear(x, w, **more)
    assert names(calls) == {"fg_gemm_large"}
    monkeypatch.setattr(linear, "force", "library")
    assert linear.qkv_parts(on_gpu(100, 1024), linear.StreamedMatrix(on_gpu(1024, 1024), packed(1024, 1024))) is None
    monkeypatch.setattr(linear, "force", None)
    assert linear.qkv_parts(on_gpu(100, 1024), linear.StreamedMatrix(on_gpu(1024, 1024), packed(1024, 1024))) is not None
