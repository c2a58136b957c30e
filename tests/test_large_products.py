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


def test_sizes_are_worked_out_once(calls, monkeypatch):
    """A step of a few dozen rows waits for the host: what depends on a product's sizes alone is not worked out at every call."""
    asked = []
    for name in ("large_whole_tiles", "large_plan", "parts_plan"):
        work = getattr(ops, name)
        monkeypatch.setattr(ops, name, lambda *a, name=name, work=work: asked.append(name) or work(*a))
    x, w = on_gpu(45, 1088), linear.StreamedMatrix(on_gpu(1040, 1088), packed(1040, 1088))
    for _ in range(3):
        linear.linear(x, w, partials_ok=True)
        linear.linear(x, w, epilogue="silu_mul")
        linear.qkv_parts(x, w)
    assert names(calls) == {"fg_gemm_large"} and len(calls) == 9
    assert sorted(asked) == ["large_plan"] * 2 + ["large_whole_tiles"] * 2 + ["parts_plan"]  # (two of the three are one tile and split)


def test_what_goes_to_the_large_tiles(calls, monkeypatch):
    """Rows, k, strides, alignment and epilogues that they take, and those that go other ways or are refused as before."""
    monkeypatch.setattr(linear, "_settle", lambda what, n, k, rows, candidates, *a, **b: candidates[-1][0])
    monkeypatch.setattr(torch.nn.functional, "linear", lambda x, w: on_gpu(x.shape[0], w.shape[0]))

    def large(M, N, K, more, ldx=0, matrix=None):
        calls.clear()
        x = on_gpu(M, ldx or K)[:, :K].as_subclass(OnGpu)
        linear.linear(x, linear.StreamedMatrix(on_gpu(N, K), packed(N, K)) if matrix is None else matrix, **more)
        return "fg_gemm_large" in names(calls)

    parts, gated, f32 = {"partials_ok": True}, {"epilogue": "gelu_tanh_mul"}, {"out_dtype": torch.float32}
    for M, N, K, more, want in [(16, 64, 64, gated, False), (17, 64, 64, gated, True), (17, 64, 72, gated, False),
                                (17, 64, 72, parts, False), (17, 40, 128, parts, True), (512, 64, 64, {}, False), (513, 64, 64, {}, True),
                                (513, 64, 96, {}, False), (40, 16384, 64, f32, True), (40, 16383, 64, f32, False), (513, 64, 64, f32, True),
                                (40, 64, 64, dict(parts, **f32), False)]:
        assert large(M, N, K, more) == want, (M, N, K, more)
    assert large(20, 64, 64, gated, ldx=72) and not large(20, 64, 64, gated, ldx=68)
    assert not large(20, 64, 64, gated, matrix=on_gpu(64, 64))  # no packed copy
    x = on_gpu(20, 64 + 8)
    for bad in (lambda: ops.gemm_large(x[:, :40], packed(64, 40)), lambda: ops.gemm_large(x[:, 1:65], packed(64, 64)),
                lambda: ops.gemm_large(x[:, :64], packed(64, 64), k_splits=2), lambda: ops.gemm_large(x[:, :64], packed(72, 64), None, True),
                lambda: ops.gemm_large(x[:, :64], packed(64, 64), torch.float32, True), lambda: ops.gemm_large(x[:0, :64], packed(64, 64)),
                lambda: ops.gemm_large(x[:, :64], packed(64, 64), tile=1), lambda: ops.gemm_large(x[:, :64], packed(64, 128))):
        for _ in range(2):  # (also when asked again)
            calls.clear()
            with pytest.raises(KernelArgumentError):
                bad()
            assert not calls


def test_parts_plan_leaves_whole_splits_and_a_workgroup_a_unit(monkeypatch):
    """Every split of k of the q/k/v product has at least 6 steps, none is empty, and there are no more workgroups than compute units."""
    monkeypatch.setattr(ops, "_n_cus", 256)
    cut = 0
    for M in (17, 32, 63, 64, 65, 96, 127, 128):
        for N in (48, 1536, 3072, 5120, 6144, 12288, 16384, 40000):
            for K in (64, 704, 768, 1152, 1536, 2048, 4096, 8192):
                tile, splits = ops.parts_plan(M, N, K)
                steps, wgs = K // 64, -(-M // (tile // 1000)) * -(-N // (tile % 1000))
                assert tile in (64128, 128128) and splits in (1, 2, 3, 4)
                assert splits == 1 or (wgs * splits <= 256 and steps // splits >= 6 and -(-steps // splits) * (splits - 1) < steps)
                cut += splits > 1
    assert cut > 100
