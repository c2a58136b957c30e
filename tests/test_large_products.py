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
    x, w = on_gpu(70, 1088), linear.StreamedMatrix(on_gpu(1040, 1088), packed(1040, 1088))
    for _ in range(3):
        linear.linear(x, w, partials_ok=True)
        linear.linear(x, w, epilogue="silu_mul")
        linear.qkv_parts(x, w)
        first = list(asked) if not calls[3:] else first
    assert names(calls) == {"fg_gemm_large"} and len(calls) == 9
    assert set(asked) == {"large_whole_tiles", "large_plan", "parts_plan"} and asked == first


def test_which_kernel_takes_a_product(calls, monkeypatch):
    """Rows, k, strides, alignment and epilogues that the large tiles and the wide kernel take without a measurement, and those that go
    other ways or are refused."""
    monkeypatch.setattr(linear, "_settle", lambda what, n, k, rows, candidates, *a, **b: candidates[-1][0])
    monkeypatch.setattr(torch.nn.functional, "linear", lambda x, w: on_gpu(x.shape[0], w.shape[0]))

    def took(M, N, K, more, ldx=0, matrix=None):
        calls.clear()
        x = on_gpu(M, ldx or K)[:, :K].as_subclass(OnGpu)
        linear.linear(x, linear.StreamedMatrix(on_gpu(N, K), packed(N, K)) if matrix is None else matrix, **more)
        entries = [entry for entry in names(calls) if entry in (large, wide)]
        return entries[0] if entries else False

    large, wide = "fg_gemm_large", "fg_gemm_skinny64"
    parts, gated, f32 = {"partials_ok": True}, {"epilogue": "gelu_tanh_mul"}, {"out_dtype": torch.float32}
    for M, N, K, more, want in [(16, 64, 64, gated, False), (32, 64, 64, gated, wide), (33, 64, 64, gated, large), (17, 20480, 64, gated, large),
                                (64, 64, 1088, gated, wide), (65, 64, 1088, gated, large), (40, 64, 72, gated, False),
                                (33, 64, 72, parts, False), (33, 40, 128, parts, large), (32, 40, 128, parts, wide), (17, 4096, 4096, parts, large),
                                (512, 64, 64, {}, False), (513, 64, 64, {}, large), (513, 64, 96, {}, False), (513, 64, 4096, {}, False),
                                (513, 64, 4096, f32, large), (40, 24576, 64, f32, large), (40, 24575, 64, f32, False), (129, 24576, 64, f32, False),
                                (385, 24576, 64, f32, large), (129, 49152, 64, f32, large), (513, 64, 64, f32, large), (40, 64, 64, dict(parts, **f32), False)]:
        assert took(M, N, K, more) == want, (M, N, K, more)
    assert took(40, 64, 64, gated, ldx=72) == large and not took(40, 64, 64, gated, ldx=68)
    assert not took(40, 64, 64, gated, matrix=on_gpu(64, 64))  # no packed copy
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


@pytest.mark.parametrize("gated,partials", [(False, False), (False, True), (True, False)])
def test_large_plan_fits(monkeypatch, gated, partials):
    """Whatever the sizes: a tile that the kernel has, no empty split of k, no more workgroups than places where k is cut, and
    partial sums within the room that is kept for them; more than 64 rows of a small product go to tiles of 64 rows."""
    monkeypatch.setattr(ops, "_n_cus", 256)
    small = 0
    for M in (17, 64, 65, 100, 128, 129, 300, 512, 513, 1000, 2049, 4096, 16384):
        for N in (16, 512, 1040, 2048, 4096, 11264, 28672):
            for K in (64, 320, 704, 1408, 2048, 4096, 14336):
                tile, splits = ops.large_plan(M, N, K, gated, partials)
                assert tile in ops.LARGE_TILES and (not gated or tile % 1000 != 192)
                steps, tiles = K // 64, -(-M // (tile // 1000)) * -(-N // (tile % 1000))
                assert splits == 1 or (partials and -(-steps // splits) * (splits - 1) < steps and tiles * splits <= 512 and steps // splits >= 5
                                       and splits * M * N * 4 <= ops.gemm_large_scratch(M, N))
                small += M > 64 and tile == 64128
    assert small > 50


def test_expert_tile_rows():
    """Tiles of few rows while the experts get few, of 64 to 128 rows beyond, of 256 for one or two a expert where enough workgroups with a
    long k are left; sizes that the large tiles do not take keep their tiles."""
    from fastgen_amd.parts.moe import expert_tile_rows

    for per, E, D, F, want in [(9.9, 32, 2048, 768, 16), (10, 32, 2048, 768, 128), (111, 32, 2048, 768, 128), (112, 32, 2048, 768, 256),
                               (288, 32, 2048, 768, 256), (289, 32, 2048, 768, 128), (13, 8, 2048, 3584, 16), (14, 8, 2048, 3584, 128),
                               (150, 8, 2048, 3584, 128), (150, 32, 1024, 2048, 128), (150, 16, 4096, 2048, 256), (150, 16, 2048, 704, 128),
                               (13, 4, 96, 100, 16), (14, 4, 96, 100, 32), (24, 4, 96, 100, 128), (24, 4, 96, 24, 32)]:
        assert expert_tile_rows(per, E, D, F) == want, (per, E, D, F)
