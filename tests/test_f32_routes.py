"""Which kernels take a 32-bit product and what is behind it (no GPU: the launches are recorded)."""

import pytest
import torch

from fastgen_amd.kernels import ops


@pytest.fixture
def launched(monkeypatch):
    """The entries that are called, in order."""
    names = []

    class Recorder:
        def __getattr__(self, name):
            return lambda *a: names.append(name) or 0

    monkeypatch.setattr(ops._lib, "load", lambda name: Recorder())
    monkeypatch.setattr(ops, "_gpu", lambda *t: None)
    monkeypatch.setattr(ops, "_stream", lambda t: 0)
    monkeypatch.setattr(ops, "compute_units", lambda: 256)
    return names


def operands(M, N, K):
    x, w = torch.empty(1, K).expand(M, K), torch.empty(1, K).expand(N, K)
    cut = ops.CutWeight(torch.empty(-(-N // 16), K // 32, 3, 64, 8, dtype=torch.bfloat16), N, K)
    return x, w, cut


@pytest.mark.parametrize("M,N,K,in_norm", [(4, 5120, 13824, True), (8, 6144, 6144, True), (9, 5120, 13824, False), (12, 6144, 6144, False),
                                           (64, 8192, 8192, False), (400, 5120, 5120, False), (64, 4096, 4096, True), (400, 3072, 8192, True)])
def test_sums_of_wide_rows_are_added_in_the_norm_for_few_rows_only(launched, M, N, K, in_norm):
    x, w, cut = operands(M, N, K)
    ops.gemm_f32_norm(x, w, torch.empty(M, N), torch.empty(N), 1e-5, cut)
    assert ("fg_gemm_f32_sum_norm" in launched) == in_norm and ("fg_add_rmsnorm" in launched) != in_norm


@pytest.mark.parametrize("M,N,K,parts", [(64, 3072, 8192, False), (49, 6144, 4096, False), (64, 11264, 2048, False), (64, 5120, 13824, False),
                                         (48, 11264, 2048, True), (65, 3072, 8192, True), (72, 6144, 4096, True), (64, 4096, 4096, True),
                                         (400, 3072, 8192, True), (16, 3072, 3072, False)])
def test_four_blocks_of_rows_of_a_large_matrix_stay_as_they_are(launched, M, N, K, parts):
    x, w, cut = operands(M, N, K)
    ops.gemm_f32(x, w, cut)
    ops.gemm_f32_norm(x, w, torch.empty(M, N), torch.empty(N), 1e-5, cut) if N <= 8192 else ops.gemm_f32_gated(x, w, "silu", cut)
    assert launched.count("fg_gemm_f32_parts") == launched.count("fg_gemm_f32_cut") == (2 if parts else 0)
