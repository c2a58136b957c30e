"""What the compiler makes of the prompt attention's kernels, as far as it decides how many workgroups a compute unit holds."""

import re
import shutil
import subprocess

import pytest

from fastgen_amd.kernels import _lib


@pytest.fixture(scope="module")
def hipcc():
    try:
        path = _lib._hipcc()
    except Exception:
        path = None
    if not path or not (shutil.which(path)):
        pytest.skip("no compiler")
    return path


@pytest.mark.parametrize("head_dim", [128, 224, 256])
def test_launch_for_both_kinds_keeps_a_units_workgroups(hipcc, tmp_path, head_dim):
    """The launch that takes decoded tokens beside prompt portions has the LDS of the one for portions alone, and as many waves
    fit a SIMD."""
    flags = [f for f in _lib.HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.run([hipcc, *flags, f"-DFG_HD={head_dim}", "-S", "--offload-device-only", f"-I{_lib.CSRC}", str(_lib.CSRC / "attention_mfma.hip"),
                    "-o", str(tmp_path / "listing")], check=True, capture_output=True, timeout=300)
    held = {}
    for name, body in re.findall(r"^(_Z\d+attn_tile_kernel\w+):(.*?^; Occupancy: \d+)", (tmp_path / "listing").read_text(), re.S | re.M):
        pages, pair, both = re.match(r"_Z\d+attn_tile_kernelILi(\d)ELb(\d)EJ(.*?)EE", name).groups()
        lds, waves = re.search(r"\.amdhsa_group_segment_fixed_size (\d+)", body), re.search(r"; Occupancy: (\d+)", body)
        held[pages, pair, "SplitPart" in both, "KeyParts" in both, "TwoSums" in both] = int(lds[1]), int(waves[1])
    forms = [f for f in held if f[2]]
    assert len(forms) == (4 if head_dim <= 128 else 1)
    for pages, pair, _, *more in forms:
        assert held[(pages, pair, True, *more)] == held[(pages, pair, False, *more)], (pages, pair, more)
