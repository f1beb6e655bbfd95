"""The row statistics kernels as they are compiled (CPU: hipcc cross-compiles)."""

import os
import re
import subprocess

import pytest

from rl_project_amd import build as B


def test_no_private_memory_in_lds(tmp_path):
    """No kernel keeps a thread's variables in LDS: the compiler indexes them
    through the launch packet, which lies in host memory (12 us per launch), and
    what LDS there is holds the waves' partials."""
    try:
        hipcc = B.hipcc()
    except RuntimeError:
        pytest.skip("hipcc not available")
    src, out = os.path.join(B.CSRC, "fl_rowstats.hip"), str(tmp_path / "rs.s")
    subprocess.run([hipcc, *B.HIPCC_FLAGS, "--offload-device-only", "-S", src, "-o", out], check=True, capture_output=True)
    text = open(out).read()
    assert len(re.findall(r"^\s*\.amdhsa_kernel ", text, flags=re.M)) == 18   # 3 dtypes, with and without KL, 3 splits
    assert set(re.findall(r"\.amdhsa_user_sgpr_dispatch_ptr (\d)", text)) == {"0"}
    assert set(re.findall(r"\.amdhsa_private_segment_fixed_size (\d+)", text)) == {"0"}
    assert max(map(int, re.findall(r"\.amdhsa_group_segment_fixed_size (\d+)", text))) <= 1024
