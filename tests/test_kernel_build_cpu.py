"""What the compiler says about kernels with assembly in them."""
import os
import subprocess

import pytest

import build_ext


@pytest.mark.skipif(not os.path.exists(build_ext.HIPCC), reason="no HIP compiler")
def test_assembly_keeps_reserved_registers(tmp_path):
    """A reserved register (m0) in a clobber list is not kept track of: the compiler warns, and may go on with its old value."""
    cmd = [build_ext.HIPCC, f"--offload-arch={build_ext.ARCH}", "-O3", "-fPIC", "-std=c++17", *build_ext.NO_PACKED_FP32, "--offload-device-only",
           "-c", str(build_ext.HIP_DIR / "flash_attn.hip"), "-o", str(tmp_path / "o")]
    out = subprocess.run(cmd, capture_output=True, text=True, check=True).stderr
    assert "clobber" not in out, out[:500]
