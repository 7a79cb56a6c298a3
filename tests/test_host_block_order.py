"""Block order of the z-stencil passes (csrc/lbm_common.h), compiled for the host."""
from __future__ import annotations

import os
import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc needed")
def test_block_order_by_size(tmp_path):
    exe = tmp_path / "block_order"
    subprocess.run([HIPCC, "--offload-host-only", "-std=c++17", "-O1", str(HERE / "host_abi" / "block_order.hip"),
                    "-o", str(exe)], check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    p = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, timeout=60)
    assert p.returncode == 0, p.stdout
