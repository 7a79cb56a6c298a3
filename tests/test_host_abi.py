"""The C ABI's host code without a device: csrc/abi.hip compiled for the host
against a stand-in runtime and stand-in launchers (tests/host_abi/stubs.h), one
program per question.  Nothing runs on a GPU."""
from __future__ import annotations

import os
import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
ABI = HERE.parent / "pour-over-coffee-lbm_amd" / "csrc" / "abi.hip"


def _hipcc():
    return shutil.which("hipcc") or ("/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else None)


pytestmark = pytest.mark.skipif(_hipcc() is None or shutil.which("g++") is None, reason="hipcc and g++ needed")


def _host_object(src, obj):
    subprocess.run([_hipcc(), "--offload-host-only", "-std=c++17", "-O1", "-fPIC", "-c", str(src), "-o", str(obj)],
                   check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    return obj


@pytest.fixture(scope="module")
def abi(tmp_path_factory):
    return _host_object(ABI, tmp_path_factory.mktemp("abi") / "abi.o")


def _run(abi, tmp_path, name):
    exe = tmp_path / name
    subprocess.run(["g++", "-o", str(exe), str(abi), str(_host_object(HERE / "host_abi" / (name + ".hip"), tmp_path / "t.o")),
                    "-Wl,--unresolved-symbols=ignore-all"], check=True)
    p = subprocess.run([str(exe)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert p.returncode == 0, p.stdout


def test_step_record_refuses_overlapping_states(abi, tmp_path):
    _run(abi, tmp_path, "step_record")


def test_a_failed_launch_leaves_nothing_queued(abi, tmp_path):
    _run(abi, tmp_path, "failed_launch")


def test_counts_start_from_zero_after_a_failed_call(abi, tmp_path):
    _run(abi, tmp_path, "counts")


def test_undefined_bits_of_what_do_nothing(abi, tmp_path):
    _run(abi, tmp_path, "what_bits")


def test_velocity_across_a_written_buffer_is_refused(abi, tmp_path):
    _run(abi, tmp_path, "thermal_velocity")


def test_creating_a_context_waits_for_nothing(abi, tmp_path):
    _run(abi, tmp_path, "create")
