"""Runs the native port of the reference's board tests (tests/cpp/npu_backend_test.cpp)
against the C++ npu::Backend / npu::Linear mirror, and the checks of the host-buffer calls'
host side (tests/cpp/host_calls_test.cpp), which need no GPU."""
import os
import subprocess

import pytest

BUILD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "_build")
BIN = os.path.join(BUILD, "npu_backend_test")
HOST_BIN = os.path.join(BUILD, "host_calls_test")


def _run_bin(path, mode, timeout):
    if not os.path.exists(path):
        pytest.fail(f"{path} is not built: run python -m open_rknpu2_lm_infer_amd.build")
    r = subprocess.run([path, mode], capture_output=True, text=True, timeout=timeout)
    print(r.stdout[-4000:])
    assert r.returncode == 0, r.stdout[-4000:] + r.stderr[-2000:]
    return r.stdout


def _run(mode, timeout):
    assert f"PASS {mode} tests" in _run_bin(BIN, mode, timeout)


def test_npu_mirror_host_logic():
    _run("cpu", 60)


@pytest.mark.parametrize("mode", ["exit", "no_pinned", "capture", "blocks"])
def test_host_calls(mode):
    assert f"PASS {mode}" in _run_bin(HOST_BIN, mode, 60)


@pytest.mark.gpu
def test_npu_mirror_reference_board_tests():
    _run("gpu", 110)
