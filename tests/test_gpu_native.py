"""Runs the native (no Python in the measured program) parity test of the C ABI.

tests/native/test_mhc_layer is built beforehand (make -C tests/native, or __graft_entry__.build());
it compares every output of the dynamic and static layer calls with the plain-C fp64 oracle at
1e-5 and exits non-zero on any mismatch.
"""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
EXE = os.path.join(HERE, "native", "test_mhc_layer")


@pytest.mark.gpu
def test_native_operator_parity_executable():
    """tests/native/test_ops: mhc_sinkhorn_knopp_* and mhc_rmsnorm_* against the C oracle."""
    exe = os.path.join(HERE, "native", "test_ops")
    assert os.path.exists(exe), "build tests/native first (make -C tests/native)"
    p = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    print(p.stdout[-4000:])
    assert p.returncode == 0, p.stdout[-4000:] + p.stderr[-2000:]
    assert "all comparisons passed" in p.stdout


@pytest.mark.gpu
def test_native_parity_executable():
    assert os.path.exists(EXE), "build tests/native first (make -C tests/native)"
    p = subprocess.run([EXE], capture_output=True, text=True, timeout=100)
    print(p.stdout[-3000:])
    assert p.returncode == 0, p.stdout[-3000:] + p.stderr[-2000:]
    assert "all comparisons passed" in p.stdout


# the tables follow the kernels that ran: the tiled backward of four and of eight streams, and the two-launch one
@pytest.mark.gpu
@pytest.mark.parametrize("B,n,C,tiled", [(1280, 4, 512, True), (2000, 8, 1024, True), (64, 8, 512, False)])
def test_phase_profile_names_the_kernels_that_ran(B, n, C, tiled):
    exe = os.path.join(os.path.dirname(HERE), "mhc.cu_amd", "native", "phase_profile")
    p = subprocess.run([exe, "--batch", str(B), "--hidden", str(C), "--expansion", str(n)], capture_output=True, text=True, timeout=100)
    assert p.returncode == 0, p.stdout[-2000:] + p.stderr[-2000:]
    assert ("slab backward kernel" in p.stdout) == tiled and ("sample-resident backward kernel" in p.stdout) != tiled, p.stdout
