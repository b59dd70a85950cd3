"""The step's kernels run on the host, threads as fibers, with every buffer between pages that cannot be
touched (host/kernel_bounds.cpp): no access lies outside a buffer, in either access form of the spectral
kernel, and launches meant to give the same bits give them."""

import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CXX = "/opt/rocm/llvm/bin/clang++"  # the kernels use its vector types


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not os.path.exists(CXX):
        pytest.skip("no clang++")
    exe = str(tmp_path_factory.mktemp("bounds") / "kernel_bounds")
    csrc = os.path.join(HERE, "..", "mhdflows.jl_amd", "csrc")
    host = os.path.join(HERE, "host")
    subprocess.run([CXX, "-x", "c++", "-std=c++17", "-O1", "-w", "-I", host, "-I", csrc,
                    os.path.join(host, "kernel_bounds.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("T", ["float", "double"])
def test_steps_stay_inside_their_buffers(program, T):
    r = subprocess.run([program, T], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stderr
