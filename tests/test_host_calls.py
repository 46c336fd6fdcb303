"""What the library's host code asks of the HIP runtime, over a stand-in for
it (native/host_calls_check.cpp): runs without a GPU.

* adjoint_stray: the gradient with a per-step time step sums no entry that
  nothing wrote, also for a node of no element.
* densities_captured: the nodal mean densities are formed again after the
  densities changed, whatever was captured in between.
* densities_uniform: means are formed only where densities may differ.
* other_device: calls without a stream run on the context's device, whichever
  is current.
* passes_by_size, passes_by_option: whether a run takes the separate, the paired
  or the solo pass, on both sides of the lines and with every option that
  excludes one.
* pinned_memory, transfers: the transfers' pinned memory is shared, bounded and
  given back; they work without memory for the ring and from several threads.
"""
import os
import shutil
import subprocess

import pytest

from weldformfem_amd import _lib

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "native", "host_calls_check.cpp")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    out = str(tmp_path_factory.mktemp("host_calls") / "host_calls_check")
    subprocess.run([gxx, "-O1", "-std=c++17", "-pthread", "-rdynamic", SRC, "-ldl", "-o", out], check=True,
                   capture_output=True)
    return out


CHECKS = ["adjoint_stray", "densities_captured", "densities_uniform", "other_device_fp64", "other_device_mixed",
          "pinned_memory", "transfers", "passes_by_size", "passes_by_option"]


@pytest.mark.parametrize("check", CHECKS)
def test_host_calls(program, check):
    r = subprocess.run([program, _lib.LIB_PATH, check], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
