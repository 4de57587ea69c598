"""Headers of the library on the CPU: workgroups emulated lane by lane
(tests/host/hip/hip_runtime.h), wavefronts running ahead of each other as far as
the barriers let them."""

import os
import subprocess

import numpy as np
import pytest
from scipy.optimize import linear_sum_assignment

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = os.path.join(ROOT, "tests", "host")
CLANG = os.environ.get("FO_HOST_CLANG", "/opt/rocm/llvm/bin/clang++")


def build(tmp_path_factory, name):
    exe = str(tmp_path_factory.mktemp("host") / name)
    r = subprocess.run([CLANG, "-O1", "-std=c++17", "-w", "-I", HOST, "-I",
                        os.path.join(ROOT, "fastoverlap_amd", "csrc"),
                        os.path.join(HOST, name + ".cpp"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


@pytest.fixture(scope="session")
def lap_block(tmp_path_factory):
    return build(tmp_path_factory, "lap_block")


@pytest.mark.parametrize("reverse", [0, 1])
@pytest.mark.parametrize("threads,n", [(64, 1), (64, 40), (128, 3), (128, 65), (256, 64), (512, 33)])
def test_assignment_search_in_any_wavefront_order(lap_block, threads, n, reverse):
    """Unrelated costs leave many free rows, each a search that ends at a
    barrier: no wavefront may still wait inside it when another has left."""
    r = subprocess.run([lap_block, str(threads), str(n), "7", str(reverse)],
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    rows, costs = r.stdout.splitlines()
    got = np.array(rows.split(), int)
    c = np.array(costs.split(), float).reshape(n, n)
    np.testing.assert_array_equal(got, linear_sum_assignment(c)[1])


def test_staging_buffers_change_hands_between_threads(tmp_path_factory):
    """Positions set while another thread reads the same batch, two readers and
    two writers: no buffer serves two batches, none is lost or freed twice."""
    r = subprocess.run([build(tmp_path_factory, "staging")], capture_output=True, text=True,
                       timeout=60)
    assert (r.returncode, r.stdout) == (0, "ok\n"), r.stdout + r.stderr
