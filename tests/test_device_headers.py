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


def test_jacobi_sweeps_with_equal_eigenvalues(tmp_path_factory):
    """Equal eigenvalues (the fits of cubic and icosahedral clusters) take no more
    sweeps than distinct ones."""
    spectra = [(0, 1, 2, 3), (0, 1, 1, 2), (0, 1, 1, 1), (0, 0, 1, 1), (1, 1, 1, 1), (0, 0, 0, 0),
               (1e-3, 4000, 4001, 4002), (0, 1, 1, 1 + 1e-7)]
    spectra = [s + (off,) for off in (0, 1e-12, 1e-9, 1e-6, 1e-3) for s in spectra]
    r = subprocess.run([build(tmp_path_factory, "jacobi")] + [repr(float(v)) for s in spectra for v in s],
                       capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    for spec, line in zip(spectra, r.stdout.splitlines()):
        sweeps, err, orth = line.split()
        assert int(sweeps) <= 8, (spec, line)
        # the matrix is rounded as it is formed (four terms an entry), then once a
        # rotation of a row; V by three roundings in each of at most 48 rotations
        assert float(err) <= 16 * 2.0 ** -52 and float(orth) <= 48 * 3 * 2.0 ** -53, (spec, line)


@pytest.mark.parametrize("atoms,angle,noise", [(13, 1e-4, 0.02), (13, 1.0, 0.02), (1000, 1e-2, 0.02),
                                               (1000, 1.0, 0.02), (100, 1.0, 1.0)])
def test_fitted_distance_is_that_of_its_matrix(tmp_path_factory, atoms, angle, noise):
    """The smallest eigenvalue within a rounding, half of it after the root,
    which rounds once more: 2^-52 together, however far the larger eigenvalues lie."""
    r = subprocess.run([build(tmp_path_factory, "fit"), str(atoms), str(angle), str(noise)],
                       capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    assert float(r.stdout) <= 2.0 ** -52


def test_finish_takes_eight_wavefronts_only_where_they_win(tmp_path_factory):
    """Batches on both sides of each line of the rule, as measured."""
    rule = {(1, 0, 38): 64, (4096, 0, 191): 64, (1, 0, 192): 256, (64, 0, 512): 256,
            (64, 64, 513): 512, (256, 256, 1000): 512, (4096, 1, 600): 512, (4064, 64, 600): 512,
            (4128, 128, 600): 256, (1024, 1024, 600): 256,
            (320, 320, 600): 256, (512, 512, 700): 256, (1280, 256, 600): 256}
    r = subprocess.run([build(tmp_path_factory, "finish_rule")] + [str(v) for k in rule for v in k],
                       capture_output=True, text=True, timeout=60)
    assert [int(v) for v in r.stdout.split()] == list(rule.values())
