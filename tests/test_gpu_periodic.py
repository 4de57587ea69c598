"""GPU parity of the periodic path against the FP64 oracle (identical
argmax and permutation, distance within 1e-8, |f| grid within 1e-5 of its
maximum)."""

import sys

import numpy as np
import pytest

import fastoverlap_amd as fo
from fastoverlap_amd import _lib, workloads as W
from fastoverlap_amd.batch import PeriodicBatch
from oracle import fo_oracle as O

pytestmark = pytest.mark.gpu

DIST_TOL = 1e-8
GRID_TOL = 1e-5


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def test_structure_factors_match_oracle(gpu):
    say("case: calcFourierCoeff N=40 n=5")
    rng = np.random.default_rng(0)
    box = np.array([5.0, 6.0, 5.5])
    X = rng.random((40, 3)) * box * 1.7 - 2.0   # unwrapped coordinates
    groups = [np.arange(30), np.arange(30, 40)]
    pa = fo.PeriodicAlign(40, box, groups, n=5)
    C = pa.calcFourierCoeff(X)
    ref = O.PeriodicOracle(40, box, groups, n=5).calc_fourier_coeff(X)
    np.testing.assert_allclose(C, ref, atol=1e-11 * np.abs(ref).max())


def test_blj256_known_answer_dropin(gpu, blj256):
    say("case: BLJ256 PeriodicAlign drop-in (n=9, F=40)")
    p1, p2 = blj256
    box = np.ones(3) * 5.975206329
    groups = [np.arange(204), np.arange(204, 256)]
    pa = fo.PeriodicAlign(256, box, groups)
    dist, X1, X2, perm, disp = pa(p1, p2)
    P = O.PeriodicOracle(256, box, groups)
    (odist, oX1, oX2, operm, odisp), oind, ofabs = P.align(p1, p2)
    assert dist == pytest.approx(1.559, abs=1e-3)
    assert abs(dist - odist) <= DIST_TOL
    np.testing.assert_array_equal(perm, operm)
    assert tuple(pa.last["peaks"]["ind"][0]) == oind
    np.testing.assert_allclose(X2, oX2, atol=1e-9)
    # the attributes after a plain call describe that call's configuration:
    # |f|, the complex transform f (phase included) and the product C
    assert np.abs(pa.fabs - ofabs).max() <= GRID_TOL * ofabs.max()
    C, _ = P.overlap_grid(p1, p2)
    f = np.fft.fftn(C, P.fshape, axes=(0, 1, 2))
    assert np.abs(pa.f - f).max() <= GRID_TOL * np.abs(f).max()
    np.testing.assert_allclose(pa.C, C, atol=1e-11 * np.abs(C).max())
    np.testing.assert_allclose(np.abs(pa.f), pa.fabs, rtol=1e-5, atol=1e-6 * ofabs.max())


def test_c1_parity_64_grid(gpu):
    c = W.config1()
    say("case: C1 N=256 nk=8 F=64")
    with PeriodicBatch([256], c["box"], [0.3], 8, 64, [c["groups"]], 10,
                       _lib.PER_KEEP_GRID) as b:
        b.set_positions(c["pos1"], c["pos2"])
        b.run()
        r = b.results()
        pk = b.peaks()
        grid = b.grid(0)
    P = O.PeriodicOracle(256, c["box"], c["groups"], scale=0.3, n=8, fshape=(64, 64, 64))
    (odist, oX1, oX2, operm, odisp), oind, ofabs = P.align(c["pos1"], c["pos2"])
    assert tuple(pk["ind"][0]) == oind
    np.testing.assert_array_equal(r["perm"][0], operm)
    assert abs(r["dist"][0] - odist) <= DIST_TOL
    assert np.abs(grid - ofabs).max() <= GRID_TOL * ofabs.max()
    # the partner is a noisy permuted translate: the LAP recovers it
    np.testing.assert_array_equal(c["true_perm"][r["perm"][0]], np.arange(256))


def test_quick_align_with_coefficients(gpu, blj256):
    say("case: BLJ256 align with precomputed coefficients (Cs=)")
    p1, p2 = blj256
    box = np.ones(3) * 5.975206329
    groups = [np.arange(204), np.arange(204, 256)]
    pa = fo.PeriodicAlign(256, box, groups)
    c1, c2 = pa.calcFourierCoeff(p1), pa.calcFourierCoeff(p2)
    a = pa.align(p1, p2)
    b = pa.align(p1, p2, [c1, c2])
    assert a[0] == b[0]
    np.testing.assert_array_equal(a[3], b[3])


def test_align_group_matches_pairwise(gpu):
    say("case: alignGroup 3 structures N=64")
    rng = np.random.default_rng(8)
    box = np.full(3, 4.2)
    base = rng.random((64, 3)) * box
    coords = [base + rng.normal(scale=0.05, size=base.shape) + s
              for s in (0.0, 1.3, -0.6)]
    pa = fo.PeriodicAlign(64, box)
    D = pa.alignGroup(coords)
    P = O.PeriodicOracle(64, box)
    for i in range(3):
        for j in range(3):
            (od, *_), _, _ = P.align(coords[i], coords[j])
            assert abs(D[i, j] - od) <= DIST_TOL


def test_periodic_batch_independence(gpu):
    say("case: periodic batch of 6 vs alone")
    rng = np.random.default_rng(3)
    box = np.full(3, 5.0)
    p1, p2 = [], []
    for k in range(6):
        X = rng.random((90, 3)) * box
        p1.append(X)
        p2.append(X[rng.permutation(90)] + rng.random(3) * box + rng.normal(scale=0.02,
                                                                           size=X.shape))
    s, nk, F = fo.periodic_defaults(90, box)
    with PeriodicBatch([90] * 6, box, s, nk, F) as b:
        b.set_positions(p1, p2)
        b.run()
        r = b.results()
    with PeriodicBatch([90], box, s, nk, F) as b1:
        b1.set_positions(p1[4], p2[4])
        b1.run()
        r1 = b1.results()
    assert r1["dist"][0] == r["dist"][4]
    np.testing.assert_array_equal(r1["perm"][0], r["perm"][4])


def test_dropin_repeated_calls_reuse_the_batch(gpu):
    """Repeated PeriodicAlign calls on one instance reuse its device batch
    (graph replays after the first call); every result is identical to a
    fresh instance's."""
    c = W.config1()
    partners = [c["pos2"], c["pos2"] + np.array([0.7, -1.3, 2.2]), c["pos2"]]
    pa = fo.PeriodicAlign(256, c["box"], c["groups"], scale=0.3, n=8)
    for k, p2 in enumerate(partners):
        say(f"case: C1 partner {k} on one instance")
        d, X1, X2, perm, disp = pa.align(c["pos1"], p2)
        fresh = fo.PeriodicAlign(256, c["box"], c["groups"], scale=0.3, n=8)
        df, X1f, X2f, permf, dispf = fresh.align(c["pos1"], p2)
        assert d == df, (k, d, df)
        np.testing.assert_array_equal(perm, permf)
        np.testing.assert_array_equal(disp, dispf)
        np.testing.assert_array_equal(X2, X2f)


@pytest.mark.parametrize("sizes,nk", [((1,), 0), ((3, 2), 1), ((64, 1), 7), ((65, 0, 4), 8),
                                      ((63,), 15), ((130, 5), 16), ((66,), 24), ((7, 68), 31)])
def test_structure_factors_tiles_and_product(gpu, sizes, nk):
    """Structure factors at the edges of the 64-atom tiles and of the 16-wide
    column tiles (2 nk + 1 = 15, 17, 31, 33, 49, 63), with empty groups,
    unwrapped positions and a box that is not a cube; Hermitian to the last
    bit, and the product is the one from the same coefficients supplied."""
    say(f"case: groups {sizes} nk={nk}")
    rng = np.random.default_rng(100 + nk)
    N = sum(sizes)
    box = np.array([5.0, 6.1, 4.3])
    pos = [(2.0 * rng.random((N, 3)) - 0.5) * box for _ in range(2)]
    at = np.concatenate([[0], np.cumsum(sizes)])
    perm = rng.permutation(N)
    groups = [perm[at[i]:at[i + 1]] for i in range(len(sizes))]
    F = max(2 * nk + 1, 4)
    with PeriodicBatch([N], box, 0.3, nk, F, [groups], 10, _lib.PER_KEEP_COEFFS) as b:
        b.set_positions(*pos)
        b.run(_lib.PSTAGE_SF)
        C, Cp = b.coeffs(), b.product()[0]
    with PeriodicBatch([N], box, 0.3, nk, F, [groups], 10, _lib.PER_INPUT_COEFFS) as b:
        b.set_positions(*pos)
        b.set_coeffs(*C)
        b.run(_lib.PSTAGE_SF)
        np.testing.assert_array_equal(b.product()[0], Cp)
    k = np.arange(-nk, nk + 1)
    for Cs, x in zip(C, pos):
        e = [np.exp(-2j * np.pi * np.outer(x[:, q] / box[q], k)) for q in range(3)]
        for Cg, g in zip(Cs, groups):
            ref = np.einsum("ja,jb,jc->abc", e[0][g], e[1][g], e[2][g])
            # per atom and axis the reference's angle, below 2 pi nk 1.5, is
            # off by at most three roundings of it; a dozen roundings besides
            tol = len(g) * 3 * (2 * np.pi * nk * 1.5 * 3 + 12) * 2.0 ** -53
            assert np.abs(Cg - ref).max() <= tol
            np.testing.assert_array_equal(Cg[::-1, ::-1, ::-1], Cg.conj())


def _refine_reference(x, y, box, groups, disp, niter):
    """The LAP + mean-shift iteration with scipy's assignment solver."""
    from scipy.optimize import linear_sum_assignment

    def wrap(v):
        return v - np.round(v / box) * box

    def assign(d):
        perm = np.arange(len(x))
        for g in groups:
            c = np.linalg.norm(wrap(x[g][:, None] - (y[g] - d)[None]), axis=2)
            perm[g] = g[linear_sum_assignment(c)[1]]
        return perm

    def shift(d, perm):
        return d - wrap(x - (y[perm] - d)).mean(0)

    perm = assign(disp)
    for _ in range(niter):
        disp = shift(disp, perm)
        new = assign(disp)
        same = np.array_equal(new, perm)
        perm = new
        if same:
            break
    disp = shift(disp, perm)
    return perm, disp, np.linalg.norm(wrap(x - (y[perm] - disp)))


@pytest.mark.parametrize("sizes,noise,niter", [
    ((1,), 0.02, 10), ((63, 0, 2), 0.02, 10), ((64,), 0.3, 10), ((65, 1, 64), 0.3, 10),
    ((256,), 0.02, 0), ((257, 130), 0.25, 10), ((2000,), 0.02, 1)])
def test_refine_nearest_rows_and_assignment(gpu, sizes, noise, niter):
    """The refinement from a given displacement at the edges of the nearest-row
    kernel's 64 columns and 256-row tiles, with empty and one-atom groups,
    with many free rows (noise 0.25 and above: later assignments rescan
    columns) and with positions too many for LDS (2000)."""
    say(f"case: groups {sizes} noise {noise} niter {niter}")
    rng = np.random.default_rng(sum(sizes) + niter)
    N = sum(sizes)
    box = np.array([1.0, 1.15, 0.9]) * (N / 1.1) ** (1 / 3) + 0.5
    at = np.concatenate([[0], np.cumsum(sizes)])
    order = rng.permutation(N)
    groups = [order[at[i]:at[i + 1]] for i in range(len(sizes))]
    x = rng.random((N, 3)) * box
    perm = np.arange(N)
    for g in groups:
        perm[g] = rng.permutation(g)
    y = x[perm] + 0.4 + rng.normal(scale=noise, size=x.shape)
    d0 = np.full(3, 0.4 + 0.01)
    with PeriodicBatch([N], box, 0.3, 2, 12, [groups], niter) as b:
        b.set_positions(x, y)
        b.set_disp(d0)
        b.run(_lib.PSTAGE_REFINE)
        r = b.results()
    rp, rd, dist = _refine_reference(x, y, box, groups, d0, niter)
    np.testing.assert_array_equal(r["perm"][0], rp)
    # sums of N terms below the box length
    tol = 8 * N * box.max() * 2.0 ** -53
    np.testing.assert_allclose(r["disp"][0], rd, rtol=0, atol=tol)
    assert abs(r["dist"][0] - dist) <= tol


@pytest.mark.parametrize("nk,F,mirror", [(1, 4, False), (4, 9, True), (15, 31, False),
                                         (15, 64, True), (16, 33, False), (16, 36, True),
                                         (31, 63, True)])
def test_selected_peak_and_neighbours(gpu, nk, F, mirror):
    """The selected grid maximum, its value and the interpolated displacement
    against a 64-bit FFT, on both sides of the k-cube where the selection
    evaluates one x a pass (nk 15 / 16); inversion-symmetric structures
    (mirror) give pairs of equal maxima, evaluated one by one."""
    say(f"case: nk={nk} F={F} mirror={mirror}")
    rng = np.random.default_rng(nk * F)
    box = np.array([4.0, 4.4, 3.7])
    x, y = (rng.random((20, 3)) - 0.5 for _ in range(2))
    if mirror:
        x, y = np.concatenate([x, -x]), np.concatenate([y, -y])
    x, y = x * box, y * box
    N = len(x)
    with PeriodicBatch([N], box, 0.25, nk, F) as b:
        b.set_positions(x, y)
        b.run(_lib.PSTAGE_SF | _lib.PSTAGE_GRID)
        C, pk = b.product()[0], b.peaks()
    f = np.abs(np.fft.fftn(C, (F, F, F)))
    i = pk["ind"][0]
    # an FFT of F points a side: below 16 log2(F) roundings of sum |C|
    tol = 16 * np.log2(F) * 2.0 ** -53 * np.abs(C).sum()
    assert f[tuple(i)] >= f.max() - tol
    assert abs(pk["value"][0] - f.max()) <= tol
    disp = np.zeros(3)
    for ax in range(3):
        up, dn = i.copy(), i.copy()
        up[ax], dn[ax] = (i[ax] + 1) % F, (i[ax] - 1) % F
        y1, y2, y3 = f[tuple(up)], f[tuple(i)], f[tuple(dn)]
        curv = 2 * (2 * y2 - y1 - y3)
        disp[ax] = (i[ax] - (y3 - y1) / curv) * box[ax] / F
        # numerator and denominator are each off by a few tol
        assert abs(pk["disp"][0, ax] - disp[ax]) <= 16 * tol / abs(curv) * box[ax] / F + 1e-14


@pytest.mark.parametrize("nk,F,P", [(1, 3, 1), (7, 16, 2), (8, 17, 256), (8, 64, 64), (15, 45, 1),
                                    (16, 36, 1), (23, 47, 1), (24, 81, 1), (31, 63, 66)])
def test_real_planes_within_the_selection_bound(gpu, nk, F, P):
    """|f| of the real-basis planes (structure factors) and of the complex ones
    (the same coefficients supplied) against a 64-bit FFT at the edges of the
    basis tiles (2 nk + 1 = 15, 17, 31, 33, 47, 49, 63), odd F, and with one
    or four planes a workgroup: within the bound the selection relies on."""
    say(f"case: nk={nk} F={F} P={P}")
    rng = np.random.default_rng(nk + F)
    box = np.array([4.0, 4.4, 3.7])
    N = 12
    x, y = rng.random((P, N, 3)) * box, rng.random((P, N, 3)) * box
    NB = 2 * nk + 1
    with PeriodicBatch([N] * P, box, 0.25, nk, F, None, 10,
                       _lib.PER_KEEP_GRID | _lib.PER_KEEP_COEFFS) as b:
        b.set_positions(list(x), list(y))
        b.run(_lib.PSTAGE_SF | _lib.PSTAGE_GRID)
        C, coef, pk = b.product(), b.coeffs(), b.peaks()
        grids = {p: b.grid(p) for p in {0, P - 1}}
    for p, g in grids.items():
        f = np.abs(np.fft.fftn(C[p], (F, F, F)))
        A = np.abs(C[p]).sum()
        assert np.abs(g - f).max() <= (9 * NB + 64) * 2.0 ** -24 * A
        assert abs(pk["delta"][p] - (9 * NB + 64) * 2.0 ** -24 * A) <= 1e-12 * A
        assert f[tuple(pk["ind"][p])] >= f.max() * (1 - 1e-12)
    with PeriodicBatch([N], box, 0.25, nk, F, None, 10,
                       _lib.PER_KEEP_GRID | _lib.PER_INPUT_COEFFS) as b:
        b.set_positions(x[0], y[0])
        b.set_coeffs(coef[0][:1], coef[1][:1])
        b.run(_lib.PSTAGE_SF | _lib.PSTAGE_GRID)
        f = np.abs(np.fft.fftn(C[0], (F, F, F)))
        A = np.abs(C[0]).sum()
        assert np.abs(b.grid(0) - f).max() <= (4 * NB + 32) * 2.0 ** -24 * A


@pytest.mark.parametrize("pairs", [1, 96])
def test_periodic_read_back_in_one_transfer(gpu, pairs):
    """``read()`` gives what ``results()`` and ``peaks()`` give, through the
    staging buffer and directly (96 pairs of 64 atoms), with positions set
    again before the first ones have run."""
    say(f"case: {pairs} pairs")
    rng = np.random.default_rng(pairs)
    box = np.array([4.0, 4.4, 3.7])
    x, y = (rng.random((pairs * 64, 3)) * box for _ in range(2))
    with PeriodicBatch([64] * pairs, box, 0.25, 4, 16, None, 10, 0) as b:
        b.set_positions(y, y)
        b.set_positions(x, y)
        b.run(sync=False)
        r, pk = b.read()
        for got, ref in ((r, b.results()), (pk, b.peaks())):
            assert got.keys() == ref.keys()
            for k in ref:
                for u, v in zip(got[k], ref[k]):
                    np.testing.assert_array_equal(u, v)
        cells = (r["X1"][0] - x[:64]) / box  # the structure in the home cell
        np.testing.assert_allclose(cells, np.round(cells), atol=1e-12)


@pytest.mark.parametrize("nk,F,N", [(4, 20, 30), (8, 64, 256), (14, 60, 1000), (16, 70, 500)])
def test_real_planes_round_no_more_than_complex_planes(gpu, nk, F, N):
    """|f| against a 64-bit FFT of the same product: the rms error of the
    real-basis planes is no larger than that of the complex transform (the same
    coefficients supplied), also for structures that nearly match, whose product
    falls off slowest."""
    rng = np.random.default_rng(nk)
    box = np.array([1.0, 1.1, 0.95]) * (N / 1.185) ** (1 / 3)
    err = np.zeros(2)
    for seed in range(3):
        say(f"case: nk={nk} F={F} N={N} seed {seed}")
        x = rng.random((N, 3)) * box
        y = rng.random((N, 3)) * box if seed == 2 else x + 0.3 * box + rng.normal(scale=0.02, size=x.shape)
        coef = None
        for k, flag in enumerate((_lib.PER_KEEP_COEFFS, _lib.PER_INPUT_COEFFS)):
            with PeriodicBatch([N], box, 0.3, nk, F, None, 10, _lib.PER_KEEP_GRID | flag) as b:
                b.set_positions(x, y)
                if k:
                    b.set_coeffs(*coef)
                b.run(_lib.PSTAGE_SF | _lib.PSTAGE_GRID)
                coef = coef or b.coeffs()
                f = np.abs(np.fft.fftn(b.product()[0], (F, F, F)))
                err[k] += np.square(b.grid(0) - f).mean() / np.square(f).mean()
    say("rms error, real and complex:", np.sqrt(err / 3))
    assert err[0] <= err[1]
