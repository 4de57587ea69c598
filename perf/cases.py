"""Workloads of the framework, as its users run them.

Every case is a dict of plain values.  ``prepare`` draws its inputs from a
seed and builds the handle a user's program keeps (aligner, batch, server,
transform); ``run`` is one pass through the public Python interface with new
positions handed in and every answer read back; ``exact`` gives the answers
in 64 bits with numpy alone.

Structures are planted: the second structure of a pair is a rotated (or
translated), permuted copy of the first with N(0, 0.02) noise, the inputs of
the alignment workloads of this repository.  The best assignment is then the
planted one and the aligned distance follows from a quaternion or mean-shift
fit over it.  Clusters are spherical cuts of one relaxed random packing
(0.964 volume units per atom, neighbours about 0.9 or further apart, as the
cluster mixes of ``fastoverlap_amd/workloads.py``); periodic systems are
relaxed random packings of their own.
"""

import math

import numpy as np
import torch

from fastoverlap_amd import _lib
from fastoverlap_amd.batch import (PeriodicBatch, SphericalBatch, dense_to_compact,
                                   periodic_defaults)
from fastoverlap_amd.periodic import PeriodicAlign
from fastoverlap_amd.serve import Server
from fastoverlap_amd.soft import SOFT
from fastoverlap_amd.spherical import SphericalAlign

NOISE = 0.02          # of the planted copies
ATOM_VOLUME = 0.964   # volume per atom of the cluster mixes
SAMPLE = 4096         # atoms of the packing that clusters are cut from


def listed():
    return [
        # one pair through the drop-in class, the interactive call: 38 atoms
        # (the Lennard-Jones cluster of the examples), Jmax 15
        dict(name="cluster_call_38", kind="cluster_call", natoms=38, L=15, species=1, scale=0.3),
        # one periodic pair through the drop-in class: 256 atoms, 204 + 52
        dict(name="periodic_call_256", kind="periodic_call", natoms=256, nk=8, density=1.185,
             species=2, scale=0.3),
        # a small ragged batch of small clusters at low degrees, automatic width
        dict(name="cluster_batch_64", kind="cluster_batch", pairs=64, nmin=13, nmax=55, lmin=8,
             lmax=15, grid=32, species=2, scale=0.0, invert=True),
        # the large ragged batch of mixed clusters: the throughput workload
        dict(name="cluster_batch_4096", kind="cluster_batch", pairs=4096, nmin=13, nmax=147,
             lmin=16, lmax=25, grid=64, species=2, scale=0.3, invert=True),
        # the largest clusters and degree: 1000 atoms, Jmax 40, grid 128
        dict(name="cluster_batch_n1000", kind="cluster_batch", pairs=64, nmin=1000, nmax=1000,
             lmin=40, lmax=40, grid=128, species=2, scale=0.2, invert=True),
        # the drop-in classes' default grid 2 (Jmax + 1), here 42: no power of
        # two; only the given orientation
        dict(name="cluster_batch_grid42", kind="cluster_batch", pairs=96, nmin=20, nmax=120,
             lmin=20, lmax=20, grid=42, species=1, scale=0.3, invert=False),
        # harmonic-basis alignment of many pairs of one cluster size
        dict(name="harmonic_batch_32", kind="harmonic_batch", pairs=32, natoms=55, L=15, nmax=15,
             species=1, scale=0.3),
        # a batch of equal periodic systems
        dict(name="periodic_batch_128", kind="periodic_batch", pairs=128, nmin=256, nmax=256,
             nk=8, grid=64, density=1.185, species=2, aspect=1.0),
        # a ragged batch of the largest periodic systems at the default
        # k-cube and grid, in a box that is not a cube
        dict(name="periodic_batch_n1024", kind="periodic_batch", pairs=24, nmin=601, nmax=1024,
             nk=14, grid=60, density=1.2, species=2, aspect=1.17),
        # all pairs of a group of periodic structures (distance matrix)
        dict(name="periodic_group_12", kind="periodic_group", structures=12, natoms=256, nk=8,
             density=1.185, species=2),
        # requests of both kinds and every size through the server
        dict(name="served_mix_96", kind="served", requests=96, nmin=13, nmax=300, lmin=15,
             lmax=30, pmin=64, pmax=512, species=2),
        # the SO(3) transform itself: forward of a complex grid, inverse of
        # two coefficient sets, bandwidth 32
        dict(name="soft_bw32", kind="soft", bw=32),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _least_degree(natoms):
    """Degree from which a cluster's surface is resolved (15 at 500 atoms)."""
    return max(8, math.ceil(3.1 * (3 * ATOM_VOLUME * natoms / (4 * math.pi)) ** (1 / 3)))


def draw(rng):
    """One more case of the same ranges (no more work than the largest)."""
    kind = rng.choice(["cluster_call", "periodic_call", "cluster_batch", "cluster_batch",
                       "cluster_batch", "harmonic_batch", "periodic_batch", "periodic_batch",
                       "periodic_group", "served", "soft"])
    species = rng.randint(1, 2)
    if kind == "cluster_call":
        n = _log_int(rng, 13, 500)
        return dict(kind=kind, natoms=n, L=rng.randint(_least_degree(n), 30), species=species,
                    scale=0.3)
    if kind == "periodic_call":
        n = _log_int(rng, 64, 1024)
        return dict(kind=kind, natoms=n, nk=math.ceil(1.3 * n ** (1 / 3)),
                    density=rng.choice([1.0, 1.185, 1.2]), species=species, scale=0.3)
    if kind == "cluster_batch":
        nmin = _log_int(rng, 13, 600)
        nmax = min(1000, int(nmin * rng.uniform(1.0, 4.0)))
        lmin = rng.randint(_least_degree(nmax), 36)
        lmax = min(40, lmin + rng.randint(0, 9))
        pow2 = 32 if lmax <= 15 else 64 if lmax <= 31 else 128
        direct = lmax <= 25 and rng.random() < 0.3
        case = dict(kind=kind, pairs=_log_int(rng, 1, 4096), nmin=nmin, nmax=nmax, lmin=lmin,
                    lmax=lmax, grid=2 * (lmax + 1) if direct else pow2, species=species,
                    scale=rng.choice([0.0, 0.2, 0.3]), invert=rng.random() < 0.8)
        if direct:  # the direct transform costs more per pair
            case["pairs"] = min(case["pairs"], 256)
        top = work(listed()[3])["flops"]
        while case["pairs"] > 1 and work(case)["flops"] > 0.4 * top:
            case["pairs"] = (case["pairs"] + 1) // 2
        return case
    if kind == "harmonic_batch":
        n = _log_int(rng, 13, 100)
        return dict(kind=kind, pairs=_log_int(rng, 1, 64), natoms=n,
                    L=rng.randint(_least_degree(n), 15), nmax=rng.randint(8, 15), species=species, scale=0.3)
    if kind == "periodic_batch":
        nmin = _log_int(rng, 64, 1024)
        nmax = min(1024, int(nmin * rng.uniform(1.0, 2.0)))
        nk = math.ceil(1.3 * nmax ** (1 / 3))
        pairs = min(_log_int(rng, 1, 256), max(1, 24 * 1024 ** 2 // nmax ** 2))
        return dict(kind=kind, pairs=pairs, nmin=nmin, nmax=nmax, nk=nk,
                    grid=periodic_defaults(nmax, [1.0] * 3)[2], density=rng.uniform(0.9, 1.2),
                    species=species, aspect=rng.choice([1.0, 0.83, 1.17]))
    if kind == "periodic_group":
        n = _log_int(rng, 64, 400)
        return dict(kind=kind, structures=rng.randint(2, 12), natoms=n,
                    nk=math.ceil(1.3 * n ** (1 / 3)), density=rng.choice([1.0, 1.185, 1.2]),
                    species=species)
    if kind == "served":
        return dict(kind=kind, requests=_log_int(rng, 4, 96), nmin=13, nmax=rng.randint(60, 300),
                    lmin=15, lmax=rng.randint(15, 30), pmin=64, pmax=rng.randint(100, 512),
                    species=species)
    return dict(kind="soft", bw=rng.randint(8, 40))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _relax(X, box, dmin, valid, iters=80):
    """Push overlapping spheres of X (B, N, 3) in periodic boxes (B, 3) apart."""
    N = X.shape[1]
    off = ~torch.eye(N, dtype=torch.bool, device=X.device)[None] & valid[:, :, None] & valid[:, None, :]
    for _ in range(iters):
        d = X[:, :, None, :] - X[:, None, :, :]
        d -= torch.round(d / box[:, None, None, :]) * box[:, None, None, :]
        r = d.square().sum(-1).sqrt().clamp_min(1e-6)
        push = torch.where(off, (1.03 * dmin - r).clamp_min(0.0) / r, 0.0)
        X = X + 0.4 * (push[..., None] * d).sum(2)
        X = X - torch.floor(X / box[:, None, :]) * box[:, None, :]
    return X


def _packings(rng, natoms, boxes, dmin):
    """Relaxed random packings, one per (natoms[i], boxes[i]); float64 arrays."""
    out, i = [], 0
    while i < len(natoms):
        j = i + 1
        while j < len(natoms) and (j + 1 - i) * max(natoms[i:j + 1]) ** 2 <= 1 << 24:
            j += 1
        n = max(natoms[i:j])
        X = rng.random((j - i, n, 3)) * np.asarray(boxes[i:j])[:, None, :]
        valid = np.arange(n)[None, :] < np.asarray(natoms[i:j])[:, None]
        box = torch.tensor(np.asarray(boxes[i:j]), dtype=torch.float32, device=_dev())
        X = _relax(torch.tensor(X, dtype=torch.float32, device=_dev()), box, dmin,
                   torch.tensor(valid, device=_dev())).double().cpu().numpy()
        out += [X[k, :natoms[i + k]].copy() for k in range(j - i)]
        i = j
    return out


def _rotation(rng):
    w, x, y, z = (lambda q: q / np.linalg.norm(q))(rng.normal(size=4))
    return np.array([[1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w)],
                     [2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w)],
                     [2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)]])


def _groups(n, species):
    k = n if species == 1 else int(round(0.7 * n))
    return [np.arange(k)] if k == n else [np.arange(k), np.arange(k, n)]


def _shuffle(rng, groups, n):
    perm = np.arange(n)
    for g in groups:
        perm[g] = g[rng.permutation(len(g))]
    return perm


def _clusters(seed, natoms, species):
    """Planted cluster pairs: per pair pos1, pos2, groups and the planted
    assignment (pos2[assign] matches pos1)."""
    rng = np.random.default_rng(seed)
    side = (SAMPLE * ATOM_VOLUME) ** (1 / 3)
    X = torch.tensor(_packings(rng, [SAMPLE], [[side] * 3], 0.9)[0], dtype=torch.float32,
                     device=_dev())
    c = torch.tensor(rng.random((len(natoms), 3)) * side, dtype=torch.float32, device=_dev())
    cuts = []
    for k in range(0, len(natoms), 512):
        d = X[None] - c[k:k + 512, None]
        d -= torch.round(d / side) * side
        near = d.square().sum(-1).argsort(dim=1)[:, :max(natoms)]
        cuts.append(torch.gather(d, 1, near[..., None].expand(-1, -1, 3)).double().cpu().numpy())
    cuts = np.concatenate(cuts)
    out = []
    for p, n in enumerate(natoms):
        x = cuts[p, :n][rng.permutation(n)]
        g = _groups(n, species)
        perm = _shuffle(rng, g, n)
        y = x.dot(_rotation(rng).T)[perm] + rng.normal(scale=NOISE, size=(n, 3))
        out.append((x, y, g, np.argsort(perm)))
    return out


def _box(n, density, aspect=1.0):
    a = (n / density / aspect) ** (1 / 3)
    return np.array([a, a, a * aspect])


def _periodic(seed, natoms, density, species, aspect=1.0, copies=None):
    """Planted periodic pairs, or ``copies`` structures of one system."""
    rng = np.random.default_rng(seed)
    boxes = [_box(n, density, aspect) for n in natoms]
    out = []
    for x, box in zip(_packings(rng, natoms, boxes, 0.8 * density ** (-1 / 3)), boxes):
        n = len(x)
        g = _groups(n, species)
        if copies is None:
            perm = _shuffle(rng, g, n)
            t = (0.05 + 0.9 * rng.random(3)) * box
            y = x[perm] + t + rng.normal(scale=NOISE, size=(n, 3))
            out.append((x, y, g, np.argsort(perm), box, t))
        else:
            perms = [_shuffle(rng, g, n) for _ in range(copies)]
            out.append(([x[q] + rng.random(3) * box + rng.normal(scale=NOISE, size=(n, 3))
                         for q in perms], g, perms, box))
    return out


def _ints(key, n, lo, hi):
    """n sizes in lo..hi, hi among them; a case's sizes do not depend on its
    seed, so its outputs keep their shapes."""
    return [int(v) for v in np.random.default_rng(key).integers(lo, hi + 1, n - 1)] + [hi]


def _inputs(case, seed):
    """The drawn structures of a case (the same for one seed)."""
    k = case["kind"]
    if k == "cluster_call":
        return _clusters(seed, [case["natoms"]], case["species"])
    if k == "cluster_batch":
        return _clusters(seed, _ints(1, case["pairs"], case["nmin"], case["nmax"]), case["species"])
    if k == "harmonic_batch":
        return _clusters(seed, [case["natoms"]] * case["pairs"], case["species"])
    if k == "periodic_call":
        return _periodic(seed, [case["natoms"]], case["density"], case["species"])
    if k == "periodic_batch":
        return _periodic(seed, _ints(2, case["pairs"], case["nmin"], case["nmax"]),
                         case["density"], case["species"], case["aspect"])
    if k == "periodic_group":
        return _periodic(seed, [case["natoms"]], case["density"], case["species"],
                         copies=case["structures"])[0]
    if k == "served":
        # seven of ten requests are clusters
        nc = max(1, (7 * case["requests"]) // 10)
        cl = _clusters(seed, _ints(3, nc, case["nmin"], case["nmax"]), case["species"])
        pe = _periodic([seed, 1], _ints(4, case["requests"] - nc, case["pmin"], case["pmax"]),
                       1.2, case["species"])
        order = np.random.default_rng(5).permutation(case["requests"])
        Ls = _ints(6, nc, case["lmin"], case["lmax"])
        return [(cl[i], Ls[i]) if i < nc else (pe[i - nc], None) for i in order]
    # soft: a complex grid, two Hermitian coefficient sets (dense layout)
    rng = np.random.default_rng(seed)
    bw = case["bw"]
    n, W = 2 * bw, 2 * bw - 1
    grid = rng.normal(size=(n, n, n)) + 1j * rng.normal(size=(n, n, n))
    m = (np.arange(W) + bw - 1) % W - (bw - 1)
    neg, sign = (-m) % W, (-1.0) ** (m[:, None] + m[None, :])
    sets = []
    for _ in range(2):
        f = rng.normal(size=(bw, W, W)) + 1j * rng.normal(size=(bw, W, W))
        f *= np.exp(-0.1 * np.arange(bw))[:, None, None]  # overlaps fade with the degree
        f = 0.5 * (f + sign * np.conj(f[:, neg][:, :, neg]))
        l = np.arange(bw)[:, None, None]
        sets.append(np.where((abs(m)[None, :, None] <= l) & (abs(m)[None, None, :] <= l), f, 0))
    return grid, sets


def _on_device(arrays):
    return torch.tensor(np.concatenate(arrays), dtype=torch.float64, device=_dev())


def prepare(case, seed):
    k = case["kind"]
    x = _inputs(case, seed)
    s = {"kind": k}
    if k == "cluster_call":
        p1, p2, g, _ = x[0]
        s.update(pos1=p1, pos2=p2, align=SphericalAlign(case["scale"], case["L"], g))
    elif k in ("cluster_batch", "harmonic_batch"):
        natoms = [len(q[0]) for q in x]
        if k == "cluster_batch":
            flags = 0 if case["invert"] else _lib.SPH_NO_INVERT
            b = SphericalBatch(natoms, _ints(7, case["pairs"], case["lmin"], case["lmax"]),
                               case["scale"], case["grid"],
                               [q[2] for q in x], flags)
        else:
            b = SphericalBatch(natoms, case["L"], case["scale"], 2 * (case["L"] + 1),
                               [q[2] for q in x], harmonic=(case["nmax"], 1.0))
        s.update(batch=b, pos1=_on_device([q[0] for q in x]), pos2=_on_device([q[1] for q in x]))
    elif k == "periodic_call":
        p1, p2, g, _, box, _ = x[0]
        s.update(pos1=p1, pos2=p2,
                 align=PeriodicAlign(len(p1), box, g, scale=case["scale"], n=case["nk"]))
    elif k == "periodic_batch":
        scale = [periodic_defaults(len(q[0]), q[4])[0] for q in x]
        b = PeriodicBatch([len(q[0]) for q in x], np.array([q[4] for q in x]), scale, case["nk"],
                          case["grid"], [q[2] for q in x])
        s.update(batch=b, pos1=_on_device([q[0] for q in x]), pos2=_on_device([q[1] for q in x]))
    elif k == "periodic_group":
        coords, g, _, box = x
        s.update(coords=coords, align=PeriodicAlign(case["natoms"], box, g, n=case["nk"]))
    elif k == "served":
        reqs = []
        for q, L in x:
            r = dict(pos1=q[0], pos2=q[1], groups=q[2])
            reqs.append(dict(r, kind=1, box=q[4]) if L is None else
                        dict(r, kind=0, L=L, scale=0.3))
        s.update(requests=reqs, server=Server(max_batch=64, streams=2))
    else:
        grid, (a, b) = x
        batch = SphericalBatch([1], case["bw"] - 1, 1.0, 2 * case["bw"],
                               flags=_lib.SPH_GENERAL | _lib.SPH_KEEP_GRID)
        s.update(soft=SOFT(case["bw"]), data=grid, batch=batch, a=dense_to_compact(a),
                 b=dense_to_compact(b))
    if torch.cuda.is_available():
        torch.cuda.synchronize()
    return s


def run(s):
    k = s["kind"]
    if k == "cluster_call":
        dist, X1, X2 = s["align"](s["pos1"], s["pos2"])
        return dict(dist=dist, X1=X1, X2=X2)
    if k == "periodic_call":
        dist, X1, X2, perm, disp = s["align"](s["pos1"], s["pos2"])
        return dict(dist=dist, X1=X1, X2=X2, perm=perm, disp=disp)
    if k in ("cluster_batch", "harmonic_batch", "periodic_batch"):
        b = s["batch"]
        b.set_positions_device(s["pos1"].data_ptr(), s["pos2"].data_ptr())
        b.run()
        r = b.results()
        out = dict(dist=r["dist"], X1=np.concatenate(r["X1"]), X2=np.concatenate(r["X2"]),
                   perm=np.concatenate(r["perm"]))
        if k == "periodic_batch":
            return dict(out, disp=r["disp"])
        return dict(out, rmat=r["rmat"], inverted=r["inverted"])
    if k == "periodic_group":
        dists, aligned = s["align"].alignGroup(s["coords"], keepCoords=True)
        return dict(dists=dists, aligned=aligned)
    if k == "served":
        ids = [s["server"].submit(r) for r in s["requests"]]
        res = [s["server"].wait(i) for i in ids]
        return dict(dist=np.array([r["dist"] for r in res]),
                    X2=np.concatenate([r["X2"] for r in res]),
                    perm=np.concatenate([r["perm"] for r in res]))
    b = s["batch"]
    b.set_coeffs(s["a"], s["b"])
    b.run(_lib.STAGE_GRID)
    return dict(grids=b.grid(0), coeffs=s["soft"].SOFT(s["data"]))


# ---------------------------------------------------------------------------
# work and exact answers
# ---------------------------------------------------------------------------

def _sizes(case):
    n = case.get("natoms", 0.5 * (case.get("nmin", 0) + case.get("nmax", 0)))
    L = case.get("L", 0.5 * (case.get("lmin", 0) + case.get("lmax", 0)))
    return n, L


def _cluster_flops(n, L, grid, species):
    """Coefficients of the rows m1 >= 0, the grid transform of them (one beta
    sum for both orientations) and two evaluations of the refinement."""
    K = (L + 1) * (2 * L + 1) * (2 * L + 3) / 3
    pairs = n * n * (1.0 if species == 1 else 0.58)
    coef = 2 * pairs * (L + 1) ** 2 + 4 * n * K
    soft = 2 * grid * K + 5 * grid ** 3 * math.log2(grid)
    return coef + soft + 2 * 32 * K


def _periodic_flops(n, nk, grid):
    nb = 2 * nk + 1
    half = 0.5 * nb ** 3  # C(-k) = conj C(k)
    return 2 * 8 * n * half + 5 * grid ** 3 * math.log2(grid) + 20 * n * n


def work(case):
    k = case["kind"]
    n, L = _sizes(case)
    if k in ("cluster_call", "cluster_batch"):
        pairs = case.get("pairs", 1)
        grid = case.get("grid", 2 * (L + 1))
        return {"bytes": pairs * n * (4 * 24 + 8), "flops":
                pairs * _cluster_flops(n, L, grid, case["species"])}
    if k == "harmonic_batch":
        K = (L + 1) * (2 * L + 1) * (2 * L + 3) / 3
        coef = (case["nmax"] + 1) * (8 * n * (L + 1) * (L + 2) / 2 + 4 * K)
        return {"bytes": case["pairs"] * n * (4 * 24 + 8), "flops":
                case["pairs"] * (coef + _cluster_flops(0, L, 2 * (L + 1), 1))}
    if k in ("periodic_call", "periodic_batch"):
        pairs = case.get("pairs", 1)
        grid = case.get("grid") or periodic_defaults(n, [1.0] * 3, None, case["nk"])[2]
        return {"bytes": pairs * n * (4 * 24 + 8), "flops":
                pairs * _periodic_flops(n, case["nk"], grid)}
    if k == "periodic_group":
        m = case["structures"]
        grid = periodic_defaults(n, [1.0] * 3, None, case["nk"])[2]
        return {"bytes": m * n * 24 + m * m * n * 48, "flops":
                m * m * (_periodic_flops(0, case["nk"], grid) + 20 * n * n)}
    if k == "served":
        nc = max(1, (7 * case["requests"]) // 10)
        p = 0.5 * (case["pmin"] + case["pmax"])
        nk = math.ceil(1.3 * p ** (1 / 3))
        grid = 32 if L <= 15 else 64
        return {"bytes": (nc * n + (case["requests"] - nc) * p) * (3 * 24 + 8), "flops":
                nc * _cluster_flops(n, L, grid, case["species"]) +
                (case["requests"] - nc) * _periodic_flops(p, nk, 4 * nk + 4)}
    bw = case["bw"]
    g = 2 * bw
    K = bw * (2 * bw - 1) * (2 * bw + 1) / 3
    return {"bytes": g ** 3 * (16 + 8) + 3 * 16 * K,
            "flops": 2 * 4 * g * K + 3 * 5 * g ** 3 * math.log2(g)}


def _fit(x, y):
    """Superposition of y on x (both (n, 3)): distance, the centred x, the
    rotated centred y and the matrix acting on rows of y."""
    x, y = x - x.mean(0), y - y.mean(0)
    u, _, vt = np.linalg.svd(y.T.dot(x))
    u[:, -1] *= np.sign(np.linalg.det(u) * np.linalg.det(vt))
    R = u.dot(vt)
    return np.linalg.norm(x - y.dot(R)), x, y.dot(R), R


def _wrap(v, box):
    return v - np.round(v / box) * box


def _shift_fit(x, y, box, t):
    """Mean-shift fit of the matched y on x near the displacement t."""
    disp = t - _wrap(x - (y - t), box).mean(0)
    x2, y2 = _wrap(x, box), _wrap(y - disp, box)
    return np.linalg.norm(_wrap(x2 - y2, box)), x2, y2, disp


def _wigner(bw):
    """sqrt((2l+1)/2) d^l_{m1 m2}(beta_k) at [l, m1, m2, k] (m modulo 2 bw - 1),
    beta_k = pi (2k+1) / (4 bw): closed form at l = max(|m1|, |m2|), then the
    three-term recurrence in l."""
    W, n = 2 * bw - 1, 2 * bw
    beta = np.pi * (2 * np.arange(n) + 1) / (2 * n)
    c, s, cb = np.cos(beta / 2), np.sin(beta / 2), np.cos(beta)
    out = np.zeros((bw, W, W, n))
    for m1 in range(-bw + 1, bw):
        for m2 in range(-bw + 1, bw):
            l0, mu, nu = max(abs(m1), abs(m2)), abs(m1 - m2), abs(m1 + m2)
            sg = -1.0 if m2 < m1 and mu % 2 else 1.0
            lg = 0.5 * (math.lgamma(mu + nu + 1) - math.lgamma(mu + 1) - math.lgamma(nu + 1))
            prev, cur = 0.0, sg * np.exp(lg + mu * np.log(s) + nu * np.log(c))
            out[l0, m1, m2] = cur
            for l in range(l0, bw - 1):
                e = math.sqrt(((l + 1) ** 2 - m1 ** 2) * ((l + 1) ** 2 - m2 ** 2))
                t = (l + 1) * (2 * l + 1) * (cb - (m1 * m2 / (l * (l + 1)) if l else 0.0)) * cur
                if l:
                    t = t - (l + 1) / l * math.sqrt((l * l - m1 * m1) * (l * l - m2 * m2)) * prev
                prev, cur = cur, t / e
                out[l + 1, m1, m2] = cur
    return out * np.sqrt((2 * np.arange(bw) + 1) / 2)[:, None, None, None]


def exact(case, seed):
    k = case["kind"]
    x = _inputs(case, seed)
    if k in ("cluster_call", "cluster_batch", "harmonic_batch"):
        fits = [_fit(q[0], q[1][q[3]]) for q in x]
        if k == "cluster_call":
            return dict(dist=fits[0][0], X1=fits[0][1], X2=fits[0][2])
        return dict(dist=np.array([f[0] for f in fits]), X1=np.concatenate([f[1] for f in fits]),
                    X2=np.concatenate([f[2] for f in fits]),
                    perm=np.concatenate([q[3] for q in x]),
                    rmat=np.array([f[3] for f in fits]),
                    inverted=np.zeros(len(x), bool))
    if k in ("periodic_call", "periodic_batch"):
        fits = [_shift_fit(q[0], q[1][q[3]], q[4], q[5]) for q in x]
        if k == "periodic_call":
            d, x1, x2, disp = fits[0]
            return dict(dist=d, X1=x1, X2=x2, perm=x[0][3], disp=disp)
        return dict(dist=np.array([f[0] for f in fits]), X1=np.concatenate([f[1] for f in fits]),
                    X2=np.concatenate([f[2] for f in fits]),
                    perm=np.concatenate([q[3] for q in x]), disp=np.array([f[3] for f in fits]))
    if k == "periodic_group":
        coords, _, perms, box = x
        m, n = len(coords), case["natoms"]
        dists, aligned = np.zeros((m, m)), np.zeros((2, m, m, n, 3))
        for i in range(m):
            for j in range(m):
                y = coords[j][np.argsort(perms[j])[perms[i]]]
                t = -_wrap(coords[i][0] - y[0], box)
                dists[i, j], aligned[0, i, j], aligned[1, i, j], _ = _shift_fit(coords[i], y, box, t)
        return dict(dists=dists, aligned=aligned)
    if k == "served":
        dist, X2, perm = [], [], []
        for q, L in x:
            y = q[1][q[3]]
            f = _shift_fit(q[0], y, q[4], q[5]) if L is None else _fit(q[0], y)
            dist.append(f[0])
            X2.append(f[2])
            perm.append(q[3])
        return dict(dist=np.array(dist), X2=np.concatenate(X2), perm=np.concatenate(perm))
    grid, sets = x
    bw = case["bw"]
    n, W = 2 * bw, 2 * bw - 1
    D = _wigner(bw)
    m = (np.arange(W) + bw - 1) % W - (bw - 1)
    grids = []
    for f in sets:
        S = np.zeros((n, n, n), complex)
        S[m[:, None, None], np.arange(n)[None, :, None], m[None, None, :]] = np.einsum(
            "lab,labk->akb", f, D)
        grids.append(np.fft.ifftn(S, axes=(0, 2)).real * n * n)
    a = (2 * np.arange(n) + 1) * np.pi / (4 * bw)
    j = 2 * np.arange(bw) + 1
    w = (np.sin(a[:, None] * j) / j).sum(1) * 2 * np.sin(a) / bw
    S2 = np.fft.fftn(grid, axes=(0, 2)) / (n * n)
    S2 = S2[m[:, None, None], np.arange(n)[None, :, None], m[None, None, :]]
    return dict(grids=np.array(grids), coeffs=np.einsum("labk,akb,k->lab", D, S2, w))
