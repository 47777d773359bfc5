"""GPU checks of the shared rough-wall launches of a projection step: forcing of
several fields at once (targets on faces, edges and corners, whose images lie in
the halo shell and in the wall planes; a component without records; one whose
sources are targets, which takes the field-by-field passes), and column slabs
at their limits (none, whole columns, overlapping, past the walls)."""
import sys

import numpy as np
import pytest

import projection as PJ
import dnsproj.projection as DP
from dnsproj import workloads as W

pytestmark = pytest.mark.gpu
NX, NZ, NY = 12, 10, 9


def host(t):
    import torch
    torch.cuda.synchronize()
    return t.cpu().numpy()


def make_step(c):
    s = DP.ProjectionStep(NX, NZ, NY, c["yu"], c["inv_dx"], c["inv_dz"], c["dtmax"])
    s.set_walls(c["walls"])
    s.load(c["fields"])
    return s


def records(rng, n, overlap):
    """n records with distinct targets, corners first; sources are other points,
    or (overlap) targets too."""
    pts = [(i, j, k) for i in (0, NX - 1) for j in (0, NZ - 1) for k in (0, 3, NY - 1)]
    rest = [(int(i), int(j), int(k)) for i, j, k in rng.integers(0, (NX, NZ, NY), size=(400, 3))]
    pts += [p for p in dict.fromkeys(rest) if p not in pts]
    tgt, src = pts[:n], pts[n:]
    ijk, c = [], []
    for r, t in enumerate(tgt):
        a, b = (tgt[(r + 1) % n], tgt[(r + 2) % n]) if overlap else (src[r % len(src)], src[(r + 7) % len(src)])
        ijk.append([*t, *a, *b])
        c.append(rng.standard_normal(3))
    return np.array(ijk, dtype=np.int32), np.array(c)


@pytest.mark.parametrize("kinds", [("d", "d", "d"), ("d", None, "d"), ("o", "d", None), (None, None, "d")])
def test_forcing_set_matches_oracle(cuda, kinds):
    print("[gpu-case] forcing set", kinds, flush=True)
    sys.stdout.flush()
    c = W.projection_case(NX, NZ, NY, seed=5, k_rough=0.0)
    c["walls"] = np.array([0.25, -0.5, 0.125, 1.0, 0.5, -0.75])
    base = make_step(c)
    base.enqueue()
    ref = {n: host(base.read(n)) for n in "UVW"}
    base.close()
    rng = np.random.default_rng(7)
    s = make_step(c)
    fs = DP.IbmForcingSet.__new__(DP.IbmForcingSet)
    fs.handles, recs = {}, {}
    for n, kind in zip("UVW", kinds):
        if kind:
            recs[n] = records(rng, 40, kind == "o")
            fs.handles[n] = DP.IbmForcing(NX, NZ, NY, 1, 0, *recs[n])
            assert fs.handles[n].info["disjoint"] == (kind == "d")
    s.set_ibm(fs)
    s.enqueue()
    for q, n in enumerate("UVW"):
        A = ref[n]
        if n in recs:
            A = PJ.ibm_exec(A, recs[n][0].reshape(-1, 3, 3), recs[n][1], NX, NZ, NY, 1, 0)
        PJ.set_val_slice(A, 0, 0, c["walls"][q])
        PJ.set_val_slice(A, -1, -1, c["walls"][3 + q])
        assert np.array_equal(host(s.read(n)), A), n
    s.close()


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_column_limits_match_oracle(cuda, seed):
    print("[gpu-case] column limits", seed, flush=True)
    sys.stdout.flush()
    c = W.projection_case(NX, NZ, NY, seed=5, k_rough=0.0)
    c["walls"] = np.array([0.25, -0.5, 0.125, 1.0, 0.5, -0.75])
    base = make_step(c)
    base.enqueue()
    ref = {n: host(base.read(n)) for n in "UVW"}
    base.close()
    rng = np.random.default_rng(seed)
    s = make_step(c)
    cols = {}
    for n in ("U", "V", "W")[: 2 + seed % 2]:
        cols[n] = rng.integers(-2, NY + 3, size=(2, NZ, NX)).astype(np.int32)
        s.set_columns(*cols[n], component=n)
    s.enqueue()
    for q, n in enumerate("UVW"):
        A, w = ref[n], c["walls"]
        if n in cols:
            bot, top = np.minimum(cols[n][0], NY), np.maximum(cols[n][1], -1)
            A = PJ.ibm_part2(A, bot, top, NY if n == "V" else NY - 1, w[q], w[3 + q])
        PJ.halo_periodic_xz(A)
        PJ.set_val_slice(A, 0, 1 if n == "V" else 0, w[q])
        PJ.set_val_slice(A, -1, -1, w[3 + q])
        assert np.array_equal(host(s.read(n)), A), n
    s.close()
