"""GPU check of the tridiagonal shapes chosen by ny (variants 2 and 6) in the
layouts of the blocked solve, at the edges of every chunk count's range: the
blocked solve against the in-place stages with the same variant (1e-13 of the
max-abs, the bar of the other shapes)."""
import sys

import numpy as np
import pytest

import dnsproj as D
from dnsproj import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ny", [32, 33, 48, 49, 57, 64, 128, 129, 320, 321, 512, 513, 545, 770, 1024])
def test_rule_shapes_blocked(cuda, ny):
    import torch
    nx, nz = 64, 96
    print("[gpu-case] blocked rule shape", ny, flush=True)
    sys.stdout.flush()
    yu = W.tanh_faces(ny, 1.2)
    f = torch.from_numpy(np.random.default_rng(ny).uniform(-1, 1, size=(ny, nz, nx))).to("cuda:0")
    bands = D.mk_P_abc(yu, False) + D.mk_P_abc(yu, True)
    s = D.PoissonSolver(nx, nz, ny, nx / W.LX, nz / W.LZ, bands)
    for tv in (2, 6):
        s.set_variants(0, 0, tv)
        out = []
        for blocked in (False, True):
            s.set_blocked(blocked)
            assert s.blocked == (True, blocked)
            P = torch.zeros_like(f)
            s.solve(f, P)
            torch.cuda.synchronize()
            out.append(P.cpu().numpy())
        assert np.abs(out[1] - out[0]).max() <= 1e-13 * np.abs(out[0]).max(), tv
    s.close()
