"""GPU check of the solver tuner's data: after many repetitions the work array
still holds ordinary values (transforms and solves repeated in place without a
refill end in infinities or in zeros), and the tuned solve is right."""
import sys

import numpy as np
import pytest

import oracle as O
import dnsproj as D
from dnsproj import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nz,ny,precision", [(256, 32, 40, 0), (64, 96, 48, 1), (50, 64, 33, 0), (192, 42, 36, 0)])
def test_tuner_keeps_ordinary_values(cuda, nx, nz, ny, precision):
    import torch
    print("[gpu-case] tuner data", nx, nz, ny, precision, flush=True)
    sys.stdout.flush()
    yu = W.tanh_faces(ny, 1.4)
    bands = D.mk_P_abc(yu, False) + D.mk_P_abc(yu, True)
    idx, idz = nx / W.LX, nz / W.LZ
    s = D.PoissonSolver(nx, nz, ny, idx, idz, bands, precision=precision)
    work = torch.zeros((ny, nz, nx), dtype=torch.float64, device="cuda:0")
    t = s.autotune(work=work, reps=300)
    assert all(v > 0 or v == -1 for k in t for v in t[k] if k.endswith("_ms"))
    top = float(work.abs().max())
    assert 1e-100 < top < 1e100
    f = np.random.default_rng(nx).uniform(-1, 1, size=(ny, nz, nx))
    P = torch.from_numpy(f).to("cuda:0")
    s.run(P)
    torch.cuda.synchronize()
    g, r = P.cpu().numpy(), O.solve(f, idx, idz, bands)
    r = r - r.mean()
    assert np.abs(g - g.mean() - r).max() <= 1e-12 * np.abs(r).max()
    s.close()
