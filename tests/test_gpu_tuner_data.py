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


def test_tuner_on_an_array_aligned_to_eight_bytes(cuda):
    """A work array that is not 16-byte aligned runs other x kernels and no blocked
    solve: those knobs are not timed and stay as they were set."""
    import torch
    nx, nz, ny = 128, 64, 40
    print("[gpu-case] tuner, 8-byte aligned work", flush=True)
    yu = W.tanh_faces(ny, 1.4)
    bands = D.mk_P_abc(yu, False) + D.mk_P_abc(yu, True)
    s = D.PoissonSolver(nx, nz, ny, nx / W.LX, nz / W.LZ, bands)
    work = torch.zeros(nx * nz * ny + 1, dtype=torch.float64, device="cuda:0")[1:].view(ny, nz, nx)
    assert work.data_ptr() % 16 == 8
    for xv, zv, tv in ((1, 0, 1), (3, 1, 5)):
        s.set_variants(xv, zv, tv)
        before = s.solve_variants
        t = s.autotune(work=work, reps=3)
        assert s.solve_variants == before
        assert t["x_ms"] == [-1.0] * 4 and t["picked"][0] == xv
        assert min(t["z_ms"]) > 0 and min(t["tri_ms"]) > 0
    s.close()
