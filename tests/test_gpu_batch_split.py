"""GPU checks of the batched solve that runs its large instances alone (FP64
tridiagonal variant 6): batches with instances on both sides of the bound, only
small and only large ones, against the shared launches (another partition of
the rows and another transform layout: 1e-12 of the solution), eagerly and in a
replayed graph.  An instance below the bound equals variant 4 bit for bit."""
import sys

import numpy as np
import pytest

import dnsproj as D
from dnsproj import workloads as W

pytestmark = pytest.mark.gpu

BOUND = 6 << 20  # points


def say(*a):
    print("[gpu-case]", *a, flush=True)
    sys.stdout.flush()


def case(nx, nz, ny):
    yu = W.tanh_faces(ny, 1.3)
    return dict(nx=nx, nz=nz, ny=ny, inv_dx=nx / W.LX, inv_dz=nz / W.LZ,
                bands=D.mk_P_abc(yu, False) + D.mk_P_abc(yu, True))


@pytest.mark.parametrize("sizes", [
    [(64, 32, 5), (128, 32, 1024), (512, 128, 97), (64, 32, 33), (96, 768, 86), (256, 96, 255), (512, 96, 128)],
    [(32, 32, 2), (64, 128, 50)],
    [(384, 192, 86), (768, 64, 130)],
], ids=["both", "small", "large"])
def test_large_instances_alone(cuda, sizes):
    import torch
    say("batch split", sizes)
    cases = [case(*s) for s in sizes]
    b = D.PoissonBatch(cases)
    gen = torch.Generator(device="cuda:0").manual_seed(3)
    f = [torch.rand((ny, nz, nx), dtype=torch.float64, device="cuda:0", generator=gen) - 0.5 for nx, nz, ny in sizes]
    P = [torch.full_like(t, float("nan")) for t in f]
    b.bind(f, P)
    assert b.variants[2] == 6
    b.set_variants(2, 1, 4)
    b.run()
    torch.cuda.synchronize()
    ref = [t.clone() for t in P]
    b.set_variants(2, 1, 6)

    def check(tag):
        torch.cuda.synchronize()
        for (nx, nz, ny), t, r in zip(sizes, P, ref):
            if nx * nz * ny < BOUND:
                assert torch.equal(t, r), (tag, nx, nz, ny)
            else:
                a, c = t - t.mean(), r - r.mean()
                assert float((a - c).norm() / c.norm()) <= 1e-12, (tag, nx, nz, ny)
            t.fill_(float("nan"))

    b.run()
    check("eager")
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        b.run()
    for rep in range(3):
        g.replay()
        check(("replay", rep))
    b.close()
