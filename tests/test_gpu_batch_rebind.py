"""GPU check of a batch bound a second time: a graph captured under the first
binding solves the arrays of the second one, for the instances of the shared
launches and for those that run alone, and leaves the first arrays untouched."""
import sys

import pytest

import dnsproj as D
from dnsproj import workloads as W

pytestmark = pytest.mark.gpu


def case(nx, nz, ny):
    yu = W.tanh_faces(ny, 1.3)
    return dict(nx=nx, nz=nz, ny=ny, inv_dx=nx / W.LX, inv_dz=nz / W.LZ,
                bands=D.mk_P_abc(yu, False) + D.mk_P_abc(yu, True))


@pytest.mark.parametrize("sizes", [[(64, 32, 33), (256, 96, 256)], [(512, 128, 97), (96, 64, 40), (384, 768, 24)]])
def test_captured_run_follows_a_second_bind(cuda, sizes):
    import torch
    print("[gpu-case] batch rebind", sizes, flush=True)
    sys.stdout.flush()
    b = D.PoissonBatch([case(*s) for s in sizes])
    gen = torch.Generator(device="cuda:0").manual_seed(11)

    def arrays():
        f = [torch.rand((ny, nz, nx), dtype=torch.float64, device="cuda:0", generator=gen) - 0.5
             for nx, nz, ny in sizes]
        return f, [torch.full_like(t, float("nan")) for t in f]
    sets = [arrays() for _ in range(3)]  # all kept alive: a stale address is a wrong result, not a fault
    ref = []
    for f, P in sets:
        b.bind(f, P)
        b.run()
        torch.cuda.synchronize()
        ref.append([t.clone() for t in P])
        for t in P:
            t.fill_(float("nan"))
    b.bind(*sets[0])
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        b.run()
    for q in (0, 1, 2, 1):
        b.bind(*sets[q])
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        for t, r, s in zip(sets[q][1], ref[q], sizes):
            assert torch.equal(t, r), (q, s)
            t.fill_(float("nan"))
        for o in range(3):
            assert o == q or all(bool(t.isnan().all()) for t in sets[o][1]), (q, o)
    b.close()
