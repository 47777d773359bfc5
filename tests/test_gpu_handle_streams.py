"""GPU checks of solves that overlap on one handle: a handle whose lengths are not
all compile-time ones (so that its solve holds no workspace) solves different
arrays on two streams at once, launched one by one and as two graphs, and every
result equals the one solved alone, bit for bit."""
import sys

import pytest

import dnsproj as D
from dnsproj import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nz,ny", [(80, 48, 64), (240, 120, 160), (560, 280, 70), (512, 140, 96), (320, 128, 96)])
def test_two_streams_on_one_handle(cuda, nx, nz, ny):
    import torch
    print("[gpu-case] one handle, two streams", nx, nz, ny, flush=True)
    sys.stdout.flush()
    yu = W.tanh_faces(ny, 1.4)
    bands = D.mk_P_abc(yu, False) + D.mk_P_abc(yu, True)
    s = D.PoissonSolver(nx, nz, ny, nx / W.LX, nz / W.LZ, bands)
    assert s.blocked == (False, False)
    s.set_blocked(True)
    assert s.blocked == (False, False)
    gen = torch.Generator(device="cuda:0").manual_seed(nx)
    f = [torch.rand((ny, nz, nx), dtype=torch.float64, device="cuda:0", generator=gen) - 0.5 for _ in range(2)]
    P = [torch.empty_like(t) for t in f]
    ref = []
    for t in f:
        s.solve(t, P[0])
        torch.cuda.synchronize()
        ref.append(P[0].clone())
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]

    def check(tag):
        torch.cuda.synchronize()
        for q in range(2):
            assert torch.equal(P[q], ref[q]), (tag, q)
            P[q].fill_(float("nan"))
        torch.cuda.synchronize()

    for rep in range(10):
        for _ in range(4):
            for q in (rep % 2, 1 - rep % 2):
                s.solve(f[q], P[q], stream=streams[q])
        check(("launched", rep))
    graphs = []
    for q in range(2):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=streams[q]):
            s.solve(f[q], P[q])
        graphs.append(g)
    for rep in range(5):
        for _ in range(4):
            for q in range(2):
                with torch.cuda.stream(streams[q]):
                    graphs[q].replay()
        check(("replayed", rep))
    s.close()


@pytest.mark.parametrize("nx,nz,ny", [(80, 48, 64), (320, 128, 96)])
def test_step_takes_its_fields_only(cuda, nx, nz, ny):
    """A projection step at such lengths holds its 11 halo fields, P and tables:
    no optional workspace that could take the memory of a field."""
    import dnsproj.projection as DP
    print("[gpu-case] step footprint", nx, nz, ny, flush=True)
    s = DP.ProjectionStep(nx, nz, ny, W.tanh_faces(ny, 1.4), nx / W.LX, nz / W.LZ, 1e-4)
    fields = 8 * (11 * (nx + 2) * (nz + 2) * (ny + 2) + nx * nz * ny)
    assert fields <= s.footprint < fields + 4 * nx * nz * ny
    s.close()
