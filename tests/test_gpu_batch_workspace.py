"""GPU checks of the workspace of a batch's large instances (FP64 tridiagonal
variant 6): who allocates it and when, and a batch without memory for it."""
import sys

import pytest

import dnsproj as D
from dnsproj import workloads as W

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-case]", *a, flush=True)
    sys.stdout.flush()


def case(nx, nz, ny):
    yu = W.tanh_faces(ny, 1.3)
    return dict(nx=nx, nz=nz, ny=ny, inv_dx=nx / W.LX, inv_dz=nz / W.LZ,
                bands=D.mk_P_abc(yu, False) + D.mk_P_abc(yu, True))


def free_bytes():
    import torch
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_workspace_comes_with_the_first_bind_that_needs_it(cuda):
    import torch
    sizes = [(512, 256, 200), (64, 32, 40)]
    field = 8 * 512 * 256 * 200  # bytes; the allocator rounds, so half of it tells one from none
    say("batch workspace", sizes)
    f = [torch.rand((ny, nz, nx), dtype=torch.float64, device="cuda:0") - 0.5 for nx, nz, ny in sizes]
    P = [torch.zeros_like(t) for t in f]

    def taken(precision, variants=None):
        b = D.PoissonBatch([case(*s) for s in sizes], precision=precision)
        if variants:
            b.set_variants(*variants)
        n0 = free_bytes()
        b.bind(f, P)
        n1 = free_bytes()
        b.bind(f, P)
        assert free_bytes() == n1
        b.run()
        torch.cuda.synchronize()
        b.close()
        return n0 - n1
    free = free_bytes()
    b = D.PoissonBatch([case(*s) for s in sizes])
    assert free - free_bytes() < field // 2  # none at creation
    b.close()
    assert taken(D.PRECISION_FP64) > field // 2
    assert taken(D.PRECISION_FP64, (2, 1, 4)) < field // 2
    assert taken(D.PRECISION_MIXED) < field // 2
    assert taken(D.PRECISION_MIXED, (2, 1, 6)) > field // 2


def test_batch_without_memory_for_its_workspace(cuda):
    """All device memory but 2 GB taken: variant 6 of an instance of 3.2 GB runs as
    variant 4, bit for bit; bound again with memory, alone."""
    import torch
    sizes = [(512, 768, 1024), (64, 32, 40)]
    say("batch without its workspace", sizes)
    f = [torch.rand((ny, nz, nx), dtype=torch.float64, device="cuda:0") - 0.5 for nx, nz, ny in sizes]
    P = [torch.zeros_like(t) for t in f]
    b = D.PoissonBatch([case(*s) for s in sizes])
    v = b.variants
    assert v[2] == 6
    b.set_variants(v[0], v[1], 4)
    b.bind(f, P)
    b.run()
    torch.cuda.synchronize()
    ref = [t.clone() for t in P]
    b.set_variants(*v)
    torch.cuda.empty_cache()
    fill = []
    while free_bytes() > 2 << 30:
        fill.append(torch.empty(min(free_bytes() - (3 << 29), 32 << 30), dtype=torch.uint8, device="cuda:0"))
    say("filled", len(fill), free_bytes())
    for t in P:
        t.zero_()
    b.bind(f, P)
    b.run()
    torch.cuda.synchronize()
    for t, r in zip(P, ref):
        assert torch.equal(t, r)
    del fill
    torch.cuda.empty_cache()
    n0 = free_bytes()
    b.bind(f, P)
    assert n0 - free_bytes() > 4 * 512 * 768 * 1024
    b.run()
    torch.cuda.synchronize()
    a, c = P[0] - P[0].mean(), ref[0] - ref[0].mean()
    assert float((a - c).norm() / c.norm()) <= 1e-12
    assert torch.equal(P[1], ref[1])
    b.close()
