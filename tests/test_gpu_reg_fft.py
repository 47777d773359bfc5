"""GPU checks of the register-direct transforms (lengths 16..768 with prime
factors up to 13) against the oracle: every radix in the first, middle and
paired stage, odd and even butterfly counts, the shortest and the longest
lengths, odd nx (16-byte pairs not aligned), a ragged last block of x rows, an
odd number of lines, and arrays aligned to 8 bytes only.

Tolerances are those of the other FP64 transforms: 1e-13 of the output's
max-abs per stage (a few ulp times the number of stages), 1e-12 for a solve
(mean removed)."""
import sys

import numpy as np
import pytest

import oracle as O
import dnsproj as D
from dnsproj import workloads as W

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-case]", *a, flush=True)
    sys.stdout.flush()


def to_dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).to("cuda:0")


def to_host(t):
    import torch
    torch.cuda.synchronize()
    return t.cpu().numpy()


def case(nx, nz, ny):
    rng = np.random.default_rng(nx * 1000 + nz + ny)
    yu = W.tanh_faces(ny, float(rng.uniform(1.2, 2.2)))
    return yu, rng.uniform(-1, 1, size=(ny, nz, nx))


# (nx, nz, ny): two-stage, three-stage and four-stage plans; 625 = 5 5 5 5 and
# 343 = 7 7 7 have odd butterfly counts only; 50, 90, 150 pair an odd radix
# with an even count (N/2 inside a pair); 169, 121 the largest primes twice
SIZES = [(16, 16, 5), (18, 20, 33), (21, 45, 7), (22, 26, 9), (49, 77, 3), (50, 90, 5), (105, 50, 77), (121, 169, 3),
         (150, 343, 3), (104, 88, 35), (200, 100, 33), (288, 280, 34), (312, 39, 3), (560, 140, 3), (576, 576, 3),
         (624, 312, 33), (625, 48, 3), (728, 16, 5), (756, 704, 2), (729, 65, 3), (672, 144, 40)]


@pytest.mark.parametrize("nx,nz,ny", SIZES)
def test_stages_and_solve_match_oracle(cuda, nx, nz, ny):
    say("reg fft", nx, nz, ny)
    yu, f = case(nx, nz, ny)
    bands = D.mk_P_abc(yu, False) + D.mk_P_abc(yu, True)
    idx, idz = nx / W.LX, nz / W.LZ
    s = D.PoissonSolver(nx, nz, ny, idx, idz, bands)
    t = to_dev(f)
    s.forward(t)
    ref = O.forward(f)
    assert np.abs(to_host(t) - ref).max() <= 1e-13 * np.abs(ref).max()
    t = to_dev(ref)
    s.backward(t)
    back = O.backward(ref)
    assert np.abs(to_host(t) - back).max() <= 1e-13 * np.abs(back).max()
    sol = O.solve(f, idx, idz, bands)
    r = sol - sol.mean()
    src = to_dev(f)
    for blocked in (True, False):
        s.set_blocked(blocked)
        P = to_dev(np.zeros_like(f))
        s.solve(src, P)
        g = to_host(P)
        assert np.abs(g - g.mean() - r).max() <= 1e-12 * np.abs(r).max(), blocked
        Q = to_dev(f)
        s.run(Q)
        assert np.array_equal(to_host(Q), g), blocked
    assert np.array_equal(to_host(src), f)
    s.close()


@pytest.mark.parametrize("nx,nz,ny", [(80, 48, 36), (45, 36, 5), (624, 24, 33)])
def test_arrays_aligned_to_eight_bytes(cuda, nx, nz, ny):
    import torch
    say("reg fft, 8-byte aligned", nx, nz, ny)
    yu, f = case(nx, nz, ny)
    bands = D.mk_P_abc(yu, False) + D.mk_P_abc(yu, True)
    idx, idz = nx / W.LX, nz / W.LZ
    s = D.PoissonSolver(nx, nz, ny, idx, idz, bands)
    buf = torch.zeros(f.size + 1, dtype=torch.float64, device=cuda)
    P = buf[1:].view(f.shape)
    assert P.data_ptr() % 16 == 8
    P.copy_(to_dev(f))
    s.run(P)
    g, r = to_host(P), O.solve(f, idx, idz, bands)
    r = r - r.mean()
    assert np.abs(g - g.mean() - r).max() <= 1e-12 * np.abs(r).max()
    s.close()
