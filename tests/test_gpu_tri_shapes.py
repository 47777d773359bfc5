"""GPU checks of the tridiagonal shapes chosen by ny (variants 2 and 6) at the
edges of every chunk count's range: fewest and most rows a chunk, a last chunk
that is nearly empty, one and two passes, in place and through the blocked
layouts, where 8-mode groups share a block of 16 x rows.

The in-place kernel is compared with the serial Thomas sweep per mode
(1e-11 of the mode's max-abs, the bar of the other partitioned shapes); the
blocked solve with the in-place one (1e-13 of the max-abs)."""
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


@pytest.mark.parametrize("ny", [2, 5, 8, 33, 45, 48, 49, 57, 64, 120, 128, 129, 145, 305, 320, 321, 497, 512, 513, 545,
                                770, 993, 1024])
def test_rule_shapes_match_serial_and_blocked(cuda, ny):
    nx, nz = 48, 18
    say("rule shape", ny)
    yu = W.tanh_faces(ny, 1.2)
    rng = np.random.default_rng(ny)
    f = rng.uniform(-1, 1, size=(ny, nz, nx))
    bands = D.mk_P_abc(yu, False) + D.mk_P_abc(yu, True)
    idx, idz = nx / W.LX, nz / W.LZ
    s = D.PoissonSolver(nx, nz, ny, idx, idz, bands)
    S = O.forward(f)
    ref = O.tridiag(S, idx, idz, bands)
    scale = np.abs(ref).max(axis=0, keepdims=True)
    s.set_strategy(D.FFT_AUTO, D.TRIDIAG_PARTITION)
    src = to_dev(f)
    for tv in (2, 6):
        s.set_variants(0, 0, tv)
        t = to_dev(S)
        s.tridiag(t)
        assert np.all(np.abs(to_host(t) - ref) <= 1e-11 * scale + 1e-300), tv
        out = []
        for blocked in (False, True):
            s.set_blocked(blocked)
            P = to_dev(np.zeros_like(f))
            s.solve(src, P)
            out.append(to_host(P))
        assert np.abs(out[1] - out[0]).max() <= 1e-13 * np.abs(out[0]).max(), tv
    s.close()


@pytest.mark.parametrize("ny", [2, 8, 33, 48, 49, 96, 128, 129, 280, 512, 513, 1024])
def test_rule_shapes_of_fp32_spectra(cuda, ny):
    """The mixed form's 32-mode shapes, whose two group lists pair 16-mode
    groups: the same modes run in FP32 as with 16-mode workgroups, and one
    refinement meets the residual bar of the other shapes (1e-10)."""
    nx, nz = 96, 32
    say("fp32 rule shape", ny)
    yu = W.tanh_faces(ny, 1.2)
    rhs = W.rhs_band_limited((ny, nz, nx), 2, yu=yu)
    idx, idz = nx / W.LX, nz / W.LZ
    bands = D.mk_P_abc(yu, False) + D.mk_P_abc(yu, True)
    s = D.PoissonSolver(nx, nz, ny, idx, idz, bands, precision=D.PRECISION_MIXED)
    src = to_dev(rhs)
    s.set_mixed_variants(0, 0, 0)
    n32 = s.mixed_info[2]
    for tv in (2, 6):
        s.set_mixed_variants(0, 0, tv)
        assert s.mixed_info[2] == n32, tv
        for fp32 in (False, True):
            s.set_mixed_fp32(fp32)
            P = to_dev(np.zeros_like(rhs))
            s.solve_mixed(src, P, 1)
            rel = s.residual(src, P)
            assert rel <= 1e-10, (tv, fp32, rel)
    s.close()
