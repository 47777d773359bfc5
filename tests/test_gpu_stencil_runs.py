"""GPU checks of the plane-marching stencil kernels for every run length that
the grid size selects (2, 4, 8 and 16 planes per workgroup), with a last run
that is cut short: thin, tall grids, bit-identical to the oracle."""
import sys

import numpy as np
import pytest

import projection as PJ
import dnsproj.projection as DP
from dnsproj import workloads as W

pytestmark = pytest.mark.gpu


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a).copy()).to("cuda:0")


@pytest.mark.parametrize("ny", [37, 4097, 8203, 16405, 32781])
def test_rhs_varprop_runs_bitexact(cuda, ny):
    import torch
    nx, nz = 5, 3
    print("[gpu-case] runs", ny, flush=True)
    sys.stdout.flush()
    rng = np.random.default_rng(ny)
    Uh, Wh, Vh, Pn, Po, dn, rho = (rng.standard_normal((ny + 2, nz + 2, nx + 2)) for _ in range(7))
    rho = 0.1 + np.abs(rho)
    g = PJ.geom_coeffs(W.tanh_faces(ny, 1.6))
    P = dev(np.zeros((ny, nz, nx)))
    rm = PJ.rho_min(rho)
    DP.build_p_rhs_varprop(P, dev(Uh), dev(Wh), dev(Vh), dev(Pn), dev(Po), dev(rho), dev(dn), dev(g["inv_dy_p"]),
                           dev(g["inv_dy_p_pad"]), dev(np.array([rm])), 40.0, 3.5, 2.25, 3.5 ** 2, 2.25 ** 2)
    ref = PJ.build_p_rhs_varprop(Uh, Wh, Vh, Pn, Po, rho, dn, g["inv_dy_p"], g["inv_dy_p_pad"], 40.0, 3.5, 2.25,
                                 3.5 ** 2, 2.25 ** 2, rm)
    torch.cuda.synchronize()
    assert np.array_equal(P.cpu().numpy(), ref)
