"""GPU checks of the plane-marching kernels (momentum, energy right-hand side,
Poisson right-hand side) at the edges of their 64 x 4 tiles and of their runs of
planes, where lanes past the last column repeat its point and waves past the
last row only stage: the whole predictor and the right-hand side against the
oracle, with the bars of the other sizes."""
import sys

import numpy as np
import pytest

import projection as PJ
import test_gpu_predictor as TP
import dnsproj.projection as DP
from dnsproj import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["incomp", "nicoud"])
@pytest.mark.parametrize("nx,nz,ny", [(1, 4, 5), (63, 5, 4), (64, 4, 17), (65, 3, 18), (66, 9, 3), (130, 6, 7)])
def test_predictor_tile_edges(cuda, kind, nx, nz, ny):
    TP.say("ring tiles", kind, nx, nz, ny)
    TP.test_predictor_matches_oracle(cuda, kind, nx, nz, ny)


@pytest.mark.parametrize("nx,nz,ny", [(1, 1, 1), (63, 4, 2), (64, 5, 3), (65, 8, 1), (129, 3, 35)])
def test_rhs_varprop_tile_edges_bitexact(cuda, nx, nz, ny):
    import torch
    TP.say("ring tiles rhs", nx, nz, ny)
    sys.stdout.flush()

    def dev(a):
        return torch.from_numpy(np.ascontiguousarray(a).copy()).to("cuda:0")
    rng = np.random.default_rng(nx + ny)
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


@pytest.mark.parametrize("nx,nz,ny", [(512, 128, 100), (512, 128, 257)])
def test_predictor_stores_past_the_caches(cuda, nx, nz, ny):
    """Sizes from which the momentum and property kernels (6.8 M padded points)
    and also the energy right-hand side (17 M) store past the caches."""
    TP.say("ring tiles large", nx, nz, ny)
    TP.test_predictor_matches_oracle(cuda, "nicoud", nx, nz, ny)
