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


@pytest.mark.parametrize("nx,nz,ny", [(1, 1, 1), (65, 8, 1), (129, 3, 35), (1, 1, 32753), (2, 3, 32757), (65, 1, 16383),
                                      (63, 5, 16381), (66, 9, 8189)])
@pytest.mark.parametrize("kmin", [0, 1])
def test_update_varprop_tile_edges_bitexact(cuda, nx, nz, ny, kmin):
    """The marching kernel takes grids of 2048 workgroups of 16 planes and more:
    thin, tall ones here."""
    import torch
    TP.say("ring tiles update", nx, nz, ny, kmin)

    def dev(a):
        return torch.from_numpy(np.ascontiguousarray(a).copy()).to("cuda:0")
    rng = np.random.default_rng(nx + ny)
    U, V, Wv, Uh, Vh, Wh, Pn, Po, rho = (rng.standard_normal((ny + 2, nz + 2, nx + 2)) for _ in range(9))
    rho = 0.1 + np.abs(rho)
    p = rng.standard_normal((ny, nz, nx))
    g = PJ.geom_coeffs(W.tanh_faces(ny, 1.6))
    walls = dict(zip(PJ.WALL_KEYS, (0.5, -0.25, 0.125, 1.0, -1.5, 2.0)))
    rm = PJ.rho_min(rho)
    ref = PJ.update_vars(p, U, V, Wv, Uh, Vh, Wh, g["dPdy_ddy_hi"], g["dPdy_ddy_lo"], 0.003, 3.0, 2.0, kmin, walls,
                         use_incompressible=False, P_now=Pn, P_old=Po, rho=rho, rho_min_v=rm)
    t = [dev(U), dev(V), dev(Wv), dev(np.zeros_like(U)), dev(Pn), dev(Po)]
    DP.update_vars(dev(p), t[3], t[4], t[5], t[0], t[1], t[2], dev(Uh), dev(Vh), dev(Wh), dev(rho),
                   dev(g["dPdy_ddy_hi"]), dev(g["dPdy_ddy_lo"]), dev(np.array([rm])),
                   dev(np.array([walls[k] for k in PJ.WALL_KEYS])), kmin, 0.003, 3.0, 2.0, use_incompressible=False)
    torch.cuda.synchronize()
    for q in range(6):
        assert np.array_equal(t[q].cpu().numpy(), ref[q]), q
