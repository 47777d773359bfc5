"""The work a channel-flow code has this library do, as cases to be timed.

Kinds of case:
  solve      one pressure Poisson solve rhs -> P on a kept solver (FP64 form,
             or the mixed form with one FP64 refinement)
  batch      independent FP64 solves of uneven sizes, bound once
  step       one pressure-projection step (right-hand side, solve, gradient
             correction, rough-wall forcing and columns) on resident fields
  time_step  one full time step: predictor (momentum, temperature, properties,
             energy right-hand side) and projection

Sizes are the reference's example grids, the benchmark's and test suite's
grids, and the serving ensemble's.  A kept solver, step or batch is what a
time loop holds; fields come from a seed on the GPU.
"""
import ctypes
import json
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "dns-supercritical-ibm_amd"))

import dnsproj as D  # noqa: E402
from dnsproj import predictor as PR  # noqa: E402
from dnsproj import projection as DP  # noqa: E402
from dnsproj import workloads as W  # noqa: E402

DEV = "cuda"
F8 = torch.float64
STRETCH = 1.8          # tanh stretching of the wall-normal faces
DT = 1e-4              # time step of the step and time_step cases
WALLS = (0.0, 0.0, 0.0)
# temperatures at the bottom and top walls: within the supercritical-CO2
# tables, or the ratio-4 channel of the power laws
T_WALLS = {"cubic": (316.0, 299.0), "power": (1.0, 4.0), "incompressible": (1.0, 0.0)}
CT_LENGTHS = (32, 64, 96, 128, 192, 256, 384, 512, 768)
MAX_POINTS = 624 * 312 * 770


def listed():
    return [
        # the smallest solve a test channel makes: launches and latency
        dict(name="solve_64x32x64", kind="solve", form="fp64", nx=64, nz=32, ny=64, tuned=False),
        # lengths with odd factors and an odd number of rows
        dict(name="solve_105x50x77", kind="solve", form="fp64", nx=105, nz=50, ny=77, tuned=False),
        # the smallest grid of the serving ensemble
        dict(name="solve_256x128x192", kind="solve", form="fp64", nx=256, nz=128, ny=192, tuned=False),
        # the grit-blasted Ret180 example's grid
        dict(name="solve_560x280x280", kind="solve", form="fp64", nx=560, nz=280, ny=280, tuned=False),
        # the benchmark's grid with tuned kernels, as the benchmark runs it
        dict(name="solve_768x384x384", kind="solve", form="fp64", nx=768, nz=384, ny=384, tuned=True),
        # the Ret540 example's grid, the largest field
        dict(name="solve_624x312x770", kind="solve", form="fp64", nx=624, nz=312, ny=770, tuned=False),
        # the mixed-precision form at a mid-size grid of the serving ensemble
        dict(name="mixed_512x256x256", kind="solve", form="mixed", nx=512, nz=256, ny=256, tuned=False),
        # an ensemble's pressure solves of uneven sizes in one call
        dict(name="batch_16_uneven", kind="batch", n=16, pick=2),
        # variable-density projection step over a rough bottom wall, one graph
        dict(name="step_384x192x256", kind="step", nx=384, nz=192, ny=256, density="variable", rough=True, graph=True),
        # full time step, supercritical-CO2 property tables, rough bottom wall
        dict(name="time_step_384x192x256", kind="time_step", nx=384, nz=192, ny=256, props="cubic", rough=True,
             graph=True),
        # a small variable-property channel with power laws: launches count
        dict(name="time_step_96x48x65", kind="time_step", nx=96, nz=48, ny=65, props="power", rough=False, graph=True),
        # constant-property time step, launched kernel by kernel
        dict(name="time_step_incomp_200x100x129", kind="time_step", nx=200, nz=100, ny=129, props="incompressible",
             rough=False, graph=False),
    ]


def _fft_lengths(lo, hi):
    out = []
    for n in range(lo, hi + 1):
        m = n
        for p in (2, 3, 5, 7, 11, 13):
            while m % p == 0:
                m //= p
        if m == 1:
            out.append(n)
    return out


def _log_pick(rng, values):
    """One of the increasing `values`, spread over their logarithm."""
    x = math.exp(rng.uniform(math.log(values[0]), math.log(values[-1])))
    return min(values, key=lambda v: abs(math.log(v / x)))


def draw(rng):
    kind = rng.choices(("solve", "mixed", "batch", "step", "time_step"), (50, 10, 10, 15, 15))[0]
    if kind == "batch":
        return dict(kind="batch", n=rng.randint(2, 24), pick=rng.randint(10, 1 << 20))
    if kind == "mixed":
        return dict(kind="solve", form="mixed", nx=rng.choice(CT_LENGTHS), nz=rng.choice(CT_LENGTHS[:-1]),
                    ny=rng.randint(32, 320), tuned=False)
    # three quarters round lengths (multiples of 16 or 8), the rest any length the transforms take
    every = _fft_lengths(24, 768)
    most = MAX_POINTS if kind == "solve" else 20_000_000
    while True:
        xs = [n for n in every if n % 16 == 0] if rng.random() < 0.75 else every
        zs = [n for n in every if n % 8 == 0 and n <= 640] if rng.random() < 0.75 else [n for n in every if n <= 640]
        nx, nz, ny = _log_pick(rng, xs), _log_pick(rng, zs), round(math.exp(rng.uniform(math.log(24), math.log(800))))
        if nx * nz * ny <= most:
            break
    if kind == "solve":
        return dict(kind="solve", form="fp64", nx=nx, nz=nz, ny=ny, tuned=rng.random() < 0.25)
    rough, graph = rng.random() < 0.5, rng.random() < 0.75
    if kind == "step":
        return dict(kind="step", nx=nx, nz=nz, ny=ny, density=rng.choice(("variable", "constant")), rough=rough,
                    graph=graph)
    props = rng.choice(("cubic", "power", "incompressible"))
    return dict(kind="time_step", nx=nx, nz=nz, ny=ny, props=props, rough=rough, graph=graph)


# ---------------------------------------------------------------------------
# inputs (from the seed alone)
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _faces(ny):
    j = np.arange(ny + 1, dtype=np.float64)
    return 1.0 + np.tanh(STRETCH * (2.0 * j / ny - 1.0)) / np.tanh(STRETCH)


def _bands(yu, pinned):
    """The wall-normal Poisson bands for faces yu (pinned: of the mean mode)."""
    yp = 0.5 * (yu[:-1] + yu[1:])
    pad = np.concatenate([[2 * yu[0] - yp[0]], yp, [2 * yu[-1] - yp[-1]]])
    dy = 0.5 * (pad[2:] - pad[:-2])
    a, c = 1.0 / ((pad[1:-1] - pad[:-2]) * dy), 1.0 / ((pad[2:] - pad[1:-1]) * dy)
    b = -(a + c)
    b[0] += -a[0] if pinned else a[0]
    b[-1] += c[-1]
    a[0] = c[-1] = 0.0
    return a, b, c


def _rhs(shape, seed):
    """A right-hand side: U(-1, 1) noise over a few smooth modes."""
    g = _gen(seed)
    f = torch.rand(shape, generator=g, dtype=F8, device=DEV).mul_(2.0).sub_(1.0)
    return f.add_(_smooth(shape, g, 1.0, 2))


def _smooth(shape, g, amp, modes=4):
    """Sum of a few random x-z Fourier modes with random wall-normal profiles
    of amplitude `amp`."""
    ny, nz, nx = shape
    r = torch.rand((modes, 5), generator=g, dtype=F8, device=DEV).cpu().numpy()
    y = torch.linspace(0, math.pi, ny, dtype=F8, device=DEV)
    z, x = (torch.arange(n, dtype=F8, device=DEV) * (2 * math.pi / n) for n in (nz, nx))
    out = torch.zeros(shape, dtype=F8, device=DEV)
    for m in range(modes):
        kx, kz, ky = 1 + int(4 * r[m, 0]), 1 + int(4 * r[m, 1]), 1 + int(3 * r[m, 2])
        prof = amp * torch.sin(ky * y + 6.0 * r[m, 3])
        cx, cz = torch.cos(kx * x + 6.0 * r[m, 4]), torch.cos(kz * z + 6.0 * r[m, 3])
        out.add_((prof[:, None] * cz[None, :])[:, :, None] * cx)
    return out


def _noise(t, g, amp):
    """t plus white noise, its periodic halos restored."""
    t.add_(torch.randn(t.shape, generator=g, dtype=F8, device=DEV), alpha=amp)
    _halo(t)
    return t


def _rough(case, seed):
    """Rough bottom wall of height 1/8: forcing records per velocity component
    and the columns inside the wall."""
    nx, nz, ny = case["nx"], case["nz"], case["ny"]
    h = W.rough_height_map(nx, nz, 0.125, int(seed))
    return W.rough_wall_ibm(nx, nz, ny, _faces(ny), h)


def _step_fields(case, seed):
    """Fields of a projection step: predicted velocities, density, pressure
    history and the last divergence."""
    nx, nz, ny = case["nx"], case["nz"], case["ny"]
    sh = (ny + 2, nz + 2, nx + 2)
    g = _gen(seed)
    yc = torch.linspace(-1, 1, ny + 2, dtype=F8, device=DEV)[:, None, None]
    f = {"U_hat": _noise(_smooth(sh, g, 0.05).add_(1.5 * (1 - yc * yc)), g, 0.01),
         "V_hat": _noise(_smooth(sh, g, 0.05), g, 0.01), "W_hat": _noise(_smooth(sh, g, 0.05), g, 0.01)}
    if case["density"] == "variable":
        temp = _noise(_smooth(sh, g, 0.05).add_(0.5 + 0.5 * yc), g, 0.01)
        f["rho"] = 1.0 - 0.45 * (1.0 + torch.tanh((temp - 0.5) / 0.05))
        f.update(P_now=_noise(_smooth(sh, g, 0.01), g, 1e-3), P_old=_noise(_smooth(sh, g, 0.01), g, 1e-3),
                 div_now=_noise(_smooth(sh, g, 0.01), g, 1e-4))
    return f


def _time_fields(case, seed):
    """Fields of a time step as a restart has them: velocities, temperature,
    and (variable properties) the properties at that temperature, the energy
    right-hand side and div_now."""
    nx, nz, ny = case["nx"], case["nz"], case["ny"]
    sh = (ny + 2, nz + 2, nx + 2)
    g = _gen(seed)
    yc = torch.linspace(-1, 1, ny + 2, dtype=F8, device=DEV)[:, None, None]
    f = {"U": _noise(_smooth(sh, g, 0.05).add_(1.5 * (1 - yc * yc)), g, 1e-3),
         "V": _noise(_smooth(sh, g, 0.05), g, 1e-3), "W": _noise(_smooth(sh, g, 0.05), g, 1e-3)}
    for n in "UVW":
        _walls(f[n], n == "V", 0.0, 0.0)
    lo, hi = T_WALLS[case["props"]]
    span = abs(hi - lo)
    T = _noise(_smooth(sh, g, 0.04 * span).add_(0.5 * (lo + hi) + 0.4 * (hi - lo) * yc), g, 1e-3 * span)
    T.clamp_(min(lo, hi), max(lo, hi))
    _walls(T, False, lo, hi)
    f["T"] = T
    if case["props"] != "incompressible":
        p = _exact_props(*_laws(case["props"]), T)
        f.update({n: p[n] for n in ("rho", "mu", "cp", "cond", "buoy")})
        f["RHS_energy"] = _at(_smooth(sh, g, 0.05), 0, 0, 0).contiguous()
        f["div_now"] = _noise(_smooth(sh, g, 1e-4), g, 1e-6)
    return f


def _laws(props):
    if props == "cubic":  # the supercritical-CO2 example's spline tables
        tab = json.load(open(os.path.join("tests", "golden", "props_wan2025.json")))
        laws = {q: ("cubic", [tuple(s) for s in segs]) for q, segs in tab["laws"].items()}
        return laws, ("formula",), ("linear", *tab["buoyancy"])
    laws = {"enth": ("power", 1.0, 1.0), "rho": ("power", 1.0, -1.0), "mu": ("power", 1.0 / 180.0, -0.5),
            "cond": ("power", 1.0 / (180.0 * 0.76), -0.5), "cp": ("const", 1.0), "drho_dT": ("power", -1.0, -2.0)}
    return laws, ("const", 1.0), ("none",)


def _phys(props):
    """nu, cond, mean pressure gradient and gravity of a time_step case."""
    return {"cubic": (6e-5, 0.08, 1.0, 1e-3), "power": (1 / 180.0, 1 / 136.8, 1.0, 0.0),
            "incompressible": (1 / 180.0, 1 / 136.8, 1.0, 0.0)}[props]


class _Array:
    """A device array of a handle, seen through __cuda_array_interface__."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner  # the array lives as long as its handle
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f8", "data": (int(ptr), False),
                                         "version": 2}


def _view(owner, ptr, shape):
    return torch.as_tensor(_Array(owner, ptr, shape), device=DEV)


def _step_view(step, name):
    ptr = ctypes.c_void_p()
    D._check(D.lib().dnsp_step_field(step._h, DP.STEP_FIELDS.index(name), ctypes.byref(ptr)))
    return _view(step, ptr.value, step.shape(name))


def _pred_view(pred, name):
    ptr = ctypes.c_void_p()
    D._check(D.lib().dnsp_predictor_field(pred._h, PR.PRED_FIELDS.index(name), ctypes.byref(ptr), None))
    return _view(pred, ptr.value, pred.shape(name))


def _batch_cases(case):
    rng = random.Random(case["pick"])
    return [dict(nx=rng.choice(W.CONFIG3_NX), nz=rng.choice(W.CONFIG3_NZ), ny=rng.choice(W.CONFIG3_NY))
            for _ in range(case["n"])]


def _inv_d(nx, nz):
    return nx / W.LX, nz / W.LZ


STEP_OUT = ("U", "V", "W", "P_per", "P_now", "P_old", "P")
TIME_OUT = ("U", "V", "W", "P")
PRED_OUT = ("T", "Ru_old", "Rv_old", "Rw_old", "Rt_old")
PROP_OUT = ("mu", "cond", "buoy", "cp", "enth", "divjac", "T_ext", "RHS_energy")


def prepare(case, seed):
    kind = case["kind"]
    if kind == "solve":
        nx, nz, ny = case["nx"], case["nz"], case["ny"]
        yu = _faces(ny)
        bands = D.mk_P_abc(yu, False) + D.mk_P_abc(yu, True)
        mixed = case["form"] == "mixed"
        s = D.PoissonSolver(nx, nz, ny, *_inv_d(nx, nz), bands,
                            precision=D.PRECISION_MIXED if mixed else D.PRECISION_FP64)
        P = torch.empty((ny, nz, nx), dtype=F8, device=DEV)
        if case["tuned"]:
            s.autotune(work=P, reps=5)
        return dict(kind="mixed" if mixed else "solve", solver=s, rhs=_rhs((ny, nz, nx), seed), P=P)
    if kind == "batch":
        cases = _batch_cases(case)
        for c in cases:
            c["inv_dx"], c["inv_dz"] = _inv_d(c["nx"], c["nz"])
            yu = _faces(c["ny"])
            c["bands"] = D.mk_P_abc(yu, False) + D.mk_P_abc(yu, True)
        b = D.PoissonBatch(cases)
        rhs = [_rhs((c["ny"], c["nz"], c["nx"]), seed + 1000 * i) for i, c in enumerate(cases)]
        P = [torch.empty_like(f) for f in rhs]
        b.bind(rhs, P)
        return dict(kind="batch", batch=b, P=P)
    nx, nz, ny = case["nx"], case["nz"], case["ny"]
    yu = _faces(ny)
    if kind == "step":
        s = DP.ProjectionStep(nx, nz, ny, yu, *_inv_d(nx, nz), DT, incompressible=case["density"] == "constant")
        s.set_walls(WALLS + WALLS)
        if case["rough"]:
            recs, bot, top = _rough(case, seed)
            s.set_ibm(DP.IbmForcingSet(nx, nz, ny, recs))
            s.set_columns(bot, top)
        for name, t in _step_fields(case, seed).items():
            s.write(name, t)
        st = dict(kind="step", step=s, graph=case["graph"], out={n: _step_view(s, n) for n in STEP_OUT})
        if case["graph"]:
            st["stream"] = _captured(lambda q: s.capture(stream=q))
        return st
    props = case["props"]
    s = DP.ProjectionStep(nx, nz, ny, yu, *_inv_d(nx, nz), DT, incompressible=props == "incompressible")
    nu, cond, sf, gy = _phys(props)
    p = PR.Predictor(s, yu, nu, cond, WALLS + (T_WALLS[props][0],) + WALLS + (T_WALLS[props][1],), Sf_x=sf,
                     Gb=(0.0, gy, 0.0))
    out = {n: _step_view(s, n) for n in TIME_OUT}
    out.update({n: _pred_view(p, n) for n in PRED_OUT})
    forcing = None
    if case["rough"]:
        recs, bot, top = _rough(case, seed)
        forcing = DP.IbmForcingSet(nx, nz, ny, recs)
        p.set_ibm(forcing.handles)
        p.set_columns(bot, top)
    if props != "incompressible":
        laws, divjac, buoy = _laws(props)
        for q, law in laws.items():
            p.set_law(q, law)
        p.set_derived(divjac, buoy)
        out.update({n: _pred_view(p, n) for n in PROP_OUT})
        out.update(rho=_step_view(s, "rho"), div_now=_step_view(s, "div_now"))
    for name, t in _time_fields(case, seed).items():
        (s if name in DP.STEP_FIELDS else p).write(name, t)
    st = dict(kind="time_step", step=s, pred=p, forcing=forcing, graph=case["graph"], out=out)
    if case["graph"]:
        st["stream"] = _captured(lambda q: p.capture(with_step=True, stream=q))
    return st


def _captured(capture):
    """Records a graph on a side stream; it is replayed on the current one."""
    q = torch.cuda.Stream()
    q.wait_stream(torch.cuda.current_stream())
    capture(q)
    return q


def run(state):
    kind = state["kind"]
    if kind == "solve":
        return state["solver"].solve(state["rhs"], state["P"])
    if kind == "mixed":
        return state["solver"].solve_mixed(state["rhs"], state["P"], 1)
    if kind == "batch":
        state["batch"].run()
        return state["P"]
    if kind == "step":
        if state["graph"]:
            state["step"].launch()
        else:
            state["step"].enqueue()
        return state["out"]
    if state["graph"]:
        state["pred"].launch()
    else:
        state["pred"].enqueue()
        state["step"].enqueue()
    return state["out"]


def _solve_work(nx, nz, ny):
    """rhs read and P written once; two transforms each way and the sweep."""
    n = nx * nz * ny
    return 16 * n, n * (5 * (math.log2(nx) + math.log2(nz)) + 10)


def work(case):
    if case["kind"] == "batch":
        w = [_solve_work(c["nx"], c["nz"], c["ny"]) for c in _batch_cases(case)]
        return {"bytes": sum(b for b, _ in w), "flops": sum(f for _, f in w)}
    nx, nz, ny = case["nx"], case["nz"], case["ny"]
    n = nx * nz * ny
    solve_bytes, flops = _solve_work(nx, nz, ny)
    if case["kind"] == "solve":
        return {"bytes": solve_bytes, "flops": flops * (2 if case["form"] == "mixed" else 1)}
    if case["kind"] == "step":
        # variable: hats, rho, P_now, P_old, div_now in; U, V, W, P_per, P_now, P_old, P out
        fields = 14 if case["density"] == "variable" else 8
        return {"bytes": 8 * fields * n, "flops": flops + (110 if case["density"] == "variable" else 25) * n}
    # state in: U, V, W, T, four histories (and mu, cp, rho, div_now, buoy, RHS_energy, P_now, P_old);
    # out: the same, P, P_per (and the properties)
    fields = 16 + 22 if case["props"] != "incompressible" else 8 + 10
    return {"bytes": 8 * fields * n, "flops": flops + (520 if case["props"] != "incompressible" else 190) * n}


# ---------------------------------------------------------------------------
# the same results in 64 bits from torch alone
# ---------------------------------------------------------------------------
def _exact_solve(f, yu):
    ny, nz, nx = f.shape
    idx, idz = _inv_d(nx, nz)
    S = torch.fft.fft(torch.fft.rfft(f, dim=2), dim=1)
    mean = S[:, 0, 0].real.clone()
    kx = torch.arange(nx // 2 + 1, dtype=F8, device=DEV)
    kz = torch.arange(nz, dtype=F8, device=DEV)
    lam = -4 * idx * idx * torch.sin(kx * (math.pi / nx)).square()[None, :] \
        - 4 * idz * idz * torch.sin(kz * (math.pi / nz)).square()[:, None]
    a, b, c = _bands(yu, False)
    lam[0, 0] = -1.0  # replaced below
    cp = torch.empty((ny,) + lam.shape, dtype=F8, device=DEV)
    for k in range(ny):
        den = lam + b[k]
        if k:
            den -= a[k] * cp[k - 1]
            S[k] -= a[k] * S[k - 1]
        S[k] /= den
        cp[k] = c[k] / den
    for k in range(ny - 2, -1, -1):
        S[k] -= cp[k] * S[k + 1]
    del cp
    a, b, c = _bands(yu, True)
    d, e = mean.cpu().numpy(), np.zeros(ny)
    for k in range(ny):
        den = b[k] - (a[k] * e[k - 1] if k else 0.0)
        d[k] = (d[k] - (a[k] * d[k - 1] if k else 0.0)) / den
        e[k] = c[k] / den
    for k in range(ny - 2, -1, -1):
        d[k] -= e[k] * d[k + 1]
    S[:, 0, 0] = torch.from_numpy(d).to(DEV)
    return torch.fft.irfft(torch.fft.ifft(S, dim=1), n=nx, dim=2)


def _at(A, di, dj, dk):
    """Interior-shaped view of a padded array, shifted."""
    ny, nz, nx = (n - 2 for n in A.shape)
    return A[1 + dk:1 + dk + ny, 1 + dj:1 + dj + nz, 1 + di:1 + di + nx]


def _halo(A, planes=slice(None)):
    """Periodic x and z halos of the given padded planes."""
    B = A[planes]
    B[:, :, 0], B[:, :, -1] = B[:, :, -2].clone(), B[:, :, 1].clone()
    B[:, 0, :], B[:, -1, :] = B[:, -2, :].clone(), B[:, 1, :].clone()


def _col(v):
    return torch.as_tensor(np.ascontiguousarray(v), dtype=F8, device=DEV)[:, None, None]


def _force(A, rec):
    """Rough-wall forcing of a padded field, with its periodic images."""
    ijk, c = rec
    ijk = torch.from_numpy(ijk.astype(np.int64)).to(DEV)
    c = torch.from_numpy(c).to(DEV)
    nz2, nx2 = A.shape[1], A.shape[2]
    ny, nz, nx = (n - 2 for n in A.shape)
    ijk = torch.stack([ijk[:, q] % (nx, nz, ny)[q % 3] for q in range(9)], dim=1)  # indices wrap as read
    pos = [((ijk[:, 3 * q + 2] + 1) * nz2 + ijk[:, 3 * q + 1] + 1) * nx2 + ijk[:, 3 * q] + 1 for q in range(3)]
    flat = A.view(-1)
    v = c[:, 1] * flat[pos[1]] + c[:, 2] * flat[pos[2]] + c[:, 0]
    flat[pos[0]] = v
    i, j, k = ijk[:, 0], ijk[:, 1], ijk[:, 2]
    for si in (-1, 0, 1):
        for sj in (-1, 0, 1):
            for sk in (-1, 0, 1):
                q = (i + si * nx, j + sj * nz, k + sk * ny)
                m = (q[0] >= -1) & (q[0] <= nx) & (q[1] >= -1) & (q[1] <= nz) & (q[2] >= -1) & (q[2] <= ny)
                if (si, sj, sk) != (0, 0, 0) and bool(m.any()):
                    flat[((q[2][m] + 1) * nz2 + q[1][m] + 1) * nx2 + q[0][m] + 1] = v[m]


def _columns(A, bot, top, kmax, wb, wt):
    ny = A.shape[0] - 2
    k = torch.arange(-1, ny + 1, device=DEV)[:, None, None]
    b, t = (torch.from_numpy(v.astype(np.int64)).to(DEV)[None] for v in (bot, top))
    B = A[:, 1:-1, 1:-1]
    B[(k >= 0) & (k <= torch.clamp(b, max=ny))] = wb
    B[(k >= torch.clamp(t, min=-1)) & (k <= kmax)] = wt


def _exact_projection(F, yu, nx, nz, variable):
    """Right-hand side, solve and gradient correction on the fields F (padded;
    U_hat, V_hat, W_hat and, with `variable`, rho, P_now, P_old, div_now)."""
    idx, idz = _inv_d(nx, nz)
    yp = 0.5 * (yu[:-1] + yu[1:])
    pad = np.concatenate([[2 * yu[0] - yp[0]], yp, [2 * yu[-1] - yp[-1]]])
    idy, idyp = _col(1.0 / np.diff(yu)), 1.0 / np.diff(pad)
    ny = yp.size
    Uh, Vh, Wh = F["U_hat"], F["V_hat"], F["W_hat"]
    div = (_at(Uh, 1, 0, 0) - _at(Uh, 0, 0, 0)) * idx + (_at(Wh, 0, 1, 0) - _at(Wh, 0, 0, 0)) * idz \
        + (_at(Vh, 0, 0, 1) - _at(Vh, 0, 0, 0)) * idy
    if variable:
        rho = F["rho"]
        rmin = _at(rho, 0, 0, 0).min()
        Ps = 2 * F["P_now"] - F["P_old"]

        def flux(d):
            s = 1.0 - rmin * (0.5 / _at(rho, *d) + 0.5 / _at(rho, 0, 0, 0))
            return s * (_at(Ps, *d) - _at(Ps, 0, 0, 0))

        rhs = rmin / DT * (div - _at(F["div_now"], 0, 0, 0)) \
            + (flux((1, 0, 0)) + flux((-1, 0, 0))) * (idx * idx) + (flux((0, 1, 0)) + flux((0, -1, 0))) * (idz * idz) \
            + (flux((0, 0, 1)) * _col(idyp[1:]) + flux((0, 0, -1)) * _col(idyp[:-1])) * idy
    else:
        rhs = div / DT
    P = _exact_solve(rhs, yu)
    del rhs, div
    per = torch.empty_like(Uh)
    per[1:-1, 1:-1, 1:-1] = P
    per[0, 1:-1, 1:-1], per[-1, 1:-1, 1:-1] = P[0], P[-1]
    _halo(per)

    def grad(d):
        if not variable:
            return P, _at(per, *d)
        ir, im = 0.5 / _at(F["rho"], 0, 0, 0) + 0.5 / _at(F["rho"], *d), 1.0 / rmin
        return P * im + (ir - im) * _at(Ps, 0, 0, 0), _at(per, *d) * im + (ir - im) * _at(Ps, *d)

    out = {n: torch.zeros_like(Uh) for n in "UVW"}
    f, b = grad((-1, 0, 0))
    _at(out["U"], 0, 0, 0).copy_(_at(Uh, 0, 0, 0) - DT * (f - b) * idx)
    f, b = grad((0, -1, 0))
    _at(out["W"], 0, 0, 0).copy_(_at(Wh, 0, 0, 0) - DT * (f - b) * idz)
    f, b = grad((0, 0, -1))
    dy = np.concatenate([[np.inf], np.diff(yp)])
    _at(out["V"], 0, 0, 0).copy_(_at(Vh, 0, 0, 0) - DT * (f - b) * _col(1.0 / dy))
    for n in "UVW":
        _walls(out[n], n == "V", 0.0, 0.0)
    out.update(P=P, P_per=per)
    if variable:
        out.update(P_now=per, P_old=F["P_now"])
    return out


def _walls(A, is_v, bottom, top):
    """Periodic halos, then the wall planes over the whole padded plane."""
    _halo(A)
    A[0], A[-1] = bottom, top
    if is_v:
        A[1] = bottom


def _exact_step(case, seed):
    nx, nz, ny = case["nx"], case["nz"], case["ny"]
    F = _step_fields(case, seed)
    out = _exact_projection(F, _faces(ny), nx, nz, case["density"] == "variable")
    if case["rough"]:
        recs, bot, top = _rough(case, seed)
        for n in "UVW":
            _columns(out[n], bot, top, ny if n == "V" else ny - 1, 0.0, 0.0)
            _walls(out[n], n == "V", 0.0, 0.0)
            _force(out[n], recs[n])
            out[n][0], out[n][-1] = 0.0, 0.0
    return {n: out.get(n) for n in STEP_OUT}


def _second(x0, x1, x2, wall):
    """d/dy and d2/dy2 weights at x1 of the parabola through three values, the
    value at a wall (`wall` -1: below, 1: above) being given at the wall."""
    s, n = x0 - x1, x2 - x1
    if wall < 0:
        det = n * n * s - 2 * n * s * s
        d1 = (n * n / det, (-n * n + 2 * s * s) / det, -2 * s * s / det)
        return d1, (-2 * n / det, 2 * (n - s) / det, 2 * s / det)
    if wall > 0:
        det = -2 * n * n * s + n * s * s
        d1 = (-2 * n * n / det, (2 * n * n - s * s) / det, s * s / det)
        return d1, (2 * n / det, 2 * (-n + s) / det, -2 * s / det)
    det = n * n * s - n * s * s
    return (n * n / det, (-n * n + s * s) / det, -s * s / det), (-2 * n / det, 2 * (n - s) / det, 2 * s / det)


def _exact_props(laws, divjac, buoy, T):
    def law(q):
        spec = laws[q]
        if spec[0] == "const":
            return torch.full_like(T, spec[1])
        if spec[0] == "power":
            return spec[1] * T ** spec[2]
        seg = torch.tensor([[math.inf if s[0] is None else s[0], *s[1:]] for s in spec[1]], dtype=F8, device=DEV)
        s = seg[torch.searchsorted(seg[:-1, 0].contiguous(), T)]
        d = T - s[..., 1]
        return s[..., 2] + d * (s[..., 3] + d * (s[..., 4] + d * s[..., 5]))

    p = {q: law(q) for q in ("enth", "rho", "mu", "cond", "cp")}
    p["divjac"] = -law("drho_dT") / (p["rho"].square() * p["cp"]) if divjac[0] == "formula" \
        else torch.full_like(T, divjac[1])
    p["buoy"] = buoy[1] * (p["rho"] - buoy[2]) if buoy[0] == "linear" else torch.zeros_like(T)
    return p


class _Step64:
    """One time step's predictor part in 64 bits."""

    def __init__(self, case, seed):
        self.nx, self.nz, self.ny = case["nx"], case["nz"], case["ny"]
        self.yu = yu = _faces(self.ny)
        self.idx, self.idz = _inv_d(self.nx, self.nz)
        self.props = case["props"]
        self.variable = self.props != "incompressible"
        self.nu, self.cond, self.sf, self.gy = _phys(self.props)
        self.tw = T_WALLS[self.props]
        yp = 0.5 * (yu[:-1] + yu[1:])
        ext = np.concatenate([[yu[0]], yp, [yu[-1]]])
        ny = self.ny
        c = [_second(ext[i], ext[i + 1], ext[i + 2], -1 if i == 0 else (1 if i == ny - 1 else 0)) for i in range(ny)]
        v = [((0.0,) * 3, (0.0,) * 3) if i == 0 else _second(yu[i - 1], yu[i], yu[i + 1], 0) for i in range(ny)]
        self.c1, self.c2 = ([_col(np.array([r[m][q] for r in c])) for q in range(3)] for m in range(2))
        self.v1, self.v2 = ([_col(np.array([r[m][q] for r in v])) for q in range(3)] for m in range(2))
        down = np.concatenate([[0.0], yu[1:-1] - yp[:-1]])
        up = np.concatenate([[1.0], yp[1:] - yu[1:-1]])
        self.ib, self.it = _col(1 - down / (up + down)), _col(1 - up / (up + down))
        self.idyu = _col(1.0 / np.diff(ext)[:-1])
        w = (ext[0] - ext[1]) / (ext[2] - ext[1]), (ext[-1] - ext[-2]) / (ext[-3] - ext[-2])
        self.extrap = (1 - w[0], w[0], 1 - w[1], w[1])
        self.rough = _rough(case, seed) if case["rough"] else None

    def _d(self, A, w):
        """First derivatives (x, z, y) at interior points; w: y weights."""
        return (0.5 * self.idx * (_at(A, 1, 0, 0) - _at(A, -1, 0, 0)),
                0.5 * self.idz * (_at(A, 0, 1, 0) - _at(A, 0, -1, 0)),
                _at(A, 0, 0, -1) * w[0] + _at(A, 0, 0, 0) * w[1] + _at(A, 0, 0, 1) * w[2])

    def _lap(self, A, w2):
        c = _at(A, 0, 0, 0)
        return (_at(A, 1, 0, 0) - 2 * c + _at(A, -1, 0, 0)) * self.idx ** 2 \
            + (_at(A, 0, 1, 0) - 2 * c + _at(A, 0, -1, 0)) * self.idz ** 2 \
            + _at(A, 0, 0, -1) * w2[0] + c * w2[1] + _at(A, 0, 0, 1) * w2[2]

    def momentum(self, U, V, Wz, mu, rho, dv, b):
        def avg(A, *ds):
            return sum(_at(A, *d) for d in ds) / len(ds)

        o, idx, idz = (0, 0, 0), self.idx, self.idz
        ux, uz, uy = self._d(U, self.c1)
        wx, wz, wy = self._d(Wz, self.c1)
        vx, vz, vy = self._d(V, self.v1)
        u, v, w = _at(U, *o), _at(V, *o), _at(Wz, *o)
        v_u = avg(V, o, (-1, 0, 0), (0, 0, 1), (-1, 0, 1))
        w_u = avg(Wz, o, (-1, 0, 0), (0, 1, 0), (-1, 1, 0))
        u_w = avg(U, o, (0, -1, 0), (1, 0, 0), (1, -1, 0))
        v_w = avg(V, o, (0, -1, 0), (0, 0, 1), (0, -1, 1))
        u_v = avg(U, (0, 0, -1), (1, 0, -1)) * self.ib + avg(U, o, (1, 0, 0)) * self.it
        w_v = avg(Wz, (0, 0, -1), (0, 1, -1)) * self.ib + avg(Wz, o, (0, 1, 0)) * self.it
        lu, lw, lv = self._lap(U, self.c2), self._lap(Wz, self.c2), self._lap(V, self.v2)
        cu, cw, cv = u * ux + v_u * uy + w_u * uz, u_w * wx + v_w * wy + w * wz, u_v * vx + v * vy + w_v * vz
        if not self.variable:
            return -cu + self.nu * lu + self.sf, -cv + self.nu * lv, -cw + self.nu * lw
        m, Ra, Rb, Rc = mu, *self.c1
        d0, e = _at(dv, *o), (-1, 0, 0)
        visc = avg(m, e, o) * (lu + (d0 - _at(dv, *e)) * idx / 3) \
            + (2 * ux - (2 / 3) * avg(dv, e, o)) * (_at(m, *o) - _at(m, *e)) * idx \
            + (uy + (avg(V, o, (0, 0, 1)) - avg(V, e, (-1, 0, 1))) * idx) * (
                avg(m, (-1, 0, -1), (0, 0, -1)) * Ra + avg(m, e, o) * Rb + avg(m, (-1, 0, 1), (0, 0, 1)) * Rc) \
            + (uz + (avg(Wz, o, (0, 1, 0)) - avg(Wz, e, (-1, 1, 0))) * idx) * (
                avg(m, (-1, 1, 0), (0, 1, 0)) - avg(m, (-1, -1, 0), (0, -1, 0))) * (0.5 * idz)
        Ru = (visc - cu + self.sf) / avg(rho, e, o)
        e = (0, -1, 0)
        visc = avg(m, e, o) * (lw + (d0 - _at(dv, *e)) * idz / 3) \
            + (wx + (avg(U, o, (1, 0, 0)) - avg(U, e, (1, -1, 0))) * idz) * (
                avg(m, (1, -1, 0), (1, 0, 0)) - avg(m, (-1, -1, 0), (-1, 0, 0))) * (0.5 * idx) \
            + (wy + (avg(V, o, (0, 0, 1)) - avg(V, e, (0, -1, 1))) * idz) * (
                avg(m, (0, -1, -1), (0, 0, -1)) * Ra + avg(m, e, o) * Rb + avg(m, (0, -1, 1), (0, 0, 1)) * Rc) \
            + (2 * wz - (2 / 3) * avg(dv, e, o)) * (_at(m, *o) - _at(m, *e)) * idz
        Rw = (visc - cw) / avg(rho, e, o)
        e, iy = (0, 0, -1), self.idyu
        visc = avg(m, e, o) * (lv + (d0 - _at(dv, *e)) * iy / 3) \
            + (vx + (avg(U, o, (1, 0, 0)) - avg(U, e, (1, 0, -1))) * iy) * (
                avg(m, (1, 0, -1), (1, 0, 0)) - avg(m, (-1, 0, -1), (-1, 0, 0))) * (0.5 * idx) \
            + (2 * vy - (2 / 3) * avg(dv, e, o)) * (_at(m, *o) - _at(m, *e)) * iy \
            + (vz + (avg(Wz, o, (0, 1, 0)) - avg(Wz, e, (0, 1, -1))) * iy) * (
                avg(m, (0, 1, -1), (0, 1, 0)) - avg(m, (0, -1, -1), (0, -1, 0))) * (0.5 * idz)
        Rv = (visc - cv + self.gy * avg(b, o, e)) / avg(rho, e, o)
        return Ru, Rv, Rw

    def open(self, F):
        """Periodicity and walls, or the rough wall's forcing and wall planes."""
        if self.rough is None:
            for n in "UVW":
                _walls(F[n], n == "V", 0.0, 0.0)
            _walls(F["T"], False, *self.tw)
        else:
            for n in "UVW":
                _force(F[n], self.rough[0][n])
            for n, (lo, hi) in dict(U=(0, 0), V=(0, 0), W=(0, 0), T=self.tw).items():
                F[n][0], F[n][-1] = lo, hi
        if self.variable:
            e, dv = self.extrap, F["div_now"]
            dv[0] = e[0] * dv[1] + e[1] * dv[2]
            dv[-1] = e[2] * dv[-2] + e[3] * dv[-3]

    def predictor(self, F):
        self.open(F)
        U, V, Wz, T = F["U"], F["V"], F["W"], F["T"]
        R = self.momentum(U, V, Wz, F.get("mu"), F.get("rho"), F.get("div_now"), F.get("buoy"))
        hats = {}
        for n, r in zip("UVW", R):
            h = hats[n + "_hat"] = torch.zeros_like(U)
            old = F["R%s_old" % n.lower()]
            new = _at(F[n], 0, 0, 0) + DT * (1.5 * r - 0.5 * old)
            first = 1 if n == "V" else 0
            _at(h, 0, 0, 0)[first:] = new[first:]
            old[first:] = r[first:]
        tx, tz, ty = self._d(T, self.c1)
        o = (0, 0, 0)
        conv = 0.5 * (_at(U, *o) + _at(U, 1, 0, 0)) * tx + 0.5 * (_at(Wz, *o) + _at(Wz, 0, 1, 0)) * tz \
            + 0.5 * (_at(V, *o) + _at(V, 0, 0, 1)) * ty
        if self.variable:
            r = -conv + F["RHS_energy"] / (_at(F["rho"], *o) * _at(F["cp"], *o))
        else:
            r = -conv + self.cond * self._lap(T, self.c2)
        _at(T, *o).add_(DT * (1.5 * r - 0.5 * F["Rt_old"]))
        F["Rt_old"] = r
        four = dict(hats, T=T)
        for n, A in four.items():
            if self.rough is not None:
                lo, hi = self.tw if n == "T" else (0.0, 0.0)
                _columns(A, self.rough[1], self.rough[2], self.ny if n == "V_hat" else self.ny - 1, lo, hi)
            _walls(A, n == "V_hat", *(self.tw if n == "T" else (0.0, 0.0)))
        F.update(hats)
        if self.variable:
            Te = F["T_ext"] = T.clone()
            if self.rough is not None:
                _columns(Te, self.rough[1], self.rough[2], self.ny - 1, *self.tw)
                _halo(Te[1:-1])
            F.update(_exact_props(*_laws(self.props), Te))
            q = F["cond"]
            g, t = self._d(q, self.c1), self._d(T, self.c1)
            rhs = _at(q, *o) * self._lap(T, self.c2) + g[0] * t[0] + g[1] * t[1] + g[2] * t[2]
            F["RHS_energy"] = rhs
            dv = F["div_now"] = torch.zeros_like(T)
            _at(dv, *o).copy_(_at(F["divjac"], *o) * rhs)
            if self.rough is not None:
                _columns(dv, self.rough[1], self.rough[2], self.ny - 1, 0.0, 0.0)
            _halo(dv)
            dv[0] = dv[-1] = 0.0


def _exact_time_step(case, seed):
    nx, nz, ny = case["nx"], case["nz"], case["ny"]
    s = _Step64(case, seed)
    F = _time_fields(case, seed)
    F.update({n: torch.zeros((ny, nz, nx), dtype=F8, device=DEV) for n in ("Ru_old", "Rv_old", "Rw_old", "Rt_old")})
    s.predictor(F)
    F.update({n: torch.zeros_like(F["U"]) for n in ("P_now", "P_old")})
    F.update({n: v for n, v in _exact_projection(F, s.yu, nx, nz, s.variable).items() if n in TIME_OUT})
    return {n: F[n] for n in TIME_OUT + PRED_OUT + (PROP_OUT + ("rho", "div_now") if s.variable else ())}


def exact(case, seed):
    if case["kind"] == "solve":
        shape = (case["ny"], case["nz"], case["nx"])
        return _exact_solve(_rhs(shape, seed), _faces(case["ny"]))
    if case["kind"] == "batch":
        return [_exact_solve(_rhs((c["ny"], c["nz"], c["nx"]), seed + 1000 * i), _faces(c["ny"]))
                for i, c in enumerate(_batch_cases(case))]
    if case["kind"] == "step":
        return _exact_step(case, seed)
    return _exact_time_step(case, seed)
