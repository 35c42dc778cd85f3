"""The work that users of this package have it do, as measurable cases.

Most of it is the time step (`DuctSolver.time_step`, three RKW3+CN substeps
with their pressure projections), in the forms a run is configured with: the
plain FP64 drop-in with the MUDPACK replica (the default projection), the
consistent projection with FP32 cycles (eager and replayed from HIP graphs),
with and without the subgrid models, on free-slip and on periodic z ends, on
rectilinear and on curvilinear grids, and with the learned initial guess.
Beside it: the drop-in transforms and the drop-in tridiagonal solver on device
arrays, and the statistics a run writes every few steps.

A step case is a run in progress: `prepare` uploads a seeded state (the Ekman
profile with noise in every kept Fourier mode, as a restart at step 3, so the
subgrid models run from the first step), projects it as the start-up does, and
`run` advances it by one step and returns the state's five fields.
"""
import math
import os

import numpy as np
import torch

import ekman_bl_amd
from ekman_bl_amd import solver as S
from ekman_bl_amd.grid import tanh_grid
from ekman_bl_amd.params import YMAX, YMIN, ZMAX, ZMIN, config, mg_factors, params_from_fixture

DEV = "cuda:0"
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(ekman_bl_amd.__file__)))
GOLDEN = os.path.join(ROOT, "tests", "golden")


# -- the cases ------------------------------------------------------------------
def listed():
    return [
        # the 64x65x65 neutral configuration, plain form: the smallest run, launch-bound
        _step("plain_64x65x65", 64, 65, 65, "plain", th=0),
        # the same grid in the form that meets the divergence bound, replayed from graphs
        _step("fp32_graph_64x65x65", 64, 65, 65, "fp32", th=0, graph=True),
        # the stratified 256x193x257 configuration in the plain form (the reference's algorithm)
        _step("plain_256x193x257", 256, 193, 257, "plain"),
        # the same in the headline form
        _step("fp32_256x193x257", 256, 193, 257, "fp32"),
        # the same started from the learned guess (bf16 network on the matrix cores)
        _step("learned_256x193x257", 256, 193, 257, "learned"),
        # the reference run's own configuration: periodic multigrid z ends, no specified
        # side, type-6 rows, vertical sponge, constant pressure gradient, 256x129x321
        dict(name="fp32_reference_run", kind="reference_run", form="fp32", graph=False),
        # the stratified 512x257x513 configuration, replayed from graphs
        _step("fp32_graph_512x257x513", 512, 257, 513, "fp32", graph=True),
        # both subgrid models on the z-y plane of the 1024x385x769 configuration
        _step("les_fp32_256x385x769", 256, 385, 769, "fp32", les=1),
        # a sheared (curvilinear) grid with both subgrid models: cross terms everywhere
        _step("les_fp32_skewed_128x97x129", 128, 97, 129, "fp32", les=1, skew=1),
        # the transform drop-ins there and back on one field of the 256x193x257 grid
        dict(name="fft_256", kind="fft", nx=256, npencil=193 * 257),
        # the tridiagonal drop-in: one line per x point and z row of a small duct
        dict(name="thomas_192", kind="thomas", n=192, batch=257 * 65),
        # the statistics of the 256x193x257 run (x means, fluxes, higher moments)
        dict(name="stats_256x193x257", kind="stats", nx=256, ny2=193, nz2=257),
    ]


def _step(name, nx, ny2, nz2, form, th=1, les=0, skew=0, periodic=0, graph=False):
    c = dict(kind="step", nx=nx, ny2=ny2, nz2=nz2, form=form, th=th, les=les, skew=skew, periodic=periodic,
             graph=bool(graph))
    return dict(c, name=name) if name else c


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _points(rng, lo, hi):
    """m 2^k + 1 points (the multigrid's rule) with a log-uniform size target."""
    want = _log(rng, lo, hi)
    best = [m * 2 ** k + 1 for m in (2, 3, 5, 7) for k in range(1, 9) if lo <= m * 2 ** k + 1 <= hi]
    best.sort(key=lambda n: abs(math.log(n / want)))
    return rng.choice(best[:3])


def draw(rng):
    u = rng.random()
    if u < 0.08:
        nx = 2 ** rng.randint(4, 10)
        return dict(kind="fft", nx=nx, npencil=max(1, int(_log(rng, 2e3, 1.3e7) / nx)))
    if u < 0.14:
        n = int(_log(rng, 16, 800))
        return dict(kind="thomas", n=n, batch=max(1, int(_log(rng, 1e4, 4e6) / n)))
    if u < 0.20:
        return dict(kind="stats", nx=2 ** rng.randint(5, 8), ny2=_points(rng, 33, 193), nz2=_points(rng, 33, 257))
    if u < 0.26:  # planes the network takes: 32 m + 1 points each way
        return _step(None, 2 ** rng.randint(5, 8), 32 * rng.randint(2, 6) + 1, 32 * rng.randint(2, 8) + 1, "learned")
    form = "plain" if u < 0.50 else "fp32"
    most = 13e6 if form == "plain" else 60e6
    while True:
        nx = 2 ** rng.randint(5, 9)
        ny2, nz2 = _points(rng, 33, 385), _points(rng, 33, 769)
        if 3e4 <= nx * ny2 * nz2 <= most:
            break
    bc = rng.random()
    return _step(None, nx, ny2, nz2, form, th=int(rng.random() < 0.8), les=int(bc < 0.4), skew=int(rng.random() < 0.15),
                 periodic=int(bc > 0.75), graph=rng.random() < 0.5)


# -- states ---------------------------------------------------------------------
class _Buffer:
    """A device buffer of a solver as an array-interface object; a tensor made of it
    holds it, and so keeps the solver, whose memory it shows, alive."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f8", "data": (ptr, False), "version": 3}


def _fields(s):
    """The state's fields U1, U2, U3, P, TH: views of the solver's device buffers."""
    import ctypes
    p, out = s.p, []
    for f in range(5 if s.p.n_th else 4):
        ptr = ctypes.c_void_p()
        if S.lib().ekm_field_device_ptr(s.h, f, ctypes.byref(ptr)) != 0:
            raise RuntimeError("ekm_field_device_ptr")
        out.append(torch.as_tensor(_Buffer(s, ptr.value, (p.ny + 2, p.nz + 2, p.nx + 2)), device=DEV))
    return out


def _params(case):
    """(params, xpoint, ypoint, th_bar, wind) of a step or statistics case."""
    if case["kind"] == "reference_run":
        p, xp, yp = params_from_fixture(os.path.join(GOLDEN, "grid_yz_unst.json"),
                                        os.path.join(GOLDEN, "input_unst.dat"))
        p.proj_mode = 2 if case["form"] == "fp32" else 0
        return p, xp, yp, 1e-3 * yp, p.wbulk0
    cfg = config(2 if case.get("th", 1) else 1)
    p = cfg.params
    p.nx, p.ny, p.nz = case["nx"], case["ny2"] - 2, case["nz2"] - 2
    p.mg_ixp, p.mg_iex = mg_factors(p.nz + 2)
    p.mg_jyq, p.mg_jey = mg_factors(p.ny + 2)
    if case["kind"] == "step":
        p.proj_mode = 0 if case["form"] == "plain" else 2
        p.proj_guess = 2 if case["form"] == "learned" else 0
        p.les_model = 2 if case["les"] else 0
        if case["periodic"]:  # the reference run's boundary set with a specified pressure top
            for c in range(3):
                p.u_bc[c][ZMIN] = p.u_bc[c][ZMAX] = 6
            p.th_bc[YMIN] = 5
            p.th_bc[ZMIN] = p.th_bc[ZMAX] = 6
            p.mudpack_bc[0] = p.mudpack_bc[1] = 0
    # a step below the CFL limit from the start
    p.delta_t = min(p.delta_t, 0.3 * min(p.lx / p.nx, p.lz / p.nz))
    xp, yp = tanh_grid(p.ny, p.nz, p.ly, p.lz, cfg.gamma)
    if case.get("skew"):
        xp = xp + 0.05 * np.sin(0.3 * yp)
    return p, xp, yp, None, 1.0


def _state(p, yp, seed, ug, with_p):
    """Fourier U1, U2, U3, P, TH (device, complex128): the Ekman profile with 5%
    noise, theta with 1% noise, P zero or 1% noise; modes above NX/3 zero."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    y = torch.from_numpy(yp).to(DEV)[:, :, None]
    eta = y / math.sqrt(2.0 * p.nu / p.f0) if p.f0 > 0 else y
    base = [ug * (1.0 - torch.exp(-eta) * torch.cos(eta)), 0.0 * eta, -ug * torch.exp(-eta) * torch.sin(eta),
            0.0 * eta, 0.0 * eta]
    amp = [0.05 * ug, 0.05 * ug, 0.05 * ug, 0.01 if with_p else 0.0, 0.01 if p.n_th else 0.0]
    out = []
    for b, a in zip(base, amp):
        c = torch.zeros((p.ny + 2, p.nz + 2, p.nx // 2 + 1), dtype=torch.complex128, device=DEV)
        if a:
            u = b + a * (torch.rand((p.ny + 2, p.nz + 2, p.nx), dtype=torch.float64, device=DEV, generator=g) - 0.5)
            c[..., : p.nx // 3 + 1] = torch.fft.rfft(u, dim=-1, norm="forward")[..., : p.nx // 3 + 1]
            c[..., 0] = c[..., 0].real + 0j
        out.append(c)
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "fft":
        g = torch.Generator(device=DEV).manual_seed(seed)
        v = torch.zeros((case["npencil"], case["nx"] + 2), dtype=torch.float64, device=DEV)
        v[:, : case["nx"]] = torch.rand(v[:, : case["nx"]].shape, dtype=torch.float64, device=DEV, generator=g) - 0.5
        return dict(case=case, v=v)
    if kind == "thomas":
        return dict(case=case, **_thomas(case, seed))
    p, xp, yp, tb, ug = _params(case)
    s = S.DuctSolver(p, xp, yp, th_bar=tb)
    cu = [c.cpu().numpy() for c in _state(p, yp, seed, ug, kind == "stats")]
    s.set_state(*cu, time=0.0, time_step=3)
    st = dict(case=case, solver=s)
    if kind != "stats":
        s.rem_div_curv()
        if case["form"] == "learned":
            from ekman_bl_amd import warmstart as W
            st["net"] = W.WarmStartNet(p.nz + 2, p.ny + 2, 2 * (p.nx // 3 + 1))
            st["net"].load(os.path.join(os.path.dirname(W.__file__), "data", "wsnet.npz"))
            st["net"].attach(s)
        st["fields"] = _fields(s)
    del cu
    torch.cuda.empty_cache()
    return st


def _thomas(case, seed):
    """Crank-Nicolson diffusion rows with zero-flux ends, one coefficient per row and
    line, so a solve damps what varies along a line and keeps its mean part."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    n, m = case["n"], case["batch"]
    r = 0.1 + 2.0 * torch.rand((n, m), dtype=torch.float64, device=DEV, generator=g)
    a, c = -r, -r.flip(0)
    a[0], c[-1] = 0.0, 0.0
    return dict(a=a.contiguous(), b=(1.0 - a - c).contiguous(), c=c.contiguous(),
                g=1.0 + torch.rand((n, m), dtype=torch.float64, device=DEV, generator=g))


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "fft":
        v, L = st["v"], S.lib()
        stream = torch.cuda.current_stream().cuda_stream
        a = L.ekm_fft_x_to_fourier_dev(v.data_ptr(), case["nx"], case["npencil"], stream)
        b = L.ekm_fft_x_to_physical_dev(v.data_ptr(), case["nx"], case["npencil"], stream)
        if a or b:
            raise RuntimeError(f"transform: {a} {b}")
        return v
    if kind == "thomas":
        n, m = st["g"].shape
        e = S.lib().ekm_thomas_real_dev(st["a"].data_ptr(), st["b"].data_ptr(), st["c"].data_ptr(),
                                        st["g"].data_ptr(), n - 1, m - 1, torch.cuda.current_stream().cuda_stream)
        if e:
            raise RuntimeError(f"thomas: {e}")
        return st["g"]
    s = st["solver"]
    if kind == "stats":
        return {"stats": s.x_stats(), "moments": s.x_moments()}
    s.time_step(1, graph=case["graph"])
    return st["fields"]


# -- what a pass cannot do without ------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "fft":
        n = float(case["npencil"]) * case["nx"]
        return {"bytes": 16.0 * n, "flops": 2 * 2.5 * n * math.log2(case["nx"])}
    if kind == "thomas":
        n = float(case["n"]) * case["batch"]
        return {"bytes": 5 * 8.0 * n, "flops": 8.0 * n}
    p = _params(case)[0]
    n = float(p.nx) * (p.ny + 2) * (p.nz + 2)
    f = 4 + p.n_th
    if kind == "stats":
        return {"bytes": 8.0 * n * f, "flops": n * (3 * 2.5 * math.log2(p.nx) + 50)}
    # per substep the state (and the RK history of the transported fields) is read and
    # written; transforms of the transported fields there and back, their fluxes, the
    # implicit sweeps, and one residual's worth of work per Poisson unknown
    sub = n * ((f - 1) * (4 * 2.5 * math.log2(p.nx) + 120) + 60)
    return {"bytes": 3 * 8.0 * n * (2 * f + 2 * (f - 1)), "flops": 3 * sub}


def tolerance(case):
    kind = case["kind"]
    if kind == "fft":
        return {"rel": 2e-15, "max": 4e-14}
    if kind == "thomas":
        return {"rel": 2e-15, "max": 2e-14}
    if kind == "stats":
        return {"rel": 1e-12, "max": 1e-10}
    if case["form"] == "plain":
        # four times what the pressure of the plain step and the oracle's, with their
        # sums in another order, differ by over a few steps (5.4e-12)
        return {"rel": 2.2e-11, "max": 2e-9}
    # the projection stops at max|residual| <= 1e-12, and two correct iterations stop at
    # different points below it: with the plain and the GCR(1) outer iteration the pressure
    # (the sum of phi / H_BAR) differs by up to 1.5e-6 (5.5e-5 at a point) over three steps
    return {"rel": 6e-6, "max": 2.2e-4}


def exact(case, seed):
    kind = case["kind"]
    if kind == "fft":
        nx = case["nx"]
        v = prepare(case, seed)["v"]
        c = torch.fft.rfft(v[:, :nx], dim=-1)
        c[:, nx // 3 + 1:] = 0
        out = torch.zeros_like(v)
        out[:, :nx] = torch.fft.irfft(c, n=nx, dim=-1)
        return out
    if kind == "thomas":
        t = _thomas(case, seed)
        n = case["n"]
        b, g = t["b"].clone(), t["g"].clone()
        for j in range(1, n):
            w = t["a"][j] / b[j - 1]
            b[j] -= w * t["c"][j - 1]
            g[j] -= w * g[j - 1]
        g[n - 1] /= b[n - 1]
        for j in range(n - 2, -1, -1):
            g[j] = (g[j] - t["c"][j] * g[j + 1]) / b[j]
        return g
    if kind != "stats":
        return None  # a whole step: its layers have no closed form outside this package
    p, _, yp, _, ug = _params(case)
    f = [torch.fft.irfft(c, n=p.nx, dim=-1, norm="forward") for c in _state(p, yp, seed, ug, True)]
    mean = [a.mean(-1) for a in f]
    u, v, w, q, t = (a - m[..., None] for a, m in zip(f, mean))
    av = lambda *x: torch.stack([y for y in x]).prod(0).mean(-1).cpu().numpy()  # noqa: E731
    sq = lambda x: (x * x).sum(-1).cpu().numpy()  # noqa: E731
    names = S.DuctSolver.XSTATS
    vals = [m.cpu().numpy() for m in mean] + [sq(u), sq(v), sq(w), sq(t)] + [
        av(u, v), av(u, w), av(w, v), av(q, w), av(q, v), av(t, v), av(t, w)]
    mom = [av(u, u), av(v, v), av(w, w), av(u, u, u), av(v, v, v), av(w, w, w), av(u, u, u, u), av(v, v, v, v),
           av(w, w, w, w), av(u, u, v), av(w, w, v), av(u, u, u, v), av(w, w, w, v)]
    return {"stats": dict(zip(names, vals)), "moments": dict(zip(S.DuctSolver.XMOMENTS, mom))}
