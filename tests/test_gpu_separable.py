"""The separable solver of the consistent projection (proj_mode 2 on grids
without cross terms) against the FP64 line-multigrid cycles of proj_mode 1,
which never take it: both stop at max|residual| <= tol, so after two
substeps the velocities agree to 1e-8 and the pressure, which sums
phi / H_BAR, to 1e-6 (the bounds of the other comparisons of two converged
projections, which are quoted for tol = 1e-12 on the 65 x 65 plane; the
residual is J div u, so tol scales with J, the cell area, here).  Planes at the edges of the solver's tiles (columns around 64
and 128 per wavefront stripe and workgroup, rows around the 16-row tiles),
every set of sides, and z spacings from uniform to so uneven that the passes
leave work to the V cycles (more than 5 cycles of a solve, the passes being at
most 5) or the operator is not taken as separable and the FP32 V cycles do all
of it (the outer iteration, proj_krylov, then changes their number)."""
import numpy as np
import pytest

from ekman_bl_amd import solver as S
from ekman_bl_amd.grid import tanh_grid
from ekman_bl_amd.ic import ekman_initial
from ekman_bl_amd.params import config, mg_factors

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def _run(p, xp, yp, ic, mode, guess=0, krylov=1, tol=1e-12):
    q = p.copy()
    tol *= min(1.0, 64.0 / (p.nz + 1) * 64.0 / (p.ny + 1))
    q.proj_mode, q.proj_tol, q.proj_maxit, q.proj_guess, q.proj_krylov = mode, tol, 50, guess, krylov
    s = S.DuctSolver(q, xp, yp)
    s.set_initial_physical(*ic)
    for _ in range(2):
        s.rk_duct()
    d, cyc, out = s.diag(), s.solve_cycles(), s.get_state()
    s.close()
    assert d.status == 0 and d.mg_unconverged == 0 and d.div_max < 1e-10
    return out, cyc


@pytest.mark.parametrize("nx,ny2,nz2,bcs,wave", [
    (16, 33, 33, (2, 2, 2, 1), 0.0),     # one stripe, columns of several solves per workgroup
    (16, 41, 65, (2, 2, 2, 1), 0.0),     # one point past a stripe
    (32, 49, 129, (1, 1, 1, 1), 0.0),    # specified sides: 47 rows, columns without an unknown
    (8, 129, 385, (2, 2, 2, 2), 0.0),    # no specified side: singular kx = 0; 129 rows
    (16, 65, 193, (2, 1, 1, 2), 0.0),    # one specified end per direction
    (8, 33, 641, (0, 0, 2, 1), 0.0),     # periodic, the longest lines
    (8, 65, 97, (0, 0, 2, 2), 0.0),      # periodic and singular
    (32, 33, 33, (2, 2, 2, 1), 0.1),     # uneven z: all 5 passes
    (32, 33, 33, (2, 2, 2, 1), 0.14),    # too uneven: V cycles throughout
])
def test_separable_solver_matches_fp64_cycles(nx, ny2, nz2, bcs, wave):
    z = np.linspace(0.0, 1.0, nz2)
    p, xp, yp, ic = _case(nx, ny2, nz2, bcs, z + wave * np.sin(2 * np.pi * z))
    ref, _ = _run(p, xp, yp, ic, 1)
    for guess in (0, 1):
        got, cyc = _run(p, xp, yp, ic, 2, guess)
        _compare(f"separable {nx}x{ny2}x{nz2} {bcs} wave {wave} guess {guess}", got, ref, cyc)
        if wave <= 0.1:
            assert cyc.max() <= 5    # the passes alone


def _case(nx, ny2, nz2, bcs, z):
    """Parameters, grid and initial condition of a neutral case with the z
    points z (0..1) in every row and the tanh spacing in y."""
    cfg = config(1)
    p = cfg.params
    p.nx, p.ny, p.nz = nx, ny2 - 2, nz2 - 2
    p.mg_ixp, p.mg_iex = mg_factors(nz2)
    p.mg_jyq, p.mg_jey = mg_factors(ny2)
    p.delta_t = 0.02
    for k, b in enumerate(bcs):
        p.mudpack_bc[k] = b
    if bcs[0] == 0:
        for c in range(3):
            p.u_bc[c][2] = p.u_bc[c][3] = 6
    xp, yp = tanh_grid(p.ny, p.nz, p.ly, p.lz, cfg.gamma)
    xp = np.broadcast_to(z * p.lz, xp.shape).copy()
    return p, xp, yp, ekman_initial(p, yp, 3, 0.05, 0.0)


def _compare(what, got, ref, cyc):
    r = [_rel(a, b) for a, b in zip(got[:4], ref[:4])]
    print(f"[{what}] velocities {max(r[:3]):.1e} pressure {r[3]:.1e} cycles max {cyc.max()}", flush=True)
    assert max(r[:3]) < 1e-8 and r[3] < 1e-6


@pytest.mark.parametrize("bcs,wave,tol", [
    ((2, 2, 2, 1), 0.125, 1e-13), ((0, 0, 2, 1), 0.125, 1e-13),
    ((2, 2, 2, 2), 0.126, 5e-15), ((0, 0, 2, 2), 0.125, 1e-13),   # singular: kx = 0 is among those that go on
])
def test_passes_hand_over_to_v_cycles(bcs, wave, tol):
    """A z spacing just within what is taken as separable, and a tolerance that
    5 passes do not reach: V cycles go on from where the passes ended, with
    either outer iteration, from zero and from a guess."""
    z = np.linspace(0.0, 1.0, 33)
    p, xp, yp, ic = _case(32, 33, 33, bcs, z + wave * np.sin(2 * np.pi * z))
    ref, _ = _run(p, xp, yp, ic, 1, tol=tol)
    for krylov in (0, 1):
        for guess in (0, 1):
            got, cyc = _run(p, xp, yp, ic, 2, guess, krylov, tol)
            _compare(f"hand-over {bcs} krylov {krylov} guess {guess}", got, ref, cyc)
            assert (cyc > 5).sum() > 10 and cyc[:2].max() > 5


@pytest.mark.parametrize("nx,ny2,nz2,bcs,krylovs", [
    (16, 33, 33, (2, 2, 2, 1), (0, 1)), (16, 41, 65, (1, 1, 1, 1), (0, 1)),
    (16, 33, 97, (0, 0, 2, 1), (0, 1)),
    (16, 33, 65, (2, 2, 2, 2), (0, 1)), (16, 33, 97, (0, 0, 2, 2), (0, 1)),  # singular
    (8, 33, 641, (0, 0, 2, 1), (0, 1)),
    (8, 33, 385, (2, 2, 2, 1), (1,)),  # plain refinement diverges here, in FP64 too
])
def test_v_cycles_without_cross_terms(nx, ny2, nz2, bcs, krylovs):
    """A z spacing that changes by 1.3 from one cell to the next is not taken as
    separable: the FP32 V cycles of grids without cross terms, with lines of
    every length class, both outer iterations and every kind of z ends."""
    h = np.ones(nz2 - 1)
    h[(nz2 - 1) // 3: 2 * (nz2 - 1) // 3] = 1.3
    z = np.concatenate([[0.0], np.cumsum(h)])
    p, xp, yp, ic = _case(nx, ny2, nz2, bcs, z / z[-1])
    ref, cref = _run(p, xp, yp, ic, 1)
    most = {}
    for krylov in krylovs:
        for guess in (0, 1):
            got, cyc = _run(p, xp, yp, ic, 2, guess, krylov)
            _compare(f"V cycles {nx}x{ny2}x{nz2} {bcs} krylov {krylov} guess {guess}", got, ref, cyc)
            if guess == 0:
                most[krylov] = int(cyc.max())
    # from the same start the FP32 cycles contract as the FP64 ones do, to the
    # cycle in which the tolerance is met
    assert abs(most[1] - int(cref.max())) <= 1
    assert len(krylovs) == 1 or most[0] > most[1]


def test_repeated_solves_are_identical():
    """The products and scans have a fixed order: two runs agree bit for bit."""
    cfg = config(1)
    p = cfg.params
    xp, yp = tanh_grid(p.ny, p.nz, p.ly, p.lz, cfg.gamma)
    ic = ekman_initial(p, yp, 3, 0.05, 0.0)
    a, _ = _run(p, xp, yp, ic, 2)
    b, _ = _run(p, xp, yp, ic, 2)
    assert all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("nx,ny2,nz2,bcs", [
    (128, 97, 129, (2, 2, 2, 1)),     # two points per thread and a remainder
    (128, 129, 193, (2, 2, 2, 1)),    # four points per thread and a remainder
    (128, 129, 193, (2, 2, 2, 2)),    # singular kx = 0: the start's residual is stored
])
def test_residual_pass_splits(nx, ny2, nz2, bcs):
    """The residual pass with several points per thread, from a zero start and
    from a guess, within the bounds of the comparison above."""
    p, xp, yp, ic = _case(nx, ny2, nz2, bcs, np.linspace(0.0, 1.0, nz2))
    ref, _ = _run(p, xp, yp, ic, 1)
    for guess in (0, 1):
        got, cyc = _run(p, xp, yp, ic, 2, guess)
        _compare(f"residual pass {nx}x{ny2}x{nz2} {bcs} guess {guess}", got, ref, cyc)
        assert cyc.max() <= 5
