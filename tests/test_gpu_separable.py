"""The separable solver of the consistent projection (proj_mode 2 on grids
without cross terms) against the FP64 line-multigrid cycles of proj_mode 1,
which never take it: both stop at max|residual| <= tol, so after two
substeps the velocities agree to 1e-8 and the pressure, which sums
phi / H_BAR, to 1e-6 (the bounds of the other comparisons of two converged
projections, which are quoted for tol = 1e-12 on the 65 x 65 plane; the
residual is J div u, so tol scales with J, the cell area, here).  Planes at the edges of the solver's tiles (columns around 64
and 128 per wavefront stripe and workgroup, rows around the 16-row tiles),
every set of sides, and z spacings from uniform to so uneven that the passes
leave work to the V cycles or the operator is not taken as separable."""
import numpy as np
import pytest

from ekman_bl_amd import solver as S
from ekman_bl_amd.grid import tanh_grid
from ekman_bl_amd.ic import ekman_initial
from ekman_bl_amd.params import config, mg_factors

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def _run(p, xp, yp, ic, mode, guess=0):
    q = p.copy()
    tol = 1e-12 * min(1.0, 64.0 / (p.nz + 1) * 64.0 / (p.ny + 1))
    q.proj_mode, q.proj_tol, q.proj_maxit, q.proj_guess = mode, tol, 50, guess
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
    (32, 33, 33, (2, 2, 2, 1), 0.1),     # uneven z: more passes, then V cycles
    (32, 33, 33, (2, 2, 2, 1), 0.14),    # too uneven: V cycles throughout
])
def test_separable_solver_matches_fp64_cycles(nx, ny2, nz2, bcs, wave):
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
    z = np.linspace(0.0, 1.0, nz2)
    xp = np.broadcast_to((z + wave * np.sin(2 * np.pi * z)) * p.lz, xp.shape).copy()
    ic = ekman_initial(p, yp, 3, 0.05, 0.0)
    ref, _ = _run(p, xp, yp, ic, 1)
    for guess in (0, 1):
        got, cyc = _run(p, xp, yp, ic, 2, guess)
        r = [_rel(a, b) for a, b in zip(got[:4], ref[:4])]
        print(f"[separable {nx}x{ny2}x{nz2} {bcs} wave {wave} guess {guess}] velocities {max(r[:3]):.1e} "
              f"pressure {r[3]:.1e} cycles max {cyc.max()}", flush=True)
        assert max(r[:3]) < 1e-8 and r[3] < 1e-6
        if wave == 0.0:
            assert cyc.max() <= 5    # the passes alone


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
    cfg = config(1)
    p = cfg.params
    p.nx, p.ny, p.nz = nx, ny2 - 2, nz2 - 2
    p.mg_ixp, p.mg_iex = mg_factors(nz2)
    p.mg_jyq, p.mg_jey = mg_factors(ny2)
    p.delta_t = 0.02
    for k, b in enumerate(bcs):
        p.mudpack_bc[k] = b
    xp, yp = tanh_grid(p.ny, p.nz, p.ly, p.lz, cfg.gamma)
    ic = ekman_initial(p, yp, 3, 0.05, 0.0)
    ref, _ = _run(p, xp, yp, ic, 1)
    for guess in (0, 1):
        got, cyc = _run(p, xp, yp, ic, 2, guess)
        r = [_rel(a, b) for a, b in zip(got[:4], ref[:4])]
        assert max(r[:3]) < 1e-8 and r[3] < 1e-6 and cyc.max() <= 5
