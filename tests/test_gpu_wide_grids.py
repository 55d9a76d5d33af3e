"""Row pitches of 2^23 points and more, and arrays of 4 GiB and more in the FP64
coarse CG's arena: a V-cycle is compared with that of a narrow grid of the same
columns."""
import numpy as np
import pytest


def _vcycle(W, nx, first, precision):
    """V-cycle of a residual on 64 columns from `first`, on uniform ice: the
    correction on the 192 columns around them, outside which it is zero."""
    ny, dx = 2, 4000.0
    grid = W.Grid(nx=nx, ny=ny, nσ=2, x0=0.0, y0=0.0, dx=dx, dy=dx)
    ic = W.InitialConditions(initial_thickness=np.full((nx, ny), 1000.0, order="F"))
    sp = W.SolverParams(maxiter_picard=1, maxiter_coarse=1, levels=3)
    m = W.Model(grid=grid, bed_elevation=np.full((nx, ny), -500.0, order="F"), solver_params=sp,
                params=W.Params(default_temperature=265.700709), initial_conditions=ic,
                parallel_spec=W.HIPSpec(precision))
    print("[gpu] model of %d x %d made" % (nx, ny), flush=True)
    W.update_preconditioner(m)
    W.push_fields(m)
    spec = m.parallel_spec
    assert spec._lib.wavi_update_geometry(spec.ctx) == 0
    assert spec._lib.wavi_inner_update(spec.ctx) == 0
    rng = np.random.default_rng(4)
    ru, rv = np.zeros((nx + 1, ny), order="F"), np.zeros((nx, ny + 1), order="F")
    ru[first:first + 64] = rng.standard_normal((64, ny))
    rv[first:first + 64] = rng.standard_normal((64, ny + 1))
    eu, ev, it = W.vcycle(m, ru, rv)
    assert it == 1
    spec.close()
    win = slice(first - 64, first + 128)
    for e in (eu, ev):
        assert not e[:first - 64].any() and not e[first + 128:].any()
    return eu[win].copy(), ev[win].copy()


# the tiles' sums are the same; only their sum over the tiles, in FP64, is in
# another order, which can move the step length by roundings
@pytest.mark.gpu
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-10), ("mixed", 1e-5)])
def test_widest_pitch_equals_a_narrow_grid(W, precision, tol):
    nx = 1 << 23
    print("[gpu] V-cycle on %d x 2, %s" % (nx, precision), flush=True)
    ref = _vcycle(W, 256, 96, precision)
    got = _vcycle(W, nx, nx - 4096 + 96, precision)
    for a, b in zip(got, ref):
        assert np.abs(b).max() > 0.0
        assert np.abs(a - b).max() <= tol * np.abs(b).max()
