"""Values that are not finite where there is no ice (missing data) reach no
result: the operator against the oracle, bit for bit, and a solve whose
Dirichlet velocities off the ice are NaN."""
import numpy as np
import pytest

from helpers import iceberg, ragged


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny", [(20, 20), (40, 24), (33, 17)])
def test_operator_takes_nothing_from_off_the_masks(W, oracle, nx, ny):
    print("[gpu] operator with NaN off the ice %dx%d" % (nx, ny), flush=True)
    m = iceberg(W, nx=nx, ny=ny)[0] if nx == ny else ragged(W, nx=nx, ny=ny)
    o = oracle.OracleModel(m)
    W.update_preconditioner(m)
    W.push_fields(m)
    spec = m.parallel_spec
    assert spec._lib.wavi_update_geometry(spec.ctx) == 0
    assert spec._lib.wavi_inner_update(spec.ctx) == 0
    o.update_geometry()
    o.inner_update()
    rng = np.random.default_rng(nx)
    off_u, off_v = ~m.fields.gu.mask, ~m.fields.gv.mask
    # off the masks only, then one point on each mask too
    for bad in (np.nan, np.inf, -np.inf):
        xu, xv = rng.standard_normal(off_u.shape), rng.standard_normal(off_v.shape)
        xu[off_u], xv[off_v] = bad, bad
        for on in (False, True):
            if on:
                for x, off in ((xu, off_u), (xv, off_v)):
                    i, j = np.argwhere(~off)[rng.integers((~off).sum())]
                    x[i, j] = bad
            yu, yv = W.op_apply(m, xu, xv, sampled=False)
            with np.errstate(invalid="ignore"):
                ou, ov = o.op_apply(xu, xv)
            np.testing.assert_array_equal(yu, ou)
            np.testing.assert_array_equal(yv, ov)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_missing_dirichlet_data_off_the_ice(W, precision):
    print("[gpu] NaN velocities off the ice %s" % precision, flush=True)
    out = []
    for missing in (0.0, np.nan):
        m = iceberg(W, precision)[0]
        gu, gv = m.fields.gu, m.fields.gv
        assert (gu.u_isfixed & ~gu.mask).any() and (gv.v_isfixed & ~gv.mask).any()
        gu.u[~gu.mask] = missing
        gv.v[~gv.mask] = missing
        W.update_geometry(m)
        W.update_velocities(m)
        out.append((m.fields.gu.u[gu.mask], m.fields.gv.v[gv.mask], dict(m.last_report)))
    assert np.isfinite(out[0][0]).all() and np.abs(out[0][0]).max() > 1.0
    np.testing.assert_array_equal(out[1][0], out[0][0])
    np.testing.assert_array_equal(out[1][1], out[0][1])
    assert out[0][2] == out[1][2]


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_context_recovers_from_a_solve_that_ended_in_nan(W, precision):
    """Nothing of a NaN solve stays in the context's work arrays: with its fields
    put back it gives what a new context gives."""
    print("[gpu] solve after a NaN solve, %s" % precision, flush=True)
    out = []
    for spoiled in (False, True):
        m = ragged(W, precision=precision)
        m.solver_params.maxiter_coarse = 60
        if spoiled:
            clean = {(c, a): m._array(c, a).copy(order="F") for c, a, _ in W.model.FIELD_MAP}
            m.fields.gu.u[10, 10] = np.nan
            W.update_geometry(m)
            W.update_velocities(m)
            assert np.isnan(m.fields.gu.u).mean() > 0.5
            for (c, a), v in clean.items():
                setattr(m.params if c == "params" else getattr(m.fields, c), a, v)
        W.update_geometry(m)
        W.update_velocities(m)
        out.append((m.fields.gu.u, m.fields.gv.v, m.last_report))
    np.testing.assert_array_equal(out[1][0], out[0][0])
    np.testing.assert_array_equal(out[1][1], out[0][1])
    assert out[1][2] == out[0][2] and np.isfinite(out[0][0]).all()
