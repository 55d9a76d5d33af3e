"""The coarse CG in one launch of resident workgroups: the same bits and
the same iteration counts as the launches per iteration, on
both sides of the tile counts where the folding of its sums (32 tiles) and its
form (one launch or launches per iteration) change, for every Haar level, and
where its waits run out at once and the CG runs again in one workgroup."""
import numpy as np
import pytest


def _mode(W, m, resident):
    spec = m.parallel_spec
    assert spec._lib.wavi_set_coarse_cg(spec.ctx, W._lib.WAVI_CG_AUTO if resident else W._lib.WAVI_CG_LAUNCHES) == 0


def _solve(W, monkeypatch, nx, ny, levels=3, resident=True, polls=None, maxiter_coarse=40, calls=2, **kw):
    if polls is not None:
        monkeypatch.setenv("WAVI_CG_POLLS", str(polls))
    m = W.workloads.channel_solve(nx=nx, ny=ny, nσ=4, maxiter_picard=3, **kw)
    m.solver_params.levels = levels
    m.solver_params.maxiter_coarse = maxiter_coarse
    out = []
    for _ in range(calls):
        W.update_geometry(m)
        _mode(W, m, resident)
        W.update_velocities(m)
        out.append((m.fields.gu.u.copy(), m.fields.gv.v.copy(), dict(m.last_report)))
    monkeypatch.delenv("WAVI_CG_POLLS", raising=False)
    return out


def _equal(a, b):
    for (u, v, r), (x, y, q) in zip(a, b):
        np.testing.assert_array_equal(u, x)
        np.testing.assert_array_equal(v, y)
        assert r == q


# 6 tiles; 31, 32 and 33 tiles in a row; 11 x 3; 246; 441 and 504 (two per CU); 512 and 891 (the launches)
@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nx,ny", [(80, 10), (495, 14), (511, 15), (527, 12), (161, 33), (640, 80), (1007, 111), (1007, 120),
                                   (1023, 127), (1280, 160)])
def test_resident_cg_equals_the_launches(W, monkeypatch, nx, ny, precision):
    print("[gpu] resident CG %s %dx%d" % (precision, nx, ny), flush=True)
    _equal(_solve(W, monkeypatch, nx, ny, precision=precision),
           _solve(W, monkeypatch, nx, ny, precision=precision, resident=False))


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny", [(77, 35), (250, 62)])
@pytest.mark.parametrize("levels", [0, 1, 2])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_resident_cg_at_every_level(W, monkeypatch, nx, ny, levels, precision):
    print("[gpu] resident CG %s %dx%d levels %d" % (precision, nx, ny, levels), flush=True)
    _equal(_solve(W, monkeypatch, nx, ny, levels, precision=precision),
           _solve(W, monkeypatch, nx, ny, levels, precision=precision, resident=False))


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny", [(80, 10), (250, 62)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_waits_that_run_out_start_the_cg_over(W, monkeypatch, nx, ny, precision):
    """polls = 0: the first poll that does not find its words ends the launch;
    the CG then runs in one workgroup from the same start, and the context
    takes the launches per iteration from then on."""
    print("[gpu] resident CG without polls %s %dx%d" % (precision, nx, ny), flush=True)
    _equal(_solve(W, monkeypatch, nx, ny, polls=0, precision=precision),
           _solve(W, monkeypatch, nx, ny, precision=precision, resident=False))


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny", [(64, 16), (250, 62)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_resident_cg_in_the_adjoint(W, nx, ny, precision):
    """The Jacobi-preconditioned form, inside the linear solves."""
    print("[gpu] resident CG in the adjoint %s %dx%d" % (precision, nx, ny), flush=True)
    res = []
    for on in (True, False):
        logc = W.workloads.inversion_logc_true(nx, ny, seed=4)
        m = W.workloads.inversion_model(logc, precision, nσ=4, n_picard=2)
        W.update_geometry(m)
        _mode(W, m, on)
        g = m.grid
        rng = np.random.default_rng(1)
        J, grad, rep = W.misfit_gradient(m, 2, 100 * rng.random(g.xxu.shape), 10 * rng.random(g.yyv.shape))
        res.append((J, grad, rep))
    assert res[0][0] == res[1][0]
    np.testing.assert_array_equal(res[0][1], res[1][1])
    assert res[0][2] == res[1][2]


@pytest.mark.gpu
@pytest.mark.parametrize("polls", [None, 0])
def test_resident_batch_equals_the_launches(W, monkeypatch, polls):
    """Members of different sizes in one launch, each against its own solve by
    launches; polls = 0: all of them start over in one workgroup."""
    print("[gpu] resident batch, polls %s" % polls, flush=True)
    if polls is not None:
        monkeypatch.setenv("WAVI_CG_POLLS", str(polls))
    sizes = [(80, 10), (160, 20), (77, 35), (511, 15)]
    ms = [W.workloads.channel_solve(nx=a, ny=b, nσ=4, maxiter_picard=3, precision="mixed") for a, b in sizes]
    for m in ms:
        m.solver_params.maxiter_coarse = 40
        W.update_geometry(m)
    W.update_velocities_batch(ms, lockstep=True)
    for m, (a, b) in zip(ms, sizes):
        got = [(m.fields.gu.u, m.fields.gv.v, dict(m.last_report))]
        _equal(got, _solve(W, monkeypatch, a, b, precision="mixed", resident=False, calls=1))
