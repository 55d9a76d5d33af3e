"""Which form the coarse CG takes (wavi_coarse_cg_runs), and that its result is
that of the launches per iteration, bit for bit."""
import ctypes

import numpy as np
import pytest


def runs(W, m):
    """(launches, resident, workgroup, gave up) so far"""
    got = (ctypes.c_int64 * W._lib.WAVI_CG_RAN_COUNT)()
    assert m.parallel_spec._lib.wavi_coarse_cg_runs(m.parallel_spec.ctx, got) == 0
    return tuple(got)


def model(W, nx, ny, precision, maxiter_coarse=40, maxiter_picard=3, mode=None, seed=2):
    m = W.workloads.channel_solve(nx=nx, ny=ny, nσ=4, maxiter_picard=maxiter_picard, precision=precision, seed=seed)
    m.solver_params.maxiter_coarse = maxiter_coarse
    W.update_geometry(m)
    if mode is not None:
        set_mode(m, mode)
    return m


def set_mode(m, mode):
    assert m.parallel_spec._lib.wavi_set_coarse_cg(m.parallel_spec.ctx, mode) == 0


def assert_same(m, ref):
    np.testing.assert_array_equal(m.fields.gu.u, ref.fields.gu.u)
    np.testing.assert_array_equal(m.fields.gv.v, ref.fields.gv.v)
    assert m.last_report == ref.last_report


# tiles: 6, 33, 246, 256, 260, 441, 504, 512, 891; resident up to 504 (FP64) and 256 (mixed)
@pytest.mark.gpu
@pytest.mark.parametrize("precision,most", [("fp64", 504), ("mixed", 256)])
@pytest.mark.parametrize("nx,ny,tiles", [(80, 10, 6), (527, 12, 33), (640, 80, 246), (255, 255, 256), (1039, 63, 260),
                                         (1007, 111, 441), (1007, 120, 504), (1023, 127, 512), (1280, 160, 891)])
def test_form_by_the_number_of_tiles(W, nx, ny, tiles, precision, most):
    print("[gpu] form of the coarse CG %s %dx%d" % (precision, nx, ny), flush=True)
    m = model(W, nx, ny, precision)
    W.update_velocities(m)
    n = m.last_report["picard_iters"] - m.last_report["converged"]
    assert n > 0 and runs(W, m) == ((0, n, 0, 0) if tiles <= most else (n, 0, 0, 0))
    ref = model(W, nx, ny, precision, mode=W._lib.WAVI_CG_LAUNCHES)
    W.update_velocities(ref)
    assert runs(W, ref) == (n, 0, 0, 0)
    assert_same(m, ref)
    set_mode(ref, W._lib.WAVI_CG_WORKGROUP)
    if tiles == 6:
        W.update_velocities(ref)
        assert runs(W, ref)[2] > 0


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_form_when_waits_run_out(W, monkeypatch, precision):
    print("[gpu] form without polls %s" % precision, flush=True)
    monkeypatch.setenv("WAVI_CG_POLLS", "0")
    m = model(W, 250, 62, precision)
    W.update_velocities(m)
    n = m.last_report["picard_iters"] - m.last_report["converged"]
    assert n > 1 and runs(W, m) == (n - 1, 0, 0, 1)


@pytest.mark.gpu
def test_form_in_a_gradient(W):
    print("[gpu] form in a gradient", flush=True)
    m = W.workloads.inversion_model(W.workloads.inversion_logc_true(64, 16, seed=4), "fp64", nσ=4, n_picard=2)
    W.update_geometry(m)
    rng = np.random.default_rng(1)
    W.misfit_gradient(m, 2, 100 * rng.random(m.grid.xxu.shape), 10 * rng.random(m.grid.yyv.shape))
    got = runs(W, m)
    assert got[1] > 4 and got == (0, got[1], 0, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("polls", [None, "0"])
def test_form_in_a_lockstep_batch(W, monkeypatch, polls):
    """Every member resident, or every member's first CG started over; with one
    member by launches, all are."""
    print("[gpu] forms in a batch, polls %s" % polls, flush=True)
    if polls is not None:
        monkeypatch.setenv("WAVI_CG_POLLS", polls)
    ms = [model(W, a, b, "mixed") for a, b in ((80, 10), (160, 20), (77, 35), (511, 15))]
    W.update_velocities_batch(ms, lockstep=True)
    for m in ms:
        n = m.last_report["picard_iters"] - m.last_report["converged"]
        assert n > 1 and runs(W, m) == ((0, n, 0, 0) if polls is None else (n - 1, 0, 0, 1))
    if polls is None:
        before = [runs(W, m) for m in ms]
        set_mode(ms[1], W._lib.WAVI_CG_LAUNCHES)
        for m in ms:
            m.fields.gu.u[...] = 0.0
            m.fields.gv.v[...] = 0.0
        W.update_velocities_batch(ms, lockstep=True)
        for m, b in zip(ms, before):
            assert runs(W, m)[1:] == b[1:] and runs(W, m)[0] > b[0]


def set_waits(m, polls=-1, tag=0):
    return m.parallel_spec._lib.wavi_set_coarse_cg_waits(m.parallel_spec.ctx, polls, tag)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nx,ny", [(80, 10), (250, 62)])
@pytest.mark.parametrize("maxiter_coarse", [1, 40])
def test_tags_that_run_out(W, nx, ny, precision, maxiter_coarse):
    """The words of the first call hold the first tags (1 with one iteration);
    in the second call the tags run out and those come again, which is right only
    if the words were cleared."""
    print("[gpu] tags run out %s %dx%d, %d iterations" % (precision, nx, ny, maxiter_coarse), flush=True)
    m, ref = (model(W, nx, ny, precision, maxiter_coarse=maxiter_coarse, maxiter_picard=1, mode=mode)
              for mode in (None, W._lib.WAVI_CG_LAUNCHES))
    for tag in (0, 2 ** 32 - 2 * (maxiter_coarse + 2), 0, 0, 0):
        assert set_waits(m, tag=tag) == 0
        for x in (m, ref):
            W.update_velocities(x)
        assert_same(m, ref)
    assert runs(W, m) == (0, 5, 0, 0)
    assert set_waits(m, tag=1) == W._lib.WAVI_EARG
    assert set_waits(m, polls=2 ** 21 + 1) == W._lib.WAVI_EARG


@pytest.mark.gpu
def test_tags_that_run_out_in_a_batch(W):
    print("[gpu] tags run out in a batch", flush=True)
    sizes = ((80, 10), (160, 20), (77, 35))
    ms = [model(W, a, b, "mixed", maxiter_coarse=1, maxiter_picard=1) for a, b in sizes]
    refs = [model(W, a, b, "mixed", maxiter_coarse=1, maxiter_picard=1, mode=W._lib.WAVI_CG_LAUNCHES) for a, b in sizes]
    for tag in (0, 2 ** 32 - 6, 0, 0, 0):
        assert set_waits(ms[1], tag=tag) == 0
        W.update_velocities_batch(ms, lockstep=True)
        for m, ref in zip(ms, refs):
            W.update_velocities(ref)
            assert_same(m, ref)
    assert all(runs(W, m) == (0, 5, 0, 0) for m in ms)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_resident_again_after_a_lost_wait(W, precision):
    """256 CGs by launches after a loss, 512 after a second one in a row; then the
    waits are polled again and the form is resident for good."""
    print("[gpu] resident again after a lost wait, %s" % precision, flush=True)
    m, ref = (model(W, 80, 10, precision, maxiter_coarse=4, maxiter_picard=1, mode=mode)
              for mode in (None, W._lib.WAVI_CG_LAUNCHES))
    rng = np.random.default_rng(0)
    ru, rv = rng.standard_normal(m.fields.gu.u.shape), rng.standard_normal(m.fields.gv.v.shape)

    def vcycles(n):
        for _ in range(n):
            got, want = W.vcycle(m, ru, rv), W.vcycle(ref, ru, rv)
        for a, b in zip(got, want):
            np.testing.assert_array_equal(a, b)
        return runs(W, m)

    assert vcycles(1) == (0, 1, 0, 0)
    assert set_waits(m, polls=0) == 0
    assert vcycles(1) == (0, 1, 0, 1)
    assert vcycles(256) == (256, 1, 0, 1)
    assert vcycles(1) == (256, 1, 0, 2)
    assert set_waits(m, polls=2 ** 21) == 0
    assert vcycles(512) == (768, 1, 0, 2)
    assert vcycles(300) == (768, 301, 0, 2)
    assert set_waits(m, polls=0) == 0
    assert vcycles(1) == (768, 301, 0, 3)
    assert vcycles(257) == (1024, 301, 0, 4)


@pytest.mark.gpu
@pytest.mark.parametrize("precision,timer,lockstep", [("fp64", "cg_iter_fp64", False), ("mixed", "cg_iter_mixed", False),
                                                      ("mixed", "cg_iter_mixed", True)])
def test_launches_know_the_length_of_a_resident_cg(W, precision, timer, lockstep):
    """After a CG of 40 iterations the launches are queued in a first chunk of 32,
    which is timed whole; without its length they begin with chunks of 2, 4, 8, 16."""
    print("[gpu] launches after a resident CG, %s, lockstep %s" % (precision, lockstep), flush=True)
    m = model(W, 80, 10, precision, maxiter_coarse=40, maxiter_picard=1)
    lib, ctx = m.parallel_spec._lib, m.parallel_spec.ctx
    if lockstep:
        W.update_velocities_batch([m], lockstep=True)
    else:
        W.update_velocities(m)
    assert m.last_report["coarse_cg_iters"] == [40] and runs(W, m) == (0, 1, 0, 0)
    set_mode(m, W._lib.WAVI_CG_LAUNCHES)
    assert lib.wavi_profile_enable(ctx, 1) == 0
    W.update_velocities(m)
    ms, n = ctypes.c_double(), ctypes.c_int64()
    assert lib.wavi_profile_read(ctx, W._lib.KT[timer], ctypes.byref(ms), ctypes.byref(n)) == 0
    assert lib.wavi_profile_enable(ctx, 0) == 0
    assert m.last_report["coarse_cg_iters"] == [40] and runs(W, m) == (1, 1, 0, 0)
    assert n.value == 32 and ms.value > 0.0
