"""All fields at once (wavi_set_fields, wavi_get_fields) against one by one,
below and above the size from which they are copied one by one."""
import ctypes

import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny", [(17, 5), (80, 10), (400, 60)])
def test_fields_at_once_equal_one_by_one(W, nx, ny):
    print("[gpu] fields %dx%d" % (nx, ny), flush=True)
    m = W.workloads.channel_solve(nx=nx, ny=ny, nσ=4, maxiter_picard=1)
    W.update_preconditioner(m)
    rng = np.random.default_rng(nx)
    ref = {}
    for c, a, fid in W.model.FIELD_MAP:
        old = m._array(c, a)
        new = rng.random(old.shape) > 0.5 if old.dtype == np.bool_ else rng.standard_normal(old.shape)
        if a == "u":  # C order, which has to be converted
            new = np.ascontiguousarray(new)
        setattr(m.params if c == "params" else getattr(m.fields, c), a, new)
        ref[fid] = new
    W.push_fields(m)
    lib, ctx = m.parallel_spec._lib, m.parallel_spec.ctx
    for c, a, fid in W.model.FIELD_MAP:
        buf = np.empty(ref[fid].size)
        assert lib.wavi_get_field(ctx, W._lib.FIELD[fid], W._lib.dptr(buf), buf.size) == 0
        np.testing.assert_array_equal(buf.reshape(ref[fid].shape, order="F"), ref[fid].astype(float), err_msg=fid)
    W.pull_fields(m)
    for c, a, fid in W.model.FIELD_MAP:
        got = m._array(c, a)
        assert got is not ref[fid] and got.dtype == ref[fid].dtype
        np.testing.assert_array_equal(got, ref[fid], err_msg=fid)
    ids, size = (ctypes.c_int * 1)(0), (ctypes.c_size_t * 1)(3)
    ptr = (ctypes.c_void_p * 1)(np.empty(3).__array_interface__["data"][0])
    assert lib.wavi_set_fields(ctx, 1, ids, ptr, size) == W._lib.WAVI_EDIM
    assert lib.wavi_get_fields(ctx, 1, (ctypes.c_int * 1)(-1), ptr, size) == W._lib.WAVI_EARG
    assert lib.wavi_set_fields(None, 1, ids, ptr, size) == W._lib.WAVI_EARG
