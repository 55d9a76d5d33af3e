"""The +-1 Haar transforms by lines (haar_line_P, haar_line_R) and the
wavefront tree sums, against the oracle.  Both keep the oracle's order of
additions, so the bar is equality (of values: the sign of a zero may differ)."""
import numpy as np
import pytest

from helpers import channel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("levels", [0, 1, 2, 3])
@pytest.mark.parametrize("nx,ny", [(24, 10), (17, 15), (31, 18), (33, 16), (47, 33)])
def test_haar_lines_every_level_and_partial_block(W, oracle, levels, nx, ny):
    """Both components and directions on grids whose last blocks hold 1, 2,
    15, 16 and other counts of points in x and y."""
    print("[gpu] haar lines levels %d %dx%d" % (levels, nx, ny), flush=True)
    m = channel(W, nx=nx, ny=ny)
    m.solver_params.levels = levels
    W.update_preconditioner(m)
    o = oracle.OracleModel(m)
    rng = np.random.default_rng(levels)
    for comp, shape in (("u", (nx + 1, ny)), ("v", (nx, ny + 1))):
        x = rng.standard_normal(shape) * 10.0 ** rng.uniform(-8, 8, shape)
        for d in ("inverse", "inverse_t"):
            assert np.array_equal(W.haar(m, comp, d, x), o.haar(comp, d, x)), (comp, d)
