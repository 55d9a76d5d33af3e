"""The resident coarse CG where others hold room on the chip: launches per
iteration, the same bits, and the resident form again once there is room."""
import ctypes

import pytest

import room
from test_gpu_cg_forms import assert_same, model, runs

UNITS = 256 * 64  # CUs, units of a CU


def _bus(lib):
    buf = ctypes.create_string_buffer(64)
    assert lib.hipDeviceGetPCIBusId(buf, 64, 0) == 0
    return buf.value.decode()


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_room_held_by_another_process(W, tmp_path, precision):
    print("[gpu] room held by another process, %s" % precision, flush=True)
    m = model(W, 250, 62, precision, maxiter_picard=2)
    ref = model(W, 250, 62, precision, maxiter_picard=2, mode=W._lib.WAVI_CG_LAUNCHES)
    exe, bus = room.build(tmp_path), _bus(m.parallel_spec._lib)

    def solve():
        before = runs(W, m)
        for x in (m, ref):
            W.update_velocities(x)
        assert_same(m, ref)
        n = m.last_report["picard_iters"] - m.last_report["converged"]
        assert n > 0
        got = tuple(a - b for a, b in zip(runs(W, m), before))
        assert got in ((n, 0, 0, 0), (0, n, 0, 0))
        return "resident" if got[1] else "launches"

    assert solve() == "resident"
    for kill in (False, True):
        h = room.Holder(exe, bus, UNITS)
        assert h.take(UNITS // 2 + 1)
        assert solve() == "launches"
        h.give(UNITS // 2 + 1)
        assert h.take(UNITS // 8) and solve() == "resident"
        h.end(kill)
        assert solve() == "resident"


@pytest.mark.gpu
def test_members_that_do_not_fit_together(W):
    """FP64 members of 441 tiles on four threads: one of them may be resident."""
    print("[gpu] FP64 members of 441 tiles on four threads", flush=True)
    kw = dict(maxiter_coarse=300, maxiter_picard=6)
    ms = [model(W, 1007, 111, "fp64", seed=k, **kw) for k in range(4)]
    W.update_velocities_batch(ms, nthreads=4)
    total = [sum(c) for c in zip(*(runs(W, m) for m in ms))]
    assert total[0] > 0 and total[1] > 0 and total[2:] == [0, 0]
    for k, m in enumerate(ms):
        ref = model(W, 1007, 111, "fp64", seed=k, mode=W._lib.WAVI_CG_LAUNCHES, **kw)
        W.update_velocities(ref)
        assert_same(m, ref)
