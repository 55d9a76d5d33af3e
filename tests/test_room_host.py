"""The account of the room that waiting launches take of a GPU, among processes
(wavi_room.h; no GPU needed)."""
import os

import pytest

import room


@pytest.fixture
def holders(tmp_path):
    exe = room.build(tmp_path)
    bus = "test:%d" % os.getpid()
    made = []

    def make(name=bus):
        made.append(room.Holder(exe, name, 1000))
        return made[-1]
    yield make
    for h in made:
        if h.p.poll() is None:
            h.end()
    path = "/dev/shm/wavi_hip_room1.%d.%s" % (os.geteuid(), bus.replace(":", "-"))
    if os.path.exists(path):
        os.unlink(path)


def test_alone_all_of_the_chip_beside_another_half(holders):
    a, b = holders(), holders()
    assert a.take(1000) and not a.take(1) and not b.take(1)
    a.give(1000)
    assert b.take(300) and a.take(200) and not a.take(1) and not b.take(1)
    b.give(300)
    assert a.take(300) and not a.take(1)
    a.give(500)
    assert b.take(501) and not a.take(1)


@pytest.mark.parametrize("kill", [False, True])
def test_what_an_ended_process_held_is_free(holders, kill):
    a, b = holders(), holders()
    assert a.take(1000) and not b.take(1)
    a.end(kill)
    assert b.take(1000)
    c = holders()  # on the line of the ended one
    assert not c.take(1)
    b.give(1000)
    assert c.take(1000)


def test_no_line_no_room(holders):
    hs = [holders() for _ in range(65)]
    assert all(h.take(1) for h in hs[:64]) and not hs[64].take(1)
    hs[10].end()
    late = holders()
    assert late.take(1) and not hs[64].take(1)


def test_own_account_without_shared_memory(holders):
    a, b = holders("x" * 300), holders("x" * 300)  # too long a name
    assert a.take(1000) and b.take(1000) and not a.take(1)
    a.give(1000)
    assert a.take(400) and a.take(100) and not a.take(1)
