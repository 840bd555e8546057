"""The wait bound (adcgpu_set_wait_limit) is each wait's own: a solve of many
short waits, several times longer than the bound in all, ends with the
oracle's result, one and two chunks a block."""
from __future__ import annotations

import dataclasses

import pytest

from adcirc_amd import meshgen
from adcirc_amd.model import set_wait_limit
from gpu_helpers import build_pair, case_setup, compare, log, step_pair

pytestmark = pytest.mark.gpu

# 170 iterations and more take 1.1 ms, a wait some 10 us.
LIMIT = 0.3e-3


@pytest.mark.parametrize("blocks", [0, 3])
def test_long_solve_of_short_waits(blocks):
    case = meshgen.basin(nx=124, ny=50, lx=123.0e3, ly=49.0e3)
    # a step so long that the matrix is nearly the stiffness matrix, and a tolerance at
    # rounding level: some 180 iterations
    run = dataclasses.replace(case.run, itmax=256, convcr=1.0e-30, dtdp=600.0)
    d = case_setup(case)
    g, o = build_pair(d, run)
    if blocks:
        g.set_jcg_blocks(blocks)
    log(f"basin {int(d['np'])} nodes, {blocks or 'all'} blocks, every wait bounded by "
        f"{1e3 * LIMIT} ms: 3 steps bit-exact")
    set_wait_limit(LIMIT)
    try:
        for it in range(1, 4):
            step_pair(g, o, it)
            bad = compare(g, o, it)
            assert not bad, f"step {it}: " + "; ".join(bad)
    finally:
        set_wait_limit(0.5)
    n, _ = g.numitr()
    log(f"last solve {n} iterations")
    assert n >= 170
    g.close()
