"""The register-resident JCG (k_jcg_reg) where its layout has edges: systems
that end at, one past and inside a 2048-row chunk or a two-chunk tile, one and
two chunks per block, rows with more entries than the register slots (kept in
LDS), and a random numbering (every block's window is the whole system).
Bit-exact against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from adcirc_amd import meshgen
from adcirc_amd.fort14 import Mesh
from gpu_helpers import build_pair, case_setup, compare, log, step_pair

pytestmark = pytest.mark.gpu


def _basin(nx, ny):
    return meshgen.basin(nx=nx, ny=ny, lx=1000.0 * (nx - 1), ly=1000.0 * (ny - 1))


def _scattered(n, seed=5, shuffle=False):
    """Delaunay mesh of random points (up to a dozen neighbours a node) in a
    basin of n-node size, numbered west to east or at random."""
    from scipy.spatial import Delaunay
    rng = np.random.default_rng(seed)
    side = int(np.sqrt(n))
    edge = np.linspace(0.0, 1000.0 * side, side)
    ring = [np.column_stack([edge, 0 * edge]), np.column_stack([edge, 0 * edge + edge[-1]]),
            np.column_stack([0 * edge, edge])[1:-1],
            np.column_stack([0 * edge + edge[-1], edge])[1:-1]]
    inner = rng.uniform(300.0, edge[-1] - 300.0, (n - 4 * side + 4, 2))
    p = np.concatenate(ring + [inner])
    p = p[rng.permutation(p.shape[0]) if shuffle else np.lexsort((p[:, 1], p[:, 0]))]
    nm = Delaunay(p).simplices.astype(np.int64)
    a = ((p[nm[:, 1], 0] - p[nm[:, 0], 0]) * (p[nm[:, 2], 1] - p[nm[:, 0], 1])
         - (p[nm[:, 2], 0] - p[nm[:, 0], 0]) * (p[nm[:, 1], 1] - p[nm[:, 0], 1]))
    nm[a < 0] = nm[a < 0][:, [0, 2, 1]]
    nm = nm[np.abs(a) > 1.0]
    on = lambda c, v: np.flatnonzero(np.abs(p[:, c] - v) < 1e-6)  # noqa: E731
    east, west, south, north = on(0, edge[-1]), on(0, 0.0), on(1, 0.0), on(1, edge[-1])
    op = east[np.argsort(p[east, 1])] + 1
    land = np.concatenate([north[np.argsort(-p[north, 0])], west[np.argsort(-p[west, 1])][1:-1],
                           south[np.argsort(p[south, 0])]]) + 1
    case = _basin(8, 8)
    mesh = Mesh("scattered", p[:, 0], p[:, 1], np.full(p.shape[0], 30.0),
                (nm + 1).astype(np.int32), [op.astype(np.int32)], [(0, land.astype(np.int32))])
    emo = np.full((op.shape[0], 1), 0.5)
    return meshgen.Case(mesh, case.run, emo, np.zeros_like(emo))


CASES = {
    "2048 rows": (lambda: _basin(64, 32), 0),
    "2049 rows": (lambda: _basin(683, 3), 0),
    "4096 rows, two chunks a block": (lambda: _basin(128, 32), 2),
    "4097 rows, two chunks a block": (lambda: _basin(241, 17), 3),
    "6200 rows, two chunks a block": (lambda: _basin(124, 50), 3),
    "9000 rows, up to a dozen neighbours": (lambda: _scattered(9000), 0),
    "9000 rows, the same, two chunks a block": (lambda: _scattered(9000), 4),
    "9000 rows at random": (lambda: _scattered(9000, shuffle=True), 0),
}


@pytest.mark.parametrize("name", list(CASES))
def test_edges_bitexact(name):
    make, blocks = CASES[name]
    case = make()
    d = case_setup(case)
    g, o = build_pair(d, case.run)
    if blocks:
        g.set_jcg_blocks(blocks)
    log(f"case {name}: {int(d['np'])} nodes, {g.jcg_shape()} JCG shape; 12 steps bit-exact")
    for it in range(1, 13):
        step_pair(g, o, it)
        bad = compare(g, o, it)
        assert not bad, f"step {it}: " + "; ".join(bad)
    g.close()
