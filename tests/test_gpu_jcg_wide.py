"""The solver kernels for matrices that the register-resident solve cannot hold:
k_jcg and k_jcg_batch, each with one and two starts.  A mesh numbered at random
(every row block references all rows: the products gather from memory) and a mesh
of overlapping layers (twelve neighbours a node, a bandwidth of 5,002: the
pseudo-residual is staged in LDS).  Alone bit-exact against the oracle, in a batch
bit for bit the member's own run."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from adcirc_amd import _lib, meshgen
from adcirc_amd.fort14 import Mesh
from adcirc_amd.model import Batch
from gpu_helpers import build_pair, case_setup, compare, log, step_pair

pytestmark = pytest.mark.gpu

REG_LDS_DOUBLES = 152 * 1024 // 8  # what the register-resident solve may keep per block
STAGED_BANDWIDTH = 5632            # the widest whose pseudo-residual is staged


def _random():
    """The basin of 22,500 nodes, numbered at random."""
    case = meshgen.basin(nx=150, ny=150, lx=149.0e3, ly=149.0e3)
    m = case.mesh
    order = np.random.default_rng(5).permutation(m.x.shape[0])
    inv = np.empty_like(order)
    inv[order] = np.arange(order.shape[0])
    ren = lambda ids: (inv[np.asarray(ids, np.int64) - 1] + 1).astype(np.int32)  # noqa: E731
    mesh = dataclasses.replace(m, x=m.x[order], y=m.y[order], dp=m.dp[order], nm=ren(m.nm),
                               open_bnd=[ren(s) for s in m.open_bnd],
                               land_bnd=[(ib, ren(s)) for ib, s in m.land_bnd])
    return dataclasses.replace(case, mesh=mesh)


def _layers(nx=5, ny=5000):
    """Three layers of triangles over the same grid, numbered along its long side:
    neighbours (0,1), (1,0), (1,1), (0,2), (1,-1), (1,2) and their opposites."""
    i, j = np.meshgrid(np.arange(nx), np.arange(ny), indexing="ij")
    node = lambda a, b: (a * ny + b + 1).ravel()  # noqa: E731
    a, b = i[:-1, :-1], j[:-1, :-1]
    nm = [np.column_stack([node(a, b), node(a + 1, b), node(a + 1, b + 1)]),
          np.column_stack([node(a, b), node(a + 1, b + 1), node(a, b + 1)])]
    a, b = i[:-1, :-2], j[:-1, :-2]
    nm.append(np.column_stack([node(a, b), node(a + 1, b + 1), node(a, b + 2)]))
    nm.append(np.column_stack([node(a, b), node(a + 1, b + 2), node(a, b + 1)]))
    x, y = 1000.0 * i.ravel(), 1000.0 * j.ravel()
    left, right = node(0 * j[0], j[0]), node(0 * j[0] + nx - 1, j[0])
    bottom, top = node(i[:, 0], 0 * i[:, 0]), node(i[:, 0], 0 * i[:, 0] + ny - 1)
    op = bottom.astype(np.int32)
    land = np.concatenate([right, top[::-1][1:-1], left[::-1]]).astype(np.int32)
    case = meshgen.basin(nx=8, ny=8)
    mesh = Mesh("layers", x, y, np.full(x.shape[0], 20.0), np.vstack(nm).astype(np.int32), [op],
                [(0, land)])
    emo = np.full((op.shape[0], 1), 0.5)
    return meshgen.Case(mesh, case.run, emo, np.zeros_like(emo))


def _shape(d):
    """(bandwidth, the fewest LDS doubles that some 2048-row block of the
    register-resident solve needs for its window and its entries past eight)."""
    n, w = int(d["np"]), int(d["mnei"])
    nei = np.asarray(d["neitab"], np.int64).reshape(w, n) - 1
    row = np.broadcast_to(np.arange(n), nei.shape)
    col = np.where(nei >= 0, nei, row)
    over = np.maximum((nei >= 0).sum(0) - 1 - 8, 0)
    need = 0
    for c in range(0, n, 2048):
        e = min(n, c + 2048)
        lo, hi = min(c, col[:, c:e].min()), max(e, col[:, c:e].max() + 1)
        need = max(need, (c - lo) + 2048 + (hi - e) + 1 + 1.25 * over[c:e].sum())
    return int(np.abs(col - row).max()), need


MESHES = {"random numbering": _random, "overlapping layers": _layers}


@pytest.fixture(scope="module", params=list(MESHES))
def setup(request):
    case = MESHES[request.param]()
    d = case_setup(case)
    bw, need = _shape(d)
    assert need > REG_LDS_DOUBLES
    assert (bw <= STAGED_BANDWIDTH) == (request.param == "overlapping layers")
    log(f"{request.param}: {int(d['np'])} nodes, bandwidth {bw}, MNEI {int(d['mnei'])}")
    return case, d


@pytest.mark.parametrize("warm", [0, 2])
def test_alone_bitexact(setup, warm):
    """The learned start untrained: its correction is zero, the start the same."""
    case, d = setup
    run = dataclasses.replace(case.run, warm_start=warm)
    g, o = build_pair(d, run)
    for it in range(1, 9):
        step_pair(g, o, it)
        bad = compare(g, o, it)
        assert not bad, f"step {it}: " + "; ".join(bad)
    g.close()


@pytest.mark.parametrize("warm", [0, 2])
def test_batch_members_equal_their_own_runs(setup, warm):
    case, d = setup
    run = dataclasses.replace(case.run, warm_start=warm)
    params = (0.05 * np.random.default_rng(5).standard_normal(_lib.ML_NPARAM)).astype(np.float32)
    models = []
    for k in range(4):  # two members, and their own runs
        g, _ = build_pair(d, run)
        eta = g.get("eta2") + 0.1 * (1 + k % 2) * np.cos(np.asarray(d["y"]) / 40.0e3)
        g.cold_start(eta, d["nodecode0"], d["noff0"])
        if warm == 2:
            g.ml_params(params)
        models.append(g)
    b = Batch(models[:2])
    b.run(1, 25)
    b.close()
    for x, y in zip(models[:2], models[2:]):
        y.run_resident(1, 25)
        for f in ("eta1", "eta2", "etas", "uu2", "vv2", "tk", "etamax", "coef"):
            u, v = x.get(f), y.get(f)
            assert np.array_equal(u, v), (f, int((u != v).sum()))
        assert x.run_stats() == y.run_stats()
    assert not np.array_equal(models[0].get("eta2"), models[1].get("eta2"))
    for g in models:
        g.close()
