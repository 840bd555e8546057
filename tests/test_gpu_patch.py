"""The GWCE and momentum passes over patches (k_gwce, k_mom) where the patches
have edges: fewer nodes than one patch, exactly one patch of nodes and one more,
a hub with almost as many neighbours as a row may have (rows past the columns
read ahead), an edge with three elements (rows summed slot by slot), geometry
that the coordinates do not give (kept per patch), and ALPHAL other than 1.
Bit-exact against the oracle."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from adcirc_amd import meshgen
from adcirc_amd.fort14 import Mesh
from gpu_helpers import build_pair, case_setup, compare, log, step_pair

pytestmark = pytest.mark.gpu


def _basin(nx, ny):
    return meshgen.basin(nx=nx, ny=ny, lx=1000.0 * (nx - 1), ly=1000.0 * (ny - 1))


def _beach(nx, ny):
    return meshgen.beach(nx=nx, ny=ny, lx=200.0 * (nx - 1), ly=200.0 * (ny - 1))


def _wheel(spokes):
    """A hub and a rim; the first third of the rim is the open boundary."""
    a = 2.0 * np.pi * np.arange(spokes) / spokes
    x, y = np.append(0.0, 3000.0 * np.cos(a)), np.append(0.0, 3000.0 * np.sin(a))
    rim = np.arange(spokes) + 2
    nm = np.column_stack([np.ones(spokes), rim, np.roll(rim, -1)]).astype(np.int32)
    k = spokes // 3
    land = np.append(rim[k - 1:], rim[0]).astype(np.int32)
    case = _basin(8, 8)
    mesh = Mesh("wheel", x, y, np.full(spokes + 1, 20.0), nm, [rim[:k].astype(np.int32)], [(0, land)])
    emo = np.full((k, 1), 0.5)
    return meshgen.Case(mesh, case.run, emo, np.zeros_like(emo))


def _fin(case):
    """One more element on an interior edge of the middle of the mesh."""
    m = case.mesh
    tri = m.nm[m.nm.shape[0] // 2]
    a, b = int(tri[0]), int(tri[1])
    dx, dy = m.x[b - 1] - m.x[a - 1], m.y[b - 1] - m.y[a - 1]
    x = np.append(m.x, 0.5 * (m.x[a - 1] + m.x[b - 1]) - 0.3 * dy)
    y = np.append(m.y, 0.5 * (m.y[a - 1] + m.y[b - 1]) + 0.3 * dx)
    nm = np.vstack([m.nm, [[a, b, x.shape[0]]]]).astype(np.int32)
    mesh = dataclasses.replace(m, x=x, y=y, dp=np.append(m.dp, 20.0), nm=nm)
    return dataclasses.replace(case, mesh=mesh)


def _off(d):
    """Areas one unit in the last place off: not what the coordinates give."""
    d["areas"] = np.nextafter(d["areas"], np.inf)


CASES = {
    "12 nodes": (lambda: _basin(4, 3), None),
    "96 nodes": (lambda: _basin(12, 8), None),
    "97 to 99 nodes": (lambda: _basin(11, 9), None),
    "wheel of 28 spokes": (lambda: _wheel(28), None),
    "three elements on an edge": (lambda: _fin(_basin(20, 12)), None),
    "stored geometry": (lambda: _basin(40, 23), _off),
    "stored geometry, wet/dry": (lambda: _beach(41, 21), _off),
    "wet/dry, 67 x 31": (lambda: _beach(67, 31), None),
}


@pytest.mark.parametrize("name", list(CASES))
def test_edges_bitexact(name):
    make, edit = CASES[name]
    case = make()
    d = case_setup(case)
    if edit:
        edit(d)
    g, o = build_pair(d, case.run)
    log(f"case {name}: {int(d['np'])} nodes, 15 steps bit-exact")
    for it in range(1, 16):
        step_pair(g, o, it)
        bad = compare(g, o, it)
        assert not bad, f"step {it}: " + "; ".join(bad)
    g.close()


@pytest.mark.parametrize("lumped", [False, True])
def test_alphal_from_the_host(lumped):
    """ALPHAL other than 1 at some elements: the matrix, the right-hand side and
    the momentum pass take it."""
    case = _basin(30, 17)
    run = dataclasses.replace(case.run, ilump=1, dtdp=0.5) if lumped else case.run
    d = case_setup(case)
    g, o = build_pair(d, run)
    al = np.ones(int(d["ne"]))
    al[::7] = 0.75
    g.set("alphal", al)
    p = o.lib.adco_array(o.h, b"alphal")
    np.ctypeslib.as_array(p, (al.size,))[:] = al
    log(f"ALPHAL 0.75 at every seventh element, lumped {lumped}: 10 steps bit-exact")
    for it in range(1, 11):
        step_pair(g, o, it)
        bad = compare(g, o, it)
        assert not bad, f"step {it}: " + "; ".join(bad)
    g.close()


@pytest.mark.parametrize("shape", [(60, 40), (200, 160), (620, 230)])
def test_many_wetting_candidates_bitexact(shape):
    """Shallow water over a rough bed, wet and dry all over: thousands of wetting
    candidates a step, in one block of the ordered friction updates and in many,
    and in more than one list of element tiles (over 262,144 elements)."""
    from adcirc_amd.model import cold_wetdry_state
    case = _beach(*shape)
    rng = np.random.default_rng(7)
    m = case.mesh
    dp = 0.15 + 0.25 * rng.standard_normal(m.x.shape[0])
    case = dataclasses.replace(case, mesh=dataclasses.replace(m, dp=dp),
                               run=dataclasses.replace(case.run, dtdp=0.5))
    d = case_setup(case)
    eta = 0.3 * np.sin(m.x / 700.0) * np.cos(m.y / 900.0)
    e2, nc, nf = cold_wetdry_state(d, case.run, eta)
    d["eta2_0"], d["nodecode0"], d["noff0"] = e2, nc, nf
    g, o = build_pair(d, case.run)
    log(f"rough bed {int(d['np'])} nodes, {int((nc == 0).sum())} dry: 6 steps bit-exact")
    for it in range(1, 7):
        step_pair(g, o, it)
        bad = compare(g, o, it)
        assert not bad, f"step {it}: " + "; ".join(bad)
    g.close()
