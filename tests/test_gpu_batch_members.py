"""Batches whose members differ: what goes out in one launch per pass (the common
wet/dry members, alike in precision and forcing) beside members that take their
passes one by one.  Every member ends bit for bit where its own resident run
ends."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from adcirc_amd import _lib, meshgen
from conftest import load_golden
from gpu_helpers import case_setup, golden_tables, log

pytestmark = pytest.mark.gpu

FIELDS = ("eta1", "eta2", "etas", "uu2", "vv2", "qx2", "qy2", "h1", "h2", "tk", "etamax", "umax",
          "coef", "alphal", "totalarea", "nodecode", "noff", "mju", "etamax_it", "umax_it")


class _Spec:
    def __init__(self, what, d, run, holland=None, precision=_lib.FP64, params=None):
        self.what, self.d, self.run, self.holland = what, d, run, holland
        self.precision, self.params = precision, params

    def model(self):
        from adcirc_amd.model import Model
        d, run = self.d, self.run
        t = golden_tables(d)
        nb = run.nbfr
        g = Model(t, run, tau0var=d["tau0var"], evm=d["evm"], fric=d["fric"],
                  corif=np.full(t["np"], run.cori), emo=np.asarray(d["emo"]).reshape(t["neta"], nb),
                  efa=np.asarray(d["efa"]).reshape(t["neta"], nb), precision=self.precision,
                  qnam=d.get("qnam"), qnph=d.get("qnph"))
        g.cold_start(d["eta2_0"], d["nodecode0"], d["noff0"])
        if self.params is not None:
            g.ml_params(self.params)
        if self.holland is not None:
            g.holland(0.0, self.holland)
        return g


@pytest.fixture(scope="module")
def coastal():
    case = meshgen.coastal(6000)
    d = case_setup(case)
    storms = meshgen.storm_ensemble(case, 6, seed=3)

    def spec(k, what=None, precision=_lib.FP64, params=None, **over):
        run = dataclasses.replace(case.run, **over)
        return _Spec(what or f"storm {k}", d, run, storms[k] if run.nws else None, precision, params)
    return spec


def _beach(k):
    case = meshgen.beach()
    hol = list(case.run.holland)
    hol[0] += 5.0 * k
    return _Spec(f"beach {k}", case_setup(case), case.run, tuple(hol))


def _basin(what, name, run):
    return _Spec(what, load_golden(name), run)


def _members(name, storm):
    mixed = _lib.MIXED
    if name == "mixed precision":
        return [storm(k, precision=mixed) for k in range(3)]
    if name == "FP64 beside mixed":
        return [storm(0), storm(1, precision=mixed), storm(2), storm(3, precision=mixed)]
    if name == "mixed, two meshes":
        return [storm(0, precision=mixed), storm(1, precision=mixed), _beach(0), storm(2, precision=mixed)]
    if name == "storms beside calm":
        calm = [storm(k, what=f"calm {k}", holland=None) for k in range(2)]
        return [calm[0], storm(0), calm[1], storm(1)]
    if name == "beside rivers":
        return [storm(0), _basin("rivers", "basin_river", meshgen.basin_river().run), storm(1)]
    if name == "beside a tidal potential":
        return [_basin("tide", "basin_tide", meshgen.basin_tide().run), storm(0), storm(1)]
    if name == "beside the learned start":
        rng = np.random.default_rng(5)
        params = (0.05 * rng.standard_normal(_lib.ML_NPARAM)).astype(np.float32)
        return [storm(0), storm(1), storm(2, what="learned", warm_start=2, params=params), storm(3)]
    if name == "beside the lumped GWCE":
        return [storm(0), storm(2, what="lumped", ilump=1), storm(1)]
    if name == "extrapolated starts":
        return [storm(0, warm_start=1), storm(1), storm(2, warm_start=1)]
    raise KeyError(name)


CASES = ("mixed precision", "FP64 beside mixed", "mixed, two meshes", "storms beside calm",
         "beside rivers", "beside a tidal potential", "beside the learned start",
         "beside the lumped GWCE", "extrapolated starts")


@pytest.mark.parametrize("name", CASES)
def test_members_equal_their_own_runs(name, coastal):
    """Two runs of the batch, of odd and even length: the members' arguments
    alternate with the time levels."""
    from adcirc_amd.model import Batch
    specs = _members(name, coastal)
    log(f"batch {name}: {[s.what for s in specs]}, 45 + 30 steps")
    members = [s.model() for s in specs]
    singles = [s.model() for s in specs]
    hols = [s.holland for s in specs]
    b = Batch(members)
    for it0, n in ((1, 45), (46, 30)):
        b.run(it0, n, holland=hols)
        for g, h in zip(singles, hols):
            g.run_resident(it0, n, holland=h)
        for s, x, y in zip(specs, members, singles):
            for f in FIELDS:
                u, v = x.get(f), y.get(f)
                assert np.array_equal(u, v), (name, s.what, it0, f, int((u != v).sum()))
            assert x.run_stats() == y.run_stats(), (name, s.what, it0)
    b.close()
    for g in members + singles:
        g.close()
