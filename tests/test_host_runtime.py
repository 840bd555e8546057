"""The library's host code over a HIP runtime without a device
(hip_host_stub.cpp: kernels are not run, calls can be made to fail): what a
failed call leaves behind, which launch a small solve takes, and contexts
driven from several threads.  Each check runs in a process of its own, where
the stub is loaded ahead of the library."""
from __future__ import annotations

import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def stub_path(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("stub") / "libhip_host_stub.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-pthread",
                    "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include",
                    os.path.join(HERE, "hip_host_stub.cpp"), "-o", out], check=True)
    return out


def _child(stub_path, check, *args):
    code = ("import sys; sys.path[:0] = [%r, %r]; import test_host_runtime as t; t.%s(%s)"
            % (os.path.dirname(HERE), HERE, check, ", ".join(map(repr, (stub_path,) + args))))
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.returncode, r.stdout[-2000:], r.stderr[-2000:])


class _Stub:
    def __init__(self, path):
        self.lib = C.CDLL(path, C.RTLD_GLOBAL)  # found before the HIP runtime's symbols
        for f in ("ordinary", "cooperative", "dead_uses", "live_streams"):
            getattr(self.lib, "stub_" + f).restype = C.c_long
        self.lib.stub_last_pinned.restype = C.c_void_p
        for f in ("fail_copy", "fail_cooperative"):
            getattr(self.lib, "stub_" + f).argtypes = [C.c_long]

    def __getattr__(self, name):
        return getattr(self.lib, "stub_" + name)


def _models(n, nodes=2000, **over):
    import dataclasses
    from adcirc_amd import meshgen
    from adcirc_amd.model import Model
    from gpu_helpers import case_setup, golden_tables
    case = meshgen.coastal(nodes)
    run = dataclasses.replace(case.run, **over)
    d = case_setup(case)
    t = golden_tables(d)
    got = []
    for _ in range(n):
        g = Model(t, run, emo=np.asarray(d["emo"]).reshape(t["neta"], -1),
                  efa=np.asarray(d["efa"]).reshape(t["neta"], -1))
        g.cold_start(d["eta2_0"], d["nodecode0"], d["noff0"])
        got.append(g)
    return got, run


def _step(m, it):
    w = np.zeros(m.np_)
    m.timestep(it, (w, w, w))


# ---- a run of a batch that fails part way
def child_failed_batch(path, what):
    from adcirc_amd.model import Batch
    stub = _Stub(path)
    models, run = _models(3)
    streams = stub.live_streams()
    failed = 0
    for nth in range(1, 200):
        b = Batch(models)
        getattr(stub, "fail_" + what)(nth)
        try:
            b.run(1, 3, holland=[run.holland] * 3)
            done = True
        except RuntimeError as e:
            assert "stub error" in str(e), e
            done = False
        getattr(stub, "fail_" + what)(0)
        b.close()
        assert stub.live_streams() == streams
        # no member holds the batch's stream, and none counts as solving: a small
        # solve takes the ordinary launch
        for m in models:
            coop = stub.cooperative()
            _step(m, 5)
            m.synchronize()
            assert stub.dead_uses() == 0, (nth, stub.dead_uses())
            assert stub.cooperative() == coop, nth
        if done:
            break
        failed += 1
    assert done and failed > 0, failed
    for m in models:
        m.close()
    assert stub.live_streams() == 0 and stub.dead_uses() == 0


@pytest.mark.parametrize("what", ["copy", "cooperative"])
def test_failed_batch_gives_the_streams_back(stub_path, what):
    """Each copy, or each cooperative launch, of a three-step run fails in turn."""
    _child(stub_path, "child_failed_batch", what)


# ---- the launch of a small solve
def child_launch_choice(path):
    stub = _Stub(path)
    (a, b), _ = _models(2)

    def cooperative(m, it):
        before = stub.cooperative()
        _step(m, it)
        return stub.cooperative() - before

    assert cooperative(a, 1) == 0      # alone
    assert cooperative(a, 2) == 0
    assert cooperative(b, 1) == 1      # a's solves have not been waited for
    assert cooperative(a, 3) == 1
    for wait in (a.synchronize, a.numitr, a.last_solve, lambda: a.get("eta2"), a.save_state,
                 lambda: a.set("tk", a.get("tk"))):
        b.synchronize()
        _step(a, 4)
        wait()
        assert cooperative(b, 2) == 0, wait   # a has been waited for
    a.close()
    b.close()


def test_launch_follows_what_is_solving(stub_path):
    """A small solve takes the ordinary launch exactly while no other context has
    solves that nobody has waited for; every call that waits counts."""
    _child(stub_path, "child_launch_choice")


def child_given_up(path):
    stub = _Stub(path)
    (m,), _ = _models(1)
    given = C.c_int.from_address(stub.last_pinned())
    it = 0

    def cooperative(n):
        nonlocal it
        before = stub.cooperative()
        for _ in range(n):
            it += 1
            _step(m, it)
        return stub.cooperative() - before

    assert cooperative(3) == 0
    n = 512
    for _ in range(3):
        given.value = 1                      # what k_jcg_mem leaves
        assert cooperative(n) == n
        assert given.value == 0
        assert cooperative(2) == 0
        n *= 2
    m.lib.adcgpu_set_jcg_giveup(m.h, 0)
    given.value = 1
    assert cooperative(512) == 512
    assert cooperative(1) == 0
    m.close()


def test_given_up_launch_brings_back_the_cooperative_one(stub_path):
    """After a small solve's launch was given up (the chip is shared) the context's
    solves take the cooperative launch, each time for twice as long."""
    _child(stub_path, "child_given_up")


def child_snapshot_layout(path):
    _Stub(path)
    (m,), _ = _models(1)
    np_, ne, mnei = m.np_, m.ne, m.mnei
    a = m.save_state()
    noffold = 16 + 25 * 8 * np_ + 5 * 4 * np_ + 4 * ne
    assert a.size == (noffold + 4 * ne + 8 * ne + 8 * mnei * np_ + 8 * max(m.neta, 1) * mnei
                      + 8 * 8 + 12 * 8 + 16 * 4)
    b = np.random.default_rng(1).integers(0, 256, a.size).astype(np.uint8)
    b[:16] = a[:16]
    m.load_state(b)
    b[noffold:noffold + 4 * ne] = 0  # NOFFOLD: once kept, not read
    assert np.array_equal(m.save_state(), b)
    m.close()


def test_snapshot_layout(stub_path):
    """The snapshot's layout is that of earlier files."""
    _child(stub_path, "child_snapshot_layout")


# ---- contexts driven from several threads
def child_threads(path, close):
    import threading
    stub = _Stub(path)
    models, _ = _models(4)
    errors = []

    def work(m):
        try:
            for it in range(1, 121):
                _step(m, it)
                if it % 3 == 0:
                    m.numitr()
            m.get("eta2")
            if close:
                m.close()
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(m,)) for m in models]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    assert stub.dead_uses() == 0
    assert stub.live_streams() == (0 if close else 4)
    # every context has been waited for: none counts as solving
    (last,), _ = _models(1)
    coop = stub.cooperative()
    _step(last, 1)
    assert stub.cooperative() == coop
    # what is open is left to the interpreter's end


@pytest.mark.parametrize("close", [True, False])
def test_contexts_of_several_threads(stub_path, close):
    """Four threads step a context each at once; the count of solving contexts ends
    at none, and the process ends cleanly with the contexts closed by their threads
    or left open."""
    _child(stub_path, "child_threads", close)
