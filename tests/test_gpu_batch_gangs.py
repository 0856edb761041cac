"""Batched synthetic solves whose instances have several bands of swept rows and
several flux workgroups each, axis-aligned and not, among them one with more
flux tiles (263 x 16) than sixteen times the device's workgroups: placed in the
graph by default from four instances on, with the bits and the inner iteration
counts of single steps."""
import importlib

import numpy as np
import pytest

from helpers import load_pkg, solver_mod
from test_gpu_synthetic_bands import _box

pytestmark = pytest.mark.gpu


def test_gangs_of_several_bands_equal_single_steps():
    load_pkg()
    batch = importlib.import_module("gsis_amd.batch")
    cases = [_box(i, j, bent, nv=4) for i, j, bent in ((70, 132, True), (70, 197, False), (132, 260, True),
                                                       (2100, 260, False))]

    def make(c):
        print("case:", c.name, flush=True)
        s = solver_mod().GsisSolver(c, mode=1, ns_maxit=15)
        s.initialize()
        return s

    both = [make(c) for c in cases]
    b = batch.Batch(both)
    assert b.ns_graph() == 4
    for _ in range(2):  # the graph is replayed
        b.step(1)
    print("batch done", flush=True)
    for c, q in zip(cases, both):
        p = make(c)
        p.step(2)
        assert p.counters()[2] == q.counters()[2] > 1
        mp, mq = p.macro(), q.macro()
        for f in ("s", "s0", "u", "taoi", "qj"):
            assert np.array_equal(mp[f], mq[f]), (c.name, f)
        p.close()


def test_three_instances_are_solved_after_the_graph():
    load_pkg()
    batch = importlib.import_module("gsis_amd.batch")
    hs = []
    for k in range(3):
        s = solver_mod().GsisSolver(_box(8 + k, 9, False, nv=4), mode=1, ns_maxit=5)
        s.initialize()
        hs.append(s)
    assert batch.Batch(hs).ns_graph() == 0


def test_batches_and_a_handle_on_threads_of_their_own():
    """Launches whose workgroups wait for each other come from three threads at once."""
    import threading

    load_pkg()
    batch = importlib.import_module("gsis_amd.batch")
    sets = [[_box(64 + 5 * k, 70 - 3 * k, k % 2 == 0, nv=4) for k in range(4)],
            [_box(40 + 9 * k, 66 + 2 * k, k % 2 == 1, nv=4) for k in range(5)], [_box(90, 100, True, nv=4)]]

    def make(c):
        print("case:", c.name, flush=True)
        s = solver_mod().GsisSolver(c, mode=1, ns_maxit=12, kstep_show=1 << 30)
        s.initialize()
        return s

    hs = [[make(c) for c in cs] for cs in sets]
    runs = [batch.Batch(hs[0]), batch.Batch(hs[1]), hs[2][0]]
    assert runs[0].ns_graph() == 4 and runs[1].ns_graph() == 5
    err = []

    def go(r):
        try:
            for _ in range(3):
                r.step(2)
            if r is hs[2][0]:
                r.counters()  # waits, and reports waits that ran out
        except Exception as e:  # noqa: BLE001 (the assertion below shows it)
            err.append(e)

    ts = [threading.Thread(target=go, args=(r,)) for r in runs]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not err, err
    print("threads done", flush=True)
    for cs, qs in zip(sets, hs):
        for c, q in zip(cs, qs):
            p = make(c)
            p.step(6)
            assert p.counters()[2] == q.counters()[2]
            mp, mq = p.macro(), q.macro()
            for f in ("s", "u", "qj"):
                assert np.array_equal(mp[f], mq[f]), (c.name, f)
            p.close()
