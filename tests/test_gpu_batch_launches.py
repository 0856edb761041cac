"""A batch's launches over instances of every kind at once: strips of 16 columns
and of 8, several boundary launches in order (periodic, far-field and walls in
one instance), both forms of the moments kernel, a mass-corrected instance.
An instance's work is the single step's, so the fields are the same bits."""
import importlib

import numpy as np
import pytest

from helpers import channel_case, cylinder_case, load_pkg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wide", [True, False], ids=["strips16_and_8", "strips8"])
def test_mixed_batch_equals_single_steps(wide):
    g = load_pkg()
    solver = importlib.import_module("gsis_amd.solver")
    batch = importlib.import_module("gsis_amd.batch")

    def cases():
        # 4 x 64 strips of 16 columns: from there on a batch takes 16
        big = [g.cases.cavity_case(64, 64, kn=0.1, lid=0.2, dt=0.8)] if wide else []
        return big + [g.cases.couette_case(ny_cells=16, nx_cells=4, nv=12, kn=0.1, uwall=0.1, dt=0.5),
                      g.cases.couette_case(ny_cells=9, nx_cells=21, nv=34, kn=0.1, uwall=0.1, dt=0.5),
                      cylinder_case(), channel_case(), g.cases.cavity_case(9, 20, kn=0.1, lid=0.2, dt=0.8)]

    def make():
        out = []
        for k, c in enumerate(cases()):
            print("case:", c.name, flush=True)
            c.const["scheme"] = g.capi.SCHEME_NND
            s = solver.GsisSolver(c, kstep_show=1 << 30)
            s.initialize()
            if k == 1:
                s.set_mass_correct(True)
            out.append(s)
        return out

    single, both = make(), make()
    b = batch.Batch(both)
    for _ in range(2):  # the graph is replayed
        b.step(1)
        for s in single:
            s.step(1)
    for k, (p, q) in enumerate(zip(single, both)):
        mp, mq = p.macro(), q.macro()
        for f in ("s", "s0", "u", "cf", "taoi", "qj", "swall"):
            assert np.array_equal(mp[f], mq[f]), (k, f)
        assert np.array_equal(p.frd(), q.frd()), k
