"""Steps of several handles queued on their streams without a wait in between:
the kinetic strips of one (workgroups that wait for their neighbours) start
while the synthetic solve of another takes every CU.  The bits are those of the
handles stepped alone, and no wait runs out."""
import numpy as np
import pytest

from helpers import solver_mod
from test_gpu_synthetic_bands import _box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,nv", [(40, 12), (256, 8)])
def test_handles_step_beside_each_other(cells, nv):
    cases = [_box(cells + k, cells - k, k % 2 == 1, nv=nv, lid=0.1 + 0.01 * k) for k in range(4)]

    def make(c):
        print("case:", c.name, flush=True)
        s = solver_mod().GsisSolver(c, mode=1, ns_tol=1e-300, ns_maxit=30, kstep_show=1 << 30)
        s.initialize()
        return s

    hs = [make(c) for c in cases]
    for _ in range(3):
        for h in hs:
            h.step(1)
    together = []
    for h in hs:
        assert h.counters()[2] == 30  # waits, and reports waits that ran out
        together.append(h.macro())
        h.close()
    print("beside each other: done", flush=True)
    for c, m in zip(cases, together):
        p = make(c)
        p.step(3)
        q = p.macro()
        for f in ("s", "u", "qj"):
            assert np.array_equal(m[f], q[f]), (c.name, f)
        p.close()
