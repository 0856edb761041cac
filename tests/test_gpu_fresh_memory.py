"""Device memory is cleared before its first use: what a call queues on a
handle's stream right after an allocation is not cleared again (the clear runs
on another stream).  MassCorrect allocates on its first call and sums the mass
at once: a sum cleared too late made every density zero."""
import importlib

import numpy as np
import pytest

from helpers import load_pkg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["m0", "m1"])
def test_mass_correction_of_new_instances(mode):
    g = load_pkg()
    solver = importlib.import_module("gsis_amd.solver")
    m = g.capi.MODE_M1 if mode == "m1" else g.capi.MODE_M0
    keep = []
    for k in range(40):
        case = g.cases.cavity_case(24 + 3 * (k % 16), 12, kn=0.2, lid=0.1, dt=0.5)
        s = solver.GsisSolver(case, mode=m, ns_maxit=3, kstep_show=1 << 30)
        s.initialize()
        before = s.macro()["s"][0].sum()
        s.set_mass_correct(True)
        s.step(1)
        rho = s.macro()["s"][0]
        assert np.isfinite(rho).all(), k
        assert abs(rho.sum() / before - 1.0) < 0.01, k
        keep.append(s)
