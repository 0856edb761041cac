"""The column-pair kinetic kernel at the edges of its layout: pairs without a
right column, strips of one pair, one and several velocity tiles with a ragged
last one, odd numbers of velocities (copies of 16 bytes straddle their end) and
the smallest mesh, in both precisions and both strip widths, against the split
kernels.

Tolerance: the two paths round differently.  A step takes about 30 roundings of
terms no larger than the distribution, at most 30 * 2^-24 = 1.8e-6 of it in
FP32 and 30 * 2^-53 = 3.3e-15 in FP64; three steps, and a factor of 2 for what the
recursion passes on."""
import importlib

import numpy as np
import pytest

from helpers import load_pkg, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
@pytest.mark.parametrize("n,nv", [(4, 5), (5, 9), (15, 7), (16, 9), (17, 8), (18, 13), (33, 11)])
def test_column_pairs_agree_with_the_split_kernels(n, nv, fp32):
    g = load_pkg()
    solver = importlib.import_module("gsis_amd.solver")
    case = g.cases.cavity_case(n, nv, kn=0.1, lid=0.2, dt=0.8)
    print("case:", case.name, "fp32" if fp32 else "fp64", flush=True)
    out = {}
    for k in (g.capi.KERNEL_SPLIT, g.capi.KERNEL_AUTO, g.capi.KERNEL_STRIP16):
        s = solver.GsisSolver(case, precision=g.capi.PREC_FP32 if fp32 else g.capi.PREC_FP64, split_kernels=k)
        s.initialize()
        s.step(3)
        s.counters()  # waits, and reports a wait for a neighbouring strip that timed out
        out[k] = s.frd()
        s.close()
    ref = out.pop(g.capi.KERNEL_SPLIT)
    tol = 2 * 3 * (1.8e-6 if fp32 else 3.3e-15)
    for k, f in out.items():
        assert rel_l2(f, ref) <= tol, k
    # the two widths do the same arithmetic
    assert np.array_equal(*out.values())
