"""The synthetic solve's inner loop at the edges of its split: bands of 64
swept rows (nodes in j less 5), groups of four plane steps, flux tiles of
8 x 16 cells, and meshes whose face normals are not those of the axes; batched
launches with more workgroups than fit the device.

Bar: the oracle's inner iteration counts and 1e-10 relative L2 on the fields."""
import math

import numpy as np
import pytest

from helpers import load_oracle, load_pkg, rel_l2, solver_mod

pytestmark = pytest.mark.gpu
TOL = 1e-10


def _box(cells_i, cells_j, bent, lid=0.15, nv=8):
    g = load_pkg()
    c = g.cases
    nx, ny = cells_i + 1, cells_j + 1
    x, y = np.meshgrid(np.linspace(0.0, 1.0, nx), np.linspace(0.0, 1.0, ny), indexing="ij")
    if bent:
        x, y = x + 0.2 * y + 0.02 * np.sin(math.pi * y), y + 0.03 * np.sin(math.pi * x)
    bcs = [c.BC(2, 1, nx, 1, 1, g.capi.BC_WALL), c.BC(3, nx, nx, 1, ny, g.capi.BC_WALL),
           c.BC(4, 1, nx, ny, ny, g.capi.BC_WALL, lid, 0.0), c.BC(1, 1, 1, 1, ny, g.capi.BC_WALL)]
    v, w = c.sinh_velocity_grid(nv, 6.0)
    return c.Case(f"box{cells_i}x{cells_j}{'_bent' if bent else ''}", c.build_mesh(x, y, bcs), bcs, v, w, v.copy(),
                  w.copy(), c.constants_from_kn(0.1, dt=0.05), "rest")


@pytest.mark.parametrize("bent", [False, True], ids=["axis", "bent"])
@pytest.mark.parametrize("cells_i,cells_j", [(5, 5), (5, 69), (6, 133), (9, 67), (20, 68), (12, 69), (37, 6),
                                             (68, 132), (70, 197), (11, 263)])
def test_inner_loop_follows_the_oracle(cells_i, cells_j, bent):
    case = _box(cells_i, cells_j, bent)
    print(case.name, flush=True)
    gpu = solver_mod().GsisSolver(case, mode=1, ns_maxit=25)
    cpu = load_oracle().OracleSolver(case, mode=1, ns_maxit=25)
    for s in (gpu, cpu):
        s.initialize()
        s.step(2)
    assert gpu.counters()[2] == cpu.counters()[2] > 1
    a, b = gpu.macro(), cpu.macro()
    errs = {k: rel_l2(a[k], b[k]) for k in ("s", "s0", "cf", "u")}
    print({k: f"{v:.1e}" for k, v in errs.items()}, flush=True)
    assert max(errs.values()) <= TOL
    gpu.close()
    cpu.close()


def test_batch_larger_than_the_device_equals_single_steps():
    """300 instances, two or three workgroups each: the launch's gangs follow one another."""
    g = load_pkg()
    import importlib
    batch = importlib.import_module("gsis_amd.batch")
    sizes = [(6 + k % 7, 6 + (5 * k) % 11) for k in range(299)] + [(10, 70)]
    cases = [_box(a, b, k % 3 == 0, lid=0.05 + 0.001 * k, nv=4) for k, (a, b) in enumerate(sizes)]

    def make(c):
        s = solver_mod().GsisSolver(c, mode=1, ns_maxit=20)
        s.initialize()
        return s

    both = [make(c) for c in cases]
    b = batch.Batch(both)
    assert b.ns_graph() == len(cases)
    b.step(2)
    for k in (0, 1, 7, 150, 297, 298, 299):
        print("instance", k, cases[k].name, flush=True)
        s = make(cases[k])
        s.step(2)
        assert s.counters()[2] == both[k].counters()[2]
        for f in ("s", "u"):
            assert np.array_equal(s.macro()[f], both[k].macro()[f])
        s.close()
    b.close()
    for s in both:
        s.close()
