"""The synthetic solve on a long thin mesh, whose sweep records take 1.5 GiB of the
2 GiB that 32-bit offsets reach, against the oracle."""
import pytest

from helpers import load_oracle, rel_l2, solver_mod
from test_gpu_synthetic_bands import TOL, _box

pytestmark = pytest.mark.gpu


def test_records_beyond_one_and_a_half_gib():
    case = _box(262000, 5, True, nv=4)
    print(case.name, flush=True)
    gpu = solver_mod().GsisSolver(case, mode=1, ns_maxit=4)
    gpu.initialize()
    gpu.step(1)
    its = gpu.counters()[2]
    a = gpu.macro()
    gpu.close()
    print("gpu done", flush=True)
    cpu = load_oracle().OracleSolver(case, mode=1, ns_maxit=4)
    cpu.initialize()
    cpu.step(1)
    b = cpu.macro()
    assert its == cpu.counters()[2] > 1
    for k in ("s", "s0", "u"):
        assert rel_l2(a[k], b[k]) <= TOL, k
