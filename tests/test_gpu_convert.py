"""The conversion to NS variables in one kernel (corner S, U, its ghost
extrapolations, primitive variables) and the periodic faces in one launch, at
the smallest mesh, at padded cell counts around a workgroup's 64 and with ghost
cells that are extrapolated, copied or both, against the oracle."""
import pytest

from helpers import load_pkg, rel_l2
from test_gpu_parity import TOL, _compare, _pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,nx,ny", [("cavity", 4, 4), ("cavity", 5, 5), ("cavity", 12, 12), ("cavity", 13, 13),
                                        ("couette", 4, 4), ("couette", 12, 13), ("couette", 5, 28)])
def test_convert_against_oracle(kind, nx, ny):
    g = load_pkg()
    if kind == "cavity":
        case = g.cases.cavity_case(nx, 12, kn=0.1, lid=0.2, dt=0.8)
    else:
        case = g.cases.couette_case(ny_cells=ny, nx_cells=nx, nv=12, kn=0.1, uwall=0.1, dt=0.5)
    print("case:", case.name, flush=True)
    gpu, cpu = _pair(case)
    for k in range(2):
        gpu.step(1)
        cpu.step(1)
        _compare(gpu, cpu, f"{case.name} step {k + 1}")
        assert rel_l2(gpu.macro()["u"], cpu.macro()["u"]) <= TOL
