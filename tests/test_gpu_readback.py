"""Reading the macroscopic fields at the sizes where the way to the host changes
(S of 64 KB and just above, of one piece of 960 KB and just above) and on a
mesh that is not square, against the oracle's arrays: every component, the
ghost layers and the zeros beyond them."""
import pytest

from helpers import load_pkg
from test_gpu_parity import _compare, _pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(4, 31), (19, 19), (20, 20), (97, 97), (98, 98)])
def test_fields_read_back(nx, ny):
    g = load_pkg()
    if nx == ny:
        case = g.cases.cavity_case(nx, 6, kn=0.2, lid=0.2, dt=0.5)
    else:
        case = g.cases.couette_case(ny_cells=ny, nx_cells=nx, nv=6, kn=0.2, uwall=0.2, dt=0.5)
    gpu, cpu = _pair(case)
    gpu.step(1)
    cpu.step(1)
    _compare(gpu, cpu, case.name)
    a, b = gpu.macro(), cpu.macro()
    for f in ("s", "s0"):  # zero where there is no padded cell
        assert a[f].shape == b[f].shape
        assert not a[f][:, :2].any() and not a[f][:, :, :2].any()
        assert not a[f][:, -2:].any() and not a[f][:, :, -2:].any()
