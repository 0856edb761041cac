"""Reading the macroscopic fields around the longest read through pinned memory:
S of just under and just over 512 KB (two of the former do not fit the pinned
memory together), against the oracle's arrays."""
import numpy as np
import pytest

from helpers import load_pkg
from test_gpu_parity import _compare, _pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [69, 70])
def test_fields_read_back(n):
    gpu, cpu = _pair(load_pkg().cases.cavity_case(n, 6, kn=0.2, lid=0.2, dt=0.5))
    gpu.step(1)
    cpu.step(1)
    _compare(gpu, cpu, f"cavity {n}")
    a, b = gpu.macro(), cpu.macro()
    assert np.array_equal(a["s"] == 0.0, b["s"] == 0.0)
