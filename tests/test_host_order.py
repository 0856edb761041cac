"""The order of what the library gives to the GPU, without a GPU: the calls to the
HIP runtime go to a model (hip_order_model.cpp) that keeps account of which
operation is sure to have ended before which."""
import pathlib
import subprocess
import sys

import pytest

HERE = pathlib.Path(__file__).resolve().parent

PROLOGUE = """
import ctypes, sys
sys.path.insert(0, {here!r})
model = ctypes.CDLL({model!r}, mode=ctypes.RTLD_GLOBAL)
from helpers import load_pkg
g = load_pkg()
lib = g.capi.load_library()
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    so = tmp_path_factory.mktemp("model") / "hip_order_model.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", str(so), str(HERE / "hip_order_model.cpp")],
                   check=True)

    def go(body):  # a process of its own: the library binds to the runtime once
        code = PROLOGUE.format(here=str(HERE), model=str(so)) + body
        r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout.split()

    return go


def test_a_new_network_keeps_what_is_written_to_it(run):
    """The clears of its memory come before the default scaling, the parameters and the samples."""
    out = run("""
import numpy as np
from gsis_amd import closure
net = closure.Mlp()
print(model.model_races())
net.set_params(closure.init_params(1))
x = np.zeros((100, 8), np.float32)
net.forward(x)
net.loss_grad(x, x[:, :5])
net.forward(np.zeros((500, 8), np.float32))
net.train(x, x[:, :5], 1, 64)
print(model.model_races())
""")
    assert out == ["0", "0"]


@pytest.mark.parametrize("cells", [6, 19, 20, 30, 40, 58])
def test_short_reads_go_through_pinned_memory(run, cells):
    """The runtime's own way into pageable memory takes up to three times as long between 64 and 190 KB."""
    out = run(f"""
from gsis_amd import solver
s = solver.GsisSolver(g.cases.cavity_case({cells}, 6, kn=0.2))
s.macro()
s.counters()
model.model_shortest_pageable_read.restype = ctypes.c_size_t
print(model.model_shortest_pageable_read(), model.model_races())
""")
    assert int(out[0]) > 190 << 10
    assert out[1] == "0"
