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


BATCH = """
import importlib, math
import numpy as np
from gsis_amd import solver
batch = importlib.import_module("gsis_amd.batch")
def box(cells_i, cells_j, bent=False):
    c = g.cases
    nx, ny = cells_i + 1, cells_j + 1
    x, y = np.meshgrid(np.linspace(0.0, 1.0, nx), np.linspace(0.0, 1.0, ny), indexing="ij")
    if bent:
        x, y = x + 0.2 * y, y + 0.03 * np.sin(math.pi * x)
    bcs = [c.BC(2, 1, nx, 1, 1, -2), c.BC(3, nx, nx, 1, ny, -2), c.BC(4, 1, nx, ny, ny, -2, 0.1, 0.0),
           c.BC(1, 1, 1, 1, ny, -2)]
    v, w = c.sinh_velocity_grid(4, 6.0)
    return c.Case("box", c.build_mesh(x, y, bcs), bcs, v, w, v.copy(), w.copy(), c.constants_from_kn(0.1, dt=0.05), "rest")
def gang(case):
    s = solver.GsisSolver(case, mode=1)
    b = batch.Batch([s])
    b.set_ns_graph(1)
    n = ctypes.c_int()
    print(b.ns_graph(), model.model_launches(b"k_ns_batch", ctypes.byref(n)) > 0, n.value)
"""


@pytest.mark.parametrize("cus", [256, 64, 32])
def test_a_batched_instance_never_needs_more_workgroups_than_fit_beside_others(run, cus):
    """The workgroups of an instance in a batched launch wait for each other, so all have to be
    resident: at most half of the device's, at any size of the mesh."""
    out = run(BATCH + f"""
model.model_set_cus({cus})
for i, j in ((5, 5), (64, 64), (128, 69), (700, 260), (2100, 260), (4700, 100), (12, 260)):
    gang(box(i, j, i % 3 == 0))
""")
    rows = [out[k:k + 3] for k in range(0, len(out), 3)]
    assert len(rows) == 7
    for in_graph, launched, workgroups in rows:
        assert (in_graph, launched) == ("1", "True")
        assert 1 < int(workgroups) <= cus // 2


def test_launches_whose_workgroups_wait_for_each_other_take_turns(run):
    """A handle's inner loop and a batch's gangs, on streams and threads of their own: no two may run
    at once, as each could hold workgroup slots that the other waits for."""
    out = run(BATCH + """
import threading
def handle(n):
    return solver.GsisSolver(box(n, n + 1), mode=1, kstep_show=1 << 30)
a, b = handle(20), handle(30)
for _ in range(3):
    a.step(1)
    b.step(2)
print(model.model_beside())
both = [batch.Batch([handle(10 + k) for k in range(4)]) for _ in range(2)]
assert all(x.ns_graph() == 4 for x in both)
a.step(1)
both[0].step(1)
print(model.model_beside())
ts = [threading.Thread(target=x.step, args=(500,)) for x in both + [a]]
for t in ts: t.start()
for t in ts: t.join()
print(model.model_beside(), model.model_captured_fills(), model.model_races())
""")
    assert out == ["0", "0", "0", "0", "0"]


def test_a_batch_leaves_turns_to_others(run):
    """A batch's call of many steps queues two at a time, so that another thread's solve waits for
    two steps and not for all of them."""
    out = run(BATCH + """
b = batch.Batch([solver.GsisSolver(box(10 + k, 12), mode=1, kstep_show=1 << 30) for k in range(4)])
b.step(50)
b.step(1)
print(b.ns_graph(), model.model_queued())
""")
    assert out[0] == "4" and 1 <= int(out[1]) <= 2


@pytest.mark.parametrize("bent", [False, True], ids=["axis", "bent"])
def test_the_largest_meshes_of_the_synthetic_solve(run, bent):
    """Refused is what does not fit the 32-bit offsets into the sweep's arrays: 12 doubles for each of 64
    rows of a plane, nx - 5 planes in a single band of one row, below 2 GiB up to nx = 349530."""
    out = run(BATCH + f"""
for nx in (349530, 349531):
    q = box(nx - 1, 5, {bent})
    try:
        solver.GsisSolver(q, mode=1).close()
        print("taken")
    except g.capi.GsisError as e:
        print("2 GiB" in str(e) and "refused")
""")
    assert out == ["taken", "refused"]


@pytest.mark.parametrize("cus", [256, 64, 32])
def test_many_bands_on_few_cus(run, cus):
    """The bands of an instance are spread over every eighth workgroup only where the device has the CUs."""
    out = run(BATCH + f"""
model.model_set_cus({cus})
n = ctypes.c_int()
for j in (260, 330, 1028):
    s = solver.GsisSolver(box(20, j), mode=1, kstep_show=1 << 30)
    s.step(1)
    model.model_launches(b"k_ns_loop", ctypes.byref(n))
    print(n.value)
    s.close()
""")
    assert len(out) == 3 and all(1 < int(n) <= cus for n in out)


def test_a_step_allocates_nothing_on_the_host(run):
    """What a step launches is laid out when its handle is made: an allocation that failed in a step
    would throw through its C entry."""
    out = run(BATCH + """
model.model_own_allocations.restype = ctypes.c_long
hs = [solver.GsisSolver(c, mode=m, kstep_show=1 << 30)
      for c, m in ((box(12, 9), 0), (box(12, 9, True), 1), (g.cases.couette_case(ny_cells=9, nx_cells=6, nv=6), 0))]
n = model.model_own_allocations()
for h in hs:
    h.step(3)
    h.counters()
print(n > 0, model.model_own_allocations() - n)
""")
    assert out == ["True", "0"]


def test_a_handle_without_pinned_memory(run):
    """Pinned memory that cannot be had is no error: reads go into pageable memory, steps run."""
    out = run(BATCH + """
model.model_no_pinned_memory()
s = solver.GsisSolver(box(12, 9), mode=1, kstep_show=1 << 30)
s.step(2)
s.macro()
model.model_shortest_pageable_read.restype = ctypes.c_size_t
print(s.counters()[0], model.model_shortest_pageable_read())
""")
    assert out == ["2", "8"]
