"""Launches of small meshes on an MI355X, which are bound by their number."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# in a process of its own: torch's tracer has to be loaded before the library
HEAD = """
import sys
import numpy as np
import torch
from torch.profiler import ProfilerActivity, profile
import parabiofvm_amd

torch.cuda.init()
rng = np.random.default_rng(1)


def solver(shape, S):
    return parabiofvm_amd.DeviceSolver(3, [0] * 3, [20 * n for n in shape], [20] * 3, S, 0.01, np.full(S, 1e4, np.float32),
                                       np.full(S, 0.1, np.float32), np.zeros(S, np.float32))


def kernels(call):
    call()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        call()
        torch.cuda.synchronize()
    print("KERNELS", *[e.name.split("(")[0].split("::")[-1].replace(" ", "") for e in prof.events() if "bfvm::" in e.name])


"""

CELL = """
A, S = 60, 3
uniform = lambda *shape: rng.random(shape, dtype=np.float32)  # noqa: E731
g = solver((12, 9, 7), S)
g.set_agents({"positions": uniform(A, 3) * np.float32(139), "volumes": uniform(A) * 1000,
              "secretion_rates": uniform(A, S), "uptake_rates": uniform(A, S), "saturation_densities": uniform(A, S),
              "net_export_rates": uniform(A, S), "internalized_substrates": np.zeros((A, S), np.float32)})
g.set_compute_internalized(sys.argv[1] == "1")
g.initialize()
g.store()
kernels(lambda: (g.cell(True), g.wait()))
"""

BATCH = """
solvers = [solver(*x) for x in (((41, 37, 60), 7), ((64, 33, 50), 16), ((35, 64, 64), 5), ((50, 44, 39), 12))]
for g in solvers:
    g.set_storage(sys.argv[1])
    g.initialize()
    g.store()
b = parabiofvm_amd.Batch(solvers)
kernels(lambda: (b.timestep(False, False), b.wait()))
"""

GROWING = """
solvers = [solver(*x) for x in (((41, 37, 60), 7), ((64, 33, 50), 16), ((35, 64, 64), 5), ((70, 90, 80), 12))]
uniform = lambda *shape: rng.random(shape, dtype=np.float32)  # noqa: E731


def agents(g, A):
    S = g.S
    g.set_agents({"positions": uniform(A, 3) * np.float32(600), "volumes": uniform(A) * 1000,
                  "secretion_rates": uniform(A, S), "uptake_rates": uniform(A, S), "saturation_densities": uniform(A, S),
                  "net_export_rates": uniform(A, S), "internalized_substrates": np.zeros((A, S), np.float32)})


for g in solvers:
    agents(g, 100)
    g.initialize()
    g.store()
    g.store_agents()
b = parabiofvm_amd.Batch(solvers)
calls = []
for step in range(6):
    if step < 4:
        agents(solvers[1], 100 + 10 * step)
        solvers[1].store_agents()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        b.timestep(True, True)
        b.wait()
        torch.cuda.synchronize()
    names = [e.name for e in prof.events()]
    calls.append("%d,%d" % (names.count("hipGraphInstantiate"), names.count("hipGraphLaunch")))
    if not any("hip" in n for n in names):
        calls = []
        break
print("KERNELS", *calls)
"""


def launched(program, argument):
    r = subprocess.run([sys.executable, "-c", HEAD + program, argument], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    kernels = next(x for x in r.stdout.splitlines() if x.startswith("KERNELS")).split()[1:]
    if not kernels:
        pytest.skip("kernel tracing is not available")
    return kernels


@pytest.mark.parametrize("internalized,most", [("1", 5), ("0", 4)])
def test_recompute_launches(internalized, most):
    """Claims, terms and sums, then internalized amounts where they are kept, then densities."""
    kernels = launched(CELL, internalized)
    assert len(kernels) <= most, kernels


@pytest.mark.parametrize("storage,most", [("f32", 3), ("f16", 4)])
def test_small_batch_launches(storage, most):
    """Instances of at most 8 MB share one launch per axis (and the step of the rounding's counter)."""
    kernels = launched(BATCH, storage)
    assert len(kernels) <= most, kernels


def test_growing_batch_makes_no_graphs():
    """Agents that come between steps change the batch's launches: such steps are launched directly, and a graph is made
    once a step repeats (made, launched)."""
    assert launched(GROWING, "") == ["0,0"] * 4 + ["1,1", "0,1"]
