"""Launches of the secretion phase on an MI355X: small meshes are bound by their number."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# a process of its own: torch's tracer has to be loaded before the library
PROGRAM = """
import sys
import numpy as np
import torch
from torch.profiler import ProfilerActivity, profile
import parabiofvm_amd

torch.cuda.init()
rng = np.random.default_rng(1)
A, S = 60, 3
uniform = lambda *shape: rng.random(shape, dtype=np.float32)
g = parabiofvm_amd.DeviceSolver(3, [0] * 3, [240, 180, 140], [20] * 3, S, 0.01, np.full(S, 1e4, np.float32),
                                np.full(S, 0.1, np.float32), np.zeros(S, np.float32))
g.set_agents({"positions": uniform(A, 3) * np.float32(139), "volumes": uniform(A) * 1000,
              "secretion_rates": uniform(A, S), "uptake_rates": uniform(A, S), "saturation_densities": uniform(A, S),
              "net_export_rates": uniform(A, S), "internalized_substrates": np.zeros((A, S), np.float32)})
g.set_compute_internalized(sys.argv[1] == "1")
g.initialize()
g.store()
g.cell(True)
g.wait()
with profile(activities=[ProfilerActivity.CUDA]) as prof:
    g.cell(True)
    g.wait()
    torch.cuda.synchronize()
print("KERNELS", *[e.name.split("(")[0].split("::")[-1] for e in prof.events() if "bfvm::" in e.name])
"""


@pytest.mark.parametrize("internalized,most", [(1, 5), (0, 4)])
def test_recompute_launches(internalized, most):
    """Claims, terms and sums, then internalized amounts where they are kept, then densities."""
    r = subprocess.run([sys.executable, "-c", PROGRAM, str(internalized)], cwd=ROOT, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    kernels = next(x for x in r.stdout.splitlines() if x.startswith("KERNELS")).split()[1:]
    if not kernels:
        pytest.skip("kernel tracing is not available")
    assert len(kernels) <= most, kernels
