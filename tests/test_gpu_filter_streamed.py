"""Filter sweeps of densities larger than the Infinity Cache (256 MB) whose rows 4 does not divide, on an MI355X: y and z
stream columns of which the last is moved back into the range."""
import numpy as np
import pytest

from test_gpu_parity import assert_close

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pkg():
    import parabiofvm_amd

    parabiofvm_amd.load()
    return parabiofvm_amd


@pytest.mark.parametrize("storage,shape", [("f32", (251, 233, 241)), ("f16", (277, 311, 319)), ("bf16", (277, 311, 319))])
def test_streamed_ragged_columns(storage, shape, pkg):
    """Against the partitioned sweep (asked for by a block length): FP32 within the parity bar, 16 bits one unit of 11 or 8
    bits for each of 4 roundings (3 sweeps, the conversion) on both sides."""
    S = 5
    x = np.random.default_rng(21).random(shape[0] * shape[1] * shape[2] * S, dtype=np.float32)
    assert x.size * (4 if storage == "f32" else 2) > 256 << 20
    results = []
    for chunk in (0, 16):
        g = pkg.DeviceSolver(3, [0] * 3, [20 * n for n in shape], [20] * 3, S, 0.01,
                             np.array([1e3, 1e4, 1e5, 3e4, 3e3], np.float32), np.full(S, 0.1, np.float32),
                             np.zeros(S, np.float32))
        for axis in range(3):
            g.set_boundary(axis, axis % 2, np.linspace(0, 1, S, dtype=np.float32), np.array([1, 0, 1, 0, 1], np.uint8))
        g.set_sweep_algorithm(pkg.BFVM_SWEEP_PARTITIONED, chunk)
        g.set_storage(storage)
        g.initialize()
        g.densities[:] = x
        g.store()
        g.diffusion()
        g.load()
        results.append(g.densities.copy())
        g.close()
    a, b = results
    if storage == "f32":
        assert_close(a, b, what=f"{shape} x {S}")
    else:
        err = np.linalg.norm(a - b) / np.linalg.norm(b)
        assert err <= 2 * 4 * (2.0**-10 if storage == "f16" else 2.0**-7), err
