"""Which sweep the automatic shape takes as the diffusion coefficient grows, and its error for local sources, on an
MI355X.  a = dt * D / dx^2; the recursive filter runs up to a = 10 (decay constant mu = 0.73), the partitioned sweep
beyond and for negative diffusion."""
import numpy as np
import pytest

from test_gpu_parity import REL, assert_close

pytestmark = pytest.mark.gpu

DX, DT = 20, np.float32(0.01)


@pytest.fixture(scope="module")
def pkg():
    import parabiofvm_amd

    parabiofvm_amd.load()
    return parabiofvm_amd


def solver(pkg, n, a, chunk=None):
    D = np.array([a * DX**2 / float(DT)], dtype=np.float32)
    g = pkg.DeviceSolver(1, [0] * 3, [n * DX, DX, DX], [DX] * 3, 1, float(DT), D, np.array([0.1], np.float32),
                         np.zeros(1, np.float32))
    if chunk is not None:
        g.set_sweep_algorithm(pkg.BFVM_SWEEP_PARTITIONED, chunk)
    g.initialize()
    return g


def diffused(g, x):
    g.densities[:] = x
    g.store()
    g.diffusion()
    g.load()
    return g.densities.copy()


def exact(x, a):
    """The line's tridiagonal system in FP64 (Thomas algorithm)."""
    n = x.size
    a = float(DT) * float(np.float32(a * DX**2 / float(DT))) / DX**2
    lam = 1 + float(np.float32(0.1)) * float(DT)
    b = np.full(n, lam + 2 * a)
    b[[0, -1]] -= a
    d = x.astype(np.float64)
    for i in range(1, n):
        w = -a / b[i - 1]
        b[i] += w * a
        d[i] -= w * d[i - 1]
    d[n - 1] /= b[n - 1]
    for i in range(n - 2, -1, -1):
        d[i] = (d[i] + a * d[i + 1]) / b[i]
    return d


@pytest.mark.parametrize("a", [2.5, 9.9, 10.1, 250.0, 1e4, 1e5, 9e5])
@pytest.mark.parametrize("n", [400, 1000])
def test_local_sources(n, a, pkg):
    """A point source and a step, per voxel wherever the solution is above 1e-3 of its largest value.  The filter's
    error there is at most ln(1e3) 2^-25 / (mu |ln mu|) (the rounding of mu) + (2 / (1 - mu) + 6) 2^-24, 1.7e-6 at mu =
    0.73; the partitioned sweep's coefficients are rounded one by one, 3 roundings per element of a block of at most 64:
    4 standard deviations are 2e-6.  The bound is twice the larger; a filter used at any a reaches 1e-5 here."""
    g = solver(pkg, n, a)
    for name in ("point", "step"):
        x = np.zeros(n, dtype=np.float32)
        if name == "point":
            x[n // 3] = 1
        else:
            x[: n // 2] = 1
        want = exact(x, a)
        got = diffused(g, x)
        big = want > 1e-3 * want.max()
        err = (np.abs(got - want)[big] / want[big]).max()
        assert err <= 4e-6, (name, err)
    g.close()


@pytest.mark.parametrize("a,filter_runs", [(2.5, True), (9.9, True), (10.1, False), (1e4, False), (-0.1, False)])
def test_which_sweep_runs(a, filter_runs, pkg):
    """The partitioned sweep's result is, bit for bit, that of one of its block lengths asked for by hand; the filter's
    is none of them.  Both solve the system."""
    n = 300
    x = np.random.default_rng(8).random(n, dtype=np.float32)
    g = solver(pkg, n, a)
    got = diffused(g, x)
    same = []
    for chunk in (8, 16, 32, 48, 64):
        h = solver(pkg, n, a, chunk)
        same.append(np.array_equal(diffused(h, x).view(np.uint32), got.view(np.uint32)))
        h.close()
    assert any(same) != filter_runs, same
    assert_close(got, exact(x, a), rel=REL, what=f"a {a}")
    g.close()


@pytest.mark.parametrize("a", [2.5, 250.0])
def test_refused_tuning_leaves_the_steps(a, pkg):
    """A launch shape that does not fit is refused, and steps captured before it run on the tables that replaced theirs."""
    n = 300
    x = np.random.default_rng(9).random(n, dtype=np.float32)
    results = []
    for refused in (False, True):
        g = solver(pkg, n, a)
        g.densities[:] = x
        g.store()
        for step in range(4):
            if refused and step == 2:
                with pytest.raises(Exception):
                    g.set_sweep_tuning(0, 16, 1024)
            g.timestep(False, False)
        g.load()
        results.append(g.densities.copy())
        g.close()
    np.testing.assert_array_equal(results[0].view(np.uint32), results[1].view(np.uint32))


@pytest.mark.parametrize("a", [2.5, 9.9])
def test_values_near_the_largest(a, pkg):
    """Densities of up to 3e38: a diffused value lies within the range of the densities, and so does everything on the way
    to it."""
    n = 400
    x = (np.random.default_rng(10).random(n) * 2e38 + 1e38).astype(np.float32)
    g = solver(pkg, n, a)
    assert_close(diffused(g, x), exact(x, a), rel=REL, what=f"a {a}")
    g.close()
