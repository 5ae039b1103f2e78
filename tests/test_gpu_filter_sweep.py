"""The recursive-filter sweeps (the automatic sweep of a context) on an MI355X, at the sizes where blocks, waves and
row ends change, against the double oracle and the other sweep algorithm.

Tolerance (FP32): a sweep's relative rounding error is at most about 2/(1 - mu) + 6 units of 2^-24 per element, mu <=
0.54 for the diffusion coefficients drawn here, so 2 solves of 3 sweeps stay below 4e-6; 1e-5 is the parity bar."""
import numpy as np
import pytest

from test_gpu_parity import REL, assert_close, build_pair, random_problem

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pkg():
    import parabiofvm_amd

    parabiofvm_amd.load()
    return parabiofvm_amd


# line lengths around the blocks a lane, a wave and a workgroup hold, each with a short other axis
LENGTHS = [2, 3, 5, 16, 25, 26, 33, 51, 104, 199, 201, 257, 400, 401, 801, 1201]


@pytest.mark.parametrize("S", [1, 3, 4, 8, 12, 17])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_lengths_f32(axis, S, pkg, oracle_mod):
    for n in LENGTHS:
        if n > 401 and S > 8:  # longer than the partitioned sweep's tables allow, which every mesh must fit
            continue
        shape = [5, 3, 4]
        shape[axis] = n
        p = random_problem(3, tuple(shape), S, seed=7 * n + S)
        o, g = build_pair(pkg, oracle_mod, p, dtype=np.float64)
        g.store()
        for _ in range(2):
            o.diffusion()
            g.diffusion()
        g.load()
        assert_close(g.densities, o.densities, what=f"axis {axis} n {n} S {S}: {g.partition(axis)}")
        g.close()


@pytest.mark.parametrize("storage", ["f16", "bf16"])
@pytest.mark.parametrize("S", [1, 3, 8, 17])
def test_lengths_16bit(S, storage, pkg, oracle_mod):
    for axis in range(3):
        for n in (2, 26, 51, 104, 257, 401):
            shape = [6, 5, 7]
            shape[axis] = n
            p = random_problem(3, tuple(shape), S, seed=11 * n + S)
            o, g = build_pair(pkg, oracle_mod, p, dtype=np.float64)
            g.set_storage(storage)
            g.initialize()
            g.store()
            for _ in range(2):
                o.diffusion()
                g.diffusion()
            g.load()
            err = np.linalg.norm(g.densities - o.densities) / np.linalg.norm(o.densities)
            # 7 roundings to 11 (FP16) or 8 (BF16) significant bits, each of at most one unit in the last place
            assert err <= 7 * (2.0**-10 if storage == "f16" else 2.0**-7), (axis, n, S, err)
            g.close()


@pytest.mark.parametrize("dims,shape", [(1, (77, 1, 1)), (2, (31, 45, 1)), (3, (21, 18, 33))])
@pytest.mark.parametrize("S", [1, 2, 4, 7])
def test_filter_equals_partitioned(dims, shape, S, pkg, oracle_mod):
    """The automatic sweep and the partitioned one (asked for by a chunk length) solve the same systems."""
    p = random_problem(dims, shape, S, seed=5)
    _, g = build_pair(pkg, oracle_mod, p)
    _, h = build_pair(pkg, oracle_mod, p, algorithm=pkg.BFVM_SWEEP_PARTITIONED, chunk=16)
    for s in (g, h):
        s.store()
        s.diffusion()
        s.load()
    assert_close(g.densities, h.densities, what="filter against partitioned")


@pytest.mark.parametrize("dims,shape", [(1, (130, 1, 1)), (2, (40, 60, 1))])
def test_lines_do_not_mix(dims, shape, pkg, oracle_mod):
    """NaN and infinity in one substrate leave every other substrate's values as they are, bit for bit."""
    S = 5
    p = random_problem(dims, shape, S, seed=3, faces=False, interior=False)
    _, g = build_pair(pkg, oracle_mod, p)
    g.store()
    g.diffusion()
    g.load()
    clean = g.densities.reshape(-1, S).copy()
    for bad in (np.nan, np.inf):
        g.densities[:] = p["dens"]
        g.densities.reshape(-1, S)[7, 2] = bad
        g.store()
        g.diffusion()
        g.load()
        got = g.densities.reshape(-1, S)
        keep = [0, 1, 3, 4]
        np.testing.assert_array_equal(got[:, keep].view(np.uint32), clean[:, keep].view(np.uint32))
        assert not np.isfinite(got[:, 2]).any()


def test_large_coefficients_keep_the_partitioned_sweep(pkg, oracle_mod):
    """Coefficients outside the filter's range (mu close to 1, negative diffusion) still run."""
    p = random_problem(3, (20, 30, 10), 2, seed=13, faces=False, interior=False)
    p["D"] = np.array([1e9, 1e4], dtype=np.float32)
    o, g = build_pair(pkg, oracle_mod, p, dtype=np.float64)
    g.store()
    o.diffusion()
    g.diffusion()
    g.load()
    err = np.abs(g.densities - o.densities).reshape(-1, 2)
    assert err[:, 1].max() <= REL * np.abs(o.densities).max()
    assert np.isfinite(g.densities).all()


@pytest.mark.parametrize("S", [2, 5, 7, 13, 31])
def test_staged_rows(S, pkg, oracle_mod):
    """x rows staged several to a workgroup: lengths at which the blocks, the lines of a wave and the rows of a task
    change, with row counts that leave a short last task; the tolerance is the lengths' test's."""
    for n in (4, 21, 42, 63, 64, 65, 130, 181, 275):
        if n > 65 and S > 13:  # longer than the partitioned sweep's tables allow, which every mesh must fit
            continue
        for rows in ((2, 2), (7, 3), (5, 13)):
            p = random_problem(3, (n, *rows), S, seed=3 * n + S)
            o, g = build_pair(pkg, oracle_mod, p, dtype=np.float64)
            g.store()
            for _ in range(2):
                o.diffusion()
                g.diffusion()
            g.load()
            assert_close(g.densities, o.densities, what=f"n {n} rows {rows} S {S}: {g.partition(0)}")
            g.close()


@pytest.mark.parametrize("storage", ["f32", "f16"])
@pytest.mark.parametrize("gradient", [False, True])
def test_small_instances_share_launches(storage, gradient, pkg, oracle_mod):
    """Small meshes of a batch, whose sweeps share launches, beside one that does not, against the same meshes stepped
    one by one: the same arithmetic up to fused multiply-adds in FP32, one unit of 11 bits per rounding in FP16."""
    shapes = [((9, 7, 5), 3), ((33, 1 + 16, 4), 4), ((64, 40, 21), 13), ((5, 6, 64), 1), ((17, 50, 33), 8), ((96, 90, 64), 16)]
    problems = [random_problem(3, sh, S, seed=70 + k) for k, (sh, S) in enumerate(shapes)]
    alone, together = [], []
    for p in problems:
        for out in (alone, together):
            _, g = build_pair(pkg, oracle_mod, p)
            g.set_storage(storage)
            g.initialize()
            g.store()
            out.append(g)
    batch = pkg.Batch(together)
    for _ in range(3):
        batch.timestep(True, gradient)
        for g in alone:
            g.timestep(True, gradient)
    batch.wait()
    for k, (g, h) in enumerate(zip(together, alone)):
        g.load()
        h.load()
        if storage == "f32":
            assert_close(g.densities, h.densities, what=f"instance {k}")
        else:
            # 3 steps of 5 roundings each on both sides (3 sweeps, the conversions)
            err = np.linalg.norm(g.densities - h.densities) / np.linalg.norm(h.densities)
            assert err <= 2 * 15 * 2.0**-10, (k, err)
        if gradient and storage == "f32":
            scale = np.abs(h.gradients).max()
            assert np.abs(g.gradients - h.gradients).max() <= 4 * REL * max(scale, np.abs(h.densities).max())
    batch.close()
