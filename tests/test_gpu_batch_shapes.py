"""Launch shapes within a batch, on an MI355X: sweeps are shaped by the batch, whatever the contexts ask for; an
instance's gradient shape is its context's; the batch's autotuner times nothing and recomputes the gradients."""
import numpy as np
import pytest

from test_gpu_batch import check_gradients_of_stored
from test_gpu_parity import assert_close, build_pair, random_problem

pytestmark = pytest.mark.gpu

SHAPES = [((20, 12, 9), 4), ((11, 10, 8), 3), ((9, 14, 7), 8), ((13, 6, 10), 5), ((40, 33, 26), 12)]


@pytest.fixture(scope="module")
def pkg():
    import parabiofvm_amd

    parabiofvm_amd.load()
    return parabiofvm_amd


def solvers_of(pkg, oracle_mod, storage="f32", shapes=SHAPES):
    out = []
    for k, (shape, S) in enumerate(shapes):
        _, g = build_pair(pkg, oracle_mod, random_problem(3, shape, S, seed=500 + k))
        g.set_storage(storage)
        g.initialize()
        g.store()
        out.append(g)
    return out


def configs_of(solvers, shapes=SHAPES):
    return [{"grid": shape, "S": S, "voxel_shape": g.voxel_shape} for g, (shape, S) in zip(solvers, shapes)]


@pytest.mark.parametrize("storage", ["f32", "f16"])
@pytest.mark.parametrize("stacked", [False, True])
@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("groups", [0, 4096])
def test_gradient_shapes_of_the_contexts(groups, order, stacked, storage, pkg, oracle_mod):
    """4 and 8 rows per thread, both workgroup orders, chunks of the z planes by a workgroup count: each instance's
    gradient is that of its densities as stored."""
    solvers = solvers_of(pkg, oracle_mod, storage)
    for g in solvers:
        g.set_gradient_tuning(groups)
        g.set_gradient_stacked(stacked)
        g.set_gradient_order(order)
    batch = pkg.Batch(solvers)
    batch.timestep(True, True)
    batch.timestep(False, True)
    batch.wait()
    for g in solvers:
        g.load()
    check_gradients_of_stored(configs_of(solvers), solvers, f"groups {groups} stacked {stacked} order {order} {storage}")
    batch.close()
    for g in solvers:
        g.close()


def test_autotune_recomputes_the_gradients_each_time(pkg, oracle_mod):
    solvers = solvers_of(pkg, oracle_mod)
    batch = pkg.Batch(solvers)
    for step in range(2):
        batch.timestep(step == 0, False)
        batch.wait()
        for g in solvers:
            g.load()
        before = [g.densities.copy() for g in solvers]
        batch.autotune()
        for g, d in zip(solvers, before):
            g.gradients[:] = np.nan
            g.load()
            np.testing.assert_array_equal(g.densities.view(np.uint32), d.view(np.uint32))
        check_gradients_of_stored(configs_of(solvers), solvers, f"autotune after step {step}")
    batch.close()


@pytest.mark.parametrize("storage", ["f32", "f16"])
@pytest.mark.parametrize("setting", ["staged before", "staged", "exact", "chunk", "tuning", "workgroups"])
def test_sweeps_do_not_follow_the_contexts(setting, storage, pkg, oracle_mod):
    """Sweep algorithms, block lengths and workgroup caps that are set on the contexts, before the batch is made or
    while it exists, leave its results as they are, bit for bit (the densities of meshes without agents are the same
    from run to run)."""
    shapes = SHAPES + [((60, 50, 40), 4), ((18, 1, 33), 8)]

    def change(g):
        if "staged" in setting:
            g.set_sweep_algorithm(pkg.BFVM_SWEEP_STAGED)
        elif setting == "exact":
            g.set_sweep_algorithm(pkg.BFVM_SWEEP_EXACT)
        elif setting == "chunk":
            g.set_sweep_algorithm(pkg.BFVM_SWEEP_PARTITIONED, 32)
        elif setting == "tuning":
            for axis in range(3):
                g.set_sweep_tuning(axis, 16, 8)
        else:
            g.set_sweep_workgroups(3)

    results = []
    for changed in (False, True):
        solvers = solvers_of(pkg, oracle_mod, storage, shapes)
        if changed and setting != "exact" and setting != "staged":
            for g in solvers:
                change(g)
        batch = pkg.Batch(solvers)
        batch.timestep(False, False)
        if changed and setting in ("exact", "staged"):
            for g in solvers:
                change(g)
        batch.timestep(False, False)
        batch.wait()
        for g in solvers:
            g.load()
        results.append([g.densities.copy() for g in solvers])
        batch.close()
        for g in solvers:
            g.close()
    for k, (a, b) in enumerate(zip(*results)):
        np.testing.assert_array_equal(a.view(np.uint32), b.view(np.uint32), err_msg=f"instance {k} {shapes[k]}")


@pytest.mark.parametrize("storage", ["f32", "f16"])
@pytest.mark.parametrize("S", [1, 3, 4, 7, 13, 16])
def test_shared_launches_by_length(S, storage, pkg, oracle_mod):
    """Small instances whose sweeps share launches, lines of 2 to 257 voxels along each axis with Dirichlet faces: rows in
    one or several passes of a wave, blocks and segments at the edges of their lengths.  The same meshes stepped one by
    one differ by the two plans' roundings: FP32 within the parity bar, FP16 one unit of 11 bits per rounding."""
    shapes = []
    for n in (2, 3, 5, 17, 33, 49, 64, 65, 97, 130, 200, 257):
        for axis in range(3):
            shape = [6, 5, 7]
            shape[axis] = n
            shapes.append((tuple(shape), S))
    alone, together = (solvers_of(pkg, oracle_mod, storage, shapes) for _ in range(2))
    batch = pkg.Batch(together)
    for _ in range(2):
        batch.timestep(False, False)
        for g in alone:
            g.timestep(False, False)
    batch.wait()
    for (shape, _), g, h in zip(shapes, together, alone):
        g.load()
        h.load()
        if storage == "f32":
            assert_close(g.densities, h.densities, what=f"{shape} x {S}")
        else:
            # 2 steps of 4 roundings each on both sides (3 sweeps, the conversion)
            err = np.linalg.norm(g.densities - h.densities) / np.linalg.norm(h.densities)
            assert err <= 2 * 8 * 2.0**-10, (shape, S, err)
    batch.close()
    for g in alone + together:
        g.close()


@pytest.mark.parametrize("recompute", [False, True])
def test_direct_steps_and_replays(recompute, pkg, oracle_mod):
    """The first step of a kind after a change is launched directly, the second makes the graph, later ones replay it:
    agents that change before some of the steps, every instance against the oracle after each step."""
    shapes = [((24, 20, 18), 4), ((33, 28, 21), 3), ((140, 130, 40), 4)]
    rng = np.random.default_rng(12)
    pairs = [build_pair(pkg, oracle_mod, random_problem(3, shape, S, seed=600 + k)) for k, (shape, S) in enumerate(shapes)]

    def agents(k, A):
        S, grid = shapes[k][1], shapes[k][0]
        uniform = lambda *shape: rng.random(shape, dtype=np.float32)  # noqa: E731
        size = np.array([n * v for n, v in zip(grid, pairs[k][1].voxel_shape)], dtype=np.float32)
        a = {"positions": np.array(pairs[k][1].mins, np.float32) + uniform(A, 3) * size * np.float32(0.999),
             "volumes": uniform(A) * 1000, "secretion_rates": uniform(A, S), "uptake_rates": uniform(A, S),
             "saturation_densities": uniform(A, S), "net_export_rates": uniform(A, S),
             "internalized_substrates": np.zeros((A, S), np.float32),
             "fraction_released_at_death": np.zeros((A, S), np.float32)}
        for be in pairs[k]:
            be.set_agents({name: v.copy() for name, v in a.items()})
        pairs[k][0].initialize()
        pairs[k][1].store_agents()

    for k, (o, g) in enumerate(pairs):
        g.store()
        agents(k, 50)
    batch = pkg.Batch([g for _, g in pairs])
    for step in range(7):
        if step in (0, 1, 4):
            agents(step % 3, 60 + 20 * step)
        again = recompute or step in (0, 1, 4)  # new agents need their sums
        batch.timestep(again, step % 2 == 0 or recompute)
        for o, _ in pairs:
            o.timestep(again, step % 2 == 0 or recompute)
        batch.wait()
        for k, (o, g) in enumerate(pairs):
            g.load()
            assert_close(g.densities, o.densities, what=f"step {step} instance {k}")
    batch.close()
