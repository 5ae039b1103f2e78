"""The process's tuning cache on an MI355X: an entry is applied to the kernels it was made for and to no others."""
import numpy as np
import pytest

from test_gpu_parity import assert_close, random_problem

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pkg():
    import parabiofvm_amd

    parabiofvm_amd.load()
    return parabiofvm_amd


def solver(pkg, shape, S, D):
    p = random_problem(3, shape, S, seed=4, faces=False, interior=False)
    g = pkg.DeviceSolver(p["dims"], p["mins"], p["maxs"], p["vs"], p["S"], p["dt"], np.full(S, D, np.float32), p["decay"],
                         p["init"])
    g.initialize()
    return g


@pytest.mark.parametrize("first", [1e12, 1e4])
def test_contexts_of_one_shape_and_other_coefficients(first, pkg):
    """Diffusion coefficients decide whether an axis takes the recursive filter.  A context tuned first, on the other side
    of that line, leaves a context of the same shape its own sweep."""
    shape, S = (70, 41, 26) if first > 1e6 else (71, 42, 27), 4
    second = 1e4 if first > 1e6 else 1e12
    a, b = solver(pkg, shape, S, first), solver(pkg, shape, S, second)
    automatic = [b.partition(axis) for axis in range(3)]
    a.autotune()
    b.autotune()
    if second < 1e6:  # the filter's tuning changes its workgroup cap alone
        assert [b.partition(axis) for axis in range(3)] == automatic
    else:  # the partitioned sweep's blocks are among those that the autotuner times
        assert {b.partition(axis)[1] for axis in range(3)} <= {m for c in (16, 32, 64) for m in range(1, c + 1)}
        c = solver(pkg, shape, S, second)
        c.autotune()
        assert [c.partition(axis) for axis in range(3)] == [b.partition(axis) for axis in range(3)]
        c.close()
    a.close()
    b.close()


def test_entries_of_older_files_leave_the_automatic_kernels(pkg, tmp_path):
    """Files written when the partitioned sweep and the tiled gradient were the automatic kernels name a block length
    and tile shapes: axes that take the recursive filter keep it, and the gradient is timed anew."""
    from parabiofvm_amd import _native

    shape, S = (50, 36, 44), 4
    path = tmp_path / "old.txt"
    entry = " ".join(str(v) for v in (*shape, S, 0, 0))
    path.write_text("".join(f"sweep {axis} {entry} 16 {lines} 1024\n" for axis, lines in ((0, 2), (1, 8), (2, 8))) +
                    f"gradient {entry} 2048 1 0\n")
    g = solver(pkg, shape, S, 1e4)
    automatic = [g.partition(axis) for axis in range(3)]
    _native.tuning_load(str(path))
    g.autotune()
    assert [g.partition(axis) for axis in range(3)] == automatic
    out = tmp_path / "out.txt"
    _native.tuning_save(str(out))
    lines = out.read_text().splitlines()
    assert f"sweep 0 {entry} 16 2 1024" in lines and f"gradient {entry} 2048 1 0" in lines
    assert any(x.startswith(f"gradient_field {entry} ") for x in lines)
    assert any(x.startswith(f"sweep 0 {entry} 0 0 ") for x in lines)
    g.close()


def test_autotune_where_only_a_requested_shape_fits(pkg, oracle_mod):
    """Lines of 1200 voxels x 18 substrates fit with 4 lines or fewer to a workgroup, which the automatic shape does not
    take: a context that asked for such a shape is tuned over the shapes that fit, and steps on."""
    p = random_problem(3, (4, 1200, 3), 18, seed=6, faces=False, interior=False)
    args = (p["dims"], p["mins"], p["maxs"], p["vs"], p["S"], p["dt"], p["D"], p["decay"], p["init"])
    o, g = oracle_mod.Oracle(*args, dtype=np.float64), pkg.DeviceSolver(*args)
    g.set_sweep_tuning(1, 32, 2)
    for be in (o, g):
        be.densities[:] = p["dens"]
        be.initialize()
    g.store()
    g.timestep(False, False)
    g.autotune()
    g.timestep(False, False)
    g.load()
    for _ in range(2):
        o.diffusion()
    assert_close(g.densities, o.densities, what=f"{[g.partition(axis) for axis in range(3)]}")
    g.close()
