"""The work that a program built on parabiofvm_amd has it do, as measurable cases.

A case is a dict of plain values.  `prepare` builds what the program holds before the call (an initialized solver or
batch with its data on the GPU), `run` is one call of the public entry points, `work` the bytes and operations that
the call cannot do without, and `exact` the same call's results in 64-bit torch.

Sizes are those of this repository's workloads: the 100^3 x 4 microenvironment, the 400^3 x 8 instance with a million
clustered agents and Dirichlet conditions, the 64 uneven microenvironments of a batch (edges 32..200, 1..16
substrates), the 16-substrate clustered stress workload (reduced), the 1000-voxel lines of 2-D meshes, and small
meshes where the latency of a step counts.
"""
import random

import numpy as np
import torch

import parabiofvm_amd

DX = 20
DT = 0.01
AGENT_VOLUME = 2494.0
STEP = {"kind": "step", "nx": 1, "ny": 1, "nz": 1, "dims": 3, "substrates": 1, "storage": "f32", "agents": 0,
        "clusters": 0, "faces": False, "interior": 0.0, "reduction": "atomic", "recompute": False, "gradient": True,
        "internalized": True, "tuned": False}


def _step(name, shape, substrates, **more):
    case = dict(STEP, name=name, dims=len(shape), substrates=substrates)
    case.update(zip(("nx", "ny", "nz"), shape))
    case.update(more)
    return case


def listed():
    return [
        # a slice model of a small tissue sample: the latency of one step counts
        _step("step-2d-50x40x2", (50, 40), 2, agents=20, faces=True),
        # a small 3-D mesh with an odd substrate count, as a unit of a parameter scan
        _step("step-40x30x20x3", (40, 30, 20), 3, agents=300, faces=True, interior=0.01),
        # a large 2-D slice: lines of 1000 voxels
        _step("step-2d-1000x1000x4", (1000, 1000), 4, agents=5000, faces=True),
        # the everyday 3-D microenvironment, uniformly placed agents
        _step("step-100cube-4", (100, 100, 100), 4, agents=10_000),
        # ragged edges and a substrate count that 4 does not divide, agents that moved since the last step
        _step("step-181x97x143x5", (181, 97, 143), 5, agents=25_000, faces=True, interior=0.01, recompute=True),
        # the large single instance in a tuned production run, whole step
        _step("step-400cube-8", (400, 400, 400), 8, agents=1_000_000, clusters=16, faces=True, interior=0.01,
              tuned=True),
        # the same instance with densities stored in scaled FP16, a step without gradients
        _step("step-f16-400cube-8", (400, 400, 400), 8, agents=1_000_000, clusters=16, faces=True, interior=0.01,
              storage="f16", gradient=False, internalized=False, tuned=True),
        # 16 substrates in BF16 with crowded clusters that moved, agents combined by the sorted reduction
        _step("step-bf16-256cube-16", (256, 256, 256), 16, agents=1_000_000, clusters=64, faces=True, interior=0.005,
              storage="bf16", reduction="sorted", recompute=True, gradient=False, internalized=False),
        # gradients alone, of densities stored in FP16 (chemotaxis output at chosen steps)
        _step("gradient-f16-320cube-8", (320, 320, 320), 8, kind="gradient", storage="f16"),
        # secretion and uptake of a million clustered agents that moved, claim-and-atomics reduction
        _step("cell-1M-200cube-8", (200, 200, 200), 8, kind="cell", agents=1_000_000, clusters=16, recompute=True,
              gradient=False),
        # uneven microenvironments advanced together, whole step
        {"name": "batch-20-f32", "kind": "batch", "count": 20, "edge_min": 32, "edge_max": 200, "sub_min": 1,
         "sub_max": 16, "shape_seed": 4321, "storage": "f32", "gradient": True, "internalized": True, "tuned": True},
        # the 64-instance batch in scaled FP16, steps without gradients
        {"name": "batch-64-f16", "kind": "batch", "count": 64, "edge_min": 32, "edge_max": 200, "sub_min": 1,
         "sub_max": 16, "shape_seed": 1234, "storage": "f16", "gradient": False, "internalized": False,
         "tuned": True},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _edges3(rng, lo, hi, most):
    """Three edges of [lo, hi], the voxel count at most `most`."""
    while True:
        e = [_log(rng, lo, hi) for _ in range(3)]
        if e[0] * e[1] * e[2] <= most:
            return tuple(e)


def draw(rng):
    kind = rng.choice(["step3", "step3", "step3", "step2", "step16", "step16", "gradient", "cell", "batch", "batch"])
    faces, interior = rng.random() < 0.6, rng.choice([0.0, 0.0, 0.01, 0.03])
    recompute, tuned = rng.random() < 0.3, rng.random() < 0.3
    if kind == "batch":
        f32 = rng.random() < 0.5
        case = {"kind": "batch", "count": rng.randint(2, 20), "edge_min": 32, "edge_max": rng.choice([64, 120, 200]),
                "sub_min": 1, "sub_max": 16, "shape_seed": rng.randrange(1 << 30),
                "storage": "f32" if f32 else rng.choice(["f16", "bf16"]), "gradient": f32, "internalized": f32,
                "tuned": tuned}
        return case
    S = rng.randint(1, 16)
    if kind == "step2":
        S = rng.randint(1, 6)
        shape = (_log(rng, 20, 1200), _log(rng, 20, 1200))
    elif kind == "step3":
        shape = _edges3(rng, 16, 360, 300_000_000 // S)
    else:
        shape = _edges3(rng, 40, 360, 300_000_000 // S)
    voxels = int(np.prod(shape))
    agents = max(1, int(voxels * rng.choice([0.001, 0.01, 0.02])))
    case = _step("", shape, S, agents=min(agents, 1_000_000), clusters=rng.choice([0, 0, 16]), faces=faces,
                 interior=interior, recompute=recompute, tuned=tuned, reduction=rng.choice(["atomic", "atomic", "sorted"]))
    if kind == "step16":
        case.update(storage=rng.choice(["f16", "bf16"]), gradient=False, internalized=False)
    elif kind == "gradient":
        case.update(kind="gradient", storage=rng.choice(["f32", "f16", "bf16"]), agents=0, recompute=False)
    elif kind == "cell":
        case.update(kind="cell", recompute=True, gradient=False)
    del case["name"]
    return case


def _instances(case):
    """The microenvironments of a batch as step cases: uneven edges and substrate counts, agents on 1% of voxels."""
    rng = random.Random(case["shape_seed"])
    out = []
    for i in range(case["count"]):
        shape = tuple(rng.randint(case["edge_min"], case["edge_max"]) for _ in range(3))
        agents = max(1, shape[0] * shape[1] * shape[2] // 100)
        out.append(_step("", shape, rng.randint(case["sub_min"], case["sub_max"]), agents=agents,
                         storage=case["storage"], gradient=case["gradient"], internalized=case["internalized"]))
    return out


def _shape(case):
    return [case["nx"], case["ny"], case["nz"]]


def _inputs(case, seed):
    """The microenvironment's fields: initial densities ~ uniform[0, 1) on the GPU, the rest on the host."""
    n, S, A, dims = _shape(case), case["substrates"], case["agents"], case["dims"]
    V = n[0] * n[1] * n[2]
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = np.random.Generator(np.random.PCG64(seed))
    uniform = lambda *shape: r.random(shape, dtype=np.float32)  # noqa: E731
    x = {"densities": torch.rand(V * S, generator=g, device="cuda"),
         "D": np.exp(r.uniform(np.log(1e3), np.log(1e5), S)).astype(np.float32),
         "decay": r.uniform(0.01, 1.0, S).astype(np.float32), "faces": {}, "interior": None, "agents": None}
    if case["faces"]:
        x["faces"] = {(d, m): uniform(S) for d in range(dims) for m in (0, 1)}
    if case["interior"]:
        lin = np.unique(r.integers(0, V, max(1, int(V * case["interior"]))))
        vox = np.stack([lin % n[0], lin // n[0] % n[1], lin // (n[0] * n[1])], axis=1)[:, :dims]
        x["interior"] = (vox.astype(np.int32), uniform(lin.size, S), lin)
    if A:
        size = np.array(n[:dims], dtype=np.float64) * DX
        if case["clusters"]:
            centres = r.random((case["clusters"], dims)) * size
            pos = centres[r.integers(0, case["clusters"], A)] + r.normal(0.0, max(DX, n[0]), (A, dims))
            pos = np.mod(pos, size)
        else:
            pos = r.random((A, dims)) * size
        pos = np.minimum(pos, size * (1 - 1e-6)).astype(np.float32)
        x["agents"] = {"positions": pos, "volumes": np.full(A, AGENT_VOLUME, dtype=np.float32),
                       "secretion_rates": uniform(A, S), "uptake_rates": uniform(A, S),
                       "saturation_densities": uniform(A, S), "net_export_rates": np.zeros((A, S), np.float32),
                       "internalized_substrates": np.zeros((A, S), np.float32)}
    return x


class _View:
    """One device buffer of a solver for torch; keeps its owner alive."""

    def __init__(self, owner, pointer, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (pointer, False),
                                         "version": 2}


def _solver(case, seed):
    n, dims, S = _shape(case), case["dims"], case["substrates"]
    x = _inputs(case, seed)
    g = parabiofvm_amd.DeviceSolver(dims, [0] * 3, [v * DX for v in n], [DX] * 3, S, DT, x["D"], x["decay"],
                                    np.zeros(S, dtype=np.float32))
    for (d, m), values in x["faces"].items():
        g.set_boundary(d, m, values, np.ones(S, dtype=np.uint8))
    if x["interior"] is not None:
        g.set_interior(x["interior"][0], x["interior"][1], np.ones(x["interior"][1].shape, dtype=np.uint8))
    if x["agents"] is not None:
        g.set_agents(x["agents"])
    g.set_compute_internalized(case["internalized"])
    g.set_secretion_reduction(case["reduction"])
    g.set_storage(case["storage"])
    g.initialize()
    torch.cuda.synchronize()
    g.store_densities_device(x["densities"].data_ptr())
    g.wait()
    g.store_agents()
    return g


def _buffers(g, case, owner):
    """What a call leaves on the GPU, in place: densities in their storage form, gradients, internalized amounts."""
    b, n, S, dims = g.device_buffers(), _shape(case), case["substrates"], case["dims"]
    out = {}
    if case["kind"] != "gradient":
        typestr = {"f32": "<f4", "f16": "<f2", "bf16": "<i2"}[case["storage"]]
        d = torch.as_tensor(_View(owner, b.densities, (n[2], n[1], n[0], S), typestr), device="cuda")
        out["densities"] = d.view(torch.bfloat16) if case["storage"] == "bf16" else d
    if case["gradient"]:
        shape = (3, n[2], n[1], n[0], S) if dims == 3 else (n[1], n[0], S, dims)
        out["gradients"] = torch.as_tensor(_View(owner, b.gradients, shape, "<f4"), device="cuda")
    if case["internalized"] and case["agents"]:
        shape = (case["agents"], S)
        out["internalized"] = torch.as_tensor(_View(owner, b.internalized_substrates, shape, "<f4"), device="cuda")
    return out


def prepare(case, seed):
    """An initialized solver (or batch) with its data on the GPU.  Steps that keep the agents' sums from an earlier
    step (recompute off) come after a first step that computed them, as in a program's loop."""
    if case["kind"] == "batch":
        parts = _instances(case)
        solvers = [_solver(p, seed * 1000 + i) for i, p in enumerate(parts)]
        batch = parabiofvm_amd.Batch(solvers)
        if case["tuned"]:
            batch.autotune()
        batch.timestep(True, case["gradient"])
        batch.wait()
        out = [_buffers(g, p, batch) for g, p in zip(solvers, parts)]
        return {"case": case, "handle": batch, "out": out}
    g = _solver(case, seed)
    if case["tuned"]:
        g.autotune()
    if case["kind"] == "step" and not case["recompute"]:
        g.timestep(True, case["gradient"])
    g.wait()
    return {"case": case, "handle": g, "out": _buffers(g, case, g)}


def run(state):
    case, handle = state["case"], state["handle"]
    if case["kind"] == "batch":
        handle.timestep(False, case["gradient"])
    elif case["kind"] == "gradient":
        handle.gradient()
    elif case["kind"] == "cell":
        handle.cell(True)
    else:
        handle.timestep(case["recompute"], case["gradient"])
    return state["out"]


def work(case):
    """Densities read and written once (gradients alone: read), gradients written, agents' terms read and their
    internalized amounts updated, Dirichlet values read; secretion alone touches the agents' voxels only.
    Operations: about 5 per element and sweep, 2 per gradient component, 12 per agent and substrate."""
    if case["kind"] == "batch":
        parts = [work(p) for p in _instances(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    n, S, A, dims = _shape(case), case["substrates"], case["agents"], case["dims"]
    V = n[0] * n[1] * n[2]
    e = 4 if case["storage"] == "f32" else 2
    gradient = 4 * dims * V * S if case["gradient"] else 0
    agents = A * (4 * (dims + 1) + S * (16 if case["recompute"] else 12) + S * (8 if case["internalized"] else 0))
    dirichlet = int(V * case["interior"]) * (8 + 5 * S)
    if case["kind"] == "gradient":
        return {"bytes": e * V * S + gradient, "flops": 2 * dims * V * S}
    if case["kind"] == "cell":
        return {"bytes": agents + 2 * e * A * S, "flops": 12 * A * S}
    return {"bytes": 2 * e * V * S + gradient + agents + dirichlet,
            "flops": (5 * dims + (2 * dims if case["gradient"] else 0)) * V * S + 12 * A * S}


# ---- the same calls in 64 bits -------------------------------------------------------------------------------------


def _exact_dirichlet(d, x, case):
    flat = d.view(-1, case["substrates"])
    for (axis, m), values in x["faces"].items():  # x-, x+, y-, y+, z-, z+
        d.select(2 - axis, d.shape[2 - axis] - 1 if m else 0).copy_(torch.from_numpy(values).double().cuda())
    if x["interior"] is not None:
        flat[torch.from_numpy(x["interior"][2]).cuda()] = torch.from_numpy(x["interior"][1]).double().cuda()


def _exact_sweep(d, x, case, axis):
    """Thomas algorithm along one axis (0 = x) of d [z][y][x][s], in place."""
    n, dims, dt = d.shape[2 - axis], case["dims"], float(np.float32(DT))
    decay, r = x["decay"].astype(np.float64) * dt / dims, dt * x["D"].astype(np.float64) / DX**2
    if n == 1:
        d /= torch.from_numpy(1 + decay).cuda()
        return
    b, e = np.empty((n, r.size)), np.empty((n, r.size))
    for i in range(n):
        b[i] = 1 + decay + (r if i in (0, n - 1) else 2 * r)
        if i:
            e[i] = -r * b[i - 1]
            b[i] += r * e[i]
        b[i] = 1 / b[i]
    b, e, c = torch.from_numpy(b).cuda(), torch.from_numpy(e).cuda(), torch.from_numpy(-r).cuda()
    row = [d.select(2 - axis, i) for i in range(n)]
    for i in range(1, n):
        row[i].addcmul_(row[i - 1], e[i], value=-1)
    row[n - 1].mul_(b[n - 1])
    for i in range(n - 2, -1, -1):
        row[i].addcmul_(row[i + 1], c, value=-1).mul_(b[i])


def _exact_cell(d, x, case, internalized):
    a = {k: torch.from_numpy(v).cuda() for k, v in x["agents"].items()}
    n, S, vv, dt = _shape(case), case["substrates"], float(DX**3), float(np.float32(DT))
    voxel = torch.from_numpy((x["agents"]["positions"] / np.float32(DX)).astype(np.int64)).cuda()  # FP32 decides it
    lin = torch.zeros(case["agents"], dtype=torch.long, device="cuda")
    for axis in reversed(range(case["dims"])):
        lin = lin * n[axis] + voxel[:, axis]
    share = a["volumes"].double()[:, None] * dt / vv
    num = a["secretion_rates"].double() * a["saturation_densities"].double() * share
    den = (a["uptake_rates"].double() + a["secretion_rates"].double()) * share
    flat = d.view(-1, S)
    internalized -= vv * (num - den * flat[lin]) / (1 + den)
    at, inverse = torch.unique(lin, return_inverse=True)
    sums = [torch.zeros(at.numel(), S, dtype=torch.double, device="cuda").index_add_(0, inverse, v) for v in (num, den)]
    flat[at] = (flat[at] + sums[0]) / (1 + sums[1])


def _exact_gradient(d, dims):
    parts = []
    for axis in range(dims):
        v = d.movedim(2 - axis, 0)
        g = torch.empty_like(v)
        g[1:-1] = (v[2:] - v[:-2]) / (2 * DX)
        g[0], g[-1] = (v[1] - v[0]) / DX, (v[-1] - v[-2]) / DX
        parts.append(g.movedim(0, 2 - axis))
    return torch.stack(parts) if dims == 3 else torch.stack(parts, dim=-1)[0]


def _exact_scale(x, case):
    """The storage scale of each substrate: FP16 keeps value * 2^k with the largest of the initial densities, the
    Dirichlet values and the agents' targets in [2^10, 2^11)."""
    S = case["substrates"]
    if case["storage"] != "f16":
        return torch.ones(S, dtype=torch.double, device="cuda")
    most = x["densities"].view(-1, S).amax(0).cpu().numpy()
    for values in list(x["faces"].values()) + ([x["interior"][1]] if x["interior"] is not None else []):
        most = np.maximum(most, values.reshape(-1, S).max(0))
    return torch.from_numpy(np.ldexp(1.0, 11 - np.frexp(most)[1])).cuda()


def exact(case, seed):
    if case["kind"] == "batch":
        return [exact(p, seed * 1000 + i) for i, p in enumerate(_instances(case))]
    n, S, dims = _shape(case), case["substrates"], case["dims"]
    x = _inputs(case, seed)
    scale = _exact_scale(x, case)
    d = x.pop("densities").view(n[2], n[1], n[0], S).double()
    if case["storage"] != "f32":  # the call starts from the stored values
        kept = torch.float16 if case["storage"] == "f16" else torch.bfloat16
        d = (d * scale).to(kept).double() / scale
    if case["kind"] == "gradient":
        return {"gradients": _exact_gradient(d, dims)}
    internalized = torch.zeros(case["agents"], S, dtype=torch.double, device="cuda")
    for _ in range(1 if case["kind"] == "cell" or case["recompute"] else 2):
        if case["agents"]:
            _exact_cell(d, x, case, internalized)
        if case["kind"] == "cell":
            break
        _exact_dirichlet(d, x, case)
        for axis in range(dims):
            _exact_sweep(d, x, case, axis)
            _exact_dirichlet(d, x, case)
    out = {"densities": d * scale}
    if case["gradient"]:
        out["gradients"] = _exact_gradient(d, dims)
    if case["internalized"] and case["agents"]:
        out["internalized"] = internalized
    return out
