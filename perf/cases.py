"""The work a user has this framework do, as cases that can be timed.

Each case is one pass through the public entry points of phenlei_amd on data
that a user's program has in hand: a grid with its device context, a start
state (a restart, or the network's prediction), the warm-start network with
its weights and graph.  `listed` gives a fixed set, `draw` more of the same
ranges, `prepare` the data before a pass, `run` one pass with its whole
results, `work` the bytes and operations a pass cannot do without, and
`exact` the network's results in 64-bit arithmetic by plain torch.

Solver passes load a start state, run a chunk of outer iterations (a solve
checks its residual every 32 steps) and read the state back, as a driver that
restarts, judges or writes files between chunks does.  The context of a grid is
a program's to keep for as many start states as it has, so the states of one
case share it; every pass loads all the state that its iterations read.
"""
import json
import os

import numpy as np
import torch

import phenlei_amd as pa
from phenlei_amd import warmstart as ws

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
RAE2822 = os.path.join(ROOT, "tests", "golden", "rae2822_hybrid2d__4_0.fts")
LAYERS = 6  # the network's depth in training, inference and the shipped weights


def listed():
    """Fixed cases over the range of use."""
    return [
        # the smallest grid of the tests and of the smoke run: launches and level latency are all there is
        dict(name="hex_512", kind="hex", nx=16, ny=8, nz=4, steps=32),
        # the reference's CPU-runnable channel, the case users start with
        dict(name="hex_16k", kind="hex", nx=64, ny=32, nz=8, steps=32),
        # one case of an inviscid sweep at its own size, ragged in every direction
        dict(name="hex_254k", kind="hex", nx=127, ny=77, nz=26, steps=32),
        # laminar flow over a hybrid grid (prism layers and tetrahedra), the 1M-cell configuration
        dict(name="hybrid_1m", kind="hybrid", nx=128, nz=16, n_prism=15, n_tet=77, steps=32, precision=0),
        # the mixed-precision form on a smaller hybrid grid of odd sizes
        dict(name="hybrid_mixed_135k", kind="hybrid", nx=61, nz=9, n_prism=13, n_tet=37, steps=32, precision=1),
        # RANS of the swept wing with its wall forces, the production workload
        dict(name="wing_sa_2m", kind="wing", n_chord=60, n_span=30, n_prism=30, n_tet=29, steps=32),
        # a sweep of inviscid cases solved together in the mixed form
        dict(name="batch_16", kind="batch", cases=16, n_min=50000, n_max=150000, grid_seed=20241202, steps=32),
        # the reference's own 2-D example: node gradients, several LU-SGS sweep pairs (eager launches)
        dict(name="rae2822", kind="rae2822", mach=0.2, sweeps=5, venkat=50.0, cfl=100.0, steps=32),
        # a host solver that calls the hooks one by one, least-squares gradient
        dict(name="hooks_81k", kind="hooks", nx=47, nz=11, n_prism=11, n_tet=23, steps=8),
        # the warm-start network's prediction for one grid of a sweep, FP32
        dict(name="net_forward_200k", kind="net", nx=64, ny=56, nz=56, bf16=0, train=0),
        # the same with BF16 hidden layers on a larger grid of odd size
        dict(name="net_bf16_622k", kind="net", nx=151, ny=71, nz=58, bf16=1, train=0),
        # one training step's loss and gradients
        dict(name="net_gradient_123k", kind="net", nx=79, ny=39, nz=40, bf16=0, train=1),
    ]


def _log(rng, a, b):
    return int(round(a * (b / a) ** rng.random()))


def draw(rng):
    """One more case of the ranges above."""
    kind = rng.choice(["hex", "hex", "hybrid", "hybrid", "wing", "batch", "rae2822", "hooks", "net", "net", "net"])
    if kind == "hex":
        nz = _log(rng, 4, 40)
        return dict(kind=kind, nx=rng.randint(4 * nz, 8 * nz), ny=rng.randint(2 * nz, 4 * nz), nz=nz, steps=32)
    if kind == "hybrid":
        nx = _log(rng, 24, 128)
        return dict(kind=kind, nx=nx, nz=rng.randint(5, 16), n_prism=rng.randint(8, 16), n_tet=rng.randint(20, 77),
                    steps=32, precision=rng.randint(0, 1))
    if kind == "wing":
        nc = _log(rng, 16, 56)
        return dict(kind=kind, n_chord=nc, n_span=max(8, nc // 2 + rng.randint(-2, 2)), n_prism=rng.randint(12, 30),
                    n_tet=rng.randint(8, 29), steps=32)
    if kind == "batch":
        lo = _log(rng, 4000, 50000)
        return dict(kind=kind, cases=rng.randint(3, 16), n_min=lo, n_max=3 * lo, grid_seed=rng.randint(1, 10**6),
                    steps=32)
    if kind == "rae2822":
        return dict(kind=kind, mach=round(rng.uniform(0.2, 0.73), 3), sweeps=rng.randint(2, 5),
                    venkat=rng.choice([5.0, 50.0]), cfl=rng.choice([30.0, 100.0]), steps=rng.randint(8, 32))
    if kind == "hooks":
        return dict(kind=kind, nx=rng.randint(20, 64), nz=rng.randint(5, 12), n_prism=rng.randint(8, 15),
                    n_tet=rng.randint(15, 40), steps=8)
    nz = _log(rng, 8, 56)
    train = rng.randint(0, 1)
    return dict(kind=kind, nx=rng.randint(2 * nz, 3 * nz) if not train else rng.randint(nz, 2 * nz),
                ny=rng.randint(nz, 2 * nz) if nz < 50 else nz + rng.randint(0, 9), nz=nz, bf16=0 if train else
                rng.randint(0, 1), train=train)


# ---------------------------------------------------------------- contexts
_kept = {}


def _keep(case, make):
    """The grid and context of a case's geometry, built once for its states."""
    key = json.dumps({k: v for k, v in case.items() if k not in ("name", "steps")}, sort_keys=True)
    if key not in _kept:
        _kept.clear()
        _kept[key] = make(case)
    return _kept[key]


def _batch_cases(case):
    """(nx, ny, nz, bump, mach, alpha) of each case of a sweep: cells drawn
    between n_min and n_max with the channel's 8:4:1 aspect."""
    rng = np.random.default_rng(case["grid_seed"])
    out = []
    for _ in range(case["cases"]):
        n = rng.uniform(case["n_min"], case["n_max"])
        nz = max(2, int(round((n / 32.0) ** (1.0 / 3.0))))
        ny = 4 * nz
        out.append((max(4, int(round(n / (ny * nz)))), ny, nz, float(rng.uniform(0.02, 0.08)),
                    float(rng.uniform(0.3, 0.8)), float(rng.uniform(-2.0, 6.0))))
    return out


def _make_solver(case):
    kind = case["kind"]
    if kind == "hex":
        mesh = pa.Mesh.bump_hex(case["nx"], case["ny"], case["nz"], 0.05)
        params = pa.default_params(mach=0.5, cfl_start=10.0, cfl_end=10.0)
    elif kind in ("hybrid", "hooks"):
        mesh = pa.Mesh.bump_hybrid(case["nx"], case["nz"], case["n_prism"], 1e-4, case["n_tet"], 0.1, 1, 0.05)
        params = pa.default_params(mach=0.3, viscous=1, reynolds=5e5, cfl_start=10.0, cfl_end=10.0,
                                   precision=case.get("precision", 0), gradient=1 if kind == "hooks" else 0)
    elif kind == "wing":
        mesh = pa.Mesh.swept_wing(case["n_chord"], case["n_span"], case["n_prism"], 1e-5, case["n_tet"])
        params = ws.wing_params(dict(mach=0.6, alpha=2.0))
    elif kind == "rae2822":
        mesh = pa.Mesh.from_fts(RAE2822)
        params = pa.default_params(mach=case["mach"], alpha_deg=2.79, reynolds=6.5e6, viscous=3, gradient=2,
                                   venkat_k=case["venkat"], cfl_start=0.01, cfl_end=case["cfl"], cfl_vary_step=500,
                                   n_lusgs_sweeps=case["sweeps"])
    elif kind == "batch":
        cs = _batch_cases(case)
        mesh = pa.Mesh.concat([pa.Mesh.bump_hex(nx, ny, nz, h) for nx, ny, nz, h, _, _ in cs])
        params = [pa.default_params(mach=m, alpha_deg=a, cfl_start=10.0, cfl_end=10.0, precision=1)
                  for *_, m, a in cs]
    else:
        raise ValueError(kind)
    return mesh, params, pa.Solver(mesh, params)


def _make_net(case):
    mesh = pa.Mesh.bump_hex(case["nx"], case["ny"], case["nz"], 0.05)
    rng = np.random.default_rng(7)
    net = pa.Mpnn(layers=LAYERS)
    scale = dict(W0=np.sqrt(2.0 / 8), A=0.5 * np.sqrt(1.0 / 128), B=0.5 * np.sqrt(1.0 / 128), Wo=np.sqrt(1.0 / 128),
                 b0=0.1, c=0.1, bo=0.1)
    weights = {k: (scale[k] * rng.standard_normal(shape)).astype(np.float32) for k, shape in net.layout()}
    net.set_params(weights)
    net.set_graph(mesh=mesh)
    net.set_forward_precision(bool(case["bf16"]))
    c = mesh.connectivity()
    nb = c["n_bface"]
    pairs = np.stack([c["left"][nb:], c["right"][nb:]])
    return mesh, net, weights, pairs


def _start(mesh, params, rng):
    """A restart-like state: each case's freestream with a disturbance of up
    to a percent in every cell."""
    plist = params if isinstance(params, list) else [params]
    q = np.empty((5, mesh.n_total))
    for k, p in enumerate(plist):
        cells, ghosts = mesh.case_slices(k) if len(plist) > 1 else (slice(0, mesh.n_cell), slice(mesh.n_cell, None))
        q_inf = ws.freestream(p.mach, p.alpha_deg)
        q[:, ghosts] = q_inf[:, None]
        scale = np.array([1.0, 1.0, 1.0, 0.0 if mesh.dim == 2 else 1.0, q_inf[4]])
        n = cells.stop - cells.start
        q[:, cells] = q_inf[:, None] + 0.01 * scale[:, None] * (2.0 * rng.random((5, n)) - 1.0)
    return q


def _features(case, rng):
    """Features of the flow cases a prediction is asked for on this grid, and
    targets of a training step."""
    mesh = _keep(case, _make_net)[0]
    X = ws.features(mesh, 0.05, float(rng.uniform(0.3, 0.8)), float(rng.uniform(-2.0, 6.0)))
    T = (0.1 * (2.0 * rng.random((mesh.n_cell, 5)) - 1.0)).astype(np.float32)
    return X, T


def prepare(case, seed):
    """What a program holds before the pass: context or network, and inputs
    drawn from the seed."""
    rng = np.random.default_rng(seed)
    if case["kind"] == "net":
        _, net, _, _ = _keep(case, _make_net)
        X, T = _features(case, rng)
        return dict(case=case, net=net, X=X, T=T)
    mesh, params, solver = _keep(case, _make_solver)
    st = dict(case=case, solver=solver, q=_start(mesh, params, rng))
    if case["kind"] in ("wing", "rae2822"):  # a RANS restart: nu~ and the eddy viscosity too
        st["nut"] = 3.0 * (0.9 + 0.2 * rng.random(mesh.n_total))
        st["vist"] = 1e-3 * (0.9 + 0.2 * rng.random(mesh.n_total))
    return st


def run(state):
    """One pass; returns everything it computes."""
    case = state["case"]
    if case["kind"] == "net":
        net = state["net"]
        if case["train"]:
            net.set_data(state["X"], state["T"])
            loss, grad = net.gradient()
            return dict(loss=loss, grad=grad)
        net.set_data(state["X"])
        return dict(y=net.forward())
    s = state["solver"]
    s.set_state(state["q"])
    if "nut" in state:
        s.set_field("nut", state["nut"])
        s.set_field("vist", state["vist"])
    if case["kind"] == "hooks":
        fixed = 0
        for step in range(1, case["steps"] + 1):
            s.load_residuals()
            s.boundary()
            s.gamma_t()
            s.gradient()
            s.limiter()
            s.update_residuals()
            s.spectrum_radius()
            s.time_step(step)
            fixed += s.lusgs()
        return dict(norm=s.residual_norm(), q=s.get_state(), residual=s.get_residual(), fixed=fixed)
    out = dict(history=s.iterate(1, case["steps"]), q=s.get_state())
    if "nut" in state:
        out["nut"] = s.get_field("nut")
        forces = s.forces()
        out["forces"] = np.array([forces[k] for k in ("CL", "CD", "CA_p", "CN_p", "CA_f")])
    return out


# ------------------------------------------------------------------ floors
def _sizes(case):
    """(cells, faces) of a case's grid (the wing's and hybrid's faces to a
    few percent)."""
    kind = case["kind"]
    if kind in ("hex", "net"):
        n = case["nx"] * case["ny"] * case["nz"]
        return n, 3 * n
    if kind in ("hybrid", "hooks"):
        n = case["nx"] * case["nz"] * (2 * case["n_prism"] + 6 * case["n_tet"])
        return n, 2.07 * n
    if kind == "wing":
        n = int(1.9 * case["n_chord"]) * int(1.4 * case["n_span"]) * 2 * (2 * case["n_prism"] + 6 * case["n_tet"])
        return n, 2.15 * n
    if kind == "batch":
        n = sum(c[0] * c[1] * c[2] for c in _batch_cases(case))
        return n, 3 * n
    return 36036, 59370


def work(case):
    """Bytes and operations of one pass.  A solver step reads the state, the
    cell and face geometry and the connectivity once and writes the state; a
    network layer reads and writes each cell's 128 features once."""
    n, f = _sizes(case)
    if case["kind"] == "net":
        dense = 2 * (8 * 128 + LAYERS * 2 * 128 * 128 + 128 * 5)
        if case["train"]:
            return {"bytes": n * (52 + 24 + LAYERS * 3 * 1024), "flops": 3 * n * dense}
        return {"bytes": n * (52 + 24 + LAYERS * 1024), "flops": n * dense}
    steps = case["steps"]
    sa = case["kind"] in ("wing", "rae2822")
    viscous = sa or case["kind"] in ("hybrid", "hooks")
    pairs = case.get("sweeps", 1)
    step_bytes = n * (80 + 48 + (40 if sa else 0)) + f * 64
    step_flops = f * (800 + (350 if viscous else 0) + 120 + 420 * pairs + (150 if sa else 0)) + n * 300
    return {"bytes": steps * step_bytes + 80 * n, "flops": steps * step_flops}


# ------------------------------------------------------------ 64-bit values
def exact(case, seed):
    """The network's results in 64-bit torch on the same inputs.  A solver
    pass (its sweeps run cell after cell) has none in reasonable time."""
    if case["kind"] != "net":
        return None
    _, _, weights, pairs = _keep(case, _make_net)
    X, T = _features(case, np.random.default_rng(seed))
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    p = {k: torch.from_numpy(v.astype(np.float64)).to(dev) for k, v in weights.items()}
    x = torch.from_numpy(X.astype(np.float64)).to(dev)
    pr = torch.from_numpy(pairs.astype(np.int64)).to(dev)
    n = x.shape[0]
    deg = torch.zeros(n, dtype=torch.float64, device=dev)
    one = torch.ones(pr.shape[1], dtype=torch.float64, device=dev)
    deg.index_add_(0, pr[0], one)
    deg.index_add_(0, pr[1], one)
    deg = deg.clamp(min=1.0)[:, None]

    def scatter(v):  # sum over face neighbours
        s = torch.zeros_like(v)
        s.index_add_(0, pr[0], v[pr[1]])
        s.index_add_(0, pr[1], v[pr[0]])
        return s

    h = torch.relu(x @ p["W0"] + p["b0"])
    z0, hs, ms, zs = h, [h], [], []
    for i in range(LAYERS):
        m = scatter(h) / deg
        z = h @ p["A"][i] + m @ p["B"][i] + p["c"][i]
        h = h + torch.relu(z)
        if case["train"]:
            ms.append(m)
            zs.append(z)
            hs.append(h)
    y = h @ p["Wo"] + p["bo"]
    if not case["train"]:
        return dict(y=y.cpu().numpy())
    t = torch.from_numpy(T.astype(np.float64)).to(dev)
    g = {k: torch.zeros_like(v) for k, v in p.items()}
    loss = float(((y - t) ** 2).mean())
    dy = 2.0 * (y - t) / (n * 5)
    g["Wo"], g["bo"] = hs[-1].T @ dy, dy.sum(0)
    dh = dy @ p["Wo"].T.contiguous()
    for i in reversed(range(LAYERS)):
        dz = dh * (zs[i] > 0)
        g["A"][i], g["B"][i], g["c"][i] = hs[i].T @ dz, ms[i].T @ dz, dz.sum(0)
        dh = dh + dz @ p["A"][i].T.contiguous() + scatter((dz @ p["B"][i].T.contiguous()) / deg)
    dz = dh * (z0 > 0)
    g["W0"], g["b0"] = x.T @ dz, dz.sum(0)
    return dict(loss=loss, grad={k: v.cpu().numpy() for k, v in g.items()})
