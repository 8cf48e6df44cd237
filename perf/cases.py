"""The work that users of ndg_cuda_amd have it do, as cases that can be timed and compared: whole
solves, blocks of time steps, receiver records, the adjoint gradient, the error estimator, an
hp-adaptive run and the output interpolation, each through the package's public classes.

A case is a dict of plain values. Every mesh is an nx x ny grid of [-1, 1]^2 in Hilbert order with
seeded vertex jitter; every initial field is a sum of seeded radial pulses. exact() evaluates the
same discretisation with torch in 64 bits, from the mesh description alone.
"""
import math

import numpy as np
import torch

import ndg_cuda_amd as nd
from ndg_cuda_amd import adjoint

CFL = 0.5


def listed():
    return [
        # A whole small solve, 289 steps of a 16 x 16 periodic mesh: launches and latency count.
        {"name": "solve_periodic_16x16_N6", "kind": "solve", "nx": 16, "ny": 16, "N": 6, "bc": "periodic",
         "jitter": 0.0, "precision": "fp64", "graph": "off", "t_end": 0.5},
        # A small ragged mesh with every kind of boundary (inflow reads the stage time).
        {"name": "solve_boundaries_23x19_N4", "kind": "solve", "nx": 23, "ny": 19, "N": 4, "bc": "mixed",
         "jitter": 0.15, "precision": "fp64", "graph": "off", "t_end": 0.6},
        # A mid-size solve between the two regimes, with the step captured as a graph.
        {"name": "solve_graph_64x64_N5", "kind": "solve", "nx": 64, "ny": 64, "N": 5, "bc": "periodic",
         "jitter": 0.1, "precision": "fp64", "graph": "sequential", "t_end": 0.15},
        # The large production run between two outputs: 512 x 512 jittered walls, order 8.
        {"name": "steps_walls_512x512_N8", "kind": "steps", "nx": 512, "ny": 512, "N": 8, "bc": "walls",
         "jitter": 0.15, "precision": "fp64", "graph": "off", "steps": 200},
        # The same kind of run in the FP32 compensated form.
        {"name": "steps_fp32c_384x384_N7", "kind": "steps", "nx": 384, "ny": 384, "N": 7, "bc": "periodic",
         "jitter": 0.0, "precision": "fp32c", "graph": "off", "steps": 200},
        # A small mesh of the highest order.
        {"name": "steps_61x47_N16", "kind": "steps", "nx": 61, "ny": 47, "N": 16, "bc": "walls",
         "jitter": 0.1, "precision": "fp64", "graph": "off", "steps": 100},
        # Orders 4 to 12 by distance to the pulses, tuned and captured with parallel branches.
        {"name": "steps_orders_256x256_N4_12", "kind": "orders", "nx": 256, "ny": 256, "N": 4, "N_max": 12,
         "bc": "walls", "jitter": 0.0, "precision": "fp64", "graph": "parallel", "steps": 200},
        # A forward run of an inversion: pressure at 32 receivers after every step.
        {"name": "receivers_128x128_N8", "kind": "receivers", "nx": 128, "ny": 128, "N": 8, "bc": "periodic",
         "jitter": 0.0, "precision": "fp64", "graph": "off", "steps": 400, "receivers": 32},
        # Its gradient by checkpoints and recomputation.
        {"name": "gradient_128x128_N8", "kind": "gradient", "nx": 128, "ny": 128, "N": 8, "bc": "periodic",
         "jitter": 0.0, "precision": "fp64", "graph": "off", "steps": 200, "receivers": 32, "interval": 50},
        # An hp-adaptive run from the mesh description on: orders raised and elements split.
        {"name": "adaptive_96x96_N4_12", "kind": "adaptive", "nx": 96, "ny": 96, "N": 4, "N_max": 12,
         "bc": "periodic", "jitter": 0.0, "precision": "fp64", "graph": "off", "interval": 20, "t_end": 0.06},
        # The error estimate that decides an adaptation, on a large mesh.
        {"name": "estimate_256x256_N8", "kind": "estimate", "nx": 256, "ny": 256, "N": 8, "bc": "walls",
         "jitter": 0.1, "precision": "fp64", "graph": "off"},
        # One output event: every field, its time derivative and errors on 10 x 10 points an element.
        {"name": "output_96x96_N8", "kind": "output", "nx": 96, "ny": 96, "N": 8, "bc": "periodic",
         "jitter": 0.1, "precision": "fp64", "graph": "off", "points": 10},
    ]


def draw(rng):
    """One more case: any kind, sizes spread over the logarithm of their range, any order."""
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["solve", "solve", "steps", "steps", "orders", "receivers", "gradient", "adaptive",
                       "estimate", "output"])
    c = {"kind": kind, "bc": rng.choice(["periodic", "walls", "mixed"]),
         "jitter": rng.choice([0.0, round(rng.uniform(0.02, 0.2), 3)]), "precision": "fp64",
         "graph": rng.choice(["off", "off", "sequential"])}
    if kind == "solve":
        c.update(nx=size(6, 80), ny=size(6, 80), N=rng.randint(2, 12))
        # some 100 to 300 steps of the CFL size
        steps = rng.randint(100, 300)
        c["t_end"] = round(steps * CFL * 2.0 / max(c["nx"], c["ny"]) * (1 - 2 * c["jitter"]) / c["N"] ** 2, 6)
    elif kind == "steps":
        c.update(N=rng.randint(1, 16), precision=rng.choice(["fp64", "fp64", "fp32c"]))
        top = min(512, int(2000 / (c["N"] + 1)))
        c.update(nx=size(20, top), ny=size(20, top), steps=rng.randint(40, 200))
    elif kind == "orders":
        lo = rng.randint(2, 5)
        c.update(nx=size(24, 256), ny=size(24, 256), N=lo, N_max=lo + 2 * rng.randint(1, 4),
                 precision=rng.choice(["fp64", "fp64", "fp32c"]), graph=rng.choice(["off", "sequential", "parallel"]),
                 steps=rng.randint(40, 200))
    elif kind in ("receivers", "gradient"):
        c.update(nx=size(12, 128), ny=size(12, 128), N=rng.randint(3, 9), bc="periodic",
                 steps=rng.randint(50, 200), receivers=rng.randint(1, 48))
        if kind == "gradient":
            c.update(interval=rng.randint(11, 60))
    elif kind == "adaptive":
        c.update(nx=size(16, 96), ny=size(16, 96), N=rng.randint(3, 5), N_max=12, interval=rng.randint(8, 20))
        c.update(bc="periodic", jitter=0.0)
        c["t_end"] = round(rng.randint(60, 120) * CFL * 2.0 / max(c["nx"], c["ny"]) / c["N"] ** 2, 6)
    elif kind == "estimate":
        c.update(N=rng.randint(2, 16))
        top = min(384, int(2000 / (c["N"] + 1)))
        c.update(nx=size(16, top), ny=size(16, top))
    else:
        c.update(nx=size(8, 128), ny=size(8, 128), N=rng.randint(1, 12), points=rng.randint(2, 12))
    return c


# ---- inputs ----------------------------------------------------------------------------------


def hilbert_cells(nx, ny):
    """The cells of an nx x ny grid in the order of the Hilbert curve over the smallest square of
    a power of two that holds them, as two index arrays."""
    n = 1
    while n < max(nx, ny):
        n *= 2
    d = np.arange(n * n, dtype=np.int64)
    x, y, t, s = np.zeros_like(d), np.zeros_like(d), d.copy(), 1
    while s < n:
        rx = (t // 2) & 1
        ry = (t ^ rx) & 1
        flip = (ry == 0) & (rx == 1)
        x, y = np.where(flip, s - 1 - x, x), np.where(flip, s - 1 - y, y)
        x, y = np.where(ry == 0, y, x), np.where(ry == 0, x, y)
        x, y = x + s * rx, y + s * ry
        t, s = t // 4, 2 * s
    keep = (x < nx) & (y < ny)
    return x[keep], y[keep]


BC_SIDES = {  # bottom, right, top, left
    "walls": (nd.BC_WALL, nd.BC_WALL, nd.BC_WALL, nd.BC_WALL),
    "mixed": (nd.BC_WALL, nd.BC_OUTFLOW, nd.BC_SYMMETRY, nd.BC_INFLOW),
    "periodic": (nd.BC_PERIODIC,) * 4,
}


def description(case, seed):
    """The case's mesh: nodes with jittered interior, elements in Hilbert order with corners bottom
    right, top right, top left, bottom left, and boundary bars against the element edges."""
    nx, ny = case["nx"], case["ny"]
    rng = np.random.default_rng([seed, 1])
    X, Y = np.meshgrid(np.linspace(-1, 1, nx + 1), np.linspace(-1, 1, ny + 1), indexing="ij")
    if case["jitter"]:
        move = rng.uniform(-1, 1, (2, nx - 1, ny - 1)) * case["jitter"]
        X[1:-1, 1:-1] += move[0] * (2.0 / nx)
        Y[1:-1, 1:-1] += move[1] * (2.0 / ny)
    node = np.arange((nx + 1) * (ny + 1)).reshape(nx + 1, ny + 1)
    i, j = hilbert_cells(nx, ny)
    quads = np.stack([node[i + 1, j], node[i + 1, j + 1], node[i, j + 1], node[i, j]], axis=1)
    sides = [np.stack([node[1:, 0], node[:-1, 0]], 1), np.stack([node[-1, 1:], node[-1, :-1]], 1),
             np.stack([node[:-1, -1], node[1:, -1]], 1), np.stack([node[0, :-1], node[0, 1:]], 1)]
    kinds = BC_SIDES[case["bc"]]
    start = np.cumsum([0] + [len(s) for s in sides])
    bar_type = np.concatenate([np.full(len(s), k, dtype=np.int32) for s, k in zip(sides, kinds)])
    donor = np.full(start[-1], -1, dtype=np.int64)
    if case["bc"] == "periodic":
        for s in range(4):
            o = (s + 2) % 4
            donor[start[s]:start[s + 1]] = np.arange(start[o], start[o + 1])
    desc = nd.MeshDescription(np.stack([X.ravel(), Y.ravel()], 1), quads.astype(np.int64),
                              np.concatenate(sides).astype(np.int64), bar_type, donor)
    if case["kind"] == "orders":
        # the refined places belong to the mesh, so that every seed has the same number of unknowns
        c = desc.xy[quads].mean(axis=1)
        p = pulses_of(case, 0)
        d = np.min(np.hypot(c[:, None, 0] - p[None, :, 0], c[:, None, 1] - p[None, :, 1]) / p[None, :, 2], axis=1)
        step = np.select([d < 1.0, d < 2.0, d < 3.0, d < 4.5], [8, 6, 4, 2], 0)
        desc.quad_N = np.minimum(case["N"] + step, case["N_max"]).astype(np.int32)
    return desc


def pulses_of(case, seed):
    """Radial pulses {x0, y0, width, amplitude}: eight narrow ones where orders adapt to them, else
    three wide enough for every order to resolve them, and for the estimate 64 more that no order
    resolves. An adaptive run has the same pulses for every seed but for a shift by whole cells,
    which changes the values of every element and not the number of refined ones."""
    kind, cell = case["kind"], 2.0 / max(case["nx"], case["ny"])

    def some(rng, n, lo, hi):
        return np.column_stack([rng.uniform(-0.7, 0.7, n), rng.uniform(-0.7, 0.7, n), rng.uniform(lo, hi, n),
                                rng.uniform(0.2, 1.0, n)])
    if kind == "adaptive":
        pulses = some(np.random.default_rng([0, 2]), 8, 0.05, 0.2)
        n = np.array([case["nx"], case["ny"]])
        shift = np.random.default_rng([seed, 2]).integers(0, n) * (2.0 / n)
        pulses[:, :2] = (pulses[:, :2] + shift + 1.0) % 2.0 - 1.0
        return pulses
    rng = np.random.default_rng([seed, 2])
    if kind == "orders":
        return some(rng, 8, 0.05, 0.2)
    wide = some(rng, 3, 0.15, 0.4)
    return np.concatenate([wide, some(rng, 64, 0.25 * cell, 0.6 * cell)]) if kind == "estimate" else wide


def receivers_of(case, seed):
    rng = np.random.default_rng([seed, 3])
    n = case["receivers"]
    element = rng.integers(0, case["nx"] * case["ny"], n)
    points = rng.uniform(-0.9, 0.9, (n, 2))
    data = 0.05 * np.sin(np.arange(case["steps"])[:, None] * rng.uniform(0.01, 0.05, n) + rng.uniform(0, 6, n))
    return element, points, data


def frozen_step(case):
    """The step of runs whose step the caller gives: the CFL step of the unjittered cell, with the
    margin that the largest jitter needs."""
    return CFL * 2.0 / max(case["nx"], case["ny"]) * (1 - 2 * case["jitter"]) / case["N"] ** 2


def prepare(case, seed):
    kind = case["kind"]
    desc = description(case, seed)
    pulses = pulses_of(case, seed)
    N_max = case.get("N_max", case["N"])
    ndg = nd.NDG_t(N_max, case.get("points", 5))
    state = {"case": case, "ndg": ndg, "desc": desc, "pulses": pulses, "time": 0.0}
    if kind in ("solve", "adaptive"):
        state["solver"] = nd.Solver2D_t(CFL, [case["t_end"]])
    else:
        state["solver"] = nd.Solver2D_t(CFL, [0.0])
    if kind == "adaptive":
        return state
    mesh = nd.Mesh2D_t(desc, case["N"], N_max, case.get("points", 5), 0, 0, 0, 1e-6, 1e-14, 0.0, ndg)
    mesh.initial_conditions(pulses)
    if kind == "output":  # an output event comes in the middle of a run
        state["solver"].run_steps(mesh, 10)
    mesh.set_precision(case["precision"])
    if case["graph"] == "parallel":
        mesh.autotune(5)
    mesh.set_graph(case["graph"])
    state["mesh"] = mesh
    if kind in ("receivers", "gradient"):
        element, points, data = receivers_of(case, seed)
        state["receivers"] = adjoint.Receivers(element, points)
        state["data"] = data
        state["dt"] = frozen_step(case)
    mesh.synchronize()
    return state


def run(state):
    case, solver, mesh = state["case"], state["solver"], state.get("mesh")
    kind = case["kind"]
    if kind == "solve":
        mesh.initial_conditions(state["pulses"])
        steps = solver.solve(state["ndg"], mesh)
        return {"steps": steps, "time": solver.time_, "state": mesh.get_solution()}
    if kind in ("steps", "orders"):
        state["time"] = solver.run_steps(mesh, case["steps"], state["time"])
        return {"time": state["time"], "state": mesh.get_solution()}
    if kind == "receivers":
        mesh.initial_conditions(state["pulses"])
        records = adjoint.record_receivers(mesh, state["receivers"], state["dt"], case["steps"])
        return {"records": records, "state": mesh.get_solution()}
    if kind == "gradient":
        J, gp, gu, gv, gc = adjoint.adjoint_gradient(mesh, state["receivers"], state["dt"], case["steps"],
                                                     case["interval"], state["data"])
        return {"J": J, "gradient": (gp, gu, gv), "dc": gc}
    if kind == "adaptive":
        mesh = nd.Mesh2D_t(state["desc"], case["N"], case["N_max"], 5, 1, case["interval"], 0, 1e-6, 1e-14, 0.0,
                           state["ndg"])
        mesh.initial_conditions(state["pulses"], period=(2.0, 2.0))
        steps = solver.solve(state["ndg"], mesh)
        out = {"steps": steps, "orders": mesh.orders_, "state": mesh.get_solution(),
               "points": mesh.get_interpolated_solution()}
        mesh.close()
        return out
    if kind == "estimate":
        error, sigma, refine, coarsen = mesh.estimate_error()
        return {"error": error, "sigma": sigma, "refine": refine, "coarsen": coarsen}
    return mesh.get_complete_solution(0.1)


# ---- what a pass cannot do without -----------------------------------------------------------


def work(case):
    """Bytes and operations of one pass. A stage reads the state, the RK register (but at the
    step's first stage), the neighbours' traces and the geometry, and writes the state and the
    register (but at the last), in 8-byte values, or 4-byte values with a low word of the state in
    the FP32 form. The transposed stages of a gradient are counted as forward stages with the stage
    input read too, and the forward pass twice (once recomputed)."""
    K, N = case["nx"] * case["ny"], case["N"]
    orders = np.full(K, N)
    kind = case["kind"]
    if kind == "orders":
        orders = description(case, 0).quad_N.astype(np.int64)
    nf = orders + 1.0
    values = float((3 * nf * nf).sum())
    traces = float((12 * nf).sum())
    if case["precision"] == "fp32c":
        stage_bytes = values * (8 * 2 + 4 * 4 / 3) + traces * 4 + 80 * K
    else:
        stage_bytes = values * (8 * 2 + 8 * 4 / 3) + traces * 8 + 80 * K
    # contractions along both directions, lifts, fluxes and metrics, and the update
    stage_flops = float((12 * nf ** 3 + 90 * nf * nf + 100 * nf).sum())
    if kind in ("solve", "adaptive"):
        # element sizes vary with the jitter; the count of the unjittered mesh stands for all
        steps = math.ceil(case["t_end"] / (CFL * 2.0 / max(case["nx"], case["ny"]) / N ** 2))
    else:
        steps = case.get("steps", 0)
    out = values * 8
    if kind in ("solve", "steps", "orders", "adaptive"):
        return {"bytes": 3 * steps * stage_bytes + out, "flops": 3 * steps * stage_flops}
    if kind == "receivers":
        return {"bytes": 3 * steps * stage_bytes + out + 8 * steps * case["receivers"],
                "flops": 3 * steps * stage_flops}
    if kind == "gradient":
        return {"bytes": 3 * steps * (3 * stage_bytes + 8 * values) + out, "flops": 3 * steps * 3 * stage_flops}
    if kind == "estimate":
        modes = min(N + 1, 4)
        # the spectra's coefficients by one contraction per direction
        return {"bytes": values / 3 * 8 + K * 25, "flops": K * 2.0 * modes * ((N + 1) ** 2 + (N + 1) ** 2) * 2}
    n = case["points"]
    points = K * n * n
    per_field = 2.0 * ((N + 1) ** 2 * n + (N + 1) * n * n)
    return {"bytes": stage_bytes + points * 88.0 + 84.0 * K, "flops": stage_flops + K * 9 * per_field}


# ---- the same discretisation in 64 bits ------------------------------------------------------


class Rule:
    """Legendre-Gauss nodes, weights, the weak derivative matrix and end-point values of an order."""

    def __init__(self, N, device):
        x, w = np.polynomial.legendre.leggauss(N + 1)
        self.N, self.x, self.w = N, x, w
        self.bary = np.array([1.0 / np.prod(x[i] - np.delete(x, i)) for i in range(N + 1)])
        D = np.zeros((N + 1, N + 1))
        for i in range(N + 1):
            for j in range(N + 1):
                if i != j:
                    D[i, j] = self.bary[j] / self.bary[i] / (x[i] - x[j])
            D[i, i] = -D[i].sum()
        at = [self.at([-1.0])[0], self.at([1.0])[0]]

        def move(a):
            return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=device)
        self.Dh = move(-(D.T * w[None, :]) / w[:, None])
        self.ends = move(np.stack(at))           # values at -1 and +1
        self.lift = move(np.stack(at) / w)       # and divided by the weights
        self.nodes = move(x)

    def at(self, points):
        """Lagrange polynomials at points, [point][node]."""
        rows = []
        for p in points:
            d = p - self.x
            hit = np.abs(d) < 1e-15
            rows.append(hit.astype(float) if hit.any() else (self.bary / d) / (self.bary / d).sum())
        return np.array(rows)


class Reference:
    """The DG-SEM operator on a description of quadrilaterals, elements grouped by order."""

    def __init__(self, desc, N):
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        K = len(desc.quads)
        order = np.full(K, N) if desc.quad_N is None else np.asarray(desc.quad_N).astype(np.int64)
        self.K, self.order = K, order
        xy, quads = np.asarray(desc.xy), np.asarray(desc.quads)
        P = xy[quads]
        ends = np.stack([quads, np.roll(quads, -1, axis=1)], axis=2).reshape(-1, 2)
        edge = ends.min(axis=1) * len(xy) + ends.max(axis=1)
        by = np.argsort(edge, kind="stable")
        pair = edge[by][:-1] == edge[by][1:]
        nb = np.full(4 * K, -1)
        nb[by[:-1][pair]], nb[by[1:][pair]] = by[1:][pair], by[:-1][pair]
        bars, bar_type = np.asarray(desc.bars), np.asarray(desc.bar_type)
        bar_edge = bars.min(axis=1) * len(xy) + bars.max(axis=1)
        bar_side = by[np.searchsorted(edge[by], bar_edge)]
        kind = np.zeros(4 * K, dtype=np.int64) - 1
        periodic = bar_type == nd.BC_PERIODIC
        kind[bar_side[~periodic]] = bar_type[~periodic]
        nb[bar_side[periodic]] = bar_side[np.asarray(desc.bar_donor)[periodic]]
        edge_vec = np.roll(P, -1, axis=1) - P
        length = np.hypot(edge_vec[..., 0], edge_vec[..., 1])
        diag = np.minimum(np.hypot(*(P[:, 1] - P[:, 3]).T), np.hypot(*(P[:, 2] - P[:, 0]).T))
        self.delta_min = np.minimum(length.min(axis=1), diag)

        def move(a, dtype=torch.float64):
            return torch.as_tensor(np.ascontiguousarray(a), dtype=dtype, device=self.dev)
        self.rules = {int(n): Rule(int(n), self.dev) for n in np.unique(order)}
        self.groups = []
        place, which = np.zeros(K, dtype=np.int64), np.zeros(K, dtype=np.int64)
        for g, n in enumerate(self.rules):
            mine = np.nonzero(order == n)[0]
            place[mine], which[mine] = np.arange(len(mine)), g
        for g, (n, rule) in enumerate(self.rules.items()):
            mine = np.nonzero(order == n)[0]
            Pg, xn = move(P[mine]), rule.nodes
            xi, eta = xn[None, :, None], xn[None, None, :]

            def line(a, b, c, d, t):  # ((1 - t) (Pa - Pb) + (1 + t) (Pc - Pd)) / 4
                return ((1 - t)[..., None] * (Pg[:, a] - Pg[:, b])[:, None, None] +
                        (1 + t)[..., None] * (Pg[:, c] - Pg[:, d])[:, None, None]) / 4
            d_xi, d_eta = line(1, 0, 2, 3, eta), line(3, 0, 2, 1, xi)
            ev = move(edge_vec[mine])
            le = torch.linalg.vector_norm(ev, dim=2)
            sides = (4 * mine[:, None] + np.arange(4)).reshape(-1)
            out = nb[sides]
            same = (out >= 0) & (which[out // 4] == g)
            G = {"N": n, "rule": rule, "mine": move(mine, torch.int64), "P": Pg, "x_xi": d_xi[..., 0],
                 "y_xi": d_xi[..., 1], "x_eta": d_eta[..., 0], "y_eta": d_eta[..., 1], "half": le / 2,
                 "nx": ev[..., 1] / le, "ny": -ev[..., 0] / le,
                 "gather": move(np.where(same, 4 * place[out // 4] + out % 4, 0), torch.int64), "walls": [],
                 "mortars": []}
            G["J"] = G["x_xi"] * G["y_eta"] - G["x_eta"] * G["y_xi"]
            for k in np.unique(kind[sides]):
                if k >= 0:
                    G["walls"].append((int(k), move(np.nonzero(kind[sides] == k)[0], torch.int64)))
            for h, m in enumerate(self.rules):
                other = np.nonzero((out >= 0) & (which[out // 4] == h))[0] if h != g else []
                if len(other):
                    r = self.rules[m]
                    face = rule if n > m else r
                    G["mortars"].append({
                        "sides": move(other, torch.int64), "group": h,
                        "from": move(4 * place[out[other] // 4] + out[other] % 4, torch.int64),
                        "own": move(rule.at(face.x)), "ext": move(r.at(face.x)),
                        "back": move((rule.at(face.x) * face.w[:, None] / rule.w[None, :]).T)})
            self.groups.append(G)

    def pulses(self, pulses):
        fields = []
        for G in self.groups:
            x = G["rule"].nodes
            xi, eta, P = x[None, :, None, None], x[None, None, :, None], G["P"][:, None, None]
            X = (P[..., 0, :] * (1 - xi) * (1 - eta) + P[..., 1, :] * (1 + xi) * (1 - eta) +
                 P[..., 2, :] * (1 + xi) * (1 + eta) + P[..., 3, :] * (1 - xi) * (1 + eta)) / 4
            q = torch.zeros((len(G["mine"]), 3) + X.shape[1:3], dtype=torch.float64, device=self.dev)
            for x0, y0, width, a in pulses:
                r2 = (X[..., 0] - x0) ** 2 + (X[..., 1] - y0) ** 2
                q[:, 0] += a * torch.exp(-math.log(2.0) * r2 / width ** 2)
            fields.append(q)
        return fields

    def step_size(self):
        return float(np.min(CFL * self.delta_min / self.order ** 2))

    def rhs(self, fields, t):
        traces = []
        for G, q in zip(self.groups, fields):
            e = G["rule"].ends
            at_xi = torch.einsum("si,efij->sefj", e, q)    # at xi = -1, +1
            at_eta = q @ e.T                                # [e][f][i][-1, +1]
            traces.append(torch.stack([at_eta[..., 0], at_xi[1], at_eta[..., 1].flip(-1), at_xi[0].flip(-1)], 1))
        out = []
        for G, q, tr in zip(self.groups, fields, traces):
            n1 = G["N"] + 1
            own = tr.reshape(-1, 3, n1)
            nx, ny, half = (G[k].reshape(-1, 1) for k in ("nx", "ny", "half"))
            ext = own[G["gather"]].flip(-1)
            for kind, at in G["walls"]:
                a, x, y, s = own[at], nx[at], ny[at], half[at]
                if kind in (nd.BC_WALL, nd.BC_SYMMETRY):
                    un, ut = a[:, 1] * x + a[:, 2] * y, -a[:, 1] * y + a[:, 2] * x
                    ghost = torch.stack([a[:, 0], -un * x - ut * y, -un * y + ut * x], 1) * s[:, None]
                elif kind == nd.BC_OUTFLOW:
                    ghost = a * s[:, None]
                elif kind == nd.BC_INFLOW:
                    e, k = at // 4, at % 4
                    x1 = (1 + G["rule"].nodes)[None, :, None] / 2
                    X = G["P"][e, k][:, None] * (1 - x1) + G["P"][e, (k + 1) % 4][:, None] * x1
                    kx = 0.707106781186548
                    arg = kx * (X[..., 0] + 0.2) + kx * (X[..., 1] + 0.2) - t
                    p = torch.exp(-arg ** 2 / 0.120112240878645 ** 2)
                    ghost = torch.stack([p, kx * p, kx * p], 1)
                else:
                    ghost = torch.zeros_like(a)
                ext = ext.index_copy(0, at, ghost)
            flux = self.flux(own, ext, nx, ny) * half[:, None]
            for m in G["mortars"]:
                at = m["sides"]
                a = own[at] @ m["own"].T
                b = (traces[m["group"]].reshape(-1, 3, m["ext"].shape[1])[m["from"]] @ m["ext"].T).flip(-1)
                f = self.flux(a, b, nx[at], ny[at]) @ m["back"].T
                flux = flux.index_copy(0, at, f * half[at][:, None])
            F = flux.reshape(-1, 4, 3, n1)
            p, u, v = q[:, 0], q[:, 1], q[:, 2]
            A = torch.stack([G["y_eta"] * u - G["x_eta"] * v, G["y_eta"] * p, -G["x_eta"] * p], 1)
            B = torch.stack([-G["y_xi"] * u + G["x_xi"] * v, -G["y_xi"] * p, G["x_xi"] * p], 1)
            lift, Dh = G["rule"].lift, G["rule"].Dh
            d = torch.matmul(Dh, A) + torch.matmul(B, Dh.T)
            d = d + lift[1][:, None] * F[:, 1, :, None, :] + lift[0][:, None] * F[:, 3].flip(-1)[:, :, None, :]
            d = d + F[:, 2].flip(-1)[..., None] * lift[1] + F[:, 0][..., None] * lift[0]
            out.append(-d / G["J"][:, None])
        return out

    @staticmethod
    def flux(a, b, nx, ny):
        wl = a[:, 0] + a[:, 1] * nx + a[:, 2] * ny
        wr = b[:, 0] - b[:, 1] * nx - b[:, 2] * ny
        return torch.stack([(wl - wr) / 2, nx * (wl + wr) / 2, ny * (wl + wr) / 2], 1)

    def step(self, fields, t, dt, c=1.0):
        reg = [torch.zeros_like(q) for q in fields]
        for a, b, g in ((0.0, 0.0, 1 / 3), (-5 / 9, 1 / 3, 15 / 16), (-153 / 128, 3 / 4, 8 / 15)):
            G = self.rhs(fields, t + b * dt)
            reg = [a * r + c * d for r, d in zip(reg, G)]
            fields = [q + g * dt * r for q, r in zip(fields, reg)]
        return fields

    def packed(self, fields):
        """Fields p, u, v of every element one after another, in the description's order."""
        size = (self.order + 1) ** 2
        start = np.cumsum(size) - size
        out = [torch.empty(int(size.sum()), dtype=torch.float64, device=self.dev) for _ in range(3)]
        for G, q in zip(self.groups, fields):
            first = torch.as_tensor(start, device=self.dev)[G["mine"]]
            at = first[:, None] + torch.arange((G["N"] + 1) ** 2, device=self.dev)
            for f in range(3):
                out[f][at] = q[:, f].reshape(len(at), -1)
        return tuple(o.cpu().numpy() for o in out)


def exact(case, seed):
    kind = case["kind"]
    if kind == "adaptive":  # the mesh follows the run
        return None
    K, N = case["nx"] * case["ny"], case["N"]
    if case.get("steps", 100) * K * (N + 1) ** 2 > 6e9:
        return None
    desc = description(case, seed)
    ref = Reference(desc, N)
    with torch.set_grad_enabled(kind == "gradient"):
        q = ref.pulses(pulses_of(case, seed))
        if kind == "estimate":
            # the decay rate is a fit through logarithms of coefficients at rounding level where the
            # field is smooth or zero: no value of its own there
            return {"error": estimate(ref, q[0]), "sigma": None, "refine": None, "coarsen": None}
        if kind == "output":
            t, dt = 0.0, ref.step_size()
            for _ in range(10):
                q, t = ref.step(q, t, dt), t + dt
            return output(case, ref, q[0])
        if kind == "solve":
            t, dt0, steps = 0.0, ref.step_size(), 0
            while t < case["t_end"]:
                dt = min(dt0, case["t_end"] - t) if t + dt0 > case["t_end"] else dt0
                q, t, steps = ref.step(q, t, dt), t + dt, steps + 1
            return {"steps": steps, "time": t, "state": ref.packed(q)}
        if kind in ("steps", "orders"):
            t, dt = 0.0, ref.step_size()
            for _ in range(case["steps"]):
                q, t = ref.step(q, t, dt), t + dt
            return {"time": t, "state": ref.packed(q)}
        element, points, data = receivers_of(case, seed)
        rule, dt = ref.rules[N], frozen_step(case)
        wx, wy = (torch.as_tensor(rule.at(points[:, k]), device=ref.dev) for k in (0, 1))
        element = torch.as_tensor(element, device=ref.dev)

        def record(q):
            return torch.einsum("rij,ri,rj->r", q[0][element, 0], wx, wy)
        if kind == "receivers":
            rows = []
            for _ in range(case["steps"]):
                q = ref.step(q, 0.0, dt)
                rows.append(record(q))
            return {"records": torch.stack(rows).cpu().numpy(), "state": ref.packed(q)}
        return gradient(case, ref, q[0], record, torch.as_tensor(data, device=ref.dev), dt)


def gradient(case, ref, q0, record, data, dt):
    """Reverse-mode gradient of the misfit, one block of steps kept at a time."""
    block, steps = 5, case["steps"]
    starts, q = [], q0
    with torch.no_grad():
        for n in range(steps):
            if n % block == 0:
                starts.append(q)
            q = ref.step([q], 0.0, dt)[0]
    J, lam, dc = 0.0, torch.zeros_like(q0), 0.0
    for b in range(len(starts) - 1, -1, -1):
        q = first = starts[b].detach().requires_grad_(True)
        c = torch.ones((), dtype=torch.float64, device=ref.dev, requires_grad=True)
        misfit = 0.0
        for n in range(b * block, min(steps, (b + 1) * block)):
            q = ref.step([q], 0.0, dt, c)[0]
            misfit = misfit + ((record([q]) - data[n]) ** 2).sum() / 2
        lam, g = torch.autograd.grad(misfit + (q * lam).sum(), (first, c))
        J, dc = J + float(misfit.detach()), dc + float(g)
    return {"J": J, "gradient": ref.packed([lam]), "dc": dc}


def estimate(ref, q):
    """Error of the pressure from the last min(N + 1, 4) modes (all with the larger index of the two
    directions equal) and the decay fitted through them."""
    G = ref.groups[0]
    rule, N = G["rule"], G["N"]
    V = np.polynomial.legendre.legvander(rule.x, N)
    M = torch.as_tensor((V * rule.w[:, None]).T * (np.arange(N + 1) + 0.5)[:, None], device=ref.dev)
    modes = (M @ q[:, 0] @ M.T).abs()
    n = min(N + 1, 4)
    spec = []
    for k in range(N + 1 - n, N + 1):
        spec.append(modes[:, :k, k].sum(1) + modes[:, k, :k].sum(1) + modes[:, k, k])
    spec = torch.stack(spec, 1)
    at = torch.arange(N + 1 - n, N + 1, dtype=torch.float64, device=ref.dev)
    logs = spec.log()
    xa, ya = at.mean(), logs.mean(1)
    slope = ((at - xa) * (logs - ya[:, None])).sum(1) / ((at - xa) ** 2).sum()
    C, sigma = (ya - slope * xa).exp(), slope.abs()
    return (spec[:, -1] ** 2 + C ** 2 * 0.5 / sigma * (-2 * sigma * (N + 1)).exp()).sqrt().cpu().numpy()


def output(case, ref, q):
    G, n, t = ref.groups[0], case["points"], 0.1
    rule, P, K = G["rule"], G["P"][:, None, None], ref.K
    x = rule.nodes

    def mapped(xi, eta):
        return (P[..., 0, :] * (1 - xi) * (1 - eta) + P[..., 1, :] * (1 + xi) * (1 - eta) +
                P[..., 2, :] * (1 + xi) * (1 + eta) + P[..., 3, :] * (1 - xi) * (1 + eta)) / 4
    X = mapped(x[None, :, None, None], x[None, None, :, None])
    kx = 0.707106781186548
    p = torch.exp(-(kx * (X[..., 0] + 0.2) + kx * (X[..., 1] + 0.2) - t) ** 2 / 0.120112240878645 ** 2)
    wave = torch.stack([p, kx * p, kx * p], 1)
    grid = np.linspace(-1, 1, n)
    I = torch.as_tensor(rule.at(grid), device=ref.dev)
    s = torch.as_tensor(grid, device=ref.dev)
    XY = mapped(s[None, :, None, None], s[None, None, :, None])

    def points(f):
        return (I @ f @ I.T).cpu().numpy()
    d, w = ref.rhs([q], t)[0], (wave - q).abs()
    out = {"x": XY[..., 0].cpu().numpy(), "y": XY[..., 1].cpu().numpy()}
    for k, name in enumerate("puv"):
        out[name] = points(q[:, k])
        out["d%s_dt" % name] = points(d[:, k])
        out["%s_analytical_error" % name] = points(w[:, k])
        out["%s_error" % name] = out["%s_sigma" % name] = None
    out.update(N=np.full(K, G["N"], dtype=np.int32), refine=None, coarsen=None, split_level=None, status=None,
               rotation=None)
    return out
