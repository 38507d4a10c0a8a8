"""The calls whose time matters to a user of this framework, with their inputs, outputs, least work and exact answers.

A case is one call (or the few calls of one time step) of an ocean or shallow-water run: the explicit step, the
split-explicit step with its implicit free surface, the multi-level step, the column physics after a step, and the
free-surface solve and its network by themselves.  Sizes are those of this repository's configurations: J5 shallow
water with one layer, the J7 ocean with 20 layers, the J8 ocean with 30, ensembles and hierarchies of them, and odd
layer counts between.

The prognostic state lives on the device and is returned as it lies there (wtg_state_device_ptrs); fields that the API
hands out on the host (the free surface, the network's gradients) come back as host arrays, as a program gets them.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import wavetrisk_hydrostatic_amd as W
from wavetrisk_hydrostatic_amd import cases as C
from wavetrisk_hydrostatic_amd import learned as LC

GRAV, RHO0 = 9.80616, 1028.0
DIFFUSION_VISC = {1: (1e3, 1e3, 1e4, 1e4), 2: (1e12, 1e12, 1e13, 1e13)}  # m^2/s and m^4/s, stable on the J8 grid
SOLVE_TOL = 1e-9


def listed():
    return [
        # 100-step shallow-water runs (TC5) on one layer: every launch is tiny, so latency and launches count
        {"name": "sw_J5_L1_graph", "kind": "rk4", "level": 5, "layers": 1, "members": 1, "precision": "fp64", "graph": True,
         "diffusion": 0, "steps": 5},
        # an ordinary ocean with the test cases' hyperdiffusion hooks on an odd number of layers
        {"name": "rk4_J6_L7_hyperdiffusion", "kind": "rk4", "level": 6, "layers": 7, "members": 1, "precision": "fp64",
         "graph": False, "diffusion": 2, "steps": 1},
        # the headline: the explicit ocean step at J8 with 30 layers, FP64 and FP32-bulk
        {"name": "rk4_J8_L30", "kind": "rk4", "level": 8, "layers": 30, "members": 1, "precision": "fp64", "graph": False,
         "diffusion": 0, "steps": 1},
        {"name": "rk4_J8_L30_fp32bulk", "kind": "rk4", "level": 8, "layers": 30, "members": 1, "precision": "bulk",
         "graph": False, "diffusion": 0, "steps": 1},
        # the mode-split ocean step: J7 with V-cycles on its hierarchy, J8 with BiCGSTAB on the one level, and a small
        # FP32-bulk ensemble with learned cycles
        {"name": "split_J7_L20_vcycle", "kind": "split", "level": 7, "layers": 20, "members": 1, "precision": "fp64",
         "solver": "vcycle", "steps": 2},
        {"name": "split_J8_L30_bicgstab", "kind": "split", "level": 8, "layers": 30, "members": 1, "precision": "fp64",
         "solver": "bicgstab", "steps": 2},
        {"name": "split_J7_L11_ensemble", "kind": "split", "level": 7, "layers": 11, "members": 3, "precision": "bulk",
         "solver": "learned", "steps": 2},
        # the same ocean on a full hierarchy of levels, explicit and mode-split
        {"name": "ml_split_J5_J7_L20", "kind": "ml_split", "level": 7, "layers": 20, "steps": 1},
        # a free-surface solve by itself, host right-hand side in and surface out
        {"name": "solve_J7_vcycle", "kind": "solve", "level": 7, "members": 1, "solver": "vcycle"},
        # the column physics after a step
        {"name": "remap_J8_L30_ppr", "kind": "remap", "level": 8, "layers": 30, "members": 1, "scheme": W.REMAP_PPR},
        {"name": "vdiff_J8_L30_tke", "kind": "vdiff", "level": 8, "layers": 30, "members": 1, "tke": True},
        # one gradient of the learned correction's network (its training's forward and backward)
        {"name": "mlp_gradients_4096", "kind": "mlp", "rows": 4096},
    ]


def _layers(rng, level, members=1, least=1):
    """a layer count, spread over its logarithm up to the largest case's nodes x layers"""
    most = min(45, 30 * 4 ** (8 - level) // members)
    return max(least, min(most, int(math.exp(rng.uniform(math.log(least), math.log(most + 1))))))


def draw(rng):
    kind = rng.choice(["rk4", "rk4", "rk4", "split", "split", "ml_rk4", "ml_split", "solve", "remap", "vdiff", "mlp"])
    if kind == "rk4":
        level, diffusion = rng.randint(4, 8), rng.choice([0, 0, 0, 1, 2])
        members = rng.choice([1, 1, 2, 3, 5]) if level < 8 else 1
        graph = rng.random() < 0.4 and not diffusion
        return {"kind": kind, "level": level, "layers": _layers(rng, level, members), "members": members,
                "precision": "fp64" if diffusion else rng.choice(["fp64", "bulk"]), "graph": graph, "diffusion": diffusion,
                "steps": rng.randint(1, 5) if level < 7 else 1}
    if kind == "split":
        level, solver = rng.randint(6, 8), rng.choice(["bicgstab", "vcycle", "learned"])
        members = rng.choice([1, 2, 4]) if level < 8 else 1
        return {"kind": kind, "level": level, "layers": min(30, _layers(rng, level, members)), "members": members,
                "precision": rng.choice(["fp64", "bulk"]), "solver": solver, "steps": rng.randint(1, 2)}
    if kind in ("ml_rk4", "ml_split"):
        level = rng.randint(6, 7)
        return {"kind": kind, "level": level, "layers": min(24, _layers(rng, level)), "steps": 1}
    if kind == "solve":
        level = rng.randint(6, 8)
        return {"kind": kind, "level": level, "members": rng.choice([1, 1, 2, 5]) if level < 8 else 1,
                "solver": rng.choice(["vcycle", "learned"])}
    if kind == "remap":
        level = rng.randint(4, 8)
        members = rng.choice([1, 1, 3]) if level < 8 else 1
        return {"kind": kind, "level": level, "layers": _layers(rng, level, members, 3), "members": members,
                "scheme": rng.choice([W.REMAP_PPR, W.REMAP_PPR, W.REMAP_PIECEWISE_LINEAR, W.REMAP_PIECEWISE_CONSTANT])}
    if kind == "vdiff":
        level = rng.randint(4, 8)
        members = rng.choice([1, 1, 3]) if level < 8 else 1
        return {"kind": kind, "level": level, "layers": _layers(rng, level, members, 3), "members": members,
                "tke": rng.random() < 0.7}
    return {"kind": kind, "rows": int(math.exp(rng.uniform(math.log(100), math.log(20000))))}


# ---- inputs ---------------------------------------------------------------

_grids = {}


def _grid(level, lowest):
    """a program builds its grid once and makes every context from it"""
    if (level, lowest) not in _grids:
        _grids[level, lowest] = W.Grid(level=level, min_level=lowest, domain_level=2)
    return _grids[level, lowest]


def _levels(case):
    """levels of the case's hierarchy, coarse to fine (one level where the call takes one)"""
    hi = case["level"]
    if case["kind"] in ("ml_rk4", "ml_split", "solve") or case.get("solver") in ("vcycle", "learned"):
        return list(range(hi - 2, hi + 1))
    return [hi]


def _case_grids(case):
    ls = _levels(case)
    return [_grid(l, ls[0]) for l in ls]


def _ocean(grid, case, seed):
    """topography [M, NC] and state [M L, ...] of the case's members on one grid"""
    L, M = case["layers"], case.get("members", 1)
    if case["kind"] == "rk4" and L == 1:
        topo, m, t, u = C.tc5(grid, 1, u0=15.0 + seed % 7)
        return np.repeat(topo[None], M, 0), np.repeat(m, M, 0), np.repeat(t, M, 0), np.repeat(u, M, 0)
    topo, m, t, u = C.ocean(grid, L, seed=seed)
    rng = np.random.default_rng(seed + 1)
    if case["kind"] in ("remap", "vdiff"):  # layers that have drifted from their coordinates, the buoyancy with them
        x = grid.array("x") / grid.radius
        a, b = (rng.uniform(-0.04, 0.04, (L, 1)) for _ in range(2))
        f = 1.0 + a * x[2] + b * x[0] * x[1]
        m, t = m * f, t * f * (1.0 + 0.02 * rng.uniform(-1, 1, (L, 1)))
    topos = topo + 50.0 * np.arange(M)[:, None] * np.cos(grid.array("x")[2] / grid.radius)
    if M == 1:
        return topos, m, t, u
    bump = 1.0 + 0.01 * np.arange(M)[:, None, None]
    return topos, (m * bump).reshape(M * L, -1), (t * bump).reshape(M * L, -1), np.tile(u, (M, 1, 1))


def _step(grid, case, topos, mass):
    """time step: half the gravity wave's limit for the explicit step, the ocean's baroclinic step for the split one"""
    if case["kind"] in ("rk4", "ml_rk4"):
        own = grid.layout.owned_edge_cells()
        L = case["layers"]
        depth = float(mass[:L].sum(0).max()) / RHO0
        return 0.5 * float(grid.array("len")[:, own].min()) / (math.sqrt(GRAV * depth) + 30.0)
    return {"split": 900.0, "ml_split": 300.0, "solve": 1800.0}.get(case["kind"], 900.0)


def _targets(L):
    """two hybrid coordinates that a run remaps onto: Chebyshev, and one refined towards the surface"""
    s = np.arange(L + 1) / L
    return [(1.0 - b, b) for b in ((1.0 + np.cos(s * np.pi)) / 2.0, 1.0 - s ** 0.8)]


def _forcing(rng, M, L, NC):
    hooks = dict(bottom_buoy_flux=rng.uniform(-3e-7, 3e-7, M * NC), top_buoy_flux=rng.uniform(-1e-6, 1e-6, M * NC),
                 tau_mag=rng.uniform(0.02, 0.2, M * NC), wind_flux=rng.uniform(-2e-4, 2e-4, (M * 3, NC)))
    coef = (np.full((M * (L + 1), NC), 1.2e-5), np.full((M * (L + 1), NC), 1.2e-4),
            rng.uniform(1e-6, 3e-5, (M * L, 1)) * rng.uniform(0.5, 1.5, NC))
    return hooks, coef


def _solve_fields(grid, members, seed):
    """per member (topography, old free surface, right-hand side) of seeded draws"""
    draws = [LC.draw_fields([grid], seed * 16 + k)[0] for k in range(members)]
    return [np.stack([d[k] for d in draws]) for k in range(3)]


class _Program:
    """the handles that a program keeps; destroyed hierarchy first"""

    def __init__(self):
        self.ctxs, self.h, self.ml, self.mlp = [], None, None, None

    def __del__(self):
        if self.h is not None and self.mlp is not None:
            self.h.set_learned(None)
        for x in [self.ml, self.h, self.mlp] + self.ctxs:
            if x is not None:
                x.close()


class _DeviceArray:
    """device memory of the framework as another library sees it (CUDA array interface), and its owner"""

    def __init__(self, ptr, shape, owner):
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f8", "data": (ptr, False), "version": 3,
                                         "strides": None}
        self.owner = owner


def _resident(state, ctx):
    """mass, temp and velocity of slot 0 where they lie on the device"""
    p = [ctypes.c_void_p() for _ in range(3)]
    if W.load_library().wtg_state_device_ptrs(ctx._h, 0, *map(ctypes.byref, p)) != 0:
        raise RuntimeError("wtg_state_device_ptrs failed")
    key = tuple(x.value for x in p)
    if key not in state["views"]:
        n, nc = ctx.nlayers * ctx.members, ctx.layout.ncells
        state["views"][key] = [torch.as_tensor(_DeviceArray(a, s, state["program"]), device="cuda")
                               for a, s in zip(key, ((n, nc), (n, nc), (n, 3, nc)))]
    return state["views"][key]


def _mg_params(case):
    if case["kind"] == "ml_split":
        return W.MgParams.defaults(coarse_tol=SOLVE_TOL, fine_tol=SOLVE_TOL, coarse_iter=400, max_vcycle=50)
    return W.MgParams.defaults(coarse_tol=1e-2, fine_tol=SOLVE_TOL, coarse_iter=400, max_vcycle=40)


def prepare(case, seed):
    kind, M = case["kind"], case.get("members", 1)
    prog = _Program()
    state = {"case": case, "program": prog, "views": {}, "calls": 0}
    if kind == "mlp":
        rng = np.random.default_rng(seed)
        prog.mlp = W.MLP(max_batch=case["rows"], seed=seed % 1000)
        state["x"], state["t"] = _mlp_rows(rng, case["rows"])
        return state
    grids = _case_grids(case)
    state["params"] = _mg_params(case)
    multi = kind in ("ml_rk4", "ml_split")
    for k, g in enumerate(grids):
        top = k == len(grids) - 1
        full = top or multi
        if kind == "solve":
            topos, eta_old, rhs = _solve_fields(g, M, seed)
            c = W.Context(g, nlayers=1, members=M)
        else:
            sub = case if full else {**case, "layers": 1, "kind": "coarse"}
            topos, m, t, u = _ocean(g, sub, seed)
            c = W.Context(g, nlayers=sub["layers"], members=M, nslots=1)
        prog.ctxs.append(c)
        c.set_topography(topos[0] if M == 1 else topos)
        if kind == "solve":
            c.fs_set_params(_step(g, case, None, None))
            c.fs_upload(W.FS_ETA_OLD, eta_old[0] if M == 1 else eta_old)
            if top:
                state["rhs"] = rhs[0] if M == 1 else rhs
                state["guess"] = np.zeros_like(state["rhs"])
            continue
        if full:
            c.upload_state(0, m, t, u)
        if kind in ("split", "ml_split"):
            c.fs_set_params(_step(grids[-1], case, topos, None), 0.6, 0.8)
            if full:
                eta = m.reshape(M, case["layers"], -1).sum(1) / RHO0 + topos
                c.fs_upload(W.FS_ETA, eta[0] if M == 1 else eta)
    top = prog.ctxs[-1]
    if len(grids) > 1 and kind != "ml_rk4":
        prog.h = W.Hierarchy(prog.ctxs)
        if case.get("solver") == "learned":
            prog.mlp = LC.load_network(prog.h.npatches * M)
            prog.h.set_learned(prog.mlp)
    if multi:
        prog.ml = W.MultiLevel(prog.ctxs)
        prog.ml.forward(0)  # the coarser levels start as the finest one's restrictions
    if case.get("precision") == "bulk":
        top.set_precision(W.PRECISION_FP32_BULK)
        if kind == "rk4":
            top.set_stage_shape(W.SHAPE_LAYER_PAIRS)
    if case.get("graph"):
        top.set_graph(True)
    if case.get("diffusion"):
        top.set_diffusion((case["diffusion"],) * 3, DIFFUSION_VISC[case["diffusion"]])
    if kind in ("rk4", "ml_rk4"):
        state["dt"] = _step(grids[-1], case, topos, m)
    if kind == "remap":
        state["targets"] = _targets(case["layers"])
    if kind == "vdiff":
        hooks, coef = _forcing(np.random.default_rng(seed + 2), M, case["layers"], grids[-1].layout.ncells)
        top.set_vdiff(tke_closure=int(case["tke"]), bottom_friction=4e-4)
        top.vdiff_set_coefficients(*coef)
        top.vdiff_set_forcing(**hooks)
        state["dt"] = _step(grids[-1], case, None, None)
    return state


def _mlp_rows(rng, rows):
    x = rng.standard_normal((rows, W.MLP_IN)).astype(np.float32)
    x[:, 64:] = np.abs(x[:, 64:]) * 0.5
    return x, (0.5 * rng.standard_normal((rows, W.MLP_OUT))).astype(np.float32)


# ---- one pass -------------------------------------------------------------

def run(state):
    case, prog = state["case"], state["program"]
    kind = case["kind"]
    if kind == "mlp":
        loss, grads = prog.mlp.gradients(state["x"], state["t"])
        return [loss, grads]
    top = prog.ctxs[-1]
    if kind == "rk4":
        top.rk4(0, state["dt"], case["steps"])
        return _resident(state, top)
    if kind == "split":
        if prog.h is None:
            top.rk4_split(0, case["steps"], SOLVE_TOL, 400)
        else:
            prog.h.rk4_split(0, case["steps"], W.SOLVE_LEARNED if case["solver"] == "learned" else W.SOLVE_VCYCLE,
                             state["params"])
        return _resident(state, top) + [top.fs_download(W.FS_ETA)]
    if kind == "ml_rk4":
        prog.ml.rk4(0, state["dt"], case["steps"])
        return [_resident(state, c) for c in prog.ctxs]
    if kind == "ml_split":
        prog.ml.rk4_split(prog.h, 0, case["steps"], state["params"])
        return [_resident(state, c) + [c.fs_download(W.FS_ETA)] for c in prog.ctxs]
    if kind == "solve":
        top.fs_upload(W.FS_RHS, state["rhs"])
        top.fs_upload(W.FS_ETA, state["guess"])
        prog.h.solve(W.SOLVE_LEARNED if case["solver"] == "learned" else W.SOLVE_VCYCLE, state["params"])
        return top.fs_download(W.FS_ETA)
    if kind == "remap":  # a run's layers differ from the target at every remap: the two targets in turn
        a, b = state["targets"][state["calls"] % 2]
        state["calls"] += 1
        top.remap(0, case["scheme"], a, b)
        return _resident(state, top)
    top.vertical_diffusion(0, state["dt"], 2)
    return _resident(state, top)


# ---- least work and tolerances ----------------------------------------------

def work(case):
    """Bytes: every stage of a step reads its state and the step's first one and writes the next (a stage reads its
    neighbours' values of the one before, and a state does not fit a cache), and the geometry once a stage; the column
    physics and the solve read their inputs and write their results once.  FLOPs: the operations of the discrete
    equations for each node and layer."""
    kind = case["kind"]
    if kind == "mlp":
        per_row = 2 * (192 * 128 + 128 * 128 + 128 * 64)
        return {"bytes": case["rows"] * (192 + 64) * 4 + 2 * 4 * 49472, "flops": 3 * per_row * case["rows"]}
    M = case.get("members", 1)
    nodes = M * sum(10 * 4 ** l for l in (_levels(case) if kind.startswith("ml") else [case["level"]]))
    if kind == "solve":  # right-hand side, depth, old surface, edge weights read, surface written
        return {"bytes": nodes * 8 * 12, "flops": nodes * 40 * 10}
    nl = nodes * case["layers"]
    stage = nl * 8 * 13.75 + nodes * 8 * 19
    if kind in ("rk4", "ml_rk4") and case.get("precision") == "bulk":
        stage = nl * 80 + nodes * 80
    if kind in ("rk4", "ml_rk4"):
        n = 4 * case["steps"]
        return {"bytes": n * stage, "flops": n * nl * (290 + 120 * case.get("diffusion", 0))}
    if kind in ("split", "ml_split"):
        n = 4 * case["steps"]
        return {"bytes": n * stage + case["steps"] * (nl * 8 * 13 + nodes * 8 * 12), "flops": n * nl * 300}
    if kind == "remap":
        return {"bytes": nl * 8 * 10 + nodes * 8, "flops": nl * 4 * 80}
    reads_writes = 5 + 4 + (6 if case["tke"] else 2)  # m, t, 3 u in, t, 3 u out, Kt, Kv, TKE in and out
    return {"bytes": nl * 8 * reads_writes + nodes * 8 * 16, "flops": nl * (4 * 20 + (60 if case["tke"] else 8))}


def tolerance(case):
    """About four times what the calls differ by from their 64-bit answers (or, multi-level, in another order of sums):
    FP64 steps carry the rounding of pressures into weak velocities, a solve ends at SOLVE_TOL of its right-hand side."""
    kind = case["kind"]
    if kind == "mlp":  # bf16 weights, activations and output gradients
        return {"rel": 1e-2}
    if case.get("precision") == "bulk":
        return {"rel": 2e-7}
    return {"rel": {"rk4": 4e-12, "ml_rk4": 1e-11, "remap": 1e-13, "vdiff": 1e-13}.get(kind, 1e-8)}


# ---- exact answers (plain torch in 64 bits) ----------------------------------

class _Mesh:
    """one level's geometry and ghost maps as torch arrays; neighbours are shifts of the flat cell index"""

    def __init__(self, grid, device):
        lay = grid.layout
        self.n, self.S, self.nc, self.dev = lay.n, lay.S, lay.ncells, device
        put = lambda a: torch.as_tensor(np.array(a), device=device)  # noqa: E731
        self.len, self.ped, self.area = put(grid.array("len")), put(grid.array("pedlen")), put(grid.array("area"))
        self.hinv, self.tri, self.cor = put(grid.array("hex_inv")), put(grid.array("triarea")), put(grid.array("coriolis"))
        src, es, sg = grid.array("node_src"), grid.array("edge_src"), grid.array("edge_sign")
        c = np.arange(self.nc)
        h = np.nonzero((src >= 0) & (src != c))[0]
        self.nd, self.ns = put(h), put(src[h])
        slot = np.arange(3 * self.nc)
        eh = np.nonzero((es >= 0) & (es != slot))[0]
        flat = lambda s: (s % 3) * self.nc + s // 3  # noqa: E731
        self.ed, self.es, self.esg = put(flat(eh)), put(flat(es[eh])), put(sg[eh].astype(float))
        self.owned = put(lay.owned_edge_cells())
        self.masters = put(lay.owned_cells())
        own_ped, own_len = self.ped.clone().reshape(-1), self.len.clone().reshape(-1)
        own_ped[self.ed], own_len[self.ed] = own_ped[self.es], own_len[self.es]
        self.pedf, self.lenf = own_ped.reshape(3, -1), own_len.reshape(3, -1)  # of the edge's owner
        acc, w = [], []
        for o in range(6):  # Qperp weights of the five other edges, starting from each of the six
            part = self.area[o].clone()
            acc = [0.5 - part * self.hinv]
            for i in range(1, 5):
                part = part + self.area[(i + o) % 6]
                acc.append(0.5 - part * self.hinv)
            w.append([a if i % 2 == 0 else -a for i, a in enumerate(acc)])
        self.w = w

    def at(self, f, di, dj):
        return torch.roll(f, -(dj * self.S + di), -1)

    def cells(self, i, j):
        return torch.arange(10, device=self.dev) * self.S * self.S + (j + 2) * self.S + i + 2

    def node_fill(self, f):
        f[..., self.nd] = f[..., self.ns]

    def edge_fill(self, u):
        v = u.reshape(u.shape[:-2] + (-1,))
        v[..., self.ed] = v[..., self.es] * self.esg

    def fill(self, s):
        self.node_fill(s[0])
        self.node_fill(s[1])
        self.edge_fill(s[2])

    def square(self):
        """cells of [0, n]^2 outside the owned ones"""
        n, k = self.n, torch.arange(self.n + 1, device=self.dev)
        edge = [self.cells(int(i), n) for i in k] + [self.cells(n, int(i)) for i in k[:-1]]
        return torch.cat(edge)

    def div(self, F):
        a = self.at
        return (F[0] - a(F[0], -1, 0) + a(F[1], -1, -1) - F[1] + F[2] - a(F[2], 0, -1)) * self.hinv

    def grad(self, q, length):
        a = self.at
        return torch.stack([(a(q, 1, 0) - q) / length[0], (q - a(q, 1, 1)) / length[1], (a(q, 0, 1) - q) / length[2]])

    def mean(self, q):
        a = self.at
        return [0.5 * (q + a(q, 1, 0)), 0.5 * (q + a(q, 1, 1)), 0.5 * (q + a(q, 0, 1))]


def _corner_sums(g, P, vL, vU):
    """circulations of the four merged corner triangles of every lozenge"""
    n, x = g.n, g.cells
    f = lambda e, i, j: P[e][x(i, j)]  # noqa: E731
    return {"mm": f(2, 0, -1) - f(0, -1, 0) + f(0, -1, -1), "pm": -f(0, n, 0) + f(0, n - 1, -1) + f(1, n - 1, -1),
            "mp": f(2, 0, n) - f(1, -1, n - 1) - f(2, -1, n - 1), "pp": f(0, n, n) - f(0, n, n + 1) - f(2, n, n)}


def _vorticity(g, u):
    P = u * g.len
    a, n, x = g.at, g.n, g.cells
    vL = (P[0] + a(P[2], 1, 0) + P[1]) / g.tri[0]
    vU = -(P[1] + P[2] + a(P[0], 0, 1)) / g.tri[1]
    c = _corner_sums(g, P, vL, vU)
    vL[x(-1, -1)] = vU[x(-1, -1)] = c["mm"] / g.tri[0][x(-1, -1)]
    vL[x(n - 1, -1)] = vU[x(n, -1)] = c["pm"] / g.tri[0][x(n - 1, -1)]
    vU[x(-1, n - 1)] = vL[x(-1, n)] = c["mp"] / g.tri[1][x(-1, n - 1)]
    vL[x(n, n)] = vU[x(n, n)] = c["pp"] / g.tri[0][x(n, n)]
    return vL, vU


def _masters_only(g, f):
    out = torch.zeros_like(f)
    out[..., g.masters] = f[..., g.masters]
    g.node_fill(out)
    return out


def _laplacian(g, q):
    F = g.grad(q, g.lenf) * g.pedf
    g.edge_fill(F)
    return _masters_only(g, g.div(F))


def _curl_edges(g, vL, vU, ped):
    return torch.stack([(vL - g.at(vU, 0, -1)) / ped[0], (vL - vU) / ped[1], (g.at(vL, -1, 0) - vU) / ped[2]])


def _hooks(g, order, m, t, u):
    """scalar fluxes and velocity source of the diffusion hooks of one layer"""
    vm, vt, vd, vr = DIFFUSION_VISC[order]
    F = u * g.pedf
    divu = g.div(F)
    local = divu[g.square()]
    divu = _masters_only(g, divu)
    divu[g.square()] = local  # each lozenge's own divergence beside its far edges
    vL, vU = _vorticity(g, u)
    qm, qt, sign = m, t, -1.0
    if order == 2:
        divu, qm, qt, sign = _laplacian(g, divu), _laplacian(g, m), _laplacian(g, t), 1.0
        rot = torch.zeros_like(u)
        curl = -_curl_edges(g, vL, vU, torch.where(g.ped != 0, g.ped, torch.ones_like(g.ped)))
        rot[:, g.owned] = curl[:, g.owned]
        g.edge_fill(rot)
        vL, vU = _vorticity(g, rot)
    fluxes = [sign * v * g.grad(q, g.lenf) * g.pedf for v, q in ((vm, qm), (vt, qt))]
    return fluxes, -sign * (vd * g.grad(divu, g.len) - vr * _curl_edges(g, vL, vU, g.ped))


def _trend(g, topo, mass, temp, velo, diffusion=0):
    a, n, x = g.at, g.n, g.cells
    L = mass.shape[0]
    dm, dt, du = torch.zeros_like(mass), torch.zeros_like(temp), torch.zeros_like(velo)
    p_low = GRAV * (mass - temp).sum(0)
    phi_low = GRAV * topo
    for k in range(L):
        m, t, u = mass[k], temp[k], velo[k]
        p_up = p_low - GRAV * (m - t)
        phi_up = phi_low + GRAV * m / RHO0
        press, phi = 0.5 * (p_low + p_up), 0.5 * (phi_low + phi_up)
        p_low, phi_low = p_up, phi_up
        P = u * g.len
        A = g.area
        circL, circU = P[0] + a(P[2], 1, 0) + P[1], -(P[1] + P[2] + a(P[0], 0, 1))
        pvL = (g.cor[0] + circL) / (m * A[0] + a(m * A[2], 1, 0) + a(m * A[4], 1, 1))
        pvU = (g.cor[1] + circU) / (m * A[1] + a(m * A[3], 1, 1) + a(m * A[5], 0, 1))
        qe = torch.stack([0.5 * (a(pvU, 0, -1) + pvL), 0.5 * (pvU + pvL), 0.5 * (pvU + a(pvL, -1, 0))])
        flux = u * g.pedf
        hm = torch.stack([flux[e] * f for e, f in enumerate(g.mean(m))])
        ht = torch.stack([flux[e] * f for e, f in enumerate(g.mean(t))])
        source = None
        if diffusion:
            (fm, ft), source = _hooks(g, diffusion, m, t, u)
            hm, ht = hm + fm, ht + ft
        c = _corner_sums(g, P, None, None)
        M_ = lambda p, i, j: m[x(i, j)] * A[p - 1][x(i, j)]  # noqa: E731
        L_ = lambda f, i, j: f[x(i, j)]  # noqa: E731
        # the lozenge's pentagon corners: potential vorticity of the merged triangle and of its two neighbours
        big = (L_(g.cor[0], -1, -1) + c["mm"]) / (M_(1, -1, 0) + M_(3, 0, 0) + M_(5, 0, 1))
        wl = (L_(g.cor[0], -1, 0) + L_(circL, -1, 0)) / (M_(6, -1, 0) + M_(4, 0, 0) + M_(5, 0, 0) + M_(3, 0, -1))
        su = (L_(g.cor[1], 0, -1) + L_(circU, 0, -1)) / (M_(2, 0, -1) + M_(4, 1, 0) + M_(6, 0, 0))
        # (the masses follow the corner routine's own triangles)
        qe[0][x(-1, 0)], qe[2][x(0, -1)] = 0.5 * (wl + big), 0.5 * (su + big)
        sw = (L_(g.cor[0], n - 1, -1) + c["pm"]) / (M_(1, n - 1, -1) + M_(3, n, -1) + M_(5, n, 0) + M_(6, n, 0))
        l0 = (L_(g.cor[0], n, 0) + L_(circL, n, 0)) / (M_(1, n, 0) + M_(3, n + 1, 0) + M_(5, n + 1, 1))
        u0 = (L_(g.cor[1], n - 1, -1) + L_(circU, n - 1, -1)) / (M_(2, n - 1, -1) + M_(4, n, 0) + M_(6, n - 1, 0))
        qe[0][x(n, 0)], qe[1][x(n - 1, -1)] = 0.5 * (sw + l0), 0.5 * (sw + u0)
        sw = (L_(g.cor[1], -1, n - 1) + c["mp"]) / (M_(2, -1, n - 1) + M_(3, 0, n) + M_(4, 0, n) + M_(6, -1, n))
        u0 = (L_(g.cor[1], 0, n) + L_(circU, 0, n)) / (M_(2, 0, n) + M_(4, 1, n + 1) + M_(6, 0, n + 1))
        l0 = (L_(g.cor[0], -1, n - 1) + L_(circL, -1, n - 1)) / (M_(1, -1, n - 1) + M_(3, 0, n - 1) + M_(5, 0, n))
        qe[2][x(0, n)], qe[1][x(-1, n - 1)] = 0.5 * (sw + u0), 0.5 * (l0 + sw)
        ne = (L_(g.cor[0], n, n) + c["pp"]) / (M_(3, n + 1, n) + M_(1, n, n) + M_(2, n, n) + M_(6, n, n + 1))
        wl = (L_(g.cor[0], n - 1, n) + L_(circL, n - 1, n)) / (M_(1, n - 1, n) + M_(3, n, n) + M_(5, n, n + 1))
        su = (L_(g.cor[1], n, n - 1) + L_(circU, n, n - 1)) / (M_(2, n, n - 1) + M_(4, n + 1, n) + M_(6, n, n))
        qe[0][x(n, n)], qe[2][x(n, n)] = 0.5 * (ne + su), 0.5 * (ne + wl)
        K = P * (u * g.ped)
        ke = (K[0] + K[1] + K[2] + a(K[2], 0, -1) + a(K[1], -1, -1) + a(K[0], -1, 0)) * g.hinv / 4.0
        bern, exner = ke + phi + press / RHO0, -phi
        dm[k][g.masters], dt[k][g.masters] = -g.div(hm)[g.masters], -g.div(ht)[g.masters]
        ring = [(0, [(1, 0, 0), (2, 0, 0), (0, -1, 0), (1, -1, -1), (2, 0, -1)],
                 (1, 0), 3, [(1, 0, -1), (2, 1, -1), (0, 1, 0), (1, 1, 0), (2, 1, 0)]),
                (1, [(2, 0, 0), (0, -1, 0), (1, -1, -1), (2, 0, -1), (0, 0, 0)],
                 (1, 1), 4, [(2, 1, 0), (0, 1, 1), (1, 1, 1), (2, 1, 1), (0, 0, 1)]),
                (2, [(0, -1, 0), (1, -1, -1), (2, 0, -1), (0, 0, 0), (1, 0, 0)],
                 (0, 1), 5, [(0, 0, 1), (1, 0, 1), (2, 0, 1), (0, -1, 1), (1, -1, 0)])]
        theta = g.mean(t / m)
        gB, gE = g.grad(bern, g.len), g.grad(exner, g.len)
        for e, near, nb, o, far in ring:
            q = torch.zeros_like(m)
            for i, (f, di, dj) in enumerate(near):
                q += a(hm[f], di, dj) * 0.5 * (a(qe[f], di, dj) + qe[e]) * g.w[e][i]
            for i, (f, di, dj) in enumerate(far):
                q += a(hm[f], di, dj) * 0.5 * (a(qe[f], di, dj) + qe[e]) * a(g.w[o][i], *nb)
            d = -q / g.len[e] - gB[e] - theta[e] * gE[e]
            if source is not None:
                d = d + source[e]
            du[k][e][g.owned] = d[g.owned]
    return dm, dt, du


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _members(case, seed, grid, mesh):
    """per member: topography and ghost-filled state"""
    topos, m, t, u = _ocean(grid, case, seed)
    L, put = case["layers"], lambda a: torch.as_tensor(np.array(a), device=mesh.dev)  # noqa: E731
    for k in range(case.get("members", 1)):
        s = slice(k * L, (k + 1) * L)
        topo, state = put(topos[k]), [put(m[s]), put(t[s]), put(u[s])]
        mesh.node_fill(topo)
        mesh.fill(state)
        yield topo, state, _step(grid, case, topos, m)


def _advance(s, d, h, g, extra=None):
    out = [a.clone() for a in s]
    out[0][:, g.masters] += h * d[0][:, g.masters]
    out[1][:, g.masters] += h * d[1][:, g.masters]
    du = d[2] if extra is None else d[2] + extra
    out[2][:, :, g.owned] += h * du[:, :, g.owned]
    g.fill(out)
    return out


def _apply(g, csq, coef, q):
    F = torch.stack(g.mean(csq)) * g.grad(q, g.lenf) * g.pedf
    return _masters_only(g, coef * g.div(F) - q)


def _solve(g, csq, coef, rhs, guess):
    """conjugate gradients to rounding: the operator is symmetric under the cells' areas"""
    W_ = torch.zeros_like(rhs)
    W_[g.masters] = 1.0 / g.hinv[g.masters]
    dot = lambda a, b: (W_ * a * b).sum()  # noqa: E731
    u = guess.clone()
    r = _masters_only(g, _apply(g, csq, coef, u) - rhs)
    p, rr = r.clone(), dot(r, r)
    stop = 1e-28 * dot(rhs, rhs)
    for _ in range(5000):
        if rr <= stop:
            break
        Ap = -_apply(g, csq, coef, p)
        al = rr / dot(p, Ap)
        u, r = u + al * p, r - al * Ap
        new = dot(r, r)
        p, rr = r + (new / rr) * p, new
    return u


def _flux_divergence(g, s):
    F = sum(u * torch.stack(g.mean(m)) for m, u in zip(s[0], s[2])) * g.pedf
    return _masters_only(g, g.div(F))


def _rescale(g, topo, eta, s):
    ratio = (eta - topo) / (s[0].sum(0) / RHO0)
    for a in s[:2]:
        a[:, g.masters] *= ratio[g.masters]
        g.node_fill(a)


def _split_steps(g, topo, s, dt, steps, th1=0.6, th2=0.8):
    eta = s[0].sum(0) / RHO0 + topo
    for _ in range(steps):
        before = _flux_divergence(g, s)
        push = th1 * GRAV * g.grad(eta, g.len)
        y = s
        for k in range(4):
            _rescale(g, topo, eta, y)
            y = _advance(s, _trend(g, topo, *y), dt / (4 - k), g, push)
        s = y
        rhs = _masters_only(g, -eta + dt * (th2 * _flux_divergence(g, s) + (1.0 - th2) * before) / RHO0)
        eta = _solve(g, GRAV * (topo.abs() + eta), th1 * th2 * dt * dt, rhs, eta)
        _rescale(g, topo, eta, s)
        s[2][:, :, g.owned] -= th1 * dt * GRAV * g.grad(eta, g.len)[:, g.owned]
        g.fill(s)
    return s, eta


def _tridiagonal(lo, di, up, rhs):
    """rows of [..., L, columns]; lo[k] and up[k] couple row k to k - 1 and k + 1"""
    L = di.shape[0]
    d, b = [di[0]], [rhs[0]]
    for k in range(1, L):
        f = lo[k] / d[-1]
        d.append(di[k] - f * up[k - 1])
        b.append(rhs[k] - f * b[-1])
    x = [b[-1] / d[-1]]
    for k in range(L - 2, -1, -1):
        x.append((b[k] - up[k] * x[-1]) / d[k])
    return torch.stack(x[::-1])


def _mixing_lengths(dz, nsq, tau, e):
    """dissipation and mixing length at the interfaces: turbulent lengths bounded by the distances to both ends"""
    first = torch.sqrt(2.0 * e / nsq.clamp(min=1e-20))
    dn, up = [torch.full_like(tau, 0.04)], [(0.4 * 2e5 / (RHO0 * GRAV) * tau).clamp(min=0.04)]
    for k in range(1, len(first)):
        dn.append(torch.minimum(first[k], dn[-1] + dz[k - 1]))
    for k in range(len(first) - 2, -1, -1):
        up.append(torch.minimum(first[k], up[-1] + dz[k]))
    dn, up = torch.stack(dn), torch.stack(up[::-1])
    return torch.sqrt(up * dn).clamp(min=0.01), torch.minimum(up, dn).clamp(min=0.01)


def _eddy_coefficients(dz, nsq, shear, tau, e):
    kv = (0.1 * _mixing_lengths(dz, nsq, tau, e)[1] * torch.sqrt(e)).clamp(1.2e-4, 1e-2)
    ri = nsq / (shear + 1e-20)
    pr = torch.where(ri < 0.2, torch.ones_like(ri), torch.where(ri <= 2.0, 5.0 * ri, torch.full_like(ri, 10.0)))
    return (kv / pr).clamp(1.2e-5, 1e-2), kv


def _diffuse(dt, K, dz, dzl, rhs, bottom=0.0, reference_top=False):
    """backward Euler of one column field with diffusivity K at the inner interfaces"""
    c = dt * K[1:-1] / dzl
    zero = torch.zeros_like(c[:1])
    lo, up = torch.cat([zero, -c / dz[1:]]), torch.cat([-c / dz[:-1], zero])
    di = 1.0 - (lo + up)
    di[0] += bottom
    if reference_top:  # the reference's top row takes the entry of the row below
        di[-1] = 1.0 - up[-2]
    return _tridiagonal(lo, di, up, rhs)


def _exact_vdiff(g, case, topo, s, dt, hooks, coef):
    m, t, u = s
    Kt, Kv, tke = coef
    bot, top, tau, wind = hooks
    dz = m / RHO0
    dzl = 0.5 * (dz[:-1] + dz[1:])
    if case["tke"]:
        K = (u * g.len) * (u * g.ped)
        a = g.at
        speed = torch.sqrt(2.0 * (K.sum(1) + a(K[:, 2], 0, -1) + a(K[:, 1], -1, -1) + a(K[:, 0], -1, 0)) * g.hinv / 4.0)
        zero = torch.zeros_like(dz[:1])
        shear = torch.cat([zero, ((speed[1:] - speed[:-1]) / dzl) ** 2, zero])
        b = t / m
        nsq = GRAV * (b[1:] - b[:-1]) / dzl
        nsq = torch.cat([nsq[:1], nsq, nsq[-1:]])
        e = torch.cat([torch.full_like(zero, 1e-6 / math.sqrt(2.0)), tke.clamp(min=1e-6)])
        i = slice(1, -1)
        sink = -0.7 * torch.sqrt(e) / _mixing_lengths(dz, nsq, tau, e)[0]
        gain = Kv * shear - Kt * nsq
        kup, klo = 0.5 * (Kv[1:-1] + Kv[2:]), 0.5 * (Kv[1:-1] + Kv[:-2])
        up, lo = -dt * kup / (dzl * dz[1:]), -dt * klo / (dzl * dz[:-1])
        up[-1], lo[0] = 0.0, 0.0
        new = _tridiagonal(lo, 1.0 - (up + lo) - dt * sink[i], up, e[i] + dt * gain[i]).clamp(min=1e-6)
        e = torch.cat([e[:1], new, (67.83 * tau / RHO0).clamp(min=1e-4)[None]])
        Kt, Kv = _eddy_coefficients(dz, nsq, shear, tau, e)
    else:
        z = torch.cat([topo[None], topo + dz.cumsum(0)])
        f = torch.exp((z - z[-1]) / 10.0)
        Kt, Kv = 1.2e-5 + 1e-2 * f, 1.2e-4 + 1e-2 * f
    rhs = t / m
    rhs[0] -= dt * bot / dz[0]
    rhs[-1] += dt * top / dz[-1]
    new_t = m * _diffuse(dt, Kt, dz, dzl, rhs, reference_top=True)
    out = [m.clone(), t.clone(), u.clone()]
    out[1][:, g.masters] = new_t[:, g.masters]
    for e_, dze in enumerate(g.mean(dz)):
        rhs = u[:, e_].clone()
        rhs[-1] += dt * wind[e_] / dze[-1]
        new_u = _diffuse(dt, Kv, dze, 0.5 * (dze[:-1] + dze[1:]), rhs, bottom=dt * 4e-4 / dze[0])
        out[2][:, e_, g.owned] = new_u[:, g.owned]
    g.fill(out)
    return out


def _primitive_slopes(x, f, at):
    """derivative at point `at` of the polynomial through the primitive of cell means f between the points x"""
    h = [b - a for a, b in zip(x, x[1:])]
    P = [torch.zeros_like(x[0]) for _ in x]
    for j in range(at + 1, len(x)):
        P[j] = P[j - 1] + h[j - 1] * f[j - 1]
    for j in range(at - 1, -1, -1):
        P[j] = P[j + 1] - h[j] * f[j]
    d = torch.zeros_like(x[0])
    for j in range(len(x)):
        if j == at:
            continue
        w = torch.ones_like(d)
        for k in range(len(x)):
            if k != j:
                w = w / (x[j] - x[k])
                if k != at:
                    w = w * (x[at] - x[k])
        d = d + P[j] * w
    return d


def _parabola(f0, el, er):
    return 1.5 * f0 - 0.25 * (er + el), 0.5 * (er - el), -1.5 * f0 + 0.75 * (er + el)


def _ppr_cells(x, f):
    """the limited parabolas a + b s + c s^2, s in [-1, 1], of the cells between the interfaces x"""
    N, h, where = len(f), x[1:] - x[:-1], torch.where
    if N <= 3:
        E = [f[0]] + [(h[i] * f[i - 1] + h[i - 1] * f[i]) / (h[i - 1] + h[i]) for i in range(1, N)] + [f[-1]]
    else:
        E = [_primitive_slopes(x[:4], f[:3], i) for i in range(2)]
        E += [_primitive_slopes(x[i - 2:i + 3], f[i - 2:i + 2], 2) for i in range(2, N - 1)]
        E += [_primitive_slopes(x[-4:], f[-3:], i) for i in (2, 3)]
    out = []
    for i in range(N):
        f0, fl, fr = f[i], f[max(i - 1, 0)], f[min(i + 1, N - 1)]
        h0, hl, hr = h[i], h[max(i - 1, 0)], h[min(i + 1, N - 1)]
        dm, dp = f0 - fl, fr - f0
        d0 = 0.5 * ((hr * f0 + h0 * fr) / (h0 + hr) - (h0 * fl + hl * f0) / (hl + h0))
        lim = (torch.minimum(dm.abs(), dp.abs()) / d0.abs().clamp(min=1e-14)).clamp(max=1.0) * d0
        d0 = where(dm * dp > 0.0, lim, torch.zeros_like(d0))
        el, er = E[i], E[i + 1]
        el = where((fl - el) * (el - f0) <= 0.0, f0 - d0, el)
        er = where((fr - er) * (er - f0) <= 0.0, f0 + d0, er)
        c = _parabola(f0, el, er)
        turn = where(c[2].abs() > 0.5 * c[1].abs(), -0.5 * c[1] / c[2], torch.full_like(f0, 9.0))
        right, left = (turn >= -1.0) & (turn <= 0.0), (turn > 0.0) & (turn <= 1.0)
        er, el = where(right, 3.0 * f0 - 2.0 * el, er), where(left, 3.0 * f0 - 2.0 * er, el)
        flat = dp * dm < 0.0
        c = _parabola(f0, el, er)
        out.append([where(flat, f0, c[0]), where(flat, torch.zeros_like(f0), c[1]), where(flat, torch.zeros_like(f0), c[2])])
    return [torch.stack([o[k] for o in out]) for k in range(3)]


def _remap_ppr(x, f, xn):
    a, b, c = _ppr_cells(x, f)
    h = x[1:] - x[:-1]
    mean = (a + c / 3.0) * h
    total = torch.cat([torch.zeros_like(mean[:1]), mean.cumsum(0)])
    j = (torch.searchsorted(x.T.contiguous(), xn.T.contiguous(), right=True).T - 1).clamp(0, len(f) - 1)
    hj = h.gather(0, j)
    s = 2.0 * (xn - x.gather(0, j)) / hj - 1.0
    part = lambda v: a.gather(0, j) * v + b.gather(0, j) * v ** 2 / 2 + c.gather(0, j) * v ** 3 / 3  # noqa: E731
    I_ = total.gather(0, j) + 0.5 * hj * (part(s) - part(torch.full_like(s, -1.0)))
    return (I_[1:] - I_[:-1]) / (xn[1:] - xn[:-1])


def _remap_flux(x, f, xn, scheme):
    """remap0 / remap1: fluxes through the moved interfaces of constant / reconciled linear profiles"""
    h, dz, where = x[1:] - x[:-1], (xn - x)[1:-1], torch.where
    zero = torch.zeros_like(f[:1])
    if scheme == W.REMAP_PIECEWISE_CONSTANT:
        F = dz.clamp(max=0.0) * f[:-1] + dz.clamp(min=0.0) * f[1:]
    else:
        d = (f[1:] - f[:-1]) / (h[1:] + h[:-1])
        d = torch.cat([d[:1], d, d[-1:]])
        slope = where(d[1:] * d[:-1] < 0.0, torch.zeros_like(f), 2.0 * d[1:] * d[:-1] / (d[1:] + d[:-1]))
        R, Lf = f + slope * h, f - slope * h
        for _ in range(10):
            E = torch.cat([Lf[:1], 0.5 * (R[:-1] + Lf[1:]), R[-1:]])
            dR, dL = E[1:] - f, f - E[:-1]
            c = where(dR * dL < 0.0, torch.zeros_like(f), where(dR.abs() > dL.abs(), dL, dR))
            R, Lf = f + c, f - c
        rise = dz > 0.0
        slope = R - Lf
        F = dz * (where(rise, Lf[1:], R[:-1]) + 0.5 * where(rise, slope[1:], slope[:-1]) * dz / where(rise, h[1:], h[:-1]))
    F = torch.cat([zero, F, zero])
    return (h * f + F[1:] - F[:-1]) / (xn[1:] - xn[:-1])


def _exact_remap(g, case, topo, s):
    av, bv = (torch.as_tensor(np.array(v), device=g.dev)[:, None] for v in _targets(case["layers"])[0])
    x = torch.cat([topo[None], topo + (s[0] / RHO0).cumsum(0)])
    xn = av * x[-1] + bv * topo
    column = _remap_ppr if case["scheme"] == W.REMAP_PPR else lambda *a: _remap_flux(*a, case["scheme"])
    mass = RHO0 * (xn[1:] - xn[:-1])
    c = g.masters
    out = [v.clone() for v in s]
    out[0][:, c] = mass[:, c]
    out[1][:, c] = mass[:, c] * column(x[:, c], (s[1] / s[0])[:, c], xn[:, c])
    c = g.owned
    for e, (xo, xe) in enumerate(zip(g.mean(x), g.mean(xn))):
        out[2][:, e, c] = column(xo[:, c], s[2][:, e, c], xe[:, c])
    g.fill(out)
    return out


def _exact_mlp(case, seed):
    """loss and gradient of the network in 64 bits, from the parameters that the seed gives it"""
    net = W.MLP(max_batch=16, seed=seed % 1000)
    params = torch.as_tensor(net.params).double().requires_grad_()
    net.close()
    x, t = (torch.as_tensor(v).double() for v in _mlp_rows(np.random.default_rng(seed), case["rows"]))
    at = 0
    for k, (i, o) in enumerate(((192, 128), (128, 128), (128, 64))):
        w, b = params[at:at + i * o].reshape(i, o), params[at + i * o:at + i * o + o]
        at += i * o + o
        x = x @ w + b
        if k < 2:
            x = torch.nn.functional.gelu(x)
    loss = ((x - t) ** 2).sum() / (2.0 * case["rows"])
    loss.backward()
    return [loss.detach(), params.grad]


def exact(case, seed):
    kind, dev = case["kind"], _device()
    if kind in ("ml_rk4", "ml_split"):
        return None  # the transforms between levels: over 20 seconds in plain array operations
    if kind == "mlp":
        return _exact_mlp(case, seed)
    grid = _case_grids(case)[-1]
    g = _Mesh(grid, dev)
    if kind == "solve":
        outs = []
        for topo, eta_old, rhs in zip(*_solve_fields(grid, case["members"], seed)):
            f = [torch.as_tensor(a, device=dev).clone() for a in (topo, eta_old, rhs)]
            for a in f:
                g.node_fill(a)
            dt = _step(grid, case, None, None)
            outs.append(_solve(g, GRAV * (f[0].abs() + f[1]), dt * dt, f[2], torch.zeros_like(f[2])).cpu().numpy())
        return outs[0] if case["members"] == 1 else np.stack(outs)
    outs = []
    for topo, s, dt in _members(case, seed, grid, g):
        if kind == "rk4":
            for _ in range(case["steps"]):
                y = s
                for k in range(4):
                    y = _advance(s, _trend(g, topo, *y, case["diffusion"]), dt / (4 - k), g)
                s = y
            outs.append(s)
        elif kind == "split":
            s, eta = _split_steps(g, topo, s, dt, case["steps"])
            outs.append(s + [eta.cpu().numpy()])
        elif kind == "remap":
            outs.append(_exact_remap(g, case, topo, s))
        else:
            k, L, nc = len(outs), case["layers"], g.nc
            put = lambda a: torch.as_tensor(np.array(a), device=dev)  # noqa: E731
            hooks, coef = _forcing(np.random.default_rng(seed + 2), case["members"], L, nc)
            hooks = [put(h.reshape(case["members"], -1, nc)[k]) for h in hooks.values()]
            for h in hooks:
                g.node_fill(h) if len(h) == 1 else g.edge_fill(h)
            coef = [put(a.reshape(case["members"], -1, nc)[k]) for a in coef]
            outs.append(_exact_vdiff(g, case, topo, s, _step(grid, case, None, None),
                                     [h[0] if len(h) == 1 else h for h in hooks], coef))
    parts = [torch.cat([o[k] for o in outs]) for k in range(3)]
    if kind == "split":
        parts.append(outs[0][3] if len(outs) == 1 else np.stack([o[3] for o in outs]))
    return parts
