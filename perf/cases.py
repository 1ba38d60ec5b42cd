"""What a user of the beam Newton path has it do, as cases that can be timed.

Every case is a time-stepping program: a structure is set up and brought a few steps into its
motion, that state is saved, and ONE pass restores it, applies the steps' inputs, advances and
reads the motion back (the correction iteration of a program that couples the blades to an
aerodynamic or CFD solver, and the restart of a load case).  Kinds:

  terms      one element's residual and iteration matrix through the allocation-free entry point
  blade      the blade interface (one prescribed-root blade, loads per node, motion per node)
  beam       one beam driven from the host: dynamic or static, either form, either tangent
  rotor      one three-blade rotor with prescribed hub motion, driven from the host
  points     a beam with point masses and a spring (plain form)
  ensemble   many independent rotors as load cases, inputs as a device schedule
  structure  tower, shaft and blades joined into one large system (plain form)
"""

import functools
import math

import numpy as np
import torch

import openturbine_amd as ota
from openturbine_amd import workloads as W

F64 = torch.float64
_LIB = []


def _lib():
    if not _LIB:
        _LIB.append(ota.KynLib())
    return _LIB[0]


# --------------------------------------------------------------------------------------
# cases
# --------------------------------------------------------------------------------------
def listed():
    return [
        # the smallest call: a serving loop asks for the terms of one full-size blade element
        {"name": "terms_21", "kind": "terms", "nodes": 21, "qps": 40},
        # one blade of a coupled turbine program, the reference's blade interface test in size
        {"name": "blade_11", "kind": "blade", "nodes": 11, "sections": 21, "steps": 2},
        # the FP32-tangent cantilever (8 nodes, 11 points: an odd quadrature), 4 steps
        {"name": "beam_fp32_8", "kind": "beam", "nodes": 8, "qps": 11, "form": "fused", "tangent": "fp32",
         "static": False, "refine": 1, "bound": 10.0, "steps": 4},
        # static load stepping in the reference's launch structure, a ragged size
        {"name": "beam_static_16", "kind": "beam", "nodes": 16, "qps": 17, "form": "plain", "tangent": "fp64",
         "static": True, "refine": 0, "bound": 0.0, "steps": 2},
        # one rotor stepped from the host, 11 nodes and 20 points per blade
        {"name": "rotor_11", "kind": "rotor", "nodes": 11, "qps": 20, "form": "fused", "tangent": "fp64",
         "refine": 0, "bound": 0.0, "steps": 4},
        # point masses and a spring beside the beam: the plain form's other elements
        {"name": "points_plain", "kind": "points", "h": 0.005, "steps": 3},
        # the throughput workload: 4096 rotors, FP32 tangent, refinement in the converging iteration
        {"name": "ensemble_fp32_4096", "kind": "ensemble", "rotors": 4096, "nodes": 0, "form": "fused",
         "tangent": "fp32", "refine": 1, "bound": 10.0, "steps": 4},
        # a day's load cases of one turbine design, refinement in every Newton iteration
        {"name": "ensemble_fp32_96", "kind": "ensemble", "rotors": 96, "nodes": 0, "form": "fused",
         "tangent": "fp32", "refine": 1, "bound": 0.0, "steps": 4},
        # load cases in full FP64
        {"name": "ensemble_fp64_512", "kind": "ensemble", "rotors": 512, "nodes": 0, "form": "fused",
         "tangent": "fp64", "refine": 0, "bound": 0.0, "steps": 2},
        # the reference's launch structure over an ensemble
        {"name": "ensemble_plain_256", "kind": "ensemble", "rotors": 256, "nodes": 0, "form": "plain",
         "tangent": "fp64", "refine": 0, "bound": 0.0, "steps": 2},
        # a whole turbine structure of 8459 dofs, both tangents
        {"name": "structure_fp64", "kind": "structure", "nodes": 21, "tower": 8, "shaft": 8, "blade": 16,
         "tangent": "fp64", "refine": 0, "steps": 2},
        {"name": "structure_fp32", "kind": "structure", "nodes": 21, "tower": 8, "shaft": 8, "blade": 16,
         "tangent": "fp32", "refine": 2, "steps": 2},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["terms", "blade", "beam", "beam", "rotor", "points", "ensemble", "ensemble", "ensemble",
                       "structure", "structure"])
    nodes = rng.randint(5, 21)
    qps = rng.randint(nodes, 2 * nodes)
    fp32 = rng.random() < 0.5
    prec = {"tangent": "fp32", "refine": 1, "bound": rng.choice([10.0, 0.0])} if fp32 else \
        {"tangent": "fp64", "refine": 0, "bound": 0.0}
    if kind == "terms":
        return {"kind": kind, "nodes": nodes, "qps": qps}
    if kind == "blade":
        return {"kind": kind, "nodes": nodes, "sections": rng.randint(nodes, 40), "steps": rng.randint(1, 4)}
    if kind == "beam":
        static = not fp32 and rng.random() < 0.4
        return {"kind": kind, "nodes": nodes, "qps": qps, "form": rng.choice(["fused", "plain"]), "static": static,
                "steps": rng.randint(1, 6), **prec}
    if kind == "rotor":
        return {"kind": kind, "nodes": nodes, "qps": qps, "form": rng.choice(["fused", "fused", "plain"]),
                "steps": rng.randint(1, 6), **prec}
    if kind == "points":
        return {"kind": kind, "h": round(rng.uniform(0.002, 0.01), 4), "steps": rng.randint(1, 8)}
    if kind == "ensemble":
        plain = not fp32 and rng.random() < 0.3
        rotors = _log_int(rng, 2, 256 if plain else 1024)
        return {"kind": kind, "rotors": rotors, "nodes": rng.choice([0, 0, nodes]), "form": "plain" if plain else "fused",
                "steps": rng.randint(1, 3), **prec}
    return {"kind": kind, "nodes": rng.randint(8, 21), "tower": rng.randint(2, 10), "shaft": rng.randint(1, 8),
            "blade": rng.randint(2, 16), "tangent": prec["tangent"], "refine": 2 if fp32 else 0,
            "steps": rng.randint(1, 2)}


# --------------------------------------------------------------------------------------
# inputs: model specs and the inputs of every step (warm-up steps first)
# --------------------------------------------------------------------------------------
def _root_motion(omega, t, p):
    """Rigid rotation of a root at p (hub axis x): {u, quaternion}."""
    q = np.array([math.cos(0.5 * omega * t), math.sin(0.5 * omega * t), 0.0, 0.0])
    c, s = math.cos(omega * t), math.sin(omega * t)
    return np.concatenate([[0.0, c * p[1] - s * p[2] - p[1], s * p[1] + c * p[2] - p[2]], q])


class _Problem:
    """Distinct specs, how they are repeated, and every step's inputs:
    cdisp [steps][constraints][7] or None, loads [steps][loaded nodes][6] on load_nodes."""

    def __init__(self, specs, order, warm, steps):
        self.specs, self.order, self.warm, self.steps = specs, order, warm, steps
        self.node_off = np.concatenate([[0], np.cumsum([specs[k].num_nodes for k in order])])
        self.cdisp, self.load_nodes, self.loads = None, None, None
        self.h = specs[0].h

    def rotor_motion(self):
        """Prescribed roots of every rotor in order, from each spec's hub speeds."""
        per_spec = []
        for sp in self.specs:
            roots = [sp.x0[c.target, :3] for c in sp.constraints]
            per_spec.append(np.array([[_root_motion(om, self.h * (k + 1), p) for p, om in zip(roots, sp.meta["omegas"])]
                                      for k in range(self.warm + self.steps)]))
        self.cdisp = np.ascontiguousarray(np.concatenate([per_spec[k] for k in self.order], axis=1))

    def tip_loads(self, nodes, gen, sigma, tau):
        """Forces on `nodes`: normal(0, sigma) in every step, correlated over tau seconds."""
        rho = math.exp(-self.h / tau)
        f = gen.standard_normal((len(nodes), 3))
        self.load_nodes = np.asarray(nodes)
        self.loads = np.zeros((self.warm + self.steps, len(nodes), 6))
        for k in range(self.warm + self.steps):
            self.loads[k, :, :3] = sigma * f
            f = rho * f + math.sqrt(1.0 - rho * rho) * gen.standard_normal(f.shape)

    def nodal_loads(self, k):
        f = np.zeros((int(self.node_off[-1]), 6))
        f[self.load_nodes] = self.loads[k]
        return f


@functools.lru_cache(maxsize=2)
def _designs(distinct, nodes):
    return W.ensemble_config_specs(num_rotors=distinct, fixed_nodes=nodes or None)


def _problem(case, seed):
    gen = np.random.default_rng(seed)
    key = int(gen.integers(1 << 30))
    kind = case["kind"]
    if kind in ("terms", "rotor"):
        spec = W.rotor_config_spec(num_nodes=case["nodes"], num_qps=case["qps"], omega=gen.uniform(0.8, 1.2),
                                   length=gen.uniform(50.0, 70.0), seed=key)
        p = _Problem([spec], [0], 2, case.get("steps", 0))
        p.rotor_motion()
    elif kind == "beam":
        spec = W.cantilever_config_spec(num_nodes=case["nodes"], num_qps=case["qps"])
        spec.is_dynamic = not case["static"]
        p = _Problem([spec], [0], 1, case["steps"])
        tip, amp = spec.meta["tip_node"], gen.uniform(0.4, 1.0) * (3e4 if case["static"] else 1e5)
        p.load_nodes = np.array([tip])
        p.loads = np.zeros((1 + case["steps"], 1, 6))
        for k in range(1 + case["steps"]):
            p.loads[k, 0, 1:3] = amp * (k + 1) / (2.0 + case["steps"]) * np.array([0.3, 1.0])
    elif kind == "points":
        spec = W.beam_mass_spring_spec(h=case["h"])
        p = _Problem([spec], [0], 2, case["steps"])
        p.tip_loads([spec.meta["tip_node"], spec.meta["extra_node"]], gen, 2e3, 0.1)
    elif kind == "ensemble":
        distinct = min(case["rotors"], 64)
        specs = _designs(distinct, case["nodes"])  # the designs are the same, their load cases the seed's
        p = _Problem(specs, [r % distinct for r in range(case["rotors"])], 2, case["steps"])
        p.rotor_motion()
        tips = np.concatenate([p.node_off[r] + specs[k].meta["tips"] for r, k in enumerate(p.order)])
        p.tip_loads(tips, gen, 1e4, 0.1)
    else:
        spec = W.structure_config_spec(num_nodes=case["nodes"], num_qps=2 * case["nodes"] - 2, tower_elems=case["tower"],
                                       shaft_elems=case["shaft"], blade_elems=case["blade"], seed=key)
        p = _Problem([spec], [0], 1, case["steps"])
        p.tip_loads(spec.meta["tips"], gen, 1e4, 0.1)
    return p


def _blade_inputs(case, seed):
    """A straight blade along x with tapered sections, hub speed about z, loads on every node."""
    gen = np.random.default_rng(seed)
    grid, M, C = W.section_properties(int(gen.integers(1 << 30)), 0, num_stations=case["sections"], size_factor=4.0)
    omega, total = gen.uniform(0.5, 1.0), 2 + case["steps"]
    loads = np.cumsum(gen.standard_normal((total, case["nodes"], 6)) * np.array([1e2, 1e3, 1e3, 10.0, 10.0, 10.0]), axis=0)
    return {"length": 40.0, "grid": grid, "M": M, "C": C, "omega": omega, "h": 0.01, "rho": 0.9, "total": total,
            "loads": loads, "root": np.array([2.0, 0.0, 0.0]), "gravity": np.array([0.0, 0.0, -9.81])}


def _blade_root(b, k):
    a = b["omega"] * b["h"] * (k + 1)
    c, s, p = math.cos(a), math.sin(a), b["root"]
    return np.array([c * p[0] - p[0], s * p[0], 0.0, math.cos(a / 2), 0.0, 0.0, math.sin(a / 2)])


# --------------------------------------------------------------------------------------
# a pass
# --------------------------------------------------------------------------------------
def prepare(case, seed):
    lib = _lib()
    if case["kind"] == "blade":
        b = _blade_inputs(case, seed)
        om = np.array([0.0, 0.0, b["omega"]])
        beam = ota.beam_input(
            element_order=case["nodes"] - 1, ref_grid=[0.0, 1.0], ref_coords=[[0, 0, 0], [b["length"], 0, 0]],
            twist_grid=[0.0, 1.0], twist=[0.0, 0.0], section_grid=b["grid"], section_mass=b["M"],
            section_stiffness=b["C"], prescribe_root_motion=True, root_position=(*b["root"], 1, 0, 0, 0),
            root_velocity=(*np.cross(om, b["root"]), *om),
            root_acceleration=(*np.cross(om, np.cross(om, b["root"])), 0, 0, 0))
        g = ota.KynBladeInterface(lib, {"gravity": b["gravity"], "time_step": b["h"], "rho_inf": b["rho"], "max_iter": 20,
                                        "atol": 1e-8, "rtol": 1e-6}, beam)
        state = {"case": case, "blade": g, "inputs": b}
        for k in range(2):
            _blade_step(state, k)
        g.save_state()
        return state
    p = _problem(case, seed)
    fp32 = case.get("tangent") == "fp32"
    plain = case["kind"] in ("points", "structure") or case.get("form") == "plain"
    g = ota.KynSystem(lib, [p.specs[k] for k in p.order], exec_mode=ota.EXEC_PLAIN if plain else ota.EXEC_FUSED,
                      precision=ota.TANGENT_FP32 if fp32 else ota.TANGENT_FP64, refine_sweeps=case.get("refine", 0),
                      refine_err_bound=case.get("bound", 0.0))
    state = {"case": case, "system": g, "problem": p}
    if case["kind"] == "ensemble":
        w = p.warm
        g.set_schedule(w, p.cdisp[:w], p.load_nodes, p.loads[:w])
        g.step_many(w, use_graph=False)
        state["window"] = [np.ascontiguousarray(a) for a in (p.cdisp[w:], p.loads[w:])]
    else:
        state["inputs"] = []
        for k in range(p.warm + p.steps):
            d = {}
            if p.cdisp is not None:
                d["constraint_disp"] = {c: p.cdisp[k, c] for c in range(p.cdisp.shape[1])}
            if p.loads is not None:
                d["nodal_loads"] = p.nodal_loads(k)
            state["inputs"].append(d)
        for k in range(p.warm):
            g.step(state["inputs"][k])
    g.save_state()
    if case["kind"] == "terms":
        N = case["nodes"]
        state["out"] = np.zeros((N, 6)), np.zeros((N, N, 36))
    return state


def _blade_step(state, k):
    g, b = state["blade"], state["inputs"]
    g.set_root_displacement(_blade_root(b, k))
    for i in range(g.n):
        g.set_node_loads(i, b["loads"][k, i])
    g.step()


def run(state):
    case = state["case"]
    if case["kind"] == "blade":
        g = state["blade"]
        g.restore_state()
        for k in range(2, 2 + case["steps"]):
            _blade_step(state, k)
        motion = [g.motion(i) for i in range(g.n)]
        return [np.stack([m[c] for m in motion]) for c in range(4)]
    g, p = state["system"], state["problem"]
    if case["kind"] == "terms":
        r, m = state["out"]
        g._check(g.lib.L.kyn_element_terms_noalloc(g.h, 1, r.ctypes.data_as(ota._dp), m.ctypes.data_as(ota._dp)))
        return [r, m]
    g.restore_state()
    if case["kind"] == "ensemble":
        cdisp, loads = state["window"]
        g.set_schedule(case["steps"], cdisp, p.load_nodes, loads)
        g.step_many(case["steps"], use_graph=True)
    else:
        for k in range(p.warm, p.warm + p.steps):
            g.step(state["inputs"][k])
    return [g.get(f) for f in _fields(case)]


def _fields(case):
    """The motion a program reads: displacements and rates; from the FP32-tangent form the rates
    of single systems, and of an ensemble the displacements (a Newton path of one more iteration
    moves a rotor's rates at the convergence tolerance)."""
    if case.get("tangent") == "fp32":
        return ["q"] if case["kind"] == "ensemble" else ["q", "v"]
    return ["q", "v", "vd"]


# --------------------------------------------------------------------------------------
# the work of a pass
# --------------------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "blade":
        elems = [(case["nodes"], case["sections"])]
    elif kind in ("terms", "beam"):
        elems = [(case["nodes"], case["qps"])]
    elif kind == "rotor":
        elems = [(case["nodes"], case["qps"])] * 3
    elif kind == "points":
        elems = [(8, 11)]
    elif kind == "ensemble":
        sizes = [case["nodes"]] if case["nodes"] else [6, 11, 16, 21]
        elems = [(n, 2 * n - 2) for n in sizes for _ in range(round(3 * case["rotors"] / len(sizes)))]
    else:
        ne = case["tower"] + case["shaft"] + 3 * case["blade"]
        elems = [(case["nodes"], 2 * case["nodes"] - 2)] * ne
    # Newton iterations a step takes on average
    iters = {"terms": 0, "blade": 3, "beam": 4, "rotor": 5, "points": 3, "ensemble": 5.3, "structure": 6}[kind]
    read = sum(8.0 * (38 * n + 87 * q) for n, q in elems)  # state, loads, section and quadrature data
    contract = sum(144.0 * n * n * q for n, q in elems)
    solve = sum((2.0 / 3.0) * (6 * n + 6) ** 3 + 2.0 * (6 * n + 6) ** 2 for n, q in elems)
    if kind == "terms":
        n = case["nodes"]
        return {"bytes": read + 8.0 * (6 * n + 36 * n * n), "flops": contract}
    wrote = sum(8.0 * 38 * n for n, q in elems)
    return {"bytes": read + wrote, "flops": case["steps"] * iters * (contract + solve)}


# --------------------------------------------------------------------------------------
# the same steps in 64 bits with plain torch
# --------------------------------------------------------------------------------------
def _mul(a, b):
    """Quaternion product."""
    a0, a1, a2, a3 = a.unbind(-1)
    b0, b1, b2, b3 = b.unbind(-1)
    return torch.stack([a0 * b0 - a1 * b1 - a2 * b2 - a3 * b3, a0 * b1 + a1 * b0 + a2 * b3 - a3 * b2,
                        a0 * b2 - a1 * b3 + a2 * b0 + a3 * b1, a0 * b3 + a1 * b2 - a2 * b1 + a3 * b0], -1)


def _conj(q):
    return q * torch.tensor([1.0, -1.0, -1.0, -1.0], dtype=F64, device=q.device) / q.norm(dim=-1, keepdim=True)


def _rot(q):
    a, b, c, d = q.unbind(-1)
    return torch.stack([a * a + b * b - c * c - d * d, 2 * (b * c - a * d), 2 * (b * d + a * c),
                        2 * (b * c + a * d), a * a - b * b + c * c - d * d, 2 * (c * d - a * b),
                        2 * (b * d - a * c), 2 * (c * d + a * b), a * a - b * b - c * c + d * d], -1).reshape(*q.shape[:-1], 3, 3)


def _skew(v):
    x, y, z = v.unbind(-1)
    o = torch.zeros_like(x)
    return torch.stack([o, -z, y, z, o, -x, -y, x, o], -1).reshape(*v.shape[:-1], 3, 3)


def _vec(M, v):
    return (M * v[..., None, :]).sum(-1)


def _diag2(R):
    out = torch.zeros(*R.shape[:-2], 6, 6, dtype=F64, device=R.device)
    out[..., :3, :3] = R
    out[..., 3:, 3:] = R
    return out


def _section(R, M):
    R2 = _diag2(R)
    return R2 @ M @ R2.transpose(-1, -2).contiguous()


def _inertial(r, ud, w, wd, r0, Ms, g):
    """Mass, gyroscopic and inertia-stiffness matrices, inertial and gravity forces."""
    M = _section(_rot(_mul(r, r0)), Ms)
    m = M[..., 0, 0]
    me = torch.stack([M[..., 5, 1], -M[..., 5, 0], M[..., 4, 0]], -1)  # m eta
    rho = M[..., 3:, 3:]
    W_, Wd, Me = _skew(w), _skew(wd), _skew(me)
    N = W_ @ W_ + Wd
    Fi = torch.cat([m[..., None] * ud + _vec(N, me), _vec(Me, ud) + _vec(rho, wd) + _vec(W_ @ rho, w)], -1)
    Fg = torch.cat([m[..., None] * g, _vec(Me, g.expand_as(me))], -1)
    G, K = torch.zeros_like(M), torch.zeros_like(M)
    T = lambda A: A.transpose(-1, -2)  # noqa: E731
    Hw = _skew(_vec(rho, w))
    G[..., :3, 3:] = W_ @ T(Me) + T(_skew(_vec(W_, me)))
    G[..., 3:, 3:] = W_ @ rho - Hw
    K[..., :3, 3:] = N @ T(Me)
    K[..., 3:, 3:] = _skew(ud) @ Me + rho @ Wd - _skew(_vec(rho, wd)) + W_ @ (rho @ W_ - Hw)
    return M, G, K, Fi, Fg


def _stiffness(r, rp, up, r0, x0p, Cs):
    C = _section(_rot(_mul(r, r0)), Cs)
    a, b, c, d = r.unbind(-1)
    E = torch.stack([-b, a, -d, c, -c, d, a, -b, -d, -c, b, a], -1).reshape(*r.shape[:-1], 3, 4)
    strain = torch.cat([x0p + up - _vec(_rot(r), x0p), 2 * _vec(E, rp)], -1)
    F = _vec(C, strain)
    X = _skew(x0p + up)
    Xt = X.transpose(-1, -2)
    Nt, Mt = _skew(F[..., :3]), _skew(F[..., 3:])
    O, P, Q = (torch.zeros_like(C) for _ in range(3))
    O[..., :3, 3:] = C[..., :3, :3] @ X - Nt
    O[..., 3:, 3:] = C[..., 3:, :3] @ X - Mt
    P[..., 3:, :3] = Xt @ C[..., :3, :3] + Nt
    P[..., 3:, 3:] = Xt @ C[..., :3, 3:]
    Q[..., 3:, 3:] = Xt @ (C[..., :3, :3] @ X - Nt)
    Fd = torch.cat([torch.zeros_like(F[..., :3]), _vec(Xt, F[..., :3])], -1)
    return C, O, P, Q, F, Fd


def _lagrange(x, xs):
    """Values and derivatives [N][Q] of the Lagrange basis on xs at points x."""
    N, Q = len(xs), len(x)
    phi, dphi = np.zeros((N, Q)), np.zeros((N, Q))
    for i in range(N):
        oth = [k for k in range(N) if k != i]
        phi[i] = np.prod([(x - xs[k]) / (xs[i] - xs[k]) for k in oth], axis=0)
        for j in oth:
            dphi[i] += np.prod([(x - xs[k]) / (xs[i] - xs[k]) for k in oth if k != j] + [np.ones(Q)], axis=0) / (xs[i] - xs[j])
    return phi, dphi


class _Group:
    """Blocks of one topology, batched: n nodes, E elements of N nodes and Q points, constraints
    (type, base, target), point masses and springs."""

    def __init__(self, dev, params, model, members):
        t = lambda a: torch.tensor(np.asarray(a), dtype=F64, device=dev)  # noqa: E731
        self.dev, self.p, self.model = dev, params, torch.tensor(model, device=dev)
        first = members[0]
        self.n, self.cons = len(first["x0"]), first["cons"]
        self.x0 = t(np.stack([b["x0"] for b in members]))
        self.q = t(np.stack([b["u"] for b in members]))
        self.v = t(np.stack([b["v"] for b in members]))
        self.vd = t(np.stack([b["vd"] for b in members]))
        self.a, self.f = self.vd.clone(), torch.zeros_like(self.v)
        self.B = len(members)
        self.g = t(first["gravity"])
        self.rows = [5 if c[0] == W.REVOLUTE_JOINT else 6 for c in self.cons]
        self.off = [6 * self.n + sum(self.rows[:k]) for k in range(len(self.rows))]
        self.size = 6 * self.n + sum(self.rows)
        self.cdisp = t(np.tile([0.0, 0, 0, 1, 0, 0, 0], (self.B, max(1, len(self.cons)), 1)))
        el = first["elems"]
        self.enodes = torch.tensor(np.stack([e["nodes"] for e in el]), device=dev)
        quad = np.asarray(el[0]["quad"])
        xi = 2.0 * np.asarray(first["s"])[el[0]["nodes"]] - 1.0
        phi, dphi = _lagrange(quad[:, 0], xi)
        self.phi, self.dphi, self.w = t(phi), t(dphi), t(quad[:, 1])
        M, C = [], []
        for b in members:
            for e in b["elems"]:
                sx = 2.0 * np.asarray(e["s"]) - 1.0
                M.append(np.stack([np.interp(quad[:, 0], sx, e["M"][:, k]) for k in range(36)], -1))
                C.append(np.stack([np.interp(quad[:, 0], sx, e["C"][:, k]) for k in range(36)], -1))
        shape = (self.B, len(el), len(quad), 6, 6)
        self.Ms, self.Cs = t(np.stack(M)).reshape(shape), t(np.stack(C)).reshape(shape)
        xe = self.x0[:, self.enodes]
        d = torch.einsum("beid,iq->beqd", xe[..., :3], self.dphi)
        self.J = d.norm(dim=-1)
        self.x0p = d / self.J[..., None]
        r = torch.einsum("beid,iq->beqd", xe[..., 3:], self.phi)
        self.r0 = r / r.norm(dim=-1, keepdim=True)
        self.masses = [(k, t(m).reshape(6, 6)) for k, m in first["masses"]]
        self.springs = first["springs"]

    def displaced(self):
        h = self.p["h"]
        rv = h * self.qd[..., 3:]
        ang = rv.norm(dim=-1, keepdim=True)
        f = torch.where(ang < 1e-12, torch.zeros_like(ang), torch.sin(ang / 2) / torch.where(ang < 1e-12, torch.ones_like(ang), ang))
        dq = torch.cat([torch.cos(ang / 2), rv * f], -1)
        return torch.cat([self.qp[..., :3] + h * self.qd[..., :3], _mul(dq, self.qp[..., 3:])], -1)

    def predict(self):
        p, h = self.p, self.p["h"]
        self.qp = self.q
        an = (p["af"] * self.vd - p["am"] * self.a) / (1 - p["am"])
        vn = self.v + h * (1 - p["gamma"]) * self.a + p["gamma"] * h * an
        self.qd = self.v + (0.5 - p["beta"]) * h * self.a + p["beta"] * h * an
        self.a, self.v, self.vd = an, vn, torch.zeros_like(vn)
        self.q = self.displaced()
        self.lam = torch.zeros(self.B, self.size - 6 * self.n, dtype=F64, device=self.dev)

    def tangent(self):
        """The stored tangent of every node: rotations about h q_delta."""
        rv = self.p["h"] * self.qd[..., 3:]
        ang = rv.norm(dim=-1)[..., None, None]
        one = torch.ones_like(ang)
        safe = torch.where(ang > 1e-16, ang, one)
        t1 = torch.where(ang > 1e-16, (torch.cos(ang) - 1) / safe**2, 0 * one)
        t2 = torch.where(ang > 1e-16, (1 - torch.sin(ang) / safe) / safe**2, 0 * one)
        S = _skew(rv)
        T = torch.zeros(*rv.shape[:-1], 6, 6, dtype=F64, device=self.dev)
        eye = torch.eye(3, dtype=F64, device=self.dev)
        T[..., :3, :3] = eye
        T[..., 3:, 3:] = (eye + t1 * S + t2 * (S @ S)).transpose(-1, -2)
        return T

    def element_terms(self, T):
        """Residuals [B][E][N][6] and iteration matrices [B][E][N][6][N][6]."""
        p, phi, dphi = self.p, self.phi, self.dphi
        qe, ve, ae = self.q[:, self.enodes], self.v[:, self.enodes], self.vd[:, self.enodes]
        at = lambda v: torch.einsum("beid,iq->beqd", v, phi)  # noqa: E731
        r = at(qe[..., 3:])
        r = r / r.norm(dim=-1, keepdim=True)
        ddx = lambda v: torch.einsum("beid,iq->beqd", v, dphi) / self.J[..., None]  # noqa: E731
        M, G, K, Fi, Fg = _inertial(r, at(ae[..., :3]), at(ve[..., 3:]), at(ae[..., 3:]), self.r0, self.Ms, self.g)
        C, O, P, Q, Fc, Fd = _stiffness(r, ddx(qe[..., 3:]), ddx(qe[..., :3]), self.r0, self.x0p, self.Cs)
        w, wJ, wdJ = self.w, self.w * self.J, self.w / self.J
        res = torch.einsum("iq,beqd->beid", dphi * w, Fc) + torch.einsum("iq,beqd->beid", phi, wJ[..., None] * (Fd + Fi - Fg))
        N, nq = phi.shape
        B, E = self.J.shape[:2]
        pair = lambda a, b: (a[:, None, :] * b[None, :, :]).reshape(N * N, nq)  # noqa: E731
        s = lambda c, A: (c[..., None, None] * A).reshape(B, E, nq, 36)  # noqa: E731
        wb = w.expand_as(self.J)
        left = torch.cat([pair(phi, phi), pair(phi, dphi), pair(dphi, phi), pair(dphi, dphi)], 1)
        right = torch.cat([s(wJ, K + Q), s(wb, P), s(wb, O), s(wdJ, C)], 2)
        U = (left @ right).reshape(B, E, N, N, 6, 6) @ T[:, self.enodes][:, :, None]
        U = U + (pair(phi, phi) @ s(wJ, p["bp"] * M + p["gp"] * G)).reshape(B, E, N, N, 6, 6)
        return res, U.permute(0, 1, 2, 4, 3, 5)

    def constraint(self, k):
        """Residual [B][6], gradients (base or None, target) [B][6][6] of constraint k."""
        typ, base, target, axes, X0 = self.cons[k]
        dev, B = self.dev, self.B
        tq = self.q[:, target]
        X = torch.tensor(X0, dtype=F64, device=dev).expand(B, 3) if typ != W.PRESCRIBED_BC else torch.zeros(B, 3, dtype=F64, device=dev)
        two = typ in (W.RIGID_JOINT, W.REVOLUTE_JOINT)
        bq = self.q[:, base] if two else self.cdisp[:, k]
        if typ == W.FIXED_BC:
            X = self.x0[:, target, :3]
        u1, R1, u2, R2 = bq[:, :3], bq[:, 3:], tq[:, :3], tq[:, 3:]
        RX = _vec(_rot(R1), X)
        res = torch.zeros(B, 6, dtype=F64, device=dev)
        res[:, :3] = u2 + X - u1 - RX
        tg, bg = torch.zeros(B, 6, 6, dtype=F64, device=dev), torch.zeros(B, 6, 6, dtype=F64, device=dev)
        eye = torch.eye(3, dtype=F64, device=dev)
        tg[:, :3, :3], bg[:, :3, :3] = eye, -eye
        if typ != W.REVOLUTE_JOINT:
            C = _rot(_mul(R2, _conj(R1)))
            res[:, 3:] = torch.stack([C[:, 2, 1] - C[:, 1, 2], C[:, 0, 2] - C[:, 2, 0], C[:, 1, 0] - C[:, 0, 1]], -1) / 2
            A = 0.5 * (C.diagonal(dim1=-2, dim2=-1).sum(-1)[:, None, None] * eye - C)
            tg[:, 3:, 3:] = A.transpose(-1, -2)
            bg[:, :3, 3:], bg[:, 3:, 3:] = _skew(RX), -A
        else:
            ax = [torch.tensor(a, dtype=F64, device=dev).expand(B, 3) for a in axes]
            x, y, z = _vec(_rot(R1), ax[0]), _vec(_rot(R2), ax[1]), _vec(_rot(R2), ax[2])
            res[:, 3], res[:, 4] = (z * x).sum(-1), (y * x).sum(-1)
            xz, xy = torch.linalg.cross(x, z), torch.linalg.cross(x, y)
            tg[:, 3, 3:], tg[:, 4, 3:], bg[:, 3, 3:], bg[:, 4, 3:] = -xz, -xy, xz, xy
        return res, (bg if two else None), tg, base, target

    def solve(self):
        """One Newton iteration: sum over rows of the weighted increments squared [B], then the update."""
        p, n, B = self.p, self.n, self.B
        cond = p["beta"] * p["h"] ** 2
        T = self.tangent()
        A = torch.zeros(B, self.size, self.size, dtype=F64, device=self.dev)
        b = torch.zeros(B, self.size, dtype=F64, device=self.dev)
        b[:, :6 * n] = -self.f.reshape(B, -1)
        if len(self.enodes):
            res, S = self.element_terms(T)
            for e in range(len(self.enodes)):
                idx = (6 * self.enodes[e][:, None] + torch.arange(6, device=self.dev)).reshape(-1)
                A[:, idx[:, None], idx[None, :]] += cond * S[:, e].reshape(B, len(idx), len(idx))
                b[:, idx] += res[:, e].reshape(B, -1)
        for k, Mm in self.masses:
            M, G, K, Fi, Fg = _inertial(self.q[:, k, 3:], self.vd[:, k, :3], self.v[:, k, 3:], self.vd[:, k, 3:],
                                        self.x0[:, k, 3:], Mm, self.g)
            sl = slice(6 * k, 6 * k + 6)
            A[:, sl, sl] += cond * (p["bp"] * M + p["gp"] * G + K @ T[:, k])
            b[:, sl] += Fi - Fg
        for i, j, ks, l0 in self.springs:
            r = self.x0[:, j, :3] - self.x0[:, i, :3] + self.q[:, j, :3] - self.q[:, i, :3]
            ln = r.norm(dim=-1)
            c1, c2 = ks * (l0 / ln - 1), ks * l0 / ln**3
            rr = _skew(r) @ _skew(r)
            a = (c1 - c2 * ln * ln)[:, None, None] * torch.eye(3, dtype=F64, device=self.dev) - c2[:, None, None] * rr
            si, sj = slice(6 * i, 6 * i + 3), slice(6 * j, 6 * j + 3)
            for u, v_, sg in ((si, si, 1), (sj, sj, 1), (si, sj, -1), (sj, si, -1)):
                A[:, u, v_] += sg * cond * a
            b[:, si] += c1[:, None] * r
            b[:, sj] -= c1[:, None] * r
        for k in range(len(self.cons)):
            res, bg, tg, base, target = self.constraint(k)
            rows, o = self.rows[k], self.off[k]
            lam = self.lam[:, o - 6 * n:o - 6 * n + rows]
            for gr, node in ((tg, target), (bg, base)):
                if gr is None:
                    continue
                sl = slice(6 * node, 6 * node + 6)
                A[:, o:o + rows, sl] += gr[:, :rows] @ T[:, node]
                A[:, sl, o:o + rows] += gr[:, :rows].transpose(-1, -2)
                b[:, sl] += (gr[:, :rows] * lam[..., None]).sum(1)
            b[:, o:o + rows] = res[:, :rows]
        rhs = -b
        rhs[:, :6 * n] *= cond
        x = torch.linalg.solve(A, rhs[..., None])[..., 0]
        x[:, 6 * n:] /= cond
        return x

    def update(self, x, active):
        """Applies the increments of the blocks still iterating; returns their error sums [B]."""
        p, n = self.p, self.n
        d, dl = x[:, :6 * n].reshape(self.B, n, 6), x[:, 6 * n:]
        err = ((d / (p["atol"] + p["rtol"] * (self.qd * p["h"]).abs())) ** 2).sum((1, 2))
        err = err + ((dl / (p["atol"] + p["rtol"] * self.lam.abs())) ** 2).sum(1)
        m = active[self.model][:, None, None].to(F64)
        self.qd = self.qd + m * d / p["h"]
        if p["dynamic"]:
            self.v, self.vd = self.v + m * p["gp"] * d, self.vd + m * p["bp"] * d
        self.lam = self.lam + m[:, :, 0] * dl
        self.q = torch.where(m > 0, self.displaced(), self.q)
        return err

    def finish(self):
        self.a = self.a + (1 - self.p["af"]) / (1 - self.p["am"]) * self.vd


def _params(h, rho, atol, rtol, max_iter, dynamic):
    am, af = (2 * rho - 1) / (rho + 1), rho / (rho + 1)
    gamma = 0.5 + af - am
    beta = 0.25 * (gamma + 0.5) ** 2
    return {"h": h, "am": am, "af": af, "gamma": gamma, "beta": beta, "atol": atol, "rtol": rtol, "max_iter": max_iter,
            "gp": gamma / (h * beta) if dynamic else 0.0,
            "bp": (1 - am) / (h * h * beta * (1 - af)) if dynamic else 0.0, "dynamic": dynamic}


def _axes(axis):
    """The revolute joint's frame: its unit axis and two unit vectors normal to it."""
    x = np.asarray(axis, dtype=float) / np.linalg.norm(axis)
    v, c = np.cross([1.0, 0.0, 0.0], x), x[0]
    V = np.array([[0, -v[2], v[1]], [v[2], 0, -v[0]], [-v[1], v[0], 0]])
    R = np.eye(3) + V + V @ V / (1 + c)
    return [R[:, 0], R[:, 1], R[:, 2]]


def _blocks(sp):
    """A spec's independent blocks: one per beam where every constraint holds a single node."""
    elem = lambda b, nodes: {"nodes": nodes, "quad": b.quad, "s": b.section_s, "M": b.section_M, "C": b.section_C}  # noqa: E731
    base = {"gravity": sp.gravity, "masses": [], "springs": []}
    if len(sp.beams) > 1 and all(c.type in (W.FIXED_BC, W.PRESCRIBED_BC) for c in sp.constraints):
        for b in sp.beams:
            ids = np.asarray(b.nodes)
            where = {int(k): i for i, k in enumerate(ids)}
            cons = [(c.type, 0, where[int(c.target)], None, None) for c in sp.constraints if int(c.target) in where]
            yield ids, [k for k, c in enumerate(sp.constraints) if int(c.target) in where], {
                **base, "x0": sp.x0[ids], "u": sp.u[ids], "v": sp.v[ids], "vd": sp.vd[ids], "s": sp.s[ids], "cons": cons,
                "elems": [elem(b, np.arange(len(ids)))]}
        return
    cons = []
    for c in sp.constraints:
        two = c.type in (W.RIGID_JOINT, W.REVOLUTE_JOINT)
        cons.append((c.type, int(c.base), int(c.target), _axes(c.axis) if c.type == W.REVOLUTE_JOINT else None,
                     sp.x0[c.target, :3] - sp.x0[c.base, :3] if two else np.zeros(3)))
    yield np.arange(sp.num_nodes), list(range(len(cons))), {
        **base, "x0": sp.x0, "u": sp.u, "v": sp.v, "vd": sp.vd, "s": sp.s, "cons": cons,
        "elems": [elem(b, np.asarray(b.nodes)) for b in sp.beams], "masses": [(e.node, e.M) for e in sp.masses],
        "springs": [(e.n1, e.n2, e.k, e.l0) for e in sp.springs]}


class _Exact:
    def __init__(self, specs, order, params):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.dev, self.p = dev, params
        found, node0, con0 = {}, 0, 0
        ndofs = []
        for m, k in enumerate(order):
            sp, nd = specs[k], 0
            for ids, cids, b in _blocks(sp):
                key = (len(b["x0"]), len(b["elems"]), len(b["elems"][0]["quad"]), tuple(c[:3] for c in b["cons"]))
                found.setdefault(key, []).append((m, node0 + ids, con0 + np.array(cids, dtype=int), b))
                nd += 6 * len(ids) + sum(5 if c[0] == W.REVOLUTE_JOINT else 6 for c in b["cons"])
            ndofs.append(nd)
            node0 += sp.num_nodes
            con0 += len(sp.constraints)
        self.nodes = node0
        self.ndofs = torch.tensor(ndofs, dtype=F64, device=dev)
        self.groups = []
        for mem in found.values():
            g = _Group(dev, params, [x[0] for x in mem], [x[3] for x in mem])
            g.ids = torch.tensor(np.stack([x[1] for x in mem]), device=dev)
            g.cids = torch.tensor(np.stack([x[2] for x in mem]), device=dev)
            self.groups.append(g)

    def step(self, cdisp, load_nodes, loads):
        f = torch.zeros(self.nodes, 6, dtype=F64, device=self.dev)
        if loads is not None:
            f[torch.tensor(np.asarray(load_nodes, dtype=np.int64), device=self.dev)] = torch.tensor(loads, dtype=F64, device=self.dev)
        for g in self.groups:
            g.f = f[g.ids]
            if cdisp is not None:
                g.cdisp = torch.tensor(cdisp, dtype=F64, device=self.dev)[g.cids]
            g.predict()
        active = torch.ones(len(self.ndofs), dtype=torch.bool, device=self.dev)
        for _ in range(self.p["max_iter"]):
            total = torch.zeros_like(self.ndofs)
            for g in self.groups:
                total.index_add_(0, g.model, g.update(g.solve(), active))
            active = active & (torch.sqrt(total / self.ndofs) > 1.0)
            if not bool(active.any()):
                break
        for g in self.groups:
            g.finish()

    def get(self, field):
        out = torch.zeros(self.nodes, 7 if field in ("q", "x") else 6, dtype=F64, device=self.dev)
        for g in self.groups:
            if field == "x":
                val = torch.cat([g.x0[..., :3] + g.q[..., :3], _mul(g.q[..., 3:], g.x0[..., 3:])], -1)
            else:
                val = getattr(g, field)
            out[g.ids] = val
        return out.cpu().numpy()


def exact(case, seed):
    if case["kind"] == "blade":
        b = _blade_inputs(case, seed)
        N, L = case["nodes"], b["length"]
        xi = np.polynomial.legendre.Legendre.basis(N - 1).deriv().roots().real if N > 2 else np.zeros(0)
        s = (np.concatenate([[-1.0], np.sort(xi), [1.0]]) + 1) / 2
        om, r0 = np.array([0.0, 0.0, b["omega"]]), b["root"]
        x0 = np.zeros((N, 7))
        x0[:, 0], x0[:, 3] = s * L, 1.0
        x0[:, :3] += r0
        rel = x0[:, :3] - r0
        v = np.concatenate([np.cross(om, r0) + np.cross(om, rel), np.tile(om, (N, 1))], 1)
        vd = np.concatenate([np.cross(om, np.cross(om, r0)) + np.cross(om, np.cross(om, rel)), np.zeros((N, 3))], 1)
        grid = b["grid"]  # trapezoidal quadrature at the section stations
        wq = np.concatenate([[grid[1] - grid[0]], grid[2:] - grid[:-2], [grid[-1] - grid[-2]]]) / (grid[-1] - grid[0])
        quad = np.stack([2 * (grid - grid[0]) / (grid[-1] - grid[0]) - 1, wq], 1)
        spec = W.ModelSpec("blade", x0, np.tile([0.0, 0, 0, 1, 0, 0, 0], (N, 1)), v, vd, s,
                           [W.BeamSpec(np.arange(N), grid, b["M"], b["C"], quad)],
                           [W.ConstraintSpec(W.PRESCRIBED_BC, 0, 0)], b["gravity"])
        e = _Exact([spec], [0], _params(b["h"], b["rho"], 1e-8, 1e-6, 20, True))
        for k in range(b["total"]):
            e.step(_blade_root(b, k)[None], np.arange(N), b["loads"][k])
        return [e.get(f) for f in ("x", "q", "v", "vd")]
    p = _problem(case, seed)
    if len(p.order) * (p.warm + p.steps) > 2600:
        return None
    sp = p.specs[0]
    e = _Exact(p.specs, p.order, _params(sp.h, sp.rho_inf, sp.atol, sp.rtol, sp.max_iter, sp.is_dynamic))
    for k in range(p.warm + p.steps):
        e.step(None if p.cdisp is None else p.cdisp[k], p.load_nodes, None if p.loads is None else p.loads[k])
    if case["kind"] == "terms":
        g = e.groups[0]
        res, S = g.element_terms(g.tangent())
        N = case["nodes"]
        return [res[1, 0].cpu().numpy(), S[1, 0].permute(0, 2, 1, 3).reshape(N, N, 36).cpu().numpy()]
    return [e.get(f) for f in _fields(case)]
