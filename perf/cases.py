"""Performance cases: the work that programs have this framework do.

A simulation holds one engine (nbody_create_engine) for one set of bodies, and
its solvers call engine.fcompute(t, y, f) on state buffers, combine the
derivatives with the engine's vector ops, and step.  The cases below are such
calls, from a thousand bodies (where launches and latency count) to the four
million of the Barnes-Hut workload.

A state is (engine, buffers); the engine -- with its masses, tree and scratch --
is shared by the states of a case, as a simulation's stage buffers share it.
"""
from __future__ import annotations

import functools
import math

import torch

from nbody_amd import nbody_create_engine, nbody_create_solver, nbody_data

MIN_DISTANCE = 1e-8      # the force law's clamp on r^2
TIME_STEP = 1e-3      # time step of the rk4 case


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed() -> list[dict]:
    return [
        # one whole rk4 step (4 force evaluations and their combinations) of the
        # small unit ball that runs start with; FP64 is the default precision
        {"name": "rk4_step_fp64_1024", "kind": "rk4", "bodies": "ball", "n": 1024},
        # one force evaluation of a medium FP64 run with a ragged body count
        {"name": "direct_fp64_20011", "kind": "direct", "precision": "fp64", "bodies": "plummer", "n": 20011},
        # FP64 forces of the cold-cube workload (rkfeagin10 and bs call this 150 times a step)
        {"name": "direct_fp64_65536", "kind": "direct", "precision": "fp64", "bodies": "cube", "n": 65536},
        # small FP32 run: the sort and the launches weigh as much as the pairs
        {"name": "direct_fp32_4000", "kind": "direct", "precision": "fp32", "bodies": "plummer", "n": 4000},
        # the cold cube's split-precision forces (FP32 tiles + FP64 neighbours)
        {"name": "direct_fp32_corr_65536", "kind": "direct", "precision": "fp32_corr", "bodies": "cube", "n": 65536},
        # the headline direct sum: one rkdp stage of the 2^18 Plummer sphere
        {"name": "direct_fp32_262144", "kind": "direct", "precision": "fp32", "bodies": "plummer", "n": 262144},
        # Barnes-Hut with the reference's arithmetic (the engine's default
        # precision and walk) at theta 0.5: heap build + per-body FP64 walk
        {"name": "bh_fp64_131072", "kind": "bh", "tree": "heap", "precision": "fp64", "walk": "body",
         "multipole": "monopole", "far": "per_body", "ratio": 2.0, "near": 3.0, "bodies": "plummer", "n": 131072},
        # the FP32 monopole group walk on the heap tree at theta 0.5
        {"name": "bh_group_262144", "kind": "bh", "tree": "heap", "precision": "fp32", "walk": "group",
         "multipole": "monopole", "far": "per_body", "ratio": 2.0, "near": 3.0, "bodies": "plummer", "n": 262144},
        # two colliding Plummer spheres, two-level quadrupole walk on the heap tree, theta 0.6
        {"name": "bh_two_level_1048576", "kind": "bh", "tree": "heap", "precision": "fp32", "walk": "group",
         "multipole": "quadrupole", "far": "local", "ratio": 1.667, "near": 3.0, "bodies": "two_plummer",
         "n": 1048576},
        # Morton-tree walk of an ordinary, ragged body count
        {"name": "bh_morton_100003", "kind": "bh", "tree": "morton", "precision": "fp32", "walk": "group",
         "multipole": "quadrupole", "far": "local", "ratio": 1.667, "near": 2.0, "bodies": "plummer", "n": 100003},
        # the fastest Barnes-Hut force evaluation of the 4M Plummer workload (theta 0.6, near 2)
        {"name": "bh_morton_4194304", "kind": "bh", "tree": "morton", "precision": "fp32", "walk": "group",
         "multipole": "quadrupole", "far": "local", "ratio": 1.667, "near": 2.0, "bodies": "plummer", "n": 4194304},
        # the compensated 12-term combination that ends an rkfeagin10 step of 2^20 bodies
        {"name": "fmaddn_corr_1048576", "kind": "fmaddn_corr", "terms": 12, "n": 1048576},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["rk4", "direct", "direct", "direct", "direct", "bh64", "group", "two_level", "morton", "morton",
                       "fmaddn_corr"])
    if kind == "rk4":
        return {"kind": "rk4", "bodies": rng.choice(["ball", "plummer"]), "n": _log_int(rng, 64, 16384)}
    if kind == "direct":
        precision = rng.choice(["fp64", "fp64", "fp32", "fp32", "fp32_corr"])
        n = _log_int(rng, 256, 131072 if precision == "fp64" else 262144)
        return {"kind": "direct", "precision": precision, "bodies": rng.choice(["plummer", "cube", "ball"]), "n": n}
    if kind == "fmaddn_corr":
        return {"kind": "fmaddn_corr", "terms": rng.randint(1, 16), "n": _log_int(rng, 1000, 1048576)}
    case = {"kind": "bh", "tree": "heap", "precision": "fp32", "walk": "group", "multipole": "quadrupole",
            "far": "local", "ratio": round(rng.uniform(1.25, 2.0), 3), "near": rng.choice([2.0, 2.5, 3.0]),
            "bodies": rng.choice(["plummer", "two_plummer"])}
    if kind == "bh64":
        case.update(precision="fp64", walk="body", multipole="monopole", far="per_body", n=1 << rng.randint(10, 17))
    elif kind == "group":
        case.update(multipole="monopole", far="per_body", n=1 << rng.randint(12, 18))
    elif kind == "two_level":
        case.update(n=1 << rng.randint(14, 20))
    else:
        case.update(tree="morton", n=_log_int(rng, 2000, 4194304))
    return case


# ---------------------------------------------------------------------------
# bodies, made on the GPU
# ---------------------------------------------------------------------------
def _generator(seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _uniform(g, *shape) -> torch.Tensor:
    return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64)


def _isotropic(g, length: torch.Tensor) -> torch.Tensor:
    z = (1.0 - 2.0 * _uniform(g, length.numel())) * length
    rxy = (length * length - z * z).clamp_min(0.0).sqrt()
    phi = 2.0 * math.pi * _uniform(g, length.numel())
    return torch.stack((rxy * phi.cos(), rxy * phi.sin(), z))


def _plummer(g, n: int, offset: float, drift: float) -> torch.Tensor:
    """[6, n]: Plummer sphere (a = M = 1, cut at 10 a) shifted along x."""
    top = (1.0 + 1.0 / 100.0) ** -1.5                     # mass within 10 a
    x = (_uniform(g, n) * top).clamp_min(1e-12)
    r = 1.0 / (x ** (-2.0 / 3.0) - 1.0).sqrt()
    q = torch.linspace(0.0, 1.0, 4097, device="cuda", dtype=torch.float64)
    cdf = torch.cumsum(q * q * (1.0 - q * q).clamp_min(0.0) ** 3.5, 0)
    speed = q[torch.searchsorted(cdf / cdf[-1], _uniform(g, n)).clamp_max(4096)]
    vesc = math.sqrt(2.0) * (1.0 + r * r) ** -0.25
    y = torch.cat((_isotropic(g, r), _isotropic(g, speed * vesc)))
    y[0] += offset
    y[3] += drift
    return y


def _state(kind: str, n: int, seed: int) -> torch.Tensor:
    """Positions and velocities in the engines' layout [x y z vx vy vz], [6, n]."""
    g = _generator(seed)
    if kind == "plummer":
        return _plummer(g, n, 0.0, 0.0)
    if kind == "two_plummer":
        h = n // 2
        return torch.cat((_plummer(g, h, -5.0, 0.25), _plummer(g, n - h, 5.0, -0.25)), 1).contiguous()
    if kind == "ball":
        pos = _isotropic(g, _uniform(g, n) ** (1.0 / 3.0))
        return torch.cat((pos, 0.3 * torch.randn(3, n, generator=g, device="cuda", dtype=torch.float64)))
    if kind == "cube":                                     # cold start: bodies at rest
        return torch.cat((2.0 * _uniform(g, 3, n) - 1.0, torch.zeros(3, n, device="cuda", dtype=torch.float64)))
    raise ValueError(kind)


def _masses(kind: str, n: int) -> torch.Tensor:
    """The masses belong to the simulation, not to a state: the same for every seed."""
    if kind == "cube":
        m = torch.exp(0.5 * torch.randn(n, generator=_generator(n), device="cuda", dtype=torch.float64))
        return m / m.sum()
    return torch.full((n,), (2.0 if kind == "two_plummer" else 1.0) / n, device="cuda", dtype=torch.float64)


# ---------------------------------------------------------------------------
# engines and states
# ---------------------------------------------------------------------------
def _engine_params(case: dict) -> dict:
    if case["kind"] == "bh":
        return {"engine": "hip_bh", "distance_to_node_radius_ratio": case["ratio"], "tree_layout": "heap_stackless",
                "force_precision": case["precision"], "bh_walk": case["walk"], "bh_tree": case["tree"],
                "bh_multipole": case["multipole"], "bh_far_field": case["far"], "bh_quad_near": case["near"]}
    return {"engine": "hip", "force_precision": case.get("precision", "fp64")}


@functools.lru_cache(maxsize=1)
def _simulation(key: tuple):
    """The engine of a case (and its solver), initialised with the bodies' masses."""
    case = dict(key)
    n = case["n"]
    bodies = case.get("bodies", "ball")
    data = nbody_data()
    data.set_quiet(True)
    y = _state(bodies, n, 1)
    data.set_bodies(y[:3].t().contiguous().cpu().numpy(), y[3:].t().contiguous().cpu().numpy(),
                    _masses(bodies, n).cpu().numpy())
    engine = nbody_create_engine(_engine_params(case))
    if engine is None or not engine.init(data):
        raise RuntimeError(f"no engine for {case}")
    solver = None
    if case["kind"] == "rk4":
        solver = nbody_create_solver({"solver": "rk4", "max_step": TIME_STEP})
        solver.set_engine(engine)
    return engine, solver


class _DeviceArray:
    """An engine buffer as torch sees it (no copy); a tensor made from it keeps
    it, and so the buffer's owner, alive."""

    def __init__(self, mem, owner, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f8", "data": (mem.device_ptr(), False),
                                         "version": 2}


def _view(mem, owner, *shape) -> torch.Tensor:
    return torch.as_tensor(_DeviceArray(mem, owner, shape), device="cuda")


class _Buffers:
    """Engine buffers that go back to the engine with the state."""

    def __init__(self, engine, nbytes: int, count: int):
        self.engine = engine
        self.mem = engine.create_buffers(nbytes, count)
        if len(self.mem) != count:
            raise MemoryError("out of memory: engine buffers")

    def __del__(self):
        self.engine.free_buffers(self.mem)


def prepare(case: dict, seed: int) -> dict:
    engine, solver = _simulation(tuple(sorted((k, v) for k, v in case.items() if k != "name")))
    n = case["n"]
    state = {"kind": case["kind"], "engine": engine, "solver": solver}
    if case["kind"] == "fmaddn_corr":
        terms = case["terms"]
        buf = _Buffers(engine, 48 * n, terms + 2)
        g = _generator(seed)
        for k, m in enumerate(buf.mem):
            # a state of order 1, a small correction, and derivatives of order 1
            scale = 1e-17 if k == 1 else 1.0
            _view(m, buf, 6 * n).copy_(scale * torch.randn(6 * n, generator=g, device="cuda", dtype=torch.float64))
        state.update(buf=buf, coef=_coefficients(terms),
                     out=(_view(buf.mem[0], buf, 6 * n), _view(buf.mem[1], buf, 6 * n)))
    else:
        buf = _Buffers(engine, 48 * n, 1 if solver is not None else 2)
        _view(buf.mem[0], buf, 6, n).copy_(_state(case["bodies"], n, seed))
        result = _view(engine.get_y() if solver is not None else buf.mem[1], buf, 6, n)
        state.update(buf=buf, y=engine.get_y(), out=(result[:3], result[3:]))
    torch.cuda.synchronize()      # the engine's stream is not torch's
    return state


def run(state: dict):
    engine, buf = state["engine"], state["buf"].mem
    if state["kind"] == "fmaddn_corr":
        engine.fmaddn_corr(buf[0], buf[1], buf[2:], state["coef"], len(state["coef"]))
    elif state["kind"] == "rk4":
        engine.copy_buffer(state["y"], buf[0])        # the saved state that the step starts from
        state["solver"].advise(TIME_STEP)
    else:
        engine.fcompute(0.0, buf[0], buf[1])
    return state["out"]


def _coefficients(terms: int) -> list[float]:
    return [1e-3 / (3.0 + k) for k in range(terms)]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case: dict) -> dict:
    n = case["n"]
    if case["kind"] == "fmaddn_corr":
        return {"bytes": 8.0 * 6 * n * (case["terms"] + 4), "flops": 5.0 * 6 * n * case["terms"]}
    evaluation = 8.0 * n * (6 + 1 + 6)                    # state and masses in, derivative out
    if case["kind"] == "rk4":
        return {"bytes": 2 * 48.0 * n + 8.0 * n, "flops": 4 * 20.0 * n * n}
    if case["kind"] == "direct":
        return {"bytes": evaluation, "flops": 20.0 * n * n}
    # Barnes-Hut: a compact tree's cells at this opening ratio (about 60 per
    # halving of the distance at ratio 2), and each node record written and read once
    cells = min(float(n), 7.5 * case["ratio"] ** 3 * math.log2(n))
    flops_per_cell = 20.0 if case["multipole"] == "monopole" else 50.0
    return {"bytes": evaluation + 2 * 2 * 64.0 * n, "flops": flops_per_cell * cells * n}


# ---------------------------------------------------------------------------
# how far another correct implementation may be
# ---------------------------------------------------------------------------
def tolerance(case: dict):
    if case["kind"] in ("rk4", "fmaddn_corr") or case.get("precision") == "fp64":
        return "exact"          # the FP64 paths reproduce the CPU engines bit for bit
    if case["kind"] == "direct":
        return {"rel": 2e-5, "max": 2e-3}      # measured against 64 bits: 2e-7 to 6e-6, set by close pairs
    # Barnes-Hut in FP32: which cells a group opens may differ, within the method's
    # own error (measured against the direct sum: 1.4e-3 and 4.9e-3)
    return {"rel": 5e-3 if case["multipole"] == "quadrupole" else 2e-2, "max": 0.5}


# ---------------------------------------------------------------------------
# the same in 64 bits, by plain torch
# ---------------------------------------------------------------------------
def _accelerations(y: torch.Tensor, m: torch.Tensor) -> torch.Tensor:
    n = y.shape[1]
    out = torch.empty(3, n, device="cuda", dtype=torch.float64)
    rows = max(1, (1 << 26) // n)
    for i in range(0, n, rows):
        d = [y[k][None, :] - y[k, i:i + rows, None] for k in range(3)]
        r2 = (d[0] * d[0]).add_(d[1] * d[1]).add_(d[2] * d[2]).clamp_min_(MIN_DISTANCE)
        w = m[None, :] / (r2 * r2.sqrt())
        for k in range(3):
            out[k, i:i + rows] = (d[k] * w).sum(1)
    return out


def _derivative(y: torch.Tensor, m: torch.Tensor) -> torch.Tensor:
    return torch.cat((y[3:], _accelerations(y, m)))


def exact(case: dict, seed: int):
    n = case["n"]
    if case["kind"] == "fmaddn_corr":
        # the compensated sum's state; its correction term has no value in 64 bits
        g = _generator(seed)
        rows = [(1e-17 if k == 1 else 1.0) * torch.randn(6 * n, generator=g, device="cuda", dtype=torch.float64)
                for k in range(case["terms"] + 2)]
        total = rows[0]
        for c, r in zip(_coefficients(case["terms"]), rows[2:]):
            total = total + c * r
        return total, None
    if n > 262144:
        return None                                       # a direct sum over these bodies takes too long
    y = _state(case["bodies"], n, seed)
    m = _masses(case["bodies"], n)
    if case["kind"] == "rk4":
        h = TIME_STEP
        k1 = _derivative(y, m)
        k2 = _derivative(y + 0.5 * h * k1, m)
        k3 = _derivative(y + 0.5 * h * k2, m)
        k4 = _derivative(y + h * k3, m)
        y = y + (h / 6.0) * (k1 + 2.0 * k2 + 2.0 * k3 + k4)
        return y[:3], y[3:]
    f = _derivative(y, m)
    return f[:3], f[3:]
