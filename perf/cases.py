"""Performance cases: the work that programs built on this engine have it do,
through the public entry points of `marbles_amd`, at the sizes, storages and
layouts they use.

Kinds of case
  flow         a compact level advanced by `Level.advance` (the hot path)
  diagnostics  macroscopic fields, vorticity, tags and conservation sums of a
               compact level (what a program does between steps for output)
  fab          a level in the reference's box layout advanced by
               `Level.advance`, ghosts of every layer filled afterwards
  stages       one step of the reference's schedule, stage by stage, on the
               box layout (the drop-in use, where the caller owns the loop)
  amr          a two-level hierarchy advanced by `Hierarchy.advance`, ghosts
               of every layer filled afterwards
  adjoint      an objective of the isothermal solver and its gradient through
               torch autograd

Initial states are seeded smooth fields (density, velocity, temperature) about
the flow's reference state, so every population differs from cell to cell.
`exact` restates the step in plain torch at 64 bits.
"""
from __future__ import annotations

import math

import numpy as np
import torch
import torch.utils.checkpoint

from marbles_amd import Hierarchy, Level, configs
from marbles_amd.adjoint import IsoSolver, flow_loss

# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------


def listed() -> list[dict]:
    return [
        # the smallest boxes people start with (tutorial and regression sizes,
        # 16^3 to 32^3): a handful of microseconds of work per step, so the
        # launches and the host path decide
        {"name": "periodic_24_f64", "kind": "flow", "flow": "periodic", "nx": 24, "ny": 24, "nz": 24,
         "storage": "f64", "steps": 10, "tuned": False, "forces": False},
        # the cylinder validation run: the deck's 660 x 123 x 4 domain, the
        # force on the body sampled every 25 steps
        {"name": "cylinder_turek_f64", "kind": "flow", "flow": "cylinder", "nx": 660, "ny": 123, "nz": 4,
         "storage": "f64", "steps": 25, "tuned": False, "forces": True},
        # an ordinary production box whose extents are no round numbers, rows
        # wider than 256 cells, the level's own kernel
        {"name": "channel_301_f64", "kind": "flow", "flow": "channel", "nx": 301, "ny": 150, "nz": 131,
         "storage": "f64", "steps": 5, "tuned": False, "forces": False},
        # the benchmark workload: 256^3 channel with a sphere, FP64, the
        # kernel chosen by the autotuner as the benchmark does
        {"name": "channel_256_f64_tuned", "kind": "flow", "flow": "channel", "nx": 256, "ny": 256, "nz": 256,
         "storage": "f64", "steps": 6, "tuned": True, "forces": False},
        # walled duct with the Channel inlet profile, shifted FP32 storage at
        # a moderate size
        {"name": "duct_160_f32s", "kind": "flow", "flow": "profile", "nx": 160, "ny": 80, "nz": 80,
         "storage": "f32s", "steps": 10, "tuned": False, "forces": False},
        # a large periodic box in shifted FP32 storage (the precision study's
        # family)
        {"name": "periodic_320_f32s", "kind": "flow", "flow": "periodic", "nx": 320, "ny": 320, "nz": 320,
         "storage": "f32s", "steps": 4, "tuned": False, "forces": False},
        # the benchmark channel in scaled FP16 storage, fields read back
        {"name": "channel_256_f16s", "kind": "flow", "flow": "channel", "nx": 256, "ny": 256, "nz": 256,
         "storage": "f16s", "steps": 6, "tuned": False, "forces": False},
        # output of a run: fields, vorticity, refinement tags, conservation
        {"name": "diagnostics_200", "kind": "diagnostics", "flow": "channel", "nx": 200, "ny": 160, "nz": 144,
         "storage": "f64"},
        # the reference's box layout (boxes of at most 32 cells, three ghost
        # layers) driven by the batched step
        {"name": "fab_128_f64", "kind": "fab", "nx": 128, "ny": 96, "nz": 72, "max_box": 32, "steps": 5},
        # the same layout driven stage by stage, uneven boxes
        {"name": "stages_90_f64", "kind": "stages", "nx": 90, "ny": 72, "nz": 56, "max_box": 32},
        # two levels: uneven coarse boxes, a fine level over a fifth of the
        # volume (the two-level benchmark's family at a size that prepares
        # quickly)
        {"name": "amr_128_f64", "kind": "amr", "nx": 128, "ny": 128, "nz": 64, "nbox": 256, "box_seed": 3,
         "steps": 6, "graph": False},
        # gradient of the flow objective through autograd, every state kept
        {"name": "adjoint_96", "kind": "adjoint", "nx": 96, "ny": 80, "nz": 64, "steps": 40, "every": -1},
    ]


def _log(rng, lo, hi) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _extents(rng, lo_cells, hi_cells, min_edge, max_edge):
    """Extents with a cell count log-uniform in [lo_cells, hi_cells], uneven
    and often odd."""
    cells = math.exp(rng.uniform(math.log(lo_cells), math.log(hi_cells)))
    e = cells ** (1.0 / 3.0)
    a, b = rng.uniform(0.7, 1.4), rng.uniform(0.7, 1.4)
    n = [int(e * a), int(e * b), int(e / (a * b))]
    return [max(min_edge, min(max_edge, k)) for k in n]


def draw(rng) -> dict:
    kind = rng.choice(["flow"] * 6 + ["diagnostics", "fab", "stages", "amr", "adjoint"])
    if kind == "flow":
        flow = rng.choice(["periodic", "channel", "channel", "profile", "cylinder", "pressure"])
        storage = rng.choice(["f64", "f64", "f32s", "f16s"])
        if flow == "cylinder":
            nx, ny, nz = _log(rng, 240, 700), _log(rng, 90, 150), rng.choice([4, 4, 6, 8])
            storage = "f64"
        else:
            nx, ny, nz = _extents(rng, 2e4, 1.2e7 if storage == "f64" else 2.4e7, 20, 400)
        cells = nx * ny * nz
        steps = rng.randint(2, 12) if cells < 2e6 else rng.randint(2, 4)
        return {"kind": "flow", "flow": flow, "nx": nx, "ny": ny, "nz": nz, "storage": storage, "steps": steps,
                "tuned": False, "forces": flow == "cylinder"}
    if kind == "diagnostics":
        nx, ny, nz = _extents(rng, 6e4, 8e6, 24, 320)
        return {"kind": kind, "flow": "channel", "nx": nx, "ny": ny, "nz": nz,
                "storage": rng.choice(["f64", "f32s", "f16s"])}
    if kind in ("fab", "stages"):
        nx, ny, nz = _extents(rng, 3e4, 1.5e6, 18, 160)
        case = {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "max_box": rng.choice([16, 24, 32, 64])}
        if kind == "fab":
            case["steps"] = rng.randint(1, 6)
        return case
    if kind == "amr":
        # extents are multiples of the largest box edge
        nx, ny, nz = 64 * rng.choice([1, 2]), 64 * rng.choice([1, 2]), 64
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "nbox": int(rng.uniform(0.4, 1.6) * nx * ny * nz / 4096),
                "box_seed": rng.randint(0, 999), "steps": rng.randint(1, 5), "graph": rng.random() < 0.3}
    nx, ny, nz = _extents(rng, 3e4, 4e5, 20, 120)
    return {"kind": "adjoint", "nx": nx, "ny": ny, "nz": nz, "steps": rng.randint(8, 30),
            "every": rng.choice([-1, 0])}


def _ncell(case):
    return case["nx"], case["ny"], case["nz"]


def _cfg(case) -> dict:
    """The workload description (physics, boundaries, body) of a case."""
    n = _ncell(case)
    flow = case.get("flow", "periodic")
    if flow == "channel":
        r = max(3.0, 0.094 * min(n))
        return configs.channel_sphere(n, radius=r, center=(n[0] // 4 + 4.0, n[1] / 2.0, n[2] / 2.0), tau=0.55)
    if flow == "profile":
        return configs.channel_profile(n, kind="channel", tau=0.55)
    if flow == "pressure":
        return configs.pressure_case("outlet", ncell=n)
    if flow == "cylinder":
        cfg = configs.cylinder_deck("turek_2d2")
        if n != cfg["ncell"]:
            # another channel of the deck's family, the body scaled with the height
            s = n[1] / 123.0
            cfg.update(ncell=n, prob_lo=(0.0, 0.0, -n[2] / 2.0), prob_hi=(float(n[0]), float(n[1]), n[2] / 2.0))
            cfg["eb"] = dict(cfg["eb"], center=(60.0 * s, 60.0 * s, 0.0), radius=15.0 * s)
        return cfg
    tau, t0 = 0.55, 0.2
    return {
        "name": "periodic_{}x{}x{}".format(*n), "ncell": n, "periodic": (1, 1, 1), "prob_lo": (0.0, 0.0, 0.0),
        "prob_hi": tuple(float(k) for k in n), "bc_lo": (0, 0, 0), "bc_hi": (0, 0, 0), "velocity_bc": None,
        "nu": (tau - 0.5) * t0, "T0": t0, "ic": {"type": "constant", "density": 1.0, "mach": (0.0, 0.0, 0.0),
                                                 "temperature": t0},
        "eb": {"type": "all_regular"}, "max_box": case.get("max_box"),
    }


def _fields(case, cfg, seed):
    """(rho, u, v, w, T) over the domain, each (nz, ny, nx): the workload's
    initial state plus two seeded separable Fourier modes per field."""
    n = _ncell(case)
    g = torch.Generator().manual_seed(1000003 * int(seed) + 17)
    gamma = cfg["ic"].get("adiabatic_exponent", 5.0 / 3.0)
    t0 = cfg["ic"].get("temperature", cfg["T0"])
    cs = math.sqrt(gamma * t0)
    u0 = [m * cs for m in cfg["ic"].get("mach", (0.0, 0.0, 0.0))]
    small = case.get("flow") == "cylinder"
    amp = [1e-3, 5e-4, 5e-4, 5e-4, 1e-3 * t0] if small else [1e-2, 0.02, 0.02, 0.02, 0.02 * t0]
    base = [cfg["ic"].get("density", 1.0), *u0, t0]
    out = []
    for b, a in zip(base, amp):
        acc = torch.full((n[2], n[1], n[0]), b, dtype=torch.float64)
        for _ in range(2):
            k = torch.randint(1, 4, (3,), generator=g)
            ph = torch.rand(3, generator=g, dtype=torch.float64) * (2.0 * math.pi)
            ax = [torch.cos(2.0 * math.pi * k[d] * (torch.arange(n[d], dtype=torch.float64) + 0.5) / n[d] + ph[d])
                  for d in range(3)]
            acc += (0.5 * a * ax[2])[:, None, None] * ax[1][None, :, None] * ax[0][None, None, :]
        out.append(acc)
    return out


def _level(case, cfg, seed):
    boxed = case["kind"] in ("fab", "stages")
    storage = case.get("storage", "f64")
    boxes = configs.chop_boxes(cfg["ncell"], cfg.get("max_box")) if boxed else None
    lvl = Level(cfg["ncell"], cfg["periodic"], cfg["prob_lo"], cfg["prob_hi"], boxes=boxes, ng=3 if boxed else 0,
                layout="fab" if boxed else "compact", storage=storage)
    gamma = cfg.get("adiabatic_exponent", 5.0 / 3.0)
    lvl.set_phys(cfg["nu"], cfg.get("alpha"), adiabatic_exponent=gamma)
    lvl.set_bc(cfg["bc_lo"], cfg["bc_hi"], cfg.get("velocity_bc"))
    if storage != "f64":
        lvl.set_shift_state(*configs.reference_state(cfg))
    configs.set_eb_flags(lvl, cfg["eb"])
    fields = [f.numpy() for f in _fields(case, cfg, seed)]
    if boxed:
        fields = [np.concatenate([_fab(f, lo, hi, 3).ravel() for lo, hi in boxes]) for f in fields]
    lvl.init_fields(*fields, adiabatic_exponent=gamma)
    return lvl


def _fab(dom, lo, hi, ng):
    """The box [lo, hi] grown by ng out of a periodic domain array (..., nz, ny, nx)."""
    n = dom.shape[::-1]
    ix = [np.arange(lo[d] - ng, hi[d] + ng + 1) % n[d] for d in range(3)]
    return dom[..., ix[2][:, None, None], ix[1][None, :, None], ix[0][None, None, :]]


class _Device:
    """Device memory of the engine, wrapped for torch (no copy); keeps its
    owner alive for as long as a tensor looks at it."""

    def __init__(self, owner, ptr, count, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": typestr, "data": (ptr, False), "version": 3,
                                         "strides": None}


def _populations(state, lvl, lattice=0):
    """Torch view of a level's current populations: on the box layout one
    lattice (boxes back to back, 27 components each, ghosts included), on
    the compact layout both (27, cells, 2)."""
    ptr, nbytes = lvl.population_ptr(lattice)
    key = (ptr, lattice)
    view = state["views"].get(key)
    if view is None:
        es = 8 if lvl.storage == "f64" else 4
        count = nbytes // es * (2 if lvl.layout == "compact" else 1)
        owner = state.get("hierarchy", lvl)
        view = torch.as_tensor(_Device(owner, ptr, count, "<f8" if es == 8 else "<f4"), device="cuda")
        state["views"][key] = view
    return view


def _stream():
    return torch.cuda.current_stream().cuda_stream


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case, "views": {}}
    if kind == "amr":
        cfg = configs.amr_two_level(ncell=_ncell(case), nbox=case["nbox"], seed=case["box_seed"])
        cfg["ic"]["seed"] = int(seed)
        st["hierarchy"] = Hierarchy(cfg)
        return st
    if kind == "adjoint":
        ns, tau, u0 = _adjoint_inputs(case, seed)
        st["solver"] = IsoSolver(_ncell(case), T0=1.0 / 3.0, u_in=0.04)
        st["params"] = [t.cuda().requires_grad_() for t in (ns, tau, u0)]
        return st
    cfg = _cfg(case)
    lvl = st["level"] = _level(case, cfg, seed)
    cells = case["nx"] * case["ny"] * case["nz"]
    if kind == "flow" and case["tuned"]:
        lvl.autotune(reps=3, stream=_stream())
    if kind == "diagnostics":
        st["macro"] = torch.empty(5 * cells, dtype=torch.float64, device="cuda")
        st["vort"] = torch.empty(4 * cells, dtype=torch.float64, device="cuda")
        st["tags"] = torch.empty(cells, dtype=torch.uint8, device="cuda")
    if case.get("storage") == "f16s":
        st["macro"] = torch.empty(5 * cells, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    return st


def run(state):
    case = state["case"]
    kind = case["kind"]
    s = _stream()
    if kind == "flow":
        lvl = state["level"]
        lvl.advance(case["steps"], stream=s)
        if case["storage"] == "f16s":
            lvl.macro_fields(state["macro"], stream=s)
            return {"macro": state["macro"]}
        out = {"populations": _populations(state, lvl)}
        if case["forces"]:
            out["force"] = lvl.eb_force(stream=s)
        return out
    if kind == "diagnostics":
        lvl = state["level"]
        lvl.macro_fields(state["macro"], stream=s)
        lvl.vorticity(state["vort"], stream=s)
        cells = state["tags"].numel()
        lvl.tag_cells(state["vort"][3 * cells:], "greater", 2e-3, state["tags"], stream=s)
        return {"macro": state["macro"], "vorticity": state["vort"], "tags": state["tags"],
                "conservation": lvl.conservation(stream=s)}
    if kind == "fab":
        lvl = state["level"]
        lvl.advance(case["steps"], stream=s)
        for lattice in (0, 1):
            lvl.fillpatch(lattice, stream=s)
        return [_populations(state, lvl, lattice) for lattice in (0, 1)]
    if kind == "stages":
        lvl = state["level"]
        for lattice in (0, 1):
            lvl.fillpatch(lattice, stream=s)
        for lattice in (0, 1):
            lvl.stream(lattice, stream=s)
        lvl.collide(stream=s)
        return [_populations(state, lvl, lattice) for lattice in (0, 1)]
    if kind == "amr":
        h = state["hierarchy"]
        h.advance(case["steps"], stream=s, graph=case["graph"])
        # every ghost layer of both levels, as before an output or a stage call
        for lattice in (0, 1):
            h.crse.fillpatch(lattice, stream=s)
            h.explode(lattice, stream=s)
        return [_populations(state, lvl, lattice) for lvl in h.levels for lattice in (0, 1)]
    ns, tau, u0 = state["params"]
    loss = flow_loss(state["solver"], ns, tau, u0, case["steps"], case["every"])
    return [loss.detach(), *torch.autograd.grad(loss, (ns, tau, u0))]


# ---------------------------------------------------------------------------
# the work a pass cannot do without
# ---------------------------------------------------------------------------

_FLOPS_THERMAL = 900  # moments, equilibria and relaxation of 54 populations
_FLOPS_ISO = 450


def work(case) -> dict:
    """Bytes: every population of every update read once and written once
    (the lattice-update roofline's convention: a step is one sweep over the
    state), and each further output written once."""
    cells = case["nx"] * case["ny"] * case["nz"]
    kind = case["kind"]
    per_update = {"f64": 864, "f32s": 432, "f16s": 216}[case.get("storage", "f64")]
    if kind == "flow":
        extra = 40 * cells + per_update // 2 * cells if case["storage"] == "f16s" else 0
        return {"bytes": cells * case["steps"] * per_update + extra, "flops": cells * case["steps"] * _FLOPS_THERMAL}
    if kind == "diagnostics":
        return {"bytes": cells * (per_update // 2 + 40 + 32 + 1), "flops": cells * 200}
    if kind in ("fab", "stages"):
        steps = case.get("steps", 1)
        return {"bytes": cells * steps * per_update, "flops": cells * steps * _FLOPS_THERMAL}
    if kind == "amr":
        cfg = configs.amr_two_level(ncell=_ncell(case), nbox=case["nbox"], seed=case["box_seed"])
        fine = sum(math.prod(h - l + 1 for l, h in zip(lo, hi)) for lo, hi in cfg["fine_boxes"])
        updates = (cells + 2 * fine) * case["steps"]
        return {"bytes": updates * per_update, "flops": updates * _FLOPS_THERMAL}
    # forward: read and write the state; reverse: read the kept state and the
    # adjoint state, write the adjoint state; the gradients once
    steps = case["steps"]
    return {"bytes": cells * steps * 27 * 8 * 5 + cells * 8 * 8, "flops": cells * steps * _FLOPS_ISO * 3}


# ---------------------------------------------------------------------------
# the same results in plain torch at 64 bits
# ---------------------------------------------------------------------------

_C = [(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1),
      (1, 1, 0), (-1, -1, 0), (1, -1, 0), (-1, 1, 0), (1, 0, 1), (-1, 0, -1), (1, 0, -1), (-1, 0, 1),
      (0, 1, 1), (0, -1, -1), (0, 1, -1), (0, -1, 1),
      (1, 1, 1), (-1, -1, -1), (1, -1, 1), (-1, 1, -1), (1, -1, -1), (-1, 1, 1), (1, 1, -1), (-1, -1, 1)]
_OPP = [_C.index(tuple(-a for a in c)) for c in _C]
_W = [{0: 8.0 / 27.0, 1: 2.0 / 27.0, 2: 1.0 / 54.0, 3: 1.0 / 216.0}[sum(a * a for a in c)] for c in _C]


def _exact_device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _phi(c, u, p):
    return c * 0.5 * u + abs(c) * (1.5 * p - 1.0) - p + 1.0


def _feq(q, rho, u, p):
    c = _C[q]
    return rho * _phi(c[0], u[0], p[0]) * _phi(c[1], u[1], p[1]) * _phi(c[2], u[2], p[2])


def _g_state(rho, u, temp, energy2, cv):
    """Heat flux and second-moment coefficients of the energy equilibrium; the
    temperature they use subtracts only u_x^2 (the reference's expansion)."""
    tv = 0.5 / cv * (energy2 / rho - u[0] * u[0] + u[1] * u[1] + u[2] * u[2])
    p = rho * tv
    h = energy2 / (2.0 * rho) + p / rho
    hp = h + p / rho
    q = [2.0 * rho * u[a] * h for a in range(3)]
    r = {(a, b): 2.0 * rho * u[a] * u[b] * hp + (2.0 * p * h if a == b else 0.0) for a in range(3)
         for b in range(a, 3)}
    return q, r


def _geq(k, energy2, qeq, r):
    c = _C[k]
    v = energy2
    for a in range(3):
        if c[a]:
            v = v + 3.0 * c[a] * qeq[a]
    for a in range(3):
        v = v + 4.5 * (c[a] * c[a] - 1.0 / 3.0) * (r[a, a] - energy2 / 3.0)
        for b in range(a + 1, 3):
            if c[a] * c[b]:
                v = v + 9.0 * c[a] * c[b] * r[a, b]
    return _W[k] * v


def _equilibrium(rho, u, temp, gamma):
    """f and g equilibria of a prescribed state (gas constant 1), (27, ...)."""
    cv = 1.0 / (gamma - 1.0)
    p = [u[a] * u[a] + temp for a in range(3)]
    e2 = rho * (2.0 * cv * temp + u[0] * u[0] + u[1] * u[1] + u[2] * u[2])
    qeq, r = _g_state(rho, u, temp, e2, cv)
    f = torch.stack([_feq(k, rho, u, p) for k in range(27)])
    return f, torch.stack([_geq(k, e2, qeq, r) for k in range(27)])


def _fluid(cfg, dev):
    """1 where a cell is fluid: a cell is solid when all 8 of its nodes lie in the body."""
    n = cfg["ncell"]
    eb = cfg["eb"]
    if eb["type"] == "all_regular":
        return torch.ones(n[2], n[1], n[0], dtype=torch.bool, device=dev)
    nodes = [cfg["prob_lo"][d] + torch.arange(n[d] + 1, dtype=torch.float64, device=dev) - eb["center"][d]
             for d in range(3)]
    d2 = nodes[0][None, None, :] ** 2 + nodes[1][None, :, None] ** 2
    if eb["type"] == "sphere":
        d2 = d2 + nodes[2][:, None, None] ** 2
    inside = (d2 <= eb["radius"] ** 2).expand(n[2] + 1, n[1] + 1, n[0] + 1)
    solid = torch.ones(n[2], n[1], n[0], dtype=torch.bool, device=dev)
    for a in (0, 1):
        for b in (0, 1):
            for c in (0, 1):
                solid &= inside[c:c + n[2], b:b + n[1], a:a + n[0]]
    return ~solid


class _Box:
    """A single-level domain with its boundaries, advanced in torch: pull with
    halfway bounce-back, then the collide.  Faces: periodic; velocity inlet at
    x-lo; outflow at x-hi; no-slip walls in y and z."""

    def __init__(self, cfg, fields, dev):
        self.cfg, self.dev = cfg, dev
        self.n = cfg["ncell"]
        self.gamma = cfg.get("adiabatic_exponent", 5.0 / 3.0)
        self.cv = 1.0 / (self.gamma - 1.0)
        self.fluid = _fluid(cfg, dev)
        fields = [x.to(dev) for x in fields]
        self.f, self.g = _equilibrium(fields[0], fields[1:4], fields[4], self.gamma)
        self.f *= self.fluid
        self.g *= self.fluid
        if not cfg["periodic"][0]:
            self._inlet()

    def _inlet(self):
        """Equilibria of the ghost column at x-lo over (27, nz + 2, ny + 2), indices shifted by one."""
        v, (nx, ny, nz) = self.cfg["velocity_bc"], self.n
        temp, gamma = v["initial_temperature"], v["adiabatic_exponent"]
        um = v["Mach_ref"] * math.sqrt(gamma * temp)
        jy = torch.arange(-1, ny + 1, dtype=torch.float64, device=self.dev)[None, :]
        jz = torch.arange(-1, nz + 1, dtype=torch.float64, device=self.dev)[:, None]
        if v["kind"] == "constant":
            ux = torch.full((nz + 2, ny + 2), um, dtype=torch.float64, device=self.dev)
        elif v["kind"] == "channel":
            ux = 16.0 * um * (jy * (ny - 1 - jy)) * (jz * (nz - 1 - jz)) / float(ny) ** 4
        else:
            y = jy + 0.5
            ux = (4.0 * um * y * (ny - y) / float(ny) ** 2).expand(nz + 2, ny + 2)
        zero = torch.zeros_like(ux)
        rho = torch.full_like(ux, v["initial_density"])
        self.inlet = _equilibrium(rho, [ux, zero, zero], torch.full_like(ux, temp), gamma)

    def _pull(self, pop, inlet):
        nx, ny, nz = self.n
        per = self.cfg["periodic"]
        out = torch.empty_like(pop)
        for q, (cx, cy, cz) in enumerate(_C):
            own = pop[_OPP[q]]
            v = torch.where(torch.roll(self.fluid, (cz, cy, cx), (0, 1, 2)), torch.roll(pop[q], (cz, cy, cx), (0, 1, 2)),
                            own)
            if not per[0]:
                if cx == 1:
                    v[:, :, 0] = inlet[q][1 - cz:1 - cz + nz, 1 - cy:1 - cy + ny]
                elif cx == -1:
                    v[:, :, nx - 1] = torch.roll(pop[q][:, :, nx - 1], (cz, cy), (0, 1))
            if not per[1] and cy:
                j = 0 if cy == 1 else ny - 1
                v[:, j] = own[:, j]
            if not per[2] and cz:
                k = 0 if cz == 1 else nz - 1
                v[k] = own[k]
            out[q] = v
        return out

    def _gradient(self, a, x):
        """Central difference, one-sided next to the domain's box or a solid cell."""
        ax = 2 - a
        n = x.shape[ax]
        pos = torch.arange(n, device=self.dev).view([-1 if d == ax else 1 for d in range(3)])
        up = torch.roll(self.fluid, -1, ax) & (pos < n - 1)
        lo = torch.roll(self.fluid, 1, ax) & (pos > 0)
        xp, xm = torch.roll(x, -1, ax), torch.roll(x, 1, ax)
        zero = torch.zeros((), dtype=x.dtype, device=self.dev)
        return torch.where(up & lo, 0.5 * (xp - xm), torch.where(up, xp - x, torch.where(lo, x - xm, zero)))

    def macro(self, f, g):
        rho = f.sum(0)
        safe = torch.where(self.fluid, rho, torch.ones_like(rho))
        u = [sum(f[q] * c[a] for q, c in enumerate(_C) if c[a]) / safe for a in range(3)]
        e2 = g.sum(0)
        temp = 0.5 / self.cv * (e2 / safe - (u[0] * u[0] + u[1] * u[1] + u[2] * u[2]))
        temp = torch.where(self.fluid, temp, torch.ones_like(temp))
        return safe, u, e2, temp

    def step(self):
        cfg = self.cfg
        self.f = self._pull(self.f, None if cfg["periodic"][0] else self.inlet[0])
        self.g = self._pull(self.g, None if cfg["periodic"][0] else self.inlet[1])
        f, g = self.f, self.g
        rho, u, e2, temp = self.macro(f, g)
        dq = [self._gradient(a, rho * u[a] * (1.0 - 3.0 * temp - u[a] * u[a])) for a in range(3)]
        alpha = cfg.get("alpha") or cfg["nu"]
        omega = 1.0 / (cfg["nu"] / temp + 0.5)
        ratio = 1.0 / (alpha / temp + 0.5) / omega
        corr = (2.0 - omega) / (2.0 * omega * rho)
        p = [u[a] * u[a] + temp + corr * dq[a] for a in range(3)]
        press = {}
        for a in range(3):
            for b in range(a, 3):
                press[a, b] = press[b, a] = sum(f[q] * (c[a] * c[b]) for q, c in enumerate(_C) if c[a] * c[b])
        qeq, r = _g_state(rho, u, temp, e2, self.cv)
        for a in range(3):
            flux = sum(g[q] * c[a] for q, c in enumerate(_C) if c[a])
            noneq = flux - 2.0 * (u[0] * press[a, 0] + u[1] * press[a, 1] + u[2] * press[a, 2]) - u[a] * dq[a]
            qeq[a] = ratio * qeq[a] + (1.0 - ratio) * noneq
        minus1 = torch.full((), -1.0, dtype=torch.float64, device=self.dev)
        for q in range(27):
            f[q] = torch.where(self.fluid, f[q] + omega * (_feq(q, rho, u, p) - f[q]), minus1)
            g[q] = torch.where(self.fluid, g[q] + omega * (_geq(q, e2, qeq, r) - g[q]), minus1)


def _exact_macro(box):
    rho, u, _, temp = box.macro(box.f, box.g)
    fields = [torch.where(box.fluid, x, torch.zeros_like(x)) for x in (rho, *u, temp)]
    return fields, torch.cat([x.reshape(-1) for x in fields])


def exact(case, seed):
    kind = case["kind"]
    if kind == "amr":
        return None  # two levels and their transfers have no short restatement
    dev = _exact_device()
    if kind == "adjoint":
        return _exact_adjoint(case, seed, dev)
    if case.get("flow") == "pressure":
        return None  # the pressure faces' sums have no short restatement
    cfg = _cfg(case)
    box = _Box(cfg, _fields(case, cfg, seed), dev)
    if kind == "diagnostics":
        fields, macro = _exact_macro(box)
        grad = [[torch.where(box.fluid, box._gradient(a, fields[1 + b]), torch.zeros_like(fields[0]))
                 for b in range(3)] for a in range(3)]
        w = [grad[1][2] - grad[2][1], grad[2][0] - grad[0][2], grad[0][1] - grad[1][0]]
        w.append(torch.sqrt(w[0] ** 2 + w[1] ** 2 + w[2] ** 2))
        fl = box.fluid
        sums = [(box.f.sum(0) * fl).sum()]
        sums += [(sum(box.f[q] * c[a] for q, c in enumerate(_C) if c[a]) * fl).sum() for a in range(3)]
        sums.append((box.g.sum(0) * fl).sum())
        return {"macro": macro, "vorticity": torch.cat([x.reshape(-1) for x in w]), "tags": None,
                "conservation": torch.stack(sums)}
    for _ in range(case.get("steps", 1)):
        box.step()
    if kind in ("fab", "stages"):
        out = []
        for pop in (box.f, box.g):
            pop = pop.cpu().numpy()
            out.append(torch.from_numpy(np.concatenate(
                [_fab(pop, lo, hi, 3).ravel() for lo, hi in _boxes(cfg)])))
        return out
    if case["storage"] == "f16s":
        return {"macro": _exact_macro(box)[1]}
    f, g = box.f, box.g
    if case["storage"] == "f32s":
        rho0, t0 = configs.reference_state(cfg)
        one = torch.ones((), dtype=torch.float64, device=dev)
        zero = torch.zeros((), dtype=torch.float64, device=dev)
        sf, sg = _equilibrium(rho0 * one, [zero] * 3, t0 * one, box.gamma)
        f, g = f - sf.view(27, 1, 1, 1), g - sg.view(27, 1, 1, 1)
    out = {"populations": torch.stack([f, g], dim=-1).reshape(-1)}
    if case["forces"]:
        out["force"] = _exact_force(box)
    return out


def _boxes(cfg):
    """The domain in boxes of at most cfg["max_box"] cells a side, x fastest."""
    m, n = cfg["max_box"], cfg["ncell"]
    return [((x, y, z), tuple(min(a + m, k) - 1 for a, k in zip((x, y, z), n)))
            for z in range(0, n[2], m) for y in range(0, n[1], m) for x in range(0, n[0], m)]


def _exact_force(box):
    """Momentum exchange: 2 c_q f_q(x - c_q) over solid cells x with a fluid
    face neighbour and fluid sources (none of them beyond a face here)."""
    fl = box.fluid
    near = torch.zeros_like(fl)
    for d in range(3):
        near |= torch.roll(fl, 1, d) | torch.roll(fl, -1, d)
    edge = near & ~fl
    out = torch.zeros(3, dtype=torch.float64, device=box.dev)
    for q, (cx, cy, cz) in enumerate(_C):
        hit = edge & torch.roll(fl, (cz, cy, cx), (0, 1, 2))
        s = (torch.roll(box.f[q], (cz, cy, cx), (0, 1, 2)) * hit).sum()
        for a in range(3):
            out[a] += 2.0 * _C[q][a] * s
    return out


# ---------------------------------------------------------------------------
# isothermal solver with partial bounce-back
# ---------------------------------------------------------------------------


def _adjoint_inputs(case, seed):
    """Solid fraction (smooth seeded blobs, about 15 % in the mean), tau, and
    a perturbed uniform initial velocity."""
    nx, ny, nz = _ncell(case)
    g = torch.Generator().manual_seed(7919 * int(seed) + 5)
    z, y, x = (torch.arange(n, dtype=torch.float64) for n in (nz, ny, nx))
    s = torch.zeros(nz, ny, nx, dtype=torch.float64)
    width = 2.0 * (min(nx, ny, nz) / 12.0) ** 2
    for _ in range(16):
        c = torch.rand(3, generator=g, dtype=torch.float64)
        s += (torch.exp(-(z - c[0] * nz) ** 2 / width)[:, None, None]
              * torch.exp(-(y - c[1] * ny) ** 2 / width)[None, :, None]
              * torch.exp(-(x - c[2] * nx) ** 2 / width)[None, None, :])
    s = s.clamp(0, 1)
    s = (s * (0.15 / s.mean())).clamp(0, 1)
    u0 = torch.zeros(3, nz, ny, nx, dtype=torch.float64)
    u0[0] = 0.04
    ph = torch.rand(3, 3, generator=g, dtype=torch.float64) * (2.0 * math.pi)
    for a in range(3):
        u0[a] += 0.004 * (torch.cos(2.0 * math.pi * z / nz + ph[a, 0])[:, None, None]
                          * torch.cos(2.0 * math.pi * y / ny + ph[a, 1])[None, :, None]
                          * torch.cos(2.0 * math.pi * x / nx + ph[a, 2])[None, None, :])
    tau = torch.tensor(0.6 + 0.05 * float(torch.rand((), generator=g)), dtype=torch.float64)
    return s, tau, u0


def _iso_step(f, ns, tau, inlet, rt):
    pulled = []
    for q, (cx, cy, cz) in enumerate(_C):
        v = torch.roll(f[q], (cz, cy), (0, 1))
        if cx == 1:
            v = torch.cat([inlet[q].expand_as(v[:, :, :1]), v[:, :, :-1]], 2)
        elif cx == -1:
            v = torch.cat([v[:, :, 1:], v[:, :, -1:]], 2)
        pulled.append(v)
    fs = torch.stack(pulled)
    rho = fs.sum(0)
    u = [sum(fs[q] * c[a] for q, c in enumerate(_C) if c[a]) / rho for a in range(3)]
    dq = []
    for a in range(3):
        x = rho * u[a] * (1.0 - 3.0 * rt - u[a] * u[a])
        ax, n = 2 - a, f.shape[3 - a]
        if n > 1:
            inner = 0.5 * (x.narrow(ax, 2, n - 2) - x.narrow(ax, 0, n - 2))
            lo = x.narrow(ax, 1, 1) - x.narrow(ax, 0, 1)
            hi = x.narrow(ax, n - 1, 1) - x.narrow(ax, n - 2, 1)
            dq.append(torch.cat([lo, inner, hi], ax))
        else:
            dq.append(torch.zeros_like(x))
    omega = 1.0 / tau
    corr = (2.0 - omega) / (2.0 * omega * rho)
    p = [u[a] * u[a] + rt + corr * dq[a] for a in range(3)]
    feq = torch.stack([_feq(q, rho, u, p) for q in range(27)])
    return (1.0 - ns) * (fs + omega * (feq - fs)) + ns * fs[_OPP]


def _exact_adjoint(case, seed, dev):
    ns, tau, u0 = (t.to(dev).requires_grad_() for t in _adjoint_inputs(case, seed))
    rt = 1.0 / 3.0
    one = torch.ones((), dtype=torch.float64, device=dev)
    zero = torch.zeros((), dtype=torch.float64, device=dev)
    uin = [0.04 * one, zero, zero]
    inlet = torch.stack([_feq(q, one, uin, [v * v + rt for v in uin]) for q in range(27)])
    rho = torch.ones(ns.shape, dtype=torch.float64, device=dev)
    u = [u0[0], u0[1], u0[2]]
    f = torch.stack([_feq(q, rho, u, [v * v + rt for v in u]) for q in range(27)])
    for _ in range(case["steps"]):
        f = torch.utils.checkpoint.checkpoint(_iso_step, f, ns, tau, inlet, rt, use_reentrant=False)
    rho = f.sum(0)
    u = [sum(f[q] * c[a] for q, c in enumerate(_C) if c[a]) / rho for a in range(3)]
    loss = u[0][:, :, -1].mean() + 1e-3 * (0.5 * rho * (u[0] ** 2 + u[1] ** 2 + u[2] ** 2)).sum()
    return [loss.detach(), *torch.autograd.grad(loss, (ns, tau, u0))]
