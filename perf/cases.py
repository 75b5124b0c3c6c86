"""Performance cases: what a user's program has the framework do, one pass per call of `run`.

A case is a dict of plain values.  Kinds:
  step       Simulation.step of one run (beam deposit, plasma sweep, beam push), one workgroup or several
  pipelined  Simulation.run_pipelined: a run's next time steps, several in flight
  batch      Batch.step: many independent runs in one launch, replayed as a graph
  gradient   SpreadObjective.value_and_grad: one step and its adjoint
  laser      Laser.step (one box) or laser_step_batched (several)
  deposit    beam_deposit of one beam, on the caller's device arrays
  advance    beam_advance of one beam, on the caller's device arrays
  thomas     thomas_batched, system-major or element-major
"""
import ctypes as C
import math
import os
import random
import tempfile

import numpy as np
import torch

import quarz_amd as qa
from quarz_amd import configs
from quarz_amd.witness import SpreadObjective


def listed():
    return [
        # The smallest run: a quick look at a short linear wake on a coarse grid; latency and launches count.
        {"name": "step_small", "kind": "step", "modes": 0, "cells": 64, "slices": 101, "dxi": 0.05, "ppc": 2, "ntheta": 1,
         "ions": False, "nd": 2000, "nw": 0, "groups": 0},
        # The everyday axisymmetric blowout run (256 cells, ppc 4, 1e5 driver particles), one step at a time.
        {"name": "step_m0", "kind": "step", "modes": 0, "cells": 256, "slices": 801, "dxi": 0.01, "ppc": 4, "ntheta": 1,
         "ions": False, "nd": 100000, "nw": 0, "groups": 0},
        # Modes 0 and 1 on the stretched 512-cell grid with driver and witness: the hosing study, one workgroup.
        {"name": "step_m1", "kind": "step", "modes": 1, "cells": 512, "slices": 401, "dxi": 0.01, "ppc": 1, "ntheta": 8,
         "ions": False, "nd": 60000, "nw": 30000, "groups": 0},
        # The largest plasma: 1024 cells, electrons and mobile ions, 32768 particles per slice; several workgroups.
        {"name": "step_m1_ions", "kind": "step", "modes": 1, "cells": 1024, "slices": 251, "dxi": 0.02, "ppc": 2,
         "ntheta": 8, "ions": True, "nd": 100000, "nw": 50000, "groups": 0},
        # A production run with its time steps in flight, each on several workgroups.
        {"name": "pipelined_m1", "kind": "pipelined", "modes": 1, "cells": 512, "slices": 401, "dxi": 0.01, "ppc": 1,
         "ntheta": 8, "ions": False, "nd": 60000, "nw": 30000, "groups": 6, "steps": 4, "depth": 4, "chunks": 16},
        # A parameter scan: independent axisymmetric runs of uneven cells and slices, the replayed batched step.
        {"name": "batch_m0", "kind": "batch", "runs": 60, "max_cells": 1024, "max_slices": 600, "beam": 4000},
        # The witness-profile optimisation: objective and gradient of one step by the adjoint.
        {"name": "gradient_m0", "kind": "gradient", "slices": 1100, "nd": 40000, "nw": 20000, "every": 64},
        # One laser pulse in a plasma channel, one time step.
        {"name": "laser_one", "kind": "laser", "boxes": 1, "nodes": 321, "slices": 401, "scheme": "bdf2",
         "circular": False, "plasma": True},
        # A scan of laser pulses of uneven grids and boxes, one time step of all of them.
        {"name": "laser_scan", "kind": "laser", "boxes": 40, "nodes": 513, "slices": 301, "scheme": "trapezoid",
         "circular": True, "plasma": True},
        # The sources of a full-size beam in modes 0 and 1.
        {"name": "deposit_m1", "kind": "deposit", "modes": 1, "cells": 512, "slices": 1001, "np": 1500000, "ngp": False},
        # The push of a full-size beam against the stored fields of modes 0 and 1.
        {"name": "advance_m1", "kind": "advance", "modes": 1, "cells": 512, "slices": 1001, "np": 1500000, "pusher": 0},
        # Many independent tridiagonal systems, stored one after another.
        {"name": "thomas_rows", "kind": "thomas", "nodes": 513, "batch": 4096, "element_major": False},
    ]


# ---------------------------------------------------------------------------------------------------- drawn cases
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "pipelined", "batch", "gradient", "laser", "laser", "deposit", "advance", "thomas", "thomas"])
    if kind in ("step", "pipelined"):
        m1 = rng.random() < 0.5
        cells = _log(rng, 48, 512 if m1 else 1024)
        ntheta = rng.choice([4, 8]) if m1 else rng.choice([1, 2])
        ppc = 1 if m1 else rng.randint(1, 4)
        ions = rng.random() < 0.25
        groups = rng.choice([0, 0, 2, 3, 5]) if kind == "step" else rng.choice([1, 2, 4, 6])
        if cells * ppc * ntheta * (2 if ions else 1) > 4096:
            ppc, ions = 1, False
        case = {"kind": kind, "modes": int(m1), "cells": cells, "slices": _log(rng, 80, 380 if m1 else 800),
                "dxi": rng.choice([0.01, 0.02]), "ppc": ppc, "ntheta": ntheta, "ions": ions, "nd": _log(rng, 1000, 100000),
                "nw": rng.choice([0, _log(rng, 1000, 50000)]), "groups": groups}
        if kind == "pipelined":
            case.update(steps=rng.randint(2, 4), depth=rng.randint(2, 4), chunks=rng.randint(4, 16))
        return case
    if kind == "batch":
        return {"kind": kind, "runs": rng.randint(3, 60), "max_cells": rng.choice([256, 512, 1024]),
                "max_slices": _log(rng, 120, 600), "beam": _log(rng, 500, 4000)}
    if kind == "gradient":
        return {"kind": kind, "slices": rng.randint(1041, 1100), "nd": _log(rng, 5000, 40000), "nw": _log(rng, 2000, 20000),
                "every": rng.choice([32, 64, 100])}
    if kind == "laser":
        one = rng.random() < 0.5
        return {"kind": kind, "boxes": 1 if one else rng.randint(2, 40), "nodes": _log(rng, 40, 1025 if one else 513),
                "slices": _log(rng, 40, 301), "scheme": rng.choice(["trapezoid", "bdf2", "euler"]),
                "circular": rng.random() < 0.5, "plasma": rng.random() < 0.7}
    if kind == "deposit":
        return {"kind": kind, "modes": rng.choice([0, 1]), "cells": _log(rng, 64, 512), "slices": _log(rng, 64, 1001),
                "np": _log(rng, 2000, 1500000), "ngp": rng.random() < 0.3}
    if kind == "advance":
        return {"kind": kind, "modes": rng.choice([0, 1]), "cells": _log(rng, 64, 512), "slices": _log(rng, 64, 1001),
                "np": _log(rng, 2000, 1500000), "pusher": rng.choice([0, 0, 1, 2, 3])}
    return {"kind": kind, "nodes": _log(rng, 9, 513), "batch": _log(rng, 3, 4096), "element_major": rng.random() < 0.5}


# ---------------------------------------------------------------------------------------------- decks and device views
class _View:
    """A device array of the library as an object that torch wraps without a copy; the tensor keeps its owner alive."""

    def __init__(self, ptr, shape, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f8", "data": (int(ptr), False), "version": 2}


def _view(ptr, shape, owner):
    return torch.as_tensor(_View(ptr, shape, owner), device="cuda")


class _Species(C.Structure):
    _fields_ = [(n, C.c_void_p) for n in ("x", "y", "px", "py", "dl", "w", "hist")] + [
        ("np", C.c_int), ("cap", C.c_int), ("q", C.c_double), ("m", C.c_double)]


class _Sweep(C.Structure):
    """qz_sweep_args up to its species (include/quarz_amd.h)."""
    _fields_ = [("grid", qa.RadialGridC), ("modes", C.c_int), ("picard", C.c_int), ("nslices", C.c_int), ("k_begin", C.c_int),
                ("k_end", C.c_int), ("ab_order", C.c_int), ("ngp", C.c_int), ("dxi", C.c_double), ("delta_min", C.c_double),
                ("max_qsa", C.c_double), ("ab_c", C.c_double * 5), ("op", C.c_void_p * 12), ("flux_coef", C.c_double),
                ("grad", C.c_void_p * 4), ("fac", C.c_void_p * 4), ("bsrc", C.c_void_p), ("ncb", C.c_int),
                ("bg", C.c_void_p), ("fld", C.c_void_p), ("ncf", C.c_int), ("diag", C.c_void_p), ("ncd", C.c_int),
                ("nspecies", C.c_int), ("sp", _Species * 2)]


def _sim_views(sim):
    """The run's device arrays, as its argument block names them: fields, diagnostics, sources, plasma state."""
    block = C.create_string_buffer(max(8192, int(qa.lib().qz_sweep_args_bytes())))
    qa.check(qa.lib().qz_sim_prepare_sweep(sim.h, block))
    a = _Sweep.from_buffer(block)
    out = {"fld": _view(a.fld, (sim.K, sim.M, sim.NCF), sim), "diag": _view(a.diag, (sim.K, sim.M, sim.NCD), sim),
           "bsrc": _view(a.bsrc, (sim.K, sim.M, sim.NCB), sim)}
    for s in range(a.nspecies):
        for name in ("x", "y", "px", "py", "dl", "w"):
            out["sp%d.%s" % (s, name)] = _view(getattr(a.sp[s], name), (a.sp[s].np,), sim)
    return out


_GRIDS = {}


def _grid(cells, axis=None, wall=0.05):
    """(nodes, path of a grid file) of `cells` stretched cells, the smallest at the axis."""
    key = (cells, axis, wall)
    if key not in _GRIDS:
        h0 = 1e-3 if axis is None else axis
        reach = sum(min(h0 * 1.05 ** c, wall) for c in range(cells))
        R = min(10.0, reach)
        if reach < 4.0:   # few cells: a uniform grid
            nodes = [4.0 * j / cells for j in range(cells + 1)]
        else:
            nodes, _ = configs.stretched_nodes(cells, R, h0, wall)
        fd, path = tempfile.mkstemp(prefix="quarz_grid_", suffix=".txt")
        with os.fdopen(fd, "w") as f:
            f.writelines("%.17g\n" % x for x in nodes)
        _GRIDS[key] = (nodes, path)
    return _GRIDS[key]


def _beam(name, n, n0, sr, sxi, xi0, seed, x0=0.0):
    return {name + ".n0": n0, name + ".sigma_r": sr, name + ".sigma_xi": sxi, name + ".x0": x0, name + ".xi0": xi0,
            name + ".gamma": 2000, name + ".espread": 0.01, name + ".emit_n": 0.002, name + ".cut": 3,
            name + ".nparticles": n, name + ".seed": seed}


def _sim(cells, slices, dxi, modes, ppc, ntheta, ions, nd, nw, groups, seed):
    rnd = random.Random(seed)
    L = (slices - 1) * dxi
    s = min(1.0, L / 10)
    keys = {"xi.convention": "z-t", "modes": modes, "grid.type": "file", "grid.file": _grid(cells)[1], "xi.min": "%.6f" % -L,
            "xi.max": 0, "xi.step": dxi, "time.dt": 10, "time.steps": 1000000, "pusher.beam": "vay", "pusher.ab_order": 3,
            "plasma.species": "electrons ions" if ions else "electrons", "electrons.ppc": ppc, "electrons.ntheta": ntheta,
            "beams": "driver witness" if nw else "driver", "sweep.groups": groups}
    if modes:
        keys["solver.picard"] = 3
    if ions:
        keys.update({"ions.charge": 1, "ions.mass": 1836, "ions.mobile": 1, "ions.ppc": ppc, "ions.ntheta": ntheta})
    keys.update(_beam("driver", nd, "%.6f" % rnd.uniform(1.5, 3), 0.3, s, -3.2 * s, rnd.randint(1, 10 ** 8),
                      "%.6f" % (rnd.uniform(0.02, 0.1) if modes else 0)))
    if nw:
        keys.update(_beam("witness", nw, "%.6f" % rnd.uniform(1, 4), 0.1, 0.03 * L, -0.85 * L, rnd.randint(1, 10 ** 8)))
    return qa.Simulation("\n".join("%s = %s" % kv for kv in keys.items()))


def _seeded(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _kernel_grid(cells):
    """(nodes, 1 / h, 1 / hat volumes) of the stretched grid, on the host."""
    r = np.asarray(_grid(cells)[0])
    h = np.diff(r)
    V = np.zeros(cells + 1)
    V[1:] += r[:-1] * h / 2 + h * h / 3
    V[:-1] += r[:-1] * h / 2 + h * h / 6
    return r, 1 / h, 1 / (2 * np.pi * V)


def _beam_particles(n, slices, dxi, seed):
    """A bunch of n particles in the order of their sampling, as a beam is made."""
    g = _seeded(seed)
    draw = lambda: torch.randn(n, generator=g, device="cuda", dtype=torch.float64)  # noqa: E731
    L = (slices - 1) * dxi
    p = {"x": 0.3 * draw() + 0.05, "y": 0.3 * draw(), "px": 0.01 * draw(), "py": 0.01 * draw(), "pz": 2000 + 20 * draw(),
         "xi": (0.5 * L + 0.15 * L * draw()).clamp(0.0, L), "w": 1e-5 * (0.5 + torch.rand(n, generator=g, device="cuda", dtype=torch.float64))}
    return p


def _scan_runs(case):
    """(cells, slices, driver particles) of every run of a scan; the sizes do not depend on the inputs' seed."""
    rnd = random.Random(case["runs"])
    out = [(case["max_cells"], case["max_slices"], case["beam"])]
    while len(out) < case["runs"]:
        out.append((rnd.choice([c for c in (128, 256, 384, 512, 768, 1024) if c <= case["max_cells"]]),
                    rnd.randint(max(60, case["max_slices"] // 8), case["max_slices"]),
                    rnd.randint(case["beam"] // 4, case["beam"])))
    return out


def _laser_sizes(case):
    """(nodes, slices) of every box; the sizes do not depend on the inputs' seed."""
    rnd = random.Random(case["boxes"])
    out = [(case["nodes"], case["slices"])]
    while len(out) < case["boxes"]:
        out.append((rnd.randint(max(20, case["nodes"] // 2), case["nodes"]),
                    rnd.randint(max(20, case["slices"] // 2), case["slices"])))
    return out


# -------------------------------------------------------------------------------------------------------------- prepare
def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind in ("step", "pipelined"):
        sim = _sim(case["cells"], case["slices"], case["dxi"], case["modes"], case["ppc"], case["ntheta"], case["ions"],
                   case["nd"], case["nw"], case["groups"], seed)
        st["out"] = _sim_views(sim)
        if kind == "pipelined":
            sim.step()   # a pipelined run goes on from a started one
        st["sim"] = sim
    elif kind == "batch":
        rnd = random.Random(seed)
        sims = [_sim(cells, slices, 0.01, 0, 4, 1, False, n, max(n // 3, 100), 1, rnd.randint(1, 10 ** 8))
                for cells, slices, n in _scan_runs(case)]
        st["out"] = [_sim_views(s)["fld"] for s in sims]
        b = qa.Batch(sims, graph=True)
        b.step()   # the start-up step of the beams, then the step whose graph is kept
        b.step()
        st["batch"], st["sims"] = b, sims
    elif kind == "gradient":
        deck = configs.c4_deck(nd=case["nd"], nw=case["nw"])
        rnd = random.Random(seed)
        over = {"xi.min": "%.2f" % (-(case["slices"] - 1) * 0.01), "driver.seed": rnd.randint(1, 10 ** 8),
                "witness.seed": rnd.randint(1, 10 ** 8)}
        st["objective"] = SpreadObjective(deck, beam=1, nseg=configs.C4_SEGMENTS, overrides=over, method="adjoint",
                                          every=case["every"])
        st["profile"] = np.array(configs.c4_initial_profile(seed))
        st["out"] = {"fld": _sim_views(st["objective"].sims[0])["fld"]}
    elif kind == "laser":
        st["lasers"], st["chi"] = [], []
        for K, nodes, scheme, p, chi in _laser_boxes(case, seed):
            L = qa.Laser(nodes, K, 0.0, 0.05, 2.0, p["k0"], scheme=scheme, circular=case["circular"])
            L.gaussian(p["a0"], p["w0"], p["L0"], p["xi0"], p["focus"])
            st["lasers"].append(L)
            st["chi"].append(None if chi is None else torch.from_numpy(chi).cuda())
    elif kind in ("deposit", "advance"):
        r, ih, iv = _kernel_grid(case["cells"])
        st["arrays"] = [torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (r, ih, iv)]
        st["grid"] = qa.radial_grid(*st["arrays"])
        K, dxi = case["slices"], 0.01
        st["box"] = qa.BeamGridC(0.0, dxi, K, 0, K, 1 if case.get("ngp") else 0)
        st["p"] = _beam_particles(case["np"], K, dxi, seed)
        if kind == "deposit":
            st["bsrc"] = torch.zeros(K, case["cells"] + 1, 15 if case["modes"] else 5, dtype=torch.float64, device="cuda")
            st["work"] = torch.empty(qa.beam_deposit_workspace_bytes(case["np"], K, case["cells"]), dtype=torch.uint8,
                                     device="cuda")
        else:
            st["fld"] = _fields(case, seed, st["arrays"][0])
    else:
        g = _seeded(seed)
        rnd = lambda: torch.rand(case["batch"], case["nodes"], generator=g, device="cuda", dtype=torch.float64)  # noqa: E731
        a, c = rnd() - 0.5, rnd() - 0.5
        sys = [a, 2 + rnd(), c, rnd() - 0.5]   # diagonally dominant
        if case["element_major"]:
            sys = [v.t().contiguous() for v in sys]
        st["sys"] = sys
        st["x"] = torch.zeros_like(sys[3])
        n = int(qa.lib().qz_tridiag_workspace_doubles(case["nodes"], case["batch"]))
        st["work"] = torch.empty(n, dtype=torch.float64, device="cuda")
    return st


def _laser_boxes(case, seed):
    """(slices, nodes, scheme, pulse, susceptibility) of every box of a case, on the host."""
    rnd = random.Random(seed)
    rng = np.random.default_rng(seed)
    out = []
    for M, K in _laser_sizes(case):
        nodes = 14.0 * (np.arange(M) / (M - 1)) ** rnd.uniform(1.0, 1.3)
        p = {"k0": rnd.uniform(10, 25), "a0": rnd.uniform(0.1, 2), "w0": rnd.uniform(2, 3.5), "L0": rnd.uniform(1.0, 2.0),
             "xi0": 0.025 * K, "focus": rnd.uniform(-20, 40)}
        chi = None
        if case["plasma"]:   # a channel with a density ramp along the box
            chi = 0.5 * np.linspace(0.5, 1.5, K)[:, None] * (1 + nodes[None, :] ** 2 / 16) * (1 + 0.05 * rng.standard_normal((K, M)))
        out.append((K, nodes, case["scheme"], p, chi))
    return out


def _fields(case, seed, r):
    """Stored fields that focus the beam (E_r = r / 2) with small oscillations in every component."""
    K, M, nc = case["slices"], case["cells"] + 1, 18 if case["modes"] else 6
    g = _seeded(seed + 1)
    ph = 6.28 * torch.rand(nc, generator=g, device="cuda", dtype=torch.float64)
    k = torch.arange(K, device="cuda", dtype=torch.float64) * 0.01
    f = 1e-3 * torch.sin(k[:, None, None] + r[None, :, None] + ph)
    f[:, 0] = 0
    f[:, :, 0] += 0.5 * r
    return f.contiguous()


# ------------------------------------------------------------------------------------------------------------------ run
def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "step":
        sim = st["sim"]
        sim.step()
        return [st["out"]] + [sim.beam(b) for b in range(sim.nbeams)]
    if kind == "pipelined":
        sim = st["sim"]
        work = sim.run_pipelined(case["steps"], chunks=case["chunks"], depth=case["depth"])
        return [st["out"], work] + [sim.beam(b) for b in range(sim.nbeams)]
    if kind == "batch":
        st["batch"].step()
        return st["out"]
    if kind == "gradient":
        J, grad = st["objective"].value_and_grad(st["profile"])
        return {"J": float(J), "grad": grad, "fld": st["out"]["fld"]}
    if kind == "laser":
        ls = st["lasers"]
        if len(ls) == 1:
            ls[0].step(st["chi"][0])
        else:
            qa.laser_step_batched(ls, st["chi"])
        out = []
        for L in ls[:30]:   # envelope and ponderomotive arrays where they are
            for what, n in ((0, 2), (1, 3)):
                p = C.c_void_p()
                qa.check(qa.lib().qz_laser_device(L.h, what, C.byref(p)))
                out.append(_view(p.value, (L.K, L.M, n), L))
        return out
    if kind == "deposit":
        st["bsrc"].zero_()
        qa.beam_deposit(st["grid"], st["box"], case["modes"], -1.0, st["p"], st["bsrc"], st["work"])
        return st["bsrc"]
    if kind == "advance":
        qa.beam_advance(st["grid"], st["box"], case["modes"], -1.0, case["pusher"], st["p"], st["fld"], 2.0, 2.0, True)
        return st["p"]
    a, b, c, d = st["sys"]
    qa.thomas_batched(a, b, c, d, st["x"], st["work"], element_major=case["element_major"])
    return st["x"]


# ----------------------------------------------------------------------------------------------------------------- work
def _step_work(modes, M, K, npl, nb):
    fp, fn = (679, 508) if modes else (361, 84)   # operations per particle and per node of a slice
    ncf, ncb, ncd = (18, 15, 9) if modes else (6, 5, 3)
    return 8 * K * M * (ncf + 2 * ncb + ncd) + 160 * nb, K * (npl * fp + M * fn)


def work(case):
    kind = case["kind"]
    if kind in ("step", "pipelined"):
        npl = case["cells"] * case["ppc"] * case["ntheta"] * (2 if case["ions"] else 1)
        b, f = _step_work(case["modes"], case["cells"] + 1, case["slices"], npl, case["nd"] + case["nw"])
        n = case.get("steps", 1)
        return {"bytes": n * b, "flops": n * f}
    if kind == "batch":
        w = [_step_work(0, cells + 1, slices, 4 * cells, n + max(n // 3, 100)) for cells, slices, n in _scan_runs(case)]
        return {"bytes": sum(b for b, _ in w), "flops": sum(f for _, f in w)}
    if kind == "gradient":   # the step, its recomputation and a reverse sweep of about twice the forward's operations
        b, f = _step_work(0, 513, case["slices"], 2048, case["nd"] + case["nw"])
        return {"bytes": 3 * b, "flops": 4 * f}
    if kind == "laser":
        n = sum(M * K for M, K in _laser_sizes(case))
        return {"bytes": n * 8 * (2 + 2 + 3 + (1 if case["plasma"] else 0)), "flops": 90 * n}
    if kind == "deposit":
        nc = 15 if case["modes"] else 5
        return {"bytes": 56 * case["np"] + 8 * nc * case["slices"] * (case["cells"] + 1),
                "flops": case["np"] * (60 + (4 if not case["ngp"] else 2) * (50 if case["modes"] else 15))}
    if kind == "advance":
        nc = 18 if case["modes"] else 6
        return {"bytes": 104 * case["np"] + 8 * nc * case["slices"] * (case["cells"] + 1), "flops": case["np"] * (9 * nc + 150)}
    n = case["nodes"] * case["batch"]
    return {"bytes": 40 * n, "flops": 9 * n}


# ---------------------------------------------------------------------------------------------------------------- exact
def exact(case, seed):
    kind = case["kind"]
    if kind == "thomas":
        return _exact_thomas(case, seed)
    if kind == "deposit":
        return _exact_deposit(case, seed)
    if kind == "advance":
        return _exact_advance(case, seed)
    if kind == "laser" and sum(M * K for M, K in _laser_sizes(case)) < 1.5e6:
        out = []
        for box in _laser_boxes(case, seed)[:30]:
            out += _exact_laser(case, *box)
        return out
    return None   # a whole step: its trajectories have no closed form


def _exact_thomas(case, seed):
    a, b, c, d = [v.cpu().numpy() for v in prepare(case, seed)["sys"]]
    if not case["element_major"]:
        a, b, c, d = a.T, b.T, c.T, d.T
    M = a.shape[0]
    cp, x = np.zeros_like(a), np.zeros_like(a)
    cp[0], x[0] = c[0] / b[0], d[0] / b[0]
    for i in range(1, M):
        m = b[i] - a[i] * cp[i - 1]
        cp[i] = c[i] / m
        x[i] = (d[i] - a[i] * x[i - 1]) / m
    for i in range(M - 2, -1, -1):
        x[i] -= cp[i] * x[i + 1]
    return np.ascontiguousarray(x if case["element_major"] else x.T)


def _cells(case, p):
    """Radial cell and weight, slice and weight, radius and direction of every particle."""
    r, ih, iv = _kernel_grid(case["cells"])
    K, dxi, N = case["slices"], 0.01, case["cells"]
    rad = np.hypot(p["x"], p["y"])
    j = np.clip(np.searchsorted(r, rad, side="right") - 1, 0, N - 1)
    t = np.clip((rad - r[j]) * ih[j], 0, 1)
    s = p["xi"] / dxi
    return r, iv, rad, j, t, s, K, dxi


def _exact_deposit(case, seed):
    p = {k: v.cpu().numpy() for k, v in _beam_particles(case["np"], case["slices"], 0.01, seed).items()}
    r, iv, rad, j, t, s, K, dxi = _cells(case, p)
    M = case["cells"] + 1
    k = np.floor(s + 0.5 if case["ngp"] else s).astype(np.int64)
    tk = np.zeros_like(s) if case["ngp"] else s - k
    inside = rad <= r[-1]
    c, sn = p["x"] / rad, p["y"] / rad
    gam = np.sqrt(1 + p["px"] ** 2 + p["py"] ** 2 + p["pz"] ** 2)
    om = (1 + p["px"] ** 2 + p["py"] ** 2) / (gam * (gam + p["pz"]))
    vx, vy, vz = p["px"] / gam, p["py"] / gam, p["pz"] / gam
    vals = [om, vz, c * vx + sn * vy, c * vy - sn * vx, np.ones_like(c)]
    if case["modes"]:
        c2, s2 = c * c - sn * sn, 2 * c * sn
        vals += [om * c, -om * sn, vz * c, -vz * sn, vx, vy, vx * c2 + vy * s2, vy * c2 - vx * s2, c, -sn]
    out = np.zeros((K * M, len(vals)))
    for a in (0, 1):
        for b in (0, 1):
            w = -p["w"] * (tk if a else 1 - tk) * (t if b else 1 - t) / dxi
            kk = k + a
            ok = inside & (kk >= 0) & (kk < K) & ((a == 0) | (not case["ngp"]))
            at = (kk * M + j + b)[ok]
            w = (w * iv[j + b])[ok]
            for n, v in enumerate(vals):
                out[:, n] += np.bincount(at, weights=w * v[ok], minlength=K * M)
    return out.reshape(K, M, -1)


def _exact_advance(case, seed):
    st = prepare(case, seed)
    f = st["fld"].cpu().numpy()
    p = {k: v.cpu().numpy() for k, v in st["p"].items()}
    r, iv, rad, j, t, s, K, dxi = _cells(case, p)
    k = np.clip(np.floor(s).astype(np.int64), 0, K - 2)
    tk = np.where(s > K - 1, 1.0, s - k)

    def at(n):
        return (1 - tk) * ((1 - t) * f[k, j, n] + t * f[k, j + 1, n]) + tk * ((1 - t) * f[k + 1, j, n] + t * f[k + 1, j + 1, n])

    c, sn = p["x"] / rad, p["y"] / rad
    c2, s2 = c * c - sn * sn, 2 * c * sn

    def vector(r0, i0, r1, i1, r2, i2):
        x, y = at(r1) * c - at(i1) * sn, at(r1) * sn + at(i1) * c
        if case["modes"]:
            x, y = x + at(r0) + at(r2) * c2 - at(i2) * s2, y + at(i0) + at(r2) * s2 + at(i2) * c2
        return x, y

    def scalar(m0, r1, i1):
        return at(m0) + (2 * (at(r1) * c - at(i1) * sn) if case["modes"] else 0)

    E = np.stack(vector(6, 7, 0, 1, 8, 9) + (scalar(4, 14, 15),))
    B = np.stack(vector(10, 11, 2, 3, 12, 13) + (scalar(5, 16, 17),))
    u = np.stack([p["px"], p["py"], p["pz"]])
    dt, eps = 2.0, -1.0

    def cross(a, b):
        return np.cross(a, b, axis=0)

    def dot(a, b):
        return (a * b).sum(0)

    def implicit(a, b):   # u = a + u x b / gamma(u)
        b2, ab = dot(b, b), dot(a, b)
        q = 0.5 * (1 + dot(a, a) - b2)
        g2 = q + np.sqrt(q * q + b2 + ab * ab)
        g = np.sqrt(g2)
        return (g2 * a + g * cross(a, b) + ab * b) / (g2 + b2)

    e, b = eps * E, eps * B
    if case["pusher"] == 0:
        u = implicit(u + 2 * e + cross(u, b) / np.sqrt(1 + dot(u, u)), b)
    elif case["pusher"] == 1:
        um = u + e
        tt = b / np.sqrt(1 + dot(um, um))
        u = um + cross(um + cross(um, tt), 2 / (1 + dot(tt, tt)) * tt) + e
    elif case["pusher"] == 2:
        um = u + e
        sg, us = 1 + dot(um, um) - dot(b, b), dot(um, b)
        tt = b / np.sqrt(0.5 * (sg + np.sqrt(sg * sg + 4 * (dot(b, b) + us * us))))
        up = (um + dot(um, tt) * tt + cross(um, tt)) / (1 + dot(tt, tt))
        u = up + e + cross(up, tt)
    else:
        u = 2 * implicit(u + e, b) - u
    p2 = u[0] ** 2 + u[1] ** 2
    gam = np.sqrt(1 + p2 + u[2] ** 2)
    x, y = p["x"] + u[0] / gam * dt, p["y"] + u[1] / gam * dt
    xi = p["xi"] + (1 + p2) / (gam * (gam + u[2])) * dt
    w = np.where((x * x + y * y >= r[-1] ** 2) | (xi < 0) | (xi > (K - 1) * dxi), 0.0, p["w"])
    return {"x": x, "y": y, "px": u[0], "py": u[1], "pz": u[2], "xi": xi, "w": w}


def _exact_laser(case, K, nodes, scheme, p, chi):
    """One step of the envelope: [envelope, ponderomotive arrays]."""
    M, dxi, dt, k0 = len(nodes), 0.05, 2.0, p["k0"]
    N = M - 1
    h = np.diff(nodes)
    mid = 0.5 * (nodes[1:] + nodes[:-1])
    V = np.zeros(M)
    V[1:] += nodes[:-1] * h / 2 + h * h / 3
    V[:-1] += nodes[:-1] * h / 2 + h * h / 6
    la, lc = np.zeros(N), mid / h / V[:-1]
    la[1:] = (mid / h)[:-1] / V[1:-1]
    lb = -(la + lc)
    s = -p["focus"] / (0.5 * k0 * p["w0"] ** 2)
    xi = dxi * np.arange(K)
    q = 1 / (1 + 1j * s)
    a = p["a0"] * q * np.exp(-nodes ** 2 * q / p["w0"] ** 2)[None, :] * np.exp(-((xi - p["xi0"]) / p["L0"]) ** 2)[:, None]
    a[:, N] = 0
    m = (1.0 if case["circular"] else 0.5) * np.abs(a) ** 2
    prev = np.vstack([np.zeros((2, M)), m])
    pond = np.zeros((K, M, 3))
    pond[:, :, 0] = m
    hm, hp = h[:-1], h[1:]
    den = hm * hp * (hm + hp)
    pond[:, 1:N, 1] = (-hp * hp * m[:, :-2] + (hp * hp - hm * hm) * m[:, 1:-1] + hm * hm * m[:, 2:]) / den
    h1, h2 = h[N - 1], h[N - 2]
    pond[:, N, 1] = (2 * h1 + h2) / (h1 * (h1 + h2)) * m[:, N] - (h1 + h2) / (h1 * h2) * m[:, N - 1] + h1 / (h2 * (h1 + h2)) * m[:, N - 2]
    pond[:, :, 2] = (3 * m - 4 * prev[1:-1] + prev[:-2]) / (2 * dxi)
    cd, c1, c2 = {"trapezoid": (4, 4, 0), "bdf2": (3, 4, -1), "euler": (2, 2, 0)}[scheme]
    s0, s2 = 2 / (dt * dxi), 4 / dt
    alpha = cd * s0 - 1j * s2 * k0
    out = np.zeros((K, M), dtype=complex)
    x0, x1 = np.zeros(N, dtype=complex), np.zeros(N, dtype=complex)

    def H(hd, v):   # the operator on v, zero at the wall
        r = hd * v[:N]
        r[1:] += la[1:] * v[:N - 1]
        return r + lc * v[1:]

    for k in range(K):
        hd = lb - (chi[k, :N] if chi is not None else 0)
        rhs = (c1 * s0 * x0 + (s2 if scheme == "trapezoid" else c2 * s0) * x1 + 2 * H(hd, a[k])).tolist()
        d, A, Cc = (alpha - hd).tolist(), la.tolist(), lc.tolist()
        cp, dp, c_, d_ = [0] * N, [0] * N, 0.0, 0.0
        for j in range(N):
            w = d[j] + A[j] * c_
            c_ = -Cc[j] / w
            d_ = (rhs[j] + A[j] * d_) / w
            cp[j], dp[j] = c_, d_
        X, x = [0] * N, 0.0
        for j in range(N - 1, -1, -1):
            x = dp[j] - cp[j] * x
            X[j] = x
        X = np.array(X)
        full = np.append(X, 0)
        if scheme == "trapezoid":
            x0, x1 = X, 1j * k0 * X + 0.25 * dt * H(hd, full + 2 * a[k])
        else:
            x0, x1 = X, x0
        out[k] = a[k] + full
    return [np.stack([out.real, out.imag], axis=-1), pond]
