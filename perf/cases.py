"""The work a user of this framework has it do, as cases that can be timed.

A host model's time step is UpdateStateParameters followed by Solve over its grid
cells, with the concentrations resident on the GPU; besides it there are the
multi-cell State with one step size (the default form), several mechanisms in one
launch, gradients of a Solve, and the single phases of an attempt that a MICM policy
set calls one at a time.  Mechanisms and distributions are those of the benchmark
(micm_amd/synthetic.py, tests/golden/ts1_mechanism.json).

`listed()` names the cases, `draw(rng)` gives another one of the same ranges,
`prepare(case, seed)` makes what a program has in hand before the call, `run(state)` is
one pass, `work(case)` the bytes and operations it cannot do without, and
`exact(case, seed)` the results of plain torch in 64 bits.
"""
import math
import os

import numpy as np
import torch

import micm_amd
from micm_amd import _desc, _lib, mechanism_io, synthetic

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# Per mechanism: species, reactions, custom parameters, non-zeros of the Jacobian, L and U,
# FP64 operations of one forcing, Jacobian, LU and substitution (counted from the mechanism as
# bench.py does), the time step and tableau it is run with, and the mean step attempts of one
# cell's Solve over that time step.
MECHANISMS = {
    "readme": dict(n=3, r=2, p=0, nj=7, nl=6, nu=4, f=12, j=15, lu=10, s=14, dt=500.0, tableau=3, attempts=12),
    "20_50": dict(n=20, r=50, p=5, nj=124, nl=114, nu=71, f=346, j=436, lu=588, s=330, dt=300.0, tableau=4,
                  attempts=12),
    "60_200": dict(n=60, r=200, p=20, nj=646, nl=713, nu=651, f=1402, j=1915, lu=16049, s=2608, dt=300.0, tableau=4,
                   attempts=35),
    "210_560": dict(n=210, r=560, p=56, nj=2138, nl=4548, nu=4210, f=3846, j=5043, lu=246620, s=17096, dt=900.0,
                    tableau=4, attempts=69),
    "ts1": dict(n=209, r=547, p=168, nj=1950, nl=1453, nu=1137, f=4760, j=7626, lu=15425, s=4762, dt=30.0, tableau=3,
                attempts=123),
}

FORMS = {"lockstep": _lib.SOLVE_LOCKSTEP, "persistent": _lib.SOLVE_PERSISTENT, "cooperative": _lib.SOLVE_COOPERATIVE}


def listed():
    return [
        # the README example as a first user runs it: one cell, the default form, inputs and
        # results on the host; all latency
        {"name": "readme_one_cell", "kind": "facade", "mechanism": "readme", "cells": 1, "form": "lockstep"},
        # a small regional grid of the README system (the reference's 1,000-cell example)
        {"name": "readme_1000", "kind": "solve", "mechanism": "readme", "cells": 1000, "form": "cooperative",
         "threads": 128, "stage": -1},
        # a single column or box model with full chemistry: a handful of cells, an odd number
        {"name": "210_560_7", "kind": "solve", "mechanism": "210_560", "cells": 7, "form": "cooperative",
         "threads": 256, "stage": 6},
        # the headline workload, as many cells as a pass of about a second takes, in the launch
        # shape that the autotuner picks for it
        {"name": "210_560_20k", "kind": "solve", "mechanism": "210_560", "cells": 20000, "form": "cooperative",
         "threads": 256, "stage": 6},
        # the mid-size mechanism on 10,000 cells, in the autotuner's shape
        {"name": "60_200_10k", "kind": "solve", "mechanism": "60_200", "cells": 10000, "form": "cooperative",
         "threads": 256, "stage": 4},
        # the persistent form with the library's own launch shape and hand-off, for a caller
        # that does not tune, on a ragged number of cells
        {"name": "60_200_persistent", "kind": "solve", "mechanism": "60_200", "cells": 20011, "form": "persistent",
         "threads": 0, "stage": -1},
        # TS1, the reference's own benchmark mechanism, 10,000 cells, per-cell steps
        {"name": "ts1_10k", "kind": "solve", "mechanism": "ts1", "cells": 10000, "form": "cooperative", "threads": 256,
         "stage": 4},
        # one step size for all cells, what a multi-cell State of the reference does: the small
        # mechanism, where the cells' common step still reaches the end of the time step
        {"name": "20_50_lockstep", "kind": "solve", "mechanism": "20_50", "cells": 5003, "form": "lockstep",
         "threads": 0, "stage": -1},
        # three mechanisms of different sizes in one graph-captured launch (a tenth of the
        # benchmark's packed workload), launch shapes left to the library
        {"name": "packed", "kind": "packed", "small": 20000, "middle": 5000, "large": 2000},
        # gradients: recorded Solves of the mid-size mechanism, then the reverse sweep
        {"name": "adjoint_60_200", "kind": "adjoint", "mechanism": "60_200", "cells": 1024, "solves": 2},
        # the memory-bound phases one kernel at a time, as a policy set calls them at a step start
        {"name": "phases_210_560", "kind": "phases", "mechanism": "210_560", "cells": 30000},
        # the linear algebra of one attempt one kernel at a time: alpha, LU, substitution, error
        {"name": "linear_210_560", "kind": "linear", "mechanism": "210_560", "cells": 4096},
    ]


def draw(rng):
    def log_int(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    kind = rng.choice(["facade", "solve", "solve", "solve", "solve", "packed", "adjoint", "phases", "linear"])
    if kind == "facade":
        return {"kind": kind, "mechanism": "readme", "cells": log_int(1, 1000), "form": "lockstep"}
    if kind == "packed":
        return {"kind": kind, "small": log_int(100, 20000), "middle": log_int(50, 5000), "large": log_int(10, 2000)}
    if kind == "adjoint":
        return {"kind": kind, "mechanism": "60_200", "cells": log_int(16, 1024), "solves": rng.randint(1, 2)}
    if kind == "phases":
        return {"kind": kind, "mechanism": rng.choice(["60_200", "ts1", "210_560"]), "cells": log_int(300, 30000)}
    if kind == "linear":
        return {"kind": kind, "mechanism": rng.choice(["60_200", "ts1", "210_560"]), "cells": log_int(64, 4096)}
    mechanism = rng.choice(["readme", "20_50", "60_200", "60_200", "ts1", "210_560", "210_560"])
    form = rng.choice(["cooperative", "cooperative"] + (["lockstep"] if mechanism in ("readme", "20_50") else []) +
                      (["persistent"] if mechanism in ("readme", "20_50", "60_200") else []))
    most = {"readme": 100000, "20_50": 20000, "60_200": 20000, "ts1": 10000, "210_560": 20000}[mechanism]
    if form == "lockstep":
        most = 5003
    elif form == "persistent":
        most //= 2
    shapes = [(0, -1), (128, -1), (256, -1), (256, 4)]
    threads, stage = rng.choice(shapes) if form == "cooperative" else (0, -1)
    if mechanism == "210_560" and threads != 256:
        most = 2500  # these shapes run it two to three times slower
    return {"kind": "solve", "mechanism": mechanism, "cells": log_int(1, most), "form": form, "threads": threads,
            "stage": stage}


# ------------------------------------------------------------------ inputs

def _mechanism(name):
    if name == "readme":
        return synthetic.readme_mechanism()
    if name == "20_50":
        return synthetic.mechanism_20_50()
    if name == "60_200":
        return synthetic.mechanism_60_200()
    if name == "210_560":
        return synthetic.mechanism_210_560()
    return mechanism_io.load(os.path.join(ROOT, "tests", "golden", "ts1_mechanism.json"))


def _cells(name, desc, n, seed):
    """Per-cell conditions, concentrations (declared order) and custom parameters."""
    seed = 1000003 * int(seed) + 17
    if name == "readme":
        return synthetic.readme_inputs(n, seed=seed)
    if name == "210_560":
        return synthetic.inputs_210_560(desc, n, seed=seed)
    if name in ("20_50", "60_200"):
        return synthetic.inputs_60_200(desc, n, seed=seed)
    # TS1: the benchmark's initial state, each cell with a little more or less of every species
    cond, y, custom = mechanism_io.initial_arrays(desc, n)
    rs = np.random.RandomState(seed % (1 << 32))
    return synthetic.CellInputs(cond, y * rs.uniform(0.9, 1.1, y.shape), custom)


def _dev(host):
    return torch.from_numpy(_lib.to_grouped(host)).cuda()


def _empty(n, values):
    return torch.zeros((n + 63) // 64 * 64 * values, dtype=torch.float64, device="cuda")


def _device_state(name, n, seed):
    desc = _mechanism(name)
    mech = _lib.Mechanism(desc)
    cells = _cells(name, desc, n, seed)
    y = cells.variables[:, mech.species_order()]
    state = _lib.DeviceState(mech, n)
    state.set_variables(y)
    state.set_conditions(cells.conditions)
    state.set_custom_parameters(cells.custom)
    return mech, cells, state, y


def _readme_facade(case, seed):
    """The README example through the builder (README.md:95-161)."""
    foo, bar, baz = (micm_amd.Species(s) for s in ("Foo", "Bar", "Baz"))
    gas = micm_amd.Phase("gas", [foo, bar, baz])
    r1 = (micm_amd.ChemicalReactionBuilder().SetReactants([foo])
          .SetProducts([micm_amd.StoichSpecies(bar, 0.8), micm_amd.StoichSpecies(baz, 0.2)])
          .SetRateConstant(micm_amd.ArrheniusRateConstantParameters(A=1.0e-3)).SetPhase(gas).Build())
    r2 = (micm_amd.ChemicalReactionBuilder().SetReactants([foo, bar])
          .SetProducts([micm_amd.StoichSpecies(baz, 1.0)])
          .SetRateConstant(micm_amd.ArrheniusRateConstantParameters(A=1.0e-5, C=110.0)).SetPhase(gas).Build())
    solver = (micm_amd.HipSolverBuilder(micm_amd.RosenbrockSolverParameters.ThreeStageRosenbrockParameters())
              .SetSystem(micm_amd.System(gas)).SetReactions([r1, r2]).Build())
    state = solver.GetState(case["cells"], form=case["form"])
    cells = _cells("readme", None, case["cells"], seed)
    state.conditions_array[:] = cells.conditions
    order = [["Foo", "Bar", "Baz"].index(v) for v in state.variable_names]
    return solver, state, cells, order


def prepare(case, seed):
    kind = case["kind"]
    if kind == "facade":
        solver, state, cells, order = _readme_facade(case, seed)
        return {"kind": kind, "solver": solver, "state": state, "y0": cells.variables[:, order].copy()}
    if kind == "packed":
        parts = []
        for k, (name, key) in enumerate((("20_50", "small"), ("60_200", "middle"), ("210_560", "large"))):
            mech, _, state, y = _device_state(name, case[key], int(seed) * 3 + k)
            state.update_state_parameters()
            parts.append((state, _dev(y), _empty(case[key], mech.n_species)))
        return {"kind": kind, "parts": parts, "params": _lib.rosenbrock_parameters(4),
                "packed": _lib.PackedSolve([s for s, _, _ in parts], _lib.SOLVE_COOPERATIVE)}
    name, n = case["mechanism"], case["cells"]
    mech, cells, state, y = _device_state(name, n, seed)
    spec = MECHANISMS[name]
    out = {"kind": kind, "mech": mech, "state": state, "n": n, "y0": _dev(y), "dt": spec["dt"],
           "params": _lib.rosenbrock_parameters(spec["tableau"])}
    if kind == "solve":
        state.set_cooperative_shape(case["threads"], case["stage"])
        out.update(form=FORMS[case["form"]], y=_empty(n, mech.n_species))
    elif kind == "adjoint":
        # gradients are taken at a tolerance that resolves every species
        state.set_tolerances(1e-6, np.full(mech.n_species, 1e-12))
        state.update_state_parameters()
        rs = np.random.RandomState(seed % (1 << 32))
        out.update(tape=_lib.Tape(mech, n, 2200), solves=case["solves"], y=_empty(n, mech.n_species),
                   seed=_dev(rs.uniform(-1.0, 1.0, (n, mech.n_species))), gy=_empty(n, mech.n_species),
                   gk=_empty(n, mech.n_reactions))
    elif kind == "phases":
        out.update(cond=_dev(cells.conditions), custom=_dev(cells.custom), k=_empty(n, mech.n_reactions),
                   f=_empty(n, mech.n_species), jac=_empty(n, mech.nnz_jacobian))
    elif kind == "linear":
        # -J and f(y) of these cells, as the phases before leave them
        state.update_state_parameters()
        out.update(jac0=_empty(n, mech.nnz_jacobian), f=_empty(n, mech.n_species), jac=_empty(n, mech.nnz_jacobian),
                   lower=_empty(n, mech.nnz_lower), upper=_empty(n, mech.nnz_upper), x=_empty(n, mech.n_species),
                   err=torch.zeros(n, dtype=torch.float64, device="cuda"), alpha=_alpha(case))
        k = state.pointers().rate_constants
        mech.fill_and_subtract_jacobian_terms(n, k, out["y0"].data_ptr(), out["jac0"].data_ptr())
        mech.fill_and_add_forcing_terms(n, k, out["y0"].data_ptr(), out["f"].data_ptr())
    return out


def _alpha(case):
    """1 / (H gamma) of a step of a tenth of the time step."""
    spec = MECHANISMS[case["mechanism"]]
    return 1.0 / (0.1 * spec["dt"] * _lib.rosenbrock_parameters(spec["tableau"]).gamma[0])


# ------------------------------------------------------------------ one pass

def _solved(state, out):
    """Final concentrations on the device (grouped) and the per-cell outcomes."""
    state.get_variables_device(out.data_ptr())
    status, stats, final_time = state.results()
    return {"y": out, "status": status, "stats": stats, "final_time": final_time}


def run(s):
    kind = s["kind"]
    if kind == "facade":
        solver, state = s["solver"], s["state"]
        state.variables[:] = s["y0"]
        solver.UpdateStateParameters(state)
        result = solver.Solve(500.0, state)
        return {"y": state.variables, "status": state.cell_state, "stats": state.cell_stats,
                "final_time": state.cell_final_time, "state": int(result.state)}
    if kind == "packed":
        for state, y0, _ in s["parts"]:
            state.set_variables_device(y0.data_ptr())
        s["packed"].solve(900.0, s["params"])
        return [_solved(state, y) for state, _, y in s["parts"]]
    mech, state, n = s["mech"], s["state"], s["n"]
    if kind == "solve":
        state.set_variables_device(s["y0"].data_ptr())
        state.update_state_parameters()
        state.solve(s["dt"], s["params"], s["form"])
        return _solved(state, s["y"])
    if kind == "adjoint":
        s["tape"].reset()
        state.set_variables_device(s["y0"].data_ptr())
        for _ in range(s["solves"]):
            state.solve_recorded(s["dt"], s["params"], s["tape"])
        state.adjoint(s["params"], s["tape"], s["seed"].data_ptr(), s["gy"].data_ptr(), s["gk"].data_ptr())
        return {**_solved(state, s["y"]), "grad_y": s["gy"], "grad_log_k": s["gk"]}
    if kind == "phases":
        mech.calculate_rate_constants(n, s["cond"].data_ptr(), s["custom"].data_ptr(), s["k"].data_ptr())
        mech.fill_and_add_forcing_terms(n, s["k"].data_ptr(), s["y0"].data_ptr(), s["f"].data_ptr())
        mech.fill_and_subtract_jacobian_terms(n, s["k"].data_ptr(), s["y0"].data_ptr(), s["jac"].data_ptr())
        return {"k": s["k"], "f": s["f"], "jac": s["jac"]}
    s["jac"].copy_(s["jac0"])
    s["x"].copy_(s["f"])
    mech.alpha_minus_jacobian(n, s["jac"].data_ptr(), s["alpha"])
    mech.lu_decompose(n, s["jac"].data_ptr(), s["lower"].data_ptr(), s["upper"].data_ptr())
    mech.lu_solve(n, s["lower"].data_ptr(), s["upper"].data_ptr(), s["x"].data_ptr())
    mech.normalized_error(n, s["y0"].data_ptr(), s["y0"].data_ptr(), s["x"].data_ptr(),
                          state.pointers().absolute_tolerances, 1e-6, s["err"].data_ptr())
    return {"lower": s["lower"], "upper": s["upper"], "x": s["x"], "error": s["err"]}


# ------------------------------------------------------------------ work

def _solve_work(spec, cells):
    """One Solve: concentrations in and out, rate constants or what they are made of, outcomes;
    the operations of the attempts the cells take (4-stage: three forcings, four substitutions;
    3-stage: two and three)."""
    calls = 3 if spec["tableau"] == 4 else 2
    per = calls * spec["f"] + spec["j"] + spec["lu"] + spec["tableau"] * spec["s"] + 7 * spec["n"]
    return 8 * cells * (2 * spec["n"] + spec["r"] + spec["p"] + 3 + 9), cells * spec["attempts"] * per


def work(case):
    kind = case["kind"]
    if kind == "packed":
        parts = [_solve_work(MECHANISMS[m], case[k])
                 for m, k in (("20_50", "small"), ("60_200", "middle"), ("210_560", "large"))]
        return {"bytes": sum(b for b, _ in parts), "flops": sum(f for _, f in parts)}
    spec, cells = MECHANISMS[case["mechanism"]], case["cells"]
    if kind in ("facade", "solve"):
        b, f = _solve_work(spec, cells)
        return {"bytes": b, "flops": f}
    if kind == "adjoint":
        # a checkpoint per accepted step written and read; the reverse sweep factors and solves
        # each step again and solves with the transposes
        b, f = _solve_work(spec, cells * case["solves"])
        steps = 0.85 * spec["attempts"] * cells * case["solves"]
        return {"bytes": b + 16 * steps * (spec["n"] + 1) + 8 * cells * (2 * spec["n"] + spec["r"]),
                "flops": f + steps * (spec["lu"] + 2 * spec["tableau"] * spec["s"] + 8 * spec["j"])}
    n, r, p = spec["n"], spec["r"], spec["p"]
    if kind == "phases":
        return {"bytes": 8 * cells * (3 + p + r + 2 * n + spec["nj"]),
                "flops": cells * (30 * r + spec["f"] + spec["j"])}
    return {"bytes": 8 * cells * (spec["nj"] + spec["nl"] + spec["nu"] + 3 * n + 1),
            "flops": cells * (spec["lu"] + spec["s"] + 7 * n)}


# ------------------------------------------------------------------ plain torch, 64 bits

def _rates(desc, cells, device):
    """Rate constants [cells, reactions] in sorted order (Arrhenius, Troe, ternary, user-defined
    and surface) with their third bodies' concentrations."""
    T, P, rho = (torch.from_numpy(cells.conditions[:, i].copy()).to(device) for i in range(3))
    custom = torch.from_numpy(cells.custom).to(device)
    cols, c = [], 0
    for r in desc.sorted_reaction_order():
        t, p = int(desc.rate_types[r]), [float(v) for v in desc.rate_params[r]]
        if t == _desc.ARRHENIUS:
            k = p[0] * torch.exp(p[2] / T) * (T / p[3]) ** p[1] * (1.0 + p[4] * P)
        elif t in (_desc.TROE, _desc.TERNARY):
            k0 = p[0] * torch.exp(p[2] / T) * (T / 300.0) ** p[1]
            ratio = k0 * rho / (p[3] * torch.exp(p[5] / T) * (T / 300.0) ** p[4])
            k = k0 * (rho if t == _desc.TROE else 1.0) / (1.0 + ratio) * \
                p[6] ** (p[7] / (p[7] + torch.log10(ratio) ** 2))
        elif t == _desc.USER_DEFINED:
            k = custom[:, c] * p[0]
            c += 1
        else:  # surface
            radius, number = custom[:, c], custom[:, c + 1]
            speed = torch.sqrt(8.0 * synthetic.GAS_CONSTANT / (math.pi * p[1]) * T)
            k = 4.0 * number * math.pi * radius ** 2 / (radius / p[0] + 4.0 / (speed * p[2]))
            c += 2
        for i in desc.reactants[desc.reactant_offsets[r]:desc.reactant_offsets[r + 1]]:
            if i < 0:
                m = [float(v) for v in desc.parameterized[-int(i) - 1]]
                k = k * (m[0] + m[1] * T + m[2] * P + m[3] * rho)
        cols.append(k)
    return torch.stack(cols, dim=1)


def _terms(desc, order):
    """Per sorted reaction: reactant columns and (column, yield) of its products."""
    at = {int(d): i for i, d in enumerate(order)}
    out = []
    for r in desc.sorted_reaction_order():
        ins = [at[int(s)] for s in desc.reactants[desc.reactant_offsets[r]:desc.reactant_offsets[r + 1]]
               if s >= 0]
        lo, hi = desc.product_offsets[r], desc.product_offsets[r + 1]
        outs = [(at[int(s)], float(v)) for s, v in zip(desc.products[lo:hi], desc.yields[lo:hi]) if s >= 0]
        out.append((ins, outs))
    return out


def _forcing(terms, k, y):
    f = torch.zeros_like(y)
    for r, (ins, outs) in enumerate(terms):
        rate = k[r].clone()
        for i in ins:
            rate *= y[i]
        for i in ins:
            f[i] -= rate
        for i, v in outs:
            f[i] += v * rate
    return f


def _minus_jacobian(terms, k, y):
    """-J, [species, species, cells]."""
    n = y.shape[0]
    a = torch.zeros((n, n, y.shape[1]), dtype=y.dtype, device=y.device)
    for r, (ins, outs) in enumerate(terms):
        for q, j in enumerate(ins):
            d = k[r].clone()
            for i in ins[:q] + ins[q + 1:]:
                d *= y[i]
            for i in ins:
                a[i, j] += d
            for i, v in outs:
                a[i, j] -= v * d
    return a


def _factor(a):
    """Doolittle factors of a [n, n, cells], without pivoting, in place."""
    for c in range(a.shape[0] - 1):
        a[c + 1:, c] /= a[c, c]
        rows = torch.nonzero((a[c + 1:, c] != 0).any(dim=1)).flatten() + c + 1
        cols = torch.nonzero((a[c, c + 1:] != 0).any(dim=1)).flatten() + c + 1
        if len(rows) and len(cols):
            a[rows[:, None], cols[None, :]] -= a[rows, c][:, None] * a[c, cols][None, :]
    return a


def _substitute(a, b):
    """The factors' solution for b [n, cells]."""
    x = b.clone()
    n = x.shape[0]
    for i in range(1, n):
        x[i] -= (a[i, :i] * x[:i]).sum(dim=0)
    for i in range(n - 1, -1, -1):
        if i + 1 < n:
            x[i] -= (a[i, i + 1:] * x[i + 1:]).sum(dim=0)
        x[i] /= a[i, i]
    return x


def _norm(y, ynew, e, rtol=1e-6, atol=1e-3):
    q = e / (atol + rtol * torch.maximum(y.abs(), ynew.abs()))
    return q.square().mean(dim=0).sqrt().clamp_min(1e-10)


def _grouped(t):
    """[values, cells] in the grouped device layout, the padding cells zero."""
    v, n = t.shape
    g = (n + 63) // 64
    buf = torch.zeros((v, g * 64), dtype=t.dtype, device=t.device)
    buf[:, :n] = t
    return buf.reshape(v, g, 64).permute(1, 0, 2).reshape(-1)


def _solve_readme(y, k, dt, lockstep):
    """The 3-stage Rosenbrock integration of rosenbrock.inl:12-304 for a mechanism of a few
    species, every cell with its own step size or all with one; [species, cells] in and out,
    with the step size's own time."""
    p = _lib.rosenbrock_parameters(3)
    desc = _mechanism("readme")
    terms = _terms(desc, _lib.Mechanism(desc).species_order())
    n, cells = y.shape
    A, C, M, E, G = list(p.a), list(p.c), list(p.m), list(p.e), p.gamma[0]
    new_f, h_max = list(p.new_function_evaluation), dt if p.h_max == 0.0 else min(dt, p.h_max)
    h_min = 1e-15 * dt if p.h_min == 0.0 else p.h_min
    start = 1e-6 * dt if p.h_start == 0.0 else min(h_max, p.h_start)
    eye = torch.eye(n, dtype=y.dtype, device=y.device)[:, :, None]
    t = torch.zeros(cells, dtype=y.dtype, device=y.device)
    rejected = torch.zeros(cells, dtype=torch.bool, device=y.device)
    more = rejected.clone()
    H = torch.full_like(t, min(max(h_min, start), h_max))
    for _ in range(1000):
        live = (t - dt + p.round_off) <= 0
        if not live.any():
            break
        h = torch.minimum(H, dt - t)
        h = torch.where(live, h, torch.ones_like(h))
        lu = _factor(eye / (h * G) + _minus_jacobian(terms, k, y))
        f = _forcing(terms, k, y)
        K = []
        for s in range(3):
            at = s * (s - 1) // 2
            if s and new_f[s]:
                f = _forcing(terms, k, y + sum(A[at + j] * K[j] for j in range(s)))
            K.append(_substitute(lu, f + sum((C[at + j] / h * K[j] for j in range(s)), torch.zeros_like(f))))
        ynew = y + sum(M[s] * K[s] for s in range(3))
        e = sum(E[s] * K[s] for s in range(3))
        err = _norm(y, ynew, e)
        if lockstep:
            err = err.square().mean().sqrt().clamp_min(1e-10).expand_as(err)
        fac = (p.safety_factor / err ** (1.0 / p.estimator_of_local_order)).clamp(p.factor_min, p.factor_max)
        ok = live & ((err < 1) | (h < h_min))
        H2 = torch.where(ok, (h * fac).clamp(h_min, h_max), h * fac)
        H2 = torch.where(ok & rejected, torch.minimum(H2, h), H2)
        H2 = torch.where(~ok & more, h * p.rejection_factor_decrease, H2)
        t = torch.where(ok, t + h, t)
        y = torch.where(ok, ynew, y)
        more = torch.where(live, ~ok & rejected, more)
        rejected = torch.where(live, ~ok, rejected)
        H = torch.where(live, H2, H)
    return y.clamp_min(0.0), t


def exact(case, seed):
    """None for the whole Solves of the larger mechanisms and their gradients: with the slowest
    cells' thousand attempts of hundreds of dependent batched steps each they take minutes."""
    kind = case["kind"]
    device = "cuda" if torch.cuda.is_available() else "cpu"
    if kind == "packed" or kind == "adjoint" or (kind == "solve" and case["mechanism"] != "readme"):
        return None
    name = case["mechanism"]
    desc = _mechanism(name)
    cells = _cells(name, desc, case["cells"], seed)
    k = _rates(desc, cells, device).T.contiguous()
    if kind in ("facade", "solve"):
        order = _readme_facade(case, seed)[3] if kind == "facade" else _lib.Mechanism(desc).species_order()
        y = torch.from_numpy(cells.variables[:, order].T.copy()).to(device)
        y, t = _solve_readme(y, k, 500.0, case["form"] == "lockstep")
        if kind == "facade":
            return {"y": y.T.cpu().numpy(), "status": None, "stats": None, "final_time": t.cpu().numpy(), "state": None}
        return {"y": _grouped(y), "status": None, "stats": None, "final_time": t.cpu().numpy()}
    mech = _lib.Mechanism(desc)
    order, pattern = mech.species_order(), mech.patterns()
    y = torch.from_numpy(cells.variables[:, order].T.copy()).to(device)
    terms = _terms(desc, order)
    at = {q: tuple(torch.from_numpy(v).to(device) for v in pattern[q]) for q in pattern}
    if kind == "phases":
        parts = []
        for c in range(0, y.shape[1], 4096):  # a dense -J of 4,096 cells at a time
            a = _minus_jacobian(terms, k[:, c:c + 4096], y[:, c:c + 4096])
            parts.append(a[at["jacobian"][0], at["jacobian"][1]])
        return {"k": _grouped(k), "f": _grouped(_forcing(terms, k, y)), "jac": _grouped(torch.cat(parts, dim=1))}
    a = _minus_jacobian(terms, k, y)
    a.diagonal(dim1=0, dim2=1).add_(_alpha(case))
    a = _factor(a)
    x = _substitute(a, _forcing(terms, k, y))
    lower = a[at["lower"][0], at["lower"][1]].clone()
    lower[at["lower"][0] == at["lower"][1]] = 1.0
    return {"lower": _grouped(lower), "upper": _grouped(a[at["upper"][0], at["upper"][1]]), "x": _grouped(x),
            "error": _norm(y, y, x)}
