"""Performance cases: the work a user of this package has it do, with inputs and sizes.

Two paths are covered through their public entry points:

* Monte Carlo sampling: ``mc_sim`` of a drop-in script, ``DeviceReplicas.run`` for one
  chain, a parameter scan or the full 512-replica batch, and the one-launch-per-proposal
  calls (``step``, ``run_plain``);
* the voxel densities and the energy with its gradients: ``density_init``, ``energy`` and
  ``chromo_energy`` under autograd.

Chains, grids and interactions come from ``chromo_amd.workloads`` (25 nm beads in 30 nm
voxels), the drop-in scripts from the package's tutorial-sized systems.  Every Monte Carlo
pass continues the state's chains and returns all that a pass changes.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from chromo_amd import _lib as L
from chromo_amd import mc
from chromo_amd import workloads as W
from chromo_amd.binders import get_by_name, make_binder_collection
from chromo_amd.energy import EnergyModel, chromo_energy, energy, eps_index, n_theta
from chromo_amd.engine import DeviceReplicas
from chromo_amd.fields import NullField, UniformDensityField
from chromo_amd.mc import mc_controller as ctl
from chromo_amd.polymers import SSWLC, Chromatin
from chromo_amd.util.poly_paths import estimate_tangents_from_coordinates

ALL_MOVES = (30, 1, 60, 60, 10)     # proposals per sweep of chromo's all_moves
MU = (-0.4, 0.3, -1.0, 0.2)
EPS = (-4.0, -2.5, -3.0, -1.5)


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------

def _mc(name, reps, n_lo, n_hi, B, vox_lo, vox_hi, sweeps, *, steady=True, waves=0, rng="philox",
        marks="bernoulli", twist=False, fast_field=False, launch="run"):
    case = dict(kind="mc", reps=reps, n_lo=n_lo, n_hi=n_hi, B=B, vox_lo=vox_lo, vox_hi=vox_hi,
                sweeps=sweeps, steady=steady, waves=waves, rng=rng, marks=marks, twist=twist,
                fast_field=fast_field, launch=launch)
    return dict(name=name, **case) if name else case


def _script(name, n, field, steps, vox):
    case = dict(kind="script", n=n, field=field, steps=steps, vox=vox)
    return dict(name=name, **case) if name else case


def _field(name, kind, n, B, nx, ny, nz, *, marks="bernoulli"):
    case = dict(kind=kind, n=n, B=B, nx=nx, ny=ny, nz=nz, marks=marks)
    return dict(name=name, **case) if name else case


def listed():
    return [
        # One mc_step at a time, the reference's own granularity: a script that steps a
        # 1,000-bead chain and looks at it between proposals.  Launch latency.
        _mc("step_1k", 1, 1000, 1000, 2, 30, 30, 0, steady=False, rng="glibc", launch="step"),
        # One sweep with one launch per proposal on the 100,000-bead chain
        # (mc_sim(launch="plain")), for comparing a run proposal by proposal.
        _mc("plain_100k", 1, 100_000, 100_000, 2, 64, 64, 1, steady=False, rng="glibc",
            marks="markov", launch="plain"),
        # A drop-in script: one-mark chromatin of 1,000 beads in a spherical confinement,
        # 20 steps of all_moves between two looks at the chain.
        _script("script_confined_1k", 1000, "confined", 20, 16),
        # A drop-in script without a field: semiflexible homopolymer, the four geometric moves.
        _script("script_homopolymer_1k", 1000, "none", 100, 0),
        # A small parameter scan with sub-bin field weights (fast_field).
        _mc("scan16_fast", 16, 1000, 5000, 2, 24, 36, 10, fast_field=True),
        # An ordinary scan from a fresh start (initial move amplitudes), three binders.
        _mc("scan128_b3", 128, 1500, 9000, 3, 25, 45, 10, steady=False, marks="onehot"),
        # The full batch at steady-state amplitudes, two wavefronts per replica as the
        # launch-shape autotuner picks for it.
        _mc("batched512", 512, 2000, 20_000, 2, 32, 52, 20, waves=2),
        # A few very long chains with four binders.
        _mc("long4_b4", 4, 250_000, 250_000, 4, 96, 96, 10, marks="onehot"),
        # One twisting chain.
        _mc("twist_4k", 1, 4001, 4001, 1, 33, 33, 10, twist=True),
        # The densities of a million-bead chain (start of a run, after editing positions).
        _field("scatter_1m", "scatter", 1_000_000, 4, 128, 128, 128, marks="onehot"),
        # Energy and gradients of the 20,000-bead chain under autograd: a step of fitting.
        _field("grad_20k", "autograd", 20_000, 3, 48, 48, 48),
        # Energy and gradients of a million-bead chain, one evaluation.
        _field("grad_1m", "grad", 1_000_000, 4, 128, 128, 128, marks="onehot"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above."""
    kind = rng.choice(["step", "plain", "script", "scan", "scan", "batch", "long", "twist", "scatter",
                       "grad", "grad", "autograd"])
    marks = rng.choice(["bernoulli", "markov", "onehot"])
    if kind == "step":
        n = _log_int(rng, 200, 100_000)
        return _mc(None, 1, n, n, rng.randint(1, 4), 9, 40, 0, steady=False, rng="glibc", marks=marks, launch="step")
    if kind == "plain":
        n = _log_int(rng, 500, 100_000)
        return _mc(None, 1, n, n, rng.randint(1, 4), 12, 64, 1, steady=rng.random() < 0.5, rng="glibc",
                   marks=marks, launch="plain")
    if kind == "script":
        field = rng.choice(["confined", "none", "periodic"])
        return _script(None, _log_int(rng, 200, 5000), field, rng.randint(1, 60), rng.randint(11, 24))
    if kind in ("scan", "batch"):
        reps = _log_int(rng, 1, 160) if kind == "scan" else rng.randint(200, 512)
        lo = _log_int(rng, 300, 4000)
        return _mc(None, reps, lo, lo * rng.randint(1, 5), rng.randint(1, 4), 13, rng.randint(20, 48),
                   rng.randint(1, 20), steady=rng.random() < 0.6, waves=rng.choice([0, 0, 2]),
                   rng=rng.choice(["philox", "philox", "glibc"]), marks=marks, fast_field=rng.random() < 0.2)
    if kind == "long":
        n = _log_int(rng, 30_000, 400_000)
        return _mc(None, rng.randint(1, 6), n, n, rng.randint(1, 4), 48, 96, rng.randint(1, 10), marks=marks)
    if kind == "twist":
        n = _log_int(rng, 300, 20_000)
        return _mc(None, 1, n, n, rng.randint(1, 4), 13, rng.randint(16, 48), rng.randint(1, 10), steady=rng.random() < 0.5, marks=marks, twist=True)
    n = _log_int(rng, 700, 1_000_000)
    side = max(6, min(128, round(1.3 * n ** (1 / 3))))
    size = [max(5, side + rng.randint(-side // 6, side // 6)) for _ in range(3)]
    return _field(None, kind, n, rng.randint(1, 4), *[min(128, x) for x in size], marks=marks)


# ---------------------------------------------------------------------------
# States
# ---------------------------------------------------------------------------

def _replica_sizes(case):
    """(beads, voxels per side) of every replica, the longer chain in the larger grid.
    The sizes belong to the case; only the chains depend on the seed."""
    rs = np.random.RandomState(1000 + case["reps"] + case["n_lo"])
    ns = rs.randint(case["n_lo"], case["n_hi"] + 1, size=case["reps"])
    span = max(1, case["n_hi"] - case["n_lo"])
    lo, hi = case["vox_lo"], case["vox_hi"]
    vox = [hi if case["n_lo"] == case["n_hi"] else int(round(lo + (hi - lo) * ((n - case["n_lo"]) / span) ** (1 / 3)))
           for n in ns]
    return [(int(n), v) for n, v in zip(ns, vox)]


def _steady(ctrls):
    """Controllers as a long run leaves them: windows at their upper bounds."""
    for c in ctrls:
        if c.move in (L.CRANK_SHAFT, L.SLIDE, L.END_PIVOT):
            c.amp_bead = int(c.bead_hi)
        elif c.move == L.TANGENT_ROTATION:
            c.amp_bead = min(12, int(c.bead_hi))
        c.rate = 0.6
    return ctrls


def _prepare_mc(case, seed):
    rs = np.random.RandomState(seed)
    B = case["B"]
    systems = []
    make = W.make_twist_system if case["twist"] else W.make_system
    for i, (n, v) in enumerate(_replica_sizes(case)):
        s = make(n, B, v, seed=int(rs.randint(2 ** 31 - 1)), chi=float(rs.uniform(0, 2)), eps=rs.uniform(-5, -1, size=B),
                 mu=rs.uniform(-2, 1, size=B), marks=case["marks"], cross_eps=-0.5 if B == 3 else 0.0)
        s.chain.states = (rs.random_sample((n, B)) < 0.3).astype(np.int64)
        s.field.fast_field = case["fast_field"]
        if case["steady"]:
            _steady(s.ctrls)
        systems.append(s)
    mode = L.RNG_GLIBC if case["rng"] == "glibc" else L.RNG_PHILOX
    k = len(systems)
    dr = DeviceReplicas([s.chain for s in systems], [s.field for s in systems], [s.ctrls for s in systems],
                        rng_mode=mode, seeds=[int(seed) % 65521 + 1] * k if mode == L.RNG_PHILOX
                        else [int(seed) % 65521 + 1 + i for i in range(k)],
                        streams=list(range(k)) if mode == L.RNG_PHILOX else None)
    dr.np_seed([int(seed) % 65521 + i for i in range(k)])
    return dict(case=case, dr=dr, turn=0)


def _confined_walk(rs, n, radius):
    """A 25 nm random walk that stays inside a sphere around the origin."""
    steps = rs.standard_normal((n, 3))
    steps *= 25.0 / np.linalg.norm(steps, axis=1)[:, None]
    r = np.zeros((n, 3))
    x = np.zeros(3)
    for i in range(1, n):
        y = x + steps[i]
        if y @ y > (radius - 5.0) ** 2:
            y = x - steps[i]
        if y @ y > (radius - 5.0) ** 2:
            y = x * (1.0 - 25.0 / np.linalg.norm(x))
        x = r[i] = y
    return r


def _script_polymer(case, seed):
    rs = np.random.RandomState(seed)
    n = case["n"]
    bonds = np.full(n - 1, 25.0)
    np.random.seed(seed % (2 ** 31))
    if case["field"] == "none":
        p = SSWLC.gaussian_walk_polymer("poly", n, bonds, lp=53.0, binder_names=np.array(["null_reader"]))
        return p, make_binder_collection([get_by_name("null_reader")]), NullField([p])
    binders = make_binder_collection([get_by_name("HP1")])
    args = dict(states=np.zeros((n, 1), dtype=int), binder_names=np.array(["HP1"]),
                chemical_mods=(rs.random_sample((n, 1)) < 0.4).astype(int),
                chemical_mod_names=np.array(["H3K9me3"]))
    vox = case["vox"]
    if case["field"] == "confined":
        radius = 20.0 * n ** (1 / 3)
        r = _confined_walk(rs, n, radius)
        t3, t2 = estimate_tangents_from_coordinates(r)
        p = Chromatin("chr", r, bead_length=bonds, t3=t3, t2=t2, **args)
        w = 2.3 * radius
        return p, binders, UniformDensityField([p], binders, w, vox, w, vox, w, vox, confine_type="Spherical",
                                               confine_length=radius)
    p = Chromatin.gaussian_walk_polymer("chr", n, bonds, **args)
    w = 30.0 * vox
    return p, binders, UniformDensityField([p], binders, w, vox, w, vox, w, vox)


def _prepare_script(case, seed):
    p, binders, field = _script_polymer(case, seed)
    bead_b, move_b = mc.get_amplitude_bounds([p])
    make = ctl.all_moves_except_binding_state if case["field"] == "none" else ctl.all_moves
    ctrls = make(".", bead_b.bounds, move_b.bounds, controller=ctl.SimpleControl)
    return dict(case=case, p=p, binders=binders, field=field, ctrls=ctrls, seed=int(seed) % 65521 + 1)


def _energy_system(case, seed):
    rs = np.random.RandomState(seed)
    B = case["B"]
    s = W.make_system(case["n"], B, 8, seed=int(rs.randint(2 ** 31 - 1)), chi=1.3, eps=EPS[:B], mu=MU[:B],
                      marks=case["marks"], cross_eps=0.6)
    s.chain.states = rs.randint(0, 3, size=(case["n"], B))
    f = s.field
    f.nx, f.ny, f.nz = case["nx"], case["ny"], case["nz"]
    f.x_width, f.y_width, f.z_width = 30.0 * f.nx, 30.0 * f.ny, 30.0 * f.nz
    return s


def _prepare_energy(case, seed):
    s = _energy_system(case, seed)
    if case["kind"] == "scatter":
        dr = DeviceReplicas([s.chain], [s.field], [s.ctrls], rng_mode=L.RNG_PHILOX, seeds=[1], streams=[0])
        return dict(case=case, dr=dr)
    model = EnergyModel(s.chain, s.field, s.binders)
    grad = case["kind"] == "autograd"
    r = torch.tensor(s.chain.r, dtype=torch.float64, device="cuda", requires_grad=grad)
    th = torch.tensor(model.theta0, dtype=torch.float64, device="cuda", requires_grad=grad)
    return dict(case=case, model=model, r=r, th=th)


def prepare(case, seed):
    """What a program has in hand before the call: chains, fields and controllers on the GPU."""
    if case["kind"] == "mc":
        return _prepare_mc(case, seed)
    if case["kind"] == "script":
        return _prepare_script(case, seed)
    return _prepare_energy(case, seed)


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def _chain_state(dr):
    return dict(pos=dr.pos, states=dr.states, density=dr.density, rng=dr.rng, controllers=dr.ctrl)


def run(state):
    """One pass, and every value that it computes or changes."""
    case = state["case"]
    if case["kind"] == "mc":
        dr = state["dr"]
        if case["launch"] == "step":
            dr.step(state["turn"])                  # the controllers in turn: every move type
            state["turn"] = (state["turn"] + 1) % dr.nctrl[0]
        elif case["launch"] == "plain":
            dr.run_plain(case["sweeps"])
        elif case["waves"]:
            dr.run(case["sweeps"], waves=case["waves"])
        else:
            dr.run(case["sweeps"])
        return _chain_state(dr)
    if case["kind"] == "script":
        p, field = state["p"], state["field"]
        mc.seed_libc(state["seed"])                 # a stream of its own: no other chain's draws enter
        mc.mc_sim([p], state["binders"], case["steps"], state["ctrls"], field, 1.0, state["seed"])
        state["seed"] += 1
        out = dict(r=p.r, t3=p.t3, t2=p.t2, states=p.states,
                   amplitudes=np.array([[c.move.amp_bead, c.move.amp_move] for c in state["ctrls"]]))
        if case["field"] != "none":
            out["density"] = field.density
        return out
    if case["kind"] == "scatter":
        state["dr"].density_init()
        return state["dr"].density
    if case["kind"] == "grad":
        return energy(state["model"], state["r"], state["th"], grad=True)
    r, th = state["r"], state["th"]
    r.grad = th.grad = None
    E = chromo_energy(r, th, state["model"])
    E.backward()
    return E.detach(), r.grad, th.grad


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

def _proposals(amps, counts, B, n_beads):
    """Bytes and operations of one sweep from the move counts and window bounds: 72 bytes a bead read
    and (half of the moves accepted) written, 8 (B + 1) bytes a voxel, about 3 new voxels a bead."""
    byt = flops = 0.0
    for move, k in counts.items():
        amp = min(amps[move], n_beads)
        if move == "tangent":
            beads, vox, per_bead = amp / 2 + 0.5, 0.0, 144 + 24
        elif move == "binding":
            beads, vox, per_bead = 1.0, 8.0, 2 * B
        else:
            # mean of the capped exponential draw, -log10(u) * 0.45 * amplitude + 1
            beads = min(0.195 * amp + 1, amp) * (1 if move == "pivot" else 1.6)
            vox, per_bead = (8 + 3 * beads if B else 0.0), 72 * 1.5 + B
        byt += k * (beads * per_bead + vox * 8 * (B + 1) * 1.5 + 96)
        flops += k * (beads * 400 + vox * 8 * (B + 1) + 200)
    return byt, flops


def work(case):
    """Bytes and operations of one pass: inputs read once, outputs written once."""
    kind = case["kind"]
    if kind == "mc":
        names = ("crank", "pivot", "slide", "tangent", "binding")
        B = case["B"]
        byt = flops = 0.0
        for n, _ in _replica_sizes(case):
            amps = (dict(crank=min(150, n), pivot=min(150, n // 2), slide=min(150, n), tangent=12, binding=1)
                    if case["steady"] else
                    dict(crank=min(30, n), pivot=min(50, n // 4), slide=min(10, n), tangent=1, binding=1))
            if case["launch"] == "step":
                b, f = _proposals(amps, dict.fromkeys(names, 0.2), B, n)
            else:
                b, f = _proposals(amps, dict(zip(names, ALL_MOVES)), B, n)
                b, f = b * case["sweeps"], f * case["sweeps"]
            byt, flops = byt + b, flops + f
        return {"bytes": byt, "flops": flops}
    if kind == "script":
        n = case["n"]
        B = 0 if case["field"] == "none" else 1
        amps = dict(crank=min(150, n), pivot=min(150, n // 2), slide=min(150, n), tangent=10, binding=1)
        counts = (dict(crank=5, pivot=5, slide=5, tangent=5) if not B else
                  dict(crank=30, pivot=1, slide=60, tangent=60, binding=10))
        b, f = _proposals(amps, counts, B, n)
        return {"bytes": b * case["steps"], "flops": f * case["steps"]}
    n, B = case["n"], case["B"]
    V = case["nx"] * case["ny"] * case["nz"]
    if kind == "scatter":
        return {"bytes": n * (24 + B) + 8 * (B + 1) * V, "flops": n * (60 + 16 * (B + 1))}
    # r, t3, states, marks and five bond parameters in, dE/dr out
    return {"bytes": n * (24 + 24 + 2 * B + 40 + 24), "flops": n * (400 + 32 * (B + 1)) + V * 8 * B * B}


# ---------------------------------------------------------------------------
# The same results in plain float64
# ---------------------------------------------------------------------------

def _densities(s, r):
    """Voxel densities (V, B + 1) of the chain by trilinear weights, differentiable in r."""
    c, f = s.chain, s.field
    dev = r.device
    n = torch.tensor([f.nx, f.ny, f.nz], device=dev)
    width = torch.tensor([f.x_width, f.y_width, f.z_width], dtype=torch.float64, device=dev)
    dx = width / n
    vol = f.x_width * f.y_width * f.z_width / (f.nx * f.ny * f.nz)
    q = (torch.remainder(r + width / 2, width) - dx / 2) / dx
    low = torch.floor(q.detach())
    w = 1 - (q - low)
    low = low.long()
    sel = torch.cat([torch.ones(c.N, 1, dtype=torch.float64, device=dev),
                     torch.as_tensor(np.asarray(c.states), dtype=torch.float64, device=dev)], dim=1)
    rho = torch.zeros(f.nx * f.ny * f.nz, c.B + 1, dtype=torch.float64, device=dev)
    for corner in range(8):
        o = torch.tensor([corner & 1, corner >> 1 & 1, corner >> 2 & 1], device=dev)
        i = torch.remainder(low + o, n)
        wt = torch.prod(torch.where(o == 0, w, 1 - w), dim=1) / vol
        rho = rho.index_add(0, i[:, 0] + n[0] * (i[:, 1] + n[1] * i[:, 2]), wt[:, None] * sel)
    return rho, vol


def _energy_terms(s, r, theta):
    """(elastic, field, binding) energies of the chain, differentiable in r and theta."""
    c, f, B = s.chain, s.field, s.chain.B
    dev = r.device
    rho, vol = _densities(s, r)
    field = theta[0] * (vol / f.bead_vol) * torch.sum((rho[:, 0] * f.bead_vol) ** 2)
    states = np.asarray(c.states)
    names = [b.name for b in s.binders]
    for j, b in enumerate(s.binders):
        e, v = theta[eps_index(B, j, j)], b.interaction_volume
        field = field + 0.5 * e * v * vol * torch.sum(rho[:, j + 1] ** 2)
        field = field + e * (1 - v / vol) * float(np.sum(states[:, j] == 2))
        for k in range(B):
            if names[k] in b.cross_talk_interaction_energy:
                field = field + theta[eps_index(B, j, k)] * v * vol * torch.sum(rho[:, j + 1] * rho[:, k + 1])
    t3 = torch.as_tensor(c.t3, device=dev)
    eb, epar, eperp, gam, eta = torch.as_tensor(np.asarray(c.bonds), device=dev)
    d = r[1:] - r[:-1]
    par = torch.sum(t3[:-1] * d, dim=1)
    perp = d - t3[:-1] * par[:, None]
    bend = t3[1:] - t3[:-1] - perp * eta[:, None]
    elastic = torch.sum(0.5 * eb * torch.sum(bend * bend, 1) + 0.5 * epar * (par - gam) ** 2
                        + 0.5 * eperp * torch.sum(perp * perp, 1))
    binding = torch.zeros((), dtype=torch.float64, device=dev)
    for j in range(B):
        mu = theta[1 + B * (B + 1) // 2 + j]
        binding = binding + float(np.sum(np.asarray(c.F)[j, np.asarray(c.marks)[:, j], states[:, j]]))
        binding = binding - mu * float(states[:, j].sum())
    return elastic, field, binding


def exact(case, seed):
    """run()'s outputs in plain float64 torch; None for a Monte Carlo chain, whose decisions
    have no value apart from the run that makes them."""
    if case["kind"] in ("mc", "script"):
        return None
    s = _energy_system(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    r = torch.tensor(s.chain.r, dtype=torch.float64, device=dev, requires_grad=case["kind"] != "scatter")
    if case["kind"] == "scatter":
        return _densities(s, r)[0].reshape(-1)
    B = case["B"]
    theta = np.zeros(n_theta(B))
    theta[0] = s.field.chi
    for i in range(B):
        for j in range(i, B):
            theta[eps_index(B, i, j)] = EPS[i] if i == j else 0.6
        theta[1 + B * (B + 1) // 2 + i] = MU[i]
    th = torch.tensor(theta, dtype=torch.float64, device=dev, requires_grad=True)
    terms = _energy_terms(s, r, th)
    E = sum(terms)
    gr, gt = torch.autograd.grad(E, (r, th))
    if case["kind"] == "autograd":
        return E.detach(), gr, gt
    return torch.stack([E.detach(), *[t.detach() for t in terms]]), gr, gt
