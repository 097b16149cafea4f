"""Performance cases: the work that users of this framework have it do.

Four kinds of use, told apart by a case's ``path``:

* ``step``: a simulation.  ``steps`` time steps of one domain
  (``Domain.run``), after which the program takes the new state on the device
  (``Domain.device_ptr``), as one that couples, monitors or saves does.  Two
  and three phases, the Corey and the reference's closures (Brooks-Corey, van
  Genuchten), with and without the energy equation, with and without the
  non-finite check.
* ``shard``: one z slab of a domain spread over several GPUs: every step also
  writes the planes that the neighbours need (``Domain.set_halo_pack``).
* ``ensemble``: many two-phase realizations of uneven sizes advanced together
  (``Batch.run``).
* ``gradient``: one iteration of a permeability and porosity inversion, the
  loss and its gradient by the discrete adjoint
  (``autograd.history_matching_loss``), from and to host tensors as that
  wrapper works.

The physics are those of ``capaz_amd/workloads.py`` and of the reference's
decks; a seed draws porosity, permeability and a little of the initial state.
"""
from __future__ import annotations

import math

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

from capaz_amd import capaz, workloads
from capaz_amd.autograd import HistoryMatchingProblem, history_matching_loss

F64 = torch.float64

# The values of the reference's Two-phase/defines.ini that a step reads.
DECK_2PH = dict(MODEL=2, HX=5e-2, HY=5e-2, HZ=5e-2, DT=1e-4, SOURCE=30, BETA_W=4.4e-7, BETA_N=1e-6, K_0=6.64e-11,
                MU_W=0.001, MU_N=0.0009, RO_W=1000, RO_N=1460, LAMBDA_0=2.7, S_WR_0=0.09, S_N_GR=0.2, P_D_0=755,
                P_ATM=100000, G_CONST=9.807, ITERATIONS=10)


def _step(physics, nx, ny, nz, steps, check_every=0):
    return dict(path="step", physics=physics, nx=nx, ny=ny, nz=nz, steps=steps, check_every=check_every)


def listed():
    return [
        # the smallest call: a coupled program that takes the state after every step of a small domain
        dict(_step("corey3", 24, 24, 24, 1), name="injection 24^3, step by step"),
        # the two-phase Buckley-Leverett workload at its own size, read every 20 steps
        dict(_step("corey2", 40, 40, 40, 20), name="buckley-leverett 40^3"),
        # the three-phase injection at its specified size
        dict(_step("corey3", 128, 128, 128, 10), name="injection 128^3"),
        # an uneven grid, as a field model gives it, with the non-finite check on
        dict(_step("corey3", 203, 117, 83, 10, 10), name="injection 203x117x83"),
        # the headline workload
        dict(_step("corey3", 256, 256, 256, 10), name="injection 256^3"),
        # the two-phase physics at the headline's size
        dict(_step("corey2", 256, 256, 256, 10), name="buckley-leverett 256^3"),
        # the reference's three-phase deck (van Genuchten closures, 7 Newton iterations)
        dict(_step("deck3", 160, 144, 130, 5), name="van Genuchten deck"),
        # the reference's two-phase deck (Brooks-Corey closures, 10 Newton iterations)
        dict(_step("deck2", 190, 150, 110, 5), name="Brooks-Corey deck"),
        # the non-isothermal two-phase workload at its specified size
        dict(_step("energy2", 256, 256, 128, 5), name="non-isothermal 256x256x128"),
        # the reference's three-phase energy model
        dict(_step("energy3", 160, 128, 96, 5), name="energy deck"),
        # the ensemble workload, half as many realizations, launch shape chosen by the autotuner
        dict(path="ensemble", count=32, lo=32, hi=96, steps=20, autotune=True, name="ensemble of 32"),
        # an iteration of the inversion workload, a quarter of its steps
        dict(path="gradient", n=96, steps=100, every=25, columns=16, name="inversion gradient 96^3"),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["step"] * 9 + ["shard", "ensemble", "gradient"])
    if kind == "ensemble":
        lo = size(20, 60)
        return dict(path="ensemble", count=rng.randint(6, 32), lo=lo, hi=min(96, lo + size(8, 60)),
                    steps=rng.randint(5, 20), autotune=rng.random() < 0.5)
    if kind == "gradient":
        steps = rng.randint(10, 60)
        return dict(path="gradient", n=size(20, 90), steps=steps, every=rng.randint(5, steps),
                    columns=rng.randint(4, 16))
    if kind == "shard":
        return dict(path="shard", physics=rng.choice(["corey3", "corey2"]), nx=size(60, 256), ny=size(60, 256),
                    nz=size(10, 40), steps=rng.randint(1, 10), check_every=0)
    physics = rng.choice(["corey3", "corey3", "corey3", "corey2", "corey2", "deck3", "deck2", "energy2", "energy3"])
    most = {"corey3": 12e6, "corey2": 12e6, "deck3": 3e6, "deck2": 3e6, "energy2": 6e6, "energy3": 2e6}[physics]
    while True:
        nx, ny, nz = size(20, 256), size(20, 256), size(20, 256)
        if nx * ny * nz <= most:
            break
    steps = rng.choice([1, 2, 5, 10, 20] if nx * ny * nz < 1e6 else [1, 2, 5])
    return _step(physics, nx, ny, nz, steps, steps if rng.random() < 0.2 else 0)


# ---- inputs -----------------------------------------------------------------------


def _keys(physics, nx, ny, nz):
    if physics == "corey3":
        keys = workloads.three_phase_injection(4)[0]
    elif physics == "corey2":
        keys = dict(workloads.buckley_leverett_2ph(4)[0], SOURCE=max(nx, nz))
    elif physics == "deck3":
        keys = dict(workloads.REF_3PH_DECK, DT=1e-4)
    elif physics == "deck2":
        keys = dict(DECK_2PH)
    elif physics == "energy2":
        keys = dict(workloads.nonisothermal_2ph(4, 4, 4)[0], SOURCE=max(nx, nz))
    else:
        keys = workloads.energy_3ph(4, 4, 4)[0]
    return dict(keys, NX=nx, NY=ny, NZ=nz)


def _inputs(physics, keys, seed):
    """The initial fields, (Nz, Ny, Nx) on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    shape = (keys["NZ"], keys["NY"], keys["NX"])
    normal = lambda: torch.randn(shape, generator=g, device="cuda", dtype=F64)
    full = lambda v: torch.full(shape, float(v), device="cuda", dtype=F64)
    f = {"m": (0.4 * (1 + 0.05 * normal())).clamp(0.3, 0.5)}
    depth = torch.arange(shape[1], device="cuda", dtype=F64).reshape(1, -1, 1).expand(shape)
    K = 0.5 * normal() if physics == "corey3" else 0.05 * normal()
    f["K"] = keys["K_0"] * torch.exp(K)
    if physics in ("corey3", "deck3", "energy3"):
        Sw, Sn = (0.2, 0.7) if physics == "corey3" else (0.4, 0.3)
        P = full(keys["P_ATM"])
        if physics == "energy3":
            P = P + 1000.0 * keys["G_CONST"] * keys["HY"] * depth
            f["T"] = full(285.0)
        f.update(P_w=P, P_n=P.clone(), P_g=P.clone(), S_w=Sw + 0.01 * torch.tanh(normal()),
                 S_n=Sn + 0.01 * torch.tanh(normal()))
    elif physics == "deck2":
        f.update(P_w=keys["P_ATM"] + keys["RO_W"] * 0.4 * keys["G_CONST"] * keys["HY"] * depth,
                 S_n=0.1 + 0.01 * torch.tanh(normal()))
    else:
        f.update(P_w=full(keys["P_ATM"]), S_n=0.85 + 0.01 * torch.tanh(normal()))
        if physics == "energy2":
            f["T"] = full(293.0)
    return f


def _ensemble_sizes(case):
    """Edges of the realizations, spread unevenly over lo .. hi."""
    return [case["lo"] + (37 * r * r + 11 * r) % (case["hi"] - case["lo"] + 1) for r in range(case["count"])]


def _ensemble_inputs(case, seed):
    """Per realization: the correlated lognormal K and the porosity of
    workloads.ensemble (a Gaussian filter of 4 cells, ln-sigma 1)."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    keys = dict(workloads.buckley_leverett_2ph(4)[0], DT=1e-6, SOURCE=case["hi"])
    members = []
    for n in _ensemble_sizes(case):
        w = torch.randn((n, n, n), generator=g, device="cuda", dtype=F64)
        k2 = torch.fft.fftfreq(n, device="cuda", dtype=F64) ** 2
        damp = torch.exp(-2 * math.pi ** 2 * 16 * k2)
        w = torch.fft.fftn(w) * damp[:, None, None] * damp[None, :, None] * damp[None, None, :]
        w = torch.fft.ifftn(w).real.contiguous()
        w = (w - w.mean()) / w.std()
        K = workloads.K_MEAN * torch.exp(w)
        full = lambda v: torch.full((n, n, n), float(v), device="cuda", dtype=F64)
        members.append(dict(P_w=full(keys["P_ATM"]), S_n=full(0.85), K=K,
                            m=(0.4 * (K / workloads.K_MEAN) ** 0.1).clamp(0.25, 0.5)))
    return keys, members


def _gradient_inputs(case, seed):
    """The inversion of workloads.history_matching on an n^3 grid: initial
    state, trial ln K and porosity and the observed columns, on the host."""
    n = case["n"]
    rng = np.random.default_rng(int(seed))
    keys = dict(workloads.three_phase_injection(4)[0], NX=n, NY=n, NZ=n, DT=1e-6)
    shape = (n, n, n)
    P = np.full(shape, keys["P_ATM"])
    state = dict(P_w=P, P_n=P, P_g=P, S_w=0.2 + 0.01 * rng.random(shape), S_n=0.7 + 0.01 * rng.random(shape))
    lnK = np.log(workloads.K_MEAN) + 0.3 * rng.standard_normal(shape)
    m = np.clip(0.4 * (1 + 0.05 * rng.standard_normal(shape)), 0.3, 0.5)
    ik = rng.choice((n - 2) * (n - 2), size=case["columns"], replace=False)
    j = np.arange(1, n - 1)
    cells = ((1 + ik % (n - 2))[:, None] + j[None, :] * n + (1 + ik // (n - 2))[:, None] * n * n).ravel()
    steps = np.arange(case["every"], case["steps"] + 1, case["every"])
    seen = (len(steps), cells.size)
    obs = dict(cells=cells.astype(np.int64), steps=steps.astype(np.int64), S_w=0.2 + 0.01 * rng.random(seen),
               S_n=0.7 + 0.01 * rng.random(seen))
    return keys, state, lnK, m, obs


class _Array:
    """A device array of the framework as torch takes it, without a copy; a
    tensor made from it keeps `owner`, whose memory it is, alive."""

    def __init__(self, address, shape, owner):
        self.owner = owner
        self.__cuda_array_interface__ = dict(data=(address, False), shape=tuple(shape), typestr="<f8", version=3)


def _put(domain, fields):
    for name, value in fields.items():
        torch.as_tensor(_Array(domain.device_ptr(name), domain.shape, domain), device="cuda").copy_(value)


def _outputs(physics):
    return {"corey3": ("P_w", "S_w", "S_n"), "deck3": ("P_w", "S_w", "S_n"), "corey2": ("P_w", "S_n"),
            "deck2": ("P_w", "S_n"), "energy2": ("P_w", "S_n", "T"), "energy3": ("P_w", "S_w", "S_n", "T")}[physics]


def _slab(case):
    """Planes and bytes of a shard's halo buffer."""
    return (10 if case["physics"] == "corey3" else 4, case["ny"], case["nx"])


def prepare(case, seed):
    if case["path"] == "gradient":
        keys, state, lnK, m, obs = _gradient_inputs(case, seed)
        problem = HistoryMatchingProblem(keys, state, obs, case["steps"])
        return dict(case=case, problem=problem, lnK=torch.tensor(lnK, requires_grad=True),
                    m=torch.tensor(m, requires_grad=True))
    if case["path"] == "ensemble":
        keys, members = _ensemble_inputs(case, seed)
        batch = capaz.Batch(keys, [dict(dims=(n, n, n)) for n in _ensemble_sizes(case)])
        for domain, fields in zip(batch.domains, members):
            _put(domain, fields)
        torch.cuda.synchronize()
        if case["autotune"]:
            batch.autotune()
        return dict(case=case, batch=batch, views={}, step=1)
    keys = _keys(case["physics"], case["nx"], case["ny"], case["nz"])
    domain = capaz.Domain(keys)
    _put(domain, _inputs(case["physics"], keys, seed))
    state = dict(case=case, domain=domain, views={}, step=1)
    if case["check_every"]:
        domain.tune(check_every=case["check_every"])
    if case["path"] == "shard":
        state["halo"] = torch.zeros(_slab(case), device="cuda", dtype=F64)
        domain.set_halo_pack(state["halo"].data_ptr())
    torch.cuda.synchronize()
    return state


def _taken(views, domain, name, owner):
    """The field's current device array; its torch view is made once for each of the two that a step alternates."""
    address = domain.device_ptr(name)
    if address not in views:
        views[address] = torch.as_tensor(_Array(address, domain.shape, owner), device="cuda")
    return views[address]


def run(state):
    case = state["case"]
    if case["path"] == "gradient":
        lnK, m = state["lnK"], state["m"]
        lnK.grad = m.grad = None
        loss = history_matching_loss(lnK, m, state["problem"])
        loss.backward()
        return dict(loss=loss.detach(), lnK=lnK.grad, m=m.grad)
    first, state["step"] = state["step"], state["step"] + case["steps"]
    if case["path"] == "ensemble":
        batch = state["batch"]
        batch.run(case["steps"], first)
        return [{name: _taken(state["views"], d, name, batch) for name in ("P_w", "S_n")} for d in batch.domains]
    domain = state["domain"]
    domain.run(case["steps"], first)
    out = {name: _taken(state["views"], domain, name, domain) for name in _outputs(case["physics"])}
    if "halo" in state:
        out["halo"] = state["halo"]
    return out


def work(case):
    """Bytes: per step the state and the parameters once in and the new state
    once out (a step reads every cell's neighbours, so a larger grid than the
    caches hold cannot skip a sweep).  Flops: the closures, the upwind fluxes
    and the fixed Newton iterations of a cell, counted from the formulas with
    a division, a power or an exponential as one."""
    if case["path"] == "gradient":
        cells, steps = case["n"] ** 3, case["steps"]
        # forward, then the two passes of the adjoint step: the state and the
        # adjoint in and out, the parameters and their gradients
        return dict(bytes=steps * cells * (64 + 8 * (5 + 3 + 2 + 3 + 2 + 2)), flops=steps * cells * (620 + 1300))
    if case["path"] == "ensemble":
        cells = sum(n ** 3 for n in _ensemble_sizes(case))
        return dict(bytes=cells * case["steps"] * 48, flops=cells * case["steps"] * 260)
    cells = case["nx"] * case["ny"] * case["nz"]
    fields, flops = {"corey3": (8, 620), "deck3": (8, 880), "corey2": (6, 260), "deck2": (6, 420),
                     "energy2": (8, 1000), "energy3": (10, 1500)}[case["physics"]]
    extra = 8 * math.prod(_slab(case)) if case["path"] == "shard" else 0
    return dict(bytes=case["steps"] * (8 * fields * cells + extra), flops=case["steps"] * cells * flops)


# ---- the same values in plain torch -----------------------------------------------


def _grow(a):
    """Each boundary cell takes its inward neighbour's value."""
    for d in range(3):
        n = a.shape[d]
        a = torch.cat([a.narrow(d, 0, 1), a, a.narrow(d, n - 1, 1)], d)
    return a


def _in(a, axis=0, by=0):
    """The interior cells of a field, or their neighbours `by` cells along x (2), y (1) or z (0)."""
    for d in range(3):
        a = a.narrow(d, 1 + (by if d == axis else 0), a.shape[d] - 2)
    return a


def _part(x, sign):
    return (x + sign * x.abs()) / 2


def _flux(k, P, Xi, ro):
    """Divergence of one phase's upwind Darcy flux on the interior cells."""
    total = 0
    c = lambda a: _in(a)
    for axis, h in ((2, k["HX"]), (1, k["HY"]), (0, k["HZ"])):
        lift = k["G_CONST"] * c(ro) if axis == 1 else 0.0
        x1 = -(c(P) - _in(P, axis, -1)) / h + lift
        x2 = -(_in(P, axis, 1) - c(P)) / h + lift
        t1 = -(_part(x2, 1) - _part(x1, -1)) * c(Xi) * c(ro)
        t2 = -_part(x1, 1) * _in(Xi, axis, -1) * _in(ro, axis, -1)
        t3 = -_part(x2, -1) * _in(Xi, axis, 1) * _in(ro, axis, 1)
        total = total + (t1 - t2 + t3) / h
    return total


def _solve(A, b):
    """Gaussian elimination of a small system whose entries are fields."""
    n = len(b)
    A, b = [list(r) for r in A], list(b)
    for q in range(n):
        for r in range(q + 1, n):
            f = A[r][q] / A[q][q]
            A[r] = [A[r][s] - f * A[q][s] if s > q else 0.0 for s in range(n)]
            b[r] = b[r] - f * b[q]
    for q in reversed(range(n)):
        for s in range(q + 1, n):
            b[q] = b[q] - A[q][s] * b[s]
        b[q] = b[q] / A[q][q]
    return b


def _closures(k, f):
    """Relative permeabilities per phase and the two-phase capillary pressure."""
    corey = k.get("CLOSURE") == "corey"
    if k["MODEL"] == 2:
        if corey:
            se = (1 - f["S_n"] - k["S_WR_0"]) / (1 - k["S_WR_0"] - k["S_NR_0"])
            return [se.clamp(0, 1) ** 2, (1 - se).clamp(0, 1) ** 2], 0.0
        se, lam = (1 - f["S_n"] - k["S_WR_0"]) / (1 - k["S_WR_0"]), k["LAMBDA_0"]
        kr = [se ** ((2 + 3 * lam) / lam), (1 - se) ** 2 * (1 - se ** ((2 + lam) / lam))]
        return kr, k["P_D_0"] * se ** (-1 / lam)
    den = 1 - k["S_WR_0"] - k["S_NR_0"] - k["S_GR_0"]
    w, n = (f["S_w"] - k["S_WR_0"]) / den, (f["S_n"] - k["S_NR_0"]) / den
    g = 1 - w - n
    if corey:
        return [w.clamp(0, 1) ** 2, n.clamp(0, 1) ** 2, g.clamp(0, 1) ** 2], 0.0
    a = k["LAMBDA_0"] / (k["LAMBDA_0"] - 1)
    b, c = 1 / a, 2 / a
    kw = w.sqrt() * (1 - (1 - w ** a) ** b) ** 2
    kg = g.sqrt() * (1 - (1 - g) ** a) ** c
    kn = n * (1 - w).sqrt() * (1 - w ** a) ** c * n.sqrt() * (1 - (1 - n ** a) ** b) ** 2 / (1 - w) / (1 - g)
    return [torch.where(w >= 1e-3, kw, 0.0), torch.where(n >= 1e-3, kn, 0.0), torch.where(g >= 1e-3, kg, 0.0)], 0.0


def _mu(k, T):
    if T is None or k.get("ENERGY_CLOSURE") == "config":
        f = 1.0 if T is None else torch.exp(-k["MU_T_A"] * (T - k["MU_T_REF"]))
        return [k["MU_W"] * f, k["MU_N"] * f, k.get("MU_G", 0.0) * f]
    return [1 / (29.21 * T - 7506.64), 7.256e-10 * torch.exp(4141.9 / T), 1.717e-5 * (T / 273) ** 0.683]


def _density(k, a, P, T):
    """Density of phase a and its derivatives in P and T."""
    t = 0.0 if T is None else T - 273
    if a == 2:
        s = 1.0 if T is None else 273 / T
        r = k["RO_G"] * P / k["P_ATM"] * s
        return r, k["RO_G"] / k["P_ATM"] * s + 0 * P, None if T is None else -r / T
    r0, beta, alfa = [(k["RO_W"], k["BETA_W"], 1.32e-7), (k["RO_N"], k["BETA_N"], 9.2e-7)][a]
    return r0 * (1 + beta * (P - k["P_ATM"]) - alfa * t), r0 * beta + 0 * P, None if T is None else -r0 * alfa + 0 * T


def _heat(k, T):
    """Enthalpies and heat capacities of the phases and of the rock, and the rock's density."""
    t, config = T - 273, k.get("ENERGY_CLOSURE") == "config"
    sign = -1 if config else 1  # the reference's cubic term of H_w has the other sign than its c_w
    rr = k["RO_R"] if config else 2000.0
    H = [k["P_ATM"] / k["RO_W"] + t * (4194 - t * (0.575 + sign * 0.015 * t / 3)),
         k["P_ATM"] / k["RO_N"] + t * (1700 + 1.7 * t)]
    c = [4194 - 1.15 * t + 0.015 * t * t, 1700 + 3.4 * t]
    if k["MODEL"] == 3:
        H.append(k["P_ATM"] / k["RO_G"] + t * (1000 + 0.0595 * t))
        c.append(1000 + 0.119 * t)
    if config:
        return H, c, k["P_ATM"] / rr + t * k["C_R"], k["C_R"] + 0 * t, rr
    return H, c, k["P_ATM"] / rr + t * (800 + 0.375 * t), 800 + 0.75 * t, rr


def _velocity(k, P, Xi, ro, axis, h, lift):
    """Darcy velocity of every cell: central differences, one-sided at the faces."""
    n = P.shape[axis]
    mid = (P.narrow(axis, 2, n - 2) - P.narrow(axis, 0, n - 2)) / (2 * h)
    lo = (P.narrow(axis, 1, 1) - P.narrow(axis, 0, 1)) / h
    hi = (P.narrow(axis, n - 1, 1) - P.narrow(axis, n - 2, 1)) / h
    return Xi * (torch.cat([lo, mid, hi], axis) - (ro * k["G_CONST"] if lift else 0.0))


def _next(k, f):
    """One time step of the fields f (P_w, S_n, ...; m and K among them) under the deck k."""
    ph, T = k["MODEL"], f.get("T")
    config = k.get("ENERGY_CLOSURE") == "config"
    kr, Pk = _closures(k, f)
    mu = _mu(k, T)
    Xi = [-f["K"] * kr[a] / mu[a] for a in range(ph)]
    if ph == 2:
        P = [f["P_w"], f["P_w"] + Pk]
        S = [1 - f["S_n"], f["S_n"]]
    else:
        inner = torch.zeros_like(f["P_w"], dtype=torch.bool)
        inner[1:-1, 1:-1, 1:-1] = True
        P = [f["P_w"]] + [torch.where(inner, f["P_w"], f[n]) for n in ("P_n", "P_g")]
        S = [f["S_w"], f["S_n"], 1 - f["S_w"] - f["S_n"]]
    ro = [_density(k, a, P[a], T)[0] for a in range(ph)]
    m = _in(f["m"])
    A = [_in(ro[a] * S[a]) - k["DT"] / m * _flux(k, P[a], Xi[a], ro[a]) for a in range(ph)]
    p, s = _in(f["P_w"]), [_in(v) for v in S]
    t = None if T is None else _in(T)
    if T is not None:
        H, _, Hr, _, rr = _heat(k, T)
        E = f["m"] * sum(S[a] * (ro[a] * H[a] - P[a]) for a in range(ph)) + (1 - f["m"]) * (rr * Hr - P[0])
        if config:
            lam = k["LAMBDA_EFF"] + 0 * T
        else:
            lw, ln = 0.553 * (1 - 3e-3 * (T - 273)), 0.14 * (1 - 1e-3 * (T - 273))
            lam = f["m"] * (S[0] * lw + S[1] * ln + S[2] * 0.0237 * (T / 273) ** 0.82) + (1 - f["m"])
        heat, carried = 0.0, 0.0
        for axis, h in ((2, k["HX"]), (1, k["HY"]), (0, k["HZ"])):
            q = lam * T
            term = (_in(q, axis, 1) - 2 * _in(q) + _in(q, axis, -1)) / (h * h)
            heat = term if axis == 0 and not config else heat + term  # the reference keeps its z term alone
            up = axis if axis or config else 1  # and carries with the y velocity along z
            for a in range(ph):
                v = ro[a] * H[a] * _velocity(k, P[a], Xi[a], ro[a], up, (k["HZ"], k["HY"], k["HX"])[up], up == 1)
                carried = carried + (_in(v, axis, 1) - _in(v, axis, -1)) / (2 * h)
        E = _in(E) + k["DT"] * (heat - carried)
    for _ in range(int(k["ITERATIONS"])):
        one = torch.ones_like(p)
        if T is not None:
            d = [_density(k, a, p, t) for a in range(ph)]
            H, c, Hr, cr, rr = _heat(k, t)
            F = [sum(s) - 1] + [d[a][0] * s[a] - A[a] for a in range(ph)]
            F.append(m * sum(s[a] * (d[a][0] * H[a] - p) for a in range(ph)) + (1 - m) * (rr * Hr - p) - E)
            J = [[one] * ph + [0 * one, 0 * one]]
            J += [[d[a][0] if b == a else 0 * one for b in range(ph)] + [d[a][1] * s[a], d[a][2] * s[a]]
                  for a in range(ph)]
            J.append([m * (d[a][0] * H[a] - p) for a in range(ph)] +
                     [m * sum(s[a] * (d[a][1] * H[a] - 1) for a in range(ph)) - (1 - m),
                      m * sum(s[a] * (d[a][2] * H[a] + d[a][0] * c[a]) for a in range(ph)) + (1 - m) * rr * cr])
            step = _solve(J, F)
            s = [s[a] - step[a] for a in range(ph)]
            p, t = p - step[ph], t - step[ph + 1]
        elif ph == 2:
            pk = dpk = 0.0
            if k.get("CLOSURE") != "corey":
                se, lam = (1 - s[1] - k["S_WR_0"]) / (1 - k["S_WR_0"]), k["LAMBDA_0"]
                pk = k["P_D_0"] * se ** (-1 / lam)
                dpk = k["P_D_0"] * se ** (-1 / lam - 1) / (lam * (1 - k["S_WR_0"]))
            rw, dw, _ = _density(k, 0, p, None)
            rn, dn, _ = _density(k, 1, p + pk, None)
            F1, F2 = rw * (1 - s[1]) - A[0], rn * s[1] - A[1]
            a, b, c, e = dw * (1 - s[1]), -rw, dn * s[1], rn + dn * s[1] * dpk
            det = a * e - b * c
            p, n = p - (e * F1 - b * F2) / det, s[1] - (a * F2 - c * F1) / det
            s = [1 - n, n]
        else:
            rw, dw, _ = _density(k, 0, p, None)
            rn, dn, _ = _density(k, 1, p, None)
            rg, dg, _ = _density(k, 2, p, None)
            g = 1 - s[0] - s[1]
            F1, F2, F3 = rw * s[0] - A[0], rn * s[1] - A[1], rg * g - A[2]
            # rows [dw Sw, rw, 0], [dn Sn, ro0_n Sn, rn] (the reference's middle entry), [dg Sg, -rg, -rg]
            q = k["RO_N"] * s[1]
            w0, w1 = F1 / rw, dw * s[0] / rw
            n0, n1 = (F2 - q * w0) / rn, (dn * s[1] - q * w1) / rn
            dp = (F3 + rg * (w0 + n0)) / (dg * g + rg * (w1 + n1))
            p, s = p - dp, [s[0] - (w0 - w1 * dp), s[1] - (n0 - n1 * dp)]
    # the boundary cells from their inward neighbours
    Pw, out = _grow(p), dict(m=f["m"], K=f["K"])
    top, bottom = torch.zeros_like(Pw), torch.zeros_like(Pw)
    top[:, 0], bottom[:, -1] = 1, 1
    top, bottom = top.bool(), bottom.bool()
    ghy = k["G_CONST"] * k["HY"]
    if ph == 2:
        Sn = _grow(s[1])
        nz, _, nx = Pw.shape
        i, kk = torch.arange(nx, device=Pw.device), torch.arange(nz, device=Pw.device)[:, None, None]
        src = int(k["SOURCE"])
        window = top & (i >= nx // 2 - src) & (i <= nx // 2 + src) & (kk >= nz // 2 - src) & (kk <= nz // 2 + src)
        low = _grow(_in(ro[1]) * s[1] + _in(ro[0]) * (1 - s[1])) * _grow(m) * ghy
        out["S_n"] = torch.where(window, k["S_N_GR"], Sn) if src > 0 else Sn
        end = k["P_BOTTOM"] + 0 * Pw if k.get("P_BOTTOM", 0) > 0 else Pw + low
        out["P_w"] = torch.where(top, k["P_ATM"], torch.where(bottom, end, Pw))
    else:
        inject = top if k["SOURCE"] > 0 else torch.zeros_like(top)
        out["S_w"] = torch.where(inject, k["S_W_GR"], _grow(s[0]))
        out["S_n"] = torch.where(inject, k["S_N_GR"], _grow(s[1]))
        for name, r0, beta in (("P_w", k["RO_W"], k["BETA_W"]), ("P_n", k["RO_N"], k["BETA_N"])):
            lift = r0 * ghy * (1 - beta * k["P_ATM"])
            out[name] = torch.where(top, (Pw - lift) / (1 + beta * r0 * ghy),
                                    torch.where(bottom, (Pw + lift) / (1 - beta * r0 * ghy), Pw))
        r = k["RO_G"] * ghy / k["P_ATM"]
        out["P_g"] = torch.where(top, Pw / (1 + r), torch.where(bottom, Pw / (1 - r), Pw))
    if T is not None:
        T1 = _grow(t)
        if config:
            T1 = torch.where(top, k["T_TOP"], T1) if k["T_TOP"] > 0 else T1
            out["T"] = torch.where(bottom, k["T_BOTTOM"], T1) if k["T_BOTTOM"] > 0 else T1
        else:
            out["T"] = torch.where(top, 400.0, torch.where(bottom, 273.0, T1))
    return out


def _exact_gradient(case, seed):
    k, state, lnK, m, obs = _gradient_inputs(case, seed)
    names = ("P_w", "P_n", "P_g", "S_w", "S_n")
    dev = lambda a: torch.tensor(a, device="cuda")
    lnK, m = dev(lnK).requires_grad_(), dev(m).requires_grad_()
    cells, steps = dev(obs["cells"]), list(obs["steps"])

    def one(K, m, *x):
        f = _next(k, dict(zip(names, x), m=m, K=K))
        return tuple(f[n] for n in names)

    x, K, loss = tuple(dev(np.array(state[n])) for n in names), lnK.exp(), 0.0
    for t in range(1, case["steps"] + 1):
        x = checkpoint(one, K, m, *x, use_reentrant=False)
        if t in steps:
            q = steps.index(t)
            for name in ("S_w", "S_n"):
                loss = loss + 0.5 * ((x[names.index(name)].flatten()[cells] - dev(obs[name][q])) ** 2).sum()
    loss.backward()
    return dict(loss=loss.detach().cpu(), lnK=lnK.grad.cpu(), m=m.grad.cpu())


def exact(case, seed):
    if case["path"] == "gradient":
        return _exact_gradient(case, seed)
    if case["path"] == "ensemble":
        keys, members = _ensemble_inputs(case, seed)
        out = []
        for f in members:
            for _ in range(case["steps"]):
                f = _next(keys, f)
            out.append({name: f[name] for name in ("P_w", "S_n")})
        return out
    keys = _keys(case["physics"], case["nx"], case["ny"], case["nz"])
    f = _inputs(case["physics"], keys, seed)
    for _ in range(case["steps"]):
        f = _next(keys, f)
    out = {name: f[name] for name in _outputs(case["physics"])}
    if case["path"] == "shard":
        names = ("P_w", "S_w", "S_n", "P_n", "P_g") if keys["MODEL"] == 3 else ("P_w", "S_n")
        planes = []
        for name in names:
            for z in (1, case["nz"] - 2):
                # away from the boundary P_n and P_g go out as the new P_w, which the next step takes them for
                plane = f[name][z].clone()
                if name in ("P_n", "P_g"):
                    plane[1:-1, 1:-1] = f["P_w"][z][1:-1, 1:-1]
                planes.append(plane)
        out["halo"] = torch.stack(planes)
    return out
