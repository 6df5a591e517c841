"""The calls a user of this package makes, as measurable cases.

Every case is one pass of work that a simulation script (or the C host) repeats:
Metropolis sweeps of one lattice or of a batch of replicas, a step of a field
ramp, a megastep with its log line, energy differences of proposed moves, the
adjoint of a batch, a forward and backward pass through torch.autograd, and the
observables written after a megastep.  Lattices are drawn from the case's seed:
unit dipoles uniform on the sphere (the "random" initial lattice) and, for a
solid solution, a fraction of vacancies.

listed()              the cases that are always measured
draw(rng)             one more case of the same ranges
prepare(case, seed)   the context, plan and inputs a script holds before the call
run(state)            one pass and its outputs
work(case)            bytes and FP64 operations a pass cannot do without
exact(case, seed)     the outputs from plain torch in 64 bits (None where there are none)
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import starrynight_amd as sn
from starrynight_amd._lib import lib

DEVICE = "cuda:0"
POT_CUTOFF = 6        # dipole_potential's range
EFIELD_CUTOFF = 4     # the field maps' cutoff (as the C host writes them)
RADIAL_BINS = 81      # r^2 = 0..80

# what one drawn case may cost: FP64 operations of a pass, sites resident
MAX_FLOPS = 6e10
MAX_SITES = 4 * 128 ** 3


def listed():
    return [
        # the drop-in for the reference's site_energy: one move of its 25 x 25 lattice
        {"name": "site_energy_one", "kind": "site_energy", "X": 25, "Y": 25, "Z": 1, "rc": 3, "n": 1},
        # energy differences of a list of trial moves held in host memory
        {"name": "site_energy_list", "kind": "site_energy", "X": 64, "Y": 64, "Z": 64, "rc": 3, "n": 100000},
        # the reference's CPU-runnable configuration: one 25 x 25 lattice, a run of sweeps and its counters
        {"name": "square25", "kind": "sweep", "X": 25, "Y": 25, "Z": 1, "rc": 3, "replicas": 1, "spread": 0,
         "T0": 300.0, "T1": 300.0, "vacant": 0.0, "K": 0.0, "axes": False, "sweeps": 100},
        # a temperature scan of that lattice, 512 replicas at once
        {"name": "square25_scan", "kind": "sweep", "X": 25, "Y": 25, "Z": 1, "rc": 3, "replicas": 512, "spread": 0,
         "T0": 50.0, "T1": 500.0, "vacant": 0.0, "K": 0.0, "axes": False, "sweeps": 20},
        # equilibrium statistics: 64 chains of a 12^3 lattice
        {"name": "cube12_chains", "kind": "sweep", "X": 12, "Y": 12, "Z": 12, "rc": 3, "replicas": 64, "spread": 0,
         "T0": 600.0, "T1": 600.0, "vacant": 0.0, "K": 0.0, "axes": False, "sweeps": 10},
        # the example run file: a megastep of 50 sweeps of 64^3, then its log line (moment and energy)
        {"name": "cube64_megastep", "kind": "megastep", "X": 64, "Y": 64, "Z": 64, "rc": 3, "T0": 300.0,
         "vacant": 0.0, "K": 0.0, "sweeps": 50},
        # one large lattice
        {"name": "cube128", "kind": "sweep", "X": 128, "Y": 128, "Z": 128, "rc": 3, "replicas": 1, "spread": 0,
         "T0": 300.0, "T1": 300.0, "vacant": 0.0, "K": 0.0, "axes": False, "sweeps": 4},
        # a batch of uneven sizes, 16^3 to 48^3
        {"name": "uneven_batch", "kind": "sweep", "X": 16, "Y": 16, "Z": 16, "rc": 3, "replicas": 33, "spread": 32,
         "T0": 50.0, "T1": 500.0, "vacant": 0.0, "K": 0.0, "axes": False, "sweeps": 2},
        # a step of the solid-solution field ramp (half the sites vacant): new field, sweeps, polarisation
        {"name": "ramp_rc4", "kind": "ramp", "X": 128, "Y": 128, "Z": 128, "rc": 4, "replicas": 4, "T0": 300.0,
         "vacant": 0.5, "E": -0.05, "sweeps": 2},
        # local field and parameter derivatives of 32 replicas in one call
        {"name": "adjoint_batch", "kind": "adjoint", "X": 48, "Y": 48, "Z": 48, "rc": 3, "replicas": 32,
         "vacant": 0.0, "K": 0.0},
        # energy and its gradients through torch.autograd, lengths of a solid solution
        {"name": "autograd48", "kind": "autograd", "X": 48, "Y": 48, "Z": 48, "rc": 3, "vacant": 0.25, "K": 0.0},
        # what is written after a megastep: radial order, potential, field map, recombination line
        {"name": "observables64", "kind": "observables", "X": 64, "Y": 64, "Z": 64, "vacant": 0.25},
    ]


# ---- sizes ------------------------------------------------------------------

def _offsets(rc, two_d):
    """Integer offsets 0 < |r| <= rc (dz = 0 in 2D)."""
    zc = 0 if two_d else rc
    return [(x, y, z) for x in range(-rc, rc + 1) for y in range(-rc, rc + 1) for z in range(-zc, zc + 1)
            if 0 < x * x + y * y + z * z <= rc * rc]


def _boxes(case):
    """Replica sizes: all alike, or cubes growing by `spread` sites in all."""
    n, s = case.get("replicas", 1), case.get("spread", 0)
    if not s:
        return [(case["X"], case["Y"], case["Z"])] * n
    return [(case["X"] + s * k // (n - 1),) * 3 for k in range(n)]


def _sites(case):
    return sum(x * y * z for x, y, z in _boxes(case))


def _flops_per_site(rc, two_d):
    """19 per neighbour and 3 per nearest neighbour: the local field of one site."""
    return 19 * len(_offsets(rc, two_d)) + 3 * (4 if two_d else 6)


def work(case):
    kind, two_d = case["kind"], case["Z"] == 1
    N = _sites(case)
    if kind == "observables":
        radial = sum(1 for _ in _offsets(9, False) if sum(v * v for v in _) < RADIAL_BINS) + 1
        pot, field = len(_offsets(POT_CUTOFF, False)), len(_offsets(EFIELD_CUTOFF, False))
        # the radial sum is symmetric in +-r; the potential is formed once for its map and once for the
        # recombination line (two calls)
        return {"bytes": N * (4 * 32 + 2 * 8 + 24), "flops": N * (radial / 2 * 17 + 2 * pot * 7 + field * 16)}
    F = _flops_per_site(case["rc"], two_d)
    if kind == "site_energy":
        n = case["n"]
        return {"bytes": n * (4 + 24 + 8) + min(N, n * len(_offsets(case["rc"], two_d))) * 32, "flops": n * (F + 20)}
    if kind in ("adjoint", "autograd"):
        return {"bytes": N * (32 + 24) * (2 if kind == "autograd" else 1), "flops": N * (F + 40)}
    return {"bytes": N * 56.0 * case["sweeps"], "flops": N * (F + 40.0) * case["sweeps"]}


# ---- drawn cases --------------------------------------------------------------

def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _edge(rng, rc, lo, hi):
    """A lattice edge between lo and hi that splits into tiles: any from 4 rc
    on, at DipoleCutOff 5 the multiples of 10 sites."""
    v = max(4 * rc, _log(rng, lo, hi))
    return max(20, v - v % 10) if rc == 5 else v


def draw(rng):
    kind = rng.choice(["sweep", "sweep", "sweep", "sweep", "megastep", "ramp", "site_energy", "adjoint", "autograd",
                       "observables"])
    vacant = rng.choice([0.0, 0.0, 0.25, 0.5])
    K = rng.choice([0.0, 0.0, 0.0, 0.5])
    while True:
        two_d = rng.random() < 0.35 and kind not in ("ramp", "observables")
        rc = rng.choice([1, 2, 3, 3, 3, 3, 4, 4, 5])
        if two_d:
            X, Y, Z = _edge(rng, rc, 20, 1024), _edge(rng, rc, 20, 1024), 1
        else:
            X = _edge(rng, rc, 12, 128)
            Y, Z = (X, X) if rng.random() < 0.5 else (_edge(rng, rc, 12, 96), _edge(rng, rc, 12, 96))
        case = {"kind": kind, "X": X, "Y": Y, "Z": Z}
        if kind == "observables":
            case |= {"X": min(X, 64), "Y": min(Y, 64), "Z": min(Z, 64), "vacant": vacant}
        elif kind == "site_energy":
            case |= {"rc": rc, "n": _log(rng, 1, 200000)}
        elif kind == "adjoint":
            case |= {"rc": rc, "replicas": _log(rng, 1, 64), "vacant": vacant, "K": K}
        elif kind == "autograd":
            case |= {"rc": rc, "vacant": vacant, "K": K}
        elif kind == "ramp":
            case |= {"rc": rc, "replicas": _log(rng, 1, 16), "T0": 300.0, "vacant": vacant,
                     "E": round(rng.uniform(-0.1, 0.1), 4), "sweeps": _log(rng, 1, 10)}
        elif kind == "megastep":
            case |= {"rc": rc, "T0": rng.choice([150.0, 300.0, 600.0]), "vacant": vacant, "K": K,
                     "sweeps": _log(rng, 4, 50)}
        else:
            uneven = not two_d and rc <= 4 and rng.random() < 0.25
            if uneven:
                case |= {"X": 4 * rc + 3, "Y": 4 * rc + 3, "Z": 4 * rc + 3}
            case |= {"rc": rc, "replicas": rng.choice([1, 1, _log(rng, 2, 512)]), "spread": 0,
                     "T0": 100.0, "T1": rng.choice([100.0, 300.0, 500.0]), "vacant": vacant, "K": K,
                     "axes": rng.random() < 0.15, "sweeps": _log(rng, 1, 100)}
            if uneven:
                case |= {"replicas": rng.randint(4, 40), "spread": rng.randint(4, 30)}
        if _sites(case) <= MAX_SITES and work(case)["flops"] <= MAX_FLOPS:
            return case


# ---- inputs --------------------------------------------------------------------

def _lattice(N, vacant, gen):
    """(N, 4) unit dipoles uniform on the sphere; a fraction `vacant` of lengths 0, the others 1."""
    p = torch.randn((N, 3), dtype=torch.float64, device=DEVICE, generator=gen)
    lat = torch.empty((N, 4), dtype=torch.float64, device=DEVICE)
    lat[:, :3] = p / p.norm(dim=1, keepdim=True)
    if vacant > 0.0:
        lat[:, 3] = (torch.rand(N, dtype=torch.float64, device=DEVICE, generator=gen) >= vacant).to(torch.float64)
    else:
        lat[:, 3] = 1.0
    return lat


def _lattices(case, seed):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    return [_lattice(x * y * z, case.get("vacant", 0.0), gen) for x, y, z in _boxes(case)]


def _moves(case, seed):
    """Trial moves: sites and unit proposals in host memory."""
    rng = np.random.default_rng(seed)
    v = rng.normal(size=(case["n"], 3))
    v /= np.linalg.norm(v, axis=1)[:, None]
    return rng.integers(0, _sites(case), case["n"]).astype(np.int32), v


class _DeviceArray:
    """A context's lattice buffer, for torch to view in place.  torch holds
    this object as long as a tensor views it, and it holds the context: the
    buffer outlives every view."""

    def __init__(self, ctx, rows):
        self.ctx = ctx
        ptr = ctypes.c_void_p()
        st = lib().sn_lattice_device_ptr(ctx._h, 0, ctypes.byref(ptr))
        if st != 0:
            raise RuntimeError(f"sn_lattice_device_ptr: {st}")
        self.__cuda_array_interface__ = {"shape": (rows, 4), "typestr": "<f8", "data": (ptr.value, False),
                                         "version": 2}


def _replicas(case, seed):
    boxes = _boxes(case)
    R = len(boxes)
    T0, T1 = case.get("T0", 300.0), case.get("T1", case.get("T0", 300.0))
    return [sn.ReplicaParams(x, y, z, DipoleCutOff=case["rc"], CageStrain=1.0, K=case.get("K", 0.0),
                             Efield=(0.0, 0.0, case.get("E", 0.0)), ConstrainToX=case.get("axes", False),
                             T=T0 + (T1 - T0) * k / max(1, R - 1), seed=seed * 1000003 + k)
            for k, (x, y, z) in enumerate(boxes)]


_J, _E, _S = 0.9, (0.05, -0.01, 0.02), 1.1   # the autograd cases' parameters


def prepare(case, seed):
    kind = case["kind"]
    lats = _lattices(case, seed)
    state = {"case": case}
    if kind == "autograd":
        from starrynight_amd.autograd import EnergyModel
        rp = sn.ReplicaParams(case["X"], case["Y"], case["Z"], DipoleCutOff=case["rc"], K=case["K"])
        state["model"] = EnergyModel(rp)
        state["p"] = lats[0][:, :3].contiguous().requires_grad_(True)
        state["lengths"] = lats[0][:, 3].contiguous()
        state["J"], state["E"], state["s"] = (
            torch.tensor(v, dtype=torch.float64, device=DEVICE, requires_grad=True) for v in (_J, _E, _S))
        return state
    if kind == "observables":
        case = case | {"rc": 3}
    reps = _replicas(case, seed)
    ctx = state["ctx"] = sn.StarryNight(reps)
    for r, lat in enumerate(lats):
        ctx.set_lattice_device(lat, r)
    rows = _sites(case)
    if kind in ("sweep", "ramp", "megastep"):
        state["lattice"] = torch.as_tensor(_DeviceArray(ctx, rows), device=DEVICE)
    if kind == "site_energy":
        state["sites"], state["props"] = _moves(case, seed)
    if kind == "adjoint":
        state["grad"] = torch.empty((rows, 3), dtype=torch.float64, device=DEVICE)
    return state


# ---- one pass ------------------------------------------------------------------

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "autograd":
        from starrynight_amd.autograd import lattice_energy
        leaves = [state[k] for k in ("p", "J", "E", "s")]
        for t in leaves:
            t.grad = None
        e = lattice_energy(state["p"], state["lengths"], state["J"], state["E"], state["s"], state["model"])
        e.backward()
        return [e.detach()] + [t.grad for t in leaves]
    ctx = state["ctx"]
    if kind == "site_energy":
        if case["n"] == 1:
            s = int(state["sites"][0])
            Y, Z = case["Y"], case["Z"]
            return ctx.site_energy(s // (Y * Z), s // Z % Y, s % Z, state["props"][0])
        return ctx.site_energy_batch(state["sites"], state["props"])
    if kind == "adjoint":
        dparams, energy = ctx.gradient_all_device(state["grad"])
        return {"grad": state["grad"], "dparams": dparams, "energy": energy}
    if kind == "observables":
        fe, afe, count = ctx.radial_order()
        return {"fe": fe, "afe": afe, "count": count, "potential": ctx.dipole_potential(),
                "efield": ctx.dipole_efield(EFIELD_CUTOFF), "recombination": ctx.recombination()}
    R = case.get("replicas", 1)
    if kind == "ramp":
        for r in range(R):
            ctx.set_params(r, case["T0"], (0.0, 0.0, case["E"]), 1.0)
        ctx.MC_sweeps(case["sweeps"], sync=False)
        return {"moment": [ctx.moment(r) for r in range(R)], "lattice": state["lattice"]}
    ctx.MC_sweeps(case["sweeps"])
    if kind == "megastep":
        energy, parts = ctx.energy()
        return {"moment": ctx.moment(), "energy": energy, "parts": parts, "lattice": state["lattice"]}
    if R == 1:
        n = ctx.counters()
        return {"accept": n["accept"], "reject": n["reject"], "lattice": state["lattice"]}
    return {"lattice": state["lattice"]}


# ---- the same in plain torch, 64 bits --------------------------------------------

def _shift(t, o):
    """t[x + o] with periodic wrap, over the first three axes."""
    return torch.roll(t, (-o[0], -o[1], -o[2]), (0, 1, 2))


def _local_fields(lat, rc):
    """h = sum_r L_j (p_j - 3 n (n.p_j)) / d^3 and g = sum_{|r|=1} p_j of an (X, Y, Z, 4) lattice."""
    p, m = lat[..., :3], lat[..., :3] * lat[..., 3:]
    h, g = torch.zeros_like(p), torch.zeros_like(p)
    for o in _offsets(rc, lat.shape[2] == 1):
        d2 = sum(v * v for v in o)
        n = torch.tensor(o, dtype=torch.float64, device=lat.device) / math.sqrt(d2)
        q = _shift(m, o)
        h += (q - 3.0 * n * (q * n).sum(-1, keepdim=True)) / (d2 * math.sqrt(d2))
        if d2 == 1:
            g += _shift(p, o)
    return h, g


def _adjoint(lat, rc, J, E, K):
    """Energy, dE/dp and (dE/dJ, dE/dE, dE/ds, dE/dK) of one lattice (lengths as given, s = 1)."""
    h, g = _local_fields(lat, rc)
    p, L = lat[..., :3], lat[..., 3:]
    E = torch.tensor(E, dtype=torch.float64, device=lat.device)
    dd, pg, M = (L * p * h).sum(), (p * g).sum(), p.sum((0, 1, 2))
    grad = L * h - J * g + E
    ak = 0.0
    if K > 0.0:
        grad[..., :2] -= K * torch.sign(p[..., :2])
        ak = float(p[..., :2].abs().sum())
    energy = 0.5 * dd - 0.5 * J * pg + (M * E).sum() - K * ak
    dpar = [float(-0.5 * pg), *[float(v) for v in M], float(dd), -ak]
    return float(energy), grad.reshape(-1, 3), dpar


def _observables(lat):
    X, Y, Z, _ = lat.shape
    N = X * Y * Z
    p, m = lat[..., :3], lat[..., :3] * lat[..., 3:]
    fe, afe = np.zeros(RADIAL_BINS), np.zeros(RADIAL_BINS)
    count = np.zeros(RADIAL_BINS, np.int64)
    pot, field = torch.zeros_like(lat[..., 0]), torch.zeros_like(p)
    for o in [(0, 0, 0)] + _offsets(9, False):
        d2 = sum(v * v for v in o)
        d = math.sqrt(d2)
        r = torch.tensor(o, dtype=torch.float64, device=lat.device)
        n = r / d if d2 else r
        q = _shift(p, o)
        nq = (q * n).sum(-1)
        if d2 < RADIAL_BINS:
            f = float((p * q).sum())
            fe[d2] += f
            afe[d2] += f - 3.0 * float(((p * n).sum(-1) * nq).sum())
            count[d2] += N
        if 0 < d2 <= EFIELD_CUTOFF ** 2:
            field += (3.0 * n * nq[..., None] - q) / (d2 * d)
        if 0 < d2 <= POT_CUTOFF ** 2:
            pot += (_shift(m, o) * r).sum(-1) / (d2 * d)
    cnt = np.maximum(count, 1)
    x = pot * (0.165 / 5) / 0.025    # the recombination line's potential over kT
    eh, ee = torch.exp(-x).sum(), torch.exp(x).sum()
    fe_, fh_ = 1.0 / (torch.exp(x) + 1.0), 1.0 / (torch.exp(-x) + 1.0)
    rec = [eh, ee, fe_.sum(), fh_.sum(), N * N / (eh * ee), N * (fe_ * fh_).sum() / (fe_.sum() * fh_.sum()), 1.0, 1.0]
    return {"fe": fe / cnt, "afe": afe / cnt, "count": None, "potential": pot.reshape(-1).cpu().numpy(),
            "efield": (field - p / 3.0).reshape(-1, 3).cpu().numpy(), "recombination": np.array([float(v) for v in rec])}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("sweep", "ramp", "megastep"):
        return None    # a lattice of drawn proposals, chosen by decisions: nothing is summed into it
    lats = [lat.reshape(*box, 4) for lat, box in zip(_lattices(case, seed), _boxes(case))]
    if kind == "site_energy":
        # the replicas of these cases have CageStrain 1 and no field
        sites, props = _moves(case, seed)
        h, g = _local_fields(lats[0], case["rc"])
        i = torch.from_numpy(sites).to(DEVICE).long()
        flat = lats[0].reshape(-1, 4)[i]
        d = torch.from_numpy(props).to(DEVICE) - flat[:, :3]
        dE = flat[:, 3] * (d * h.reshape(-1, 3)[i]).sum(1) - (d * g.reshape(-1, 3)[i]).sum(1)
        return float(dE[0]) if case["n"] == 1 else dE.cpu().numpy()
    if kind == "autograd":
        lat = lats[0].clone()
        lat[..., 3] *= _S
        e, g, dp = _adjoint(lat, case["rc"], _J, _E, case["K"])
        t = [torch.tensor(v, dtype=torch.float64) for v in (e, dp[0], dp[1:4], dp[4] / _S)]
        return [t[0], g, t[1], t[2], t[3]]
    if kind == "adjoint":
        res = [_adjoint(lat, case["rc"], 1.0, (0.0, 0.0, 0.0), case["K"]) for lat in lats]
        return {"grad": torch.cat([r[1] for r in res]), "dparams": np.array([r[2] for r in res]),
                "energy": np.array([r[0] for r in res])}
    return _observables(lats[0])
