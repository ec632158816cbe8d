"""Performance cases: the work that a user of the package has it do, through its public entry points.

Every case is liquid water at 1 g/cm^3 under the package's own networks:
  teacher  52 symmetry functions per element, cutoff 12 Bohr, MLP 52-64-64-1
  student  34 symmetry functions per element, cutoff 8 Bohr, MLP 34-16-16-1 (packaged weights)
and one of five kinds:
  md       System + MDSimulator.run: a stretch of molecular dynamics from a stored state
  forces   energy and forces of a structure (one call, or torch.autograd through the energy)
  acsf     descriptor values, or their self-Jacobian, of selected atoms
  train    loss gradient of a batch of labelled structures (StudentTrainer)
  kalman   KalmanFilter.fit over a small labelled data set

Results of the mixed precision mode are handed on as FP32, the precision
their descriptors are computed in (a trajectory frame, an FP32 optimiser's
gradient); those of the FP64 mode stay FP64.

``exact`` evaluates the same definitions with plain torch in FP64.
"""

from __future__ import annotations

import json
import math
import random
from pathlib import Path

import numpy as np
import torch

from pantea_amd import bench_models, kalman, potential, simulation, student, water
from pantea_amd.atoms import Structure
from pantea_amd.potential import NNPSettings
from pantea_amd.units import units

ASSETS = Path(student.ASSET_DIR)
ELEMENTS = ("H", "O")                       # atom types 1, 2
PAIRS = (("H", "H"), ("H", "O"), ("O", "O"))
RADIAL_ETAS = [float(x) for x in np.geomspace(0.001, 0.5, 8)]
TEACHER_CELLS = [(eta, zeta, lam) for eta in (0.001, 0.01, 0.05) for zeta in (1.0, 4.0) for lam in (1.0, -1.0)]
MASS = {"H": 1.008, "O": 15.999}            # atomic mass units
DT = 0.5 * units.FROM_FEMTO_SECOND
T0 = 300.0
FORCE_RMS = 0.16                            # Ha/Bohr: forces of the data the packaged student was trained on
FIT_MOLECULES = 1000                        # box that the teacher's scaler is fitted on
W_ENERGY, W_FORCE = 1.0, 10.0               # loss weights of the student trainer


def listed():
    return [
        # data generation: a short teacher run on a training box (the smallest benchmark box, rc + 1 Bohr lists)
        {"name": "md_teacher_384", "kind": "md", "net": "teacher", "precision": "mixed", "molecules": 128,
         "steps": 3, "skin": 1.0},
        # the default precision of a System: reference-quality dynamics of a medium box
        {"name": "md_teacher_fp64_12k", "kind": "md", "net": "teacher", "precision": "float64", "molecules": 4096,
         "steps": 4, "skin": 0.0},
        # production dynamics: the benchmark's 98,304 atoms
        {"name": "md_teacher_98k", "kind": "md", "net": "teacher", "precision": "mixed", "molecules": 32768,
         "steps": 5, "skin": 0.0},
        # production dynamics driven by the cheaper student
        {"name": "md_student_98k", "kind": "md", "net": "student", "precision": "mixed", "molecules": 32768,
         "steps": 3, "skin": 0.0},
        # one small structure, the reference's own forces: compute_forces as a script calls it first
        {"name": "forces_fp64_96", "kind": "forces", "net": "teacher", "precision": "float64", "molecules": 32,
         "mode": "reference", "cutoff": "tanh", "autograd": False},
        # labels of a training snapshot: FP64 energy and -grad E of an odd-sized box
        {"name": "forces_fp64_1.2k", "kind": "forces", "net": "teacher", "precision": "float64", "molecules": 413,
         "mode": "full", "cutoff": "tanh", "autograd": False},
        # differentiable energy of a medium box: forward, then backward
        {"name": "autograd_mixed_12k", "kind": "forces", "net": "teacher", "precision": "mixed", "molecules": 4001,
         "mode": "full", "cutoff": "tanh", "autograd": True},
        # descriptor values of every O atom of a medium box (data preparation, scaler statistics)
        {"name": "acsf_values_fp32", "kind": "acsf", "net": "teacher", "precision": "float32", "molecules": 4096,
         "atoms": 4096, "grad": False},
        # self-Jacobians of 256 sampled atoms (ranking the symmetry functions by sensitivity)
        {"name": "acsf_grad_fp64", "kind": "acsf", "net": "teacher", "precision": "float64", "molecules": 500,
         "atoms": 256, "grad": True},
        # one optimiser batch of the student's training: 32 uneven boxes of 32 to 512 molecules
        {"name": "train_batch_32", "kind": "train", "precision": "mixed", "structures": 32, "molecules": 512},
        # Kalman filter on a few small boxes: fewer observations than weights, energies and forces
        {"name": "kalman_small", "kind": "kalman", "structures": 6, "molecules": 64, "force_fraction": 0.5},
        # Kalman filter force update of one large box: more observations than weights
        {"name": "kalman_large", "kind": "kalman", "structures": 1, "molecules": 512, "force_fraction": 1.0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("md", "md", "forces", "forces", "acsf", "train", "kalman"))
    if kind == "md":
        precision = rng.choice(("mixed", "mixed", "float64"))
        top = 32768 if precision == "mixed" else 8192
        return {"kind": kind, "net": rng.choice(("teacher", "student")), "precision": precision,
                "molecules": _log_int(rng, 32, top), "steps": rng.randint(1, 3), "skin": rng.choice((0.0, 1.0))}
    if kind == "forces":
        net = rng.choice(("teacher", "teacher", "student"))
        return {"kind": kind, "net": net, "precision": rng.choice(("mixed", "float64")),
                "molecules": _log_int(rng, 20, 16384), "mode": rng.choice(("full", "full", "reference")),
                "cutoff": rng.choice(("tanh", "tanh", "cos")) if net == "teacher" else "tanh", "autograd": False}
    if kind == "acsf":
        molecules = _log_int(rng, 32, 8192)
        if rng.random() < 0.5:
            return {"kind": kind, "net": rng.choice(("teacher", "student")), "precision": rng.choice(("float32", "float64")),
                    "molecules": molecules, "atoms": rng.randint(1, molecules), "grad": False}
        return {"kind": kind, "net": rng.choice(("teacher", "student")), "precision": "float64", "molecules": molecules,
                "atoms": min(molecules, _log_int(rng, 1, 512)), "grad": True}
    if kind == "train":
        return {"kind": kind, "precision": rng.choice(("mixed", "mixed", "float64")), "structures": rng.randint(1, 32),
                "molecules": _log_int(rng, 40, 512)}
    return {"kind": kind, "structures": rng.randint(1, 4), "molecules": _log_int(rng, 8, 320),
            "force_fraction": rng.choice((0.1, 0.5, 1.0))}


# ---- inputs ---------------------------------------------------------------------------------------------------

def _water(molecules, rng):
    """Positions (O, H, H per molecule) and box length of a water box: molecules on the jittered
    sites of a near-cubic lattice (O-O distances above 4 Bohr), random orientations."""
    L = water.box_for_density(molecules)
    k = int(math.floor(round(molecules ** (1.0 / 3.0), 9)))
    grid = next(g for g in ((k, k, k), (k, k, k + 1), (k, k + 1, k + 1), (k + 1, k + 1, k + 1)) if math.prod(g) >= molecules)
    sites = np.sort(rng.permutation(math.prod(grid))[:molecules])
    sites = np.stack([sites % grid[0], sites // grid[0] % grid[1], sites // (grid[0] * grid[1])], axis=1)
    O = (sites + 0.5 + rng.uniform(-0.06, 0.06, (molecules, 3))) * (L / np.asarray(grid))
    u = rng.normal(size=(molecules, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    v = rng.normal(size=(molecules, 3))
    v -= np.sum(v * u, axis=1, keepdims=True) * u
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    c, s = 1.81 * math.cos(math.radians(52.25)), 1.81 * math.sin(math.radians(52.25))
    pos = np.stack([O, O + c * u + s * v, O + c * u - s * v], axis=1).reshape(-1, 3)
    pos = np.mod(pos + rng.normal(scale=0.05, size=pos.shape), L)
    pos[pos >= L] = 0.0
    return pos, L


def _structure(pos, L, **more):
    return Structure.from_dict({"positions": pos, "elements": ["O", "H", "H"] * (len(pos) // 3),
                                "lattice": np.diag([L, L, L]), **more})


def _masses(molecules):
    m = np.array([MASS["O"], MASS["H"], MASS["H"]] * molecules) * units.FROM_ATOMIC_MASS
    return m.reshape(-1, 1)


def _velocities(molecules, rng):
    """Maxwell-Boltzmann velocities at T0, no net momentum."""
    m = _masses(molecules)
    v = rng.normal(size=(3 * molecules, 3)) * np.sqrt(units.BOLTZMANN_CONSTANT * T0 / m)
    return v - np.sum(m * v, axis=0) / np.sum(m)


def _teacher_weights(rng):
    """Random weights whose forces have the size of liquid water's (about 0.02 Ha/Bohr rms) and whose
    energies do not cancel (a constant per atom, as fitted networks carry in their last bias)."""
    out = {}
    for e in ELEMENTS:
        layers, fan = {}, 52
        for i, w in enumerate((64, 64, 1)):
            last = w == 1
            layers[f"layers_{2 * i}"] = {"kernel": rng.normal(0.0, (0.03 if last else 1.0) / math.sqrt(fan), (fan, w)),
                                         "bias": np.full(w, 0.3 if last else 0.0)}
            fan = w
        out[e] = layers
    return out


def _rngs(seed):
    """Generators of the network (always the same one), of the inputs and of the labels."""
    return [np.random.default_rng([s, k]) for k, s in enumerate((30, int(seed), int(seed)))]


def _potential(case, seed):
    if case.get("net", "student") == "student":
        return bench_models.water_student(ASSETS, precision="mixed")
    rng = _rngs(seed)[0]
    pot = bench_models.make_nnp(lambda e: bench_models.teacher_acsf(e, cutoff=case.get("cutoff", "tanh")), (64, 64), 2023)
    pot.set_model_params(_teacher_weights(rng))
    pot.fit_scaler([_structure(*_water(FIT_MOLECULES, rng))])
    return pot


def _labelled(case, seed):
    """The labelled boxes of a data set: (positions, box, energy, forces)."""
    _, rng, lab = _rngs(seed)
    if case["kind"] == "train":
        sizes = rng.integers(32, case["molecules"] + 1, size=case["structures"])
    else:
        sizes = rng.integers(max(2, case["molecules"] // 2), case["molecules"] + 1, size=case["structures"])
        sizes[0] = case["molecules"]
    out = []
    for nm in sizes:
        pos, L = _water(int(nm), rng)
        out.append((pos, L, float(3 * nm * (0.3 + 0.02 * lab.normal())), lab.normal(scale=FORCE_RMS, size=pos.shape)))
    return out


def _settings(case):
    return NNPSettings(elements=list(ELEMENTS), global_nodes_short=[16, 16], global_activation_short=["tanh", "tanh", "identity"],
                       symfunction_short=[], updater_type="kalman_filter", epochs=1, random_seed=2023,
                       short_force_fraction=case["force_fraction"])


def _centres(case, seed):
    """Selected O atoms (input indices 0, 3, 6, ...), ascending."""
    rng = np.random.default_rng([int(seed), 7])
    return 3 * np.sort(rng.permutation(case["molecules"])[:case["atoms"]])


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    rng = _rngs(seed)[1]
    if kind == "md":
        nm = case["molecules"]
        s = _structure(*_water(nm, rng))
        state.update(pot=_potential(case, seed), structure=s,
                     velocities=torch.as_tensor(_velocities(nm, rng), device=s.device),
                     masses=torch.as_tensor(_masses(nm), device=s.device))
    elif kind == "forces":
        state.update(pot=_potential(case, seed), structure=_structure(*_water(case["molecules"], rng)))
    elif kind == "acsf":
        state.update(acsf=_potential(case, seed).descriptors["O"], structure=_structure(*_water(case["molecules"], rng)),
                     centres=_centres(case, seed))
    elif kind == "train":
        tr = student.StudentTrainer(_potential(case, seed), precision=case["precision"], w_energy=W_ENERGY, w_force=W_FORCE)
        for pos, L, e, f in _labelled(case, seed):
            s = _structure(pos, L)
            tr.add(s, e, torch.as_tensor(f, device=s.device))
        tr.prepare(fit_scaler=False)
        state.update(trainer=tr, batch=list(range(case["structures"])))
    else:
        pot = _potential(case, seed)
        state.update(pot=pot, params=pot.models_params, settings=_settings(case),
                     data=[_structure(pos, L, forces=f, total_energy=[e]) for pos, L, e, f in _labelled(case, seed)])
    return state


# ---- one pass -------------------------------------------------------------------------------------------------

def _handed_on(precision, x):
    return x if precision == "float64" else x.float()


def run(state):
    case = state["case"]
    kind, precision = case["kind"], case.get("precision")
    if kind == "md":
        sysm = simulation.System(state["pot"], state["structure"].copy(), state["velocities"], state["masses"],
                                 force_mode="full", precision=precision, skin=case["skin"])
        md = simulation.MDSimulator(DT, simulation.BrendsenThermostat(T0, DT), integrator="physical")
        md.run(sysm, case["steps"])
        return {"positions": _handed_on(precision, sysm.positions), "velocities": _handed_on(precision, sysm.velocities),
                "forces": _handed_on(precision, sysm.forces)}
    if kind == "forces":
        pot, s = state["pot"], state["structure"]
        if case["autograd"]:
            x = s.positions.detach().requires_grad_(True)
            e = potential.energy(pot, s, x, precision=precision)
            (g,) = torch.autograd.grad(e, x)
            return {"energy": _handed_on(precision, e.detach()), "forces": _handed_on(precision, -g)}
        e, f = pot.energy_and_forces(s, mode=case["mode"], precision=precision)
        return {"energy": _handed_on(precision, e), "forces": _handed_on(precision, f)}
    if kind == "acsf":
        call = state["acsf"].grad if case["grad"] else state["acsf"]
        return call(state["structure"], atom_index=state["centres"], precision=precision)
    if kind == "train":
        loss, grad = state["trainer"].gradient(state["batch"])
        return {"loss": _handed_on(precision, loss), "grad": {e: _handed_on(precision, g) for e, g in grad.items()}}
    state["pot"].set_model_params(state["params"])
    kf = kalman.KalmanFilter.from_settings(state["pot"], state["settings"])
    history = kf.fit(state["data"], kalman.TrainingParams.from_runner(state["settings"]))
    return {"weights": kf.W, "covariance": kf.P, "loss_energy": history["loss_energy"], "loss_force": history["loss_force"]}


# ---- what one pass cannot do without --------------------------------------------------------------------------

def _descriptor_work(net, n):
    """Neighbours and live pairs of n atoms, and the operations of one descriptor forward and adjoint
    (add, multiply, compare 1, FMA 2, transcendental 1), as bench.py counts them."""
    nb, trip, g2, g3, n_eta = (107.0, 2630.0, 8, 12, 3) if net == "teacher" else (32.0, 230.0, 8, 6, 3)
    if n - 1 < nb:
        trip *= ((n - 1) / nb) ** 2
        nb = n - 1
    fwd = (15 + 6 * g2) * nb + (26 + 5 * g3) * trip
    adj = (45 + 11 * g2) * nb + (110 + 18 * n_eta) * trip
    return nb * n, fwd * n, adj * n


def work(case):
    kind = case["kind"]
    net = case.get("net", "student")
    wide, word = (52, 64) if net == "teacher" else (34, 16), 8 if case.get("precision") == "float64" else 4
    mlp = 4.0 * (wide[0] * wide[1] + wide[1] ** 2)     # forward and input gradient, per atom
    n = 3 * case["molecules"]
    if kind == "train" or kind == "kalman":
        n = 3 * case["structures"] * (case["molecules"] + (32 if kind == "train" else case["molecules"] // 2)) // 2
    edges, fwd, adj = _descriptor_work(net, n)
    if kind == "md":
        k = case["steps"]
        return {"bytes": k * (n * 200.0 + edges * 4), "flops": (k + 1) * (fwd + adj + n * mlp)}
    if kind == "forces":
        return {"bytes": n * 24.0 * 2 + edges * 4, "flops": fwd + adj + n * mlp}
    if kind == "acsf":
        c = case["atoms"]
        out = wide[0] * word * (3 if case["grad"] else 1)
        return {"bytes": n * 28.0 + c * out, "flops": (6.0 if case["grad"] else 1.0) * fwd / n * c}
    if kind == "train":
        return {"bytes": n * (wide[0] * word + 60.0) + edges * 8, "flops": adj + 2 * fwd + n * 5 * mlp}
    n_w = 1698.0
    total = {"bytes": 0.0, "flops": fwd + adj + 6 * fwd}
    for _ in range(case["structures"]):
        m = 3.0 * n / case["structures"]
        force = 2 * n_w ** 2 * m + 8.0 / 3.0 * n_w ** 3 if m > n_w else 4 * n_w ** 2 * m + 4 * m ** 2 * n_w + m ** 3 / 3
        total["flops"] += case["force_fraction"] * force + (1 - case["force_fraction"]) * 4 * n_w ** 2
        total["bytes"] += 2 * 8 * n_w ** 2 + case["force_fraction"] * 8 * n_w * m
    return total


# ---- the same in plain torch, FP64 ----------------------------------------------------------------------------

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _t(x):
    return torch.as_tensor(x, dtype=torch.float64, device=_device())


def _cutoff(kind, r, rc):
    if kind == "cos":
        return 0.5 * (torch.cos(math.pi * r / rc) + 1.0) * (r < rc)
    pre = ((math.e + 1 / math.e) / (math.e - 1 / math.e)) ** 3
    return pre * torch.tanh(1.0 - r / rc) ** 3 * (r < rc)


def _single_shift(d, L):
    d = torch.where(d > 0.5 * L, d - L, d)
    return torch.where(d < -0.5 * L, d + L, d)


def _packed(mask):
    """Column indices of the true entries of each row of a 2-D mask, padded: (index, valid)."""
    row, col = mask.nonzero(as_tuple=True)
    count = mask.sum(1)
    slot = torch.arange(row.numel(), device=mask.device) - (torch.cumsum(count, 0) - count)[row]
    idx = torch.zeros((mask.shape[0], max(1, int(count.max()))), dtype=torch.int64, device=mask.device)
    idx[row, slot] = col
    return idx, torch.arange(idx.shape[1], device=mask.device)[None, :] < count[:, None]


class _Net:
    """Symmetry functions, scaler and MLP of every element."""

    def __init__(self, case, seed):
        self.cut = case.get("cutoff", "tanh")
        if case.get("net", "student") == "teacher":
            rng = _rngs(seed)[0]
            self.rc = 12.0
            self.cells = {e: {p: TEACHER_CELLS for p in PAIRS} for e in ELEMENTS}
            params = _teacher_weights(rng)
            pos, L = _water(FIT_MOLECULES, rng)
            x, t = _t(pos), _types(len(pos))
            self.lo, self.span = {}, {}
            for e, z in (("H", 1), ("O", 2)):
                idx, ok, shift = _neighbours(x, L, self.rc, torch.nonzero(t == z)[:, 0])
                R = x[t == z][:, None] - x[idx] + shift
                G = self.descriptors(e, R, t[idx], ok, L)
                self.lo[e], self.span[e] = G.min(0).values, G.max(0).values - G.min(0).values
        else:
            self.cut = "tanh"
            spec = json.loads((ASSETS / "student.json").read_text())
            self.rc = float(spec["r_cutoff"])
            self.cells = {e: {p: [tuple(c) for c in spec["g3"][e]["-".join(p)]] for p in PAIRS} for e in ELEMENTS}
            params, self.lo, self.span = {}, {}, {}
            for e, z in (("H", 1), ("O", 8)):
                d = json.loads((ASSETS / f"scaling.{z:03d}.json").read_text())
                self.lo[e], self.span[e] = _t(d["minval"]), _t(d["maxval"]) - _t(d["minval"])
                with np.load(ASSETS / f"weights.{z:03d}.npz", allow_pickle=False) as f:
                    params[e] = {}
                    for k in f.files:
                        layer, p = k.split("/")
                        params[e].setdefault(layer, {})[p] = np.asarray(f[k], np.float64)
        self.params = {e: [_t(p[f"layers_{2 * i}"][k]) for i in range(3) for k in ("kernel", "bias")]
                       for e, p in params.items()}

    def descriptors(self, e, R, tj, ok, L):
        """(centres, functions) from R_ij = r_i - r_j (padded with ok = False)."""
        r2 = torch.where(ok, (R * R).sum(-1), 1.0)
        r = torch.sqrt(r2)
        f = _cutoff(self.cut, r, self.rc) * ok
        cols = [(torch.exp(-eta * r2) * f * (tj == z)).sum(1) for z in (1, 2) for eta in RADIAL_ETAS]
        with torch.no_grad():
            D = _single_shift(R[:, :, None] - R[:, None], L)
            d2 = (D * D).sum(-1)
            m = R.shape[1]
            live = ok[:, :, None] & ok[:, None] & (d2 < self.rc ** 2) & (d2 > 0)
            live &= torch.ones((m, m), dtype=torch.bool, device=R.device).triu(1)
            D = None
        for (a, b) in PAIRS:
            za, zb = ELEMENTS.index(a) + 1, ELEMENTS.index(b) + 1
            ja, kb = (tj == za)[:, :, None], (tj == zb)[:, None]
            sel = live & ((ja & kb) if za == zb else ((ja & kb) | ((tj == zb)[:, :, None] & (tj == za)[:, None])))
            idx, has = _packed(sel.reshape(sel.shape[0], -1))
            j, k = idx // m, idx % m
            Rj = torch.gather(R, 1, j[..., None].expand(-1, -1, 3))
            Rk = torch.gather(R, 1, k[..., None].expand(-1, -1, 3))
            with torch.no_grad():
                shift = _single_shift(Rj - Rk, L) - (Rj - Rk)
            q2 = torch.where(has, ((Rj - Rk + shift) ** 2).sum(-1), 1.0)
            S = torch.gather(r2, 1, j) + torch.gather(r2, 1, k) + q2
            F = torch.gather(f, 1, j) * torch.gather(f, 1, k) * _cutoff(self.cut, torch.sqrt(q2), self.rc) * has
            c = (Rj * Rk).sum(-1) / (torch.gather(r, 1, j) * torch.gather(r, 1, k))
            rad = {eta: torch.exp(-eta * S) * F for eta in {x[0] for x in self.cells[e][(a, b)]}}
            ang = {(z, l): 2.0 ** (1.0 - z) * (1.0 + l * c) ** int(z) for z, l in {x[1:] for x in self.cells[e][(a, b)]}}
            cols += [(rad[eta] * ang[(z, l)]).sum(1) for eta, z, l in self.cells[e][(a, b)]]
        return torch.stack(cols, dim=1)

    def mlp(self, e, x, params=None):
        W0, b0, W1, b1, W2, b2 = params or self.params[e]
        return (torch.tanh(torch.tanh(x @ W0 + b0) @ W1 + b1) @ W2 + b2)[..., 0]

    def scaled(self, e, G):
        return (G - self.lo[e]) / self.span[e]


def _types(n):
    return torch.tensor([2, 1, 1], device=_device()).repeat(n // 3)


def _neighbours(x, L, rc, centres):
    d = x[centres][:, None] - x[None]
    d = _single_shift(d, L)
    r2 = (d * d).sum(-1)
    idx, ok = _packed((r2 <= rc * rc) & (r2 > 0))
    raw = x[centres][:, None] - x[idx]
    return idx, ok, _single_shift(raw, L) - raw


def _energy_forces(net, x, L, full=True):
    """Total energy and forces, in chunks of centres of one element."""
    t = _types(x.shape[0])
    E, F = 0.0, torch.zeros_like(x)
    for e, z in (("H", 1), ("O", 2)):
        all_c = torch.nonzero(t == z)[:, 0]
        for c in torch.split(all_c, 1024 if x.shape[0] < 20000 else 512):
            idx, ok, shift = _neighbours(x, L, net.rc, c)
            R = (x[c][:, None] - x[idx] + shift).requires_grad_(True)
            en = net.mlp(e, net.scaled(e, net.descriptors(e, R, t[idx], ok, L))).sum()
            (g,) = torch.autograd.grad(en, R)
            g = g * ok[..., None]
            E = E + en.detach()
            F[c] -= g.sum(1)
            if full:
                F.index_add_(0, idx.reshape(-1), g.reshape(-1, 3))
    return E, F


def _exact_md(case, seed):
    rng = _rngs(seed)[1]
    pos, L = _water(case["molecules"], rng)
    x, v, m = _t(pos), _t(_velocities(case["molecules"], rng)), _t(_masses(case["molecules"]))
    net = _Net(case, seed)
    f = _energy_forces(net, x, L)[1]
    for _ in range(case["steps"]):
        x = torch.remainder(x + v * DT + 0.5 * (f / m) * DT * DT, L)
        new = _energy_forces(net, x, L)[1]
        v = v + 0.5 * (f / m + new / m) * DT
        f = new
        T = (m * v * v).sum() / (3 * x.shape[0] * units.BOLTZMANN_CONSTANT)
        v = v / torch.sqrt(1.0 + (T / T0 - 1.0))
    return {"positions": x, "velocities": v, "forces": f}


def _exact_acsf(case, seed):
    net = _Net(case, seed)
    pos, L = _water(case["molecules"], _rngs(seed)[1])
    x, t = _t(pos), _types(len(pos))
    out = []
    for c in torch.split(torch.as_tensor(_centres(case, seed), device=x.device), 512):
        idx, ok, shift = _neighbours(x, L, net.rc, c)
        R = (x[c][:, None] - x[idx] + shift).requires_grad_(case["grad"])
        G = net.descriptors("O", R, t[idx], ok, L)
        if case["grad"]:
            cols = [torch.autograd.grad(G[:, q].sum(), R, retain_graph=True)[0] for q in range(G.shape[1])]
            G = torch.stack([(g * ok[..., None]).sum(1) for g in cols], dim=1)
        out.append(G.detach())
    return torch.cat(out)


def _exact_train(case, seed):
    net = _Net(case, seed)
    loss = torch.zeros(2, dtype=torch.float64, device=_device())
    grad = {e: torch.zeros(sum(p.numel() for p in net.params[e]), dtype=torch.float64, device=_device()) for e in ELEMENTS}
    leaves = {e: [p.clone().requires_grad_(True) for p in net.params[e]] for e in ELEMENTS}
    flat = [p for e in ELEMENTS for p in leaves[e]]
    scale = 1.0 / case["structures"]
    for pos, L, e_ref, f_ref in _labelled(case, seed):
        x, t = _t(pos), _types(len(pos))
        E, F = 0.0, torch.zeros_like(x)
        for e, z in (("H", 1), ("O", 2)):
            c = torch.nonzero(t == z)[:, 0]
            idx, ok, shift = _neighbours(x, L, net.rc, c)
            R = (x[c][:, None] - x[idx] + shift).requires_grad_(True)
            en = net.mlp(e, net.scaled(e, net.descriptors(e, R, t[idx], ok, L)), leaves[e]).sum()
            (g,) = torch.autograd.grad(en, R, create_graph=True)
            g = g * ok[..., None]
            E = E + en
            F = F.index_add(0, c, -g.sum(1)).index_add(0, idx.reshape(-1), g.reshape(-1, 3))
        le = W_ENERGY * scale * ((E - e_ref) / len(pos)) ** 2
        lf = W_FORCE * scale * ((F - _t(f_ref)) ** 2).mean()
        got = torch.autograd.grad(le + lf, flat)
        loss += torch.stack([le.detach(), lf.detach()])
        for k, e in enumerate(ELEMENTS):
            grad[e] += torch.cat([p.reshape(-1) for p in got[6 * k:6 * k + 6]])
    return {"loss": loss, "grad": grad}


def _exact_kalman(case, seed):
    net, st = _Net(case, seed), _settings(case)
    items = []
    for pos, L, e_ref, f_ref in _labelled(case, seed):
        x, t, f_ref = _t(pos), _types(len(pos)), _t(f_ref)
        per = []
        for e, z in (("H", 1), ("O", 2)):
            c = torch.nonzero(t == z)[:, 0]
            idx, ok, shift = _neighbours(x, L, net.rc, c)
            R = (x[c][:, None] - x[idx] + shift).requires_grad_(True)
            G = net.descriptors(e, R, t[idx], ok, L)
            T = torch.stack([(torch.autograd.grad(G[:, q].sum(), R, retain_graph=True)[0] * ok[..., None]).sum(1)
                             for q in range(G.shape[1])], dim=2)          # (centres, 3, functions)
            per.append((e, net.scaled(e, G.detach()), T / net.span[e], f_ref[c]))
        items.append((len(pos), e_ref, per))
    shapes = {e: [p.shape for p in net.params[e]] for e in ELEMENTS}
    sizes = {e: sum(p.numel() for p in net.params[e]) for e in ELEMENTS}

    def unflat(e, w):
        return [p.reshape(s) for p, s in zip(torch.split(w, [math.prod(s) for s in shapes[e]]), shapes[e])]

    W = torch.cat([p.reshape(-1) for e in ELEMENTS for p in net.params[e]])
    n_w = W.numel()
    P = torch.eye(n_w, dtype=torch.float64, device=W.device) / st.kalman_epsilon
    eta, q = st.kalman_eta, st.kalman_q0
    order, shuffle, choice = list(range(len(items))), random.Random(st.random_seed), np.random.RandomState(st.random_seed)
    shuffle.shuffle(order)
    loss, count = [0.0, 0.0], [0, 0]
    for k in order:
        n, e_ref, per = items[k]
        force = choice.rand() < st.short_force_fraction
        part = dict(zip(ELEMENTS, torch.split(W, [sizes[e] for e in ELEMENTS])))
        if force:
            xi, rows = [], []
            for e, X, T, f_ref in per:
                def ydot(w, g, d, e=e):
                    return -torch.func.jvp(lambda y: net.mlp(e, y, unflat(e, w)), (g,), (d,))[1]
                Xr, Tr = X.repeat_interleave(3, 0), T.reshape(-1, T.shape[2])
                xi.append(f_ref.reshape(-1) - torch.func.vmap(ydot, (None, 0, 0))(part[e], Xr, Tr))
                J = torch.func.vmap(torch.func.grad(ydot), (None, 0, 0))(part[e], Xr, Tr)
                full = torch.zeros((J.shape[0], n_w), dtype=torch.float64, device=W.device)
                full[:, (0 if e == "H" else sizes["H"]):][:, :sizes[e]] = J
                rows.append(full)
            xi, H = torch.cat(xi), torch.cat(rows).T
        else:
            w = W.clone().requires_grad_(True)
            ws = dict(zip(ELEMENTS, torch.split(w, [sizes[e] for e in ELEMENTS])))
            E = sum(net.mlp(e, X, unflat(e, ws[e])).sum() for e, X, _, _ in per)
            H = (torch.autograd.grad(E, w)[0] / n)[:, None]
            xi = ((e_ref - E.detach()) / n).reshape(1)
        loss[force] += float((xi * xi).sum())
        count[force] += 1
        if eta < st.kalman_etamax:
            eta *= math.exp(st.kalman_eta)
        X = P @ H
        A = H.T @ X + torch.eye(H.shape[1], dtype=torch.float64, device=W.device) / eta
        K = torch.cholesky_solve(X.T, torch.linalg.cholesky(A)).T
        P = P - K @ X.T + q * torch.eye(n_w, dtype=torch.float64, device=W.device)
        W = W + K @ xi
        if q > st.kalman_qmin:
            q *= math.exp(-st.kalman_qtau)
    return {"weights": W, "covariance": P, "loss_energy": [loss[0] / max(1, count[0])], "loss_force": [loss[1] / max(1, count[1])]}


def exact(case, seed):
    kind = case["kind"]
    if kind == "md":
        return _exact_md(case, seed)
    if kind == "forces":
        pos, L = _water(case["molecules"], _rngs(seed)[1])
        e, f = _energy_forces(_Net(case, seed), _t(pos), L, full=case["mode"] == "full")
        return {"energy": e, "forces": f}
    if kind == "acsf":
        return _exact_acsf(case, seed)
    return _exact_train(case, seed) if kind == "train" else _exact_kalman(case, seed)
