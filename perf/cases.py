"""Measured cases: what a program that uses this package has it compute.

Molecular dynamics comes first, because that is what the package is for: a job
uploads a configuration, runs md_init and a number of steps, and downloads the
state and the thermo record (what the served loop, the ensemble loop and the
`rbmd -j` driver do with every system).  The systems are the package's own
workloads: the charged-LJ salt and rigid 3-site water of salt_config and
water_config, over Verlet lists and over random-batch lists, with random-batch
Ewald or grid Ewald k space, in FP64 and in mixed precision, alone and in
packs.  Sizes run over the ensemble's and the served stream's range, 600 to
300,000 atoms.  Two more kinds are the single-configuration calls of the force
error report: the real-space, random-batch and bonded forces of a
configuration, and the converged Ewald sum.

A pass of a single system starts again from the prepared configuration; a pass
of a pack is a further round of its systems, as the ensemble loop runs them.
Runs are short enough that two roundings of one trajectory stay close.  A mixed-precision run forms its pair terms and its
sines and cosines in 32 bits, so its program keeps the results in 32 bits.
"""
import dataclasses
import math

import numpy as np
import torch

from rbmd_amd import make_salt, make_water, salt_config, water_config
from rbmd_amd.accuracy import converged_kmax
from rbmd_amd.lib import Context, GpuSystem, Pack, rbe_sample_host
from rbmd_amd.serve import log_uniform_atoms, water_rbe_p
from rbmd_amd.system import water_special_lists


def listed():
    md = {"what": "md", "lists": "VERLETLIST", "coulomb": "RBE"}
    return [
        # the smallest systems of the ensemble: a step is a chain of launches
        {"name": "salt_600", **md, "kind": "salt", "atoms": 600, "precision": "fp64", "steps": 100},
        # the 4,000-ion salt workload, the everyday small run
        {"name": "salt_4k", **md, "kind": "salt", "atoms": 4000, "precision": "fp64", "steps": 100},
        # the 30,000-atom water workload, the benchmark's default line
        {"name": "water_30k", **md, "kind": "water", "atoms": 30000, "precision": "fp64", "steps": 100},
        # the same box as a production run in mixed precision
        {"name": "water_30k_mixed", **md, "kind": "water", "atoms": 30000, "precision": "mixed", "steps": 40},
        # the 300,000-atom water workload (P = 2000), the largest system served
        {"name": "water_300k_mixed", **md, "kind": "water", "atoms": 300000, "precision": "mixed", "steps": 40},
        # a large job of the served stream in FP64, an odd number of ion pairs
        {"name": "salt_99k", **md, "kind": "salt", "atoms": 99426, "precision": "fp64", "steps": 20},
        # random-batch lists on the salt with the settings of the reference's
        # salt input: cut-off 5, core 2.5, 50 samples, the erfc step table
        {"name": "salt_4k_rbl", "what": "md", "lists": "RBL", "coulomb": "RBE", "kind": "salt", "atoms": 4000,
         "precision": "fp64", "erfc": "table", "steps": 20},
        # random-batch lists on water with special bonds: core 5, 100 samples
        {"name": "water_30k_rbl", "what": "md", "lists": "RBL", "coulomb": "RBE", "kind": "water", "atoms": 30000,
         "precision": "fp64", "erfc": "analytic", "steps": 10},
        # grid Ewald, as the reference's water input asks for, with the Ewald
        # energy of every thermo row
        {"name": "water_6k_ewald", "what": "md", "lists": "VERLETLIST", "coulomb": "EWALD", "kind": "water",
         "atoms": 6000, "precision": "fp64", "kmax": 5, "steps": 20},
        # a packed ensemble: salt and water systems of mixed sizes, one launch
        # per kernel and kind
        {"name": "ensemble_32_mixed", "what": "pack", "systems": 32, "most": 12000, "precision": "mixed",
         "steps": 20},
        # forces of one configuration: real space, one random k set, bonded
        {"name": "forces_water_12k", "what": "forces", "kind": "water", "atoms": 12000, "precision": "fp64"},
        # the converged Ewald sum that force errors are measured against
        {"name": "ewald_water_12k", "what": "ewald", "kind": "water", "atoms": 12000, "precision": "fp64"},
    ]


def draw(rng):
    def atoms(least, most, multiple):
        n = int(round(math.exp(rng.uniform(math.log(least), math.log(most)))))
        return max(multiple, n - n % multiple)

    kind = rng.choice(["salt", "water"])
    per = 2 if kind == "salt" else 3
    what = rng.choice(["md", "md", "md", "rbl", "grid", "pack", "forces", "ewald"])
    if what == "md":
        n = atoms(600, 150000 if kind == "salt" else 60000, per)
        precision = rng.choice(["fp64", "mixed"])
        return {"what": "md", "lists": "VERLETLIST", "coulomb": "RBE", "kind": kind, "atoms": n,
                "precision": precision, "steps": rng.randint(20, 100 if n < 20000 and precision == "fp64" else 40)}
    if what == "rbl":
        return {"what": "md", "lists": "RBL", "coulomb": "RBE", "kind": kind, "atoms": atoms(2100, 30000, per),
                "precision": "fp64", "erfc": rng.choice(["analytic", "table"]), "steps": rng.randint(5, 10)}
    if what == "grid":
        return {"what": "md", "lists": "VERLETLIST", "coulomb": "EWALD", "kind": kind, "atoms": atoms(600, 12000, per),
                "precision": "fp64", "kmax": rng.randint(3, 6), "steps": rng.randint(10, 30)}
    if what == "pack":
        return {"what": "pack", "systems": rng.randint(8, 30), "most": rng.randint(2000, 12000),
                "precision": rng.choice(["fp64", "mixed"]), "steps": rng.randint(10, 30)}
    if what == "forces":
        return {"what": "forces", "kind": kind, "atoms": atoms(600, 30000, per), "precision": "fp64"}
    return {"what": "ewald", "kind": kind, "atoms": atoms(600, 12000, per), "precision": "fp64"}


def water(atoms, seed):
    """rigid water; above 60,000 atoms 2 x 2 x 2 copies of a box an eighth the
    size, each molecule moved a little, with velocities of its own draw"""
    n_mol = atoms // 3
    if n_mol <= 20000 or n_mol % 8:
        return make_water(n_mol=n_mol, seed=seed)
    b = make_water(n_mol=n_mol // 8, seed=seed)
    rng = np.random.default_rng(seed)
    L = b.box[0]
    cell = np.stack(np.meshgrid([0, 1], [0, 1], [0, 1], indexing="ij"), -1).reshape(8, 1, 3) * L
    move = np.repeat(rng.uniform(-0.02, 0.02, (8, n_mol // 8, 3)), 3, axis=1)
    x = np.mod(((b.x[None] + cell) + move).reshape(-1, 3), 2 * L)
    # a rigid molecule's velocities stay rigid when they are reversed or one velocity is added to all three
    sign = np.repeat(rng.choice([-1.0, 1.0], (8, n_mol // 8, 1)), 3, axis=1)
    kick = np.repeat(rng.normal(0.0, 5e-4, (8, n_mol // 8, 3)), 3, axis=1)
    v = (b.v[None] * sign + kick).reshape(-1, 3)
    mass = np.tile(b.mass, 8)
    v -= (mass[:, None] * v).sum(0) / mass.sum()
    so, si, sw = water_special_lists(n_mol, [0, 0, 0])
    base = 3 * np.arange(n_mol)
    return dataclasses.replace(
        b, hi=np.full(3, 2 * L), x=x, v=v, type=np.tile(b.type, 8), charge=np.tile(b.charge, 8), mass=mass,
        mol_id=np.repeat(np.arange(n_mol, dtype=np.int32), 3), special_offsets=so, special_ids=si, special_weights=sw,
        bond_atoms=np.stack([base, base + 1, base, base + 2], 1).reshape(-1).astype(np.int32),
        bond_k=np.full(2 * n_mol, b.bond_k[0]), bond_r0=np.full(2 * n_mol, b.bond_r0[0]),
        angle_atoms=np.stack([base + 1, base, base + 2], 1).reshape(-1).astype(np.int32),
        angle_k=np.full(n_mol, b.angle_k[0]), angle_theta0=np.full(n_mol, b.angle_theta0[0]))


def system_and_run(case, seed, kind=None, atoms=None):
    kind, atoms = kind or case["kind"], atoms or case["atoms"]
    if kind == "salt":
        s = make_salt(n_ions=atoms, seed=seed)
        r = salt_config(precision=case["precision"], seed=seed)
        rbl = {"cut_off": 5.0, "r_core": 2.5, "neighbor_sample_num": 50, "alpha": 0.1, "temp_ctrl": "BERENDSEN",
               "temperature": [1.0, 1.0, 0.5], "dt": 0.002}
    else:
        s = water(atoms, seed)
        r = water_config(precision=case["precision"], seed=seed, rbe_p=water_rbe_p(atoms))
        rbl = {"r_core": 5.0, "neighbor_sample_num": 100}
    if case.get("lists") == "RBL":
        r = dataclasses.replace(r, neighbor_type="RBL", erfc_mode=case["erfc"], **rbl)
    if case.get("coulomb") == "EWALD":
        r = dataclasses.replace(r, coulomb_type="EWALD", kmax=[case["kmax"]] * 3)
    if case["what"] in ("forces", "ewald"):  # a configuration with bonds and angles off their rest
        s = dataclasses.replace(s, x=s.x + np.random.default_rng(seed).uniform(-0.03, 0.03, s.x.shape))
        s = dataclasses.replace(s, x=np.mod(s.x, s.box))
    return s, r


def ensemble_sizes(case):
    """the case's own, so that every seed has the same work: half salt, half water"""
    rng = np.random.default_rng(case["systems"] * 100003 + case["most"])
    kinds = ["salt"] * (case["systems"] // 2) + ["water"] * (case["systems"] - case["systems"] // 2)
    return [(k, log_uniform_atoms(rng, k, 600, case["most"])) for k in kinds]


def prepare(case, seed):
    seed = int(seed) + 1
    ctx = Context(0)
    state = {"case": case, "ctx": ctx}
    if case["what"] == "pack":
        rng = np.random.default_rng(seed)
        groups = {"salt": [], "water": []}
        for kind, atoms in ensemble_sizes(case):
            g = GpuSystem(ctx, *system_and_run(case, int(rng.integers(1, 2 ** 31)), kind, atoms))
            g.md_init()
            groups[kind].append(g)
        state["packs"] = [Pack(ctx, systems) for systems in groups.values()]
        return state
    s, r = system_and_run(case, seed)
    state.update(system=s, run=r, gpu=GpuSystem(ctx, s, r))
    if case["what"] == "forces":
        state["k"] = rbe_sample_host(r.alpha, s.box, r.rbe_p, seed, 1)
    if case["what"] == "ewald":
        state["kmax"] = converged_kmax(r.alpha, s.box)
    return state


def thermo_arrays(t):
    return {"temperature": np.array([t["temperature"]]), "pressure": np.array([t["pressure"]]),
            "energies": np.array([t["e_lj"], t["e_coul"], t["e_long"], t["e_bond"], t["e_angle"]]),
            "virial": np.array(t["virial"]), "step": int(t["step"])}


def in_precision(case, out):
    if case["precision"] != "mixed":
        return out
    return {k: v.astype(np.float32) if isinstance(v, np.ndarray) and v.dtype == np.float64 else v
            for k, v in out.items()}


def run(state):
    case = state["case"]
    if case["what"] == "pack":
        for p in state["packs"]:
            p.enqueue(case["steps"])
            p.wait()
        states = [g.state() for p in state["packs"] for g in p.systems]
        return in_precision(case, {n: np.concatenate([st[i] for st in states]) for i, n in enumerate("xvf")})
    g, s = state["gpu"], state["system"]
    g.set_state(s.x, s.v)
    if case["what"] == "forces":
        g.build_neighbors(0)
        near, _, e_lj, e_coul = g.force_real()
        g.set_kvectors(state["k"])
        far, _ = g.rbe_force()
        bonded = g.force_bonded()[0] if case["kind"] == "water" else None
        return {"near": near, "e_lj": e_lj, "e_coul": e_coul, "far": far, "bonded": bonded}
    if case["what"] == "ewald":
        force, virial, energy = g.ewald_force(state["kmax"])
        return {"force": force, "virial": virial, "energy": np.array([energy])}
    g.md_init()
    if case["coulomb"] == "EWALD":  # a thermo row every ten steps
        done = 0
        while done < case["steps"]:
            n = min(10, case["steps"] - done)
            g.md_step(n)
            g.md_energy()
            done += n
    else:
        g.md_step(case["steps"])
    x, v, f, image = g.state()
    return in_precision(case, {"x": x, "v": v, "f": f, "image": image, **thermo_arrays(g.thermo())})


def k_count(case, atoms, kind):
    if case["what"] == "ewald":
        edge = (atoms / 0.5) ** (1 / 3) if kind == "salt" else (atoms / 0.10028) ** (1 / 3)
        return ((2 * converged_kmax(0.64 if kind == "salt" else 0.09, [edge])[0] + 1) ** 3 - 1) / 2
    if case.get("coulomb") == "EWALD":
        return ((2 * case["kmax"] + 1) ** 3 - 1) / 2
    return 100 if kind == "salt" else water_rbe_p(atoms)


def work(case):
    """Of one pass: 43 operations a pair within the cut-off (both sides of it)
    and 8 a pair and wave vector twice (structure factor and force); the
    configuration, velocities and forces read and written once."""
    def of(kind, atoms, steps):
        pairs = atoms * (0.5 * 4 / 3 * math.pi * 4.0 ** 3 if kind == "salt" else 0.10028 * 4 / 3 * math.pi * 1000.0)
        if case.get("lists") == "RBL":  # the core and the sample of the shell
            pairs = atoms * (0.5 * 4 / 3 * math.pi * 2.5 ** 3 + 50 if kind == "salt" else 0.10028 * 4 / 3 * math.pi * 125 + 100)
        if case["what"] == "ewald":
            pairs = 0
        return steps * (43.0 * pairs + 16.0 * atoms * k_count(case, atoms, kind)), 8.0 * 18 * atoms

    if case["what"] == "pack":
        parts = [of(k, n, case["steps"]) for k, n in ensemble_sizes(case)]
    else:
        parts = [of(case["kind"], case["atoms"], case.get("steps", 1))]
    return {"flops": sum(p[0] for p in parts), "bytes": sum(p[1] for p in parts)}


def tensors(s):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    return [torch.as_tensor(a, dtype=torch.float64, device=dev) for a in (s.x, s.charge, s.box)]


def pair_sums(s, r):
    """force and energies of every atom: Lennard-Jones (geometric epsilon,
    mean sigma) and erfc Coulomb over the minimum images within the cut-off,
    special pairs weighted"""
    x, q, box = tensors(s)
    n, dev = len(x), x.device
    qq = 332.06371 if r.unit == "REAL" else 1.0
    b = math.sqrt(r.alpha)
    typ = torch.as_tensor(s.type, device=dev).long()
    eps, sig = (torch.as_tensor(a, dtype=torch.float64, device=dev) for a in (s.eps, s.sigma))
    weighted = s.special_offsets is not None and r.special_bonds
    f, elj, ec = torch.zeros_like(x), torch.zeros_like(q), torch.zeros_like(q)
    for i0 in range(0, n, 512):
        i = slice(i0, min(n, i0 + 512))
        d = x[None] - x[i, None]
        d -= box * torch.round(d / box)
        d2 = (d * d).sum(-1)
        a, j = torch.nonzero((d2 > 1e-4) & (r.cut_off ** 2 - d2 > 1e-4), as_tuple=True)
        d, d2 = d[a, j], d2[a, j]
        a = a + i0
        w = torch.ones_like(d2)
        if weighted:
            w = torch.where(torch.div(a, 3, rounding_mode="floor") == torch.div(j, 3, rounding_mode="floor"), 0.0, w)
        e = torch.sqrt(eps[typ[a]] * eps[typ[j]])
        s6 = ((sig[typ[a]] + sig[typ[j]]) / 2) ** 6 / d2 ** 3
        rr = torch.sqrt(d2)
        c = qq * q[a] * q[j]
        near = torch.erfc(b * rr)
        g = near + 2 * b / math.sqrt(math.pi) * rr * torch.exp(-r.alpha * d2)
        k = -w * 24 * e * (2 * s6 - 1) * s6 / d2 + c * ((1 - w) - g) / (d2 * rr)
        f.index_add_(0, a, k[:, None] * d)
        elj.index_add_(0, a, w * 2 * e * (s6 - 1) * s6)
        ec.index_add_(0, a, 0.5 * c * (near - (1 - w)) / rr)
    return f, elj, ec


def wave_sums(s, r, m, scale, gauss):
    """k-space force, virial and energy terms over the wave vectors m (whole
    numbers), each with weight scale (and the Ewald Gaussian)"""
    x, q, box = tensors(s)
    qq = 332.06371 if r.unit == "REAL" else 1.0
    m = torch.as_tensor(m, dtype=torch.float64, device=x.device)
    turn = x / box
    f, vir, grid = torch.zeros_like(x), torch.zeros(len(x), 6, dtype=x.dtype, device=x.device), 0.0
    per = max(1, 40_000_000 // len(x))
    for l0 in range(0, len(m), per):
        mm = m[l0:l0 + per]
        k = 2 * math.pi * mm / box
        k2 = (k * k).sum(1)
        pre = scale / (float(s.volume) * k2)
        if gauss:
            pre = pre * torch.exp(-k2 / (4 * r.alpha))
        # the phase in turns, each axis reduced before the sum
        t = sum(torch.remainder(turn[:, d, None] * mm[None, :, d], 1.0) for d in range(3))
        t = 2 * math.pi * (t - torch.round(t))
        c, n = torch.cos(t), torch.sin(t)
        re, im = q @ c, q @ n
        g = -4 * math.pi * q[:, None] * (c * (pre * im) - n * (pre * re))
        f += g @ k
        for t6, (i, j) in enumerate(((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))):
            vir[:, t6] += x[:, i] * (g @ k[:, j]) + x[:, j] * (g @ k[:, i])
        grid += float((pre * (re * re + im * im)).sum())
    return qq * f, vir, qq * grid * 2 * math.pi


def bonded_force(s):
    """harmonic bonds and angles (rigid water: O-H1, O-H2 and H1-O-H2)"""
    x, _, box = tensors(s)
    x = x.reshape(-1, 3, 3)
    a, b = (x[:, k] - x[:, 0] for k in (1, 2))
    a, b = a - box * torch.round(a / box), b - box * torch.round(b / box)
    a.requires_grad_(True)
    b.requires_grad_(True)
    da, db = a.norm(dim=1), b.norm(dim=1)
    cos = ((a * b).sum(1) / (da * db)).clamp(-1, 1)
    e = float(s.bond_k[0]) * ((da - float(s.bond_r0[0])) ** 2 + (db - float(s.bond_r0[0])) ** 2)
    e = e + float(s.angle_k[0]) * (torch.acos(cos) - math.radians(float(s.angle_theta0[0]))) ** 2
    e.sum().backward()
    return torch.stack([a.grad + b.grad, -a.grad, -b.grad], 1).reshape(-1, 3)


def exact(case, seed):
    """The single-configuration calls, by direct sums in 64 bits.  A
    trajectory follows this package's own k-vector draws and constraint
    iterations step by step and has no value apart from them."""
    if case["what"] not in ("forces", "ewald"):
        return None
    seed = int(seed) + 1
    s, r = system_and_run(case, seed)
    if case["what"] == "ewald":
        km = converged_kmax(r.alpha, s.box)
        axis = [np.arange(-k, k + 1) for k in km]
        m = np.stack(np.meshgrid(*axis, indexing="ij"), -1).reshape(-1, 3)
        force, virial, energy = wave_sums(s, r, m[len(m) // 2 + 1:], 2.0, True)
        return {"force": force.cpu().numpy(), "virial": virial.cpu().numpy(), "energy": np.array([energy])}
    if min(s.box) < 2 * r.cut_off:
        near = e_lj = e_coul = None  # several images of an atom within the cut-off
    else:
        near, e_lj, e_coul = (t.cpu().numpy() for t in pair_sums(s, r))
    m = rbe_sample_host(r.alpha, s.box, r.rbe_p, seed, 1)  # an input of the call
    far = wave_sums(s, r, m, rbe_weight(r, s) / len(m), False)[0].cpu().numpy()
    bonded = bonded_force(s).detach().cpu().numpy() if case["kind"] == "water" else None
    return {"near": near, "e_lj": e_lj, "e_coul": e_coul, "far": far, "bonded": bonded}


def rbe_weight(r, s):
    """S: the sum of the Gaussian over all wave vectors but zero, by Jacobi's
    identity from the lattice sum (terms up to 10)"""
    h = 1.0
    for L in s.box:
        h *= math.sqrt(r.alpha * L * L / math.pi) * sum(math.exp(-r.alpha * L * L * m * m) for m in range(-10, 11))
    return h - 1.0
