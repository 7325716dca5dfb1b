"""Performance cases: the work that a program built on this library has it do.

Each case goes through the public Python entry points (copy_gpu_amd.force, .batch and
.proposal), over the sizes that the tests and the benchmark use:

  force      one force evaluation per pass at new k-vectors (rbmd_force_compute), as an
             ensemble with its own integrator calls it between its half kicks
  frames     single-point evaluation of unrelated configurations with energies and
             virial (trajectory frames): every evaluation builds the list anew
  ewald      one FP64 full-Ewald evaluation with energies (the physics reference that
             runs and k-samplers are judged against)
  md         velocity-Verlet steps on the device (rbmd_md_run): plain, thermostatted,
             with a learned k-space proposal, or with the random batch list
  batch      velocity-Verlet steps of uneven replicas (rbmd_batch_md_run)
  kspace     the k-space step without a handle (the far energy of a thermo row)
  spectrum   |rho(m)|^2 on a lattice box, the training data of the learned proposal
  mlp        a fit of the proposal network and its tabulation on the lattice box

prepare() makes what such a program holds beforehand (positions, charges, a handle,
forces of the starting positions); run() is one pass.
"""
import math

import numpy as np
import torch

from copy_gpu_amd import ForceConfig, LJCutCoulKspaceForce, systems
from copy_gpu_amd import force as force_module
from copy_gpu_amd import proposal as proposal_module
from copy_gpu_amd.batch import ReplicaBatch

DENSITY = 0.3   # reduced number density of the electrolytes
DMIN = 0.8      # their minimum separation
SKIN = 0.3


def listed():
    return [
        # the smallest electrolyte that the library's own start-up check evaluates, inside a
        # caller's integrator loop: one evaluation and one k-list per step
        {"name": "force_small", "kind": "force", "n": 4000, "P": 100, "alpha": 0.5, "rc": 5.0,
         "types": 1},
        # the large system of the benchmark: 1,048,576 ions, P = 500
        {"name": "force_large", "kind": "force", "n": 1048576, "P": 500, "alpha": 0.3, "rc": 6.0,
         "types": 1},
        # two unrelated frames of a two-type electrolyte, ragged size, energies and virial of
        # each: analysis of stored configurations
        {"name": "frames", "kind": "frames", "n": 30011, "P": 100, "alpha": 0.5, "rc": 5.0,
         "types": 2},
        # FP64 full Ewald with energies at the size of the reference's LJ_salt example
        {"name": "ewald_fp64", "kind": "ewald", "n": 6000, "alpha": 0.5, "rc": 5.0,
         "tol": 1e-10},
        # the headline run: 100,000 ions, learned proposal, P = 50
        {"name": "md_learned", "kind": "md", "n": 100000, "P": 50, "alpha": 0.5, "rc": 5.0,
         "steps": 64, "thermostat": "NONE", "learned": True, "precision": 32},
        # an NVT production run, Berendsen, between two output rows
        {"name": "md_nvt", "kind": "md", "n": 32768, "P": 100, "alpha": 0.5, "rc": 5.0,
         "steps": 50, "thermostat": "BERENDSEN", "learned": False, "precision": 32},
        # the plain LJ fluid in FP64, 4,000 atoms on an FCC lattice
        {"name": "md_lj_fp64", "kind": "lj", "nc": 10, "steps": 100},
        # the reference's own example: 1,000 ions in a 10^3 box, random batch list, RBE with
        # P = 100, Berendsen NVT
        {"name": "md_rbl", "kind": "rbl", "side": 10, "P": 100, "steps": 50},
        # 64 uneven replicas (2,048 to 65,536 ions) advanced together
        {"name": "batch", "kind": "batch", "replicas": 64, "n_min": 2048, "n_max": 65536,
         "P": 100, "steps": 8},
        # the far energy of a thermo row: the Kmax = 2 cube of the 1,000-ion example, FP64
        {"name": "kspace_small", "kind": "kspace", "n": 1000, "kmax": 2, "precision": 64},
        # one snapshot of the proposal's training data: |m_d| <= 32 at 100,000 ions
        {"name": "spectrum", "kind": "spectrum", "n": 100000, "Mg": 32},
        # a stretch of the proposal's fit on the folded |m_d| <= 32 box, and its tabulation
        {"name": "mlp_fit", "kind": "mlp", "Mg": 32, "iters": 20},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["force", "force", "frames", "ewald", "md", "md", "lj", "rbl", "batch",
                       "kspace", "spectrum", "mlp"])
    alpha, rc = rng.choice([(0.5, 5.0), (0.3, 6.0)])
    if kind == "force":
        return {"kind": kind, "n": _log_int(rng, 1000, 1000000), "P": _log_int(rng, 20, 500),
                "alpha": alpha, "rc": rc, "types": rng.choice([1, 2])}
    if kind == "frames":
        return {"kind": kind, "n": _log_int(rng, 1000, 200000), "P": _log_int(rng, 20, 400),
                "alpha": alpha, "rc": rc, "types": rng.choice([1, 2])}
    if kind == "ewald":
        return {"kind": kind, "n": _log_int(rng, 1000, 8000), "alpha": 0.5, "rc": 5.0,
                "tol": rng.choice([1e-8, 1e-10])}
    if kind == "md":
        fp64 = rng.random() < 0.2
        return {"kind": kind, "n": _log_int(rng, 1000, 20000 if fp64 else 100000),
                "P": rng.randint(20, 120), "alpha": 0.5, "rc": 5.0, "steps": rng.randint(5, 50),
                "thermostat": rng.choice(["NONE", "NONE", "BERENDSEN", "LANGEVIN"]),
                "learned": rng.random() < 0.4, "precision": 64 if fp64 else 32}
    if kind == "lj":
        return {"kind": kind, "nc": rng.randint(6, 16), "steps": rng.randint(10, 100)}
    if kind == "rbl":
        return {"kind": kind, "side": rng.randint(8, 24), "P": rng.randint(40, 120),
                "steps": rng.randint(20, 50)}
    if kind == "batch":
        return {"kind": kind, "replicas": rng.randint(3, 48), "n_min": rng.randint(1500, 3000),
                "n_max": rng.randint(5000, 40000), "P": rng.randint(40, 120),
                "steps": rng.randint(3, 12)}
    if kind == "kspace":
        return {"kind": kind, "n": _log_int(rng, 300, 50000), "kmax": rng.randint(1, 6),
                "precision": rng.choice([32, 64])}
    if kind == "spectrum":
        return {"kind": kind, "n": _log_int(rng, 4000, 60000), "Mg": rng.randint(8, 24)}
    return {"kind": "mlp", "Mg": rng.randint(8, 32), "iters": rng.randint(5, 25)}


# ------------------------------------------------------------------ inputs
def _dev(a, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a)).to("cuda", dtype)


def _ions(n, seed):
    """Positions [3][n], charges and box edge of a random electrolyte (host)."""
    x, y, z, q, L = systems.random_ions(n, DENSITY, DMIN, seed=seed)
    return (x, y, z), q, L


EPS, SIGMA = {1: (1.0,), 2: (1.0, 0.8)}, {1: (1.0,), 2: (1.0, 0.9)}


def _types(case, n, seed):
    if case["types"] == 1:
        return None
    return np.random.default_rng(seed).integers(0, 2, n).astype(np.int32)


def _seed(seed, k=0):
    return 1 + (int(seed) * 1009 + k * 7919) % (1 << 40)


def _frames(case, seed, count):
    n = case["n"]
    out = []
    for k in range(count):
        pos, q, L = _ions(n, _seed(seed, k))
        if k:
            q = out[0][1]  # the same salt in another configuration
        out.append((pos, q, L))
    return out, _types(case, n, _seed(seed))


def _lattice(case):
    """The in-built simple-cubic salt of the random batch list example at density 1."""
    s = case["side"]
    g = np.arange(s) + 0.5
    zz, yy, xx = np.meshgrid(g, g, g, indexing="ij")
    idx = np.arange(s ** 3)
    return (xx.ravel(), yy.ravel(), zz.ravel()), np.where(idx % 2 == 0, 1.0, -1.0), float(s)


def _zeros(n, dtype, count=3):
    return [torch.zeros(n, device="cuda", dtype=dtype) for _ in range(count)]


def _smooth_density(Mg, L, alpha):
    """An unnormalised proposal density of the kind that a fit gives: a(m) h(k), h smooth."""
    m = proposal_module.lattice_grid(Mg)
    k = proposal_module.kvecs(m, (L, L, L))
    kn = np.sqrt((k * k).sum(1))
    d = proposal_module.analytic_weight(m, (L, L, L), alpha) * (0.6 + 1.0 / (0.4 + kn))
    d[kn == 0.0] = 0.0
    return d


# ------------------------------------------------------------------ prepare
def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def _config(case, L, n, **kw):
    t = case.get("types", 1)
    return ForceConfig(box_len=(L, L, L), cut_off=2.5, coulomb_cut=case["rc"], skin=SKIN,
                       alpha=case["alpha"], eps=EPS[t], sigma=SIGMA[t], n_max=n, **kw)


def _prepare_force(case, seed, count=1):
    frames, types = _frames(case, seed, count)
    n, L = case["n"], frames[0][2]
    f = LJCutCoulKspaceForce(_config(case, L, n, kspace="RBE", coulomb_sample_num=case["P"]))
    f.Init(_dev(frames[0][1]), None if types is None else _dev(types, torch.int32))
    return {"kind": case["kind"], "f": f, "P": case["P"], "seed": _seed(seed), "step": 0,
            "X": [[_dev(a) for a in fr[0]] for fr in frames],
            "F": [_zeros(n, torch.float32) for _ in frames]}


def _prepare_frames(case, seed):
    return _prepare_force(case, seed, 2)


def _prepare_ewald(case, seed):
    pos, q, L = _ions(case["n"], _seed(seed))
    f = LJCutCoulKspaceForce(_config(case, L, case["n"], kspace="EWALD", precision=64,
                                     ewald_tol=case["tol"]))
    f.Init(_dev(q))
    return {"kind": "ewald", "f": f, "X": [_dev(a) for a in pos],
            "F": _zeros(case["n"], torch.float64)}


def _md_state(f, pos, vel, dtype, P, seed, dt, steps):
    n = pos[0].size
    st = {"f": f, "X": [_dev(a) for a in pos], "V": [_dev(a) for a in vel],
          "F": _zeros(n, dtype), "dt": dt, "steps": steps, "seed": _seed(seed), "step": 1}
    if P:
        f.sample_kvectors(P, st["seed"], 0)
    f.Execute(*st["X"], *st["F"])  # the forces of the starting positions
    return st


def _prepare_md(case, seed):
    n = case["n"]
    pos, q, L = _ions(n, _seed(seed))
    vel = systems.velocities(n, 1.0, seed=_seed(seed))
    f = LJCutCoulKspaceForce(_config(case, L, n, kspace="RBE", coulomb_sample_num=case["P"],
                                     precision=case["precision"]))
    f.Init(_dev(q))
    if case["learned"]:
        Mg = 32 if n > 20000 else 16
        p = proposal_module.Proposal(Mg, _smooth_density(Mg, L, case["alpha"]), 0.9,
                                     case["alpha"], (L, L, L))
        p.attach(f)
        p.close()
    st = _md_state(f, pos, vel, f.fdtype, case["P"], seed, 0.002, case["steps"])
    if case["thermostat"] != "NONE":
        f.set_thermostat(case["thermostat"], (1.0, 1.0, 0.5), seed=_seed(seed), gamma=1.0)
    return dict(st, kind="md")


def _prepare_lj(case, seed):
    x, y, z, L = systems.fcc(case["nc"], 0.8442)
    n = x.size
    vel = systems.velocities(n, 1.0, seed=_seed(seed))
    f = LJCutCoulKspaceForce(ForceConfig(box_len=(L, L, L), cut_off=2.5, coulomb_cut=0.0,
                                         skin=SKIN, alpha=0.0, kspace="NONE", precision=64,
                                         n_max=n))
    f.Init(_dev(np.zeros(n)))
    return dict(_md_state(f, (x, y, z), vel, torch.float64, 0, seed, 0.005, case["steps"]),
                kind="md")


def _prepare_rbl(case, seed):
    pos, q, L = _lattice(case)
    n = q.size
    vel = systems.velocities(n, 1.0, seed=_seed(seed))
    pice = force_module.rbl_pice_num(n, (L, L, L), min(5.0, 0.5 * L), 2.5, 50)
    f = LJCutCoulKspaceForce(ForceConfig(
        box_len=(L, L, L), cut_off=min(5.0, 0.5 * L), coulomb_cut=min(5.0, 0.5 * L), skin=SKIN,
        alpha=0.1, kspace="RBE", coulomb_sample_num=case["P"], neighbor_type="RBL", r_core=2.5,
        rbl_pice=pice, rbl_seed=_seed(seed), n_max=n))
    f.Init(_dev(q))
    st = _md_state(f, pos, vel, torch.float32, case["P"], seed, 0.002, case["steps"])
    f.set_thermostat("BERENDSEN", (1.0, 1.0, 0.5))
    return dict(st, kind="md")


def _prepare_batch(case, seed):
    sizes = systems.replica_sizes(case["replicas"], case["n_min"], case["n_max"])
    cfgs, host = [], []
    for r, n in enumerate(sizes):
        pos, q, L = _ions(n, _seed(seed, r))
        host.append((pos, systems.velocities(n, 1.0, seed=_seed(seed, r)), q))
        cfgs.append(ForceConfig(box_len=(L, L, L), cut_off=2.5, coulomb_cut=5.0, skin=SKIN,
                                alpha=0.5, kspace="RBE", coulomb_sample_num=case["P"], n_max=n))
    # one allocation per quantity, each replica a slice of it
    flat = [_dev(np.concatenate([h[0][d] for h in host])) for d in range(3)]
    flat += [_dev(np.concatenate([h[1][d] for h in host])) for d in range(3)]
    flat += _zeros(sum(sizes), torch.float32)
    b = ReplicaBatch(cfgs)
    seeds = [_seed(seed, 1000 + r) for r in range(len(sizes))]
    states, at = [], 0
    for r, n in enumerate(sizes):
        s = tuple(t[at:at + n] for t in flat)
        b.replicas[r].Init(_dev(host[r][2]))
        b.replicas[r].sample_kvectors(case["P"], seeds[r], 0)
        b.replicas[r].Execute(*s[:3], *s[6:9])
        states.append(s)
        at += n
    return {"kind": "batch", "b": b, "states": states, "seeds": seeds, "flat": flat, "step": 1,
            "steps": case["steps"]}


def _kspace_inputs(case, seed):
    pos, q, L = _ions(case["n"], _seed(seed))
    r = np.arange(-case["kmax"], case["kmax"] + 1)
    m = np.stack(np.meshgrid(r, r, r, indexing="ij"), -1).reshape(-1, 3)
    m = m[(m != 0).any(1)].astype(np.int32)
    alpha = 0.1
    k2 = ((2.0 * np.pi * m / L) ** 2).sum(1)
    return pos, q, L, alpha, m, np.exp(-k2 / (4.0 * alpha))


def _prepare_kspace(case, seed):
    pos, q, L, alpha, m, w = _kspace_inputs(case, seed)
    return {"kind": "kspace", "L": (L, L, L), "alpha": alpha, "X": [_dev(a) for a in pos],
            "q": _dev(q), "m": _dev(m.reshape(-1), torch.int32), "w": _dev(w),
            "precision": case["precision"],
            "dtype": torch.float32 if case["precision"] == 32 else torch.float64}


def _prepare_spectrum(case, seed):
    pos, q, L = _ions(case["n"], _seed(seed))
    return {"kind": "spectrum", "X": [_dev(a) for a in pos], "q": _dev(q), "L": (L, L, L),
            "Mg": case["Mg"]}


def _mlp_inputs(case, seed):
    """Training set of a screened spectrum with seeded scatter, the tabulation's features
    and a start between the network's own initial weights and a trained network's."""
    Mg, alpha = case["Mg"], 0.5
    L = (69.34 * Mg / 32.0,) * 3
    rng = np.random.default_rng(_seed(seed))
    m = proposal_module.lattice_grid(Mg)
    k2 = (proposal_module.kvecs(m, L) ** 2).sum(1)
    S2 = 1e5 * k2 / (k2 + 3.77) * rng.gamma(50.0, 0.02, len(m))
    k_scale = 2.0 * math.sqrt(alpha)
    feat, y, w, _ = proposal_module.training_set(S2, L, alpha, Mg, k_scale)
    grid = proposal_module.features(m, L, k_scale)
    p = np.zeros(proposal_module.NPARAM, np.float32)
    for lo, hi, s in ((0, 256, 6 / 68), (320, 4416, 6 / 128), (4480, 4544, 6 / 65)):
        p[lo:hi] = math.sqrt(s) * rng.uniform(-1, 1, hi - lo)
    p[256:320] = p[4416:4480] = 0.05
    p[4544] = math.log(math.e - 1.0)
    return feat, y, w, grid, p


LR = 3e-4  # the fit's late stage


def _prepare_mlp(case, seed):
    feat, y, w, grid, p = _mlp_inputs(case, seed)
    f32 = torch.float32
    return {"kind": "mlp", "net": proposal_module.ProposalMLP(1), "p": p, "feat": _dev(feat, f32),
            "y": _dev(y, f32), "w": _dev(w, f32), "grid": _dev(grid, f32),
            "iters": case["iters"]}


_PREPARE = {"force": _prepare_force, "frames": _prepare_frames, "ewald": _prepare_ewald,
            "md": _prepare_md, "lj": _prepare_lj, "rbl": _prepare_rbl, "batch": _prepare_batch,
            "kspace": _prepare_kspace, "spectrum": _prepare_spectrum, "mlp": _prepare_mlp}


# ------------------------------------------------------------------ run
def run(state):
    return _RUN[state["kind"]](state)


def _run_force(s):
    f = s["f"]
    f.sample_kvectors(s["P"], s["seed"], s["step"])
    s["step"] += 1
    f.Execute(*s["X"][0], *s["F"][0])
    return s["F"][0]


def _energies(f):
    ev = f.energy_virial()
    return {"energy": np.array([ev["e_lj"], ev["e_real"], ev["e_self"], ev["e_kspace"]]),
            "virial": ev["virial"]}


def _run_frames(s):
    f, out = s["f"], []
    for X, F in zip(s["X"], s["F"]):
        f.sample_kvectors(s["P"], s["seed"], s["step"])
        s["step"] += 1
        f.Execute(*X, *F, energy_virial=True)
        out.append({"force": F, "ev": _energies(f)})
    return out


def _run_ewald(s):
    s["f"].Execute(*s["X"], *s["F"], energy_virial=True)
    return {"force": s["F"], "ev": _energies(s["f"])}


def _run_md(s):
    s["f"].md_run(*s["X"], *s["V"], *s["F"], dt=s["dt"], nsteps=s["steps"], seed=s["seed"],
                  step0=s["step"])
    s["step"] += s["steps"]
    return {"x": s["X"], "v": s["V"], "f": s["F"]}


def _run_batch(s):
    s["b"].md_run(s["states"], 0.002, s["steps"], s["seeds"], step0=s["step"])
    s["step"] += s["steps"]
    return s["flat"]


def _run_kspace(s):
    F = _zeros(s["q"].numel(), s["dtype"])
    rho, ev = force_module.kspace_compute(s["L"], s["alpha"], *s["X"], s["q"], s["m"], s["w"], *F,
                                          precision=s["precision"])
    return {"rho": rho, "ev": ev, "force": F}


def _run_spectrum(s):
    return proposal_module.spectrum([tuple(s["X"])], s["q"], s["L"], 0.5, s["Mg"])


def _run_mlp(s):
    net = s["net"]
    net.set_params(s["p"])
    net.train(s["feat"], s["y"], s["w"], s["iters"], LR)
    return {"h": net.forward(s["grid"]), "params": net.params()}


_RUN = {"force": _run_force, "frames": _run_frames, "ewald": _run_ewald, "md": _run_md,
        "batch": _run_batch, "kspace": _run_kspace, "spectrum": _run_spectrum, "mlp": _run_mlp}


# ------------------------------------------------------------------ work
def _sphere(r):
    return 4.0 / 3.0 * math.pi * r ** 3


def _halfspace(L, alpha, tol):
    return 0.5 * _sphere(math.sqrt(-4.0 * alpha * math.log(tol)) * L / (2.0 * math.pi))


def work(case):
    """Reads of positions and charges, writes of forces (and the state of MD steps); per
    pair inside the cutoff about 40 operations (distance, erfc, LJ, force), once for both
    atoms; per atom and k-vector about 14 (phase, sine and cosine as one each, products),
    for the structure factor and again for the force."""
    kind = case["kind"]

    def ions(n, rc, P, fbytes):
        pairs = 0.5 * n * DENSITY * _sphere(rc)
        return n * (32.0 + 3.0 * fbytes), 40.0 * pairs + 28.0 * n * P

    if kind == "force":
        b, f = ions(case["n"], case["rc"], case["P"], 4)
    elif kind == "frames":
        b, f = (2.0 * v for v in ions(case["n"], case["rc"], case["P"], 4))
    elif kind == "ewald":
        L = (case["n"] / DENSITY) ** (1.0 / 3.0)
        b, f = ions(case["n"], case["rc"], _halfspace(L, case["alpha"], case["tol"]), 8)
    elif kind == "md":
        fb = case["precision"] // 8
        b, f = ions(case["n"], case["rc"], case["P"], fb)
        b, f = case["steps"] * (b + 48.0 * case["n"]), case["steps"] * f
    elif kind == "lj":
        n = 4.0 * case["nc"] ** 3
        b = case["steps"] * n * (24.0 + 24.0 + 48.0)
        f = case["steps"] * 20.0 * 0.5 * n * 0.8442 * _sphere(2.5)
    elif kind == "rbl":
        n, rc = case["side"] ** 3, min(5.0, 0.5 * case["side"])
        core = n * _sphere(2.5)
        shell = n * (_sphere(rc) - _sphere(2.5)) / 10.0
        b = case["steps"] * n * (32.0 + 12.0 + 48.0)
        f = case["steps"] * (40.0 * (core + shell) + 28.0 * n * case["P"])
    elif kind == "batch":
        lo, hi = case["n_min"], case["n_max"]
        n = case["replicas"] * (hi - lo) / math.log(hi / lo)
        b, f = ions(n, 5.0, case["P"], 4)
        b, f = case["steps"] * (b + 48.0 * n), case["steps"] * f
    elif kind == "kspace":
        n, P = case["n"], (2 * case["kmax"] + 1) ** 3 - 1
        b = n * (32.0 + 6.0 * case["precision"] / 8) + P * (20.0 + 16.0)
        f = 28.0 * n * P
    elif kind == "spectrum":
        G = (2 * case["Mg"] + 1) ** 3
        b = case["n"] * 32.0 + 8.0 * G
        # the lattice sum as one complex product per atom and half-space vector
        f = 8.0 * case["n"] * 0.5 * G
    else:
        B, G = (case["Mg"] + 1) ** 3, (2 * case["Mg"] + 1) ** 3
        b = case["iters"] * B * 24.0 + G * 20.0
        f = 2.0 * 4416.0 * ((case["iters"] + 1) * 3.0 * B + G)
    return {"bytes": float(b), "flops": float(f)}


# ------------------------------------------------------------------ exact
def exact(case, seed):
    return _EXACT[case["kind"]](case, seed) if case["kind"] in _EXACT else None


EXACT_PAIRS = 1.3e9  # pairs that a dense FP64 evaluation takes on


def _pairs(pos, q, L, rc_lj, rc, alpha, eps, sigma, types):
    """Dense FP64 LJ + erfc forces, energies and virial of a periodic box, by rows."""
    n = pos.shape[1]
    F = torch.zeros_like(pos)
    e = torch.zeros(2, dtype=torch.float64, device=pos.device)
    W = torch.zeros(6, dtype=torch.float64, device=pos.device)
    rows = max(1, int(3e7 / n))
    for a in range(0, n, rows):
        b = min(n, a + rows)
        d = pos[:, a:b, None] - pos[:, None, :]
        d -= L * torch.round(d / L)
        r2 = (d * d).sum(0)
        r2[torch.arange(b - a), torch.arange(a, b)] = 1e30
        if types is None:
            ep, sg = eps[0], sigma[0]
        else:
            ta, tb = types[a:b, None], types[None, :]
            ev = torch.tensor(eps, dtype=torch.float64, device=pos.device)
            sv = torch.tensor(sigma, dtype=torch.float64, device=pos.device)
            ep, sg = torch.sqrt(ev[ta] * ev[tb]), 0.5 * (sv[ta] + sv[tb])
        s6 = (sg * sg / r2) ** 3
        lj = r2 < rc_lj * rc_lj
        f = torch.where(lj, 24.0 * ep * (2.0 * s6 * s6 - s6) / r2, 0.0)
        e[0] += torch.where(lj, 2.0 * ep * (s6 * s6 - s6), 0.0).sum()
        if q is not None:
            r = torch.sqrt(r2)
            near = r2 < rc * rc
            qq = q[a:b, None] * q[None, :]
            ec = torch.where(near, qq * torch.erfc(math.sqrt(alpha) * r) / r, 0.0)
            g = 2.0 * math.sqrt(alpha / math.pi) * torch.exp(-alpha * r2)
            f = f + torch.where(near, (ec + qq * g) / r2, 0.0)
            e[1] += 0.5 * ec.sum()
        F[:, a:b] = (f * d).sum(2)
        for c, (i, j) in enumerate(((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))):
            W[c] += 0.5 * (f * d[i] * d[j]).sum()
    return F, e, W


def _phases(pos, m, L):
    return 2.0 * math.pi * torch.frac((m @ pos) / L)


def _rho(pos, q, m, L):
    """FP64 structure factor of integer vectors m [P, 3]."""
    re = torch.empty(len(m), dtype=torch.float64, device=pos.device)
    im = torch.empty_like(re)
    rows = max(1, int(6e7 / pos.shape[1]))
    for a in range(0, len(m), rows):
        ph = _phases(pos, m[a:a + rows], L)
        re[a:a + rows] = torch.cos(ph) @ q
        im[a:a + rows] = torch.sin(ph) @ q
    return re, im


def _kspace_exact(pos, q, m, w, L, alpha):
    """FP64 k-space forces, energy and virial of weights w at vectors m."""
    re, im = _rho(pos, q, m, L)
    k = 2.0 * math.pi * m / L
    k2 = (k * k).sum(1)
    V = L ** 3
    F = torch.zeros_like(pos)
    c = -4.0 * math.pi * w / (V * k2)
    rows = max(1, int(6e7 / pos.shape[1]))
    for a in range(0, len(m), rows):
        s = slice(a, a + rows)
        ph = _phases(pos, m[s], L)
        g = torch.cos(ph) * (c * im)[s, None] - torch.sin(ph) * (c * re)[s, None]
        F += q * (k[s].T @ g)
    e = w * (2.0 * math.pi / V) * (re * re + im * im) / k2
    bb = 2.0 * (1.0 / k2 + 1.0 / (4.0 * alpha))
    W = [(e * (1.0 - bb * k[:, d] ** 2)).sum() for d in range(3)]
    W += [-(e * bb * k[:, i] * k[:, j]).sum() for i, j in ((0, 1), (0, 2), (1, 2))]
    return F, e.sum(), torch.stack(W), torch.stack([re, im], 1)


def _rbe_weight(L, alpha, P):
    h = math.sqrt(alpha * L * L / math.pi) * sum(math.exp(-alpha * L * L * j * j)
                                                 for j in range(-10, 11))
    return (h ** 3 - 1.0) / P


def _self_energy(q, alpha):
    return -math.sqrt(alpha / math.pi) * float((q * q).sum())


def _single(case, seed, k, frame, types):
    pos, q, L = frame
    X, Q = torch.stack([_dev(a) for a in pos]), _dev(q)
    t = None if types is None else _dev(types, torch.int64)
    F, e, W = _pairs(X, Q, L, 2.5, case["rc"], case["alpha"], EPS[case["types"]],
                     SIGMA[case["types"]], t)
    # the k-list of this step is an input: the library's seeded draw, made on the host
    m, _ = systems.sample_kvectors_host(case["alpha"], [L] * 3, case["P"], _seed(seed), k)
    w = torch.full((case["P"],), _rbe_weight(L, case["alpha"], case["P"]),
                   dtype=torch.float64, device="cuda")
    Fk, ek, Wk, _ = _kspace_exact(X, Q, _dev(m), w, L, case["alpha"])
    en = np.array([float(e[0]), float(e[1]), _self_energy(Q, case["alpha"]), float(ek)])
    return list(F + Fk), {"energy": en, "virial": (W + Wk).cpu().numpy()}


def _exact_force(case, seed):
    if case["n"] ** 2 > EXACT_PAIRS:
        return None
    frames, types = _frames(case, seed, 1)
    return _single(case, seed, 0, frames[0], types)[0]


def _exact_frames(case, seed):
    if 2 * case["n"] ** 2 > 2 * EXACT_PAIRS:
        return None
    frames, types = _frames(case, seed, 2)
    out = []
    for k, fr in enumerate(frames):
        F, ev = _single(case, seed, k, fr, types)
        out.append({"force": F, "ev": ev})
    return out


def _exact_ewald(case, seed):
    pos, q, L = _ions(case["n"], _seed(seed))
    X, Q, alpha = torch.stack([_dev(a) for a in pos]), _dev(q), case["alpha"]
    F, e, W = _pairs(X, Q, L, 2.5, case["rc"], alpha, EPS[1], SIGMA[1], None)
    kmax2 = -4.0 * alpha * math.log(case["tol"])
    M = int(math.sqrt(kmax2) * L / (2.0 * math.pi)) + 1
    r = np.arange(-M, M + 1)
    m = np.stack(np.meshgrid(r[M:], r, r, indexing="ij"), -1).reshape(-1, 3)
    half = (m[:, 0] > 0) | (m[:, 1] > 0) | ((m[:, 1] == 0) & (m[:, 2] > 0))
    k2 = ((2.0 * np.pi * m / L) ** 2).sum(1)
    keep = half & (k2 <= kmax2)
    m, k2 = m[keep], k2[keep]
    Fk, ek, Wk, _ = _kspace_exact(X, Q, _dev(m), _dev(2.0 * np.exp(-k2 / (4.0 * alpha))), L,
                                  alpha)
    en = np.array([float(e[0]), float(e[1]), _self_energy(Q, alpha), float(ek)])
    return {"force": list(F + Fk), "ev": {"energy": en, "virial": (W + Wk).cpu().numpy()}}


def _exact_lj(case, seed):
    if case["steps"] * (4.0 * case["nc"] ** 3) ** 2 > 2.0 * EXACT_PAIRS:
        return None
    x, y, z, L = systems.fcc(case["nc"], 0.8442)
    X = torch.stack([_dev(a) for a in (x, y, z)])
    V = torch.stack([_dev(a) for a in systems.velocities(x.size, 1.0, seed=_seed(seed))])
    dt = 0.005

    def force():
        return _pairs(X, None, L, 2.5, 0.0, 0.0, (1.0,), (1.0,), None)[0]

    F = force()
    for _ in range(case["steps"]):
        V = V + 0.5 * dt * F
        X = X + dt * V
        X = X - L * torch.floor(X / L)
        F = force()
        V = V + 0.5 * dt * F
    return {"x": list(X), "v": list(V), "f": list(F)}


def _exact_kspace(case, seed):
    pos, q, L, alpha, m, w = _kspace_inputs(case, seed)
    X = torch.stack([_dev(a) for a in pos])
    F, e, W, rho = _kspace_exact(X, _dev(q), _dev(m), _dev(w), L, alpha)
    return {"rho": rho, "ev": torch.cat([e.reshape(1), W]), "force": list(F)}


def _exact_spectrum(case, seed):
    pos, q, L = _ions(case["n"], _seed(seed))
    X = torch.stack([_dev(a) for a in pos])
    r = np.arange(-case["Mg"], case["Mg"] + 1)
    z, y, x = np.meshgrid(r, r, r, indexing="ij")
    m = np.stack([x.ravel(), y.ravel(), z.ravel()], 1)
    G = len(m)
    h = G // 2  # the second half of the box is the mirror image of the first
    re, im = _rho(X, _dev(q), _dev(m[:h]), L)
    s = (re * re + im * im).cpu().numpy()
    return np.concatenate([s, [0.0], s[::-1]])


def _exact_mlp(case, seed):
    feat, y, w, grid, p0 = _mlp_inputs(case, seed)
    p, f, y, w = _dev(p0), _dev(feat), _dev(y), _dev(w)

    def net(p, f):
        q = p.float().bfloat16().double()  # the weights that the network uses
        q.requires_grad_(True)
        a = torch.nn.functional.silu(f @ q[:256].view(64, 4).T + q[256:320])
        a = torch.nn.functional.silu(a @ q[320:4416].view(64, 64).T + q[4416:4480])
        return q, torch.nn.functional.softplus(a @ q[4480:4544] + q[4544])

    m, v = torch.zeros_like(p), torch.zeros_like(p)
    for it in range(1, case["iters"] + 1):
        q, h = net(p, f)
        g, = torch.autograd.grad((w * (torch.log(h) - y) ** 2).sum(), q)
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        p = p - LR * (m / (1.0 - 0.9 ** it)) / (torch.sqrt(v / (1.0 - 0.999 ** it)) + 1e-8)
    with torch.no_grad():
        h = net(p, _dev(grid))[1]
    return {"h": h, "params": p.cpu().numpy()}


_EXACT = {"force": _exact_force, "frames": _exact_frames, "ewald": _exact_ewald,
          "lj": _exact_lj, "kspace": _exact_kspace, "spectrum": _exact_spectrum,
          "mlp": _exact_mlp}
