"""The framework's work as its users have it done, for timing.

Each case is one pass through the public entry points on inputs made from a
seed: force evaluations, timeblocks of simulations, batches of simulations,
trajectory gradients and radial distributions.

  listed()             the cases
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  what a script has in hand before the call
  run(state)           one pass; returns its outputs
  work(case)           bytes and floating-point operations a pass cannot do without
  exact(case, seed)    the outputs of the first pass in 64 bits, by plain torch
"""
import math

import numpy as np
import torch

import gamdpy_amd as gp
from gamdpy_amd.adjoint import DifferentiableNVE

KA_SIG = [[1.00, 0.80], [0.80, 0.88]]
KA_EPS = [[1.00, 1.50], [1.50, 0.50]]
BOND_PARAMS = [[1.1, 200.0], [1.0, 300.0]]
SCALAR_EVERY = 16        # steps between saves of a ScalarSaver
MOMENTUM_EVERY = 100     # steps between momentum resets
TIMEBLOCKS = 50000       # timeblocks a simulation is laid out for
ALL_PAIRS_MOST = 20000   # particles up to which a trajectory is followed in 64 bits


def listed():
    return [
        # a force evaluation of a small system, as a script that scores configurations
        # one by one does it: latency
        {"name": "eval_lj_500", "kind": "eval", "system": "lj", "N": 500, "rho": 0.8442, "cutoff": "SP", "lap": False},
        # the same of a large mixture, with the shifted-force cutoff and the laplacian
        # (the configurational temperature)
        {"name": "eval_ka_50021", "kind": "eval", "system": "ka", "N": 50021, "rho": 1.2, "cutoff": "SF", "lap": True},
        # the LJ benchmark of the reference at its most common size: NVE, N-squared list
        {"name": "md_lj_nve_2048", "kind": "md", "system": "lj", "N": 2048, "rho": 0.8442, "integrator": "NVE",
         "T": 1.44, "dt": 0.005, "steps": 128, "skin": 0.5, "scalars": False, "rdf_bins": 0},
        # an everyday liquid: the Kob-Andersen mixture in NVT with scalar output
        {"name": "md_ka_nvt_4000", "kind": "md", "system": "ka", "N": 4000, "rho": 1.2, "integrator": "NVT",
         "T": 2.0, "dt": 0.004, "steps": 128, "skin": 0.5, "scalars": True, "rdf_bins": 0},
        # the headline workload: a supercooled Kob-Andersen liquid (melted and cooled by a
        # temperature ramp), a partial g(r) every 100 steps beside the steps
        {"name": "md_ka_nvt_65536_rdf", "kind": "md", "system": "ka", "N": 65536, "rho": 1.2, "integrator": "NVT",
         "T": 0.45, "dt": 0.004, "steps": 100, "skin": 0.3, "scalars": False, "rdf_bins": 1000},
        # one very large system with Langevin dynamics, at the melting density
        {"name": "md_lj_langevin_1048576", "kind": "md", "system": "lj", "N": 1048576, "rho": 0.973,
         "integrator": "NVT_Langevin", "T": 0.7, "dt": 0.005, "steps": 128, "skin": 0.5, "scalars": False,
         "rdf_bins": 0},
        # constant pressure: the box and every cell change each step
        {"name": "md_lj_npt_10976", "kind": "md", "system": "lj", "N": 10976, "rho": 0.7543, "integrator": "NPT",
         "T": 2.0, "dt": 0.002, "steps": 128, "skin": 0.5, "scalars": True, "rdf_bins": 0},
        # bonded chains with the bonded pairs excluded from the pair list
        {"name": "md_chains_nvt_8788", "kind": "md", "system": "chains", "N": 8788, "rho": 0.8442,
         "integrator": "NVT", "T": 1.0, "dt": 0.002, "steps": 128, "skin": 0.5, "scalars": True, "rdf_bins": 0},
        # an ensemble of state points advanced together (the driver and lanes the autotuner
        # settles on for such a batch)
        {"name": "batch_ka_64", "kind": "batch", "replicas": 64, "Nmin": 1000, "Nmax": 8000, "steps": 64},
        # the gradient of a trajectory's g(r) for fitting a force field
        {"name": "adjoint_ka_4096", "kind": "adjoint", "N": 4096, "rho": 1.2, "steps": 200, "bins": 200,
         "rmax": 4.0},
        # the same of a small system, as a script that develops the fit uses it
        {"name": "adjoint_ka_500", "kind": "adjoint", "N": 500, "rho": 1.2, "steps": 40, "bins": 100, "rmax": 2.5},
        # g(r) of stored configurations: positions on the host, in no spatial order after a long run
        {"name": "rdf_ka_65536", "kind": "rdf", "N": 65536, "rho": 1.2, "bins": 1000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["eval", "eval", "md", "md", "md", "md", "batch", "adjoint", "rdf"])
    system = rng.choice(["lj", "ka"])
    rho = round(rng.uniform(0.75, 0.9) if system == "lj" else rng.uniform(1.1, 1.25), 3)
    if kind == "eval":
        return {"kind": kind, "system": system, "N": _log_int(rng, 300, 60000), "rho": rho,
                "cutoff": rng.choice(["SP", "SF"]), "lap": rng.random() < 0.3}
    if kind == "batch":
        lo = _log_int(rng, 600, 2500)
        return {"kind": kind, "replicas": _log_int(rng, 4, 48), "Nmin": lo, "Nmax": lo + _log_int(rng, 500, 5000),
                "steps": 64}
    if kind == "adjoint":
        N = _log_int(rng, 300, 4000)
        return {"kind": kind, "N": N, "rho": rho if system == "ka" else 1.2, "steps": rng.randint(20, 150),
                "bins": rng.randint(50, 200), "rmax": round(min(4.0, 0.5 * (N / 1.25) ** (1 / 3) - 0.25), 2)}
    if kind == "rdf":
        return {"kind": kind, "N": _log_int(rng, 1000, 60000), "rho": 1.2, "bins": rng.randint(100, 1000)}
    if rng.random() < 0.2:
        return {"kind": "md", "system": "chains", "N": 4 * rng.randint(6, 16) ** 3, "rho": 0.8442,
                "integrator": "NVT", "T": 1.0, "dt": 0.002, "steps": 100, "skin": 0.5, "scalars": True,
                "rdf_bins": 0}
    integrator = rng.choice(["NVE", "NVT", "NVT_Langevin"])
    N = _log_int(rng, 700, 200000)
    return {"kind": "md", "system": system, "N": N, "rho": rho, "integrator": integrator,
            "T": round(rng.uniform(0.8, 2.0), 2), "dt": 0.004, "steps": 100,
            "skin": round(rng.uniform(0.3, 0.5), 2), "scalars": rng.random() < 0.5,
            "rdf_bins": rng.randint(200, 1000) if 3000 < N < 60000 and rng.random() < 0.3 else 0}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _positions(N, rho, g, jitter, whole_cells=False):
    """N positions at density rho: sites of the smallest near-cubic FCC lattice
    that has them (N of its sites taken at random, all of them for
    whole_cells), each moved by up to jitter per dimension, in a cubic box.
    -> (N, 3) float32, box length"""
    n = math.ceil((N / 4) ** (1 / 3) - 1e-9)
    cells = min((a * b * c, (a, b, c)) for a in (n, n - 1) for b in (n, n - 1) for c in (n, n + 1)
                if 4 * a * b * c >= N)[1]
    corner = np.stack(np.meshgrid(*[np.arange(k) for k in cells], indexing="ij"), axis=-1).reshape(-1, 1, 3)
    sites = (corner + np.array([[0, 0, 0], [.5, .5, 0], [.5, 0, .5], [0, .5, .5]]) + 0.25).reshape(-1, 3)
    if whole_cells:
        assert len(sites) == N
    else:
        sites = sites[np.sort(g.permutation(len(sites))[:N])]
    L = float(np.float32((N / rho) ** (1 / 3)))
    r = (sites / np.array(cells) - 0.5) * L + g.uniform(-jitter, jitter, sites.shape)
    r -= L * np.round(r / L)
    return r.astype(np.float32), L


def _configuration(system, N, rho, T, seed, lap=False, jitter=0.06):
    g = np.random.default_rng(seed)
    conf = gp.Configuration(D=3, compute_flags={"lapU": True} if lap else None)
    r, L = _positions(N, rho, g, jitter, whole_cells=system == "chains")
    conf["r"] = r
    conf.simbox = gp.Orthorhombic(3, np.array([L, L, L]))
    conf["m"] = 1.0
    if system == "ka":
        conf.ptype[g.permutation(N)[:int(round(0.2 * N))]] = 1
    conf.randomize_velocities(temperature=T, seed=seed)
    return conf


def _interactions(system, conf, cutoff="SP"):
    func = (gp.apply_shifted_potential_cutoff if cutoff == "SP" else gp.apply_shifted_force_cutoff)(
        gp.LJ_12_6_sigma_epsilon)
    if system == "ka":
        return gp.PairPotential(func, params=[KA_SIG, KA_EPS, np.array(KA_SIG) * 2.5], max_num_nbs=512)
    if system == "lj":
        return gp.PairPotential(func, params=[1.0, 1.0, 2.5], max_num_nbs=256)
    # four-bead chains, one per FCC unit cell
    bonds = gp.Bonds(gp.harmonic_bond_function, BOND_PARAMS, _chain_bonds(conf.N))
    return [gp.PairPotential(func, params=[1.0, 1.0, 2.5], max_num_nbs=256,
                             exclusions=bonds.get_exclusions(conf, max_number_exclusions=4)), bonds]


def _chain_bonds(N):
    return [b for a in range(0, N, 4) for b in ([a, a + 1, 0], [a + 1, a + 2, 1], [a + 2, a + 3, 0])]


def _target(case):
    """The thermostat's temperature: constant, or from T = 2 (melt) down to a
    supercooled state point over the first blocks."""
    return case["T"] if case["T"] >= 0.7 else gp.make_function_ramp(2.0, 2.0, case["T"], 6.0)


def _start_temperature(case):
    return case["T"] if case["T"] >= 0.7 else 2.0


def _integrator(case, seed):
    T, dt = _target(case), case["dt"]
    if case["integrator"] == "NVE":
        return gp.NVE(dt=dt)
    if case["integrator"] == "NVT":
        return gp.NVT(temperature=T, tau=0.2, dt=dt)
    if case["integrator"] == "NPT":
        return gp.NPT_Atomic(temperature=T, tau=0.4, pressure=4.7, tau_p=20, dt=dt)
    return gp.NVT_Langevin(temperature=T, alpha=0.1, dt=dt, seed=seed)


def _prepare_md(case, seed):
    conf = _configuration(case["system"], case["N"], case["rho"], _start_temperature(case), seed)
    inter = _interactions(case["system"], conf)
    plan = gp.get_default_compute_plan(conf)
    plan["skin"] = case["skin"]
    actions = [gp.MomentumReset(MOMENTUM_EVERY)]
    if case["scalars"]:
        actions.append(gp.ScalarSaver(SCALAR_EVERY))
    sim = gp.Simulation(conf, inter, _integrator(case, seed), actions, num_timeblocks=TIMEBLOCKS,
                        steps_per_timeblock=case["steps"], compute_plan=plan, storage="memory", steps_in_kernel_test=0)
    rdf = gp.CalculatorRadialDistribution(conf, bins=case["rdf_bins"]) if case["rdf_bins"] else None
    conf.copy_to_device()   # the start, where the first g(r) is taken
    return {"kind": "md", "conf": conf, "sim": sim, "rdf": rdf, "blocks": sim.run_timeblocks()}


def _replica_points(case, seed):
    """(N, density, temperature) of each replica: sizes spread over the case's
    range, state points from the seed."""
    g, n = np.random.default_rng(seed), np.random.default_rng(case["replicas"])
    return [(int(n.integers(case["Nmin"], case["Nmax"] + 1)), float(g.uniform(1.1, 1.25)), float(g.uniform(0.7, 2.0)))
            for _ in range(case["replicas"])]


def _prepare_batch(case, seed):
    reps = []
    for k, (N, rho, T) in enumerate(_replica_points(case, seed)):
        conf = _configuration("ka", N, rho, T, seed + 1000 * k)
        reps.append(gp.Replica(conf, _interactions("ka", conf), gp.NVT(temperature=T, tau=0.2, dt=0.004)))
    batch = gp.BatchedSimulation(reps, num_timeblocks=TIMEBLOCKS, steps_per_timeblock=case["steps"], tp=2, skin=0.5,
                                 driver="graph")
    return {"kind": "batch", "batch": batch, "blocks": batch.run_timeblocks()}


def _prepare_adjoint(case, seed):
    conf = _configuration("ka", case["N"], case["rho"], 1.0, seed)
    traj = DifferentiableNVE(conf, dt=0.004, nsteps=case["steps"], cut=np.array(KA_SIG) * 2.5, ckpt_every=20,
                             rdf_every=10, bins=case["bins"], rmax=case["rmax"], width=0.02)
    # the structure a first fit pulls towards: none below contact, flat beyond
    target = torch.from_numpy(np.where(traj.r > 0.95, 1.0, 0.0) * np.ones((len(traj.norm), 1)))
    return {"kind": "adjoint", "traj": traj, "target": target,
            "r0": torch.from_numpy(np.array(conf["r"])), "sigma": torch.tensor(KA_SIG, dtype=torch.float32),
            "epsilon": torch.tensor(KA_EPS, dtype=torch.float32)}


def _rdf_configuration(case, seed):
    conf = _configuration("ka", case["N"], case["rho"], 1.0, seed, jitter=0.1)
    order = np.random.default_rng(seed + 1).permutation(case["N"])
    conf["r"] = np.ascontiguousarray(conf["r"][order])
    conf.ptype = np.ascontiguousarray(conf.ptype[order])
    return conf


def prepare(case, seed):
    kind = case["kind"]
    if kind == "md":
        return _prepare_md(case, seed)
    if kind == "batch":
        return _prepare_batch(case, seed)
    if kind == "adjoint":
        return _prepare_adjoint(case, seed)
    if kind == "rdf":
        conf = _rdf_configuration(case, seed)
        return {"kind": kind, "conf": conf, "rdf": gp.CalculatorRadialDistribution(conf, bins=case["bins"])}
    conf = _configuration(case["system"], case["N"], case["rho"], 1.0, seed, lap=case["lap"])
    return {"kind": "eval", "conf": conf, "evaluator": gp.Evaluator(conf, _interactions(case["system"], conf,
                                                                                      case["cutoff"]))}


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def _next_block(state, owner):
    """The next timeblock of a loop over run_timeblocks()."""
    block = next(state["blocks"], None)
    if block is None:
        state["blocks"] = owner.run_timeblocks()
        block = next(state["blocks"])
    return block


def _unwrapped(conf):
    """Positions with the box crossings undone, as a mean-square displacement
    needs them (and free of the jumps of a particle at the box's face)."""
    L = torch.from_numpy(np.asarray(conf.simbox.lengths, np.float32))
    return torch.addcmul(torch.from_numpy(conf["r"]), torch.from_numpy(conf.r_im).to(torch.float32), L)


def _state_of(conf):
    return {"r": _unwrapped(conf), "v": conf["v"], "f": conf["f"], "scalars": conf.scalars}


def run(state):
    kind = state["kind"]
    if kind == "eval":
        conf = state["conf"]
        state["evaluator"].evaluate()
        out = {"f": conf["f"], "U": conf["U"], "W": conf["W"]}
        if "lapU" in conf.sid:
            out["lapU"] = conf["lapU"]
        return out
    if kind == "md":
        conf, sim, rdf = state["conf"], state["sim"], state["rdf"]
        if rdf is not None:
            rdf.update(overlap=True)   # of the configuration so far, beside the next steps
        block = _next_block(state, sim)
        out = _state_of(conf)
        if "scalars" in sim.output.keys():
            out["saved"] = sim.output["scalars"][block]
        if sim.integrator.kind == "NPT_Atomic":
            out["box"] = conf.simbox.lengths
        if rdf is not None:
            out["counts"] = rdf.rdf_list[-1].astype(np.float32)
        return out
    if kind == "batch":
        _next_block(state, state["batch"])
        confs = [r.configuration for r in state["batch"].replicas]
        return {"r": torch.cat([_unwrapped(c) for c in confs]), "v": np.concatenate([c["v"] for c in confs]),
                "f": np.concatenate([c["f"] for c in confs]), "scalars": np.concatenate([c.scalars for c in confs])}
    if kind == "adjoint":
        r0, s, e = (state[k].clone().requires_grad_(True) for k in ("r0", "sigma", "epsilon"))
        g = state["traj"].rdf(r0, s, e)
        ((g - state["target"]) ** 2).mean().backward()
        return {"g": g.detach().to(torch.float32), "r0": r0.grad, "sigma": s.grad, "epsilon": e.grad}
    state["rdf"].update()
    return {"counts": state["rdf"].rdf_list[-1].astype(np.int64)}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _list_length(case, skin):
    return case["rho"] * 4.0 * math.pi / 3.0 * (2.5 + skin) ** 3


def work(case):
    kind = case["kind"]
    if kind == "eval":
        inside = case["rho"] * 4.0 * math.pi / 3.0 * 2.5 ** 3
        return {"bytes": case["N"] * (12 + 4 + 12 + 8), "flops": case["N"] * inside * 30}
    if kind == "md":
        N, n = case["N"], _list_length(case, case["skin"])
        rdf = 0.5 * N * N * math.pi / 6 * 12 if case["rdf_bins"] else 0.0
        return {"bytes": case["steps"] * N * ((2 if N <= 65536 else 4) * n + 92),
                "flops": case["steps"] * N * (30 * n + 40) + rdf}
    if kind == "batch":
        N = case["replicas"] * 0.5 * (case["Nmin"] + case["Nmax"])
        n = _list_length({"rho": 1.175}, 0.5)
        return {"bytes": case["steps"] * N * (2 * n + 92), "flops": case["steps"] * N * (30 * n + 40)}
    if kind == "adjoint":
        N, n = case["N"], _list_length(case, 0.5)
        frames = case["steps"] // 10 + 1
        far = case["rho"] * 4.0 * math.pi / 3.0 * (case["rmax"] + 0.1) ** 3
        return {"bytes": case["steps"] * N * (3 * 2 * n + 4 * 92) + 2 * frames * N * (2 * far + 32),
                "flops": case["steps"] * N * n * (30 + 30 + 60) + frames * N * far * 0.5 * (40 + 60)}
    return {"bytes": case["N"] * 16 + 4 * 8 * case["bins"], "flops": 0.5 * case["N"] ** 2 * math.pi / 6 * 12}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _tables(system, cutoff):
    """sigma, epsilon, cut of each type pair (the float32 values the framework is given)."""
    sig, eps = (KA_SIG, KA_EPS) if system == "ka" else ([[1.0]], [[1.0]])
    s, e, c = (torch.tensor(np.asarray(x, np.float32).astype(np.float64), device=_device())
               for x in (sig, eps, np.asarray(np.float32(sig), np.float64) * 2.5))
    return s, e, c.to(torch.float32).double(), cutoff


def _pair_sums(r, t, L, tables, excluded=None, lap=False):
    """Forces, U, W (and lapU) per particle of all pairs, rows of particles at a time."""
    sig, eps, cut, cutoff = tables
    N = len(r)
    f, out = torch.zeros_like(r), torch.zeros(3, N, dtype=r.dtype, device=r.device)
    rows = max(1, min(N, (1 << 25) // N))

    def lj(d2, s, e):
        i2 = 1.0 / d2
        x3 = (s * s * i2) ** 3
        return 4 * e * (x3 * x3 - x3), 24 * e * (2 * x3 * x3 - x3) * i2, 24 * e * (26 * x3 * x3 - 7 * x3) * i2

    uc, sc, _ = lj(cut * cut, sig, eps)
    if cutoff == "SP":
        sc = torch.zeros_like(sc)
    for a in range(0, N, rows):
        b = min(N, a + rows)
        d = r[a:b, None, :] - r[None, :, :]
        d -= L * torch.round(d / L)
        d2 = (d * d).sum(-1)
        d2[torch.arange(b - a, device=r.device), torch.arange(a, b, device=r.device)] = math.inf
        if excluded is not None:
            m = (excluded[0] >= a) & (excluded[0] < b)
            d2[excluded[0][m] - a, excluded[1][m]] = math.inf
        i, j = torch.nonzero(d2 < float(cut.max()) ** 2, as_tuple=True)
        ti, tj = t[a + i], t[j]
        d, d2, c = d[i, j], d2[i, j], cut[ti, tj]
        m = d2 < c * c
        i, d, d2, c, ti, tj = i[m], d[m], d2[m], c[m], ti[m], tj[m]
        u, s, upp = lj(d2, sig[ti, tj], eps[ti, tj])
        u = u - (uc[ti, tj] - sc[ti, tj] * c * (torch.sqrt(d2) - c))
        s = s - sc[ti, tj]
        f[a:b].index_add_(0, i, s[:, None] * d)
        terms = (0.5 * u, d2 * s / 6.0) + ((upp - 2.0 * s,) if lap else ())
        for k, x in enumerate(terms):
            out[k, a:b].index_add_(0, i, x)
    return f, out


def _bond_sums(r, L, idx, params, f, out):
    i, j = idx[:, 0], idx[:, 1]
    r0, k = params[idx[:, 2], 0], params[idx[:, 2], 1]
    d = r[j] - r[i]
    d -= L * torch.round(d / L)
    dist = torch.sqrt((d * d).sum(-1))
    u, s = 0.5 * k * (dist - r0) ** 2, -k * (dist - r0) / dist
    for a, sign in ((i, -1.0), (j, 1.0)):
        f.index_add_(0, a, sign * s[:, None] * d)
        out[0].index_add_(0, a, 0.5 * u)
        out[1].index_add_(0, a, dist * dist * s / 6.0)


def _exact_eval(case, seed):
    conf = _configuration(case["system"], case["N"], case["rho"], 1.0, seed, lap=case["lap"])
    dev = _device()
    r = torch.from_numpy(conf["r"].astype(np.float64)).to(dev)
    t = torch.from_numpy(conf.ptype.astype(np.int64)).to(dev)
    f, out = _pair_sums(r, t, float(np.float32(conf.simbox.lengths[0])), _tables(case["system"], case["cutoff"]),
                        lap=case["lap"])
    got = {"f": f, "U": out[0], "W": out[1]}
    if case["lap"]:
        got["lapU"] = out[2]
    return got


def _schedule(case):
    T = _target(case)
    return (lambda t: float(np.float32(T))) if not callable(T) else (lambda t: float(T(np.float32(t))))


def _follow(conf, system, case, integrator, T, steps):
    """The trajectory of one timeblock in 64 bits: (r unwrapped, v, f, scalars, saved rows, box)."""
    dev, N, dt = _device(), conf.N, float(np.float32(case["dt"]))
    L = float(np.float32(conf.simbox.lengths[0]))
    x = torch.from_numpy(conf["r"].astype(np.float64)).to(dev)
    v = torch.from_numpy(conf["v"].astype(np.float64)).to(dev)
    t = torch.from_numpy(conf.ptype.astype(np.int64)).to(dev)
    tables = _tables(system, "SP")
    bonds = excluded = None
    if system == "chains":
        bonds = torch.tensor(_chain_bonds(N), device=dev)
        params = torch.tensor(np.asarray(BOND_PARAMS, np.float32).astype(np.float64), device=dev)
        excluded = (torch.cat([bonds[:, 0], bonds[:, 1]]), torch.cat([bonds[:, 1], bonds[:, 0]]))
    deg = 3 * N - 3
    xi = rate_t = rate_p = 0.0
    vol = L ** 3
    K = torch.zeros(N, dtype=torch.float64, device=dev)
    saved = []
    for s in range(steps + 1):
        f, out = _pair_sums(x, t, L, tables, excluded)
        if bonds is not None:
            _bond_sums(x, L, bonds, params, f, out)
        if s == steps:
            break
        if integrator == "NVE":
            w = v + f * dt
            K = 0.125 * ((v + w) ** 2).sum(-1)
            v = w
            x = x + v * dt
        elif integrator == "NVT":
            h = 0.5 * xi * dt
            v = ((1 - h) * v + f * dt) / (1 + h)
            K = 0.5 * (v * v).sum(-1)
            x = x + v * dt
            xi += dt * float(np.float32(4.0 * np.pi * np.pi / 0.2 / 0.2)) * (2 * float(K.sum()) / (deg * T(s * dt)) - 1)
        else:
            h = 0.5 * dt * ((1 + 3 / deg) * rate_p + rate_t)
            v = ((1 - h) * v + f * dt) / (1 + h)
            K = 0.5 * (v * v).sum(-1)
            cube = 1 + 3 * dt * rate_p
            # the dilation acts on the wrapped position, the scaling on the whole
            x = (x + v * dt + rate_p * dt * (x - L * torch.round(x / L))) * cube ** (1 / 3)
            L, vol = L * cube ** (1 / 3), vol * cube
            ksum, Tk = float(K.sum()), 2 * float(K.sum()) / deg
            m = (deg - 1) * 3 / (4 * math.pi ** 2)
            mt, mp, target = m * 0.4 ** 2 * Tk, m * 20.0 ** 2 * Tk, T(s * dt)
            inner = (Tk * N + float(out[1].sum())) / vol
            ke = (2 * ksum + rate_p ** 2 * mp) / ((deg + 1) * target) - 1
            was = rate_p
            rate_t += dt * ke * (deg + 1) * target / mt
            rate_p += dt * (3 * (vol * (inner - float(np.float32(4.7))) + 0.5 * ksum / deg) / mp + rate_t * was)
        if case["scalars"] and s % SCALAR_EVERY == 0 and len(saved) < steps // SCALAR_EVERY:
            saved.append([float(out[0].sum()), float(out[1].sum()), float(K.sum())])
        if case["momentum"] and s % MOMENTUM_EVERY == 0:
            v = v - v.mean(0)
    scalars = torch.stack([out[0], out[1], K, torch.ones_like(K)], dim=1)
    return {"r": x, "v": v, "f": f, "scalars": scalars}, saved, L


def _exact_md(case, seed):
    N = case["N"]
    if N > ALL_PAIRS_MOST or case["integrator"] not in ("NVE", "NVT", "NPT"):
        return None     # too large for all pairs at every step, or with random forces of the framework's own
    conf = _configuration(case["system"], N, case["rho"], _start_temperature(case), seed)
    got, saved, L = _follow(conf, case["system"], dict(case, momentum=True), case["integrator"], _schedule(case),
                            case["steps"])
    if case["scalars"]:
        got["saved"] = torch.tensor(saved, dtype=torch.float64)
    if case["integrator"] == "NPT":
        got["box"] = torch.tensor([L, L, L], dtype=torch.float64)
    if case["rdf_bins"]:
        got["counts"] = None
    return got


def _exact_batch(case, seed):
    points = _replica_points(case, seed)
    if sum(N * N for N, _, _ in points) * case["steps"] > 6e10:
        return None     # over 20 seconds of all pairs
    parts = []
    for k, (N, rho, T) in enumerate(points):
        conf = _configuration("ka", N, rho, T, seed + 1000 * k)
        parts.append(_follow(conf, "ka", {"dt": 0.004, "scalars": False, "momentum": False}, "NVT",
                             lambda t, T=T: float(np.float32(T)), case["steps"])[0])
    return {k: torch.cat([p[k] for p in parts]) for k in parts[0]}


def _exact_adjoint(case, seed):
    if case["N"] > 800 or case["steps"] > 60:
        return None     # the graph of all pairs of every step
    conf = _configuration("ka", case["N"], case["rho"], 1.0, seed)
    dev, N = _device(), case["N"]
    L, dt = float(np.float32(conf.simbox.lengths[0])), float(np.float32(0.004))
    one = lambda x: torch.tensor(np.asarray(x, np.float32).astype(np.float64), device=dev)  # noqa: E731
    t = torch.from_numpy(conf.ptype.astype(np.int64)).to(dev)
    C = one(np.array(KA_SIG) * 2.5)[t][:, t]
    sig, eps, r0 = one(KA_SIG).requires_grad_(True), one(KA_EPS).requires_grad_(True), one(conf["r"]).requires_grad_(True)
    v = one(conf["v"])
    bins, rmax, width = case["bins"], case["rmax"], 0.02
    rk = (torch.arange(bins, dtype=torch.float64, device=dev) + 0.5) * (rmax / bins)
    upper = torch.triu_indices(N, N, offset=1, device=dev)
    cls = t[upper[0]] + t[upper[1]]

    def pairs(r):
        d = r[:, None, :] - r[None, :, :]
        return d - L * torch.round(d.detach() / L)

    def forces(r):
        d = pairs(r)
        d2 = (d * d).sum(-1)
        ok = (d2 < C * C) & ~torch.eye(N, dtype=torch.bool, device=dev)
        d2 = torch.where(ok, d2, 1.0)
        S, E = sig[t][:, t], eps[t][:, t]
        x3, c3 = (S * S / d2) ** 3, (S / C) ** 6
        s = 24 * E * ((2 * x3 * x3 - x3) / d2 - (2 * c3 * c3 - c3) / (C * C))
        return (torch.where(ok, s, 0.0)[:, :, None] * d).sum(1)

    def histogram(r):
        d = pairs(r)[upper[0], upper[1]]
        d2 = (d * d).sum(-1)
        near = d2 < (rmax + 5 * width) ** 2
        x = torch.sqrt(d2[near])[:, None] - rk[None, :]
        k = torch.exp(-0.5 * x * x / width ** 2) - math.exp(-12.5)
        k = torch.where((x.abs() < 5 * width) & (k > 0), k, 0.0)
        return torch.zeros(3, bins, dtype=torch.float64, device=dev).index_add(0, cls[near], k)

    # type classes (0, 0), (0, 1), (1, 1): the sum of the two types
    r, H, frames = r0, 0.0, 0
    for n in range(case["steps"] + 1):
        if n % 10 == 0:
            H, frames = H + histogram(r), frames + 1
        if n == case["steps"]:
            break
        v = v + forces(r) * dt
        r = r + v * dt
        r = r - L * torch.round(r.detach() / L)
    counts = np.bincount(conf.ptype, minlength=2).astype(np.float64)
    per = [counts[0] * (counts[0] - 1) / 2, counts[0] * counts[1], counts[1] * (counts[1] - 1) / 2]
    shell = 4 * math.pi * rk ** 2 / L ** 3 * math.sqrt(2 * math.pi) * width * frames
    g = H / (torch.tensor(per, dtype=torch.float64, device=dev)[:, None] * shell)
    ((g - (rk > 0.95).double()) ** 2).mean().backward()
    both = lambda x: 0.5 * (x + x.T)  # noqa: E731   (the gradient of a symmetric matrix)
    return {"g": g.detach(), "r0": r0.grad, "sigma": both(sig.grad), "epsilon": both(eps.grad)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "eval":
        return _exact_eval(case, seed)
    if kind == "md":
        return _exact_md(case, seed)
    if kind == "batch":
        return _exact_batch(case, seed)
    if kind == "adjoint":
        return _exact_adjoint(case, seed)
    return None         # whole numbers
