"""Timed cases of the molecular-dynamics framework.

Each case is work that a user's program has the library do through its public
Python entry points (``Context``, ``Batch``, ``Server``): a call that advances
a system and reads its state back (what a trajectory frame costs), forces and
energies of given coordinates, a minimization, a stream of served jobs.  The
systems are the library's own synthetic workloads (``configs``): Go and AICG2+
chains, lipid patches, HPS slabs, an open HPS cluster, a replica ensemble and
a large condensate.

* ``listed()``  the fixed cases
* ``draw(rng)`` one more case of the same ranges
* ``prepare``   systems, start states and the handle a program would hold
* ``run``       one pass
* ``work``      bytes and operations a pass cannot do without
* ``exact``     the same results in FP64 torch, where they have such a value
"""
import math

import numpy as np
import torch

from opencafemol_amd import abi, configs
from opencafemol_amd.context import Batch, Context, Server

KB = 1.380649e-23 * 6.02214076e23 / 1000.0   # kJ/mol/K
FRAME = abi.STATE_POSITIONS | abi.STATE_VELOCITIES
FRAME_ENERGY = FRAME | abi.STATE_ENERGY
EVAL = abi.STATE_FORCES | abi.STATE_ENERGY
# trajectories up to this length are compared with an FP64 integration; longer
# ones of these chaotic systems have no value that another arithmetic reaches
EXACT_STEPS = 20


# ------------------------------------------------------------------- cases
def listed():
    return [
        # the shortest call: a few steps of a 62-bead protein between reads of
        # its state (steered runs, replica exchange attempts)
        {"name": "go_62_call", "do": "steps", "model": "go", "beads": 62, "steps": 20, "energy": False},
        # the same protein's production run: a frame with energies per 1,000 steps
        {"name": "go_62_frame", "do": "steps", "model": "go", "beads": 62, "steps": 1000, "energy": True},
        # AICG2+ protein (Gaussian bonds, flexible local terms), an odd size
        {"name": "aicg2_213", "do": "steps", "model": "aicg2", "beads": 213, "steps": 500, "energy": True},
        # replica ensemble on a temperature ladder, every replica read back
        {"name": "replicas_256", "do": "replicas", "replicas": 256, "beads": 500, "steps": 2000},
        # membrane patch: WCA, iSoLF and table potentials, 3,000 beads
        {"name": "lipids_3000", "do": "steps", "model": "lipids", "beads": 3000, "steps": 400, "energy": False},
        # HPS slab at the small end of the served sizes
        {"name": "slab_2100", "do": "steps", "model": "slab", "beads": 2100, "steps": 500, "energy": True},
        # the 14,000-bead slab: production stretch with frame
        {"name": "slab_14000", "do": "steps", "model": "slab", "beads": 14000, "steps": 1000, "energy": False},
        # open boundaries, no box: a 21,000-bead HPS cluster
        {"name": "cluster_21000", "do": "steps", "model": "cluster", "beads": 21000, "steps": 300, "energy": False},
        # the 1,000,000-bead condensate (0.3 nm skin, lists at most 20 steps old)
        {"name": "condensate_1m", "do": "steps", "model": "condensate", "beads": 1000000, "steps": 200,
         "energy": False},
        # forces and energies of stored frames (re-analysis of a trajectory)
        {"name": "evaluate_14000", "do": "evaluate", "model": "slab", "beads": 14000},
        # relaxation of a packed start before a run
        {"name": "minimize_7000", "do": "minimize", "model": "slab", "beads": 7000, "iterations": 25},
        # a stream of served jobs: Go chains and HPS slabs with frames
        {"name": "served_mix", "do": "served", "jobs": 5, "beads": 6000, "steps": 4000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["steps", "steps", "steps", "steps", "evaluate", "replicas", "minimize", "served"])
    model = rng.choice(["go", "aicg2", "lipids", "slab", "slab", "cluster", "condensate"])
    beads = {"go": (30, 900), "aicg2": (30, 500), "lipids": (600, 12000), "slab": (2000, 40000),
             "cluster": (3000, 40000), "condensate": (50000, 900000)}[model]
    n = _log_int(rng, *beads)
    if kind == "steps":
        steps = _log_int(rng, 20, 200 if model == "condensate" else 1000)
        return {"do": "steps", "model": model, "beads": n, "steps": steps, "energy": rng.random() < 0.5}
    if kind == "evaluate":
        return {"do": "evaluate", "model": model, "beads": n}
    if kind == "replicas":
        return {"do": "replicas", "replicas": _log_int(rng, 4, 256), "beads": rng.randint(80, 500),
                "steps": _log_int(rng, 100, 2000)}
    if kind == "minimize":
        model = rng.choice(["lipids", "slab", "cluster"])
        return {"do": "minimize", "model": model, "beads": _log_int(rng, 2000, 14000), "iterations": rng.randint(10, 30)}
    return {"do": "served", "jobs": rng.randint(2, 5), "beads": _log_int(rng, 2000, 8000),
            "steps": 1000 * rng.randint(1, 4)}


# ------------------------------------------------------------------ inputs
def _serpentine(n_chains, chain_len, extent):
    """Chains laid along one winding path: rows of beads 0.38 nm apart (the
    bond length), rows 3 bonds apart and layers 2 bonds apart with the turns'
    beads on the way, so that every bond starts at its length; one empty site
    between chains.  About 2.9 beads/nm^3 in the layer it fills."""
    b = 0.38
    sites = n_chains * (chain_len + 1)
    nx, ny = max(2, int(extent[0] // b) - 1), max(1, int(extent[1] // (3 * b)))
    # one layer: rows run back and forth, two beads join a row to the next
    row = np.arange(nx)
    layer = []
    for r in range(ny):
        x = row if r % 2 == 0 else row[::-1]
        layer.append(np.stack([x, np.full(nx, 3 * r)], 1))
        if r + 1 < ny:
            layer.append(np.stack([np.full(2, x[-1]), 3 * r + np.array([1, 2])], 1))
    layer = np.concatenate(layer)
    nz = -(-sites // (len(layer) + 1))
    z = np.repeat(2 * np.arange(nz), len(layer) + 1)
    turned = [np.concatenate([p, p[-1:]]) for p in (layer, layer[::-1])]   # and one bead joins the layers
    xy = np.concatenate([turned[k % 2] for k in range(nz)])
    z[np.arange(1, nz + 1) * (len(layer) + 1) - 1] += 1
    path = np.concatenate([xy, z[:, None]], 1)[:sites].astype(np.float64) * b
    keep = np.arange(sites) % (chain_len + 1) < chain_len
    return path[keep]


def _hps(n_chains, chain_len, box, seed, open_boundary=False):
    x = _serpentine(n_chains, chain_len, box)
    if not open_boundary:
        x[:, 2] += 0.5 * (box[2] - x[:, 2].max())
    s, it, _ = configs.hps_slab(n_chains=n_chains, chain_len=chain_len, box=box, seed=seed, positions=x)
    if open_boundary:
        s.box = None
        for f in s.forces:
            f.use_periodic = False
    return s, it, x


def _lipids(beads, seed):
    """Stacked bilayers: lipids upright on a 1.2 nm square lattice, heads
    facing heads and tails facing tails."""
    per = max(6, round((beads / 3.0) ** (1.0 / 3.0)))
    box = (1.2 * per, 1.2 * per, 1.95 * per)
    s, it, _ = configs.lipid_patch(per ** 3, box=box, seed=seed)
    g = np.stack(np.meshgrid(*[np.arange(per)] * 3, indexing="ij"), -1).reshape(-1, 3)
    up = np.where(g[:, 2] % 2 == 0, 1.0, -1.0)
    centers = (g + 0.5) * np.array([1.2, 1.2, 1.95])
    x = np.repeat(centers, 3, axis=0)
    x[:, 2] += (up[:, None] * np.array([-0.55, 0.0, 0.55])).reshape(-1)
    rng = np.random.default_rng([seed, 11])
    return s, it, x + rng.uniform(-0.02, 0.02, size=x.shape)


def _system(model, beads, seed):
    """(system, integrator, positions) of about `beads` beads."""
    if model == "go":
        return configs.go_chain(beads, seed=seed)
    if model == "aicg2":
        return configs.aicg2_chain(beads, seed=seed)
    if model == "lipids":
        return _lipids(beads, seed)
    if model == "slab":
        chains = max(1, round(beads / 140))
        xy = max(8.0, 15.0 * math.sqrt(chains * 140 / 14000.0))
        return _hps(chains, 140, (xy, xy, 150.0), seed)
    if model == "cluster":
        xy = max(4.0, 12.0 * math.sqrt(beads / 21000.0))
        return _hps(max(1, round(beads / 140)), 140, (xy, xy, 1.0e4), seed, open_boundary=True)
    if model == "condensate":
        scale = (beads / 1.0e6) ** (1.0 / 3.0)
        chain = 1000 if beads >= 200000 else 500
        return _hps(max(1, round(beads / chain)), chain, (60.0 * scale, 60.0 * scale, 600.0 * scale), seed)
    raise ValueError(model)


def _options(model):
    return {"skin": 0.3, "rebuild_interval": 20} if model == "condensate" else {}


def _velocities(system, integrator, seed):
    """Maxwell-Boltzmann velocities (nm/ps) from the seed."""
    rng = np.random.default_rng([seed, 17])
    m = np.asarray(system.masses, dtype=np.float64)
    return rng.normal(size=(system.n, 3)) * np.sqrt(KB * integrator.temperature / m)[:, None]


def _frames(x, seed, count=3):
    """Stored frames around x: thermal displacements of 0.02 nm."""
    rng = np.random.default_rng([seed, 23])
    return [x + rng.normal(scale=0.02, size=x.shape) for _ in range(count)]


def _replica_systems(case, seed):
    """Proteins of uneven length, each on a ladder of temperatures and with a
    noise seed of its own."""
    rng = np.random.default_rng([case["beads"], case["replicas"]])   # the sizes go with the case
    n = case["replicas"]
    proteins = max(1, min(16, n // 4))
    sizes = rng.integers(50, case["beads"] + 1, proteins)
    sizes[0] = case["beads"]
    chains = [configs.go_chain(int(k), seed=seed * 97 + p) for p, k in enumerate(sizes)]
    temps = configs.temperature_ladder(n)
    out = []
    for r in range(n):
        s, it, x = chains[r % proteins]
        out.append((s, type(it)(temps[r], it.friction, it.dt, it.seed + 1000003 * r), x))
    return out


def _jobs(case, seed):
    rng = np.random.default_rng([case["beads"], case["jobs"]])   # the sizes go with the case
    jobs = []
    for k in range(case["jobs"]):
        if k % 5 in (1, 3):   # two of five are slabs
            s, it, x = _system("slab", int(rng.integers(case["beads"] // 2, case["beads"] + 1)), seed * 31 + k)
        else:
            s, it, x = configs.go_chain(int(rng.integers(50, 301)), seed=seed * 31 + k)
        steps = case["steps"] if k % 2 == 0 else case["steps"] // 2
        jobs.append({"system": s, "integrator": it, "positions": x, "velocities": _velocities(s, it, seed + k),
                     "nsteps": steps, "frame_interval": 500})
    return jobs


def prepare(case, seed):
    """The handle and inputs a program holds before the timed call."""
    do = case["do"]
    if do == "steps":
        s, it, x = _system(case["model"], case["beads"], seed)
        ctx = Context(s, it, **_options(case["model"]))
        ctx.set_positions(x)
        ctx.set_velocities(_velocities(s, it, seed))
        ctx.prepare(case["steps"])
        return {"do": do, "ctx": ctx, "steps": case["steps"], "what": FRAME_ENERGY if case["energy"] else FRAME}
    if do == "evaluate":
        s, it, x = _system(case["model"], case["beads"], seed)
        ctx = Context(s, it, **_options(case["model"]))
        frames = _frames(x, seed)
        ctx.set_positions(frames[-1])
        ctx.prepare(1)
        return {"do": do, "ctx": ctx, "frames": frames, "next": 0}
    if do == "minimize":
        if case["model"] == "slab":   # chains packed on a lattice, the start that needs it
            s, it, x = configs.hps_slab_of_size(case["beads"], seed=seed)
        else:
            s, it, x = _system(case["model"], case["beads"], seed)
            x = _frames(x, seed, 1)[0]
        ctx = Context(s, it, **_options(case["model"]))
        ctx.set_positions(x)
        ctx.prepare(1)
        return {"do": do, "ctx": ctx, "x": x, "iterations": case["iterations"]}
    if do == "replicas":
        reps = _replica_systems(case, seed)
        b = Batch([r[0] for r in reps], [r[1] for r in reps])
        for k, (s, it, x) in enumerate(reps):
            b.set_positions(k, x)
            b.set_velocities(k, _velocities(s, it, seed * 1009 + k))
        b.prepare(case["steps"])
        return {"do": do, "batch": b, "n": len(reps), "steps": case["steps"]}
    if do == "served":
        return {"do": do, "server": Server(), "jobs": _jobs(case, seed)}
    raise ValueError(do)


# -------------------------------------------------------------------- pass
def run(state):
    do = state["do"]
    if do == "steps":
        ctx = state["ctx"]
        ctx.step(state["steps"])
        return _numbers(ctx.get_state(state["what"]))
    if do == "evaluate":
        ctx = state["ctx"]
        x = state["frames"][state["next"]]
        state["next"] = (state["next"] + 1) % len(state["frames"])
        ctx.set_positions(x)
        return _numbers(ctx.get_state(EVAL))
    if do == "minimize":
        ctx = state["ctx"]
        ctx.set_positions(state["x"])
        ctx.minimize(0.1, state["iterations"])
        return _numbers(ctx.get_state(abi.STATE_POSITIONS))
    if do == "replicas":
        b = state["batch"]
        b.step(state["steps"])
        got = [b.state(k, FRAME) for k in range(state["n"])]
        return {"positions": np.concatenate([g["positions"] for g in got]),
                "velocities": np.concatenate([g["velocities"] for g in got])}
    srv = state["server"]
    frames = []
    ids = [srv.submit(j["system"], j["integrator"], j["positions"], velocities=j["velocities"],
                      nsteps=j["nsteps"], frame_interval=j["frame_interval"]) for j in state["jobs"]]
    done = srv.drain(ids, on_frame=lambda job, step, x: frames.append((job, step, x)))
    frames.sort(key=lambda f: f[:2])
    return {"positions": np.concatenate([done[j]["positions"] for j in ids]),
            "velocities": np.concatenate([done[j]["velocities"] for j in ids]),
            "frames": np.concatenate([f[2] for f in frames])}


def _numbers(st):
    """The arrays and energies of a state (its step count depends on how often
    the pass ran before and is left out)."""
    out = {k: st[k] for k in ("positions", "velocities", "forces") if k in st}
    if "potential" in st:
        out["energy"] = np.concatenate([st["energy_by_group"], [st["potential"], st["kinetic"]]])
    return out


# -------------------------------------------------------------------- work
# Per bead and step: terms and pairs inside the cutoffs of each model, with
# the operations of one bonded term (~60) and one pair (~45); the integrator
# and its noise take ~120 operations per bead.
PAIRS = {"go": 12, "aicg2": 12, "lipids": 25, "slab": 70, "cluster": 70, "condensate": 85}
TERMS = {"go": 4, "aicg2": 7, "lipids": 1, "slab": 1, "cluster": 1, "condensate": 1}


def work(case):
    do = case["do"]

    def flops(model, beads):
        return beads * (45.0 * PAIRS[model] + 60.0 * TERMS[model])

    if do == "steps":
        n = case["beads"]
        return {"bytes": 96.0 * n, "flops": case["steps"] * (flops(case["model"], n) + 120.0 * n)}
    if do == "evaluate":
        n = case["beads"]
        return {"bytes": 48.0 * n, "flops": 2.0 * flops(case["model"], n)}
    if do == "minimize":
        n = case["beads"]
        return {"bytes": 48.0 * n, "flops": case["iterations"] * 2.0 * flops(case["model"], n)}
    if do == "replicas":
        n = case["replicas"] * (50 + case["beads"]) / 2.0
        return {"bytes": 96.0 * n, "flops": case["steps"] * (flops("go", n) + 120.0 * n)}
    b = f = 0.0
    for k in range(case["jobs"]):
        model, n = ("slab", 0.75 * case["beads"]) if k % 5 in (1, 3) else ("go", 175)
        steps = case["steps"] if k % 2 == 0 else case["steps"] // 2
        b += 96.0 * n + 24.0 * n * (steps // 500)
        f += steps * (flops(model, n) + 120.0 * n)
    return {"bytes": b, "flops": f}


# ------------------------------------------------------------------- exact
def exact(case, seed):
    """FP64 values of the first pass: forces and energies, and trajectories of
    up to EXACT_STEPS steps."""
    if case["do"] == "evaluate" and case["model"] != "condensate":
        s, it, x = _system(case["model"], case["beads"], seed)
        f = _Field(s)
        x = f.tensor(_frames(x, seed)[0])
        force, e = f.force(x, f.pairs(x, 0.0))
        return {"forces": force, "energy": torch.cat([e, e.sum()[None], torch.zeros(1, dtype=e.dtype, device=e.device)])}
    if case["do"] == "steps" and case["steps"] <= EXACT_STEPS and case["model"] != "condensate":
        s, it, x = _system(case["model"], case["beads"], seed)
        f = _Field(s)
        x, v, e = _integrate(f, it, f.tensor(x), f.tensor(_velocities(s, it, seed)), case["steps"])
        out = {"positions": x, "velocities": v}
        if case["energy"]:
            ke = 0.5 * (f.mass[:, None] * v * v).sum()
            out["energy"] = torch.cat([e, e.sum()[None], ke[None]])
        return out
    return None


def _philox(counter, key):
    """Philox4x32-10 on int64 tensors holding 32-bit words."""
    mask = 0xFFFFFFFF
    c = list(counter)
    k0, k1 = key

    def mul(a, b):   # 32 x 32 -> (high, low) without leaving 63 bits
        lo = a * (b & 0xFFFF)
        hi = a * (b >> 16)
        t = hi + (lo >> 16)
        return t >> 16, ((t & 0xFFFF) << 16) | (lo & 0xFFFF)

    for _ in range(10):
        h0, l0 = mul(c[0], 0xD2511F53)
        h1, l1 = mul(c[2], 0xCD9E8D57)
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
    return c


def _noise(seed, step, n, device):
    """Three N(0,1) samples per bead: Box-Muller on the top 24 bits of the
    words counted by (step, bead)."""
    bead = torch.arange(n, dtype=torch.int64, device=device)
    zero = torch.zeros_like(bead)
    c = _philox((zero + (step & 0xFFFFFFFF), zero + (step >> 32), bead, zero), (seed & 0xFFFFFFFF, seed >> 32))
    u = [((w >> 8).to(torch.float64) + 0.5) * 2.0 ** -24 for w in c]
    r0, r1 = torch.sqrt(-2.0 * torch.log(u[0])), torch.sqrt(-2.0 * torch.log(u[2]))
    a0, a1 = 2.0 * math.pi * u[1], 2.0 * math.pi * u[3]
    return torch.stack([r0 * torch.cos(a0), r0 * torch.sin(a0), r1 * torch.cos(a1)], 1)


def _integrate(field, it, x, v, steps):
    """BAOAB: kick, drift, Ornstein-Uhlenbeck, drift, kick."""
    dt, m = it.dt, field.mass[:, None]
    c1 = math.exp(-it.friction * dt)
    sig = torch.sqrt(KB * it.temperature * (1.0 - c1 * c1) / m)
    skin = 0.5
    built = x
    pairs = field.pairs(x, skin)
    force, e = field.force(x, pairs)
    for step in range(steps):
        v = v + 0.5 * dt * force / m
        x = x + 0.5 * dt * v
        v = c1 * v + sig * _noise(it.seed, step, x.shape[0], x.device)
        x = x + 0.5 * dt * v
        if float((x - built).square().sum(1).max()) > 0.24 * skin * skin:
            built, pairs = x, field.pairs(x, skin)
        force, e = field.force(x, pairs)
        v = v + 0.5 * dt * force / m
    return x, v, e


class _Field:
    """A system's potential in FP64 torch; forces by differentiation."""

    def __init__(self, system):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.s = system
        self.mass = self.tensor(system.masses)
        self.box = None if system.box is None else self.tensor(system.box)

    def tensor(self, a, dtype=torch.float64):
        return torch.as_tensor(np.ascontiguousarray(a), dtype=dtype, device=self.dev)

    def image(self, d, periodic):
        if not periodic or self.box is None:
            return d
        return d - self.box * torch.round(d / self.box)

    def pairs(self, x, skin):
        """Per nonbonded force: the participating, allowed, not excluded pairs
        within its cutoff (+ skin)."""
        out = []
        n = self.s.n
        for f in self.s.forces:
            if f.kind < abi.EXCLUDED_VOLUME:
                out.append(None)
                continue
            cat = np.zeros(n, np.int64) if f.category is None else np.asarray(f.category, np.int64)
            members = self.tensor(np.nonzero(cat >= 0)[0], torch.int64)
            cat = self.tensor(cat, torch.int64)
            xm = x[members]
            rl2 = (f.cutoff + skin) ** 2
            rows = max(1, int(2e7 // max(1, len(members))))
            found = []
            for at in range(0, len(members), rows):
                d = self.image(xm[at:at + rows, None, :] - xm[None, :, :], f.use_periodic)
                near = (d * d).sum(-1) < rl2
                i, j = torch.nonzero(near, as_tuple=True)
                i = i + at
                keep = i < j
                found.append((members[i[keep]], members[j[keep]]))
            i, j = (torch.cat([p[k] for p in found]) for k in (0, 1))
            if f.allow is not None:
                allow = self.tensor(f.allow, torch.int64)
                keep = allow[cat[i], cat[j]] != 0
                i, j = i[keep], j[keep]
            if f.exclusions is not None and np.size(f.exclusions):
                ex = np.sort(np.asarray(f.exclusions, np.int64).reshape(-1, 2), axis=1)
                keep = ~torch.isin(i * n + j, self.tensor(ex[:, 0] * n + ex[:, 1], torch.int64))
                i, j = i[keep], j[keep]
            out.append((i, j))
        return out

    def force(self, x, pairs):
        """(forces, energy per group)."""
        x = x.detach().requires_grad_(True)
        e = torch.zeros(32, dtype=torch.float64, device=self.dev)
        for f, p in zip(self.s.forces, pairs):
            v = self.bonded(f, x) if p is None else self.nonbonded(f, x, *p)
            e = e + torch.nn.functional.one_hot(torch.tensor(f.group, device=self.dev), 32) * v.sum()
        (g,) = torch.autograd.grad(e.sum(), x)
        return -g, e.detach()

    def bonded(self, f, x):
        idx = self.tensor(f.indices, torch.int64)
        p = self.tensor(f.params).reshape(len(idx), -1)
        d = [self.image(x[idx[:, k + 1]] - x[idx[:, k]], f.use_periodic) for k in range(idx.shape[1] - 1)]
        if idx.shape[1] == 2:
            r = d[0].norm(dim=1)
            if f.kind == abi.HARMONIC_BOND:
                return 0.5 * p[:, 1] * (r - p[:, 0]) ** 2
            if f.kind == abi.GAUSSIAN_BOND:
                return p[:, 0] * torch.exp(-0.5 * ((r - p[:, 1]) / p[:, 2]) ** 2)
            q = p[:, 1] / r
            return p[:, 0] * (5.0 * q ** 12 - 6.0 * q ** 10)
        if idx.shape[1] == 3:
            th = torch.atan2(torch.linalg.cross(-d[0], d[1]).norm(dim=1), -(d[0] * d[1]).sum(1))
            if f.kind == abi.HARMONIC_ANGLE:
                return 0.5 * p[:, 1] * (th - p[:, 0]) ** 2
            return p[:, 0] * self.local_angle(np.asarray(f.globals, np.float64), th)
        n1, n2 = torch.linalg.cross(d[0], d[1]), torch.linalg.cross(d[1], d[2])
        phi = torch.atan2(d[1].norm(dim=1) * (d[0] * n2).sum(1), (n1 * n2).sum(1))
        if f.kind == abi.GAUSSIAN_DIHEDRAL:
            a = phi - p[:, 1]
            a = a - 2.0 * math.pi * torch.floor((a + math.pi) / (2.0 * math.pi))
            return p[:, 0] * torch.exp(-0.5 * (a / p[:, 2]) ** 2)
        c = [float(v) for v in f.globals]
        u = c[0] - c[7] + sum(c[2 * k - 1] * torch.cos(k * phi) + c[2 * k] * torch.sin(k * phi) for k in (1, 2, 3))
        return p[:, 0] * u

    def local_angle(self, g, th):
        """Natural cubic spline through 10 knots, walls of slope 30 outside."""
        y, tmin, tmax, emin = g[:10], g[10], g[11], g[12]
        h = (tmax - tmin) / 9.0
        a = np.eye(10)
        b = np.zeros(10)
        for k in range(1, 9):
            a[k, k - 1:k + 2] = (1.0, 4.0, 1.0)
            b[k] = 6.0 * (y[k - 1] - 2.0 * y[k] + y[k + 1]) / (h * h)
        y, y2 = self.tensor(y), self.tensor(np.linalg.solve(a, b))
        lo = torch.clamp(torch.floor((th.detach() - tmin) / h), 0, 8).to(torch.int64)
        B = (th - (tmin + lo * h)) / h
        A = 1.0 - B
        s = A * y[lo] + B * y[lo + 1] + ((A ** 3 - A) * y2[lo] + (B ** 3 - B) * y2[lo + 1]) * h * h / 6.0
        u = torch.where((th >= tmin) & (th <= tmax), s, torch.zeros_like(s))
        u = u + torch.where(th <= tmin, 30.0 * (tmin - th) + y[0], torch.zeros_like(s))
        u = u + torch.where(th >= tmax, 30.0 * (th - tmax) + y[9], torch.zeros_like(s))
        return u - emin

    def nonbonded(self, f, x, i, j):
        d = self.image(x[j] - x[i], f.use_periodic)
        r2 = (d * d).sum(1)
        keep = r2.detach() < f.cutoff ** 2
        i, j, r2 = i[keep], j[keep], r2[keep]
        r = torch.sqrt(r2)
        g = [] if f.globals is None else [float(v) for v in f.globals]
        pp = None if f.particle_params is None else self.tensor(f.particle_params).reshape(self.s.n, -1)
        mean = lambda k: 0.5 * (pp[i, k] + pp[j, k])  # noqa: E731
        zero = torch.zeros_like(r)
        rmin = 2.0 ** (1.0 / 6.0)
        if f.kind == abi.EXCLUDED_VOLUME:
            s = pp[i, 0] + pp[j, 0]
            return g[0] * ((s / r) ** 12 - (s / f.cutoff) ** 12)
        if f.kind == abi.DEBYE_HUCKEL:
            return pp[i, 0] * pp[j, 0] * g[0] * (torch.exp(-r / g[1]) / r - g[2])
        if f.kind == abi.ISOLF_ATTRACTIVE:
            sig, om, eps = mean(0), mean(2), torch.sqrt(pp[i, 1] * pp[j, 1])
            t = (r - rmin * sig) / om
            tail = torch.where(t <= 1.0, torch.cos(0.5 * math.pi * t) ** 2, zero)
            return -eps * torch.where(t <= 0.0, zero + 1.0, tail)
        if f.kind in (abi.LJ_REPULSIVE, abi.LJ_ATTRACTIVE):
            eps, sig = mean(0), mean(1)
        elif f.kind == abi.WCA:
            eps, sig = torch.sqrt(pp[i, 1] * pp[j, 1]), mean(0)
        else:
            eps, sig = zero + g[1], zero + g[0]
        s6 = (sig / r) ** 6
        lj = 4.0 * eps * (s6 * s6 - s6)
        inner = r <= rmin * sig
        if f.kind in (abi.LJ_REPULSIVE, abi.WCA):
            return torch.where(inner, lj + eps, zero)
        if f.kind == abi.UNIFORM_WCA:
            return lj + eps
        u = torch.where(inner, -eps, lj)
        if f.switch_distance > 0:
            t = torch.clamp((r - f.switch_distance) / (f.cutoff - f.switch_distance), min=0.0)
            u = u * (1.0 - t ** 3 * (10.0 - 15.0 * t + 6.0 * t * t))
        return u
