"""Performance cases of the MDDF library: the calls its users make, over the sizes they make them at.

A case is a dict of plain values.  `kind` says which entry point it goes through:

  mddf    mddf(trajectory, options) on frames in host memory
  cn      coordination_number(trajectory, options) on frames in host memory
  job     Job.submit_device + Job.finish on frames resident in device memory
  batch   submit_many: several systems at once, one job each
  served  Server: a mixed request stream over several resident systems

and `solute`/`solvent` what is counted: "globule" (a compact solute of one molecule), "chain" (an extended one),
"osmolyte" (many small solute molecules) or "self" (the solvent against itself), in "water" (3 atoms) or "urea"
(8 atoms).  Sizes are those of the repository's configurations, tests and benchmark: solutes of 120 to 20,000 atoms,
boxes of 24 to 150 A with water at 0.0334 molecules per cubic A, orthorhombic and triclinic (80 degrees), float32 and
float64 coordinates, 10 ideal-gas passes by default.
"""
import math

import numpy as np
import torch

import __graft_entry__

cm = __graft_entry__.load_package()

from complexmixtures_amd import _lib, synthetic  # noqa: E402
from complexmixtures_amd.results import setbin  # noqa: E402
from complexmixtures_amd.trajectory import unitcell_matrix  # noqa: E402

WATER_DENSITY = 0.0334
SIGMA = 0.3               # thermal jitter of the frames, A
GLOBULE_DENSITY = 0.0764  # atoms per cubic A of a compact solute (5,000 atoms in a 25 A sphere)


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def _case(**kw):
    c = dict(kind="job", solute="globule", solvent="water", n_solute=0, n_solvent=0, box=0.0, angle=90.0, dtype="f32",
             frames=1, passes=10, usecutoff=False, weights="one", groups=False)
    c.update(kw)
    return c


def listed():
    return [
        # the smallest call: a few hundred atoms, two frames, straight from host arrays (a quick look, a test, a small
        # selection); launches and host work are most of it
        _case(name="tiny_mddf", kind="mddf", solute="chain", n_solute=120, n_solvent=300, box=24.0, dtype="f64", frames=2),
        # a short trajectory of a small solvated chain, as read from a file: float64 host arrays
        _case(name="chain_mddf", kind="mddf", solute="chain", n_solute=1000, n_solvent=2000, box=40.0, dtype="f64",
              frames=20),
        # the headline workload: a protein-sized solute in a large water box, the trajectory resident in device memory
        _case(name="globule_mddf", n_solute=5000, n_solvent=40000, box=110.0, frames=120),
        # the largest solute and box of the served systems
        _case(name="large_mddf", n_solute=20000, n_solvent=112725, box=150.0, frames=16),
        # a cosolvent of 8 atoms around a polymer, triclinic cell, float64
        _case(name="polymer_urea", solute="chain", solvent="urea", n_solute=3000, n_solvent=12000, box=90.0, angle=80.0,
              dtype="f64", frames=20),
        # coordination numbers with custom groups, reweighted frames and a bulk shell, from host arrays
        _case(name="polymer_water_cn", kind="cn", solute="chain", n_solute=3000, n_solvent=15000, box=90.0, angle=80.0,
              dtype="f64", frames=20, passes=0, usecutoff=True, weights="two", groups=True),
        # a cosolvent against itself, with the ideal-gas passes
        _case(name="urea_self", solute="self", solvent="urea", n_solvent=12000, box=90.0, angle=80.0, dtype="f64",
              frames=20),
        # water against itself in a large box, coordination numbers only (the largest self requests of a served stream)
        _case(name="water_self", solute="self", n_solvent=33400, box=100.0, frames=24, passes=0),
        # the same question on a small box, with the ideal-gas passes
        _case(name="water_self_small", solute="self", n_solvent=901, box=30.0, frames=40),
        # many small solute molecules: 14-atom osmolytes in the water of an 84 A box
        _case(name="osmolyte_water", solute="osmolyte", n_solute=181, n_solvent=16667, box=84.42, frames=20),
        # uneven systems submitted together
        _case(name="batch", kind="batch", n_systems=12, frames=20, pool=11),
        # a mixed request stream: short and long requests, self and cross, with and without ideal-gas passes
        _case(name="served", kind="served", n_systems=6, n_requests=16, frames=40, pool=23),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mddf", "cn", "job", "job", "job", "self", "self", "osmolyte", "batch", "served"])
    dtype = rng.choice(["f32", "f64"])
    angle = rng.choice([90.0, 90.0, 80.0])
    passes = rng.choice([10, 10, rng.randint(1, 20)])
    weights = rng.choice(["one", "one", "two"])
    cut = rng.random() < 0.25
    if kind == "batch":
        return _case(kind="batch", n_systems=rng.randint(3, 12), frames=rng.randint(5, 20), pool=rng.randint(1, 10 ** 6))
    if kind == "served":
        return _case(kind="served", n_systems=rng.randint(2, 6), n_requests=rng.randint(4, 16), frames=rng.randint(5, 40),
                     pool=rng.randint(1, 10 ** 6))
    if kind in ("self", "osmolyte"):
        solvent = rng.choice(["water", "urea"]) if kind == "self" else "water"
        box = math.exp(rng.uniform(math.log(30.0), math.log(100.0 if solvent == "water" else 90.0)))
        cell = box ** 3 * (1.0 if angle == 90.0 else 0.95)
        n = max(20, int(cell * (WATER_DENSITY if solvent == "water" else 0.0172)))
        top = max(1, min(40, int(8e5 / n)))
        return _case(kind="job", solute=kind, solvent=solvent, n_solute=max(2, int(cell * 3e-4)) if kind == "osmolyte" else 0,
                     n_solvent=n, box=box, angle=angle, dtype=dtype, frames=rng.randint(max(1, top // 4), top),
                     passes=rng.choice([0, passes]), usecutoff=cut, weights=weights)
    solute = rng.choice(["globule", "chain"])
    solvent = rng.choice(["water", "water", "urea"])
    top = 110.0 if kind == "job" else 60.0
    box = math.exp(rng.uniform(math.log(26.0 if cut else 24.0), math.log(top)))
    if angle != 90.0:
        box = max(box, 30.0)
    cell = box ** 3 * (1.0 if angle == 90.0 else 0.95)
    most = min(20000, int(0.5 * GLOBULE_DENSITY * cell * (0.25 if solute == "chain" else 1.0)))
    n_solute = _logint(rng, 120, max(121, most))
    n_solvent = max(10, int(cell * (WATER_DENSITY if solvent == "water" else 0.0172)))
    atoms = n_solute + n_solvent * (3 if solvent == "water" else 8)
    frames = rng.randint(1, max(2, min(120, int(2.5e6 / atoms))))
    return _case(kind=kind, solute=solute, solvent=solvent, n_solute=n_solute, n_solvent=n_solvent, box=box, angle=angle,
                 dtype=dtype, frames=frames, passes=0 if kind == "cn" else passes, usecutoff=cut, weights=weights,
                 groups=kind != "job" and rng.random() < 0.25)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _cell(case):
    a = case["angle"]
    return unitcell_matrix(case["box"], case["box"], case["box"], a, a, a)


def _globule(rng, n, centre):
    """n atoms packed at the density of a compact solute: the points of a jittered lattice nearest to the centre, in
    rows (neighbours in the list are neighbours in space, as along a folded chain)."""
    h = GLOBULE_DENSITY ** (-1.0 / 3.0)
    m = int(math.ceil((3.0 * n / (4.0 * math.pi)) ** (1.0 / 3.0))) + 2
    k = np.arange(-m, m + 1, dtype=np.float64)
    p = np.stack(np.meshgrid(k, k, k, indexing="ij"), axis=-1).reshape(-1, 3)
    keep = np.sort(np.argsort((p * p).sum(axis=1), kind="stable")[:n])
    return centre + h * p[keep] + rng.normal(scale=0.35, size=(n, 3))


def _chain(rng, n, start):
    """An extended chain: 1.5 A bonds, directions correlated over about ten bonds."""
    d = rng.normal(size=(n, 3))
    w = np.exp(-np.arange(30) / 10.0)
    d = np.stack([np.convolve(d[:, k], w)[:n] for k in range(3)], axis=1)
    d *= 1.5 / np.linalg.norm(d, axis=1)[:, None]
    return start + np.cumsum(d, axis=0)


def _osmolyte():
    """14 sites: a central atom, four at 1.4 A, nine at 2.1 A from it."""
    k = np.arange(13) + 0.5
    z = 1.0 - 2.0 * k / 13.0
    a = math.pi * (1.0 + math.sqrt(5.0)) * k
    s = np.sqrt(1.0 - z * z)
    u = np.stack([s * np.cos(a), s * np.sin(a), z], axis=1)
    return np.concatenate([np.zeros((1, 3)), 1.4 * u[:4], 2.1 * u[4:]])


def _template(name):
    return {"water": synthetic.water_template, "urea": synthetic.urea_template, "osmolyte": _osmolyte}[name]()


def _frames(rng, base, nframes, dtype):
    """Frames: the base coordinates plus thermal jitter (a few draws, rolled over the atoms from frame to frame)."""
    base = base.astype(dtype)
    k = min(4, nframes)
    noise = rng.normal(scale=SIGMA, size=(k,) + base.shape).astype(dtype)
    x = np.empty((nframes,) + base.shape, dtype=dtype)
    for f in range(nframes):
        np.add(base, np.roll(noise[f % k], (f // k) * 7919, axis=0), out=x[f])
    return x


def _system(case, seed):
    """Host coordinates of a case's solute and solvent (the same array twice against itself) and its cell."""
    rng = np.random.default_rng([int(seed), 20261203])
    H = _cell(case)
    dtype = np.float32 if case["dtype"] == "f32" else np.float64
    centre = H @ np.full(3, 0.5)
    nv = case["n_solvent"]
    frac = rng.uniform(size=(nv, 3))
    if case["solute"] == "globule":
        # outside the solute
        r = (3.0 * case["n_solute"] / (4.0 * math.pi * GLOBULE_DENSITY)) ** (1.0 / 3.0) + 1.5
        for _ in range(64):
            bad = np.linalg.norm(frac @ H.T - centre, axis=1) < r
            if not bad.any():
                break
            frac[bad] = rng.uniform(size=(int(bad.sum()), 3))
    xv = synthetic.place_molecules(rng, _template(case["solvent"]), frac @ H.T)
    if case["solute"] == "self":
        x = _frames(rng, xv, case["frames"], dtype)
        return x, x, H
    if case["solute"] == "globule":
        xu = _globule(rng, case["n_solute"], centre)
    elif case["solute"] == "chain":
        xu = _chain(rng, case["n_solute"], H @ rng.uniform(size=3))
    else:
        xu = synthetic.place_molecules(rng, _template("osmolyte"), rng.uniform(size=(case["n_solute"], 3)) @ H.T)
    x = _frames(rng, np.concatenate([xu, xv]), case["frames"], dtype)
    return np.ascontiguousarray(x[:, :len(xu)]), np.ascontiguousarray(x[:, len(xu):]), H


def _shape(case):
    """(solute molecules, atoms each, solvent molecules, atoms each)"""
    nv = {"water": 3, "urea": 8}[case["solvent"]]
    if case["solute"] == "self":
        return case["n_solvent"], nv, case["n_solvent"], nv
    if case["solute"] == "osmolyte":
        return case["n_solute"], 14, case["n_solvent"], nv
    return 1, case["n_solute"], case["n_solvent"], nv


def _weights(case):
    w = np.ones(case["frames"])
    if case["weights"] == "two":
        w[case["frames"] // 2:] = 0.5
    return w


def _ranges(case):
    """dbulk, cutoff, binstep"""
    return (8.0, 11.0, 0.02) if case["usecutoff"] else (10.0, 10.0, 0.02)


def _job_kwargs(case, seed):
    mu, nu, mv, nv = _shape(case)
    dbulk, cutoff, step = _ranges(case)
    return dict(nmols_u=mu, natoms_per_mol_u=nu, nmols_v=mv, natoms_per_mol_v=nv, autocorrelation=case["solute"] == "self",
                irefatom=1, nbins=setbin(cutoff, step), binstep=step, cutoff=cutoff, dbulk=dbulk,
                usecutoff=case["usecutoff"], n_random_samples=max(1, case["passes"]),
                coordination_number_only=case["passes"] == 0, triclinic=case["angle"] != 90.0, seed=int(seed) + 1,
                n_groups_u=nu, n_groups_v=nu if case["solute"] == "self" else nv)


def _group_lists(n_atoms):
    """Custom groups of a solute: residues of 25 consecutive atoms (1-based indices)."""
    return [list(range(a + 1, min(a + 25, n_atoms) + 1)) for a in range(0, n_atoms, 25)]


def _pool_cases(case):
    """Systems of uneven size (solutes of 200 to 20,000 atoms, water boxes of 30 to 110 A)."""
    rng = np.random.default_rng([case["pool"], 7])
    subs = []
    for k in range(case["n_systems"]):
        box = float(rng.uniform(30.0, 110.0))
        n = int(min(0.4 * GLOBULE_DENSITY * box ** 3, math.exp(rng.uniform(math.log(200), math.log(20000)))))
        solute = ("globule", "chain")[k % 2]
        subs.append(_case(solute=solute, box=box, frames=case["frames"], n_solute=min(n, 4000) if solute == "chain" else n,
                          n_solvent=int(WATER_DENSITY * box ** 3)))
    return subs


def _request_cases(case, subs):
    """(system, request) pairs: 30% with ideal-gas passes, 20% of the water against itself, uneven lengths."""
    rng = np.random.default_rng([case["pool"], 11])
    reqs = []
    for _ in range(case["n_requests"]):
        k = int(rng.integers(len(subs)))
        s = dict(subs[k], frames=int(rng.integers(max(1, case["frames"] // 4), case["frames"] + 1)),
                 passes=10 if rng.random() < 0.3 else 0)
        if rng.random() < 0.2:
            s["solute"] = "self"
        reqs.append((k, s))
    return reqs


def _pool(case, seed):
    """The systems resident in device memory: (case, solute, solvent, cells)."""
    pool = []
    for k, sub in enumerate(_pool_cases(case)):
        xu, xv, H = _system(sub, int(seed) * 1000 + k)
        pool.append((sub, _lib.DeviceArray(xu), _lib.DeviceArray(xv), np.repeat(H[None], case["frames"], axis=0)))
    return pool


def prepare(case, seed):
    case = dict(case)
    if case["kind"] == "batch":
        pool = _pool(case, seed)
        return {"case": case, "pool": pool, "kw": [_job_kwargs(s, seed + k) for k, (s, _, _, _) in enumerate(pool)]}
    if case["kind"] == "served":
        pool = _pool(case, seed)
        reqs = []
        for i, (k, s) in enumerate(_request_cases(case, [p[0] for p in pool])):
            _, du, dv, cells = pool[k]
            reqs.append((s, dv if s["solute"] == "self" else du, dv, cells[:s["frames"]], _job_kwargs(s, seed + i)))
        return {"case": case, "pool": pool, "requests": reqs, "server": _lib.Server(4)}
    xu, xv, H = _system(case, seed)
    cells = np.repeat(H[None], case["frames"], axis=0)
    if case["kind"] == "job":
        du = _lib.DeviceArray(xu)
        dv = du if case["solute"] == "self" else _lib.DeviceArray(xv)
        return {"case": case, "du": du, "dv": dv, "cells": cells, "kw": _job_kwargs(case, seed),
                "frames": np.arange(1, case["frames"] + 1), "weights": _weights(case)}
    mu, nu, mv, nv = _shape(case)
    dbulk, cutoff, step = _ranges(case)
    groups = dict(group_atom_indices=_group_lists(nu), group_names=[str(k) for k in range(len(_group_lists(nu)))]) \
        if case["groups"] else {}
    solute = cm.AtomSelection(range(1, mu * nu + 1), nmols=mu, **groups)
    solvent = cm.AtomSelection(range(mu * nu + 1, mu * nu + mv * nv + 1), nmols=mv)
    rng_kw = dict(bulk_range=(dbulk, cutoff)) if case["usecutoff"] else dict(dbulk=dbulk)
    opts = cm.Options(binstep=step, n_random_samples=max(1, case["passes"]), seed=int(seed) + 1, irefatom=1, silent=True,
                      **rng_kw)
    return {"case": case, "trajectory": cm.MemoryTrajectory(xu, xv, cells, solute, solvent), "options": opts,
            "weights": None if case["weights"] == "one" else _weights(case)}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
RESULT_FIELDS = ("md_count", "md_count_random", "coordination_number", "coordination_number_random", "mddf", "kb",
                 "rdf_count", "rdf_count_random", "rdf", "kb_rdf", "solute_group_count", "solute_group_count_random",
                 "solvent_group_count", "solvent_group_count_random")


def _together(raws):
    """The outputs of several jobs: histograms one below the other, each job's solute groups as they are."""
    out = {k: np.stack([r[k] for r in raws]) for k in ("md_count", "md_count_random", "rdf_count", "rdf_count_random",
                                                        "hits_md", "hits_rdf", "hits_md_random", "hits_rdf_random")}
    out["volume_total"] = np.array([r["volume_total"] for r in raws])
    out["solvent_group_count"] = np.stack([r["solvent_group_count"] for r in raws])
    out["solvent_group_count_random"] = np.stack([r["solvent_group_count_random"] for r in raws])
    out["solute_group_count"] = [r["solute_group_count"] for r in raws]
    out["solute_group_count_random"] = [r["solute_group_count_random"] for r in raws]
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("mddf", "cn"):
        call = cm.mddf if kind == "mddf" else cm.coordination_number
        R = call(state["trajectory"], state["options"], frame_weights=state["weights"])
        out = {k: getattr(R, k) for k in RESULT_FIELDS}
        out["volume_total"] = float(R.volume.total)
        return out
    if kind == "job":
        job = _lib.Job(**state["kw"])
        job.submit_device(state["frames"], state["du"], state["dv"], 0, state["cells"], state["weights"])
        raw = job.finish()
        job.close()
        return raw
    if kind == "batch":
        n = case["frames"]
        jobs = [_lib.Job(**kw) for kw in state["kw"]]
        _lib.submit_many([(j, np.arange(1, n + 1), du, dv, 0, cells, np.ones(n))
                          for j, (_, du, dv, cells) in zip(jobs, state["pool"])])
        raws = [j.finish() for j in jobs]
        for j in jobs:
            j.close()
        return _together(raws)
    srv = state["server"]
    tickets = [srv.enqueue(np.arange(1, s["frames"] + 1), du, dv, 0, cells, np.ones(s["frames"]), **kw)
               for s, du, dv, cells, kw in state["requests"]]
    return _together([srv.wait(t)[0] for t in tickets])


# ---------------------------------------------------------------------------
# work and reference values
# ---------------------------------------------------------------------------
def _system_work(case):
    """Coordinates read once, counts written once; one distance (12 operations, 18 in a triclinic cell) for every pair
    within the cutoff at uniform density, in the real pass and in each ideal-gas pass."""
    mu, nu, mv, nv = _shape(case)
    dbulk, cutoff, step = _ranges(case)
    rc = cutoff if case["usecutoff"] else dbulk
    vol = abs(float(np.linalg.det(_cell(case))))
    share = 4.0 / 3.0 * math.pi * rc ** 3 / vol * mv * nv
    item = 4 if case["dtype"] == "f32" else 8
    coords = 3 * item * (mv * nv + (0 if case["solute"] == "self" else mu * nu))
    nbins = setbin(cutoff, step)
    pairs = share * nu * (mu * (0.5 if case["solute"] == "self" else 1.0) + case["passes"])
    return case["frames"] * coords + 8 * nbins * (4 + 2 * (nu + nv)), \
        case["frames"] * pairs * (12.0 if case["angle"] == 90.0 else 18.0)


def work(case):
    if case["kind"] in ("batch", "served"):
        subs = _pool_cases(case)
        if case["kind"] == "served":
            subs = [s for _, s in _request_cases(case, subs)]
        parts = [_system_work(s) for s in subs]
        return {"bytes": float(sum(p[0] for p in parts)), "flops": float(sum(p[1] for p in parts))}
    b, f = _system_work(case)
    return {"bytes": float(b), "flops": float(f)}


EXACT_PAIRS = 4e9   # atom pairs over all frames that the plain evaluation below takes on


def exact(case, seed):
    """The real-pass counts by an all-pairs evaluation in 64 bits (the ideal-gas passes have no value without the
    library's own random streams)."""
    if case["kind"] not in ("mddf", "cn", "job"):
        return None
    mu, nu, mv, nv = _shape(case)
    if float(mu * nu) * mv * nv * case["frames"] > EXACT_PAIRS:
        return None
    same = case["solute"] == "self"
    dbulk, cutoff, step = _ranges(case)
    rc = cutoff if case["usecutoff"] else dbulk
    nbins = setbin(cutoff, step)
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    xu, xv, H = _system(case, seed)
    w = _weights(case)
    Ht = torch.from_numpy(H).to(dev, torch.float64)
    Hi = torch.linalg.inv(Ht)
    md = torch.zeros(nbins, dtype=torch.float64, device=dev)
    rdf = torch.zeros_like(md)
    gu = torch.zeros(nu, nbins, dtype=torch.float64, device=dev)
    gv = torch.zeros(nv, nbins, dtype=torch.float64, device=dev)

    def bins(d):
        return torch.clamp(torch.ceil(d / step).long(), min=1) - 1

    for f in range(case["frames"]):
        U = torch.from_numpy(xu[f]).to(dev, torch.float64)
        V = torch.from_numpy(xv[f]).to(dev, torch.float64).reshape(mv, nv, 3)
        block = max(1, int(2e7 / (nu * mv * nv)))
        for u0 in range(0, mu, block):
            u1 = min(mu, u0 + block)
            S = U[u0 * nu:u1 * nu].reshape(u1 - u0, nu, 3)
            # [solute molecule][solvent molecule][solute atom][solvent atom]
            d = V[None, :, None, :, :] - S[:, None, :, None, :]
            d = d - torch.round(d @ Hi.T) @ Ht.T
            d = d.square().sum(-1).sqrt()
            if same:
                k = torch.arange(u0, u1, device=dev)
                d[k - u0, k] = math.inf
            m, at = d.reshape(u1 - u0, mv, nu * nv).min(-1)
            hit = m <= rc
            b, i, j = bins(m[hit]), torch.div(at[hit], nv, rounding_mode="floor"), at[hit] % nv
            one = torch.full_like(m[hit], float(w[f]))
            md.index_add_(0, b, one)
            if same:
                gu.view(-1).index_add_(0, i * nbins + b, one / 2)
                gu.view(-1).index_add_(0, j * nbins + b, one / 2)
            else:
                gu.view(-1).index_add_(0, i * nbins + b, one)
                gv.view(-1).index_add_(0, j * nbins + b, one)
            r = d[..., 0].amin(-1)
            rdf.index_add_(0, bins(r[r <= rc]), torch.full_like(r[r <= rc], float(w[f])))
    md, rdf, gu, gv = (t.cpu().numpy() for t in (md, rdf, gu, gv))
    if case["groups"]:
        gu = np.stack([gu[[a - 1 for a in g]].sum(axis=0) for g in _group_lists(nu)])
    vol = abs(float(np.linalg.det(H)))
    if case["kind"] == "job":
        out = {"md_count": md, "rdf_count": rdf, "solute_group_count": gu,
               "solvent_group_count": np.zeros((nu, nbins)) if same else gv, "volume_total": vol * float(w.sum()),
               "hits_md": None, "hits_rdf": None}
        return {**out, **{k: None for k in ("md_count_random", "rdf_count_random", "solute_group_count_random",
                                            "solvent_group_count_random", "hits_md_random", "hits_rdf_random")}}
    q = mu * float(w.sum())
    out = {k: None for k in RESULT_FIELDS}
    out.update(md_count=md / q, rdf_count=rdf / q, solute_group_count=gu / q, solvent_group_count=gv / q,
               coordination_number=np.cumsum(md / q), volume_total=vol)
    return out
