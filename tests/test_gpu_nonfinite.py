"""Coordinates that are not numbers.  A solute atom with
one takes part in no distance, as in the FP64 oracle; so does a solvent molecule
whose atoms all have one, in the real pass and as the source of placed copies.
A molecule with one such atom has no centre and counts as if all its atoms had.
Counts equal bit for bit (unit weights: exact)."""
import numpy as np
import pytest

from conftest import assert_raw_equal, gpu_raw, oracle_raw

pytestmark = pytest.mark.gpu

NU, MV, BOX, FRAMES = 70, 120, 24.0, 2
BAD = [(1, 2), (7, 0), (30, 1), (31, 2), (90, 0)]   # molecule (or solute atom), coordinate


def _traj(pkg, nv, triclinic, dtype, where, whole, value):
    """Solute atoms about the cell's origin, where an undefined position must not appear as a defined one."""
    import complexmixtures_amd.synthetic as S
    from complexmixtures_amd.trajectory import unitcell_matrix
    rng = np.random.default_rng([nv, int(triclinic)])
    H = unitcell_matrix(BOX, BOX, BOX, *((80.0, 85.0, 95.0) if triclinic else (90.0, 90.0, 90.0)))
    xu = rng.normal(scale=3.0, size=(1, NU, 3)) + rng.normal(scale=0.2, size=(FRAMES, NU, 3))
    mol = np.concatenate([np.zeros((1, 3)), rng.normal(scale=0.8, size=(nv - 1, 3))])
    xv = S.place_molecules(rng, mol, rng.uniform(size=(MV, 3)) @ H.T)
    xv = xv + rng.normal(scale=0.1, size=(FRAMES,) + xv.shape)
    for m, k in BAD:
        if where == "solute":
            xu[0, m % NU, k] = value
        elif whole:
            xv[1, m * nv:(m + 1) * nv] = value
        else:
            xv[1, m * nv + m % nv, k] = value
    su = pkg.AtomSelection(list(range(1, NU + 1)), nmols=1)
    sv = pkg.AtomSelection(list(range(NU + 1, NU + MV * nv + 1)), nmols=MV)
    return pkg.MemoryTrajectory(xu.astype(dtype), xv.astype(dtype), np.repeat(H[None], FRAMES, axis=0), su, sv)


def _options(pkg, usecutoff):
    kw = dict(bulk_range=(6.0, 9.0)) if usecutoff else dict(dbulk=9.0)
    return pkg.Options(n_random_samples=9, seed=29, silent=True, **kw)


@pytest.mark.parametrize("where", ["solute", "solvent"])
@pytest.mark.parametrize("nv,triclinic,dtype,value,usecutoff", [
    (1, False, np.float32, np.nan, False), (3, False, np.float32, np.nan, False), (3, True, np.float64, np.inf, True),
    (3, False, np.float64, -np.inf, False), (8, True, np.float32, np.nan, True), (20, False, np.float64, np.nan, False)])
def test_counts_as_the_oracle(pkg, oracle, where, nv, triclinic, dtype, value, usecutoff):
    traj = _traj(pkg, nv, triclinic, dtype, where, True, value)
    opts = _options(pkg, usecutoff)
    a, _ = oracle_raw(pkg, oracle, traj, opts, use_cells=False)
    assert_raw_equal(a, gpu_raw(pkg, traj, opts))


@pytest.mark.parametrize("nv,triclinic,value", [(3, False, np.nan), (3, True, np.inf), (8, False, np.nan)])
def test_one_atom_leaves_the_molecule_out(pkg, nv, triclinic, value):
    opts = _options(pkg, False)
    whole, one = (gpu_raw(pkg, _traj(pkg, nv, triclinic, np.float64, "solvent", w, value), opts) for w in (True, False))
    assert_raw_equal(whole, one)


def test_many_jobs_per_launch(pkg):
    """The launches over several jobs, replayed, against each job alone."""
    from complexmixtures_amd import _lib
    from complexmixtures_amd.mddf import TrajectoryMetaData, job_kwargs
    from complexmixtures_amd.results import make_result
    opts = _options(pkg, False)
    trajs = [_traj(pkg, 3, False, np.float64, w, False, np.nan) for w in ("solute", "solvent", "solvent")]
    alone = [gpu_raw(pkg, t, opts) for t in trajs]
    dev = [(_lib.DeviceArray(t.xu), _lib.DeviceArray(t.xv)) for t in trajs]
    for _ in range(3):
        jobs = []
        for t in trajs:
            tm = TrajectoryMetaData(t, opts)
            jobs.append(_lib.Job(**job_kwargs(make_result(t, opts, tm), opts, tm, False)))
        _lib.submit_many([(j, np.arange(1, FRAMES + 1), u, v, 0, t.cells, np.ones(FRAMES))
                          for j, t, (u, v) in zip(jobs, trajs, dev)])
        for j, a in zip(jobs, alone):
            assert_raw_equal(a, j.finish())
            j.close()


@pytest.mark.parametrize("mu,nu,nv,triclinic", [(0, 3, 3, False), (0, 8, 8, True), (25, 14, 3, False), (30, 20, 3, True)])
def test_molecule_pairs(pkg, oracle, mu, nu, nv, triclinic):
    """Whole molecules without a position on either side (mu = 0: the solvent against itself)."""
    traj = _traj(pkg, nv, triclinic, np.float64, "solvent", True, np.nan)
    sv = pkg.AtomSelection(list(range(1, MV * nv + 1)), nmols=MV)
    xu = traj.xv
    su = sv
    if mu:
        rng = np.random.default_rng(mu)
        xu = np.repeat(rng.uniform(0.0, BOX, size=(1, mu, 1, 3)), FRAMES, axis=0) + rng.normal(size=(FRAMES, mu, nu, 3))
        xu[0, [0, 7]] = np.nan
        xu = xu.reshape(FRAMES, mu * nu, 3)
        su = pkg.AtomSelection(list(range(1, mu * nu + 1)), nmols=mu)
        sv = pkg.AtomSelection(list(range(mu * nu + 1, mu * nu + MV * nv + 1)), nmols=MV)
    pairs = pkg.MemoryTrajectory(xu, traj.xv, traj.cells, su, sv)
    opts = pkg.Options(dbulk=7.0, n_random_samples=6, seed=31, silent=True)
    a, _ = oracle_raw(pkg, oracle, pairs, opts, use_cells=False)
    assert_raw_equal(a, gpu_raw(pkg, pairs, opts))
