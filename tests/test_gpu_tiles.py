"""The single-solute kernels at the sizes where their split of the work changes:
molecules per chunk (16 per group, up to four groups), solvent atoms per block
of tiles, merged random passes (groups of at most 16, half-cell keys from eight
per group on), staged solute atoms per round, histograms too large for LDS.
Counts equal the FP64 oracle's bit for bit (unit weights: exact)."""
import numpy as np
import pytest

from conftest import assert_raw_equal, gpu_raw, oracle_raw

pytestmark = pytest.mark.gpu


def _molecule(rng, nv):
    """nv atoms within about 1.5 A of their first one (a single atom: a point)."""
    return np.concatenate([np.zeros((1, 3)), rng.normal(scale=0.8, size=(nv - 1, 3))])


def _system(pkg, nu, nmols, nv, box=26.0, nframes=1, seed=0, triclinic=False, dtype=np.float64):
    import complexmixtures_amd.synthetic as S
    from complexmixtures_amd.trajectory import unitcell_matrix
    rng = np.random.default_rng([seed, nu, nmols, nv])
    H = unitcell_matrix(box, box, box, *((80.0, 85.0, 95.0) if triclinic else (90.0, 90.0, 90.0)))
    xu0 = H @ np.full(3, 0.5) + rng.normal(scale=3.0, size=(nu, 3))
    x0 = S.place_molecules(rng, _molecule(rng, nv), rng.uniform(size=(nmols, 3)) @ H.T)
    xu = np.stack([xu0 + rng.normal(scale=0.2, size=xu0.shape) for _ in range(nframes)]).astype(dtype)
    xv = np.stack([x0 + rng.normal(scale=0.1, size=x0.shape) for _ in range(nframes)]).astype(dtype)
    su = pkg.AtomSelection(list(range(1, nu + 1)), nmols=1)
    sv = pkg.AtomSelection(list(range(nu + 1, nu + nmols * nv + 1)), nmols=nmols)
    return pkg.MemoryTrajectory(xu, xv, np.repeat(H[None], nframes, axis=0), su, sv)


@pytest.mark.parametrize("nu,nmols,nv,passes", [
    (1, 1, 1, 1), (1, 1, 3, 10), (31, 15, 3, 1), (32, 16, 3, 7), (33, 17, 3, 8), (257, 63, 3, 16), (288, 64, 3, 17),
    (289, 65, 3, 33), (100, 129, 2, 10), (100, 40, 4, 9), (100, 40, 5, 10), (64, 33, 8, 10), (50, 21, 14, 12),
    (40, 9, 63, 3)])
@pytest.mark.parametrize("triclinic", [False, True])
def test_chunk_and_pass_group_edges(pkg, oracle, nu, nmols, nv, passes, triclinic):
    traj = _system(pkg, nu, nmols, nv, nframes=2, triclinic=triclinic)
    opts = pkg.Options(dbulk=9.0, n_random_samples=passes, seed=17, silent=True, irefatom=min(2, nv))
    a, _ = oracle_raw(pkg, oracle, traj, opts)
    assert_raw_equal(a, gpu_raw(pkg, traj, opts))


@pytest.mark.parametrize("binstep", [0.0025, 0.00125])
def test_histograms_beyond_lds(pkg, oracle, binstep):
    """4,000 bins still fit the block's LDS (the solvent groups do not), 8,000 do not."""
    traj = _system(pkg, 60, 200, 3, seed=3)
    opts = pkg.Options(dbulk=10.0, binstep=binstep, n_random_samples=10, seed=18, silent=True)
    a, _ = oracle_raw(pkg, oracle, traj, opts)
    assert_raw_equal(a, gpu_raw(pkg, traj, opts))


@pytest.mark.parametrize("columns", [1, 2, 4, 8])
def test_molecules_per_chunk(pkg, oracle, columns):
    """64, 32, 16 and 8 molecules per chunk of the real pass, shared bulk shell, FP32 input."""
    traj = _system(pkg, 700, 500, 3, box=30.0, seed=4, dtype=np.float32)
    opts = pkg.Options(bulk_range=(8.0, 11.0), n_random_samples=10, seed=19, silent=True)
    a, _ = oracle_raw(pkg, oracle, traj, opts)
    assert_raw_equal(a, gpu_raw(pkg, traj, opts, job_kw={"tuning": dict(columns=columns)}))


@pytest.mark.parametrize("nu,nmols,nv,passes,frames", [
    (3, 400, 8, 330, 2), (90, 500, 4, 200, 2), (40, 300, 1, 220, 3), (60, 150, 14, 200, 2), (30, 100, 24, 130, 3),
    (12, 60, 40, 330, 2), (130, 4, 63, 1100, 8)])
@pytest.mark.parametrize("triclinic", [False, True])
def test_chunks_of_several_blocks(pkg, oracle, nu, nmols, nv, passes, frames, triclinic):
    """Enough random slots around a sparse solute for chunks of up to 512 atoms: several blocks of 128 atoms from one
    staging, and (130 atoms) more staged atoms than the buffer takes, each block on its own."""
    traj = _system(pkg, nu, nmols, nv, nframes=frames, seed=5, triclinic=triclinic)
    traj.xu[:] = np.random.default_rng(nu).uniform(0.0, 26.0, size=traj.xu.shape[1:])
    opts = pkg.Options(dbulk=9.0, n_random_samples=passes, seed=21, silent=True, irefatom=min(2, nv))
    a, _ = oracle_raw(pkg, oracle, traj, opts, nthreads=8)
    assert_raw_equal(a, gpu_raw(pkg, traj, opts))


def test_real_chunks_of_several_blocks(pkg, oracle):
    """48 frames of 900 molecules: chunks of five molecules, two blocks of 64 lanes, in the real pass."""
    traj = _system(pkg, 20, 900, 14, nframes=48, seed=6)
    traj.xu[:] = np.random.default_rng(6).uniform(0.0, 26.0, size=traj.xu.shape[1:])
    opts = pkg.Options(dbulk=9.0, seed=22, silent=True)
    a, _ = oracle_raw(pkg, oracle, traj, opts, coordination_number_only=True, nthreads=8)
    assert_raw_equal(a, gpu_raw(pkg, traj, opts, coordination_number_only=True))


@pytest.mark.parametrize("columns,nv", [(1, 8), (2, 8), (4, 8), (8, 8), (1, 14), (2, 14), (4, 14), (8, 14), (1, 63), (2, 63),
                                        (0, 63)])
def test_atoms_per_chunk(pkg, oracle, columns, nv):
    """64 / columns atoms per chunk of molecules of other than three; where that holds no molecule, the setting is refused."""
    traj = _system(pkg, 300, 120, nv, seed=7)
    opts = pkg.Options(dbulk=9.0, n_random_samples=10, seed=23, silent=True)
    kw = {"job_kw": {"tuning": dict(columns=columns)}}
    if columns and 64 // columns < nv:
        with pytest.raises(pkg.ArgumentError):
            gpu_raw(pkg, traj, opts, **kw)
        return
    a, _ = oracle_raw(pkg, oracle, traj, opts)
    assert_raw_equal(a, gpu_raw(pkg, traj, opts, **kw))
