"""Molecule pairs on the matrix cores at the sizes where their split of the work
changes: rows per solute molecule (4, 8, 16), solvent atoms per cluster (3, 4, 8,
16), partial tiles, super tiles and clusters, cells small enough that two images
of a molecule are in reach, custom groups, and one molecule size beyond the
kernels' range.  Counts equal the FP64 oracle's bit for bit (unit weights: exact)."""
import numpy as np
import pytest

from conftest import assert_raw_equal, gpu_raw, oracle_raw

pytestmark = pytest.mark.gpu


def _traj(pkg, nu, mu, nv, mv, box=27.0, angle=90.0, nframes=2, seed=0, dtype=np.float64, groups=False, broken=True):
    """mu solute molecules of nu atoms in mv solvent molecules of nv (mu = 0: the solvent against itself)."""
    import complexmixtures_amd.synthetic as S
    from complexmixtures_amd.trajectory import unitcell_matrix
    rng = np.random.default_rng([seed, nu, mu, nv, mv])
    H = unitcell_matrix(box, box, box, angle, 90.0, 90.0)

    def side(n, m):
        mol = np.concatenate([np.zeros((1, 3)), rng.normal(scale=0.7, size=(n - 1, 3))])
        x = S.place_molecules(rng, mol, rng.uniform(size=(m, 3)) @ H.T)
        x = np.stack([x + rng.normal(scale=0.1, size=x.shape) for _ in range(nframes)])
        if broken:   # atoms and molecules in other images of the cell
            x += rng.integers(-1, 2, size=(nframes, n * m, 3)) @ H.T
        return x.astype(dtype)

    xv = side(nv, mv)
    kw = {}
    if groups:
        kw = dict(group_atom_indices=[list(range(1, nv * mv, 3)), list(range(2, nv * mv // 2))], group_names=["a", "b"])
    if mu == 0:
        s = pkg.AtomSelection(list(range(1, nv * mv + 1)), nmols=mv, **kw)
        return pkg.MemoryTrajectory(xv, xv, np.repeat(H[None], nframes, axis=0), s, s)
    off = nu * mu
    su = pkg.AtomSelection(list(range(1, off + 1)), nmols=mu)
    if groups:
        kw["group_atom_indices"] = [[i + off for i in g] for g in kw["group_atom_indices"]]
    sv = pkg.AtomSelection(list(range(off + 1, off + nv * mv + 1)), nmols=mv, **kw)
    return pkg.MemoryTrajectory(side(nu, mu), xv, np.repeat(H[None], nframes, axis=0), su, sv)


def _check(pkg, oracle, traj, **kw):
    opts = pkg.Options(seed=23, silent=True, **kw)
    cn = kw.get("n_random_samples") is None
    a, _ = oracle_raw(pkg, oracle, traj, opts, coordination_number_only=cn)
    assert_raw_equal(a, gpu_raw(pkg, traj, opts, coordination_number_only=cn))


@pytest.mark.parametrize("nu,mu,nv,mv", [
    (1, 2, 1, 1), (1, 65, 2, 17), (3, 4, 3, 16), (4, 5, 4, 15), (5, 33, 3, 257), (8, 32, 5, 33), (9, 16, 3, 100),
    (3, 50, 8, 31), (2, 300, 9, 40), (13, 17, 6, 40), (16, 15, 16, 47), (7, 20, 14, 20), (14, 12, 1, 200),
    (17, 6, 3, 60), (3, 60, 17, 9)])
@pytest.mark.parametrize("angle", [90.0, 75.0])
def test_cross_sizes(pkg, oracle, nu, mu, nv, mv, angle):
    traj = _traj(pkg, nu, mu, nv, mv, angle=angle)
    _check(pkg, oracle, traj, dbulk=8.0, n_random_samples=3, irefatom=min(2, nv))


@pytest.mark.parametrize("nv,mv,iref", [
    (1, 2, 1), (1, 260, 1), (2, 33, 2), (3, 16, 3), (3, 17, 1), (3, 1030, 2), (4, 65, 4), (5, 64, 5), (8, 31, 1),
    (8, 90, 6), (9, 16, 9), (14, 40, 5), (16, 33, 16), (17, 12, 3)])
@pytest.mark.parametrize("angle,dtype", [(90.0, np.float32), (75.0, np.float64)])
def test_self_sizes(pkg, oracle, nv, mv, iref, angle, dtype):
    traj = _traj(pkg, 0, 0, nv, mv, angle=angle, dtype=dtype)
    _check(pkg, oracle, traj, dbulk=8.0, n_random_samples=3, irefatom=iref)
    _check(pkg, oracle, traj, bulk_range=(7.0, 8.5), irefatom=iref)   # counts of the real pass alone


@pytest.mark.parametrize("mu", [0, 20])
def test_custom_groups_and_bulk_range(pkg, oracle, mu):
    traj = _traj(pkg, 5, mu, 3, 150, groups=True, seed=3)
    _check(pkg, oracle, traj, bulk_range=(6.0, 9.0), n_random_samples=4, irefatom=2)


def test_two_images_in_reach(pkg, oracle):
    """A cell of 19 A at a cutoff of 9 A: many tiles meet a cluster under two shifts or more."""
    _check(pkg, oracle, _traj(pkg, 3, 40, 2, 90, box=19.0, seed=5, broken=False), dbulk=9.0, n_random_samples=2)
    _check(pkg, oracle, _traj(pkg, 0, 0, 2, 200, box=19.0, angle=80.0, seed=6, broken=False), dbulk=9.0, n_random_samples=2)


def test_exact_ties(pkg, oracle):
    """Coordinates in whole Angstroms: ties between atom pairs and distances on the edges of bins, left to FP64."""
    x = np.round(_traj(pkg, 0, 0, 3, 40, nframes=1, seed=7, broken=False).xv)
    x[:, 1::3] = x[:, ::3] + [1.0, 0.0, 0.0]
    x[:, 2::3] = x[:, ::3] + [0.0, 1.0, 0.0]
    x[:, ::3] += [0.5, 0.0, 0.25]
    s = pkg.AtomSelection(list(range(1, 121)), nmols=40)
    traj = pkg.MemoryTrajectory(x, x, np.eye(3)[None] * 27.0, s, s)
    _check(pkg, oracle, traj, dbulk=8.0, n_random_samples=2, irefatom=2)


@pytest.mark.parametrize("binstep", [0.02, 0.01, 0.005])
def test_group_histograms_in_and_beyond_lds(pkg, oracle, binstep):
    """17 groups of 400, 800 and 1,600 bins: 27, 54 and 109 kB, of which 64 kB may lie in LDS."""
    traj = _traj(pkg, 14, 12, 3, 150, seed=8)
    _check(pkg, oracle, traj, dbulk=8.0, binstep=binstep, n_random_samples=3)


@pytest.mark.parametrize("nu,mu,nv,mv", [(1, 1100, 1, 5), (3, 1500, 1, 20), (4, 2100, 3, 33), (8, 700, 8, 17), (14, 300, 2, 16)])
def test_many_tiles_few_clusters(pkg, oracle, nu, mu, nv, mv):
    """One to three clusters a frame: their super tiles, and those tiles, split over many wavefronts."""
    _check(pkg, oracle, _traj(pkg, nu, mu, nv, mv, box=40.0, nframes=1, seed=9, angle=80.0), dbulk=9.0, n_random_samples=2)


@pytest.mark.parametrize("nu,nv", [(1, 1), (2, 3), (5, 8), (14, 3), (16, 16)])
@pytest.mark.parametrize("mv", [3, 40])
def test_exact_ties_between_species(pkg, oracle, nu, nv, mv):
    """Whole Angstroms on both sides: every pair in reach is left to FP64, few (several lanes a pair) and many."""
    t = _traj(pkg, nu, 6, nv, mv, nframes=2, seed=10, broken=False)
    t.xu[:], t.xv[:] = np.round(t.xu), np.round(t.xv)
    _check(pkg, oracle, t, dbulk=8.0, n_random_samples=3, irefatom=nv)


@pytest.mark.parametrize("n,m", [(2, 7), (8, 30), (14, 9)])
def test_exact_ties_of_larger_molecules(pkg, oracle, n, m):
    t = _traj(pkg, 0, 0, n, m, nframes=2, seed=11, broken=False)
    t.xv[:] = np.round(t.xv)
    _check(pkg, oracle, t, dbulk=8.0, n_random_samples=3, irefatom=n)


@pytest.mark.parametrize("mu,mv", [(0, 16), (0, 17), (0, 33), (0, 900), (2, 3), (15, 16), (16, 17), (17, 400), (600, 33)])
@pytest.mark.parametrize("angle,dtype", [(90.0, np.float32), (75.0, np.float64)])
def test_single_atoms(pkg, oracle, mu, mv, angle, dtype):
    """Single atoms on both sides: a row of a tile is a molecule; also whole Angstroms (FP64) and two images in reach."""
    _check(pkg, oracle, _traj(pkg, 1, mu, 1, mv, angle=angle, dtype=dtype, seed=12), dbulk=9.0, n_random_samples=3)
    t = _traj(pkg, 1, mu, 1, mv, box=20.0, angle=angle, dtype=dtype, seed=13, broken=False)
    for x in (t.xu, t.xv):
        x[:] = np.round(x)
    _check(pkg, oracle, t, bulk_range=(7.0, 9.5))
