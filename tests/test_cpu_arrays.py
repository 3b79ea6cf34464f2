"""The array forms of host preparation against the element-wise definitions."""
import warnings

import numpy as np
import pytest


def _csr_by_atom(sel, positions, groups_of):
    where = {}
    for g, inds in enumerate(groups_of.group_atom_indices):
        for a in inds:
            where.setdefault(a, []).append(g)
    lists = [where.get(sel.indices[p], []) for p in positions]
    return np.cumsum([0] + [len(x) for x in lists]), sum(lists, []) or [0]


@pytest.mark.parametrize("seed", range(40))
def test_group_csr(pkg, seed):
    """Overlapping and empty groups, another selection's atoms, positions in any order."""
    from complexmixtures_amd.selection import group_csr
    rng = np.random.default_rng(seed)
    n = int(rng.integers(1, 40))
    ind = np.sort(rng.permutation(100)[:n] + 1).tolist()
    groups = [rng.choice(ind, size=int(rng.integers(0, n + 1)), replace=False).tolist() for _ in range(int(rng.integers(1, 6)))]
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        s = pkg.AtomSelection(ind, nmols=1, group_atom_indices=groups, group_names=[str(i) for i in range(len(groups))])
    other = pkg.AtomSelection(list(range(1, 60)), nmols=1)
    for sel, m in ((s, n), (other, 59)):
        for pos in (range(m), rng.permutation(m).tolist(), []):
            ptr, idx = group_csr(sel, pos, s)
            rp, ri = _csr_by_atom(sel, pos, s)
            assert ptr.dtype == idx.dtype == np.int32 and np.array_equal(ptr, rp) and np.array_equal(idx, ri)


@pytest.mark.parametrize("step", [0.02, 0.0125, 0.3])
def test_shell_radii(pkg, step):
    from complexmixtures_amd.results import _shellradii
    assert _shellradii(700, step) == [pkg.shellradius(i, step) for i in range(1, 701)]
