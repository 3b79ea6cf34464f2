"""CPU checks of the rounding bound that the molecule-per-lane tile kernel adds
to a frame's guard band when it evaluates distances in the expanded form
relative to the chunk centre c:

    |y' - s'|^2 = (|s'|^2 - 2 y'.s') + |y'|^2,   y' = fl(y - c), s' = fl(s - c),

with |s'|^2 staged beside s', three FMAs per pair against the lane's -2 y',
and |y'|^2 added once.  The claimed bound on the distance between that FP32
value and the exact d^2 of the same FP32 coordinates is

    u (Y + S) (2 d + 7 (Y + S)),   u = 2^-24, Y = |y - c|, S = |s - c|.

The kernel's FP32 arithmetic is emulated with numpy: float32 operations round
once; an FMA is the exact float64 product plus the addend, rounded to
float32 (the float64 sum adds at most 2^-53 relative before that rounding).
"""
import numpy as np
import pytest

U = 2.0 ** -24


def f32(x):
    return np.asarray(x, dtype=np.float64).astype(np.float32)


def fma32(a, b, c):
    return f32(a.astype(np.float64) * b.astype(np.float64) + c.astype(np.float64))


def expanded_d2(y, s, c):
    """The kernel's sequence for one atom y of the lane and one staged atom s
    (arrays of shape (n, 3), float32)."""
    sp = f32(s - c)                      # staging: s' = s - c
    w = fma32(sp[:, 0], sp[:, 0], fma32(sp[:, 1], sp[:, 1], f32(sp[:, 2] * sp[:, 2])))
    ym = f32(np.float32(-2.0) * f32(y - c))   # the lane keeps -2 y'
    t = fma32(ym[:, 0], sp[:, 0], fma32(ym[:, 1], sp[:, 1], fma32(ym[:, 2], sp[:, 2], w)))
    yy2 = f32(np.float32(0.25) * fma32(ym[:, 0], ym[:, 0], fma32(ym[:, 1], ym[:, 1], f32(ym[:, 2] * ym[:, 2]))))
    return f32(t + yy2)


def adversarial(rng, n, box=110.0, yr=6.0, dmax=10.5):
    """Chunk centres anywhere in a 110 A box, lane atoms up to 6 A from the
    centre (a chunk's half-diagonal), staged atoms 0-10.5 A from the lane
    atom, all in float32 as the kernel holds them."""
    c = f32(rng.uniform(0.0, box, (n, 3)))
    y = f32(c + rng.uniform(-yr, yr, (n, 3)))
    v = rng.normal(size=(n, 3))
    v /= np.linalg.norm(v, axis=1)[:, None]
    d = rng.uniform(0.0, dmax, n)
    s = f32(y + d[:, None] * v)
    return y, s, c


def errors(y, s, c):
    d2 = np.sum((y.astype(np.float64) - s.astype(np.float64)) ** 2, axis=1)   # exact to 2^-52
    v = expanded_d2(y, s, c).astype(np.float64)
    Y = np.linalg.norm(y.astype(np.float64) - c, axis=1)
    S = np.linalg.norm(s.astype(np.float64) - c, axis=1)
    return np.abs(v - d2), np.sqrt(d2), Y, S


def test_expanded_form_within_bound():
    rng = np.random.default_rng(2026)
    y, s, c = adversarial(rng, 400_000)
    err, d, Y, S = errors(y, s, c)
    bound = U * (Y + S) * (2.0 * d + 7.0 * (Y + S)) + 1e-12
    ratio = err / bound
    assert ratio.max() <= 1.0, ratio.max()
    # not vacuous: the largest errors come within a small factor of the bound
    assert ratio.max() > 0.05, ratio.max()


def test_expanded_form_needs_the_quadratic_term():
    """The (Y + S)^2 part (norms, FMA chain, last sum) is not covered by the
    coordinate term alone: dropping it fails on these inputs."""
    rng = np.random.default_rng(2027)
    y, s, c = adversarial(rng, 400_000)
    err, d, Y, S = errors(y, s, c)
    assert (err > U * (Y + S) * 2.0 * d + 1e-12).any()


def test_direct_form_error_is_smaller_near_contact():
    """Sanity of the emulation: for the direct form (y - s)^2 on the same
    float32 coordinates the error is at most about 4 u d^2 (no cancellation)."""
    rng = np.random.default_rng(2028)
    y, s, c = adversarial(rng, 100_000)
    dx = f32(y - s)
    v = fma32(dx[:, 0], dx[:, 0], fma32(dx[:, 1], dx[:, 1], f32(dx[:, 2] * dx[:, 2]))).astype(np.float64)
    d2 = np.sum((y.astype(np.float64) - s.astype(np.float64)) ** 2, axis=1)
    assert (np.abs(v - d2) <= 5.0 * U * d2 + 1e-12).all()


def _hilbert_table():
    """The kernel's state table, read from its source."""
    import os
    import re
    src = open(os.path.join(os.path.dirname(__file__), "..", "complexmixtures.jl_amd", "csrc", "cmgpu.hip")).read()
    body = re.search(r"HILBERT\[24 \* 8\] = \{(.*?)\};", src, re.S).group(1)
    t = np.array([int(x, 16) for x in re.findall(r"0x[0-9a-f]+", body)])
    return t.reshape(24, 8)


def test_hilbert_keys_walk_the_grid():
    """Every cell of a 2^b grid gets its own key and consecutive keys are face
    neighbours (the property that keeps chunks of consecutive keys compact)."""
    t = _hilbert_table()
    for bits in (1, 2, 3, 5):
        m = 1 << bits
        g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)
        key, state = np.zeros(len(g), int), np.zeros(len(g), int)
        for b in range(bits - 1, -1, -1):
            o = ((g[:, 0] >> b) & 1) | (((g[:, 1] >> b) & 1) << 1) | (((g[:, 2] >> b) & 1) << 2)
            e = t[state, o]
            key, state = key * 8 + (e & 7), e >> 3
        assert np.array_equal(np.sort(key), np.arange(m ** 3))
        assert (np.abs(np.diff(g[np.argsort(key)], axis=0)).sum(1) == 1).all()


def test_fixed_point_tile_distance_within_guard():
    """The tile kernel's distance from fixed-point positions (integer difference
    to the chunk centre, FP32 length, expanded form by an FMA chain) and the
    direct form of a single pair against the exact d^2, on 200,000 pairs of a
    110 A box: within the chunk's and the pair's claimed guards."""
    rng = np.random.default_rng(2029)
    L, fix, n = 110.0, 28, 200_000
    E = L * 2.0 ** -fix + 1e-9
    y = rng.uniform(0.0, L, (n, 3))
    c = y + rng.uniform(-5.0, 5.0, (n, 3))
    v = rng.normal(size=(n, 3))
    d = rng.uniform(0.0, 10.5, n)
    s = y + d[:, None] * v / np.linalg.norm(v, axis=1)[:, None]
    q = [np.rint(a / L * 2.0 ** fix).astype(np.int64) for a in (y, s, c)]
    h = np.float32(L * 2.0 ** -fix)
    rel = lambda a: f32(f32(a) * np.float64(h))          # int -> float, times the FP32 unit
    yp, sp = rel(q[0] - q[2]), rel(q[1] - q[2])
    w = fma32(sp[:, 0], sp[:, 0], fma32(sp[:, 1], sp[:, 1], f32(sp[:, 2] * sp[:, 2])))
    t = f32(np.zeros(n))
    for a, b in ((sp[:, 0], -2 * yp[:, 0]), (sp[:, 1], -2 * yp[:, 1]), (sp[:, 2], -2 * yp[:, 2]), (w, np.ones(n, np.float32))):
        t = fma32(a, f32(b), t)
    got = f32(t + fma32(yp[:, 0], yp[:, 0], fma32(yp[:, 1], yp[:, 1], f32(yp[:, 2] * yp[:, 2])))).astype(np.float64)
    d2 = ((y - s) ** 2).sum(1)
    fixed = E * (2.0 * np.sqrt(3.0) * np.sqrt(d2) + 3.0 * E)
    YS = np.linalg.norm(y - c, axis=1) + np.linalg.norm(s - c, axis=1)
    bound = fixed + U * YS * (2.0 * 3.0 * np.sqrt(d2) + 7.0 * YS) + 1e-9
    ratio = np.abs(got - d2) / bound
    assert 0.05 < ratio.max() <= 1.0, ratio.max()
    e = rel(q[0] - q[1])
    direct = fma32(e[:, 0], e[:, 0], fma32(e[:, 1], e[:, 1], f32(e[:, 2] * e[:, 2]))).astype(np.float64)
    ratio = np.abs(direct - d2) / (fixed + 10.0 * U * d2 + 1e-9)
    assert 0.05 < ratio.max() <= 1.0, ratio.max()


def test_direct_distance_guard_about_a_centre():
    """The guard of a direct FP32 d^2 between two positions held relative to a
    third one (each rounded once): fixed-point units and the coordinates'
    rounding times d, rounding units times d^2; the fixed-point terms alone do
    not cover short distances between positions far from the centre."""
    import numpy as np
    rng = np.random.default_rng(3)
    box, fix, n = 48.0, 28, 200000
    unit, u, rho = box * 2.0 ** -fix, 2.0 ** -24, 3.0
    ctr = rng.integers(0, 1 << fix, size=(n, 3))
    s = ctr + np.rint(rng.uniform(-14, 14, size=(n, 3)) / unit).astype(np.int64)
    y = s + np.rint(rng.normal(size=(n, 3)) * rng.choice([0.05, 0.5, 4.0], size=(n, 1)) / unit).astype(np.int64)
    h = np.float32(unit)
    rel = [h * (p - ctr).astype(np.float32) for p in (s, y)]
    d = (rel[1] - rel[0]).astype(np.float32)
    d2 = (d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2]).astype(np.float32)
    exact = (((y - s) * unit) ** 2).sum(axis=1)
    err = np.abs(d2.astype(np.float64) - exact)
    S, Y = (np.linalg.norm((p - ctr) * unit, axis=1) for p in (s, y))
    E, r = unit + 1e-9, np.sqrt(exact)
    fixed = 3 * E * E + 1e-9 + 2 * np.sqrt(3) * E * r + (2 * rho + 4) * u * exact
    assert (err <= fixed + 2 * rho * u * (S + Y) * r).all()
    assert (err > fixed).any()


def _pair_guard(S, Y, cutoff, rho):
    """Gx of the molecule-pair kernel for tile radius S and cluster radius Y."""
    cut = cutoff + 0.5
    W, E2 = cut + S + Y, cut + 2.0 * S
    return (U * (4.0 * max(Y * (Y + 2.0 * W), (cut + S) ** 2) + 4.0 * (Y * Y + W * W) + 4.0 * E2 * E2 +
                 S * (3.0 * S + 2.0 * (cut + S)) + 3.5 * cut * (S + Y + rho * W)) + 1e-7) * (1.0 + 1e-4)


def _cell(box, angle):
    """Lattice vectors as columns, the kernel's FP32 vectors per unit, and rho."""
    import math
    c, s = math.cos(math.radians(angle)), math.sin(math.radians(angle))
    H = np.array([[1.0, c, c], [0.0, s, c * (1 - c) / s], [0.0, 0.0, 0.0]])
    H[2, 2] = math.sqrt(1.0 - H[0, 2] ** 2 - H[1, 2] ** 2)
    H *= box
    if angle == 90.0:
        H = np.diag(np.diag(H))
        return H, 3.0
    V = np.linalg.det(H)
    sp = [V / np.linalg.norm(np.cross(H[:, (k + 1) % 3], H[:, (k + 2) % 3])) for k in range(3)]
    kappa = max(sum(abs(H[r, k]) / sp[k] for k in range(3)) for r in range(3))
    return H, 5.0 * math.sqrt(3.0) * kappa


def _chain(c, a, b, order):
    """c + a . b over four components by FMAs in an order of the additions."""
    for k in order:
        c = fma32(a[k], b[k], c)
    return c


@pytest.mark.parametrize("angle", [90.0, 75.0])
@pytest.mark.parametrize("bits", [0, 4, 5, 6, 8])
def test_molecule_pair_distance_within_guard(angle, bits):
    """The two chained products of the molecule-pair kernel (|t - y'|^2 as the
    start of |t - y' + s'|^2, t between the centres of tile and cluster) in both
    layouts of the operands and both orders of their sums, with the candidate's
    code in the lowest bits: within the kernel's guard for pairs within the cutoff,
    tiles and clusters of 0.5 to 60 A radius."""
    rng = np.random.default_rng([2030, int(angle), bits])
    box, fix, cutoff, n = 240.0, 27, 10.0, 20000
    H, rho = _cell(box, angle)
    Hfix = (H * 2.0 ** -fix).astype(np.float32)
    unit = lambda m: (lambda v: v / np.linalg.norm(v, axis=1)[:, None])(rng.normal(size=(m, 3)))
    inside = lambda R: unit(n) * (R * rng.uniform(size=n) ** (1 / 3))[:, None]
    worst = 0.0
    for S, Y in [(0.5, 0.5), (3.0, 6.0), (6.0, 3.0), (12.0, 25.0), (60.0, 4.0), (4.0, 60.0), (60.0, 60.0)]:
        sr, yr = inside(S), inside(Y)
        e = unit(n) * (rng.uniform(size=n) * cutoff)[:, None]
        ti = np.rint(np.linalg.solve(H, (yr + e - sr).T).T * 2.0 ** fix).astype(np.int64)   # centres, tile minus cluster
        d2 = ((ti * 2.0 ** -fix @ H.T + sr - yr) ** 2).sum(1)
        keep = d2 <= cutoff * cutoff
        s, y = [f32(sr[keep, k]) for k in range(3)], [f32(yr[keep, k]) for k in range(3)]
        a, b, c = (f32(ti[keep, k]) for k in range(3))
        t = [f32(Hfix[0, 0] * a), f32(Hfix[1, 1] * b), f32(Hfix[2, 2] * c)]
        if angle != 90.0:
            t[0] = fma32(Hfix[0, 1], b, fma32(Hfix[0, 2], c, t[0]))
            t[1] = fma32(Hfix[1, 0], a, fma32(Hfix[1, 2], c, t[1]))
            t[2] = fma32(Hfix[2, 0], a, fma32(Hfix[2, 1], b, t[2]))
        norm = lambda v: fma32(v[0], v[0], fma32(v[1], v[1], f32(v[2] * v[2])))
        s2, y2, t2 = norm(s), norm(y), norm(t)
        one, zero = np.ones_like(s2), np.zeros_like(s2)
        m2y = [f32(-2.0 * v) for v in y]
        z = [f32(m2y[k] + f32(2.0 * t[k])) for k in range(3)]
        G = _pair_guard(S, Y, cutoff, rho)
        pk = 2.0 ** (bits - 23)
        for order in ((0, 1, 2, 3), (3, 2, 1, 0)):
            for quad in (True, False):
                first = _chain(y2, t + [t2], m2y + [one], order) if quad else _chain(zero, t + [one], m2y + [f32(y2 + t2)], order)
                got = _chain(first, s + [s2], z + [one], order)
                code = got.view(np.int32)
                coded = (code & ~((1 << bits) - 1) | rng.integers(0, 1 << bits, size=code.shape)).astype(np.int32).view(np.float32)
                # as decided: the code cleared, half its range added back
                val = ((code & ~((1 << bits) - 1)).astype(np.int32).view(np.float32) * f32(1.0 + 0.5 * pk)).astype(np.float64)
                bound = G + val * (0.5 * pk + 2.0 ** -21) + 1e-7
                worst = max(worst, (np.abs(val - d2[keep]) / bound).max())
                assert (np.abs(val - d2[keep]) <= bound).all()
                # the value compared and queued carries the code
                assert (np.abs(coded.astype(np.float64) - d2[keep]) <= G + d2[keep] * (pk + 2.0 ** -21) + 1e-7).all()
    assert worst > 0.02, worst
