"""Single pairs of the FP64 walk, relative to the pair's own force, which falls to 1e-3 .. 1e-200 of the Newtonian one.

One source of unit charge, targets without mass, no mesh: a target's acceleration is one term, S(x) d / rho^3 with
x = rho / (2 r_s).  The box edge is a power of two, so d is exact.  With u = 2^-53: v = r^2 + eps^2 takes four roundings
(4 u), which the force follows with |dlnF / dlnv| <= 2 + x^2 (both laws); 1 / rho^3, erfcx, the exponential, their
products and the sum of the term take at most ten more: |error| <= (18 + 4 x^2) u of each component.  The reference is
extended precision (within u / 16)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

L = 128.0
LD = np.longdouble
PI = LD("3.14159265358979323846264338327950288")


def _erfc(x):
    """erfc in extended precision: the all-positive series of erf up to x = 1.5, the continued fraction beyond."""
    x = np.asarray(x, LD)
    small = np.minimum(x, LD(1.5))
    t = small.copy()
    s = t.copy()
    for n in range(1, 120):
        t = t * 2 * small * small / (2 * n + 1)
        s = s + t
    near = 1 - 2 / np.sqrt(PI) * np.exp(-small * small) * s
    big = np.maximum(x, LD(1.5))
    k = np.zeros_like(big)
    for n in range(400, 0, -1):
        k = (LD(n) / 2) / (big + k)
    return np.where(x < 1.5, near, np.exp(-big * big) / np.sqrt(PI) / (big + k))


def _force(d, eps, r_s, mode):
    """S(x) d / rho^3 and x, extended precision."""
    d = d.astype(LD)
    rho = np.sqrt((d * d).sum(1) + LD(eps) * LD(eps))
    x = rho / (2 * LD(r_s))
    s = _erfc(x)
    if mode == 0:
        s = s + 2 / np.sqrt(PI) * x * np.exp(-x * x)
    return (s / rho ** 3)[:, None] * d, x


def _check(acc, d, eps, r_s, mode, charge):
    ref, x = _force(d, eps, r_s, mode)
    ref = -charge * ref  # massless m- targets are pushed by the m+ source
    bound = ((18 + 4 * x * x) * LD(2) ** -53)[:, None] * np.abs(ref) + LD(1e-290)
    assert np.all(np.abs(acc.astype(LD) - ref) <= bound), float(np.max(np.abs(acc - ref) / bound))


def _context(jtp, mode, ratio, group, leaf, r_cut, theta):
    p = jtp.default_params(L, 32)
    p.precision, p.split_mode, p.theta, p.theta_cut, p.pm_enabled = jtp.FP64, mode, theta, theta, 0
    p.group_size, p.leaf_size, p.softening = group, leaf, 0.01
    p.r_cut, p.r_s = r_cut, r_cut / ratio
    return p, jtp.ForceContext(p, 1.0, 0.0)


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("ratio", [1.0, 3.0, 4.5, 5.3])
@pytest.mark.parametrize("group", [7, 32, 64])
def test_cut_pair(jtp, mode, ratio, group):
    print(f"case: FP64 cut pair mode={mode} r_cut/r_s={ratio} group={group}", flush=True)
    rng = np.random.default_rng(11)
    p, ctx = _context(jtp, mode, ratio, group, 4, 20.0, 0.0)
    n = 1501
    e = rng.normal(size=(n, 3))
    r = np.concatenate([10.0 ** rng.uniform(-6, 0, n // 3), rng.uniform(0.0, 1.0, n - n // 3)]) * p.r_cut * (1 - 1e-9)
    x = np.concatenate([np.zeros((1, 3)), e / np.linalg.norm(e, axis=1, keepdims=True) * r[:, None]])
    pos = jtp.to_fixed(x, L)
    sp = np.concatenate([np.ones(1, np.int8), -np.ones(n, np.int8)])
    acc = ctx.compute_forces(pos, sp)[1:]
    u = pos.astype(np.int64)
    d = (u[0] - u[1:]) * (L / 2.0 ** 32)
    assert np.all((d ** 2).sum(1) < p.r_cut ** 2)
    _check(acc, d, p.softening, p.r_s, mode, 1)


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("ratio", [1.0, 3.0, 4.5, 5.3])
@pytest.mark.parametrize("group", [7, 32, 64])
def test_straddling_monopole(jtp, mode, ratio, group):
    """Two particles, one accepted node across r_cut: x from 0.06 to 6.5, across both ranges of the tail."""
    print(f"case: FP64 straddling pair mode={mode} r_cut/r_s={ratio} group={group}", flush=True)
    rng = np.random.default_rng(13)
    p, ctx = _context(jtp, mode, ratio, group, 1, 4.0, 1.0)
    clump = np.array([[-0.015625, 4.0, 4.0], [-0.015625, 4.0009765625, 4.0]])  # just below the targets' cell (edge 8)
    tg = rng.uniform(0.0, 8.0, (64, 3))
    tg[:4] = (0.5, 4.0, 4.0) + rng.uniform(-0.1, 0.1, (4, 3))
    pos = jtp.to_fixed(np.concatenate([clump, tg]), L)
    sp = np.concatenate([np.ones(2, np.int8), -np.ones(64, np.int8)])
    acc = ctx.compute_forces(pos, sp)[2:]
    u = pos.astype(np.int64).astype(np.float64)
    d = (u[:2].mean(0) - u[2:]) * (L / 2.0 ** 32)
    seen = np.any(acc != 0, axis=1)  # the group of a target sums the node or lies beyond r_cut altogether
    assert seen.sum() >= 7
    if group == 64:
        assert np.sum(seen & (np.linalg.norm(d, axis=1) > 1.5 * p.r_cut)) >= 8
    _check(acc[seen], d[seen], p.softening, p.r_s, mode, 2)
