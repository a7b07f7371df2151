"""The FP64 walk's polynomial pair laws against erfc and exp.

Cut pairs: theta = 0 (every source a particle) against the oracle's direct sum, over split ratios r_cut / r_s inside
and outside the range that the polynomials cover (beyond it the kernel calls erfc and exp).  Each pair is good to 1e-15
of its Newtonian force and the sums hold at most ~500 sources of both signs, so the bound is 1e-13 of the rms force
times the ratio of the summed magnitudes to the sum (below 100 on these boxes): 1e-11.

Monopoles of nodes that straddle r_cut: two particles as one accepted node seen by targets of zero mass spread over a
whole group cell, so that one group holds distances from well within r_cut to beyond every polynomial range.  One term
per target: 4e-15 of the Newtonian force."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RATIOS = [1.0, 3.0, 4.5, 5.4, 6.0, 9.0]


def _law(x, mode):
    s = np.array([math.erfc(v) for v in x.ravel()]).reshape(x.shape)
    return s + 2 / math.sqrt(math.pi) * x * np.exp(-x * x) if mode == 0 else s


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("ratio", RATIOS)
@pytest.mark.parametrize("group", [13, 32, 64])
def test_cut_pairs_match_direct_sum(jtp, orc, mode, ratio, group):
    print(f"case: FP64 theta=0 mode={mode} r_cut/r_s={ratio} group={group}", flush=True)
    L, n = 100.0, 3001
    rng = np.random.default_rng(5)
    x = rng.uniform(-L / 2, L / 2, (n, 3))
    x[: n // 3] = rng.normal(0, 4.0, (n // 3, 3)) + 20.0
    pos = jtp.to_fixed(x, L)
    sp = np.where(rng.random(n) < 0.5, 1, -1).astype(np.int8)
    p = jtp.default_params(L, 32)
    p.precision, p.split_mode, p.theta, p.theta_cut, p.pm_enabled, p.group_size = jtp.FP64, mode, 0.0, 0.0, 0, group
    p.r_cut, p.softening = 13.7, 0.05
    p.r_s = p.r_cut / ratio
    acc = jtp.ForceContext(p, 1.0, 19.0).compute_forces(pos, sp)
    ref = orc.short_direct(pos, sp, 1.0, 19.0, L, p.softening, p.r_cut, p.r_s, mode)
    assert np.max(np.abs(acc - ref)) < 1e-11 * np.sqrt(np.mean(ref ** 2))


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("ratio", RATIOS)
@pytest.mark.parametrize("group", [7, 32, 64])
def test_straddling_monopoles_match_the_law(jtp, mode, ratio, group):
    print(f"case: FP64 straddling monopole mode={mode} r_cut/r_s={ratio} group={group}", flush=True)
    L = 160.0  # group cells of edge 10
    rng = np.random.default_rng(3)
    clump = np.array([[-0.02, 5.0, 5.0], [-0.02, 5.001, 5.0]])  # just below the cell of the targets
    tg = rng.uniform(0.0, 10.0, (64, 3))
    tg[0] = (0.5, 5.0, 5.0)  # every group of <= 64 runs is within r_cut of the clump or skips it
    pos = jtp.to_fixed(np.concatenate([clump, tg]), L)
    sp = np.concatenate([np.ones(2, np.int8), -np.ones(len(tg), np.int8)])
    p = jtp.default_params(L, 32)
    p.precision, p.split_mode, p.theta, p.theta_cut, p.pm_enabled = jtp.FP64, mode, 1.0, 1.0, 0
    p.group_size, p.leaf_size = group, 1
    p.r_cut, p.softening = 4.0, 0.01
    p.r_s = p.r_cut / ratio
    acc = jtp.ForceContext(p, 1.0, 0.0).compute_forces(pos, sp)[2:]
    u = (pos.astype(np.int64) - 2 ** 31).astype(np.float64)
    d = (u[:2].mean(0) - u[2:]) * (L / 2.0 ** 32)
    rho = np.sqrt((d ** 2).sum(1) + p.softening ** 2)
    newton = 2.0 * d / rho[:, None] ** 3  # the two particles of the clump
    ref = -newton * _law(rho / (2 * p.r_s), mode)[:, None]
    # a target's group either sums the clump as one monopole or lies beyond r_cut altogether (acceleration zero)
    seen = np.any(acc != 0, axis=1)
    if group == 64:
        assert np.all(seen | (np.abs(ref).max(1) < 1e-15 * np.abs(newton).max(1)))
    assert seen.sum() >= 7
    assert np.all(np.abs(acc - ref)[seen] <= 4e-15 * np.linalg.norm(newton, axis=1)[seen, None])
    near = np.linalg.norm(d, axis=1) < p.r_cut
    assert np.all(seen[near])
