"""The bottom-up tree build at the edges of its workgroups, launches and rounds, bit-exact against the oracle's
Karras construction and node sums: one and several workgroups, one to three launches of lists, several rounds per
workgroup, and keys whose runs stay unmerged the longest (all equal, nested corners, few distinct cells)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

M = 384  # items of a workgroup


def _particles(kind, n, rng):
    pos = rng.integers(0, 2 ** 32, (n, 3), dtype=np.uint64).astype(np.uint32)
    if kind == "equal":
        pos[:] = pos[0]
    elif kind == "corners":  # coordinates 2^k and 2^32 - 2^k: prefix lengths of every value beside each other
        k = rng.integers(0, 32, (n, 3))
        p = (np.uint64(1) << k.astype(np.uint64)).astype(np.uint64)
        pos = np.where(rng.random((n, 3)) < 0.5, p, (2 ** 32 - p)).astype(np.uint32)
    elif kind == "cells":  # few distinct keys, long runs of duplicates
        pos = (pos >> np.uint32(30)) << np.uint32(30)
    elif kind == "halo":
        pos = (2 ** 31 + rng.normal(0, 1, (n, 3)) * 10.0 ** rng.uniform(3, 8.5, (n, 1))).astype(np.int64).astype(np.uint32)
    return pos, np.where(rng.random(n) < 0.5, 1, -1).astype(np.int8)


def _check(jtp, orc, pos, sp, precision=0):
    p = jtp.default_params(250.0, 32)
    p.precision, p.pm_enabled = precision, 0
    ctx = jtp.ForceContext(p, 1.0, 19.0)
    ctx.compute_forces(pos, sp)
    perm, keys = ctx.stage(jtp.STAGE_PERM), ctx.stage(jtp.STAGE_KEYS)
    nodes = orc.karras(keys)
    assert np.array_equal(ctx.stage(jtp.STAGE_NODES), nodes)
    sums, boxes = orc.node_sums(pos[perm], sp[perm], nodes)
    assert np.array_equal(ctx.stage(jtp.STAGE_BOXES), boxes)
    assert np.array_equal(ctx.stage(jtp.STAGE_SUMS), sums)
    mono = ctx.stage(jtp.STAGE_MONO)
    for q, o in ((sums[:, 0:4], 0), (sums[:, 4:8], 4)):
        has = q[:, 0] > 0
        cnt, s = q[has, 0], q[has, 1:4]
        assert np.all(mono[~has, o] == 0)
        if precision == 0:  # the rounded integer mean, exactly
            assert np.array_equal(mono[has, o + 1:o + 4], ((s + (cnt // 2)[:, None]) // cnt[:, None]).astype(np.float64))
        else:
            quot = s // cnt[:, None]
            rem = (s - quot * cnt[:, None]).astype(np.float64) / cnt[:, None].astype(np.float64)
            assert np.array_equal(mono[has, o + 1:o + 4], quot.astype(np.float64) + rem)


@pytest.mark.parametrize("kind", ["random", "equal", "corners", "cells", "halo"])
@pytest.mark.parametrize("n", [2, 3, M - 1, M, M + 1, 2 * M, 7 * M + 13, 64 * M, 64 * M + 1, 200 * M + 5])
def test_workgroup_edges(jtp, orc, kind, n):
    print(f"case: build {kind} n={n}", flush=True)
    pos, sp = _particles(kind, n, np.random.default_rng(n))
    _check(jtp, orc, pos, sp, precision=n % 2)


@pytest.mark.parametrize("kind", ["random", "corners", "halo"])
def test_several_rounds(jtp, orc, kind):
    n = 2 * 2048 * M + 777  # two rounds per workgroup of the first launch
    print(f"case: build {kind} n={n}", flush=True)
    pos, sp = _particles(kind, n, np.random.default_rng(9))
    _check(jtp, orc, pos, sp)
