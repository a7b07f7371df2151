"""The walk's early list where it holds some of the groups, or more are marked than it has room for.

A group is marked if the cell that encloses it reaches at least 32 group sizes beyond it.  The rule restated on the host from
the sorted keys says how many groups each case marks, so that every case is known to exercise what it is for; then a
single context, which walks the list first and the rest after it, has to give what the one-launch walk over several
boxes gives, which takes all groups in Morton order, bit for bit."""
import janus_treepm
import numpy as np
import pytest

REACH = 32
MASK = np.uint64(~((1 << 16) - 1) & (2 ** 64 - 1))
L = 50.0
# kind, particles, group size, marked groups: more than the list has room for?
CASES = [("clusters", 20011, 7, False), ("clusters", 200003, 32, False), ("clusters", 200003, 64, False),
         ("clump", 90, 1, False), ("clump", 40000, 7, True)]


def _positions(kind, n):
    """Clumps about the centres of level-4 cells (edge L / 16), whose octants lie apart in the order; or one point."""
    rng = np.random.default_rng(n)
    x = rng.uniform(-L / 2, L / 2, (n, 3))
    if kind == "clusters":
        c = (rng.integers(-8, 8, (12, 3)) + 0.5) * L / 16
        k = 4 * n // 5
        x[:k] = c[rng.integers(0, 12, k)] + rng.normal(0, L / 400, (k, 3))
    else:
        x[: 7 * n // 8] = (0.3, 0.2, 0.1)
    sp = np.where(rng.random(n) < 0.5, 1, -1).astype(np.int8)
    return janus_treepm.to_fixed((x + L / 2) % L - L / 2, L), sp


def _clz(x):
    return 64 - np.array([int(v).bit_length() for v in x])


def _marked(keys, group):
    n = len(keys)
    _, start, count = np.unique(keys >> np.uint64(51), return_index=True, return_counts=True)
    per = (count + group - 1) // group
    first = np.concatenate([s + np.arange(0, c, group) for s, c in zip(start, count)])
    last = np.minimum(first + group, np.repeat(start + count, per)) - 1
    prefix = _clz(keys[first] ^ keys[last])
    before, after = first - REACH * group, last + REACH * group
    hit = (before >= 0) & (_clz(keys[first] ^ keys[np.maximum(before, 0)]) >= prefix)
    hit |= (after < n) & (_clz(keys[first] ^ keys[np.minimum(after, n - 1)]) >= prefix)
    return int(np.sum(hit & (np.repeat(count, per) > REACH * group)))


@pytest.mark.parametrize("kind,n,group,over", CASES)
def test_cases_mark_what_they_are_for(orc, kind, n, group, over):
    marked = _marked(np.sort(orc.morton(_positions(kind, n)[0]) & MASK), group)
    room = (1024 if n < 1024 else n + n // 8) // 256 + 4096
    assert marked > room if over else 10 <= marked <= room


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kind,n,group,over", CASES)
def test_order(jtp, kind, n, group, over, precision):
    print(f"case: early list {kind} n={n} group={group} precision={precision}", flush=True)
    pos, sp = _positions(kind, n)
    p = jtp.default_params(L, 32)
    p.precision, p.group_size = precision, group
    ctx = jtp.ForceContext(p, 1.0, 19.0)
    acc = ctx.compute_forces(pos, sp)
    st = ctx.stats()
    ens = jtp.Ensemble([p, p], [1.0, 1.0], [19.0, 19.0], n_streams=2)
    dp, ds = jtp.DeviceArray.from_host(pos), jtp.DeviceArray.from_host(sp)
    da = [jtp.DeviceArray((n, 3), acc.dtype) for _ in range(2)]
    ens.compute_forces_device([n, n], [dp, dp], [ds, ds], da)
    for d in da:
        assert np.array_equal(d.download(), acc)
    assert ens.stats(1)["interactions"] == st["interactions"] > 0
    assert np.array_equal(ctx.compute_forces(pos, sp), acc)
    ens.close()
    ctx.close()
