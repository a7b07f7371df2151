"""The order in which the walk takes its groups does not show in any result.

A single context walks the groups that straddle large Morton cells first, from a list; the one-launch walk over several
boxes takes every box's groups in Morton order.  Each group's result is its own, so accelerations and interaction
counts are equal bit for bit, whatever share of the groups the list holds: none, some, or more than it has room for."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _box(kind, n, L, rng):
    x = rng.uniform(-L / 2, L / 2, (n, 3))
    if kind == "clusters":  # dense clumps on the faces of large cells, a thin rest
        c = np.round(rng.uniform(-2, 2, (12, 3))) * L / 8
        k = 4 * n // 5
        x[:k] = c[rng.integers(0, 12, k)] + rng.normal(0, L / 400, (k, 3))
    elif kind == "clump":  # coincident particles: every group of the clump is marked
        x[: 7 * n // 8] = (0.3, 0.2, 0.1)
    return (x + L / 2) % L - L / 2


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kind,n,group", [("uniform", 3000, 32), ("clusters", 20011, 32), ("clusters", 20011, 64),
                                          ("clusters", 5003, 7), ("clump", 40000, 7), ("clump", 90, 1), ("clusters", 31, 32)])
def test_order_of_the_groups(jtp, kind, n, group, precision):
    print(f"case: walk order {kind} n={n} group={group} precision={precision}", flush=True)
    L = 50.0
    rng = np.random.default_rng(n)
    sp = np.where(rng.random(n) < 0.5, 1, -1).astype(np.int8)
    pos = jtp.to_fixed(_box(kind, n, L, rng), L)
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
    again = ctx.compute_forces(pos, sp)
    assert np.array_equal(again, acc)
    ens.close()
    ctx.close()
