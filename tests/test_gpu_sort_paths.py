"""The particle sort at the edges of its paths (tiles of 2048 and 6144 keys, one segment or 128 partitioned by the top
digit), bit-exact against numpy's stable argsort of the Morton keys; the records against the permuted inputs through
the exported boxes and sums of the tree, and the deposit, which reads the tile starts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SORT_MASK = np.uint64(~((1 << 16) - 1) & (2 ** 64 - 1))


def _positions(kind, n, rng):
    pos = rng.integers(0, 2 ** 32, (n, 3), dtype=np.uint64).astype(np.uint32)
    if kind == "equal":
        pos[:] = (12345, 2 ** 31 + 7, 99)
    elif kind == "one segment":  # every key shares the top digit
        pos >>= np.uint32(3)
    elif kind == "few":  # heavy duplicates in few segments
        pos &= np.uint32(0xC0000000)
    elif kind == "halo":
        pos = (2 ** 31 + rng.normal(0, 1, (n, 3)) * 10.0 ** rng.uniform(5, 9, (n, 1))).astype(np.int64).astype(np.uint32)
    return pos


@pytest.mark.parametrize("kind", ["random", "equal", "one segment", "few", "halo"])
@pytest.mark.parametrize("n", [1, 2, 2047, 2048, 2049, 128 * 2048, 128 * 2048 + 1, 128 * 6144, 128 * 6144 + 1,
                               1_500_007, 4_194_303, 4_194_304])
def test_stable_order(jtp, orc, kind, n):
    print(f"case: sort {kind} n={n}", flush=True)
    rng = np.random.default_rng(n)
    pos = _positions(kind, n, rng)
    sp = np.where(rng.random(n) < 0.5, 1, -1).astype(np.int8)
    p = jtp.default_params(250.0, 64)
    p.tree_enabled = 0
    ctx = jtp.ForceContext(p, 1.0, 0.0)
    ctx.compute_forces(pos, sp)
    keys = orc.morton(pos) & SORT_MASK
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(ctx.stage(jtp.STAGE_PERM), order.astype(np.int32))
    assert np.array_equal(ctx.stage(jtp.STAGE_KEYS), keys[order])
    # species and cells of the records: the m+ mass on the mesh is their count (m- is massless here)
    rho = ctx.stage(jtp.STAGE_RHO).astype(np.float64)
    assert abs(rho.sum() - np.count_nonzero(sp > 0)) <= 1e-5 * max(1, n)
    occupied = np.zeros((64, 64, 64), bool)
    c = (pos[sp > 0] >> np.uint32(26)).astype(np.int64)
    for dz in (0, 1):
        for dy in (0, 1):
            for dx in (0, 1):
                occupied[(c[:, 2] + dz) % 64, (c[:, 1] + dy) % 64, (c[:, 0] + dx) % 64] = True
    assert np.all(rho.reshape(64, 64, 64)[~occupied] == 0)


@pytest.mark.parametrize("precision,pm", [(0, 1), (0, 0), (1, 1)])
@pytest.mark.parametrize("kind,n", [("random", 1), ("random", 2), ("equal", 2049), ("one segment", 2048), ("halo", 2047),
                                    ("random", 128 * 2048), ("few", 128 * 2048 + 1), ("halo", 128 * 2048 + 255)])
def test_group_cells(jtp, orc, kind, n, precision, pm):
    """The gather's level-4 cell starts: the walk's groups are the runs of <= 32 in each cell, and cover every particle."""
    print(f"case: group cells {kind} n={n} precision={precision} pm={pm}", flush=True)
    rng = np.random.default_rng(n + 1)
    pos = _positions(kind, n, rng)
    sp = np.where(rng.random(n) < 0.5, 1, -1).astype(np.int8)
    p = jtp.default_params(250.0, 64)
    p.precision, p.pm_enabled = precision, pm
    ctx = jtp.ForceContext(p, 1.0, 1.0)
    acc = jtp.DeviceArray.from_host(np.full((n, 3), np.nan, np.float64 if precision else np.float32))
    dp, ds = jtp.DeviceArray.from_host(pos), jtp.DeviceArray.from_host(sp)
    ctx.compute_forces_device(n, dp.ptr, ds.ptr, acc.ptr)
    count = np.bincount((orc.morton(pos) >> np.uint64(51)).astype(np.int64), minlength=4096)
    assert ctx.stats()["n_groups"] == np.sum((count + 31) // 32)
    assert np.all(np.isfinite(acc.download()))
