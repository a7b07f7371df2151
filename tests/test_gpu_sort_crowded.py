"""A particle set that lies in one octant cell of the key's top digit sorts about as fast as one that fills the box.

The digits' counts of a segment are added up by as many workgroups as the segment needs.  Tree only, with a short cut, so that
neither the mesh's tile table nor the walk's lists see the crowding.  Medians of the sort phase's device time; the bound
leaves room for the uneven tiles of the partition (a few per cent) and for noise.  With one workgroup to a segment the crowded
set takes 1.9 times as long."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _sort_ms(jtp, pos, reps=15):
    n = len(pos)
    p = jtp.default_params(250.0, 64)
    p.pm_enabled, p.r_cut, p.r_s = 0, 0.125, 0.028
    ctx = jtp.ForceContext(p, 1.0, 1.0)
    dp, ds = jtp.DeviceArray.from_host(pos), jtp.DeviceArray.from_host(np.ones(n, np.int8))
    da = jtp.DeviceArray((n, 3), np.float32)
    ms = []
    for _ in range(reps):
        ctx.compute_forces_device(n, dp, ds, da)
        ms.append(ctx.stats()["ms_sort"])
    perm = ctx.stage(jtp.STAGE_PERM)
    ctx.close()
    return float(np.median(ms[3:])), perm


def test_crowded_segment(jtp, orc):
    n = 4_100_000
    print(f"case: crowded sort n={n}", flush=True)
    pos = np.random.default_rng(7).integers(0, 2 ** 32, (n, 3), dtype=np.uint64).astype(np.uint32)
    spread, _ = _sort_ms(jtp, pos)
    pos >>= np.uint32(3)
    crowded, perm = _sort_ms(jtp, pos)
    mask = np.uint64(~((1 << 16) - 1) & (2 ** 64 - 1))
    assert np.array_equal(perm, np.argsort(orc.morton(pos) & mask, kind="stable").astype(np.int32))
    assert crowded < 1.5 * spread, (crowded, spread)
