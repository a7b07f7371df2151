"""The mesh solve's passes at every mesh size (x and y in one pass at G = 32, 64, 128; line blocks that end inside a
workgroup elsewhere), one mesh and both interlaced ones in the same launches, against numpy in 64 bits.

Tolerances: an FFT of G^3 points loses about log2(G^3) roundings of the largest intermediate; with the DC mode ~G^1.5
times the others' size removed only at the Green product, the 2-norm error is below 30 eps G^1.5 / 64 of the potential."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _reference(rho, L, r_s, k_min):
    G = rho.shape[0]
    i = np.fft.fftfreq(G) * G
    k = i * 2 * np.pi / L
    k2 = k[:, None, None] ** 2 + k[None, :, None] ** 2 + k[None, None, :] ** 2
    top = np.maximum(np.maximum(abs(i)[:, None, None], abs(i)[None, :, None]), abs(i)[None, None, :])
    green = np.where((top > 0) & (top >= k_min), -4 * np.pi / np.where(k2 > 0, k2, 1) * np.exp(-k2 * r_s ** 2), 0)
    return np.fft.ifftn(np.fft.fftn(rho / (L / G) ** 3) * green).real


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("G", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("k_min", [0, 3])
def test_solve(jtp, G, precision, k_min):
    print(f"case: solve G={G} precision={precision} k_min={k_min}", flush=True)
    L = 100.0
    rng = np.random.default_rng(G)
    rt = np.float64 if precision else np.float32
    rho = (1.0 + rng.standard_normal((G, G, G))).astype(rt)
    s = jtp.PoissonSolver(G, L, r_s=0.8 * L / G, k_min=k_min, precision=precision)
    ref = _reference(rho.astype(np.float64), L, 0.8 * L / G, k_min)
    got = s.solve(rho).astype(np.float64)
    eps = 2.0 ** (-53 if precision else -24)
    assert np.linalg.norm(got - ref) <= 30 * eps * max(1.0, G ** 1.5 / 64) * np.linalg.norm(ref)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("G", [32, 64, 128, 256])
def test_both_meshes_as_one_alone(jtp, G, precision):
    """The two interlaced potentials of a force evaluation, each as the solver gives it for that density alone."""
    print(f"case: two meshes G={G} precision={precision}", flush=True)
    L, n = 100.0, 5000
    rng = np.random.default_rng(1)
    pos = rng.integers(0, 2 ** 32, (n, 3), dtype=np.uint64).astype(np.uint32)
    sp = np.where(rng.random(n) < 0.5, 1, -1).astype(np.int8)
    p = jtp.default_params(L, G)
    p.precision, p.tree_enabled = precision, 0
    ctx = jtp.ForceContext(p, 1.0, 3.0)
    ctx.compute_forces(pos, sp)
    rho, phi = [ctx.stage(k) for k in (jtp.STAGE_RHO, jtp.STAGE_RHO2)], [ctx.stage(k) for k in (jtp.STAGE_PHI, jtp.STAGE_PHI2)]
    for r, f in zip(rho, phi):
        d_r, d_f = jtp.DeviceArray.from_host(r), jtp.DeviceArray(r.shape, r.dtype)
        ctx.pm_solve_device(d_r, d_f)
        assert np.array_equal(d_f.download(), f)
