"""Initial conditions take no buffer that only a force evaluation needs: the call allocates the same for an interlaced
context (whose evaluation has a second half spectrum, 17 MB here) as for a plain one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _taken(jtp, interlace):
    G, L = 128, 100.0
    p = jtp.default_params(L, G)
    p.precision, p.interlace = jtp.FP64, interlace
    ctx = jtp.ForceContext(p, 1.0, 19.0)
    dp, dv, ds = (jtp.DeviceArray((G ** 3, 3), np.uint32), jtp.DeviceArray((G ** 3, 3), np.float64),
                  jtp.DeviceArray((G ** 3,), np.int8))
    before = jtp.device_memory()[0]
    ctx.generate_ics(jtp.ic_params(box_size=L, n_grid=G), dp, dv, ds, vel_f64=True)
    taken = before - jtp.device_memory()[0]
    ctx.close()
    for d in (dp, dv, ds):
        d.free()
    return taken


def test_ic_memory(jtp):
    print("case: device memory of the initial conditions", flush=True)
    _taken(jtp, 0)  # loads the kernels
    assert abs(_taken(jtp, 1) - _taken(jtp, 0)) < 4 << 20
