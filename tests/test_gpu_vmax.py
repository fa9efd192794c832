"""max |v|^2 of the FP64 container's kick: a velocity that is not a number shows in it, particle by
particle and by bricks alike; without one it is the particles' exact maximum."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import latfield2_amd as lf  # noqa: E402
from gpu_util import announce  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 64, 3000, 40000, 50001])
@pytest.mark.parametrize("kick", [False, True])
def test_f64_vmax_keeps_nan(n, kick):
    announce(f"F64 vmax n={n} kick={kick}")
    N = 16
    rng = np.random.default_rng(n)
    pos, vel = rng.random((n, 3)), rng.standard_normal((n, 3))
    phi = lf.Field(lf.Lattice(3, N, 1), 1, lf.F64)  # zero: the velocities stay
    dt = (phi, 0.1, 0.0) if kick else (None, 0.0, 1e-3)
    for bad in (None, 0, n // 2, n - 1):
        v = vel.copy()
        if bad is not None:
            v[bad, bad % 3] = np.nan
        parts = lf.Particles(N, n, lf.F64)
        parts.addParticles(pos, v)
        vm = parts.gather_kick_drift(*dt, want_vmax=True)
        if bad is None:
            # |v|^2 is formed in FP64, fused or not: one rounding per product and sum
            assert abs(vm - np.max(np.sum(v * v, axis=1))) <= 4 * np.finfo(float).eps * vm
        else:
            assert np.isnan(vm), bad
