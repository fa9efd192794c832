"""FP32 container: the drift, which the re-bucketing evaluates as it moves the particles, against
the same formula in FP64.  The start positions are read back exactly (cell + FP32 offset); the
drift rounds the new offset to FP32 (at most 2^-25 cells, or 2^-24 where it is kept below 1),
and the positions' own FP64 roundings stay below 1e-12 cells."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import latfield2_amd as lf  # noqa: E402
from gpu_util import announce  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,n", [(8, 1), (8, 1023), (20, 4097), (64, 70001)])
@pytest.mark.parametrize("speed", [0.01, 3.0])
def test_drift_moves_every_particle_once(N, n, speed):
    announce(f"drift N={N} n={n} speed={speed}")
    rng = np.random.default_rng(N + n)
    parts = lf.Particles(N, n, lf.F32, ids=True, per_particle_mass=True)
    mass = 1.0 + np.arange(n) % 7
    assert parts.addParticles(rng.random((n, 3)), speed * rng.standard_normal((n, 3)), ids=np.arange(n, dtype=np.int64),
                              mass=mass) == n
    for dt in (0.5, -0.25):
        a = parts.download()
        parts.gather_kick_drift(None, 0.0, dt)
        b = parts.download()
        ia, ib = np.argsort(a["id"]), np.argsort(b["id"])
        assert np.array_equal(b["id"][ib], np.arange(n)) and np.array_equal(b["mass"][ib], mass)
        assert np.array_equal(a["vel"][ia], b["vel"][ib])
        X = a["pos"][ia] * N + dt * a["vel"][ia] * N
        d = np.abs(X - b["pos"][ib] * N)
        d -= N * np.rint(d / N)
        assert np.max(np.abs(d)) <= 2.0 ** -24 + 1e-12
        c = b["cell"]
        off = b["pos"] * N - np.stack([c % N, c // N % N, c // N ** 2], axis=1)
        assert np.min(off) >= -1e-12 and np.max(off) <= 1.0
        assert np.array_equal(parts.cell_counts().cpu().numpy(), np.bincount(c, minlength=N ** 3))
