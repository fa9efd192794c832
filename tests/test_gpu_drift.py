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


@pytest.mark.parametrize("N,n", [(8, 1), (8, 1023), (20, 4097), (64, 70001), (64, 300001)])
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


@pytest.mark.parametrize("N", [8, 20, 64, 160, 168])
def test_sparse_gather_matches_fp64(N):
    """Bricks of few particles, in chunks of one brick (up to 20^3 bricks of 8^3 cells) and of
    several (from 21^3), against the FP64 container.  White noise as the potential: its
    differences cancel nothing, so a velocity carries some 30 FP32 roundings of 6e-8."""
    announce(f"sparse gather N={N}")
    n = 20 * ((N + 7) // 8) ** 3 + 3
    rng = np.random.default_rng(N)
    pos, vel = rng.random((n, 3)), rng.standard_normal((n, 3))
    lat = lf.Lattice(3, N, 1)
    out = {}
    f32 = lf.Field(lat, 1, lf.F32)
    f32.t.normal_(generator=torch.Generator(device="cuda").manual_seed(N))
    f64 = lf.Field(lat, 1, lf.F64)
    f64.t.copy_(f32.t)
    for code, phi in ((lf.F32, f32), (lf.F64, f64)):
        parts = lf.Particles(N, n, code, ids=True)
        assert parts.addParticles(pos, vel, ids=np.arange(n, dtype=np.int64)) == n
        parts.gather_kick_drift(phi, 1.0 / N, 0.01)
        d = parts.download()
        i = np.argsort(d["id"])
        out[code] = (d["vel"][i], d["pos"][i])
    dv = out[lf.F32][0] - out[lf.F64][0]
    assert np.linalg.norm(dv) / np.linalg.norm(out[lf.F64][0]) <= 2e-6
    dx = np.abs(out[lf.F32][1] - out[lf.F64][1])
    assert np.max(np.minimum(dx, 1.0 - dx)) * N <= 1e-4


def test_fixed_deposits_leave_nothing_behind():
    """The fixed-point sums stay in the container between deposits: after one of any kind, target
    and halo, the next must be bit for bit that of a container without a past (integer sums do
    not depend on the order of the particles).  Few particles that move, so that most nodes with
    a value have none the next time."""
    N, n = 64, 4001
    announce("fixed deposits one after the other")
    rng = np.random.default_rng(5)
    parts = lf.Particles(N, n, lf.F32, mass=0.5)
    assert parts.addParticles(rng.random((n, 3)), rng.standard_normal((n, 3))) == n
    fields = {}
    for kind, C, target, halo in ((lf.PROJ_SCALAR, 1, lf.DEP_PERIODIC, 1), (lf.PROJ_SCALAR, 1, lf.DEP_PERIODIC, 1),
                                  (lf.PROJ_SCALAR, 1, lf.DEP_PERIODIC_SET, 2), (lf.PROJ_VECTOR, 3, lf.DEP_PERIODIC, 1),
                                  (lf.PROJ_SCALAR, 1, lf.DEP_PERIODIC_SET, 1), (lf.PROJ_SCALAR, 1, lf.DEP_UNFOLDED, 1),
                                  (lf.PROJ_SCALAR, 1, lf.DEP_PERIODIC, 2), (lf.PROJ_VECVEC, 6, lf.DEP_UNFOLDED, 1),
                                  (lf.PROJ_VECTOR, 3, lf.DEP_PERIODIC_SET, 2)):
        parts.gather_kick_drift(None, 0.0, 0.01)
        d = parts.download()
        new = lf.Particles(N, n, lf.F32, mass=0.5)
        assert new.addParticles(d["pos"], d["vel"]) == n
        got, want = (lf.Field(lf.Lattice(3, N, halo), C, lf.F32) for _ in range(2))
        start = 3.0 if target == lf.DEP_PERIODIC_SET else 0.0
        for p, f in ((parts, got), (new, want)):
            f.t.fill_(start)
            p.deposit(kind, f, target, lf.ACC_FIXED64)
        torch.cuda.synchronize()
        assert torch.equal(got.t, want.t), (kind, target, halo)
        assert float(want.t.abs().max()) > 0 and float((want.t == 0).double().mean()) > 0.3, (kind, target, halo)
