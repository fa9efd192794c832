"""FP64 container with its brick index (LDS windows of the deposits and of the gather) against
the FP64 oracle, on both sides of the rules on particles per brick and in all, with bricks that
are partial at the upper faces (N not a multiple of 8), through several steps that move particles
across bricks.  Bars: PM steps 1e-10 (FP64 sums in another order, carried through the solve),
deposits 1e-12."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import latfield2_amd as lf  # noqa: E402
import oracle as orc  # noqa: E402
from gpu_util import announce, real_np, rel_l2  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,n", [(16, 24 * 8 - 1), (16, 24 * 8), (16, 9000), (20, 24 * 27), (20, 30011),
                                 (40, 24 * 125 - 1), (40, 70001), (16, 39999), (16, 40000), (20, 45011)])
def test_f64_steps_and_projections_match_oracle(N, n):
    announce(f"F64 bricks N={N} n={n}")
    rng = np.random.default_rng(N + n)
    pos = rng.random((n, 3))
    pos[: n // 3] = (0.98 + 0.03 * rng.standard_normal((n // 3, 3))) % 1.0  # a blob over the box's corner
    vel = 2.0 * rng.standard_normal((n, 3))
    dt, mass = 0.01, 1.0 / n
    parts = lf.Particles(N, n, lf.F64, ids=True, mass=mass)
    ids = rng.permutation(n).astype(np.int64)
    assert parts.addParticles(pos, vel, ids=ids) == n
    lat = lf.Lattice(3, N, 1)
    rho, phi = lf.Field(lat, 1, lf.F64), lf.Field(lat, 1, lf.F64)
    plan = lf.PlanFFT(rho, None)
    p, v = pos.copy(), vel.copy()
    for _ in range(3):
        lf.pm_step(parts, plan, rho, phi, dt, dt)
        ref = orc.pm_step(p, v, N, dt, dt, mass_global=mass)
    torch.cuda.synchronize()
    s = slice(1, N + 1)
    # the oracle returns the density less its mean, the total mass 1
    assert rel_l2(real_np(rho)[s, s, s, 0] - 1.0, ref["rho"][s, s, s, 0]) <= 1e-10
    assert rel_l2(real_np(phi)[s, s, s, 0], ref["phi"][s, s, s, 0]) <= 1e-10
    d = parts.download()
    # upload order, whatever the steps did
    assert np.array_equal(d["id"], ids)
    step = np.abs(d["pos"] - p)
    assert np.max(np.minimum(step, 1.0 - step)) <= 1e-10
    assert rel_l2(d["vel"], v) <= 1e-10
    assert np.array_equal(d["cell"], orc.bin_keys(d["pos"], N))
    m = np.full(n, mass)
    for kind, C, project in ((lf.PROJ_SCALAR, 1, lambda f: orc.scalar_project(d["pos"], f, N, 1, mass=m)),
                             (lf.PROJ_VECTOR, 3, lambda f: orc.vector_project(d["pos"], d["vel"], f, N, 1, mass=m)),
                             (lf.PROJ_VECVEC, 6, lambda f: orc.vecvec_project(d["pos"], d["vel"], f, N, 1, mass=m)),
                             (lf.PROJ_VECTOR_NGP, 3, lambda f: orc.vector_ngp_project(d["pos"], d["vel"], f, N, 1, mass=m)),
                             (lf.PROJ_SYMTENSOR_NGP, 6,
                              lambda f: orc.symtensor_ngp_project(d["pos"], d["vel"], f, N, 1, mass=m))):
        f = lf.Field(lat, C, lf.F64)
        parts.deposit(kind, f, lf.DEP_UNFOLDED)
        torch.cuda.synchronize()
        want = orc.real_field(N, 1, C)
        project(want)
        for c in range(C):
            assert rel_l2(real_np(f)[..., c], want[..., c]) <= 1e-12, (kind, c)
    # a kick alone moves nothing, and its max |v|^2 is the particles'
    vm = parts.gather_kick_drift(phi, dt, 0.0, want_vmax=True)
    e = parts.download()
    assert np.array_equal(e["pos"], d["pos"]) and np.array_equal(e["cell"], d["cell"])
    assert abs(vm - np.max(np.sum(e["vel"] ** 2, axis=1))) <= 1e-12 * vm
    # statistics repeat exactly
    q = [lf.PQ_MVX, lf.PQ_EKIN, lf.PQ_V2]
    a = parts.reduce(q, [lf.SUM, lf.SUM, lf.MAX])
    assert a == parts.reduce(q, [lf.SUM, lf.SUM, lf.MAX])
    assert abs(a[1] - 0.5 * mass * np.sum(e["vel"] ** 2)) <= 1e-12 * a[1]


def test_f64_reordering_keeps_structs_and_upload_order():
    """more drifts than the container waits between two reorderings, with IDs, masses and a
    payload: everything comes back in upload order, and a captured run of steps that holds a
    reordering replays like eager steps"""
    N, n, dt, mass = 16, 42001, 0.01, 1.0 / 42001
    announce(f"F64 reorder N={N} n={n}")
    rng = np.random.default_rng(3)
    part = np.dtype([("ID", "<i8"), ("pos", "<f8", 3), ("vel", "<f8", 3), ("tag", "<f8")])
    a = np.zeros(n, dtype=part)
    a["ID"] = rng.permutation(n)
    a["pos"] = rng.random((n, 3))
    a["vel"] = 0.5 * rng.standard_normal((n, 3))
    a["tag"] = rng.random(n)
    lat = lf.Lattice(3, N, 1)

    def fresh():
        q = lf.Particles(N, n, lf.F64, ids=True, mass=mass)
        q.set_payload(part.itemsize)
        q.upload_structs(a)
        f = lf.Field(lat, 1, lf.F64)
        return q, f, lf.Field(lat, 1, lf.F64), lf.PlanFFT(f, None)

    eager, rho, phi, plan = fresh()
    for _ in range(70):
        lf.pm_step(eager, plan, rho, phi, dt, dt)
    e = eager.download_structs(part)
    p, v = a["pos"].copy(), a["vel"].copy()
    for _ in range(70):
        orc.pm_step(p, v, N, dt, dt, mass_global=mass)
    assert np.array_equal(e["ID"], a["ID"]) and np.array_equal(e["tag"], a["tag"])
    off = np.abs(e["pos"] - p)
    # 70 steps amplify the rounding of the sums' order; a wrong particle would be off by a cell
    assert np.max(np.minimum(off, 1.0 - off)) <= 1e-6
    captured, rho2, phi2, plan2 = fresh()
    side = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        with torch.cuda.graph(g, stream=side):
            for _ in range(35):  # the 32nd reorders
                lf.pm_step(captured, plan2, rho2, phi2, dt, dt)
        for _ in range(2):
            g.replay()
            torch.cuda.synchronize()
    c = captured.download_structs(part)
    assert np.array_equal(c["ID"], a["ID"]) and np.array_equal(c["tag"], a["tag"])
    off = np.abs(c["pos"] - p)
    assert np.max(np.minimum(off, 1.0 - off)) <= 1e-6
