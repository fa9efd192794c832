"""Which FP64 containers keep a brick index, what it costs them, and what they do on either side of the
rule (40 000 particles and 24 per 8^3-cell brick, bricks.hpp): steps against the oracle, struct members
as masses and vectors before and after the particles are put into brick order again."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import latfield2_amd as lf  # noqa: E402
import oracle as orc  # noqa: E402
from gpu_util import announce, real_np, rel_l2  # noqa: E402

pytestmark = pytest.mark.gpu

STATE, INDEX = 52, 20  # bytes a particle: cell, position, velocity; list, rank, place and an 8-byte scratch


@pytest.mark.parametrize("N,cap,index", [(16, 39999, False), (16, 40000, True), (15, 50000, False),
                                         (96, 24 * 12 ** 3 - 1, False), (96, 24 * 12 ** 3, True),
                                         (128, 90000, False), (256, 500000, False), (20, 45011, True)])
def test_index_memory(N, cap, index):
    announce(f"F64 index memory N={N} capacity={cap}")
    bricks = ((N + 7) // 8) ** 3
    got = lf.Particles(N, cap, lf.F64).bytes()
    small = 2 ** 17  # the statistics' partials
    assert cap * STATE <= got
    if index:
        assert cap * (STATE + INDEX) <= got <= cap * (STATE + INDEX) + 32 * bricks + cap // 128 + small
    else:
        assert got <= cap * STATE + small


# the occupancy rule decides on 96^3, the number of particles on 20^3 and 16^3
@pytest.mark.parametrize("N,n", [(96, 24 * 12 ** 3 - 1), (96, 24 * 12 ** 3), (20, 39999), (20, 40003), (17, 41000)])
def test_steps_on_both_sides_of_the_rule(N, n):
    announce(f"F64 rule N={N} n={n}")
    rng = np.random.default_rng(N + n)
    pos, vel = rng.random((n, 3)), 0.5 * rng.standard_normal((n, 3))
    dt, mass = 0.01, 1.0 / n
    parts = lf.Particles(N, n, lf.F64, mass=mass)
    parts.addParticles(pos, vel)
    lat = lf.Lattice(3, N, 1)
    f = lf.Field(lat, 1, lf.F64)
    phi = lf.Field(lat, 1, lf.F64)
    phi.t.copy_(torch.from_numpy(0.01 * rng.standard_normal(tuple(phi.t.shape))))
    phi.updateHalo()
    for _ in range(2):  # the second deposit follows a drift
        f.zero()
        parts.deposit(lf.PROJ_SCALAR, f, lf.DEP_UNFOLDED)
        torch.cuda.synchronize()
        d = parts.download()
        want = orc.real_field(N, 1, 1)
        orc.scalar_project(d["pos"], want, N, 1, mass=np.full(n, mass))
        assert rel_l2(real_np(f), want) <= 1e-12
        parts.gather_kick_drift(phi, dt, dt)
    # the cells are those of the moved positions
    assert np.array_equal(parts.download()["cell"], orc.bin_keys(parts.download()["pos"], N))


@pytest.mark.parametrize("n", [20011, 44444])
def test_masses_and_vectors_of_structs(n):
    """a member of the kept structs as the mass, another as the deposited vector, of particles in
    their own order (20 011) and in brick order (44 444), before and after more than 32 drifts"""
    announce(f"F64 struct members n={n}")
    N = 16
    rng = np.random.default_rng(n)
    part = np.dtype([("ID", "<i8"), ("pos", "<f8", 3), ("vel", "<f8", 3), ("mass", "<f8"), ("q", "<f8", 3), ("m4", "<f8")])
    a = np.zeros(n, dtype=part)
    a["ID"] = rng.permutation(n)
    a["pos"], a["vel"] = rng.random((n, 3)), 0.5 * rng.standard_normal((n, 3))
    a["mass"], a["m4"] = rng.random(n), rng.random(n)
    a["q"] = rng.standard_normal((n, 3))
    parts = lf.Particles(N, n, lf.F64, ids=True)
    parts.set_payload(part.itemsize)
    parts.upload_structs(a)
    lat = lf.Lattice(3, N, 1)
    for drifts in (0, 40):
        for _ in range(drifts):
            parts.gather_kick_drift(None, 0.0, 0.01)
        s = parts.download_structs(part)
        assert np.array_equal(s["ID"], a["ID"]) and np.array_equal(s["q"], a["q"]) and np.array_equal(s["m4"], a["m4"])
        for member in ("mass", "m4"):
            parts.mass_from(lf.MASS_PART, part.fields[member][1])
            # the total is summed in a fixed tree over the particles
            total = parts.reduce([lf.PQ_MASS], [lf.SUM])[0]
            assert abs(total - a[member].sum()) <= 1e-12 * total
            f = lf.Field(lat, 1, lf.F64)
            parts.deposit(lf.PROJ_SCALAR, f, lf.DEP_UNFOLDED)
            want = orc.real_field(N, 1, 1)
            orc.scalar_project(s["pos"], want, N, 1, mass=a[member])
            torch.cuda.synchronize()
            assert rel_l2(real_np(f), want) <= 1e-12, member
            for source, offset in ((s["vel"], -1), (a["q"], part.fields["q"][1])):
                parts.vector_from(offset, lf.F64)
                f = lf.Field(lat, 3, lf.F64)
                parts.deposit(lf.PROJ_VECTOR, f, lf.DEP_UNFOLDED)
                want = orc.real_field(N, 1, 3)
                orc.vector_project(s["pos"], np.ascontiguousarray(source), want, N, 1, mass=a[member])
                torch.cuda.synchronize()
                assert rel_l2(real_np(f), want) <= 1e-12, (member, offset)
