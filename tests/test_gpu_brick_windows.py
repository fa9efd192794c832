"""Window deposits and gathers of crowded bricks: how many items a workgroup takes (it depends on the
number of particles), the parts into which the dense bricks of the multi-component tiles are split, and the
lattices and numbers of particles from which those tiles are used; against the FP64 oracle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import latfield2_amd as lf  # noqa: E402
import oracle as orc  # noqa: E402
from gpu_util import announce, real_np, rel_l2  # noqa: E402

pytestmark = pytest.mark.gpu

DT = {"f32": lf.F32, "f64": lf.F64}
KINDS = {"scalar": (lf.PROJ_SCALAR, 1), "vector": (lf.PROJ_VECTOR, 3), "vecvec": (lf.PROJ_VECVEC, 6),
         "vector_ngp": (lf.PROJ_VECTOR_NGP, 3), "tensor_ngp": (lf.PROJ_SYMTENSOR_NGP, 6)}


def oracle(kind, d, N, mass, fold):
    project = dict(scalar=orc.scalar_project, vector=orc.vector_project, vecvec=orc.vecvec_project,
                   vector_ngp=orc.vector_ngp_project, tensor_ngp=orc.symtensor_ngp_project)[kind]
    comm = dict(scalar=orc.scalar_comm, vector=orc.vector_comm, vecvec=orc.vecvec_comm,
                vector_ngp=orc.vector_ngp_comm, tensor_ngp=orc.symtensor_ngp_comm)[kind]
    ref = orc.real_field(N, 1, KINDS[kind][1])
    args = (d["pos"], ref, N, 1) if kind == "scalar" else (d["pos"], d["vel"], ref, N, 1)
    project(*args, mass=mass)
    if fold:
        comm(ref, N, 1)
    return ref


# 160 is the first lattice with the multi-component tiles, 128 the last without; a tile is four bricks
@pytest.mark.parametrize("N", [128, 160, 192])
@pytest.mark.parametrize("masses", [False, True])
def test_dense_bricks_of_the_tiles(N, masses):
    """bricks just below and above the 1024 particles of a dense one, at a part's and a group's border,
    and one of several groups whose last is not full, beside sparse and empty bricks"""
    announce(f"dense bricks N={N} masses={masses}")
    orc.set_threads(16)
    rng = np.random.default_rng(N)
    counts = [1023, 1024, 1025, 2048, 8191, 8192, 8193, 20001]
    pos = [rng.random((5000, 3))]
    for i, c in enumerate(counts):
        brick = np.array([(3 * i) % (N // 8), (N // 8 - 1) * (i % 2), i])  # the upper faces among them
        pos.append((brick * 8 + 8 * rng.random((c, 3))) / N)
    pos = np.concatenate(pos)
    n = len(pos)
    vel = rng.standard_normal((n, 3))
    mass = (0.5 + rng.random(n)) / n if masses else None
    parts = lf.Particles(N, n, lf.F32, per_particle_mass=masses, mass=1.0 / n)
    parts.addParticles(pos, vel, mass)
    d = parts.download()
    for kind, (code, C) in KINDS.items():
        f = lf.Field(lf.Lattice(3, N, 1), C, lf.F32)
        f.t.fill_(7.0)
        parts.deposit(code, f, lf.DEP_PERIODIC_SET)
        torch.cuda.synchronize()
        s = slice(1, N + 1)
        ref = oracle(kind, d, N, d["mass"], True)[s, s, s]
        got = real_np(f)[s, s, s]
        for c in range(C):
            # FP32 products, as the other FP32 deposits are held to
            assert rel_l2(got[..., c], ref[..., c]) <= 1e-6, (kind, c)


# 2048 groups of two items each: below, 4 194 304 particles are taken item by item
@pytest.mark.parametrize("n", [4194303, 4194304])
@pytest.mark.parametrize("prec,tol", [("f32", 1e-6), ("f64", 1e-12)])
def test_items_per_workgroup(n, prec, tol):
    announce(f"items per workgroup n={n} {prec}")
    orc.set_threads(16)
    N = 24
    rng = np.random.default_rng(n)
    pos, vel = rng.random((n, 3)), rng.standard_normal((n, 3))
    pos[: n // 2] = (0.5 + 0.05 * rng.standard_normal((n // 2, 3))) % 1.0
    parts = lf.Particles(N, n, DT[prec], mass=1.0 / n)
    parts.addParticles(pos, vel)
    d = parts.download()
    m = np.full(n, 1.0 / n)
    for kind in ("scalar", "vector"):
        code, C = KINDS[kind]
        f = lf.Field(lf.Lattice(3, N, 1), C, DT[prec])
        parts.deposit(code, f, lf.DEP_UNFOLDED)
        torch.cuda.synchronize()
        ref = oracle(kind, d, N, m, False)
        for c in range(C):
            assert rel_l2(real_np(f)[..., c], ref[..., c]) <= tol, (kind, c)
    if prec == "f64":
        # a particle's kick does not depend on the group that it is in: the same bits from half containers
        phi = lf.Field(lf.Lattice(3, N, 1), 1, lf.F64)
        phi.interior().normal_(generator=torch.Generator(device="cuda").manual_seed(3))
        phi.updateHalo()
        parts.gather_kick_drift(phi, 0.1, 0.0)
        got = parts.download()["vel"]
        for half in (slice(0, n // 2), slice(n // 2, n)):
            q = lf.Particles(N, n // 2 + 1, lf.F64)
            q.addParticles(pos[half], vel[half])
            q.gather_kick_drift(phi, 0.1, 0.0)
            assert np.array_equal(q.download()["vel"], got[half])


@pytest.mark.parametrize("N", [64, 128, 192])
@pytest.mark.parametrize("n", [1, 700, 1500])
def test_few_particles_in_the_scalar_tiles(N, n):
    """few particles on a large lattice, without a dense brick and with one: the launch is then the
    fold's, whose workgroups outnumber the particles' work"""
    announce(f"scalar tiles N={N} n={n}")
    rng = np.random.default_rng(n)
    pos = rng.random((n, 3))
    if n > 1024:
        pos = (N // 8 - 1 + pos) * 8 / N  # all in the last brick, whose upper nodes wrap
    parts = lf.Particles(N, n, lf.F32, mass=1.0 / n)
    parts.addParticles(pos, np.zeros((n, 3)))
    d = parts.download()
    s = slice(1, N + 1)
    ref = oracle("scalar", d, N, np.full(n, 1.0 / n), True)
    for target, before in ((lf.DEP_PERIODIC_SET, 7.0), (lf.DEP_PERIODIC, 0.0)):
        f = lf.Field(lf.Lattice(3, N, 1), 1, lf.F32)
        f.t.fill_(before)
        parts.deposit(lf.PROJ_SCALAR, f, target)
        torch.cuda.synchronize()
        got = real_np(f)
        assert rel_l2(got[s, s, s], ref[s, s, s]) <= 1e-6
        got[s, s, s] = 0.0
        assert not got.any()  # the ghosts are cleared, or were and stay
