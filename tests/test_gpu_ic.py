"""Synthetic particles of the FP64 container: the same particles, in the same order, whether it keeps
them in brick order or in their own, and their cells those of their positions."""
import os
import re

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_places_come_from_the_counted_cells():
    """CPU: no kernel that puts particles at counted places evaluates their positions"""
    text = open(os.path.join(ROOT, "latfield2_amd", "csrc", "particles.hip")).read()
    bodies = re.findall(r"__global__[^{;]*\{.*?\n\}", text, flags=re.S)
    placing = [b for b in bodies if "order64(" in b]
    assert placing
    for b in placing:
        assert "ic_pos(" not in b and "ic_particle(" not in b, b.split("(")[0]


@pytest.mark.gpu
@pytest.mark.parametrize("n", [40000, 50653])
@pytest.mark.parametrize("kind", ["uniform", "lattice", "blobs"])
@pytest.mark.parametrize("masses", [False, True])
def test_f64_synthetic_particles_in_either_order(n, kind, masses):
    torch = pytest.importorskip("torch")
    import latfield2_amd as lf
    import oracle as orc
    from gpu_util import announce

    ng = round(n ** (1 / 3))
    n = ng ** 3 if kind == "lattice" else n
    announce(f"F64 synthetic particles n={n} {kind}")
    # 37^3 particles and more lie in brick order on 20^3, in their own on 128^3 (24 to a brick)
    out = []
    for N in (20, 128):
        p = lf.Particles(N, 50653, lf.F64, ids=True, per_particle_mass=masses)
        if kind == "uniform":
            p.ic_uniform(n, 0.3, 7)
        elif kind == "lattice":
            p.ic_lattice(ng, 0.001 * N, 0.3, 7)  # the displacement is given in cells
        else:
            p.ic_blobs(n, 9, 1.5, 0.02 * N, 0.2, 0.3, 7)
        torch.cuda.synchronize()
        d = p.download()
        assert np.array_equal(d["id"], np.arange(n))
        assert np.array_equal(d["cell"], orc.bin_keys(d["pos"], N))
        assert np.array_equal(d["mass"], np.ones(n))
        out.append(d)
    assert np.array_equal(out[0]["vel"], out[1]["vel"])
    # sigma of a lattice or a blob is formed as a product by N over N: one rounding each
    err = np.abs(out[0]["pos"] - out[1]["pos"])
    assert np.max(np.minimum(err, 1.0 - err)) <= 1e-15
