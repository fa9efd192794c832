"""What the differentiable run keeps for its backward pass: the gradients of a model that keeps every
step's potential and index and of one that computes them again, both against the FP64 oracle, and
the bound on the memory that keeping may take."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from gpu_util import announce, rel_l2  # noqa: E402
from latfield2_amd import F32, F64, _lib  # noqa: E402
from latfield2_amd.diffpm import DiffPM  # noqa: E402

pytestmark = pytest.mark.gpu


def model(N, n, nsteps, dt, dtype, keep):
    """a DiffPM on a handle that may spend `keep` bytes on kept potentials and indexes"""
    m = DiffPM(N, n, nsteps, 1.0 / n, dt, dtype)
    _lib.call("lf2mi_diffpm_destroy", m.h)
    m.h = None
    h = ctypes.c_void_p()
    _lib.call("lf2mi_diffpm_create_keep", N, n, nsteps, 1.0 / n, dt, m.code, keep, ctypes.byref(h))
    m.h = h
    return m


# no steps, one (nothing but an index to keep), several; one particle, ragged counts, several to a cell
@pytest.mark.parametrize("N,n,nsteps", [(8, 1, 2), (8, 700, 0), (16, 5001, 1), (16, 4099, 4), (32, 3000, 3)])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_kept_and_recomputed_gradients_match_oracle(N, n, nsteps, prec):
    import oracle as orc
    announce(f"diffpm kept and recomputed N={N} n={n} steps={nsteps} {prec}")
    dt = 0.02
    rng = np.random.default_rng(n + nsteps)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    made = [model(N, n, nsteps, dt, F64 if prec == "f64" else F32, keep) for keep in (0, 1 << 30)]
    if nsteps:
        # a potential for each step but the first and an index (4 bytes a particle and more) for each state
        tsize = 8 if prec == "f64" else 4
        more = made[1].bytes() - made[0].bytes()
        assert more >= (nsteps - 1) * (N + 2) ** 3 * tsize + nsteps * 4 * n
    # sums of some hundred terms over a few steps, as the bounds of the other tests of this run
    tol = dict(f64=(1e-11, 1e-9), f32=(1e-5, 1e-4))[prec]
    for _ in range(2):  # the second evaluation works on what the first left
        pos0, vel0, tpos = rng.random((n, 3)), rng.normal(0.0, 0.05, (n, 3)), rng.random((n, 3))
        target = orc.cic_density(tpos, N, 1.0 / n)
        L, gp, gv = orc.diffpm_loss_grad(pos0, vel0, N, 1.0 / n, dt, nsteps, target)
        for m in made:
            loss = m.forward(dev(pos0), dev(vel0), dev(target.ravel()))
            for _ in range(2):  # a backward pass can be repeated
                ggp, ggv = m.backward()
                torch.cuda.synchronize()
                assert abs(loss - L) <= tol[0] * L
                assert rel_l2(ggp.cpu().numpy(), gp) <= tol[1]
                if nsteps:
                    assert rel_l2(ggv.cpu().numpy(), gv) <= tol[1]


def test_default_keeps_at_most_an_eighth_of_the_free_memory():
    announce("diffpm memory bound")
    N, n, dt = 256, 64, 0.01
    field = 4 * (N + 2) ** 3
    torch.cuda.empty_cache()
    free, _ = torch.cuda.mem_get_info()
    steps = int(free // 8 // field) + 16  # their potentials are more than an eighth
    m = DiffPM(N, n, steps, 1.0 / n, dt, F32)
    # the fields and the FFT's workspace, tables, and some hundred bytes a particle and step
    assert m.bytes() <= 8 * field + 2 ** 24 + 4096 * n + 512 * n * steps
    assert DiffPM(N, n, 4, 1.0 / n, dt, F32).bytes() >= 8 * field  # few steps are kept: three more fields
