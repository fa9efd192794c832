"""The ghost folds on both sides of the size from which their three stages are launches of their own
(256, and 216 for six components without lower folds): the oracle's values, ghosts included, bit for bit."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import latfield2_amd as lf  # noqa: E402
import oracle as orc  # noqa: E402
from gpu_util import announce, to_np  # noqa: E402

pytestmark = pytest.mark.gpu

KINDS = [(lf.PROJ_SCALAR, 1, orc.scalar_comm), (lf.PROJ_VECTOR, 3, orc.vector_comm), (lf.PROJ_VECVEC, 6, orc.vecvec_comm),
         (lf.PROJ_VECTOR_NGP, 3, orc.vector_ngp_comm), (lf.PROJ_SYMTENSOR_NGP, 6, orc.symtensor_ngp_comm)]


AROUND = [(k, N) for k in KINDS for N in ((215, 216) if k[0] == lf.PROJ_SYMTENSOR_NGP else (255, 256, 257))]


@pytest.mark.parametrize("kind,C,comm,N", [(*k, N) for k, N in AROUND])
def test_fold_bit_exact_around_the_rule(kind, C, comm, N):
    announce(f"fold N={N} kind={kind}")
    h, G = 1, N + 2
    # only the two outermost layers on each side take part: the inside is zero
    ref = np.zeros((G, G, G, C))
    rng = np.random.default_rng(N)
    for axis in range(3):
        for part in (slice(0, 3), slice(G - 3, G)):
            idx = tuple(part if d == axis else slice(None) for d in range(3))
            ref[idx] = rng.integers(-2 ** 20, 2 ** 20, ref[idx].shape) / 64.0  # their sums are exact in FP32
    f = lf.Field(lf.Lattice(3, N, h), C, lf.F32)
    f.t.copy_(torch.from_numpy(ref.astype(np.float32)).reshape(f.t.shape))
    lf._lib.call("lf2mi_projection_comm", f.t.data_ptr(), N, h, kind, lf.F32, None)
    torch.cuda.synchronize()
    comm(ref, N, h)
    assert np.array_equal(to_np(f.t).reshape(ref.shape).astype(np.float64), ref)
