"""FP64 container under graph capture: what a capture records depends on the capture alone, and a
drift that is only recorded changes nothing that the container knows of its particles."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import latfield2_amd as lf  # noqa: E402
from gpu_util import announce  # noqa: E402

pytestmark = pytest.mark.gpu


def recorded(parts, drifts):
    """number of nodes of a capture of `drifts` drifts, which is not replayed"""
    # the HIP runtime that is loaded already
    hip = ctypes.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line))
    side = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.stream(side):
        with torch.cuda.graph(g, stream=side):
            for _ in range(drifts):
                parts.gather_kick_drift(None, 0.0, 1e-3)
    torch.cuda.synchronize()
    n = ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(ctypes.c_void_p(g.raw_cuda_graph()), None, ctypes.byref(n)) == 0
    return n.value


def container(N, n, shift=0.0):
    rng = np.random.default_rng(n)
    parts = lf.Particles(N, n, lf.F64)
    pos = rng.random((n, 3))
    parts.addParticles(pos + shift, 0.1 * rng.standard_normal((n, 3)))
    return parts, pos


def test_a_capture_counts_its_own_drifts():
    announce("F64 capture: reordering")
    parts, _ = container(16, 41000)
    one = recorded(parts, 1)
    for _ in range(31):
        parts.gather_kick_drift(None, 0.0, 1e-3)
    assert recorded(parts, 1) == one  # the 32nd drift reorders, but not in a graph of one
    assert recorded(parts, 31) == 31 * one
    assert recorded(parts, 32) > 32 * one  # this one holds a reordering, and so does every other like it
    assert recorded(parts, 32) > 32 * one
    assert recorded(parts, 1) == one


@pytest.mark.parametrize("n", [2000, 41000])
def test_a_recorded_drift_has_moved_nothing(n):
    """positions a box length away: accepted, and wrapped by the next kick, also after a drift was
    recorded and not replayed"""
    announce(f"F64 capture: positions beyond the box n={n}")
    parts, pos = container(16, n, shift=1.0)
    recorded(parts, 1)
    assert np.array_equal(parts.download()["pos"], pos + 1.0)
    phi = lf.Field(lf.Lattice(3, 16, 1), 1, lf.F64)
    parts.gather_kick_drift(phi, 0.1, 0.0)
    d = parts.download()
    assert np.array_equal(d["pos"], (pos + 1.0) - 1.0)
