"""lf2mi_poisson_green allocates and is refused under graph capture; lf2mi_poisson_green_noalloc is
captured, and its replays give what eager calls give."""
import ctypes

import pytest

torch = pytest.importorskip("torch")

import latfield2_amd as lf  # noqa: E402
from latfield2_amd import _lib  # noqa: E402
from gpu_util import announce  # noqa: E402

pytestmark = pytest.mark.gpu


def green(name, k, stream):
    return getattr(_lib.load(), name)(ctypes.c_void_p(k.t.data_ptr()), k.N, k.C, k.kh, 1.0 / k.N, 1.0, k.code,
                                      ctypes.c_void_p(stream.cuda_stream))


@pytest.mark.parametrize("code", [lf.F32, lf.F64])
def test_green_is_refused_and_noalloc_taken(code):
    announce(f"poisson_green under capture {code}")
    k = lf.KField(lf.Lattice(3, 24, 1), 1, 1, code)
    k.t.normal_(generator=torch.Generator(device="cuda").manual_seed(1))
    start = k.t.clone()
    side = torch.cuda.Stream()
    assert green("lf2mi_poisson_green_noalloc", k, side) == 0  # its first call looks the table up
    torch.cuda.synchronize()
    k.t.copy_(start)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        with torch.cuda.graph(g, stream=side):
            assert green("lf2mi_poisson_green", k, side) == -3, "refused as a HIP error"
            assert b"captur" in _lib.load().lf2mi_last_error()
            assert green("lf2mi_poisson_green_noalloc", k, side) == 0
    want = start.clone()
    for _ in range(3):
        e = lf.KField(lf.Lattice(3, 24, 1), 1, 1, code)
        e.t.copy_(want)
        torch.cuda.synchronize()
        assert green("lf2mi_poisson_green", e, torch.cuda.current_stream()) == 0
        want = e.t
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(k.t, want)
