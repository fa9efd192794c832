"""The first use of a container or a differentiable model on a stream that does not wait for the null
stream, right after it is made: their counters are clear by then."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import latfield2_amd as lf  # noqa: E402
from latfield2_amd.diffpm import DiffPM  # noqa: E402
from gpu_util import announce  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("code", [lf.F32, lf.F64])
def test_container_used_at_once_on_another_stream(code):
    announce(f"first use {code}")
    N, n = 64, 50000
    busy = torch.empty(2 ** 28, device="cuda")
    side = torch.cuda.Stream()
    for k in range(3):
        for _ in range(20):
            busy.fill_(float(k))  # the null stream has work before the clears
        p = lf.Particles(N, n, code, ids=True)
        with torch.cuda.stream(side):
            p.ic_uniform(n, 0.1, 5 + k)
            p.gather_kick_drift(None, 0.0, 0.01)
            d = p.download()
        assert np.array_equal(np.sort(d["id"]), np.arange(n))
        assert p.count() == n


def test_model_used_at_once_on_another_stream():
    announce("first use of a differentiable model")
    N, n = 32, 20000
    g = torch.Generator(device="cuda").manual_seed(2)
    x = torch.rand((n, 3), generator=g, device="cuda", dtype=torch.float64)
    ref = DiffPM(N, n, 2, 1.0 / n, 0.01, lf.F64)
    want = ref.forward(x)
    torch.cuda.synchronize()
    busy = torch.empty(2 ** 28, device="cuda")
    side = torch.cuda.Stream()
    for k in range(3):
        for _ in range(20):
            busy.fill_(float(k))
        m = DiffPM(N, n, 2, 1.0 / n, 0.01, lf.F64)
        with torch.cuda.stream(side):
            got = m.forward(x)
        # the sums of an evaluation differ in their last bits from run to run
        assert abs(got - want) <= 1e-10 * abs(want)
