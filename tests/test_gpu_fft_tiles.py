"""FFT tiles whose rows share 128-byte lines with their neighbours (k rows of odd lengths or
behind a ghost), short rows split by all threads, and the wide x-pass workgroups, against the
FP64 oracle.  Bars are those of the other transforms: FP32 2e-6 relative, FP64 1e-12 of the
largest value (a few roundings per radix pass)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import latfield2_amd as lf  # noqa: E402
import oracle as orc  # noqa: E402
from gpu_util import announce, kfield_np, real_np, rel_l2  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,tol", [("f64", 1e-12), ("f32", 2e-6)])
@pytest.mark.parametrize("N,h,kh,C", [(8, 0, 1, 3), (48, 1, 1, 6), (96, 1, 0, 3), (128, 0, 1, 1), (192, 1, 0, 1),
                                      (256, 1, 1, 3), (256, 0, 0, 1), (40, 1, 1, 6), (10, 2, 0, 3)])
def test_fft_tiles_both_ways_match_oracle(prec, tol, N, h, kh, C):
    announce(f"fft tiles {prec} N={N} h={h} kh={kh} C={C}")
    code = lf.F32 if prec == "f32" else lf.F64
    lat = lf.Lattice(3, N, h)
    r, k = lf.Field(lat, C, code), lf.KField(lat, kh, C, code)
    r.t.normal_()
    rin = np.ascontiguousarray(real_np(r))
    plan = lf.PlanFFT(r, k)

    def close(got, ref):
        return rel_l2(got, ref) <= tol if prec == "f32" else np.max(np.abs(got - ref)) <= tol * np.max(np.abs(ref))

    plan.execute(lf.FFT_FORWARD)
    torch.cuda.synchronize()
    kin = kfield_np(k).copy()
    assert close(kin, orc.fft_r2c(rin, N, h, kh))
    r.t.zero_()
    plan.execute(lf.FFT_BACKWARD)
    torch.cuda.synchronize()
    ref = orc.real_field(N, h, C)
    orc.fft_c2r(np.ascontiguousarray(kin), ref, N, h, kh)
    assert close(real_np(r), ref)
    assert np.array_equal(kfield_np(k), kin)


@pytest.mark.parametrize("prec,tol", [("f64", 1e-12), ("f32", 2e-6)])
@pytest.mark.parametrize("N", [8, 10, 12, 20, 24, 32, 40, 48])
def test_small_solves_match_numpy(prec, tol, N):
    """the solve on whole planes (up to 40) and on strided passes against the FP64 transform"""
    announce(f"small solve {prec} N={N}")
    code = lf.F32 if prec == "f32" else lf.F64
    lat = lf.Lattice(3, N, 1)
    rho, phi = lf.Field(lat, 1, code), lf.Field(lat, 1, code)
    rho.t.normal_()
    s = slice(1, N + 1)
    x = real_np(rho)[s, s, s].astype(np.float64)
    lf.poisson_solve(lf.PlanFFT(rho, None), rho, phi, 0.25, 1.0 / N ** 3)
    torch.cuda.synchronize()
    sn = 4.0 * N ** 2 * np.sin(np.pi * np.arange(N) / N) ** 2
    k2 = sn[:, None, None] + sn[None, :, None] + sn[None, None, :]
    k2[0, 0, 0] = np.inf
    want = np.fft.ifftn(-np.fft.fftn(x - 0.25, axes=(0, 1, 2)) / k2[..., None], axes=(0, 1, 2)).real
    assert rel_l2(real_np(phi)[s, s, s], want) <= tol
