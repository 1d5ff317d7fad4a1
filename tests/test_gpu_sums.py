"""GPU: the rounding of the integrals' partial sums in FP32-mixed mode.  A
thread of an x kernel adds the values of one row it holds, E of them, in FP32;
everything past that is FP64."""
import numpy as np
import pytest

from conftest import flush_print

pytestmark = pytest.mark.gpu


# elements per thread of the row transform that ends in the sums
@pytest.mark.parametrize("n,E", [(32, 8), (64, 8), (96, 12), (128, 16), (256, 16)])
def test_integral_sums_in_fp32_cover_one_row(vb, gpu, n, E):
    """A uniform field: every transform of it is exact in FP32, so each thread adds
    E equal terms, and A carries the rounding of that chain and nothing else.
    The error of a chain of m equal terms is at most about m / 3 units of 2^-24
    (half an ulp of each partial sum over the total); the values are ones whose
    chain of 2 E terms exceeds the bound of E (8.4 units at 128, 4.3 at 64)."""
    flush_print("sums", n)
    v = {64: 453, 128: 353}.get(n, 353) / 2048.0   # v^2 - 1 is exact in FP32
    eps, h, target = 2.0 * 2 * np.pi / n, 1e-14, 50.0
    # M = 1 moves the state by h (V - alpha) / 2 ~ 1e-12, far below an FP32 ulp
    p = vb.params_default(nx=n, nz=n, eps=eps, M1=1.0, M2=1.0, alpha=100.0, beta=target, time_step=h,
                          fixed_time_step=h, precision=vb.FP32_MIXED, phi_lut_mode=1)
    s = vb.Solver(p, np.full((n, n, n), v))
    assert s.step(1)["status"] == 0
    A = 0.25 / eps * (v * v - 1.0) ** 2 * 3.0 / (2.0 * np.sqrt(2.0)) * (2 * np.pi) ** 3
    # a penalty-drift step moves beta twice, beta -= A - beta0: by the A of the
    # first evaluation, whose sums are FP64, and by that of the new state
    A2 = 3.0 * target - s.state()["beta"] - A
    assert abs(A2 / A - 1.0) < E / 3.0 * 2.0 ** -24


@pytest.mark.parametrize("n,prec", [(32, "FP64"), (64, "FP32_MIXED"), (128, "FP64")])
def test_residual_between_attempts_changes_nothing(vb, gpu, n, prec):
    """vb_residual leaves another prefix (and, at 128 in FP64, another number of
    partial sums) than the attempts around it."""
    flush_print("residual between attempts", n, prec)
    eps = 2.0 * 2 * np.pi / n
    phi, _ = vb.shape(vb.SHAPE_ELLIPSOID, 4, n, n, 1.0, eps)
    p = vb.params_default(nx=n, nz=n, eps=eps, M1=1e3, M2=1e3, alpha=-1.0, beta=-1.0, time_step=1e-7,
                          fixed_time_step=0.0, precision=getattr(vb, prec))
    runs = []
    for ask in (False, True):
        s = vb.Solver(p, phi)
        for k in range(3):
            r = s.step(4)
            if ask and k < 2:   # (a query right after it reads the Euler prefix's own sums)
                assert np.isfinite(s.residual())
        runs.append((r["energy"], s.query(), s.state(), s.get_phi()))
    assert runs[0][:3] == runs[1][:3] and np.array_equal(runs[0][3], runs[1][3])
