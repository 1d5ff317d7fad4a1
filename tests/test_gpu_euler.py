"""GPU: forward-Euler steps and the residual of the Euler right-hand side against
the oracle at every length and depth with its own kernels: plane kernels, a
plane update without a plane prefix (FP64 128), flat boxes on either side of its
rule, separate kernels past 128."""
import numpy as np
import pytest

from conftest import flush_print, rel, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["FP64", "FP32_MIXED"])
@pytest.mark.parametrize("nx,nz", [(16, 16), (16, 48), (32, 16), (48, 48), (64, 64), (64, 32), (96, 96), (96, 48),
                                   (128, 16), (128, 32), (128, 48), (128, 64), (128, 128), (192, 16), (192, 64),
                                   (256, 32)])
def test_euler_steps_and_residual(vb, gpu, oracle_mod, nx, nz, prec):
    flush_print("euler", nx, nz, prec)
    # dt under the explicit limit 2 / (eps |k|^4) of the finest grid here
    eps, h, M = 2.0 * 2 * np.pi / nx, 1e-8, 1e3
    phi, _ = vb.shape(vb.SHAPE_ELLIPSOID, 7, nx, nz, 1.0, eps)
    o = oracle_mod.Oracle(nx, nz, eps=eps, M1=M, M2=M, alpha=-1.0, beta=-1.0)
    s = vb.Solver(vb.params_default(nx=nx, nz=nz, eps=eps, scheme=vb.EULER, M1=M, M2=M, alpha=-1.0, beta=-1.0,
                                    time_step=h, fixed_time_step=h, precision=getattr(vb, prec)), phi)
    fp64 = prec == "FP64"
    d = phi.copy()
    st = o.fEIF_begin(d, h, fixed_time_step=h)
    for n in (2, 1):
        assert s.step(n)["status"] == 0
        o.static_steps(d, st, n)
        # FP64: as test_euler_static_steps.  FP32-mixed: the field goes through FP32
        # transforms both ways every step, a few 1e-7 each
        assert rel_l2(s.get_phi(), d) < (1e-11 if fp64 else 3e-6)
        # rounding enters r through lap f, which grows with n against the smooth part:
        # the bounds of test_residual_matches_oracle (32^3) times (n / 32)^2
        o.set_targets(s.state()["alpha"], s.state()["beta"])
        ref = np.mean(o.sum_fgq(d) ** 2) * (2 * np.pi) ** 3
        assert rel(s.residual(), ref) < (1e-11 if fp64 else 1e-4) * max(1.0, (nx / 32.0) ** 2)
