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


@pytest.mark.parametrize("prec", ["FP64", "FP32_MIXED"])
@pytest.mark.parametrize("n", [32, 96])
def test_euler_after_shape_adjustment_on_the_device(vb, gpu, n, prec):
    """The shape loop with its decisions on the device ends behind attempts that were
    rejected or did not run; the driver that follows starts from the state's own
    integrals, as after the loop on the host."""
    flush_print("euler after shape chain", n, prec)
    eps = 2.0 * 2 * np.pi / n
    phi, _ = vb.shape(1, 20260002, n, n, 1.0, eps)
    runs = []
    for chain in (0, 8):
        s = vb.Solver(vb.params_default(nx=n, nz=n, eps=eps, scheme=vb.EULER, shape_adjust=1, M1=1e4, M2=1e4, alpha=-1.0,
                                        beta=-1.0, time_step=1e-7, fixed_time_step=1e-7, accept_chain=chain,
                                        precision=getattr(vb, prec)), phi)
        s.step(0)
        q = s.query()
        s.step(2)
        runs.append((q, s.state(), s.query(), s.get_phi()))
    assert runs[0][:3] == runs[1][:3] and np.array_equal(runs[0][3], runs[1][3])
