"""GPU: the table forms of the kernels past the plane kernels' lengths (k_ypass,
k_xrow, the stage combines): a solve of a batch is its own run, bit for bit."""
import numpy as np
import pytest

from conftest import flush_print

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nz,count,prec", [(192, 16, 4, "FP32_MIXED"), (192, 32, 3, "FP64"), (256, 16, 2, "FP32_MIXED"),
                                              (256, 32, 3, "FP64"), (128, 32, 5, "FP32_MIXED"), (128, 16, 2, "FP64"),
                                              (384, 16, 2, "FP32_MIXED")])
def test_batched_solve_is_its_own_run(vb, gpu, nx, nz, count, prec):
    flush_print("batch", nx, nz, count, prec)
    eps = 2.0 * 2 * np.pi / nx
    ps, phis = [], []
    for k in range(count):
        phi, _ = vb.shape(vb.SHAPE_ELLIPSOID, 60 + k, nx, nz, 1.0, eps)
        ps.append(vb.params_default(nx=nx, nz=nz, eps=eps, M1=1e4, M2=1e4, alpha=-1.0, beta=-1.0, time_step=1e-7,
                                    fixed_time_step=1e-7, precision=getattr(vb, prec), phi_lut_mode=1))
        phis.append(phi)
    b = vb.Batch(ps, phis)
    reps = b.step(8)
    for i in range(count):
        assert reps[i]["status"] == 0
        s = vb.Solver(ps[i], phis[i])
        s.step(8)
        assert np.array_equal(b.get_phi(i), s.get_phi()) and b.query(i) == s.query(), i
