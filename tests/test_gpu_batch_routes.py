"""GPU: the table forms of the kernels past the plane kernels' lengths (k_ypass,
k_xrow, the stage combines): a solve of a batch is its own run, bit for bit."""
import numpy as np
import pytest

from conftest import flush_print, rel, rel_l2

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


# short z under a large plane: the z kernels' wide tile (and, at 192 x 32 in FP64,
# 192 x 128 in FP64, the narrow one that such planes keep)
@pytest.mark.parametrize("nx,nz,prec", [(192, 32, "FP32_MIXED"), (192, 64, "FP32_MIXED"), (192, 64, "FP64"),
                                        (192, 32, "FP64"), (384, 32, "FP64"), (256, 128, "FP64"),
                                        (192, 128, "FP32_MIXED")])
def test_short_z_under_a_large_plane(vb, gpu, oracle_mod, nx, nz, prec):
    flush_print("short z", nx, nz, prec)
    eps, h, M = 2.0 * 2 * np.pi / nx, 1e-7, 1e4
    phi, _ = vb.shape(vb.SHAPE_ELLIPSOID, 11, nx, nz, 1.0, eps)
    o = oracle_mod.Oracle(nx, nz, eps=eps, M1=M, M2=M, alpha=-1.0, beta=-1.0)
    s = vb.Solver(vb.params_default(nx=nx, nz=nz, eps=eps, M1=M, M2=M, alpha=-1.0, beta=-1.0, time_step=h,
                                    fixed_time_step=h, precision=getattr(vb, prec)), phi)
    assert s.step(1)["status"] == 0
    d = phi.copy()
    st = o.fEIF_begin(d, h, fixed_time_step=h)
    o.fEIF_steps(d, st, 1)
    # as test_prefix_in_one_kernel (test_gpu_plane.py)
    tol = 1e-12 if prec == "FP64" else 1e-6
    assert rel_l2(s.get_phi(), d) < tol
    E, V, A, Eb = s.query()
    Eo, Vo, Ao, Ebo = o.energy(d)
    assert rel(V, Vo) < 10 * tol and rel(A, Ao) < 10 * tol
