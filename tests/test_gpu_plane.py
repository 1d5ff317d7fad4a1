"""GPU parity of the plane kernel (an ETD prefix with a whole xy plane in LDS,
csrc/vb_plane.hpp) and of the wave-wide column tiles of the stage combines, at
every length that has them and at the shortest, odd and cubic depths: one
evaluation, a penalty-drift step and the FP64 energies of a mixed state,
against the oracle."""
import numpy as np
import pytest

from conftest import flush_print, rel, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["FP64", "FP32_MIXED"])
@pytest.mark.parametrize("nx,nz", [(16, 16), (16, 48), (32, 16), (32, 32), (48, 48), (48, 16), (64, 16), (64, 96),
                                   (96, 16), (96, 48), (128, 48), (128, 64), (128, 128), (128, 192)])
def test_prefix_in_one_kernel(vb, gpu, oracle_mod, nx, nz, prec):
    flush_print("plane", nx, nz, prec)
    eps = 2.0 * 2 * np.pi / nx
    phi, _ = vb.shape(vb.SHAPE_ELLIPSOID, 11, nx, nz, 1.0, eps)
    # the reference's ETDRK4 brackets cancel at |h L^| << 1e-5: the wide interface
    # of the 16^2 plane needs a longer step, and that one weaker penalties
    h, M = (1e-5, 1e2) if nx == 16 else (1e-7, 1e4)
    o = oracle_mod.Oracle(nx, nz, eps=eps, M1=M, M2=M, alpha=-1.0, beta=-1.0)
    p = vb.params_default(nx=nx, nz=nz, eps=eps, M1=M, M2=M, alpha=-1.0, beta=-1.0, time_step=h,
                          fixed_time_step=h, precision=getattr(vb, prec))
    s = vb.Solver(p, phi)
    r = s.step(3)
    assert r["status"] == 0 and r["evaluations"] == 6
    d = phi.copy()
    st = o.fEIF_begin(d, h, fixed_time_step=h)
    o.fEIF_steps(d, st, 3)
    # FP64: as the other driver tests.  FP32-mixed: six evaluations that each add
    # h N^ with the rounding of FP32 transforms, a few 1e-7 of h N^, which is
    # itself below the field: 1e-6 of the field bounds it
    tol = 1e-12 if prec == "FP64" else 1e-6
    assert rel_l2(s.get_phi(), d) < tol
    # V and A of the state: FP64 integrals in both precisions; their difference is
    # that of the fields, to first order
    E, V, A, Eb = s.query()
    Eo, Vo, Ao, Ebo = o.energy(d)
    assert rel(V, Vo) < 10 * tol and rel(A, Ao) < 10 * tol
    if prec == "FP64":
        assert rel(Eb, Ebo) < 1e-11


# solves per batch such that all, the last ones or none of them have their planes
# in two workgroups (a round is 256 planes)
@pytest.mark.parametrize("nx,nz,count,prec", [(128, 128, 1, "FP64"), (128, 128, 2, "FP64"), (128, 128, 3, "FP32_MIXED"),
                                              (96, 48, 6, "FP64"), (64, 64, 5, "FP32_MIXED"), (64, 16, 17, "FP32_MIXED")])
def test_prefix_with_two_workgroups_per_plane(vb, gpu, nx, nz, count, prec):
    """Which planes are shared out is not seen in the result: every solve of a
    batch is its own run, bit for bit."""
    flush_print("split planes", nx, nz, count, prec)
    eps = 2.0 * 2 * np.pi / nx
    ps, phis = [], []
    for k in range(count):
        phi, _ = vb.shape(vb.SHAPE_ELLIPSOID, 30 + k, nx, nz, 1.0, eps)
        ps.append(vb.params_default(nx=nx, nz=nz, eps=eps, M1=1e4, M2=1e4, alpha=-1.0, beta=-1.0, time_step=1e-7,
                                    fixed_time_step=1e-7, precision=getattr(vb, prec), phi_lut_mode=1))
        phis.append(phi)
    b = vb.Batch(ps, phis)
    reps = b.step(3)
    for i in {0, count - 2, count - 1} & set(range(count)):
        assert reps[i]["status"] == 0
        s = vb.Solver(ps[i], phis[i])
        s.step(3)
        assert np.array_equal(b.get_phi(i), s.get_phi()) and b.query(i) == s.query(), i


@pytest.mark.parametrize("nx,nz", [(16, 16), (48, 32), (96, 16), (128, 16), (192, 16), (256, 16)])
def test_calc_operators_per_route(vb, gpu, oracle_mod, nx, nz):
    """The Laplacians and gradients where x and y run as one kernel, and past it
    (192 and 256 in FP64), and the integral of a length that no chunk divides."""
    import torch
    flush_print("calc", nx, nz)
    eps = 2.0 * 2 * np.pi / nx
    d, _ = vb.shape(vb.SHAPE_TORUS, 5, nx, nz, 1.0, eps)
    o = oracle_mod.Oracle(nx, nz, eps=eps)
    c = vb.Calc(nx, nz)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)
    real = lambda: torch.empty((nz, nx, nx), dtype=torch.float64, device=gpu)
    fd = o.r2c(d)
    # a transform rounds at ~5e-16 of the field, white over the modes; |k|^2 raises
    # that by at most 3 (n/2)^2 / (1/eps^2) ~ 120 relative to the result: 6e-14
    out, src = real(), T(fd)
    c.lap_spec(src, out)
    ref = o.lap_real(d)
    assert rel_l2(out.cpu().numpy(), ref) < 1e-12
    assert np.array_equal(src.cpu().numpy(), fd)
    c.lap_real(T(d), out)
    assert rel_l2(out.cpu().numpy(), ref) < 1e-12
    g = [real() for _ in range(3)]
    c.fftgradient(src, *g)
    for a, b in zip(g, o.fftgradient(fd)):
        assert rel_l2(a.cpu().numpy(), b) < 1e-12
    assert rel(c.intf(T(d), 1.0, 0.5), o.intf(d, 1.0, 0.5)) < 1e-13


@pytest.mark.parametrize("nx,nz", [(16, 32), (48, 16), (96, 96), (192, 16), (256, 16)])
def test_calc_fp32_round_trip_per_route(vb, gpu, oracle_mod, nx, nz):
    import torch
    u = np.random.default_rng(nx).standard_normal((nz, nx, nx)).astype(np.float32)
    c = vb.Calc(nx, nz, precision=vb.FP32_MIXED)
    ud = torch.from_numpy(u).to(gpu)
    s = torch.empty((nz, nx, nx // 2 + 1), dtype=torch.complex64, device=gpu)
    c.r2c(ud, s)
    assert rel_l2(s.cpu().numpy().astype(np.complex128), oracle_mod.Oracle(nx, nz).r2c(u.astype(np.float64))) < 2e-6
    keep = s.clone()
    back = torch.empty_like(ud)
    c.c2r(s, back)
    assert rel_l2(back.cpu().numpy(), u) < 2e-6
    assert torch.equal(s, keep)
