"""GPU: calls of the Calc operators that the timed cases do not make: outputs
over their input, non-finite modes that the reference drops."""
import numpy as np
import pytest

from conftest import flush_print, rel, rel_l2

pytestmark = pytest.mark.gpu


def _spectrum(oracle_mod, vb, nx, nz):
    eps = 2.0 * 2 * np.pi / nx
    d, _ = vb.shape(vb.SHAPE_TORUS, 5, nx, nz, 1.0, eps)
    o = oracle_mod.Oracle(nx, nz, eps=eps)
    return o, o.r2c(d)


# one length with x and y in one kernel, two past it
@pytest.mark.parametrize("nx,nz", [(48, 16), (192, 16), (256, 16)])
@pytest.mark.parametrize("which", [0, 1, 2])
def test_gradient_output_over_its_input(vb, gpu, oracle_mod, nx, nz, which):
    """A component written over the spectrum (the storage reused) leaves the other
    two components right."""
    import torch
    flush_print("gradient over fd", nx, nz, which)
    o, fd = _spectrum(oracle_mod, vb, nx, nz)
    ref = o.fftgradient(fd)
    src = torch.from_numpy(fd).to(gpu)
    g = [torch.empty((nz, nx, nx), dtype=torch.float64, device=gpu) for _ in range(3)]
    g[which] = torch.view_as_real(src).reshape(-1)[:nz * nx * nx].view(nz, nx, nx)
    vb.Calc(nx, nz).fftgradient(src, *g)
    # the tolerance of the same operator with separate buffers (test_gpu_plane.py)
    for a, b in zip(g, ref):
        assert rel_l2(a.cpu().numpy(), b) < 1e-12


@pytest.mark.parametrize("nx,nz", [(48, 16), (192, 16), (256, 16)])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_gradient_drops_its_nyquist_modes(vb, gpu, oracle_mod, nx, nz, bad):
    """gradient_kernel writes zero in a component's own Nyquist plane whatever the
    mode holds (Calc.cu:310-339)."""
    import torch
    flush_print("gradient Nyquist", nx, nz, bad)
    _, fd = _spectrum(oracle_mod, vb, nx, nz)
    c = vb.Calc(nx, nz)
    out = lambda: [torch.empty((nz, nx, nx), dtype=torch.float64, device=gpu) for _ in range(3)]
    clean = out()
    c.fftgradient(torch.from_numpy(fd).to(gpu), *clean)
    for axis, plane in enumerate([np.s_[:, :, nx // 2], np.s_[:, nx // 2, :], np.s_[nz // 2, :, :]]):
        f = fd.copy()
        f[plane] = bad
        g = out()
        c.fftgradient(torch.from_numpy(f).to(gpu), *g)
        assert torch.equal(g[axis], clean[axis]), axis


@pytest.mark.parametrize("nx,nz", [(16, 16), (96, 96), (192, 192)])
def test_get_phi_into_pinned_memory(vb, gpu, nx, nz):
    """The caller's own pinned buffer, whole or from its middle, gets what a pageable
    one gets, on the first read and on those that use a staging block."""
    import ctypes as C
    import torch
    flush_print("get_phi pinned", nx, nz)
    eps = 2.0 * 2 * np.pi / nx
    phi, _ = vb.shape(vb.SHAPE_TORUS, 5, nx, nz, 1.0, eps)
    s = vb.Solver(vb.params_default(nx=nx, nz=nz, eps=eps, M1=1e3, M2=1e3, time_step=1e-8, fixed_time_step=1e-8), phi)
    n = nx * nx * nz
    buf = torch.full((2 * n + 64,), -7.0, dtype=torch.float64, pin_memory=True)
    ref = s.get_phi()
    for off in (0, 3, n):
        buf.fill_(-7.0)
        assert vb.lib().vb_get_phi(s.h, C.c_void_p(buf.data_ptr() + 8 * off)) == 0
        out = buf.numpy()
        assert np.array_equal(out[off:off + n].reshape(ref.shape), ref)
        assert (out[:off] == -7.0).all() and (out[off + n:] == -7.0).all()
        for _ in range(3):
            assert np.array_equal(s.get_phi(), ref)


# planes on either side of the rules between one kernel per plane and separate ones
@pytest.mark.parametrize("nx,nz,prec", [(128, 16, "FP64"), (128, 32, "FP64"), (128, 48, "FP64"), (128, 32, "FP32_MIXED"),
                                        (192, 16, "FP32_MIXED"), (192, 32, "FP32_MIXED"), (192, 48, "FP32_MIXED"),
                                        (96, 64, "FP32_MIXED"), (256, 96, "FP32_MIXED"), (192, 128, "FP64")])
def test_transforms_of_few_planes(vb, gpu, oracle_mod, nx, nz, prec):
    import torch
    flush_print("few planes", nx, nz, prec)
    fp64 = prec == "FP64"
    u = np.random.default_rng(nx + nz).standard_normal((nz, nx, nx)).astype(np.float64 if fp64 else np.float32)
    c = vb.Calc(nx, nz, precision=getattr(vb, prec))
    ud = torch.from_numpy(u).to(gpu)
    s = torch.empty((nz, nx, nx // 2 + 1), dtype=torch.complex128 if fp64 else torch.complex64, device=gpu)
    c.r2c(ud, s)
    # the bounds of the round trips in test_gpu_calc.py and test_gpu_plane.py
    tol = 1e-14 if fp64 else 2e-6
    assert rel_l2(s.cpu().numpy().astype(np.complex128), oracle_mod.Oracle(nx, nz).r2c(u.astype(np.float64))) < tol
    keep, back = s.clone(), torch.empty_like(ud)
    c.c2r(s, back)
    assert rel_l2(back.cpu().numpy(), u) < tol and torch.equal(s, keep)


# with x and y in one kernel, in two, in two with aligned scratch rows
@pytest.mark.parametrize("nx,nz", [(48, 16), (128, 16), (192, 16), (256, 32)])
def test_etd41_is_the_inverse_of_its_combine(vb, gpu, oracle_mod, nx, nz):
    """vb_calc_etd41 is the combine of vb_calc_etd42 and its inverse transform
    (Calc.cu:488-517); its inputs are preserved, also where the output lies over one."""
    import torch
    flush_print("etd41", nx, nz)
    _, f = _spectrum(oracle_mod, vb, nx, nz)
    rng = np.random.default_rng(nx)
    fd = torch.from_numpy(f).to(gpu)
    nl = torch.from_numpy(oracle_mod.Oracle(nx, nz).r2c(rng.standard_normal((nz, nx, nx)))).to(gpu)
    c, eps, h = vb.Calc(nx, nz), 4 * np.pi / nx, 1e-5
    b = torch.empty_like(fd)
    c.etd42(b, fd, nl, eps, h)
    real = lambda: torch.empty((nz, nx, nx), dtype=torch.float64, device=gpu)
    ref, out, kf, kn = real(), real(), fd.clone(), nl.clone()
    c.c2r(b, ref)
    c.etd41(out, fd, nl, eps, h)
    # one inverse transform's rounding either way
    assert rel_l2(out.cpu().numpy(), ref.cpu().numpy()) < 1e-14
    assert torch.equal(fd, kf) and torch.equal(nl, kn)
    over = torch.view_as_real(nl).reshape(-1)[:nz * nx * nx].view(nz, nx, nx)
    c.etd41(over, fd, nl, eps, h)
    assert torch.equal(over, out)


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 768, 769, 1023, 1024, 1025, 4095, 4096, 4097, 100003,
                               4096 * 4096, 4096 * 4096 + 1, 2 * 4096 * 4096 + 4099])
def test_integral_of_any_length(vb, gpu, n):
    """Lengths that no chunk, round of four loads or workgroup divides, on either side
    of the chunk's first doubling."""
    import torch
    flush_print("intf_static", n)
    g = torch.Generator(device=gpu).manual_seed(n)
    u = torch.rand(n, generator=g, dtype=torch.float64, device=gpu) + 0.5
    val = torch.zeros(1, dtype=torch.float64, device=gpu)
    vb.intf_static(u, 2.0, 0.25, 3.0, val)
    torch.cuda.synchronize()
    # partial sums of at most 65536 / 1024 rounds, the rest pairwise: far below 200 ulps
    ref = (float(np.mean(u.cpu().numpy())) + 0.25) * 3.0 * 8.0
    assert rel(float(val), ref) < 200 * 2.0 ** -53


def test_get_phi_from_several_threads(vb, gpu):
    """Solvers of several sizes created, read (past the reads that make a pinned
    block) and destroyed by four threads at a time."""
    import threading
    errors = []

    def work(t):
        try:
            for r, n in enumerate([(32, 64, 96, 128)[(t + r) % 4] for r in range(4)]):
                eps = 2.0 * 2 * np.pi / n
                phi, _ = vb.shape(vb.SHAPE_ELLIPSOID, 100 * t + r, n, n, 1.0, eps)
                s = vb.Solver(vb.params_default(nx=n, nz=n, eps=eps, M1=1e3, M2=1e3, time_step=1e-7,
                                                fixed_time_step=1e-7), phi)
                first = s.get_phi()
                assert rel_l2(first, phi) < 1e-14      # the round trip of the transforms
                for _ in range(5):
                    assert np.array_equal(s.get_phi(), first)
                s.close()
        except BaseException as e:   # re-raised below, in the test's thread
            errors.append((t, e))

    flush_print("get_phi from threads")
    th = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not errors, errors
