"""The two-pass kernels (accfft_amd/csrc/fft_two.hpp): every z length, y
length (32 and 64 rows a block, M = 1, 2, 4, 8) and x length they hold, r2c,
c2r (of a spectrum with imaginary parts at DC and Nyquist, which c2r drops)
with and without PRESERVE_INPUT, the operators, the adjoints, and the
separate passes a tuning choice falls back to, against numpy's FFT and the
oracle in double precision.

Tolerances as in test_gpu_mixed_radix: at most 27 levels of rounding."""
import numpy as np
import pytest

from conftest import rel_l2, rng

pytestmark = pytest.mark.gpu

SHAPES = ([(3, 32, z) for z in (32, 64, 128, 256, 512)] +
          [(5, 64, z) for z in (32, 64, 128, 256, 512)] +
          [(x, y, 32) for x in (32, 64, 128, 256, 512) for y in (128, 256, 512)] +
          [(64, 128, 64), (64, 256, 256), (64, 512, 512), (256, 128, 128), (64, 64, 64),
           (18, 64, 64), (7, 32, 32)])


def _t(prec):
    import torch
    import accfft_amd as af
    return ((af.F64, torch.float64, torch.complex128, 1e-12) if prec == "f64"
            else (af.F32, torch.float32, torch.complex64, 1e-5))


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("shape", SHAPES)
def test_transforms(dev, shape, prec):
    import torch
    import accfft_amd as af
    fp, rdt, cdt, tol = _t(prec)
    x = rng(shape[0]).standard_normal(shape)
    xd = torch.tensor(x, dtype=rdt, device=dev)
    h = torch.empty(shape[:2] + (shape[2] // 2 + 1,), dtype=cdt, device=dev)
    ref = np.fft.rfftn(x)
    s = rng(7).standard_normal(ref.shape) + 1j * rng(8).standard_normal(ref.shape)
    t = np.fft.ifft(np.fft.ifft(s, axis=0), axis=1)
    inv = np.fft.irfft(t, n=shape[2], axis=2)
    back = torch.empty_like(xd)
    for flags in (af.ACCFFT_ESTIMATE, af.ACCFFT_ESTIMATE | af.PRESERVE_INPUT):
        p = af.Plan("r2c", shape, xd, h, fp, flags)
        for choice in (-1, -2):  # two passes, one pass per axis
            p.set_tuning(0, choice)
            p.execute_r2c(xd, h)
            torch.cuda.synchronize()
            assert rel_l2(h.cpu().numpy(), ref) < tol
            sd = torch.tensor(s, dtype=cdt, device=dev)
            p.execute_c2r(sd, back)
            torch.cuda.synchronize()
            assert rel_l2(back.cpu().numpy() / np.prod(shape), inv) < tol
            if flags & af.PRESERVE_INPUT:
                assert rel_l2(sd.cpu().numpy(), s) < 1e-6
        p.destroy()


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("shape", SHAPES + [(32, 256, 512)])
def test_c2c(dev, shape, prec):
    """Both directions, two passes and one pass per axis, and a call whose
    output is its input on the same plan."""
    import torch
    import accfft_amd as af
    fp, rdt, cdt, tol = _t(prec)
    x = rng(shape[1]).standard_normal(shape) + 1j * rng(9).standard_normal(shape)
    xd = torch.tensor(x, dtype=cdt, device=dev)
    out = torch.empty_like(xd)
    p = af.Plan("c2c", shape, xd, out, fp, af.ACCFFT_ESTIMATE)
    ref, inv = np.fft.fftn(x), np.fft.ifftn(x)
    for choice in (-1, -2):
        p.set_tuning(0, choice)
        p.execute_c2c(af.ACCFFT_FORWARD, xd, out)
        torch.cuda.synchronize()
        assert rel_l2(out.cpu().numpy(), ref) < tol
        p.execute_c2c(af.ACCFFT_BACKWARD, xd.clone(), out)
        torch.cuda.synchronize()
        assert rel_l2(out.cpu().numpy() / np.prod(shape), inv) < tol
        same = xd.clone()
        p.execute_c2c(af.ACCFFT_FORWARD, same, same)
        torch.cuda.synchronize()
        assert rel_l2(same.cpu().numpy(), ref) < tol
    p.destroy()


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("shape", [(3, 32, 64), (64, 64, 64), (64, 128, 32), (64, 256, 64),
                                   (128, 512, 32), (512, 256, 32), (256, 128, 64)])
def test_operators_and_adjoints(dev, orc, shape, prec):
    import torch
    import accfft_amd as af
    fp, rdt, cdt, tol = _t(prec)
    a = rng(3).standard_normal(shape)
    d = torch.tensor(a, dtype=rdt, device=dev)
    out = [torch.empty_like(d) for _ in range(3)]
    p = af.Plan("r2c", shape, d, out[0], fp, af.ACCFFT_ESTIMATE)
    for name in ("laplace", "biharmonic", "inv_laplace", "inv_biharmonic"):
        getattr(p, name)(d, out[0])
        torch.cuda.synchronize()
        assert rel_l2(out[0].cpu().numpy(), getattr(orc, name)(a)) < tol, name
    for method in (0, 1):
        p.poisson_solve(d, out[0], method)
        torch.cuda.synchronize()
        assert rel_l2(out[0].cpu().numpy(), orc.poisson_solve(a, method)) < tol
    p.grad(d, *out, slow=True)
    torch.cuda.synchronize()
    for x, r in zip(out, orc.grad(a, slow=True)):
        assert rel_l2(x.cpu().numpy(), r) < tol
    hs = shape[:2] + (shape[2] // 2 + 1,)
    G = rng(4).standard_normal(hs) + 1j * rng(5).standard_normal(hs)
    Gd = torch.tensor(G, dtype=cdt, device=dev)
    p.adjoint_r2c(Gd, out[0])
    torch.cuda.synchronize()
    assert rel_l2(out[0].cpu().numpy(), orc.adjoint_r2c(G, shape)) < tol
    p.adjoint_c2r(d, Gd)
    torch.cuda.synchronize()
    assert rel_l2(Gd.cpu().numpy(), orc.adjoint_c2r(a)) < tol
    p.destroy()
