"""Short power-of-two lines of passes that are too large for the mixed-radix
kernels (mix_pow2 in accfft_amd/csrc/fft_launch.hpp) and of passes just
small enough, along each axis: transforms both ways and the z derivative
against numpy's FFT and the oracle in double precision.  Tolerances as in
test_gpu_mixed_radix."""
import numpy as np
import pytest

from conftest import rel_l2, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("shape", [(512, 512, 16), (300, 100, 16), (512, 16, 500), (60, 16, 500),
                                   (16, 512, 500), (16, 60, 500), (1000, 130, 32), (260, 32, 500)])
def test_transforms(dev, orc, shape, prec):
    import torch
    import accfft_amd as af
    fp, rdt, cdt, tol = ((af.F64, torch.float64, torch.complex128, 1e-12) if prec == "f64"
                         else (af.F32, torch.float32, torch.complex64, 1e-5))
    c = rng(sum(shape)).standard_normal(shape) + 1j * rng(1).standard_normal(shape)
    cd = torch.tensor(c, dtype=cdt, device=dev)
    co = torch.empty_like(cd)
    q = af.Plan("c2c", shape, cd, co, fp, af.ACCFFT_ESTIMATE)
    q.execute_c2c(af.ACCFFT_FORWARD, cd, co)
    torch.cuda.synchronize()
    assert rel_l2(co.cpu().numpy(), np.fft.fftn(c)) < tol
    q.execute_c2c(af.ACCFFT_BACKWARD, co, cd)
    torch.cuda.synchronize()
    assert rel_l2(cd.cpu().numpy() / np.prod(shape), c) < 2 * tol
    q.destroy()
    a = c.real.copy()
    x = torch.tensor(a, dtype=rdt, device=dev)
    h = torch.empty(shape[:2] + (shape[2] // 2 + 1,), dtype=cdt, device=dev)
    back = torch.empty_like(x)
    p = af.Plan("r2c", shape, x, h, fp, af.ACCFFT_ESTIMATE)
    p.execute_r2c(x, h)
    torch.cuda.synchronize()
    assert rel_l2(h.cpu().numpy(), np.fft.rfftn(a)) < tol
    p.execute_c2r(h, back)
    torch.cuda.synchronize()
    assert rel_l2(back.cpu().numpy() / np.prod(shape), a) < 2 * tol
    p.grad(x, None, None, back, mask=4)
    torch.cuda.synchronize()
    assert rel_l2(back.cpu().numpy(), orc.grad(a, 4)[2]) < tol
    p.destroy()
