"""Prime stages of the dynamic engine: radices 11 and 13 in registers, larger
primes by the symmetric pair form with the roots in LDS (or read from the
table where the tile fills the LDS: 9973 FP32, 5003 FP64), squares and
products of primes (a second prime stage has twiddles), on every axis
against numpy's FFT in double precision.  Tolerances: a direct sum over p
terms has a relative rounding error of at most about p eps per stage and
sqrt(p) eps on random data; 1e-12 and 1e-5 leave both a factor above 10."""
import numpy as np
import pytest

from conftest import rel_l2, rng

pytestmark = pytest.mark.gpu

LENGTHS = [11, 13, 17, 22, 143, 169, 289, 323, 17 * 64, 31 * 45, 127, 509, 1021]
BIG = {"f64": [5003], "f32": [9973, 17 * 600]}


def _cases():
    for prec in ("f64", "f32"):
        for n in LENGTHS + BIG[prec]:
            for axis in range(3):
                yield prec, n, axis


@pytest.mark.parametrize("prec,n,axis", list(_cases()))
def test_prime_length(dev, prec, n, axis):
    import torch
    import accfft_amd as af
    fp, rdt, cdt, tol = ((af.F64, torch.float64, torch.complex128, 1e-12) if prec == "f64"
                         else (af.F32, torch.float32, torch.complex64, 1e-5))
    shape = [3, 3, 3]
    shape[axis] = n
    c = rng(n).standard_normal(shape) + 1j * rng(n + 1).standard_normal(shape)
    cd = torch.tensor(c, dtype=cdt, device=dev)
    co = torch.empty_like(cd)
    q = af.Plan("c2c", shape, cd, co, fp, af.ACCFFT_ESTIMATE)
    q.execute_c2c(af.ACCFFT_FORWARD, cd, co)
    torch.cuda.synchronize()
    assert rel_l2(co.cpu().numpy(), np.fft.fftn(c)) < tol
    q.execute_c2c(af.ACCFFT_BACKWARD, co, cd)
    torch.cuda.synchronize()
    assert rel_l2(cd.cpu().numpy() / np.prod(shape), c) < tol
    q.destroy()
    xd = torch.tensor(c.real.copy(), dtype=rdt, device=dev)
    h = torch.empty(shape[:2] + [shape[2] // 2 + 1], dtype=cdt, device=dev)
    p = af.Plan("r2c", shape, xd, h, fp, af.ACCFFT_ESTIMATE)
    p.execute_r2c(xd, h)
    torch.cuda.synchronize()
    assert rel_l2(h.cpu().numpy(), np.fft.rfftn(c.real)) < tol
    back = torch.empty_like(xd)
    p.execute_c2r(h, back)
    torch.cuda.synchronize()
    assert rel_l2(back.cpu().numpy() / np.prod(shape), c.real) < tol
    p.destroy()
