"""The compile-time mixed-radix kernels (accfft_amd/csrc/fft_mix.hpp): every
length of their list along every axis, transforms in both directions
against numpy's FFT in double precision, with tiles that are partly empty
(few lines) and, along x and y, more columns than one tile; and the fused
derivative and symbol passes of two-, three- and four-stage lengths, with
and without accumulation, against the oracle's operators.

Tolerances: log2(n) stages of rounding, below 1e-14 / 1e-6 relative for
these lengths; the tests hold 1e-12 and 1e-5 (operators: times the symbol's
range, as in test_gpu_ops)."""
import os
import re

import numpy as np
import pytest

from conftest import rel_l2, rng

HPP = os.path.join(os.path.dirname(__file__), "..", "accfft_amd", "csrc", "fft_mix_list.hpp")
LENGTHS = sorted(int(v) for v in re.findall(r"X\((\d+)\)", open(HPP).read()
                                            .split("#define AFFT_MIX_EACH")[0]))


def test_list_is_the_rule():
    def rest(n, primes):
        for p in primes:
            while n % p == 0:
                n //= p
        return n
    want = [n for n in range(16, 1025) if (n & (n - 1) or n <= 512) and
            (rest(n, (2, 3, 5)) == 1 or (n <= 512 and rest(n, (2, 3, 5, 7)) == 1))]
    assert LENGTHS == want


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", LENGTHS)
def test_transforms(dev, n, prec):
    import torch
    import accfft_amd as af
    fp, rdt, cdt, tol = ((af.F64, torch.float64, torch.complex128, 1e-12) if prec == "f64"
                         else (af.F32, torch.float32, torch.complex64, 1e-5))
    for shape in ((n, 3, 7), (2, n, 17), (3, 5, n)):
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
        h = torch.empty(shape[:2] + (shape[2] // 2 + 1,), dtype=cdt, device=dev)
        p = af.Plan("r2c", shape, xd, h, fp, af.ACCFFT_ESTIMATE)
        p.execute_r2c(xd, h)
        torch.cuda.synchronize()
        assert rel_l2(h.cpu().numpy(), np.fft.rfftn(c.real)) < tol
        # a spectrum with imaginary parts at DC and Nyquist, which c2r drops
        s = rng(n + 2).standard_normal(h.shape) + 1j * rng(n + 3).standard_normal(h.shape)
        back = torch.empty_like(xd)
        p.execute_c2r(torch.tensor(s, dtype=cdt, device=dev), back)
        torch.cuda.synchronize()
        t = np.fft.ifft(np.fft.ifft(s, axis=0), axis=1)
        assert rel_l2(back.cpu().numpy() / np.prod(shape), np.fft.irfft(t, n=shape[2], axis=2)) < tol
        p.destroy()


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", [16, 18, 45, 64, 70, 160, 162, 200, 256, 384, 405, 512, 625, 768])
def test_operators(dev, orc, n, prec):
    import torch
    import accfft_amd as af
    # the derivative raises mode k by k, the Laplacian by k^2, of rounding
    # noise that is flat over the modes: relative to the result's norm the
    # amplification is below 2
    fp, rdt, tol = ((af.F64, torch.float64, 1e-12) if prec == "f64"
                    else (af.F32, torch.float32, 1e-5))
    for shape in ((n, 6, 10), (5, n, 12), (4, 6, n), (3, 5, n), (n, 5, 9)):
        v = [rng(n + d).standard_normal(shape) for d in range(3)]
        d = [torch.tensor(a, dtype=rdt, device=dev) for a in v]
        out = [torch.empty_like(d[0]) for _ in range(3)]
        p = af.Plan("r2c", shape, d[0], out[0], fp, af.ACCFFT_ESTIMATE)
        p.grad(d[0], *out)
        torch.cuda.synchronize()
        for a, b in zip(out, orc.grad(v[0])):
            assert rel_l2(a.cpu().numpy(), b) < tol
        p.divergence(*d, out[0])
        torch.cuda.synchronize()
        assert rel_l2(out[0].cpu().numpy(), orc.divergence(*v)) < tol
        for name in ("laplace", "biharmonic", "inv_laplace", "inv_biharmonic"):
            getattr(p, name)(d[0], out[0])
            torch.cuda.synchronize()
            assert rel_l2(out[0].cpu().numpy(), getattr(orc, name)(v[0])) < tol, name
        p.destroy()
