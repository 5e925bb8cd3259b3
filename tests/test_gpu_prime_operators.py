"""Operators on axes with a prime factor above 13 (one, or two: a second
prime stage has twiddles): the prime stage of the run-time engine inside the
fused derivative and multiply passes, along every axis, against the oracle
in double precision.

Tolerances: a stage of prime radix p adds a relative rounding error of about
sqrt(p) eps on random data, twice in a fused pass; the symbols raise the
noise by less than a factor 2 relative to the result (as in
test_gpu_mixed_radix).  1e-12 and 1e-5 leave a factor above 10."""
import pytest

from conftest import rel_l2, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("shape", [(19, 34, 12), (12, 19, 34), (34, 12, 19), (6, 323, 10),
                                   (323, 5, 9), (4, 6, 323), (127, 3, 8), (8, 22, 26)])
def test_operators(dev, orc, shape, prec):
    import torch
    import accfft_amd as af
    fp, rdt, tol = ((af.F64, torch.float64, 1e-12) if prec == "f64"
                    else (af.F32, torch.float32, 1e-5))
    v = [rng(sum(shape) + d).standard_normal(shape) for d in range(3)]
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
