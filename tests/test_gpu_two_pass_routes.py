"""Two-pass plans (accfft_amd/csrc/fft_two.hpp): that the kernels really run
(by the plan's own launch records), with and without a tuning choice, and
the fused multiply of pass 2 at every (x length, M) tile it is built for,
against the oracle in double precision.

Tolerances as in test_gpu_two_pass: at most 27 levels of rounding each way,
1e-12 and 1e-5."""
import numpy as np
import pytest

from conftest import rel_l2, rng

pytestmark = pytest.mark.gpu


def _t(prec):
    import torch
    import accfft_amd as af
    return ((af.F64, torch.float64, torch.complex128, 1e-12) if prec == "f64"
            else (af.F32, torch.float32, torch.complex64, 1e-5))


def _kinds(p, call):
    import torch
    p.set_profiling(True)
    p.profile_reset()
    call()
    torch.cuda.synchronize()
    names = sorted(k for k, v in p.profile().items() if v[1])
    p.set_profiling(False)
    return names


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("shape,m", [((40, 64, 32), 1), ((64, 128, 64), 2), ((32, 512, 128), 8)])
def test_the_kernels_run(dev, shape, m, prec):
    """No choice: pass 1, and pass 2 or (m = 1) the plain x pass.  A choice on
    x leaves m = 1 plans as they are, one on y none of them."""
    import torch
    import accfft_amd as af
    fp, rdt, cdt, tol = _t(prec)
    a = rng(11).standard_normal(shape)
    x = torch.tensor(a, dtype=rdt, device=dev)
    h = torch.empty(shape[:2] + (shape[2] // 2 + 1,), dtype=cdt, device=dev)
    back = torch.empty_like(x)
    c = torch.tensor(a + 1j * a[::-1], dtype=cdt, device=dev)
    co = torch.empty_like(c)
    p = af.Plan("r2c", shape, x, h, fp, af.ACCFFT_ESTIMATE)
    q = af.Plan("c2c", shape, c, co, fp, af.ACCFFT_ESTIMATE)
    r = shape[1] // m
    for axis, choice in ((0, -1), (0, -2), (1, -2), (1, -1)):
        on = choice == -1 or (axis == 0 and m == 1)
        for plan, call, mode in (
                (p, lambda: p.execute_r2c(x, h), "r2c"), (p, lambda: p.execute_c2r(h, back), "c2r"),
                (q, lambda: q.execute_c2c(af.ACCFFT_FORWARD, c, co), "c2c_fwd"),
                (q, lambda: q.execute_c2c(af.ACCFFT_BACKWARD, c, co), "c2c_inv")):
            plan.set_tuning(axis, choice)
            names = _kinds(plan, call)
            assert (f"zyfft_{mode}_n{shape[2]}_zy{r}_{prec}" in names) == on, names
            assert any(f"_n{shape[0]}_xy{m}_" in k for k in names) == (on and m > 1), names
            assert len(names) == 2 or not on, names
            plan.set_tuning(axis, -1)
        torch.cuda.synchronize()
        assert rel_l2(back.cpu().numpy() / np.prod(shape), a) < 2 * tol
    p.destroy()
    q.destroy()


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("y", [128, 256, 512])
@pytest.mark.parametrize("x", [32, 64, 128, 256, 512])
def test_fused_multiply(dev, orc, x, y, prec):
    import torch
    import accfft_amd as af
    fp, rdt, cdt, tol = _t(prec)
    shape = (x, y, 32)
    a = rng(x + y).standard_normal(shape)
    d = torch.tensor(a, dtype=rdt, device=dev)
    out = [torch.empty_like(d) for _ in range(3)]
    p = af.Plan("r2c", shape, d, out[0], fp, af.ACCFFT_ESTIMATE)
    for name in ("laplace", "biharmonic", "inv_laplace"):
        names = _kinds(p, lambda: getattr(p, name)(d, out[0]))
        assert f"sfft_mult_n{x}_xy{y // 64}_{prec}" in names, names
        assert rel_l2(out[0].cpu().numpy(), getattr(orc, name)(a)) < tol, name
    p.grad(d, *out, slow=True)
    torch.cuda.synchronize()
    for g, ref in zip(out, orc.grad(a, slow=True)):
        assert rel_l2(g.cpu().numpy(), ref) < tol
    p.destroy()


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("shape,r2c,c2c", [
    # 512-point lines and tiles from 128 KiB, just below and at the number of
    # planes from which they run in two passes ((FP64, FP32) where they differ)
    ((15, 32, 512), False, False), ((16, 32, 512), True, False), ((32, 32, 512), True, True),
    ((31, 64, 512), False, False), ((32, 64, 512), True, (True, False)), ((64, 64, 512), True, True),
    ((31, 64, 256), (False, True), False), ((64, 64, 256), True, True),
    ((63, 64, 128), True, (False, True)), ((64, 64, 128), True, True)])
def test_planes(dev, shape, r2c, c2c, prec):
    import torch
    import accfft_amd as af
    fp, rdt, cdt, tol = _t(prec)
    on = [v if isinstance(v, bool) else v[prec == "f32"] for v in (r2c, c2c)]
    a = rng(sum(shape)).standard_normal(shape) + 1j * rng(1).standard_normal(shape)
    x = torch.tensor(a.real.copy(), dtype=rdt, device=dev)
    h = torch.empty(shape[:2] + (shape[2] // 2 + 1,), dtype=cdt, device=dev)
    p = af.Plan("r2c", shape, x, h, fp, af.ACCFFT_ESTIMATE)
    names = _kinds(p, lambda: p.execute_r2c(x, h))
    assert any("_zy" in k for k in names) == on[0], names
    assert rel_l2(h.cpu().numpy(), np.fft.rfftn(a.real)) < tol
    p.execute_c2r(h, x)
    torch.cuda.synchronize()
    assert rel_l2(x.cpu().numpy() / np.prod(shape), a.real) < 2 * tol
    p.destroy()
    c = torch.tensor(a, dtype=cdt, device=dev)
    co = torch.empty_like(c)
    q = af.Plan("c2c", shape, c, co, fp, af.ACCFFT_ESTIMATE)
    names = _kinds(q, lambda: q.execute_c2c(af.ACCFFT_FORWARD, c, co))
    assert any("_zy" in k for k in names) == on[1], names
    assert rel_l2(co.cpu().numpy(), np.fft.fftn(a)) < tol
    q.execute_c2c(af.ACCFFT_BACKWARD, co, c)
    torch.cuda.synchronize()
    assert rel_l2(c.cpu().numpy() / np.prod(shape), a) < 2 * tol
    p.destroy()
    q.destroy()


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("shape", [(512, 64, 128), (1024, 32, 64), (2048, 64, 32)])
def test_choices_of_the_x_pass(dev, shape, prec):
    """Where pass 2 is the plain x pass, MEASURE and every choice on x keep
    the two passes and their results."""
    import torch
    import accfft_amd as af
    fp, rdt, cdt, tol = _t(prec)
    a = rng(shape[0]).standard_normal(shape)
    x = torch.tensor(a, dtype=rdt, device=dev)
    h = torch.empty(shape[:2] + (shape[2] // 2 + 1,), dtype=cdt, device=dev)
    back = torch.empty_like(x)
    ref = np.fft.rfftn(a)
    p = af.Plan("r2c", shape, x, h, fp, af.ACCFFT_MEASURE)
    chosen = p.tuning()
    assert chosen[0] in (-1, -2, 0, 1, 2, 3) and chosen[1:] == (-1, -1)
    for choice in (chosen[0], -2, -1, 0, 1, 2, 3):
        try:
            p.set_tuning(0, choice)
        except af.AccfftError:
            continue  # no such variant of this length and precision
        names = _kinds(p, lambda: p.execute_r2c(x, h))
        assert len(names) == 2 and any("_zy" in k for k in names), names
        assert rel_l2(h.cpu().numpy(), ref) < tol, choice
        p.execute_c2r(h, back)
        torch.cuda.synchronize()
        assert rel_l2(back.cpu().numpy() / np.prod(shape), a) < 2 * tol, choice
    p.destroy()
