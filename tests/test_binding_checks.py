"""Checks the Python binding makes before a call reaches the C ABI, on the
CPU."""
import os

import pytest


def test_forked_child_asks_torch_for_its_stream(monkeypatch):
    """torch refuses the GPU in a child forked from a process that has used
    it, so the stream accessor the parent has cached is not used there."""
    import torch
    import accfft_amd as af

    def refuse():
        raise RuntimeError("Cannot re-initialize CUDA in forked subprocess")
    monkeypatch.setattr(torch.cuda, "current_stream", refuse)
    monkeypatch.setattr(af, "_raw_stream", lambda: 0)
    assert af._stream() == 0
    pid = os.fork()
    if pid == 0:
        code = 1
        try:
            af._stream()
        except RuntimeError:
            code = 0
        finally:
            os._exit(code)
    assert os.waitstatus_to_exitcode(os.waitpid(pid, 0)[1]) == 0
    assert af._stream() == 0  # the parent keeps its accessor


@pytest.mark.parametrize("xyz,given", [(1, True), (2, True), (3, True), (3, False)])
def test_masked_r2c_needs_room_for_the_half_spectrum(monkeypatch, xyz, given):
    """Without the z transform execute_r2c works in place on its input as
    rows of n[2]//2+1 complex, two reals a row more than the field of an
    out-of-place plan has."""
    import torch
    import accfft_amd as af

    class OnGpu(torch.Tensor):
        is_cuda = True
    n = (4, 3, 6)
    p = af.Plan.__new__(af.Plan)
    p._h, p.precision, p.device, p.inplace = None, af.F32, None, False
    p._in_bytes, p._out_bytes = 4 * 3 * 6 * 4, 4 * 3 * 4 * 8
    calls = []

    class Lib:
        @staticmethod
        def accfft_amd_execute_r2c(*a):
            calls.append(a)
            return af.OK
    monkeypatch.setattr(af, "lib", lambda: Lib)
    monkeypatch.setattr(af.Plan, "_bind", lambda self: None)
    field = torch.zeros(n).as_subclass(OnGpu)
    half = torch.zeros(4, 3, 4, dtype=torch.complex64).as_subclass(OnGpu)
    p._keep = (field, half)
    p.execute_r2c(field, half)  # with the z transform the field is enough
    with pytest.raises(af.AccfftError, match="bytes"):
        p.execute_r2c(field if given else None, None, xyz=xyz)
    p.execute_r2c(half, None, xyz=xyz)
    assert len(calls) == 2
