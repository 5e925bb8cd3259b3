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
