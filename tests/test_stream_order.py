"""CPU check of the order between torch's current stream and the entry points
that take no stream and start on the NULL stream: the wait is recorded before
the library is called."""
import pytest


class _Stream:
    def __init__(self, handle, log):
        self.cuda_stream, self.log = handle, log

    def wait_stream(self, other):
        self.log.append((self.cuda_stream, "waits for", other.cuda_stream))


@pytest.mark.parametrize("handle,before", [(7, [(0, "waits for", 7)]), (0, [])])
def test_factor_starts_after_the_current_stream(monkeypatch, handle, before):
    import torch
    import hplai
    log = []
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: _Stream(handle, log))
    monkeypatch.setattr(torch.cuda, "default_stream", lambda *a: _Stream(0, log))

    class Lib:
        def hplai_factor_f32(self, *args):
            log.append("factor")
            return hplai.OK

    monkeypatch.setattr(hplai, "lib", lambda: Lib())
    c = hplai.Context.__new__(hplai.Context)
    c.handle, c.device = None, 0
    c.factor(128, 64, 4096, 128)
    assert log == before + ["factor"]
