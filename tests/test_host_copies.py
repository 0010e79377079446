"""Which host-to-device copies the calls wait for, on the CPU: Tensor.to and
pin_memory are recorded in place of a GPU's."""
import pytest
import torch

from home_seek_amd import ops

CUDA = torch.device("cuda", 0)


@pytest.fixture
def copies(monkeypatch):
    """[(numel, waits)] of the copies to CUDA, in order; the tensors stay where they are."""
    log = []
    real = torch.Tensor.to

    def to(self, *args, **kw):
        if args and isinstance(args[0], (torch.device, str)) and torch.device(args[0]).type == "cuda":
            log.append((self.numel(), not kw.get("non_blocking", False)))
            return self
        return real(self, *args, **kw)

    monkeypatch.setattr(torch.Tensor, "to", to)
    monkeypatch.setattr(torch.Tensor, "pin_memory", lambda self: self)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    return log


def entry():
    return tuple(torch.zeros(4, 4, dtype=torch.int8) for _ in range(6))


def test_expert_table_is_on_the_device_when_it_returns(copies):
    """A program keeps a table and reads it on other streams than the one that was current when it was made."""
    ent = entry()
    table = ops.expert_table([None, ent], CUDA)
    assert table.tolist() == [[0] * 6, [t.data_ptr() for t in ent]]
    assert copies == [(12, True)]
