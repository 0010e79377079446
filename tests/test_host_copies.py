"""Which host-to-device copies the calls wait for, on the CPU: Tensor.to and
pin_memory are recorded in place of a GPU's."""
import contextlib

import pytest
import torch

from home_seek_amd import fused_moe, ops

CUDA = torch.device("cuda", 0)


@pytest.fixture
def current(monkeypatch):
    """The current device, as torch.cuda.device sets it."""
    now = [0]

    @contextlib.contextmanager
    def device(d):
        before, now[0] = now[0], torch.device(d).index
        yield
        now[0] = before

    monkeypatch.setattr(torch.cuda, "device", device)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: now[0])
    return now


@pytest.fixture
def copies(monkeypatch, current):
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


def test_capture_is_asked_of_the_device_that_gets_the_table(copies, current, monkeypatch):
    """The stream that copies is the table's device's, whichever device is current."""
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: current[0] == 1)
    assert ops.expert_table([entry()], torch.device("cuda", 0)).shape == (1, 6)
    with pytest.raises(RuntimeError, match="capture"):
        ops.expert_table([entry()], torch.device("cuda", 1))
    current[0] = 1  # a capture on the current device is no matter of the other one's
    assert ops.expert_table([entry()], torch.device("cuda", 0)).shape == (1, 6)
    assert len(copies) == 2


def host_calls():
    """The calls that take weights from the host, each on hidden states of another device."""
    x = torch.zeros(1, 4, dtype=torch.bfloat16, device="meta")
    fp4 = tuple(torch.zeros(4, 4, dtype=torch.int8) if q % 2 == 0 else torch.zeros(4, 4) for q in range(6))
    bf16 = tuple(torch.zeros(4, 4, dtype=torch.bfloat16) for _ in range(3))
    moe, idx, w = fused_moe.FusedMoEFFN(4, 4, 4), torch.zeros(1, 1, dtype=torch.int64), torch.ones(1, 1)
    return {
        "forward fp4": lambda to: moe.forward(x, idx, w, lambda layer, e: to(fp4), 0),
        "forward bf16": lambda to: moe.forward(x, idx, w, lambda layer, e: to(bf16), 0),
        "shared": lambda to: fused_moe.SharedExpertFFN(4, 4).forward(x[None], *to(bf16)),
        "pt": lambda to: fused_moe.fused_expert_ffn_pt(x, *to(bf16)),
        "triton bf16": lambda to: fused_moe.fused_expert_ffn_triton(x, *to(bf16)),
        "triton fp4": lambda to: (lambda e: fused_moe.fused_expert_ffn_triton(
            x, e[0], e[2], e[4], w1_scale=e[1], w3_scale=e[3], w2_scale=e[5]))(to(fp4)),
    }


@pytest.mark.parametrize("call", list(host_calls()))
def test_host_weights_are_read_when_the_call_returns(call, monkeypatch):
    """A caller may refill a pinned buffer after the call that took it; entries on the device are not waited for."""
    waits = []
    monkeypatch.setattr(ops, "expert_table", lambda entries, device, wait=True: waits.append(wait))
    monkeypatch.setattr(fused_moe, "_run_decode_chunks", lambda x, *args, **kw: torch.empty_like(x))
    run = host_calls()[call]
    run(lambda entry: entry)
    run(lambda entry: tuple(t.to("meta") for t in entry))
    run(lambda entry: (entry[0].to("meta"), *entry[1:]))
    assert waits == [True, False, True]
