"""Host side of the staged transfers, with stand-ins for the GPU: on which device's streams the
copies, events and buffers of a read-back lie."""
import types

import torch

from liteform_ae_amd import format_algos as fa


class _Cuda:
    """torch.cuda for two devices of which 0 is the current one."""

    def __init__(self):
        self.current, self.recorded = 0, []
        outer = self

        class Event:
            def __init__(self):
                self.device = outer.current             # an event belongs to the device it is made on

            def record(self):
                outer.recorded.append((self.device, outer.current))

            def synchronize(self):
                pass
        self.Event = Event

    def current_device(self):
        return self.current

    def set_device(self, device):
        self.current = device


class _OnDevice1:
    """A tensor that says it is on cuda:1."""
    device = torch.device("cuda", 1)

    def __init__(self, values):
        self.values, self.dtype = values, values.dtype

    def numel(self):
        return self.values.numel()

    def __getitem__(self, at):
        return self.values[at]


def test_read_back_uses_the_streams_of_the_tensors_device(monkeypatch):
    """The events that a read-back waits for are recorded behind its copies: on the tensors' device,
    also where another one is current."""
    cuda = _Cuda()
    empty = lambda *size, dtype, pin_memory=False: torch.empty(*size, dtype=dtype)        # noqa: E731
    monkeypatch.setattr(fa, "_torch", lambda: types.SimpleNamespace(empty=empty, uint8=torch.uint8, cuda=cuda))
    monkeypatch.setattr(fa, "_stages", {})
    rows = torch.arange(2_000_003, dtype=torch.int32)                                      # several pieces
    vals = torch.linspace(-1.0, 1.0, 1_000, dtype=torch.float32)
    with fa._Downloads([(_OnDevice1(rows), torch.int64), (_OnDevice1(vals), torch.float32)]) as down:
        assert torch.equal(down.get(0), rows.to(torch.int64)) and torch.equal(down.get(1), vals)
    assert len(cuda.recorded) == 5 and set(cuda.recorded) == {(1, 1)}
    assert [device for _, device in fa._stages] == [1]
    assert cuda.current == 0 and not fa._stage_lock.locked()
