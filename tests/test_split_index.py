"""The split-BF16 packing's index tables are shared by all calls of a shape, on
whatever stream: they must be complete when the first call returns, so they
come from the host in one blocking copy and no queued kernel writes them."""
import numpy as np
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from nsvf_amd import train

SHAPES = [(128, 32), (128, 128), (128, 128), (4, 128)]


class Ops(TorchDispatchMode):
    """The names of the torch operations called, those that write a result."""

    def __init__(self):
        super().__init__()
        self.names = set()

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.add(func._schema.name.split("::")[1])
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("backward", [False, True])
def test_no_queued_operation_makes_the_table(monkeypatch, backward):
    class Lib:
        def nsvf_mlp_split_pack(self, *args):
            self.args = args
            return 0

    fake = Lib()
    monkeypatch.setattr(train, "lib", lambda: fake)
    monkeypatch.setattr(train, "_layer_pointers", lambda w, b: (None, None, None))
    monkeypatch.setattr(train, "_stream", lambda dev: None)
    ws = [torch.zeros(s) for s in SHAPES]
    bs = [torch.zeros(s[0]) for s in SHAPES]
    with Ops() as ops:
        train._pack_split(ws, bs, 5, backward)
    assert ops.names <= {"empty", "slice", "detach", "_to_copy", "lift_fresh"}, ops.names
    f = train._x3_index(SHAPES, torch.device("cpu")).numpy()
    b = train._x3_train_index(SHAPES, torch.device("cpu")).numpy()
    nf, nb = fake.args[6:8]
    assert (nf, nb) == (f.size, b.size if backward else 0)
    idx = np.ctypeslib.as_array(
        (np.ctypeslib.ctypes.c_int64 * (nf + nb)).from_address(fake.args[5].value))
    assert np.array_equal(idx[:nf], f) and (not backward or np.array_equal(idx[nf:], b))


@pytest.mark.gpu
@pytest.mark.parametrize("widths", [[32] + [64] * 9 + [4], [32, 64, 48, 4], [32, 64, 64, 3],
                                    [32, 64, 64, 9], [20, 4], [48, 256, 256, 256, 256, 4]])
def test_any_layers_are_packed(device, widths):
    """Layers that the packing kernel does not take (many, of several widths,
    another head) have the same fragments as on the CPU, as those that it does."""
    g = torch.Generator().manual_seed(6)
    ws = [torch.randn(o, i, generator=g) for i, o in zip(widths, widths[1:])]
    bs = [torch.randn(o, generator=g) for o in widths[1:]]
    want, want_bias = train.pack_mlp_x3(ws, bs)
    frags, bias = train.pack_mlp_x3([w.to(device) for w in ws], [b.to(device) for b in bs])
    assert torch.equal(frags.cpu(), want) and torch.equal(bias.cpu(), want_bias)


def test_the_kernel_takes_equal_layers_only():
    make = lambda *widths: ([torch.zeros(o, i) for i, o in zip(widths, widths[1:])],
                            [torch.zeros(o) for o in widths[1:]])
    assert train._split_packable(*make(32, 128, 128, 128, 4))
    assert train._split_packable(*make(20, 64, 4))
    for widths in ([32] + [64] * 8 + [4], [32, 64, 48, 4], [32, 64, 64, 3], [20, 4]):
        assert not train._split_packable(*make(*widths))
    ws, bs = make(32, 64, 64, 4)
    assert not train._split_packable(ws, bs[:1] + [torch.zeros(63)] + bs[2:])


@pytest.mark.gpu
def test_first_calls_on_two_streams(device):
    """The first call of a shape on a busy stream, the second on another one."""
    g = torch.Generator().manual_seed(4)
    shapes = [(64, 32), (64, 64), (4, 64)]   # a shape that no other test packs
    ws = [torch.randn(s, generator=g) for s in shapes]
    bs = [torch.randn(s[0], generator=g) for s in shapes]
    want, want_bias = train.pack_mlp_x3(ws, bs)
    dw, db = [w.to(device) for w in ws], [b.to(device) for b in bs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(device) for _ in range(2)]
    with torch.cuda.stream(streams[0]):
        torch.cuda._sleep(50_000_000)        # some 20 ms
        first = train.pack_mlp_x3(dw, db)
    with torch.cuda.stream(streams[1]):
        second = train.pack_mlp_x3(dw, db)
    torch.cuda.synchronize()
    for frags, bias in (first, second):
        assert torch.equal(frags.cpu(), want) and torch.equal(bias.cpu(), want_bias)
