"""The arrays that a module's call takes (native.Module.__call__): outputs with room for every state only."""
import sys

import numpy as np
import pytest

from combustion_amd import native, synth
from helpers import setup


class DeviceArray:
    """What the call asks of a CUDA tensor, without a GPU."""

    is_cuda, dtype = True, "torch.float64"

    def __init__(self, *shape):
        self.shape = shape

    def __len__(self):
        return self.shape[0]

    def is_contiguous(self):
        return True

    def numel(self):
        return int(np.prod(self.shape))

    def data_ptr(self):
        return 4096


@pytest.fixture
def module(monkeypatch):
    """A module of two inputs and two outputs whose native call only records the number of states."""
    mod = native.Module.__new__(native.Module)
    mod._h, mod.program, mod.calls = None, native._Signature(2, 2), []

    class Library:
        @staticmethod
        def cb_hip_call(handle, ins, n_in, n, outs, n_out, on_device, stream, ms):
            mod.calls.append(n)
            return 0

    monkeypatch.setattr(native, "lib", lambda: Library)
    monkeypatch.setattr(native, "_addresses", lambda *a: -1)  # every array is examined by itself
    return mod


@pytest.mark.parametrize("array", [lambda *shape: np.empty(shape), DeviceArray], ids=["host", "device"])
def test_outputs_have_room_for_every_state(array, module):
    ins = [array(8), array(8)]
    for shapes in ([(8,), (7,)], [(0,), (8,)], [(2, 3), (8,)]):
        with pytest.raises(ValueError, match="room for all 8 states"):
            module(ins, [array(*s) for s in shapes])
    assert module.calls == []
    for shapes in ([(8,), (8,)], [(9,), (100,)], [(1, 8), (2, 4)]):  # longer arrays and other shapes, as ever
        module(ins, [array(*s) for s in shapes])
    assert module.calls == [8, 8, 8]
    module([array(0), array(0)], [array(0), array(0)])
    assert module.calls[-1] == 0


def test_tensors_without_the_native_helper(module, monkeypatch):
    """A library built where torch was absent has no helper; it serves tensors one by one."""
    monkeypatch.setattr(native, "_addresses", None)
    monkeypatch.setitem(sys.modules, "combustion_amd._tensors", None)
    for n in (5, 6):
        module([DeviceArray(n), DeviceArray(n)], [DeviceArray(n), DeviceArray(n)])
    assert module.calls == [5, 6]


@pytest.mark.gpu
def test_short_device_outputs_are_refused(gpu):
    import torch
    M, mech, o = setup("h2o2-10")
    mod = M.chemistry(3).assemble(form="fp64")
    T, P, Y = synth.config_states("h2o2-10", 64, 8)
    ins = [torch.from_numpy(np.ascontiguousarray(r)).to(gpu) for r in (T, P, *Y)]
    outs = [torch.empty(64, dtype=torch.float64, device=gpu) for _ in range(M.active + 2 + M.K)]
    with pytest.raises(ValueError, match="room for all 64 states"):
        mod(ins, outs[:-1] + [outs[-1][:63]])
    with pytest.raises(ValueError, match="room for all 64 states"):
        mod([x.cpu().numpy() for x in ins], [np.empty(63)] + [np.empty(64)] * (len(outs) - 1))
    assert torch.equal(torch.stack(mod(ins, outs)), torch.stack(mod(ins)))
