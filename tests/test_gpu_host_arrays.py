"""Calls on host arrays (csrc/host_arrays.hpp): states go through the staging in slices, and every state's outputs are
the ones of a call on device arrays, to the bit, whatever the slices; in place and at overlapping offsets too."""
import numpy as np
import pytest

from combustion_amd import synth
from helpers import setup


@pytest.mark.gpu
def test_slices_match_device_call(gpu):
    import torch
    M, mech, o = setup("gri-53")
    mod = M.chemistry(3).assemble(form="fp64")
    K, rows = M.K, M.active + 2 + M.K
    slot = (16 << 20) // ((K + 2 + rows) * 8) // 64 * 64  # states of one slice
    T, P, Y = synth.config_states("gri-53", 2 * slot + 65, 8)
    x = np.vstack([T, P, Y])
    want = torch.stack(mod([r.contiguous() for r in torch.from_numpy(x).to(gpu)])).cpu().numpy()
    for n in (2 * slot + 65, slot + 1, slot, 65, 1):  # shrinking batches reuse the staging
        got = np.stack(mod([np.ascontiguousarray(r[:n]) for r in x]))
        assert np.array_equal(got, want[:, :n]), n
    n = slot + 70
    ins = [r[:n].copy() for r in x]
    outs = [ins[i] if i < len(ins) else np.empty(n) for i in range(rows)]  # in place
    mod(ins, outs)
    assert np.array_equal(np.stack(outs), want[:, :n])
    buf = np.empty(n + 100)
    ins = [r[:n].copy() for r in x]
    ins[0] = buf[100:]
    ins[0][:] = x[0, :n]
    outs = [buf[:n]] + [np.empty(n) for _ in range(rows - 1)]  # the first output ends inside the temperatures
    mod(ins, outs)
    assert np.array_equal(np.stack(outs), want[:, :n])
    a = np.empty(0)
    assert all(len(r) == 0 for r in mod([a] * (K + 2)))


@pytest.mark.gpu
def test_tensors_that_are_refused_or_converted_one_by_one(gpu):
    """The native pass over tensors leaves everything but contiguous float64 CUDA tensors of one length to the checks
    on each array."""
    import torch
    M, mech, o = setup("h2o2-10")
    mod = M.chemistry(3).assemble(form="fp64")
    T, P, Y = synth.config_states("h2o2-10", 64, 8)
    ins = [torch.from_numpy(np.ascontiguousarray(r)).to(gpu) for r in (T, P, *Y)]
    want = torch.stack(mod(tuple(ins)))
    with pytest.raises(ValueError, match="contiguous float64"):
        mod([ins[0].float()] + ins[1:])
    with pytest.raises(ValueError, match="contiguous float64"):
        mod([torch.stack([ins[0], ins[0]], 1)[:, 0]] + ins[1:])
    with pytest.raises(ValueError, match="same length"):
        mod([ins[0], ins[1][:32]] + ins[2:])
    with pytest.raises(TypeError):
        mod([ins[0], ins[1].cpu()] + ins[2:])
    with pytest.raises(ValueError, match="outputs must match"):
        mod(ins, [torch.empty_like(ins[0])])
    longer = [torch.empty(100, dtype=torch.float64, device=gpu) for _ in range(M.active + 2 + M.K)]
    got = torch.stack(mod(ins, longer))[:, :64]
    assert torch.equal(got, want)
    assert torch.equal(torch.stack(mod(torch.stack(ins))), want)  # rows of one tensor
