"""A call on host arrays after an asynchronous copy into its pinned inputs, on the stream given to the call and on the
default stream."""
import numpy as np
import pytest

from combustion_amd import synth
from helpers import setup


@pytest.mark.gpu
@pytest.mark.parametrize("side", [True, False], ids=["caller's", "default"])
def test_host_call_after_a_queued_copy(side, gpu):
    import torch
    M, mech, o = setup("h2o2-10")
    mod = M.chemistry(3).assemble(form="fp64")
    n = 1 << 16
    device = torch.from_numpy(np.stack([np.ascontiguousarray(r) for a in [synth.config_states("h2o2-10", n, 8)] for r in (a[0], a[1], *a[2])])).to(gpu)
    want = torch.stack(mod(list(device))).cpu().numpy()
    filler = torch.randn(1 << 27, dtype=torch.float32, device=gpu)
    pinned = torch.full(device.shape, float("nan"), dtype=torch.float64, pin_memory=True)
    stream = torch.cuda.Stream() if side else torch.cuda.default_stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        for _ in range(20):
            filler.mul_(1.0001)  # some milliseconds of work ahead of the copy
        pinned.copy_(device, non_blocking=True)
        got = np.stack(mod(list(pinned.numpy()), stream=stream.cuda_stream or None))
    assert np.array_equal(got, want)
