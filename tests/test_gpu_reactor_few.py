"""A few reactors of a small mechanism, which fill one of its batch's parts: as in a larger batch, to the bit."""
import numpy as np
import pytest

from combustion_amd import Mechanism, synth
from combustion_amd.native import Integrator


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 8, 9])
def test_few_reactors_as_in_a_larger_batch(n, gpu):
    import torch
    M = Mechanism(synth.mechanism_path("h2o2-10"))
    T, P, Y = synth.states(M.K, 100, 3, (1000.0, 1800.0), (1.0, 5.0), 0.3)
    results = []
    for count in (n, 100):
        y, p = (torch.from_numpy(np.ascontiguousarray(a[..., :count])).to(gpu) for a in (np.vstack([T, Y]), P))
        t, h = torch.zeros(count, dtype=torch.float64, device=gpu), torch.full((count,), 1e-10, dtype=torch.float64, device=gpu)
        status, steps = torch.zeros(count, dtype=torch.int32, device=gpu), torch.zeros(count, dtype=torch.int32, device=gpu)
        Integrator(M, rtol=1e-8, atol_T=1e-6, atol_Y=1e-12).advance(y, p, t, h, status, steps, 1e-5, max_steps=64)
        results.append([x.cpu().numpy()[..., :n] for x in (y, t, h, status, steps)])
    assert results[0][4].max() > 0
    for a, b in zip(*results):
        np.testing.assert_array_equal(a, b)
