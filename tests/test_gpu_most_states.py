"""The largest batch a call takes, 2^31 - 1 states, through the one launch of both sections (more than one launch there)."""
import os

import pytest

from combustion_amd import Mechanism

HANDWRITTEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "handwritten.yaml")


@pytest.mark.gpu
def test_last_states_of_the_largest_batch(gpu):
    import torch
    n, tail = (1 << 31) - 1, 200
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 8 * 8 * n:
        pytest.skip("needs 140 GB of GPU memory")
    M = Mechanism(HANDWRITTEN)
    mod = M.chemistry(3).assemble(form="fp64")
    T, P = (torch.full((n,), v, dtype=torch.float64, device=gpu) for v in (1200.0, 101325.0))
    Y = torch.full((n,), 1.0 / M.K, dtype=torch.float64, device=gpu)
    bounds = [0, (1 << 30) - 100, n - tail]  # the batch's start, the launches' edge and its end
    for b, t in zip(bounds, (600.0, 900.0, 2000.0)):
        T[b:b + tail] = torch.linspace(t, t + 300, tail, dtype=torch.float64, device=gpu)
    ω, λ, rates, transport = (torch.zeros(n, dtype=torch.float64, device=gpu) for _ in range(4))  # the last two: any values
    outs = [ω] + [rates] * (M.active - 1) + [λ] + [transport] * (1 + M.K)
    mod([T, P] + [Y] * M.K, outs)
    for b in bounds:
        part = [x[b:b + tail].clone() for x in (T, P, Y)]
        want = mod(part[:2] + [part[2]] * M.K)
        assert torch.equal(ω[b:b + tail], want[0]) and torch.equal(λ[b:b + tail], want[M.active])
    assert not torch.equal(ω[:tail], ω[-tail:])
    del T, P, Y, ω, λ, rates, transport, outs
    torch.cuda.empty_cache()
