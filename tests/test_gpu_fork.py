"""Batches on either side of the rule that sends the transport kernel to a module's second stream (48 k states of 53
species): captured in a graph and replayed between eager work, each replay writes the eager call's bits, and a state's
outputs do not depend on the batch it came in."""
import numpy as np
import pytest

from combustion_amd import synth
from helpers import setup


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["fp64", "fast", "mixed"])
def test_replays_on_both_sides_of_the_fork(form, gpu):
    import torch
    M, mech, o = setup("gri-53")
    edge = -(-(1 << 27) // 53 ** 2)
    T, P, Y = synth.config_states("gri-53", edge, 12)
    ins = [torch.from_numpy(np.ascontiguousarray(x)).to(gpu) for x in (T, P, *Y)]
    mod = M.chemistry(3).assemble(form=form)
    s = torch.cuda.Stream()
    first = {}
    for n in (edge - 1, edge):
        part = [x[:n] for x in ins]
        outs = [torch.empty(n, dtype=torch.float64, device=gpu) for _ in range(M.active + M.K + 2)]
        torch.cuda.synchronize()
        mod(part, outs, stream=s.cuda_stream)
        torch.cuda.synchronize()
        eager = torch.stack(outs).clone()
        first[n] = eager[:, :edge - 1]
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            mod(part, outs, stream=s.cuda_stream)
        for replay in range(3):
            for x in outs:
                x.fill_(float("nan"))
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(torch.stack(outs), eager), (form, n, replay)
            _ = (ins[0] * 2).sum().item()
    assert torch.equal(first[edge - 1], first[edge])
