"""Rates and transport of a small FP64 batch in one kernel, on either side of the largest size that takes it (8192
states), and around a block's 64: a state's outputs are the same to the bit whatever its batch, alone or by two kernels,
and a captured call replays them; for the 53-species mechanism and generated ones at the ends of the range (the fewest
species whose transport has four waves, and 53 with fits of 3)."""
import numpy as np
import pytest

from combustion_amd import synth
from helpers import relative_error, setup, setup_text


@pytest.mark.gpu
@pytest.mark.parametrize("species,D", [(53, 4), (32, 4), (53, 3)])
def test_small_batches_equal_larger_ones(species, D, gpu):
    import torch
    if D == 4 and species == 53:
        M, mech, o = setup("gri-53")
    else:
        M, mech, o = setup_text(synth.generate(species, 5 * species, 6, 4, species, f"small-{species}").yaml(), D)
    mod = M.chemistry(D=D).assemble(form="fp64")
    T, P, Y = synth.states(M.K, 8193, 5, (300.0, 3000.0), (0.1, 50.0), 0.3)
    ins = [torch.from_numpy(np.ascontiguousarray(x)).to(gpu) for x in (T, P, *Y)]
    whole = torch.stack(mod(ins))  # two kernels
    ref, floor = o.batch(T[:200], P[:200], Y[:, :200], threads=8)
    err = relative_error(whole[:, :200].cpu().numpy(), ref, np.abs(floor)).max()
    print(species, D, err, flush=True)
    assert err < 1e-12
    s = torch.cuda.Stream()
    for n in (1, 63, 64, 65, 3001, 8192):
        part = [x[:n].contiguous() for x in ins]
        outs = [torch.full((n,), float("nan"), dtype=torch.float64, device=gpu) for _ in range(len(whole))]
        torch.cuda.synchronize()
        mod(part, outs, stream=s.cuda_stream)
        torch.cuda.synchronize()
        assert torch.equal(torch.stack(outs), whole[:, :n]), (species, n)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            mod(part, outs, stream=s.cuda_stream)
        for _ in range(3):
            for x in outs:
                x.fill_(float("nan"))
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(torch.stack(outs), whole[:, :n]), (species, n)


@pytest.mark.gpu
@pytest.mark.parametrize("species", [10, 24])
def test_one_lane_kernels_in_one_launch(species, gpu):
    """Mechanisms whose two sections run one lane per state, at every size in one launch of blocks of 64 states: 1e-12 of
    the oracle, and nothing written past the batch."""
    import torch
    if species == 10:
        M, mech, o = setup("h2o2-10")
    else:
        M, mech, o = setup_text(synth.generate(24, 120, 6, 4, 24, "small-24").yaml())
    mod = M.chemistry().assemble(form="fp64")
    T, P, Y = synth.states(M.K, 333, 5, (300.0, 3000.0), (0.1, 50.0), 0.3)
    ref, floor = o.batch(T, P, Y, threads=8)
    for n in (1, 63, 64, 65, 256, 257, 333):
        ins = [torch.from_numpy(np.ascontiguousarray(x[:n])).to(gpu) for x in (T, P, *Y)]
        room = torch.full((len(ref), n + 1), float("nan"), dtype=torch.float64, device=gpu)
        mod(ins, [x[:n] for x in room])
        torch.cuda.synchronize()
        assert room[:, n].isnan().all()
        err = relative_error(room[:, :n].cpu().numpy(), ref[:, :n], np.abs(floor[:, :n])).max()
        print(species, n, err, flush=True)
        assert err < 1e-12
