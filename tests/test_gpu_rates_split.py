"""The rates kernel of teams of waves (kernels/rates_split.hip) at the edges of its launch shapes: both team layouts
(two teams of four waves up to 53 species, one team of eight above) on batches around one and two groups of 64 states,
against the FP64 oracle. Tolerances as in test_gpu_ragged.py: 1e-12 of the term scale in FP64, 1e-5 with FP32 cores."""
import numpy as np
import pytest

from combustion_amd import synth
from helpers import relative_error, setup, setup_text, state_floor


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["fp64", "fast"])
@pytest.mark.parametrize("species", [53, 60])
def test_team_layouts_and_ragged_groups(species, form, gpu):
    import torch
    if species == 53:
        M, mech, o = setup("gri-53")
    else:
        M, mech, o = setup_text(synth.generate(60, 260, 14, 11, 60, "sized-60").yaml())
    prog = M.chemistry(1)
    text = prog.hip_source(form)
    assert ("#define TEAMS 2" if species == 53 else "#define TEAMS 1") in text
    mod = prog.assemble(form=form)
    T, P, Y = synth.states(M.K, 1025, 5, (500.0, 3000.0), (0.1, 50.0), 0.3)
    ref, floor = o.batch(T, P, Y, transport=False, threads=8)
    f, tol = (floor, 1e-12) if form == "fp64" else (state_floor(floor, M.active), 1e-5)
    for n in (1, 64, 65, 127, 128, 129, 1025):
        got = np.stack([x.cpu().numpy() for x in mod([torch.from_numpy(np.ascontiguousarray(x[:n])).to(gpu) for x in (T, P, *Y)])])
        err = relative_error(got, ref[:, :n], f[:, :n]).max()
        print(species, form, n, err, flush=True)
        assert err < tol, (species, form, n)
