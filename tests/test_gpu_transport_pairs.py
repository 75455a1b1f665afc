"""The FP64 transport kernel of sixteen waves per 64 states (kernels/transport_pairs.hip) at the edges of its range:
65 species (five slots a wave, most of the last ones empty), 97, and the 160 that its LDS just holds, fits of 3 and 4
coefficients, batches around one group of 64 states; 161 species stay with transport_tiled. Against the FP64 oracle at
the FP64 forms' 1e-12."""
import numpy as np
import pytest

from combustion_amd import synth
from helpers import relative_error, setup, setup_text


@pytest.mark.gpu
@pytest.mark.parametrize("species,D", [(65, 4), (97, 3), (160, 4), (161, 4)])
def test_transport_of_sixteen_waves(species, D, gpu):
    import torch
    if species == 160:
        M, mech, o = setup("large-160", D)
    else:
        M, mech, o = setup_text(synth.generate(species, 3 * species, 3, 2, species, f"sized-{species}").yaml(), D)
    prog = M.chemistry(2, D=D)
    assert ("#define WAVES 16" in prog.hip_source("fp64")) == (species <= 160)
    mod = prog.assemble(form="fp64")
    T, P, Y = synth.states(M.K, 129, 5, (300.0, 3000.0), (0.1, 50.0), 0.3)
    ref, floor = o.batch(T, P, Y, rates=False, threads=8)
    for n in (1, 64, 65, 129):
        got = np.stack([x.cpu().numpy() for x in mod([torch.from_numpy(np.ascontiguousarray(x[:n])).to(gpu) for x in (T, P, *Y)])])
        err = relative_error(got, ref[:, :n], np.abs(floor[:, :n])).max()
        print(species, D, n, err, flush=True)
        assert err < 1e-12, (species, D, n)
