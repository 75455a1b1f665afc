"""The FP64 transport kernel of four waves per 64 states (kernels/transport_split.hip) at the edges of its range: the
smallest and largest mechanisms that take it and the benchmark's, fits of 2 to 8 coefficients, and batches around one
group of 64 states, against the FP64 oracle at the FP64 forms' 1e-12."""
import numpy as np
import pytest

from combustion_amd import synth
from helpers import relative_error, setup, setup_text


@pytest.mark.gpu
@pytest.mark.parametrize("species,D", [(53, 4), (53, 2), (32, 5), (35, 8), (64, 4)])
def test_transport_of_four_waves(species, D, gpu):
    import torch
    if species == 53:
        M, mech, o = setup("gri-53", D)
    else:
        M, mech, o = setup_text(synth.generate(species, 4 * species, 3, 2, species, f"sized-{species}").yaml(), D)
    prog = M.chemistry(2, D=D)
    assert "lds_x" in prog.hip_source("fp64")
    mod = prog.assemble(form="fp64")
    T, P, Y = synth.states(M.K, 333, 5, (300.0, 3000.0), (0.1, 50.0), 0.3)
    ref, floor = o.batch(T, P, Y, rates=False, threads=8)
    for n in (1, 63, 64, 65, 333):
        got = np.stack([x.cpu().numpy() for x in mod([torch.from_numpy(np.ascontiguousarray(x[:n])).to(gpu) for x in (T, P, *Y)])])
        err = relative_error(got, ref[:, :n], np.abs(floor[:, :n])).max()
        print(species, D, n, err, flush=True)
        assert err < 1e-12, (species, D, n)


def test_wilke_factor_reproduces_its_matrix():
    """The low-rank moments against the full sums, on the CPU: the emitted text's rank is below the species count, and
    the pivoted Cholesky factor of 1/sqrt(W_k + W_j), restated here, is within rounding of every entry at that rank."""
    M, mech, o = setup("gri-53")
    text = M.chemistry(2).hip_source("fp64")
    rank = int(text.split("#define R ")[1].split()[0])
    assert rank < M.K // 2
    W = np.longdouble(M.molar_mass)
    A = 1 / np.sqrt(W[:, None] + W[None, :])
    rest, G = np.diag(A).copy(), []
    for _ in range(rank):
        p = int(np.argmax(rest / np.diag(A)))
        c = (A[:, p] - sum((g * g[p] for g in G), np.zeros(M.K, np.longdouble))) / np.sqrt(rest[p])
        rest = rest - c * c
        rest[p] = 0
        G.append(c)
    G = np.array(G, np.float64)
    assert np.abs(G.T @ G / np.float64(A) - 1).max() < 8 * 2.0 ** -53  # a few roundings of the factor's products
