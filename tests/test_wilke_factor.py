"""The factor G of 1/sqrt(W_k + W_j) that the FP64 transport kernel of four waves has in its text (CPU only): the constants
of both products, G^T y with sqrt(W_j / 8) on them and G z over sqrt(W_k), against the matrix and each other."""
import re

import numpy as np
import pytest

from combustion_amd import synth
from helpers import setup, setup_text

NUMBER = r"(-?0x[0-9a-f.]+p[+-]\d+)"


def constants(section, pattern):
    """{(i, label): value} of a wave's lines of the form of `pattern`."""
    return {(int(i), int(k)): float.fromhex(c) for i, c, k in re.findall(pattern, section)}


@pytest.mark.parametrize("species", [53, 32, 64])
def test_emitted_factor_reproduces_the_matrix(species):
    M = setup("gri-53")[0] if species == 53 else setup_text(synth.generate(species, 4 * species, 3, 2, species, f"sized-{species}").yaml())[0]
    text = M.chemistry(2).hip_source("fp64")
    K, rank, W = M.K, int(text.split("#define R ")[1].split()[0]), np.asarray(M.molar_mass)
    assert rank < K // 2
    columns = text[text.index("double z[RW][3];"):text.index("= z[i][0];")]
    rows = text[text.index("double d0[KW]"):text.index("const double den =")]
    by_column, by_row = np.zeros((K, rank)), np.zeros((K, rank))
    for wave in range(4):
        part = [re.split(r"\(wave == \d\) \{", s)[1 + wave] for s in (columns, rows)]
        for (i, j), c in constants(part[0], rf"z\[(\d+)\]\[0\] = (?:__builtin_fma\()?{NUMBER}(?:,| \*) x(\d+)").items():
            by_column[j, 4 * i + wave] = c / np.sqrt(W[j] / 8)
        for (i, q), c in constants(part[1], rf"d0\[(\d+)\] = (?:__builtin_fma\()?{NUMBER}(?:,| \*) z(\d+)_0").items():
            by_row[4 * i + wave, q] = c * np.sqrt(W[4 * i + wave])
    A = 1 / np.sqrt(W[:, None] + W[None, :])
    # the factor's remainder is below 2^-56 of an entry; its constants have three roundings each (themselves, the scaling
    # and its root), and the products of up to `rank` terms, a few of them large, one each
    assert np.abs(by_column / np.where(by_row == 0, 1, by_row) - 1)[by_row != 0].max() < 8 * 2.0 ** -53
    assert ((by_row != 0) == (by_column != 0)).all()
    for G, H in ((by_column, by_row), (by_column, by_column), (by_row, by_row)):
        assert np.abs(G @ H.T / A - 1).max() < 16 * 2.0 ** -53
