"""Rounding of the FP64 transport kernels of several waves (kernels/transport_split.hip, transport_pairs.hip): their error
against the transport formulas on the product's fits in 80-bit arithmetic, beside that of a form that divides and takes its
logarithm with the library: the straight-line program at 53 species, transport_tiled at 160."""
import numpy as np
import pytest

from combustion_amd import synth
from helpers import setup


def extended(M, T, P, Y):
    """[λ, μ, ρD_0..] in 80-bit arithmetic (transport.rs:141-177)."""
    f = lambda a: np.asarray(a).astype(np.longdouble)
    c, v, d = map(f, M.transport_fits(4, 1000.0))
    W, T, P = f(M.molar_mass), f(T), f(P)
    n = f(Y) / W[:, None]
    R = np.longdouble(1.380649e-23 * 6.02214076e23)
    C_tot = P / R / T
    x = np.maximum(n, 0) * (C_tot / n.sum(axis=0))
    x[-1] = C_tot - x[:-1].sum(axis=0)
    powers = np.stack([np.log(T / 1000) ** i for i in range(4)])
    c, v, root = c @ powers, v @ powers, np.sqrt(T)
    mass = (W[:, None] * x).sum(axis=0)
    out = [root / 2 * ((x * c).sum(axis=0) / C_tot + C_tot / (x / c).sum(axis=0)), np.zeros_like(T)]
    for k in range(M.K):
        phi = (1 + v[k] / v * np.sqrt(np.sqrt(W / W[k]))[:, None]) ** 2 / np.sqrt(8 * (1 + W[k] / W))[:, None]
        out[1] += root * x[k] * v[k] ** 2 / (x * phi).sum(axis=0)
        dk = d[k] @ powers
        dk[k] = np.inf
        out.append(root * (mass - W[k] * x[k]) / mass / R / (x / dk).sum(axis=0))
    return np.stack(out)


@pytest.mark.gpu
@pytest.mark.parametrize("name,beside", [("gri-53", "straight"), ("large-160", "fp64+tiled")])
def test_transport_rounds_no_more_than_the_library(name, beside, gpu):
    import torch
    M = setup(name)[0]
    T, P, Y = synth.config_states(name, 1024, 11)
    exact = extended(M, T, P, Y)
    ins = [torch.from_numpy(np.ascontiguousarray(r)).to(gpu) for r in (T, P, *Y)]
    error = {}
    for form in ("fp64", beside):
        got = torch.stack(M.chemistry(2).assemble(form=form)(ins)).cpu().numpy()
        e = np.abs((got - exact) / exact).astype(np.float64)
        error[form] = [e[0].mean(), e[1].mean(), e[2:].mean()]
        print(name, form, error[form], flush=True)
    for a, b in zip(error["fp64"], error[beside]):
        assert a < 1.1 * b
