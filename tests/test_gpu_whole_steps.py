"""Whole RODAS4 steps in one kernel (rosenbrock_steps in kernels/rosenbrock.hip) against the separate kernels, which one
reactor per wave still takes: the same operations in the same order, so the same bits in every state, time, step size and
count, for batches around one wave's reactors, with reactors of every status, step limits inside and at a launch's end
and an end time already reached."""
import os

import numpy as np
import pytest

from combustion_amd import Mechanism
from combustion_amd.native import Integrator

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


@pytest.mark.gpu
@pytest.mark.parametrize("n,max_steps", [(1, 200000), (9, 200000), (10, 203), (63, 5), (64, 8), (65, 9), (1000, 300), (1000, 200000)])
def test_whole_steps_equal_the_separate_kernels(gpu, n, max_steps):
    import torch
    d = np.load(os.path.join(GOLDEN, "reactor_handwritten.npz"))
    M = Mechanism(os.path.join(GOLDEN, "handwritten.yaml"))
    rng = np.random.default_rng(n)
    at = np.arange(n) % len(d["T0"])
    y0 = np.vstack([d["T0"][at] * rng.uniform(0.95, 1.05, n), d["Y0"][:, at]])
    t0 = np.where(np.arange(n) % 11 == 3, 1e-3, 0.0)      # already at the end time
    status0 = np.where(np.arange(n) % 7 == 5, np.arange(n) % 3, 0).astype(np.int32)  # some finished or collapsed before
    results = []
    for one_per_wave in (False, True):
        integ = Integrator(M, rtol=1e-8, atol_T=1e-6, atol_Y=1e-12, jacobian="analytic", one_per_wave=one_per_wave)
        y, P, t, status = (torch.from_numpy(np.ascontiguousarray(a)).to(gpu) for a in (y0, d["P"][at], t0, status0))
        h = torch.full((n,), 1e-9, dtype=torch.float64, device=gpu)
        steps = torch.full((n,), 3, dtype=torch.int32, device=gpu)
        taken = integ.advance(y, P, t, h, status, steps, 1e-3, max_steps=max_steps)
        results.append([taken] + [x.cpu().numpy() for x in (y, t, h, status, steps)])
    print(n, max_steps, results[0][0], flush=True)
    for a, b in zip(*results):
        np.testing.assert_array_equal(a, b)
    if max_steps == 200000:
        assert (results[0][4][status0 == 0] == 1).all()


@pytest.mark.gpu
def test_batches_on_either_side_of_the_rule_agree(gpu):
    """36864 reactors of six species (nine a wave) are the most that run whole steps: one more, and every reactor's values
    are the same."""
    import torch
    d = np.load(os.path.join(GOLDEN, "reactor_handwritten.npz"))
    M = Mechanism(os.path.join(GOLDEN, "handwritten.yaml"))
    results = []
    for n in (36864, 36865):
        at = np.arange(n) % len(d["T0"])
        T = d["T0"][at] * (1 + 0.05 * np.sin(np.arange(n)))
        y, P = (torch.from_numpy(np.ascontiguousarray(a)).to(gpu) for a in (np.vstack([T, d["Y0"][:, at]]), d["P"][at]))
        t, h = torch.zeros(n, dtype=torch.float64, device=gpu), torch.full((n,), 1e-9, dtype=torch.float64, device=gpu)
        status, steps = torch.zeros(n, dtype=torch.int32, device=gpu), torch.zeros(n, dtype=torch.int32, device=gpu)
        Integrator(M, rtol=1e-8, atol_T=1e-6, atol_Y=1e-12).advance(y, P, t, h, status, steps, 1e-3, max_steps=60)
        results.append([x.cpu().numpy()[..., :36864] for x in (y, t, h, status, steps)])
    for a, b in zip(*results):
        np.testing.assert_array_equal(a, b)
