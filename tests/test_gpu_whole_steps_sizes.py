"""Whole RODAS4 steps in one kernel (rosenbrock_steps) for the state sizes of 3, 4 and 8 components, with a spare lane
and without, against the separate kernels, which one reactor per wave takes: the same bits (see test_gpu_whole_steps.py)."""
import os

import numpy as np
import pytest
import yaml

from combustion_amd import Mechanism, synth
from combustion_amd.native import Integrator

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def mechanism(species):
    if species == 7:
        return Mechanism(text=synth.generate(7, 6, 1, 1, 3, "sized-7").yaml())
    names = ["O", "O2", "N2"][:species]
    doc = yaml.safe_load(open(synth.mechanism_path("h2o2-10")))
    block = {s["name"]: s for s in doc["species"]}
    doc["phases"][0]["species"] = names
    doc["species"] = [block[n] for n in names]
    doc["reactions"] = [{"equation": "2 O + M <=> O2 + M", "type": "three-body", "rate-constant": {"A": 1.2e17, "b": -1.0, "Ea": 0.0},
                         "efficiencies": {"O2": 2.5}}]
    return Mechanism(text=yaml.safe_dump(doc, sort_keys=False))


@pytest.mark.gpu
@pytest.mark.parametrize("species", [2, 3, 7])
@pytest.mark.parametrize("n,max_steps", [(1, 40), (64 // 3 + 1, 5), (333, 100)])
def test_whole_steps_equal_the_separate_kernels(species, n, max_steps, gpu):
    import torch
    M = mechanism(species)
    assert M.K == species
    T, P, Y = synth.states(species, n, 7, (1000.0, 3000.0), (0.5, 5.0), 0.5)
    results = []
    for one_per_wave in (False, True):
        integ = Integrator(M, rtol=1e-8, atol_T=1e-6, atol_Y=1e-12, jacobian="analytic", one_per_wave=one_per_wave)
        y, p = (torch.from_numpy(np.ascontiguousarray(a)).to(gpu) for a in (np.vstack([T, Y]), P))
        t, h = torch.zeros(n, dtype=torch.float64, device=gpu), torch.full((n,), 1e-10, dtype=torch.float64, device=gpu)
        status, steps = torch.zeros(n, dtype=torch.int32, device=gpu), torch.zeros(n, dtype=torch.int32, device=gpu)
        taken = integ.advance(y, p, t, h, status, steps, 1e-5, max_steps=max_steps)
        results.append([taken] + [x.cpu().numpy() for x in (y, t, h, status, steps)])
    print(species, n, results[0][0], flush=True)
    if max_steps == 100:  # (a few steps may all be rejected ones)
        assert (results[0][2] > 0).all()
    for a, b in zip(*results):
        np.testing.assert_array_equal(a, b)
