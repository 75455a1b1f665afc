"""The last mechanisms that two teams of waves take (kernels/rates_split.hip): (2 K_a + K) rows of 1 KB of LDS are all 160 KB
at 54 species with one of them inert, and 159 at 53 that all react; one more species is one team's. Rates against the FP64
oracle as in test_gpu_rates_split.py (with an inert bulk species: one that reacts has the concentration C_tot minus the
others', whose rounding alone moves the rates by more where there is little of it), and the small batches, whose both
sections go in one launch, equal to larger ones."""
import numpy as np
import pytest
import yaml

from combustion_amd import synth
from helpers import relative_error, setup_text, state_floor


def mechanism(species, inert):
    """A generated mechanism of `species` species, the last one inert or left out."""
    if inert:
        return setup_text(synth.generate(species, 5 * species, 10, 8, species, f"edge-{species}").yaml())
    doc = yaml.safe_load(synth.generate(species + 1, 5 * species, 10, 8, species, f"edge-{species}").yaml())
    last = doc["phases"][0]["species"].pop()
    doc["species"] = [s for s in doc["species"] if s["name"] != last]
    for r in doc["reactions"]:
        r.get("efficiencies", {}).pop(last, None)
    return setup_text(yaml.safe_dump(doc, sort_keys=False))


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["fp64", "fast"])
@pytest.mark.parametrize("species,teams", [(54, 2), (55, 1)])
def test_rates_at_the_edge_of_two_teams(species, teams, form, gpu):
    import torch
    M, mech, o = mechanism(species, True)
    prog = M.chemistry(1)
    assert f"#define TEAMS {teams}" in prog.hip_source(form)
    mod = prog.assemble(form=form)
    T, P, Y = synth.states(M.K, 333, 5, (500.0, 3000.0), (0.1, 50.0), 0.3)
    ref, floor = o.batch(T, P, Y, transport=False, threads=8)
    f, tol = (floor, 1e-12) if form == "fp64" else (state_floor(floor, M.active), 1e-5)
    for n in (1, 64, 127, 128, 129, 333):
        got = np.stack([x.cpu().numpy() for x in mod([torch.from_numpy(np.ascontiguousarray(x[:n])).to(gpu) for x in (T, P, *Y)])])
        err = relative_error(got, ref[:, :n], f[:, :n]).max()
        print(species, form, n, err, flush=True)
        assert err < tol, (species, form, n)


@pytest.mark.gpu
@pytest.mark.parametrize("species,inert", [(54, True), (53, False)])
def test_small_batches_at_the_edge_of_two_teams(species, inert, gpu):
    import torch
    M, mech, o = mechanism(species, inert)
    assert (M.K, M.active) == (species, species - inert)
    prog = M.chemistry()
    assert "rates_and_transport(" in prog.hip_source("fp64")
    mod = prog.assemble(form="fp64")
    T, P, Y = synth.states(M.K, 8193, 5, (300.0, 3000.0), (0.1, 50.0), 0.3)
    ins = [torch.from_numpy(np.ascontiguousarray(x)).to(gpu) for x in (T, P, *Y)]
    whole = torch.stack(mod(ins))  # two kernels
    if inert:
        ref, floor = o.batch(T[:200], P[:200], Y[:, :200], threads=8)
        assert relative_error(whole[:, :200].cpu().numpy(), ref, np.abs(floor)).max() < 1e-12
    for n in (1, 65, 8192):
        print(species, n, flush=True)
        assert torch.equal(torch.stack(mod([x[:n].contiguous() for x in ins])), whole[:, :n]), (species, n)
