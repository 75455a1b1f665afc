"""Which kernels an FP64 module of both sections compiles and prints (CPU only): rates_and_transport in the place of the
sections' own kernels where both run one lane per state, beside them for teams of four waves, none otherwise."""
import os

import pytest

from combustion_amd import synth
from helpers import setup_text


def program(species):
    return setup_text(synth.generate(species, 2 * species, 2, 1, species, f"sized-{species}").yaml())[0].chemistry(3)


@pytest.mark.parametrize("species,kernels", [(10, {"rates_and_transport"}), (24, {"rates_and_transport"}),
                                             (33, {"rates_fp64", "transport_fp64", "rates_and_transport"}), (56, {"rates_fp64", "transport_fp64"})])
def test_modules_compile_what_they_launch(species, kernels, tmp_path, monkeypatch):
    prog = program(species)
    text = prog.hip_source("fp64")
    assert ("rates_and_transport(" in text) == ("rates_and_transport" in kernels)
    rates, transport = text.split("// ---- transport ----")
    for section, name in ((rates, "rates_fp64("), (transport, "transport_fp64(")):
        assert (name in section or f"#define NAME {name[:-1]}" in section) == (name[:-1] in kernels)
    monkeypatch.setenv("COMBUSTION_AMD_KERNEL_CACHE", str(tmp_path))
    prog.compile("fp64")
    assert {f.rsplit("-", 1)[0] for f in os.listdir(tmp_path)} == kernels
