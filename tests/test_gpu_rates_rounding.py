"""Rounding of the FP64 rates of teams of waves (kernels/rates_split.hip): their error against an evaluation of the same
program in 80-bit arithmetic, beside that of the form with the library's exponential, logarithm and division."""
import ctypes as C
import re
import subprocess

import numpy as np
import pytest

from combustion_amd import synth
from helpers import setup, setup_text


def extended(text, states, rows, directory):
    """The straight-line program `text` (form "straight") on the CPU in 80-bit arithmetic, its constants as they are."""
    body = text[text.index("const double r0 = "):text.rindex("}")]
    body = re.sub(r"\(double\)in\[(\d+)\]\[id\]", r"in[\1 * n + id]", body)
    body = re.sub(r"out\[(\d+)\]\[id\]", r"out[\1 * n + id]", body)
    body = re.sub(r"(0x[0-9a-f.]+p[+-]\d+)", r"\1L", body)
    body = re.sub(r"\b(?:__builtin_)?(exp|log|fmin|fmax)\(", r"\1l(", re.sub(r"\bdouble\b", "long double", body))
    source = directory / "extended.c"
    source.write_text(f"#include <math.h>\n#include <stdbool.h>\nvoid run(const double* in, long double* out, long n) {{\n  for (long id = 0; id < n; id++) {{\n{body}\n  }}\n}}\n")
    subprocess.check_call(["gcc", "-O1", "-w", "-fPIC", "-shared", str(source), "-o", str(directory / "extended.so"), "-lm"])
    out = np.empty((rows, states.shape[1]), np.longdouble)
    C.CDLL(str(directory / "extended.so")).run(C.c_void_p(states.ctypes.data), C.c_void_p(out.ctypes.data), C.c_long(states.shape[1]))
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("species", [53, 60])
def test_rates_round_no_more_than_the_library(species, gpu, tmp_path):
    import torch
    M = setup("gri-53")[0] if species == 53 else setup_text(synth.generate(species, 300, 10, 10, species, f"sized-{species}").yaml())[0]
    T, P, Y = synth.states(M.K, 4096, 11, *synth.STATE_RANGES["gri-53"])
    states = np.ascontiguousarray(np.vstack([T, P, Y]))
    prog = M.chemistry(1)
    exact = extended(prog.hip_source("straight"), states, M.active, tmp_path)
    size = np.abs(exact).max(axis=0)
    error = {}
    for form in ("fp64", "straight"):
        got = torch.stack(prog.assemble(form=form)(list(torch.from_numpy(states).to(gpu)))).cpu().numpy()
        error[form] = (np.abs(got - exact).max(axis=0) / size).astype(np.float64)
        print(species, form, error[form].mean(), np.median(error[form]), error[form].max(), flush=True)
    # the two round in the same places but for the divisions, which are Newton steps of at most an ulp more in one
    assert error["fp64"].mean() < 1.1 * error["straight"].mean()
    assert np.median(error["fp64"]) < 1.1 * np.median(error["straight"])
