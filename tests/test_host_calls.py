"""Calls on host arrays (csrc/host_arrays.hpp) and the pointer tables of csrc/soa.hpp, run on the CPU: host_calls.cpp puts
the plumbing over HIP functions on host memory."""
import concurrent.futures
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from combustion_amd.build import CSRC, ROCM

HERE = os.path.dirname(os.path.abspath(__file__))
SLOT = (16 << 20) // (4 * 8)  # states of a slice of two inputs and two outputs


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host_calls") / "host_calls.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I" + CSRC,
                           "-I" + os.path.join(ROCM, "include"), os.path.join(HERE, "host_calls.cpp"), "-o", so])
    l = C.CDLL(so)
    l.form_new.restype = C.c_void_p
    l.form_launches.restype = C.c_size_t
    l.form_launches.argtypes = l.form_free.argtypes = [C.c_void_p]
    l.form_replay.argtypes = [C.c_void_p, C.c_size_t]
    l.form_call.argtypes = [C.c_void_p, C.POINTER(C.c_void_p), C.c_size_t, C.POINTER(C.c_void_p), C.c_int, C.c_void_p]
    l.fail_allocation.argtypes = [C.c_long]
    l.unused_allocations.restype = C.c_long
    l.queue_copy.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p, C.c_size_t]
    return l


class Form:
    def __init__(self, lib):
        self.lib, self.form = lib, lib.form_new()

    def __del__(self):
        self.lib.form_free(self.form)

    def __call__(self, ins, outs, n=None, on_device=False, stream=None):
        table = lambda arrays: (C.c_void_p * 2)(*[a.ctypes.data for a in arrays])
        if self.lib.form_call(self.form, table(ins), len(ins[0]) if n is None else n, table(outs), int(on_device), stream):
            raise MemoryError
        return self.lib.form_launches(self.form) - 1


def states(n, seed=1):
    return list(np.random.default_rng(seed).standard_normal((2, n)))


def results(a, b):
    return [a + b, a * b]


def test_host_calls_leave_the_tables_of_captured_launches(lib):
    """Host calls of more sizes than a module has pointer tables: a launch captured before them still has its own."""
    form = Form(lib)
    ins, outs = states(100), list(np.zeros((2, 100)))
    captured = form(ins, outs, on_device=True)
    most = 64 * 2200
    x, y = states(most, 2), list(np.empty((2, most)))
    want = results(*x)
    for n in range(most, 0, -64):
        y[0][:n] = y[1][:n] = 0
        form([a[:n] for a in x], [a[:n] for a in y])
        assert np.array_equal(y[0][:n], want[0][:n]) and np.array_equal(y[1][:n], want[1][:n]), n
    ins[0][:] += 1
    lib.form_replay(form.form, captured)
    assert np.array_equal(outs, results(*ins))


@pytest.mark.parametrize("stream,queued", [(8, 8), (None, None), (8, None)], ids=["caller's", "default", "default-before-caller's"])
def test_host_calls_follow_the_work_queued_before_them(stream, queued, lib):
    """Copies queued on the caller's or on the default stream, into the inputs and out of the outputs, come first."""
    form = Form(lib)
    old, ins = states(100, 3), list(np.zeros((2, 100)))
    outs, first = list(np.full((2, 100), 5.0)), np.zeros(100)
    for to, source in ((ins[0], old[0]), (ins[1], old[1]), (first, outs[0])):
        lib.queue_copy(queued, to.ctypes.data, source.ctypes.data, to.nbytes)
    form(ins, outs, stream=stream)
    assert np.array_equal(outs, results(*old))
    assert np.array_equal(first, np.full(100, 5.0))


@pytest.mark.parametrize("offset", [0, 1, SLOT // 2])
@pytest.mark.parametrize("first", ["low", "high"])
def test_outputs_that_overlap_end_as_the_later_one(first, offset, lib):
    n = 3 * SLOT // 2  # two slices, and helpers that copy
    form, ins = Form(lib), states(n)
    got, want = np.zeros(n + offset), np.zeros(n + offset)
    views = lambda a: [a[:n], a[offset:]] if first == "low" else [a[offset:], a[:n]]
    for y, r in zip(views(want), results(*ins)):
        y[:] = r
    form(ins, views(got))
    assert np.array_equal(got, want)


def test_threads_take_turns_with_the_staging(lib):
    """Host calls of several threads on one module."""
    form = Form(lib)

    def calls(seed):
        for n in (3 * SLOT // 2, 1000, SLOT):
            ins, outs = states(n, seed), list(np.empty((2, n)))
            form(ins, outs)
            if not np.array_equal(outs, results(*ins)):
                return n
        return 0

    with concurrent.futures.ThreadPoolExecutor(4) as pool:
        assert list(pool.map(calls, range(8))) == [0] * 8


@pytest.mark.timeout(100)
def test_a_host_call_that_runs_out_of_memory_fails_by_itself(lib):
    """Each allocation of a call in turn (the helper threads' among them) fails: the call works without or reports it, and
    the next one is whole."""
    ins = states(3 * SLOT // 2)
    failed = 0
    for nth in range(1000):
        form, outs = Form(lib), list(np.zeros((2, len(ins[0]))))
        lib.fail_allocation(nth)
        try:
            form(ins, outs)
            done = True
        except MemoryError:
            done = False
        finally:
            unused = lib.unused_allocations() > 0
            lib.fail_allocation(-1)
        failed += not done
        if not done:
            form(ins, outs)
        assert np.array_equal(outs, results(*ins)), nth
        if unused:
            break
    assert 0 < failed < nth
