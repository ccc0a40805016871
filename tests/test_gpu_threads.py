"""Device-resident shots built, run and fetched on several threads at once, each
on a stream of its own: the arrays of the same shots one after another.  (Argument
types set on a function object that threads share would be freed under another
thread's call.)"""
import sys
import threading

import numpy as np
import pytest

import cases
import simwave_amd as sw
from simwave_amd import hipmem
from simwave_amd.device import DeviceForward

pytestmark = pytest.mark.gpu


def test_shots_on_several_threads(gpu):
    print("shots on threads", flush=True)
    solvers = [sw.Solver(**cases.make_case(dim=2, shape=(40 + i, 50 - i), space_order=4 + 4 * (i % 2),
                                           tf=0.04)()) for i in range(6)]

    def run(solver, stream=None):
        dev = DeviceForward(solver, stream=stream)
        dev.run(stream, flags=0)       # one run a process may overlap its receivers
        return dev.results(stream)
    want = [run(s) for s in solvers]
    lib = hipmem.default_library()
    bad = []

    def work(i):
        stream = hipmem.Stream(lib)
        try:
            for _ in range(20):
                for got, ref in zip(run(solvers[i], stream), want[i]):
                    np.testing.assert_array_equal(got, ref)
        except BaseException as e:
            bad.append((i, e))
    interval = sys.getswitchinterval()
    sys.setswitchinterval(1e-5)
    try:
        threads = [threading.Thread(target=work, args=(i,)) for i in range(len(solvers))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        sys.setswitchinterval(interval)
    assert not bad, bad[0]
