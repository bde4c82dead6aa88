"""A batch whose last context has left takes a context of another shape class:
its next chunk runs that class's kernels.  On the CPU the launches are compared
with those of a new batch (tests/host_hip.py); on the GPU the results with the
same run alone, bit for bit."""
import os

import pytest

import host_hip

# (N, precision, LES): each batch holds the first class, then the second
PAIRS = [((96, 1, False), (32, 1, False)), ((32, 1, False), (32, 1, True)), ((32, 0, True), (64, 1, False))]

needs_lib = pytest.mark.skipif(not os.path.exists(host_hip.LIB), reason="libspns.so not built")


@needs_lib
@pytest.mark.parametrize("first,second", PAIRS + [(b, a) for a, b in PAIRS])
def test_launches_of_the_new_class(tmp_path, first, second):
    host_hip.run(tmp_path, """
def slot(N, prec, les):
    s = spns_amd.Solver(Nx=N, nu=1e-3, precision=prec, C_Smag=0.17 if les else 0.0)
    s.init_random(seed=1)
    s.finish_init(False)
    return s

def chunk(b, s):
    b.attach(1, s)
    log()
    b.step([0, 2])
    b.synchronize()
    return [l for l in log() if l.startswith("kernel ")]

first, second = %r, %r
runs = [slot(*first), slot(*second), slot(*second)]
b, new = spns_amd.Batch(2, 2), spns_amd.Batch(2, 2)
chunk(b, runs[0])
b.detach(1)
got, want = chunk(b, runs[1]), chunk(new, runs[2])
assert got == want, (got, want)
""" % (first, second))


@needs_lib
def test_refilled_with_its_class_it_keeps_the_chunk(tmp_path):
    # a capture must not meet another thread's context creation: callers that keep
    # the two apart do so for a batch's first chunk only
    host_hip.run(tmp_path, """
def slot(N, **kw):
    return spns_amd.Solver(Nx=N, nu=1e-3, precision=1, **kw)

def captures(b, s):
    b.attach(1, s)
    log()
    b.step([0, 2])
    n = log().count("call hipStreamBeginCapture")
    b.detach(1)
    return n

b = spns_amd.Batch(2, 2)
got = [captures(b, s) for s in (slot(32), slot(32), slot(32, omega=(0.0, 0.0, 1.0), force_eps=0.1), slot(64), slot(64), slot(32))]
assert got == [1, 0, 0, 1, 0, 1], got
""")


@needs_lib
def test_replaced_context_gives_the_class_no_more(tmp_path):
    host_hip.run(tmp_path, """
a, b, c = [spns_amd.Solver(Nx=32, nu=1e-3, precision=1) for _ in range(3)]
batch = spns_amd.Batch(2, 2)
batch.attach(0, a)
batch.attach(0, b)  # takes a's place
a.close()
batch.attach(1, c)
batch.step([1, 1])
""")


@pytest.mark.gpu
@pytest.mark.parametrize("first,second", PAIRS)
def test_results_of_the_new_class(first, second):
    import numpy as np
    import spns_amd

    def slot(N, prec, les, seed):
        s = spns_amd.Solver(Nx=N, nu=1e-3, C_At=0.5, precision=prec, C_Smag=0.17 if les else 0.0)
        s.init_random(seed=seed, k0=4.0)
        s.finish_init(False)
        return s

    b = spns_amd.Batch(2, 4)
    seed = 0
    for case in (first, second, first):
        seed += 1
        s, alone = slot(*case, seed), slot(*case, seed)
        b.attach(1, s)
        for n in (4, 3):
            b.step([0, n])
            alone.step(n)
        b.synchronize()
        assert np.array_equal(s.get_state(), alone.get_state())
        assert np.array_equal(s.spectrum(), alone.spectrum())
        b.detach(1)
        s.close()
        alone.close()
    b.close()
