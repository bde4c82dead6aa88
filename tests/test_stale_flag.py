"""When a call clears the flag by which a step skips its inverse y pass: only after
something may have set it (a step, or a batch that the context joined), on the
host-only runtime of tests/host_hip.py."""
import os

import pytest

import host_hip

pytestmark = pytest.mark.skipif(not os.path.exists(host_hip.LIB), reason="libspns.so not built")


@pytest.mark.parametrize("les", [False, True])
@pytest.mark.parametrize("graph", [False, True])
def test_clears_what_may_be_set(tmp_path, les, graph):
    host_hip.run(tmp_path, """
les, graph = %r, %r
s = spns_amd.Solver(Nx=32, nu=1e-3, precision=1, C_Smag=0.17 if les else 0.0, use_graph=graph)
state = np.zeros((3, s.nmodes), complex)
CALLS = [lambda: s.antitransform(), lambda: s.velocity_physical(), lambda: s.ccc(), lambda: s.set_state(state),
         lambda: s.init_random(seed=1), lambda: s.check_energy(1e300), lambda: s.forcing_energy_cascade(np.ones(4), 3)]

def clears(call):
    log()
    call()
    return kernels(log()).count("k_set_int")

assert s.pass_kernels()[1] == 2
for call in CALLS:
    assert clears(call) == 0                      # nothing has set it
for step in (lambda: s.step(1), lambda: s.step(3), lambda: s.profile_passes(1)):
    for call in CALLS:
        step()
        assert clears(call) >= 1                  # the step did
        assert clears(call) == 0                  # and it is clear now
b = spns_amd.Batch(1, 2)
b.attach(0, s)
for call in CALLS:
    b.step([2])                                   # sets it on the device alone
    b.synchronize()
    assert clears(call) >= 1
    b.step([1])
    b.synchronize()
    assert clears(call) >= 1
b.detach(0)
assert clears(CALLS[0]) >= 1                      # the batch's last step
""" % (les, graph))
