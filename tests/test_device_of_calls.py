"""Calls on a context of another device than the calling thread's current one,
on the host-only runtime of tests/host_hip.py, which refuses a launch or an event
across devices: each succeeds and leaves the current device as it was.  The
state is above the size at which a read goes through pinned chunks."""
import os

import pytest

import host_hip

pytestmark = pytest.mark.skipif(not os.path.exists(host_hip.LIB), reason="libspns.so not built")

CALLS = ["s.get_state()", "s.get_state_planes(3, 5)", "s.get_rhist()", "s.set_state(np.zeros((3, s.nmodes), complex))", "s.init_k41(2)",
         "s.init_random(seed=2)", "s.finish_init(False)", "s.step(1)", "s.velocity_physical()", "s.velocity_physical_step_start()",
         "s.antitransform()", "s.spectrum()", "s.scalars()", "s.check_energy(1e300)", "s.ccc()", "s.invariant_spectra()",
         "s.profile_passes(1)", "s.recalc_timestep()", "s.reconfigure(nu=1e-3)"]


@pytest.mark.parametrize("thread", [False, True])
@pytest.mark.parametrize("call", CALLS)
def test_call_from_another_device(tmp_path, call, thread):
    host_hip.run(tmp_path, """
import threading
cur = ctypes.c_int()

def create():
    return spns_amd.Solver(Nx=96, Ny=64, Nz=64, nu=1e-3, device=1, gradient_invariants=True, keep_step_start=True)

def use(s):
    hip.hipSetDevice(0)
    %s
    hip.hipGetDevice(ctypes.byref(cur))
    assert cur.value == 0, cur.value

s = create()
errors = []
if %r:
    threading.excepthook = lambda a: errors.append(a.exc_value)
    t = threading.Thread(target=use, args=(s,))
    t.start()
    t.join()
else:
    use(s)
assert not errors, errors
""" % (call, thread))
