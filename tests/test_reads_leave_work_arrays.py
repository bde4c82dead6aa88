"""Reads of the state use the context's (or batch's) own transfer
memory, not the passes' work arrays, and calls of several threads on one context
give what they give one after the other."""
import os
import threading

import numpy as np
import pytest

import host_hip

ROOM = 16 << 20


@pytest.mark.skipif(not os.path.exists(host_hip.LIB), reason="libspns.so not built")
@pytest.mark.parametrize("N", [(16, 16, 16), (96, 64, 64)])
def test_copies_come_from_the_transfer_memory(tmp_path, N):
    # every device block that a copy touches is far smaller than the work arrays
    host_hip.run(tmp_path, """
N, room = %r, %d
s = spns_amd.Solver(Nx=N[0], Ny=N[1], Nz=N[2], nu=1e-3)
b = spns_amd.Batch(1, 2)
state = np.zeros((3, s.nmodes), complex)
nbytes = state.nbytes
x2 = 9 * (3 * N[1] // 2) * (3 * N[0] // 2) * ((s.nk[2] + 15) // 16 * 16) * 16
calls = [lambda: s.get_state(), lambda: s.get_state_planes(2, 3), lambda: s.get_rhist()]
if N[0] > 16:
    b.attach(0, s)
    calls.append(lambda: b.fetch(0, state))
for i, call in enumerate(calls):
    log()
    call()
    lines = log()
    copies = [l.split() for l in lines if l.startswith("copy")]
    sizes = [max(int(c[3]), int(c[5])) for c in copies]
    # what was copied, or what the pack kernels moved themselves (16 bytes a thread)
    moved = max(sum(int(c[1]) for c in copies), sum(4096 * int(l.split()[2].split("x")[0]) for l in lines if "pack" in l))
    assert moved >= (3 * 3 * s.nk[1] * s.nk[2] * 16 if i == 1 else nbytes), (i, moved)
    assert all(x <= room and x != x2 for x in sizes), (i, sizes)
""" % (N, ROOM))


@pytest.mark.skipif(not os.path.exists(host_hip.LIB), reason="libspns.so not built")
def test_fetch_is_one_copy(tmp_path):
    # a batch's room holds a whole state of its class (26 MB here)
    host_hip.run(tmp_path, """
s = spns_amd.Solver(Nx=128, Ny=128, Nz=64, nu=1e-3)
b = spns_amd.Batch(1, 2)
b.attach(0, s)
state = np.zeros((3, s.nmodes), complex)
log()
b.fetch(0, state)
copies = [l.split() for l in log() if l.startswith("copy")]
assert [int(c[1]) for c in copies] == [state.nbytes], copies
""")


@pytest.mark.skipif(not os.path.exists(host_hip.LIB), reason="libspns.so not built")
@pytest.mark.parametrize("started", [0, 1, 2])
def test_read_without_memory_for_its_threads(tmp_path, started):
    # a thread that cannot be started is done without
    host_hip.run(tmp_path, """
s = spns_amd.Solver(Nx=96, Ny=64, Nz=64, nu=1e-3)
s.get_state()
out = np.empty((3, s.nmodes), complex)
p = out.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
log()
hip.host_hip_fail_alloc(%d)
rc = s.L.spns_get_state(s.h, p)
hip.host_hip_fail_alloc(-1)
assert rc == 0, (rc, s.L.spns_last_error(s.h))
assert len(kernels(log())) == -(-out.nbytes // (2 << 20))
""" % started)


@pytest.mark.skipif(not os.path.exists(host_hip.LIB), reason="libspns.so not built")
@pytest.mark.parametrize("prec", [0, 1])
def test_threads_take_part_by_size(tmp_path, prec):
    # outwards from 4 MiB, inwards from 8 MiB on: chunks of 2 MiB, else one copy
    host_hip.run(tmp_path, """
s = spns_amd.Solver(Nx=64, nu=1e-3, precision=%d)  # 6.7 MB
state = np.zeros((3, s.nmodes), complex)
log()
s.get_state()
assert kernels(log()).count("k_pack") == 4
s.set_state(state)
copies = [int(l.split()[1]) for l in log() if l.startswith("copy")]
assert copies[0] == state.nbytes, copies
s.get_state_planes(0, 30)  # 3.1 MB
assert kernels(log()).count("k_pack") == 1
""" % prec)


@pytest.mark.skipif(not os.path.exists(host_hip.LIB), reason="libspns.so not built")
@pytest.mark.parametrize("prec", [0, 1])
def test_small_velocity_is_one_copy(tmp_path, prec):
    host_hip.run(tmp_path, """
s = spns_amd.Solver(Nx=16, nu=1e-3, precision=%d)
log()
out = s.velocity_physical()
copies = [l.split() for l in log() if l.startswith("copy")]
assert [int(c[1]) for c in copies] == [out.nbytes], copies
""" % prec)


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("N", [(32, 32, 32), (96, 64, 64)])
def test_threads_reading_one_context(N, prec):
    import spns_amd
    s = spns_amd.Solver(Nx=N[0], Ny=N[1], Nz=N[2], nu=1e-3, C_At=0.5, precision=prec)
    s.init_random(seed=3, k0=4.0)
    s.finish_init(False)
    s.step(3)
    calls = [s.get_state, s.get_rhist, s.velocity_physical, lambda: s.get_state_planes(5, 9)]
    want = [c() for c in calls]
    wrong = []

    def loop(k):
        for i in range(12):
            j = (k + i) % len(calls)
            if not np.array_equal(calls[j](), want[j]):
                wrong.append((k, i, j))

    threads = [threading.Thread(target=loop, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong
    s.close()
