"""The drop-in's line transforms: 128-byte row pieces up to 512 points, and a
transform asks the runtime for nothing but its launches: the grids are the plan's (tests/host_hip.py counts the calls), of each plan's own device."""
import os

import pytest

import host_hip

pytestmark = pytest.mark.skipif(not os.path.exists(host_hip.LIB), reason="libspns.so not built")


@pytest.mark.parametrize("prec", [0, 1])
def test_transforms_make_no_queries(tmp_path, prec):
    host_hip.run(tmp_path, """
f = spns_amd.Fft(48, 36, 64, precision=%d)
buf = [np.zeros(48 * 36 * 66) for _ in range(2)]
log()
f.r2c(buf[0].ctypes.data, buf[1].ctypes.data)
f.c2r(buf[1].ctypes.data, buf[0].ctypes.data)
lines = log()
assert kernels(lines) == ["k_zline", "k_line", "k_line", "k_line", "k_line", "k_zline"], lines
assert not [l for l in lines if l.startswith("call")], lines
""" % prec)


@pytest.mark.parametrize("prec", [0, 1])
def test_row_pieces_of_128_bytes(tmp_path, prec):
    host_hip.run(tmp_path, """
prec = %d
for L in (16, 96, 192, 384, 512):
    f = spns_amd.Fft(L, 16, 16, precision=prec)
    buf = np.zeros((L + 8) * 24 * 24)
    log()
    f.r2c(buf.ctypes.data, buf.ctypes.data)
    x = [l for l in log() if "k_line" in l][1]
    assert "k_lineI%%sLi%%dELi%%dE" %% ("fd"[prec == 0], L, 8 if prec == 0 else 16) in x, x
""" % prec)
