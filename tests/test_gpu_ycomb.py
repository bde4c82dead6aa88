"""The combined forward y pass + epilogue (+ next inverse y pass) of the short y
lengths, DNS and LES, against the separate kernels (SPNS_EPI=split): state,
history, spectrum and scalars after four steps, and bit for bit against its own
form without the inverse pass (SPNS_YINV=0).  Against the separate kernels only
the order of the shell sums (which feed the forcing) differs: 1e-13 in FP64; in
FP32-split the history is stored in FP32, so one ulp of it may differ: 1e-7."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NY = [16, 24, 32, 48, 64, 96]  # y lengths 24, 36, 48, 72, 96, 144
CASES = [dict(Nx=16, Nz=16), dict(Nx=24, Nz=64, omega=(0.5, 0.0, 3.0), force_eps=0.1), dict(Nx=31, Mx=48, Nz=25, Mz=48)]


def _run(steps=4, **kw):
    import spns_amd
    s = spns_amd.Solver(nu=2e-3, C_At=0.5, **kw)
    s.init_random(seed=kw["Ny"], k0=4.0)
    s.finish_init(False)
    for _ in range(steps):
        s.step(1)
    out = s.get_state(), s.get_rhist(), s.spectrum(), s.scalars(), s.pass_kernels()[1]
    s.close()
    return out


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("les", [False, True])
@pytest.mark.parametrize("kw", CASES)
@pytest.mark.parametrize("Ny", NY)
def test_combined_matches_separate(monkeypatch, Ny, kw, les, prec):
    kw = dict(kw, Ny=Ny, precision=prec, C_Smag=0.17 if les else 0.0)
    a = _run(**kw)
    monkeypatch.setenv("SPNS_YINV", "0")
    b = _run(**kw)
    monkeypatch.setenv("SPNS_EPI", "split")
    c = _run(**kw)
    assert (a[4], b[4], c[4]) == (2, 1, 0)
    for x, y in zip(a[:3], b[:3]):
        assert np.array_equal(x, y)
    assert a[3] == b[3]
    tol = 1e-13 if prec == 0 else 1e-7
    for x, y in zip(a[:3], c[:3]):
        assert np.linalg.norm(x - y) <= tol * np.linalg.norm(y)
    for k in ("dt", "time", "ek", "om", "maxvel"):
        assert abs(a[3][k] - c[3][k]) <= tol * abs(c[3][k]), k
