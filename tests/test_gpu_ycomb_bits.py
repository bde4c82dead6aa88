"""The combined forward y pass + epilogue (+ next inverse y pass) against the
separate kernels (SPNS_EPI=split) at every y length that has it, with one and
with several butterflies a thread (LES from 128 on): state and history after four
steps bit for bit, in both precisions.  Without forcing nothing of the state
depends on the shell sums, whose order differs: those to 1e-13."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = [(16, 10), (24, 16), (32, 20), (36, 24), (48, 32), (64, 42), (72, 48), (96, 64), (128, 84), (144, 96), (192, 128)]


def _run(**kw):
    import spns_amd
    s = spns_amd.Solver(nu=2e-3, C_At=0.5, **kw)
    s.init_random(seed=kw["Ny"], k0=4.0)
    s.finish_init(False)
    for _ in range(4):
        s.step(1)
    out = s.get_state(), s.get_rhist(), s.spectrum(), s.pass_kernels()[1]
    s.close()
    return out


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("les", [False, True])
@pytest.mark.parametrize("My,Ny", LENGTHS)
def test_state_bits_of_the_separate_kernels(monkeypatch, My, Ny, les, prec):
    kw = dict(Nx=24, Ny=Ny, Nz=64, My=My, precision=prec, C_Smag=0.17 if les else 0.0)
    a = _run(**kw)
    monkeypatch.setenv("SPNS_EPI", "split")
    b = _run(**kw)
    assert (a[3], b[3]) == (0 if les and prec and My == 192 else 2, 0)
    assert np.array_equal(a[0], b[0])
    assert np.array_equal(a[1], b[1])
    assert np.linalg.norm(a[2] - b[2]) <= 1e-13 * np.linalg.norm(b[2])
