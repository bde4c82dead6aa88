"""The step's reductions at the edges of the finalize's shell blocks (64 shells
each): E(K), E, enstrophy, the CFL maximum, dt and the skewness sums against the
FP64 oracle, over several launches in a row.  Sums of at most ~1e5 positive
terms in FP64 in another order differ by at most ~1e-13 relative; 1e-12 as in
the parity tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("les", [False, True])
@pytest.mark.parametrize("N,M,nbins", [((16, 16, 16), None, 15), ((64, 64, 86), (96, 96, 144), 64),
                                       ((64, 64, 88), (96, 96, 144), 65), ((64, 24, 128), None, 74)])
def test_reductions_across_shell_blocks(N, M, nbins, les):
    import spns_amd
    from oracle.oracle import Oracle

    kw = dict(Nx=N[0], Ny=N[1], Nz=N[2], nu=2e-3, C_At=0.5, C_Smag=0.17 if les else 0.0)
    if M:
        kw.update(Mx=M[0], My=M[1], Mz=M[2])
    g, o = spns_amd.Solver(force_eps=0.1, **kw), Oracle(force_eps=0.1, force_kmin=1, force_kmax=2, **kw)
    assert g.nbins == nbins
    for s in (g, o):
        s.init_random(seed=5, k0=4.0)
        s.finish_init(False)
    for _ in range(3):
        g.step(1)
        o.step(1)
        a, b, sa, sb = g.spectrum(), o.spectrum(), g.scalars(), o.scalars()
        assert np.linalg.norm(a - b) <= 1e-12 * np.linalg.norm(b)
        assert abs(a.sum() - sa["ek"]) <= 1e-13 * sa["ek"]
        for k in ("time", "dt", "maxvel"):
            assert abs(sa[k] - sb[k]) <= 1e-12 * abs(sb[k]), k
        assert abs(sa["ek"] - b.sum()) <= 1e-12 * sa["ek"]
    g.close()
