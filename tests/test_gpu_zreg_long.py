"""The LES z pass with its inputs in registers at the lengths above 576, where a
block's threads are capped and (from 1152 on) hold the products of two points,
against the block-per-pencil kernel: state, energy and CFL maximum after two
steps.  FP64: rounding-level differences, 1e-13.  FP32-split: both sides carry
single-precision transforms, whose rounding moves the state by about 1e-8 in
two steps: 1e-6."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,tol", [(0, 1e-13), (1, 1e-6)])
@pytest.mark.parametrize("L", [768, 1152, 1536])
def test_matches_block_kernel(L, prec, tol):
    import spns_amd
    out = []
    for variant in (0, 1):
        s = spns_amd.Solver(Nx=24, Ny=16, Nz=2 * L // 3, nu=2e-3, C_At=0.25, C_Smag=0.17, precision=prec, zpass_variant=variant)
        s.init_random(seed=L, k0=4.0)
        s.finish_init(False)
        s.step(1)
        s.step(1)
        out.append((s.get_state(), s.scalars()))
        s.close()
    (a, qa), (b, qb) = out
    assert np.linalg.norm(a - b) <= tol * np.linalg.norm(b)
    for k in ("ek", "maxvel", "dt", "time"):
        assert abs(qa[k] - qb[k]) <= tol * abs(qb[k]), k
    # the sums of (du/dx)^2 and ^3 behind the skewness (an O(1) number)
    assert abs(qa["skewness"] - qb["skewness"]) <= 10 * tol
