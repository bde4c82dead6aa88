"""State and velocity in and out of the GPU: the packed copies against the
values themselves (bit for bit) and, for the velocity, numpy's inverse FFT of
the state.  Sizes: below and above the threaded copy's threshold (8 MiB), odd
retained counts, a chunk remainder, length-factor masks, and a z length whose
export does not fit the work arrays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [dict(Nx=16), dict(Nx=31, Ny=32, Nz=21, Mx=48, My=48, Mz=36), dict(Nx=96, Ny=64, Nz=64), dict(Nx=81, Ny=64, Nz=94, Mx=128, My=96, Mz=144)]


def _state(s, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal((3, s.nmodes)) + 1j * rng.standard_normal((3, s.nmodes))


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("kw", SIZES)
def test_state_round_trip_is_exact(kw, prec):
    import spns_amd
    s = spns_amd.Solver(nu=1e-3, precision=prec, **kw)
    for seed in (1, 2):
        u = _state(s, seed)
        s.set_state(u)
        assert np.array_equal(s.get_state(), u)
    box = u.reshape(3, *s.nk)
    for i2, n in ((0, 1), (3, 5), (s.nk[0] - 2, 2), (4, 0)):
        assert np.array_equal(s.get_state_planes(i2, n), box[:, i2:i2 + n])
    assert not s.get_rhist().any()
    s.close()


def test_length_factor_masks_zero_on_upload():
    import spns_amd
    s = spns_amd.Solver(Nx=16, Ny=16, Nz=32, Lx=1, Ly=1, Lz=2, isNotCubic=True, nu=1e-2)
    u = _state(s, 3)
    s.set_state(u)
    box = u.reshape(3, *s.nk).copy()
    box[:, :, :, 1::2] = 0.0
    assert np.array_equal(s.get_state(), box.reshape(3, -1))
    s.close()


@pytest.mark.parametrize("slots", [1, 3])
def test_batch_fetch_matches_get_state(slots):
    import spns_amd
    b = spns_amd.Batch(slots, 4)
    runs = []
    for k in range(slots):
        s = spns_amd.Solver(Nx=96, Ny=64, Nz=32, nu=1e-3, C_At=0.5, precision=1)
        s.init_random(seed=k, k0=4.0)
        s.finish_init(False)
        b.attach(k, s)
        runs.append(s)
    pins = [spns_amd.Pinned((3, s.nmodes), np.complex128) for s in runs]
    for chunk in ([3] * slots, [2] * slots):
        b.step(chunk)
        for k in range(slots):
            b.fetch(k, pins[k].array)
        b.synchronize()
        for k in range(slots):
            assert np.array_equal(pins[k].array, runs[k].get_state())
    b.close()


# FP64: an unnormalised c2r of O(1) modes, 1e-13 relative as in the transform
# tests; FP32-split: single-precision transforms, 2e-6
@pytest.mark.parametrize("prec,tol", [(0, 1e-13), (1, 2e-6)])
@pytest.mark.parametrize("kw", SIZES + [dict(Nx=16, Ny=24, Nz=16, Mz=768)])
def test_velocity_matches_numpy(kw, prec, tol):
    import spns_amd
    s = spns_amd.Solver(nu=1e-3, C_At=0.5, precision=prec, keep_step_start=True, **kw)
    s.init_random(seed=4, k0=4.0)
    s.finish_init(False)

    def phys(state):
        Mx, My, Mz = s.shape
        nk2, nk1, nk3 = s.nk
        f = np.zeros((3, My, Mx, Mz // 2 + 1), complex)
        i1 = np.where(np.arange(nk1) <= nk1 // 2, np.arange(nk1), np.arange(nk1) - nk1) % Mx
        i2 = np.where(np.arange(nk2) <= nk2 // 2, np.arange(nk2), np.arange(nk2) - nk2) % My
        f[:, i2[:, None], i1[None, :], :nk3] = state.reshape(3, *s.nk)
        return np.fft.irfftn(f, s=(My, Mx, Mz), axes=(1, 2, 3), norm="forward").transpose(0, 2, 1, 3)

    start = s.get_state()
    ref = phys(start)
    for _ in range(2):
        assert np.linalg.norm(s.velocity_physical() - ref) <= tol * np.linalg.norm(ref)
    s.step(1)
    # the last step's start field, and the current one
    assert np.linalg.norm(s.velocity_physical_step_start() - ref) <= tol * np.linalg.norm(ref)
    ref = phys(s.get_state())
    assert np.linalg.norm(s.velocity_physical() - ref) <= tol * np.linalg.norm(ref)
    s.close()
