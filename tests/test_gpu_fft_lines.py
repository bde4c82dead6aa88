"""FFT_package drop-in at the shortest and longest lengths of each dimension and
at column counts that leave a ragged last tile: both directions against numpy,
with guard values behind every buffer that must stay as they were.
Tolerances as in test_gpu_fft.py: 1e-13 (FP64), 2e-6 (FP32) of the field norm."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SHAPES = [(16, 16, 16), (16, 24, 32), (36, 64, 72), (128, 36, 48), (1536, 16, 24), (16, 1536, 36), (24, 16, 1536),
          (1152, 24, 16), (16, 1152, 16), (16, 16, 1152), (24, 576, 1024), (512, 16, 256), (192, 192, 64)]


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("shape", SHAPES)
def test_both_directions_at_the_edges(shape, prec):
    import spns_amd
    Mx, My, Mz = shape
    nk = Mz // 2 + 1
    dt = torch.float64 if prec == 0 else torch.float32
    tol = 1e-13 if prec == 0 else 2e-6
    rng = np.random.default_rng(Mx + My + Mz + prec)
    r = rng.standard_normal(shape)
    nr, nc, guard = Mx * My * 2 * nk, My * Mx * nk * 2, 64

    def buffer(n):
        return torch.full((n + guard,), 7.0, dtype=dt, device="cuda")

    rin, cbuf, rout = buffer(nr), buffer(nc), buffer(nr)
    rp = np.zeros((Mx, My, 2 * nk))
    rp[:, :, :Mz] = r
    rin[:nr] = torch.from_numpy(rp).to("cuda", dt).reshape(-1)
    f = spns_amd.Fft(Mx, My, Mz, precision=prec)
    f.r2c(rin.data_ptr(), cbuf.data_ptr())
    c = cbuf[:nc].double().cpu().numpy().reshape(My, Mx, nk, 2)
    c = c[..., 0] + 1j * c[..., 1]
    ref = np.fft.rfftn(r).transpose(1, 0, 2)
    assert np.linalg.norm(c - ref) / np.linalg.norm(ref) < tol
    # backward, from a spectrum whose end planes carry imaginary parts a c2r drops
    s = ref / r.size
    s[:, :, 0] += 0.25j * np.abs(s[0, 0, 1])
    s[:, :, -1] += 0.25j * np.abs(s[0, 0, 1])
    cbuf[:nc] = torch.from_numpy(np.stack([s.real, s.imag], -1)).to("cuda", dt).reshape(-1)
    f.c2r(cbuf.data_ptr(), rout.data_ptr())
    t = np.fft.ifftn(s, axes=(0, 1), norm="forward")
    back = np.fft.irfft(t, n=Mz, axis=2, norm="forward").transpose(1, 0, 2)
    out = rout[:nr].double().cpu().numpy().reshape(Mx, My, 2 * nk)
    assert np.linalg.norm(out[:, :, :Mz] - back) / np.linalg.norm(back) < tol
    assert (out[:, :, Mz:] == 7.0).all()  # a row's padding is not written
    for b, n in ((rin, nr), (cbuf, nc), (rout, nr)):
        assert bool((b[n:] == 7.0).all())
    f.close()
