"""Which z pass a step runs at the standard 3/2 padding, by length, precision and
model (launches on the host-only runtime of tests/host_hip.py): inputs in
registers (k_zreg) for every LES and for DNS below 768 points, except FP32 DNS
at 288 and 384, which with DNS at 768 run k_zfuse.  The tests that compare the z
passes with the block-per-pencil kernel rely on it."""
import os

import pytest

import host_hip

pytestmark = pytest.mark.skipif(not os.path.exists(host_hip.LIB), reason="libspns.so not built")


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("les", [False, True])
def test_kernel_of_each_length(tmp_path, les, prec):
    want = {L: "k_zreg" for L in (24, 36, 48, 72, 96, 144, 192, 288, 384, 576)}
    if les:
        want.update({L: "k_zreg" for L in (768, 1152, 1536)})
    else:
        want[768] = "k_zfuse"
        if prec:
            want.update({288: "k_zfuse", 384: "k_zfuse"})
    host_hip.run(tmp_path, """
want, les, prec = %r, %r, %r
for L, kernel in want.items():
    for variant, name in ((0, kernel), (1, "k_zpass")):
        s = spns_amd.Solver(Nx=16, Nz=2 * L // 3, nu=1e-3, precision=prec, C_Smag=0.17 if les else 0.0, zpass_variant=variant)
        log()
        s.step(1)
        got = [k for k in kernels(log()) if k.startswith("k_z")]
        assert got == [name], (L, variant, got)
        s.close()
""" % (want, les, prec))


def test_pencils_per_block(tmp_path):
    # DNS: two where their registers fit (FP64: not at 36, where 33 spilt, nor from 96 on)
    host_hip.run(tmp_path, """
want = {(L, 0): 2 if L in (24, 48, 72) else 1 for L in (24, 36, 48, 72, 96, 144)}
want.update({(L, 1): 2 for L in (24, 36, 48, 72, 96, 144)})
for (L, prec), pencils in want.items():
    # 24 x 24 pencils on 512 resident blocks: one per group of pencils where they are fewer
    s = spns_amd.Solver(Nx=16, Nz=2 * L // 3, nu=1e-3, precision=prec)
    log()
    s.step(1)
    blocks = [int(l.split()[2].split("x")[0]) for l in log() if "k_zreg" in l]
    assert blocks == [min(512, 576 // pencils)], (L, prec, blocks)
    s.close()
""")
