"""PLANEWAVE$FFT on the full grid over the lengths of the y and z passes: every
length with a pencil kernel of its own and one (110) that runs the run-time
kernel, on slabs whose pencil counts are no multiple of a tile.  Bounds as for
the other transforms: 1e-12 in FP64, 2e-5 in FP32."""
import math

import numpy as np
import pytest

from oracle import planewave as opw
from harness import relerr

pytestmark = pytest.mark.gpu

PAIRS = [(12, 14), (16, 18), (20, 22), (24, 28), (30, 32), (36, 40), (42, 44), (48, 56), (60, 64), (66, 70),
         (72, 80), (84, 88), (90, 96), (112, 120), (126, 128), (132, 140), (144, 110)]


@pytest.mark.parametrize("n2,n3", PAIRS)
def test_full_grid_lengths(n2, n3):
    import pwgpu
    print(f"case full-grid transform 12 x {n2} x {n3}", flush=True)
    # cutoff |G| <= 1: an edge 2 pi (m + 1/2) holds the components -m..m, 2 m + 1 = n - 1
    rbas = np.diag([2.0 * math.pi * (n / 2 - 0.5) for n in (12, n2, n3)])
    plane = pwgpu.PlaneWave(rbas, 0.5, 0.5)
    pl = opw.Plane(rbas, 0.5, 0.5)
    assert plane.nr == (12, n2, n3) == (pl.nr1, pl.nr2, pl.nr3)
    rng = np.random.default_rng(n2)
    fofg = rng.normal(size=(3, pl.ngl)) + 1j * rng.normal(size=(3, pl.ngl))
    fofr = rng.normal(size=(2, n3, n2, 12)) + 1j * rng.normal(size=(2, n3, n2, 12))
    for prec, tol in ((0, 1e-12), (1, 2e-5)):
        assert relerr(plane.fft_host("GTOR", fofg=fofg, prec=prec), pl.fft_gtor(fofg)) < tol
        assert relerr(plane.fft_host("RTOG", fofr=fofr, prec=prec), pl.fft_rtog(fofr)) < tol


@pytest.mark.parametrize("n", [12, 14, 16, 18, 20, 22, 24, 28, 32, 36, 40, 44, 48, 56, 64, 72, 80, 88, 112, 128, 144])
def test_full_grid_tiles(n):
    """Lengths of one or two stages in wide tiles (a batch that fills the chip)
    and in narrow ones (one band at a time): the same operations on each pencil,
    so the same bits; the batch against the oracle as above.  n is the length
    of the z pass, over 256 pencils, and of the y pass, over 64."""
    import pwgpu
    nb = 200 if n <= 40 else 100
    for nr in ((16, 16, n), (64, n, 12)):
        print(f"case full-grid tiles {nr}", flush=True)
        rbas = np.diag([2.0 * math.pi * (k / 2 - 0.5) for k in nr])
        plane = pwgpu.PlaneWave(rbas, 0.5, 0.5)
        pl = opw.Plane(rbas, 0.5, 0.5)
        assert plane.nr == nr
        rng = np.random.default_rng(n)
        fofg = rng.normal(size=(nb, pl.ngl)) + 1j * rng.normal(size=(nb, pl.ngl))
        fofr = rng.normal(size=(nb, *nr[::-1])) + 1j * rng.normal(size=(nb, *nr[::-1]))
        for prec, tol in ((0, 1e-12), (1, 2e-5)):
            r = plane.fft_host("GTOR", fofg=fofg, prec=prec)
            g = plane.fft_host("RTOG", fofr=fofr, prec=prec)
            for b in (0, nb - 1):
                one = slice(b, b + 1)
                assert np.array_equal(r[one], plane.fft_host("GTOR", fofg=fofg[one], prec=prec)), (nr, prec)
                assert np.array_equal(g[one], plane.fft_host("RTOG", fofr=fofr[one], prec=prec)), (nr, prec)
                assert relerr(r[one], pl.fft_gtor(fofg[one])) < tol
                assert relerr(g[one], pl.fft_rtog(fofr[one])) < tol
        plane.close()


@pytest.mark.parametrize("nb", [1, 4, 5, 7, 8, 12, 13, 15, 16, 21])
def test_x_pass_bands(nb):
    """x passes with whole octets of bands and with one to seven beyond them
    (a band per XCD, or its stripe groups on all of them)."""
    import pwgpu
    from pwgpu import model
    print(f"case x passes of {nb} bands", flush=True)
    s = model.tiny()
    plane = pwgpu.PlaneWave(s.rbas, s.epw_psi, s.epw_rho)
    pl = opw.Plane(s.rbas, s.epw_psi, s.epw_rho)
    rng = np.random.default_rng(nb)
    fofg = rng.normal(size=(nb, pl.ngl)) + 1j * rng.normal(size=(nb, pl.ngl))
    fofr = rng.normal(size=(nb, pl.nr3, pl.nr2, pl.nr1)) + 1j * rng.normal(size=(nb, pl.nr3, pl.nr2, pl.nr1))
    for prec, tol in ((0, 1e-12), (1, 2e-5)):
        assert relerr(plane.fft_host("GTOR", fofg=fofg, prec=prec), pl.fft_gtor(fofg)) < tol
        assert relerr(plane.fft_host("RTOG", fofr=fofr, prec=prec), pl.fft_rtog(fofr)) < tol
