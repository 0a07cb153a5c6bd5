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
