"""ORTHO_X in one workgroup (up to 32 bands with 8 terms of the series, 24
with 16, 16 with 32) against the oracle: one and two 16 x 16 tiles per edge
and their remainders, the widest set, the first one above it (launch chain),
and spectra of sym(CHIPSI) that ask for 4 to 32 terms.  Both sides form the
same iterates; the series is cut at 1.6e-11 of its first term and the bound is
that of the other stand-alone solves, 1e-10.
"""
import numpy as np
import pytest

from harness import relerr

pytestmark = pytest.mark.gpu


def solve_case(nb, spread, seed=5):
    rng = np.random.default_rng(seed + nb)
    q, _ = np.linalg.qr(rng.normal(size=(nb, nb)))
    e = np.geomspace(1.0, spread, nb)
    anti = 0.01 * rng.normal(size=(nb, nb))
    chipsi = (q * e) @ q.T + (anti - anti.T)
    m = rng.normal(size=(nb, nb))
    chichi = 0.02 * (m @ m.T) / nb
    d = 0.01 * rng.normal(size=(nb, nb))
    psipsi = np.eye(nb) + 0.5 * (d + d.T)
    occ = rng.choice([2.0, 2.0, 1.0, 0.3, 0.0], size=nb)
    return occ, chichi, psipsi, chipsi


@pytest.mark.parametrize("spread", [1.1, 6.0, 60.0])
@pytest.mark.parametrize("nb", [3, 4, 15, 16, 17, 20, 31, 32, 33])
def test_ortho_x_one_workgroup(nb, spread):
    import pwgpu
    from oracle import waves as owv
    occ, chichi, psipsi, chipsi = solve_case(nb, spread)
    lam0 = 0.001 * np.random.default_rng(nb).normal(size=(nb, nb))
    ref, it_ref = owv.ortho_x(occ, chichi, psipsi, chipsi, lam0.copy())
    lam, it = pwgpu.ortho_x(occ, chichi, psipsi, chipsi, lam0)
    assert it == it_ref
    assert relerr(lam, ref) < 1e-10


def test_ortho_x_one_workgroup_refuses():
    """NaN in the overlap and a diverging loop are refused as by the chain."""
    import pwgpu
    from pwgpu import PwError
    occ, chichi, psipsi, chipsi = solve_case(20, 2.0)
    bad = psipsi.copy()
    bad[0, 3] = np.nan
    with pytest.raises(PwError, match="NaN in overlap"):
        pwgpu.ortho_x(occ, chichi, bad, chipsi, np.zeros((20, 20)))
    with pytest.raises(PwError, match="diverge|not converged"):
        pwgpu.ortho_x(occ, 50.0 * chichi, 40.0 * psipsi, chipsi, np.zeros((20, 20)))
