"""ORTHO_X by row-panel chains against the oracle: remainders of the panels of
4 and 8 rows, of the column tiles of 16 and of the groups of 8 and 48 k, one
column tile per wave and more (above 256 bands), the widest set with a
Newton-Schulz step in one launch and the first one above it, 4 to 32 terms of
the series (up to 8 built in one launch).  Both sides form the same iterates;
the series is cut at 1.6e-11 of its first term and the bound is that of the
other stand-alone solves, 1e-10.
"""
import numpy as np
import pytest

from harness import relerr
from test_gpu_ortho_small import solve_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,spread", [(33, 1.1), (36, 6.0), (39, 60.0), (47, 1.1), (48, 6.0), (64, 1.1), (97, 6.0),
                                       (100, 1.1), (144, 6.0), (160, 1.1), (161, 1.1), (255, 1.1), (256, 1.1),
                                       (257, 1.1), (300, 6.0), (620, 1.1)])
def test_ortho_x_row_panels(nb, spread):
    import pwgpu
    from oracle import waves as owv
    occ, chichi, psipsi, chipsi = solve_case(nb, spread)
    lam0 = 0.001 * np.random.default_rng(nb).normal(size=(nb, nb))
    ref, it_ref = owv.ortho_x(occ, chichi, psipsi, chipsi, lam0.copy())
    lam, it = pwgpu.ortho_x(occ, chichi, psipsi, chipsi, lam0)
    assert it == it_ref
    assert relerr(lam, ref) < 1e-10


@pytest.mark.parametrize("nb", [5, 32, 33, 65])
def test_ortho_x_column_major(nb):
    """The C entry on column-major matrices gives the bits of the row-major one
    (the matrices are transposed on the device, edges of 32 x 32 tiles)."""
    import ctypes

    import pwgpu
    from pwgpu import load
    from pwgpu._lib import dptr
    occ, chichi, psipsi, chipsi = solve_case(nb, 1.1)
    lam0 = 0.001 * np.random.default_rng(nb).normal(size=(nb, nb))
    ref, it_ref = pwgpu.ortho_x(occ, chichi, psipsi, chipsi, lam0)
    col = [np.array(m.T, dtype=np.float64, order="C") for m in (chichi, psipsi, chipsi, lam0)]
    it = ctypes.c_int()
    assert load().pw_ortho_x(nb, dptr(occ), *[dptr(m) for m in col], ctypes.byref(it)) == 0
    assert it.value == it_ref
    assert np.array_equal(col[3].T, ref)


@pytest.mark.parametrize("nb", [20, 48, 146])
def test_no_terms_where_the_loop_ends(nb):
    """The series is applied once per update of the multipliers: not in the
    iteration whose GAMN is converged, in one workgroup and by panels."""
    from test_gpu_gamma import both
    print(f"case series passes nb={nb}", flush=True)
    s, o, w = both(nb, 3)
    for f in (w.etot, w.propagate, w.orthogonalize):
        f()
    assert w.geti4("ORTHOITER") > 1 and w.geti4("ORTHOEIGEN") == 0
    assert w.geti4("ORTHOPASSES") == w.geti4("ORTHOITER") - 1


@pytest.mark.parametrize("nb,spread", [(125, 6.0), (128, 6.0), (129, 6.0), (264, 1.1), (265, 1.1), (416, 1.1),
                                       (609, 1.1)])
def test_ortho_x_sixteen_rows(nb, spread):
    """Terms of the series by panels of 16 rows, from more than one panel of 8
    rows per CU on: whole panels, remainders of 1, 8, 9 and 13 rows, and the widest
    set with terms (its two panels fill a CU's LDS)."""
    import pwgpu
    from oracle import waves as owv
    print(f"case 16-row panels nb={nb}", flush=True)
    occ, chichi, psipsi, chipsi = solve_case(nb, spread)
    lam0 = 0.001 * np.random.default_rng(nb).normal(size=(nb, nb))
    ref, it_ref = owv.ortho_x(occ, chichi, psipsi, chipsi, lam0.copy())
    lam, it = pwgpu.ortho_x(occ, chichi, psipsi, chipsi, lam0)
    assert it == it_ref
    assert relerr(lam, ref) < 1e-10
