"""FP64 products on one G of each pair (G, -G) against the oracle, at the
edges of their tiles: super bands in tiles of 8 (column products; one tile per
wave up to 16, then two), real bands in blocks of 16 with at most 9 per
workgroup (row products), projector rows in blocks of 64 and 128, and a PRO
table without PRO(G) = PRO(-G), which takes the products over the whole sphere.

The random wave functions are flat in G (condition number of their overlap
below 30), so the bounds of the FP64 parity tests apply: 1e-11 on wave
functions and projections, 1e-10 on forces.
"""
import numpy as np
import pytest

from harness import oracle_waveset, relerr
from pwgpu import model

pytestmark = pytest.mark.gpu


def both(nb, nat, asym=False, seed=4):
    import pwgpu
    s = model.tiny(seed=seed, nb=nb, nat=nat, epw_psi=20.0 if nb > 40 else 4.0, epw_rho=24.0)
    o = oracle_waveset(s)
    rng = np.random.default_rng(seed)
    shape = o.psi0.shape
    psi = rng.normal(size=shape) + 1j * rng.normal(size=shape)
    o.psi0, o.psim = psi.copy(), psi.copy()
    plane = pwgpu.PlaneWave(s.rbas, s.epw_psi, s.epw_rho)
    w = pwgpu.Waves.from_system(plane, s, psi=psi)
    if asym:
        o.pro = o.pro * rng.uniform(0.5, 1.5, o.pro.shape)
        w.setr8a("PRO", o.pro)
    return s, o, w


@pytest.mark.parametrize("nb,nat", [(2, 1), (16, 8), (18, 9), (144, 2), (146, 17), (260, 3)])
def test_products(nb, nat):
    print(f"case gamma products nb={nb} nat={nat}", flush=True)
    s, o, w = both(nb, nat)
    o.etot(s.pos)
    w.etot()
    assert relerr(w.getc8a("PSI0"), o.psi0) < 1e-11
    assert relerr(w.getc8a("PROJ"), o.proj) < 1e-11
    assert relerr(w.getc8a("HPSI"), o.hpsi) < 1e-11
    assert relerr(w.getr8a("FORCE"), o.force) < 1e-10


@pytest.mark.parametrize("nb", [16, 146])
def test_products_whole_sphere(nb):
    print(f"case gamma products, PRO(G) != PRO(-G), nb={nb}", flush=True)
    s, o, w = both(nb, 3, asym=True)
    o.etot(s.pos)
    w.etot()
    assert relerr(w.getc8a("PSI0"), o.psi0) < 1e-11
    assert relerr(w.getc8a("PROJ"), o.proj) < 1e-11
    assert relerr(w.getc8a("HPSI"), o.hpsi) < 1e-11


def step(monkeypatch, s, o, w):
    """One CP step on both sides; the oracle's overlap matrices (MAT, OMAT, OOMAT) as well."""
    from oracle import waves as owv
    seen = {}
    solve = owv.ortho_x

    def ortho_x(occ, chichi, psipsi, chipsi, lam):
        seen.update(MAT=psipsi, OMAT=chipsi, OOMAT=chichi)
        return solve(occ, chichi, psipsi, chipsi, lam)

    monkeypatch.setattr(owv, "ortho_x", ortho_x)
    o.etot(s.pos)
    o.propagate()
    o.orthogonalize(s.pos, s.pos)
    for f in (w.etot, w.propagate, w.orthogonalize):
        f()
    return seen


@pytest.mark.parametrize("nb,nat", [(18, 2), (146, 2), (260, 3)])
def test_overlaps_of_a_step(nb, nat, monkeypatch):
    """The three overlap matrices of a step side by side in one launch, at the
    remainders of the band tiles; 1e-11 on the matrices and 1e-9 on the
    multipliers as in the step tests."""
    print(f"case gamma overlaps of a step nb={nb} nat={nat}", flush=True)
    s, o, w = both(nb, nat)
    for k, m in step(monkeypatch, s, o, w).items():
        assert relerr(w.getr8a(k), m) < 1e-11, k
    assert w.geti4("ORTHOITER") == o.ortho_iter
    assert relerr(w.getc8a("RLAM0").real, o.rlam0) < 1e-9


@pytest.mark.parametrize("nb", [16, 146])
def test_step_whole_sphere(nb, monkeypatch):
    """Forces and a step with PRO(G) != PRO(-G): OPSI and the overlaps with it,
    and the forces as the plain sum over the sphere, without the INVERTG
    average of dE/dP, which changes nothing where P(-G) = conj(P(G)) and which
    the kernels leave out."""
    from oracle import waves as owv
    print(f"case gamma step, PRO(G) != PRO(-G), nb={nb}", flush=True)
    monkeypatch.setattr(owv, "dedpro", lambda plane, psi, ded: np.conj(ded) @ psi)
    s, o, w = both(nb, 3, asym=True)
    mats = step(monkeypatch, s, o, w)
    assert relerr(w.getr8a("FORCE"), o.force) < 1e-10
    for k, m in mats.items():
        assert relerr(w.getr8a(k), m) < 1e-11, k
    assert relerr(w.getc8a("RLAM0").real, o.rlam0) < 1e-9
    o.switch()
    w.switch()
    o.etot(s.pos)
    w.etot()
    assert relerr(w.getr8a("FORCE"), o.force) < 1e-9
