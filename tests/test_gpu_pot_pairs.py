"""POTENTIAL$VOFRHO on one G of each pair (G, -G): every shell of compensation
moments (the kernels' LMRXX 1, 4, 9, 16, 25), atom counts that are no multiple
of an atom group or of a workgroup's waves, atoms of alternating species, no
atoms, and setup tables without T(G) = T(-G), which take every G on its own.
Bounds as in test_gpu_potential.py."""
import numpy as np
import pytest

from harness import relerr
from oracle import planewave as opw
from oracle import potential as opot
from pwgpu import model

pytestmark = pytest.mark.gpu


def check(nat, lmrxx, asym, functional=1):
    import pwgpu
    s = model.tiny(nat=max(nat, 1), seed=nat + lmrxx, epw_rho=14.0)
    s.species = [model.si_species(), model.o_species()]
    pos, isp = s.pos[:nat], np.arange(nat) % 2
    pl = opw.Plane(s.rbas, s.epw_rho, s.epw_rho)
    rng = np.random.default_rng(nat)
    rho = s.valence_density((pl.nr1, pl.nr2, pl.nr3))
    tabs = s.potential_tables(pl.g2)
    if asym:
        tabs = tabs * rng.uniform(0.7, 1.3, tabs.shape)
    qlm = rng.normal(0.0, 0.3, (nat, lmrxx))
    lmrx = np.array([lmrxx, min(lmrxx, 4)])
    for a in range(nat):
        qlm[a, lmrx[isp[a]]:] = 0.0
    o = opot.vofrho(pl, rho, pos, isp, qlm, {"pscorg": tabs[0], "vbarg": tabs[1], "g0": tabs[2], "v0": tabs[3]},
                    lmrx=lmrx, functional=functional) if nat else None
    pot = pwgpu.Potential(pwgpu.PlaneWave(s.rbas, s.epw_rho, s.epw_rho), tabs, lmrx=lmrx, functional=functional)
    g = pot.vofrho(isp, pos, qlm, rho)
    if o is None:                      # the bare density: its own Hartree energy and local potential
        o = opot.vofrho(pl, rho, np.zeros((0, 3)), np.zeros(0, dtype=int), np.zeros((0, 1)),
                        {"pscorg": tabs[0], "vbarg": tabs[1], "g0": tabs[2], "v0": tabs[3]}, lmrx=lmrx,
                        functional=functional)
    for k in ("ehartree", "exc", "rhob"):
        assert abs(g[k] - o[k]) <= 1e-10 * max(abs(o[k]), 1e-12), (k, g[k], o[k])
    assert relerr(g["v"], o["v"]) < 1e-10
    if nat:
        assert relerr(g["vqlm"], o["vqlm"]) < 1e-10
        assert relerr(g["force"], o["force"]) < 1e-9


SHELLS = [(5, 1), (18, 1), (3, 4), (5, 9), (4, 16), (3, 25), (0, 1)]


# one atom in its own density has no force beyond rounding when each G stands
# on its own, so that case has symmetric tables only
@pytest.mark.parametrize("nat,lmrxx,asym", [(1, 1, False)] + [(*c, a) for c in SHELLS for a in (False, True)])
def test_pairs(nat, lmrxx, asym):
    print(f"case vofrho pairs nat={nat} lmrxx={lmrxx} asym={asym}", flush=True)
    check(nat, lmrxx, asym)


def test_pairs_pbe():
    print("case vofrho pairs, PBE", flush=True)
    check(5, 4, False, functional=10)
    check(5, 4, True, functional=10)
