"""The tiled purification step at the edges of its tile sizes (16 up to n = 352, 32 up to 704, 48 up
to 1056), n a multiple of 16 and not: SCF energies step by step against the eigensolver's."""
from __future__ import annotations

import warnings

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_water,basis,nao", [(1, "def2-svp", 24), (2, "def2-svp", 48), (8, "def2-tzvp", 344),
                                               (15, "def2-svp", 360), (16, "def2-tzvp", 688),
                                               (17, "def2-tzvp", 731), (24, "def2-tzvp", 1032)])
def test_purified_steps_match_eigensolver(n_water, basis, nao):
    from dftax_amd import KS, becke, df, hip, scf, water_cluster
    mol = water_cluster((n_water, 1, 1), seed=7, basis=basis)
    hist = {}
    for density in ("purify", "eigh"):
        k = KS(mol, "PBE", grid=becke(10, 14), coulomb=df(engine=hip(density=density)))
        assert k.nao == nao
        with warnings.catch_warnings():
            warnings.simplefilter("ignore")          # four steps do not converge
            r = scf(k, max_iter=4)
        hist[density] = [h[0] for h in r.history]
        if density == "purify":
            assert k.coulomb.stats()["eigh_steps"] == 0
        k.coulomb.close()
    # both projectors are exact to the purification's tolerance (deviations below 1e-9 squared): the
    # repository's bound for purified against eigensolver energies, per molecule
    for a, b in zip(hist["purify"], hist["eigh"]):
        assert abs(a - b) < 1e-9 * max(1.0, abs(b) / 76.0)
