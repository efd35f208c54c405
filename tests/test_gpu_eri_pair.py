"""Three-centre integrals of the bra-pair kernel at its edges, against the oracle's engine:
contractions longer than the primitive pairs it keeps at a time, auxiliary shell counts around
its groups of 16, contracted auxiliary shells, and the cartesian spans it leaves to the
wavefront kernel."""
from __future__ import annotations

import numpy as np
import pytest

from dftax_amd.basis import BasisSet, cart_components, contracted_norm, gto_norm, ncart, nsph

pytestmark = pytest.mark.gpu

# values of normalised functions are at most ~10 and the two engines sum a few hundred terms of that
# size in FP64: the repository's bound for integrals
TOL_INT = 1e-10


def _basis(shells, spherical):
    """A BasisSet from (l, atom, centre, exps) with equal raw coefficients."""
    cols = {k: [] for k in ("l", "atom", "centre", "prim0", "nprim", "ao0", "cart0", "exps", "coefs")}
    ao = cart = 0
    for l, atom, centre, exps in shells:
        c = np.array([gto_norm(l, a) for a in exps])
        if l <= 1:
            c = c * contracted_norm(exps, c, cart_components(l)[0])
        for k, v in (("l", l), ("atom", atom), ("centre", centre), ("prim0", len(cols["exps"])), ("nprim", len(exps)),
                     ("ao0", ao), ("cart0", cart)):
            cols[k].append(v)
        cols["exps"].extend(exps)
        cols["coefs"].extend(c)
        cart += ncart(l)
        ao += nsph(l) if spherical and l >= 2 else ncart(l)
    i32 = {k: np.asarray(cols[k], np.int32) for k in ("l", "atom", "prim0", "nprim", "ao0", "cart0")}
    return BasisSet(centre=np.asarray(cols["centre"], np.float64), exps=np.asarray(cols["exps"]),
                    coefs=np.asarray(cols["coefs"]), spherical=spherical, nao=ao, nao_cart=cart, **i32)


@pytest.mark.parametrize("nprim,naux_shells,aux_prims,spherical",
                         [(1, 1, 1, True), (2, 15, 1, True), (3, 16, 2, True), (7, 17, 1, True), (2, 65, 1, True),
                          (3, 5, 2, False)])
def test_pair_kernel_classes(nprim, naux_shells, aux_prims, spherical):
    from dftax_amd import _native as N
    from dftax_amd.ks import HipDFKS, HipSpec
    from dftax_amd.system import Molecule
    from dftax_amd.xc import PBE0
    from oracle import ref
    rng = np.random.default_rng(100 * nprim + naux_shells)
    mol = Molecule(["O", "H", "H"], np.array([[0.1, -0.2, 0.3], [1.5, 0.4, -0.6], [-1.1, 1.3, 0.2]]), "sto-3g")
    xyz = np.asarray(mol.coords)
    # every l on two atoms: bra pairs on one centre and on two, each l with itself and with the others
    orb = _basis([(l, a, xyz[a], list(0.3 * 2.1 ** np.arange(nprim) * (1 + 0.1 * l + 0.05 * a)))
                  for a in (0, 1) for l in (0, 1, 2, 3)], spherical)
    aux = _basis([(l, a, xyz[a], list(rng.uniform(0.2, 3.0, aux_prims)))
                  for l in (0, 1, 2, 3, 4) for a in rng.integers(0, 3, naux_shells)], True)
    c = HipDFKS(orb, aux, mol, np.zeros((1, 3)) + 5.0, np.ones(1), PBE0(), 10, HipSpec(keep_int3c=True), chunk=None)
    g = c.matrix(N.DFKS_INT3C, (c.nao, c.nao, c.naux)).cpu().numpy()
    want = ref.int3c(orb, aux)
    assert g.shape == want.shape
    assert np.abs(g - want).max() < TOL_INT
    c.close()
