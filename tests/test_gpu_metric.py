"""The metric's factor and the fitted tensor at the edges of their blocks (64 fitting functions) and tiles
(16 fitting functions, 128 pairs and fitted functions): all eigenvalues kept (Cholesky), some under the cutoff and
32-bit handles (eigenvectors)."""
import numpy as np
import pytest

from test_gpu_eri_pair import _basis

pytestmark = pytest.mark.gpu


def _handle(orb, aux, mol, **spec):
    from dftax_amd.ks import HipDFKS, HipSpec
    from dftax_amd.xc import PBE0
    return HipDFKS(orb, aux, mol, np.zeros((1, 3)) + 5.0, np.ones(1), PBE0(), 2, HipSpec(keep_int3c=True, **spec),
                   chunk=None)


@pytest.mark.parametrize("naux,norb,close,spec", [
    (1, 1, 0.0, {}), (15, 2, 0.0, {}), (16, 15, 0.0, {}), (63, 3, 0.0, {}), (64, 16, 0.0, {}), (65, 17, 0.0, {}),
    (129, 5, 0.0, {}), (200, 16, 0.0, {}), (66, 4, 1e-4, {}), (130, 16, 1e-4, {}), (65, 4, 0.0, {"precision": "mixed"})])
def test_fitted_tensor_edges(naux, norb, close, spec):
    """B B^T = (mn|P) V+ (P|ls) with V+ over the eigenvalues above the cutoff."""
    from dftax_amd import _native as N
    from dftax_amd.system import Molecule
    from oracle import ref
    rng = np.random.default_rng(naux + norb)
    mol = Molecule(["O"] * 2, np.array([[0.0, 0.0, 0.0], [0.0, 0.1, 2.1]]), "sto-3g")
    # s fitting functions on a lattice, apart enough for a condition number of a few thousand at most
    site = 1.6 * np.indices((6, 6, 6)).reshape(3, -1).T[:naux] + rng.uniform(-0.1, 0.1, (naux, 3))
    if close:   # the last functions all but repeat the first: eigenvalues near close^2, under the cutoff of 1e-7
        site[-2:] = site[:2] + close
    aux = _basis([(0, 0, x, [0.9]) for x in site], True)
    orb = _basis([(0, 0, x, [0.8]) for x in rng.uniform(0.0, 6.0, (norb, 3))], True)
    c = _handle(orb, aux, mol, **spec)
    V, I = ref.int2c(aux), ref.int3c(orb, aux).reshape(norb * norb, naux)
    w, U = np.linalg.eigh(V)
    keep = w > 1e-7 * w[-1]
    assert c.nfit == keep.sum() == naux - (2 if close else 0)
    want = (I @ (U[:, keep] / w[keep])) @ (I @ U[:, keep]).T
    B = c.matrix(N.DFKS_BFIT, (norb * norb, c.nfit)).cpu().numpy()
    # the repository's bound for the fitted tensor
    assert np.abs(B @ B.T - want).max() < 1e-9 * max(1.0, np.abs(want).max())
    b3 = B.reshape(norb, norb, -1)
    assert np.array_equal(b3, b3.transpose(1, 0, 2))
    c.close()
