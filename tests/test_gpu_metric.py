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


def _cholesky80(V):
    L = V.astype(np.longdouble)
    for j in range(len(L)):
        L[j, j] = np.sqrt(L[j, j])
        L[j + 1:, j] /= L[j, j]
        L[j + 1:, j + 1:] -= np.outer(L[j + 1:, j], L[j + 1:, j])
    return np.tril(L)


@pytest.mark.parametrize("heavy,seed", [(3, 0), (5, 0), (5, 1), (5, 2), (6, 0)])
def test_rounding_on_molecules(heavy, seed):
    """B B^T at a molecule's conditioning (3e6 to 7e6) against 80 bits, over 200 pairs: eigenvectors of the metric are
    1.3 to 4.2e-15 off (norm against norm) on trees of 2 to 10 heavy atoms, a Cholesky factor taken atom by atom 2.0 to
    7.1e-15; a blocked factor by falling l and exponent, replayed with the integrals of the oracle, at most 1.4e-15."""
    from dftax_amd import Molecule, _native as N, tree_molecule
    from dftax_amd.basis import build_basis
    mol = tree_molecule(heavy, np.random.default_rng(heavy), basis="def2-svp")
    xyz = mol.coords + 0.05 * np.random.default_rng(seed).standard_normal(mol.coords.shape)
    mol = Molecule(mol.symbols, xyz, "def2-svp", spherical=True)
    orb, aux = (build_basis(mol.symbols, xyz, b, spherical=True) for b in ("def2-svp", "even-tempered-jk"))
    c = _handle(orb, aux, mol)
    assert c.nfit == c.naux
    V = c.matrix(N.DFKS_INT2C, (c.naux, c.naux)).cpu().numpy().astype(np.longdouble)
    rows = np.random.default_rng(0).choice(c.nao ** 2, 200, replace=False)
    I = c.matrix(N.DFKS_INT3C, (c.nao ** 2, c.naux)).cpu().numpy()[rows].T.astype(np.longdouble)
    B = c.matrix(N.DFKS_BFIT, (c.nao ** 2, c.nfit)).cpu().numpy()[rows].T.astype(np.longdouble)
    c.close()
    L = _cholesky80(0.5 * (V + V.T))
    Y = I.copy()
    for i in range(len(L)):
        Y[i] = (Y[i] - L[i, :i] @ Y[:i]) / L[i, i]
    want = Y.T @ Y
    off = np.linalg.norm((B.T @ B - want).astype(float)) / np.linalg.norm(want.astype(float))
    assert off < 2.5e-15


def _span(case):
    """Fitting functions, the metric cutoff as a multiple of the smallest eigenvalue's share (None: the default), and
    whether every eigenvalue is kept by a factor without eigenvectors."""
    rng = np.random.default_rng(5)
    if case == "wide":
        # 400 functions far apart, eigenvalues 4 pi / exponent = sqrt(i / 400): crowded at the top, where 24 Lanczos
        # steps end 1.7e-3 short, so that the bound 1.001 times the Ritz value is under the largest
        site = 1e8 * np.indices((8, 8, 8)).reshape(3, -1).T[:400] + 0.0
        return _basis([(0, 0, x, [4.0 * np.pi / np.sqrt(k / 400.0)]) for k, x in enumerate(site, 1)], True), None, False
    site = 1.6 * np.indices((5, 5, 5)).reshape(3, -1).T[:90] + rng.uniform(-0.1, 0.1, (90, 3))
    aux = _basis([(0, 0, x, [0.9]) for x in site], True)
    return aux, *{"kept": (None, True), "above": (0.97, True), "below": (1.03, False), "zero": (0.0, True)}[case]


@pytest.mark.parametrize("case", ["kept", "above", "below", "zero", "wide"])
def test_which_factor(case):
    """The Cholesky factor stands where the smallest eigenvalue is 3 % over the cutoff, and eigenvectors where it is 3 %
    under it (one function fewer) or where the bound on the largest does not hold; B B^T is that of the eigenvalues
    above the cutoff in every case."""
    from dftax_amd import _native as N
    from dftax_amd.system import Molecule
    from oracle import ref
    aux, share, chol = _span(case)
    orb = _basis([(0, 0, x, [0.8]) for x in np.random.default_rng(6).uniform(0.0, 6.0, (5, 3))], True)
    V, I = ref.int2c(aux), ref.int3c(orb, aux).reshape(25, -1)
    w, U = np.linalg.eigh(V)
    cutoff = 1e-7 if share is None else share * w[0] / w[-1]
    mol = Molecule(["O"] * 2, np.array([[0.0, 0.0, 0.0], [0.0, 0.1, 2.1]]), "sto-3g")
    c = _handle(orb, aux, mol, metric_cutoff=cutoff)
    keep = w > cutoff * w[-1]
    assert c.nfit == keep.sum() == len(w) - (case == "below")
    assert c.stats()["metric_cholesky"] == chol
    B = c.matrix(N.DFKS_BFIT, (25, c.nfit)).cpu().numpy()
    c.close()
    if chol:   # C^-T: the first fitted function is the first fitting function alone
        assert np.abs(B[:, 0] - I[:, 0] / np.sqrt(V[0, 0])).max() < 1e-12 * max(1.0, np.abs(I).max())
    want = (I @ (U[:, keep] / w[keep])) @ (I @ U[:, keep]).T
    assert np.abs(B @ B.T - want).max() < 1e-9 * max(1.0, np.abs(want).max())


def test_mixed_handle_keeps_eigenvectors():
    from dftax_amd.system import Molecule
    aux, _, _ = _span("kept")
    orb = _basis([(0, 0, np.zeros(3), [0.8])], True)
    mol = Molecule(["O"] * 2, np.array([[0.0, 0.0, 0.0], [0.0, 0.1, 2.1]]), "sto-3g")
    c = _handle(orb, aux, mol, precision="mixed")
    assert c.nfit == c.naux and c.stats()["metric_cholesky"] == 0
    c.close()


@pytest.mark.parametrize("spec", [{}, {"precision": "mixed"}])
def test_factor_on_the_calling_thread(spec, monkeypatch):
    """With a profiler tool named in the environment the metric's factor runs on the calling thread: the same B."""
    import torch
    from dftax_amd import _native as N
    from dftax_amd.system import Molecule
    torch.cuda.init()   # the tool's name is read when the runtime starts: from here on the build alone sees it
    torch.zeros(1, device="cuda")
    aux, _, _ = _span("kept")
    orb = _basis([(0, 0, np.zeros(3) + x, [0.8]) for x in (0.0, 1.0)], True)
    mol = Molecule(["O"] * 2, np.array([[0.0, 0.0, 0.0], [0.0, 0.1, 2.1]]), "sto-3g")
    got = []
    for tool in (None, "none.so"):
        if tool:
            monkeypatch.setenv("ROCP_TOOL_LIBRARIES", tool)
        c = _handle(orb, aux, mol, **spec)
        assert c.nfit == c.naux and c.stats()["metric_cholesky"] == (not spec)
        got.append(c.matrix(N.DFKS_BFIT, (4, c.nfit)).clone())
        c.close()
    assert torch.equal(*got)
