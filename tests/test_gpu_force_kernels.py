"""One-electron integrals by shell pair, Becke weights, and the gradient's kernels where the shipped force
vectors do not reach: nuclei, points and auxiliary shells around groups of 16, contractions, g spans,
cartesian spans, and molecules on both sides of what the LDS of the Becke kernels holds."""
from types import SimpleNamespace

import numpy as np
import pytest

from test_gpu_eri_pair import TOL_INT, _basis

pytestmark = pytest.mark.gpu

PARTS = ("nuclear", "one_electron", "coulomb", "exchange", "xc")
# the oracle's extrapolated differences carry ~3e-8 (tests/golden/make_forces.py): the repository's bound
TOL_FORCE = 2e-7


@pytest.mark.parametrize("natom,nprim,spherical", [(1, 1, True), (15, 2, True), (16, 3, False), (17, 1, True),
                                                   (33, 7, True), (4, 2, False)])
def test_int1e_by_pair(natom, nprim, spherical):
    from dftax_amd import _native as N
    from dftax_amd.ks import HipDFKS, HipSpec
    from dftax_amd.system import Molecule
    from dftax_amd.xc import PBE0
    from oracle import ref
    rng = np.random.default_rng(natom + 100 * nprim)
    xyz = rng.uniform(-3.0, 3.0, (natom, 3))
    mol = Molecule(["C" if i % 3 == 0 else "O" for i in range(natom)], xyz, "sto-3g")
    at = (0, natom - 1)
    orb = _basis([(l, a, xyz[a], list(0.3 * 2.1 ** np.arange(nprim) * (1 + 0.1 * l + 0.05 * k)))
                  for k, a in enumerate(at) for l in (3, 0, 2, 1)], spherical)
    aux = _basis([(0, 0, xyz[0], [0.7])], True)
    c = HipDFKS(orb, aux, mol, np.zeros((1, 3)) + 5.0, np.ones(1), PBE0(), 2, HipSpec(), chunk=None)
    got = [c.matrix(k, (c.nao, c.nao)).cpu().numpy() for k in (N.DFKS_S, N.DFKS_KINETIC, N.DFKS_NUCLEAR)]
    z = np.array([6.0 if s == "C" else 8.0 for s in mol.symbols])
    for g, want in zip(got, ref.int1e(orb, xyz, z)):
        # natom charges of up to 8 on the sums of normalised functions: the bound of one, per unit of scale
        assert np.abs(g - want).max() < TOL_INT * max(1.0, np.abs(want).max())
    c.close()


@pytest.mark.parametrize("spherical", [True, False])
def test_overlap_with_g_shells(spherical):
    from dftax_amd import _native as N
    from oracle import ref
    b = _basis([(l, 0, np.array(x), [0.4 + 0.2 * l, 1.7]) for x in ([0.0, 0.1, 0.2], [1.1, -0.7, 0.4])
                for l in (4, 2, 0, 3, 1)], spherical)
    S = N.overlap(b)
    want = ref.int1e(b, np.zeros((1, 3)), np.zeros(1))[0]
    assert np.abs(S - want).max() < TOL_INT * max(1.0, np.abs(want).max())


def _molecule(name):
    from dftax_amd.system import Molecule
    if name == "water_cartesian":
        return Molecule.from_xyz("O 0.0 0.0 0.0; H 0.80 0.62 0.05; H -0.70 0.55 -0.08", "def2-svp", spherical=False)
    rng = np.random.default_rng(7)
    n = 18
    xyz = np.array([[3.2 * (i // 2 % 3) + 0.76 * (i % 2), 3.2 * (i // 6), 0.3 * (i // 2 % 2)] for i in range(n)])
    return Molecule(["H"] * n, (xyz + rng.uniform(-0.05, 0.05, xyz.shape)) / 0.529177210903, "sto-3g", spherical=True)


@pytest.mark.parametrize("name,atoms", [("h18", (17,)), ("water_cartesian", (0, 2))])
def test_gradient_terms(name, atoms):
    import torch
    from dftax_amd import KS, becke, df, hip
    from dftax_amd.forces import gradient_parts
    from oracle import ref
    mol = _molecule(name)
    grid = becke(20, 50) if name == "h18" else becke(40, 110)
    oks = ref.OracleKS(mol, "PBE0", grid=grid)
    X = np.linalg.inv(np.linalg.cholesky(oks.S)).T
    Z = X @ np.linalg.eigh(X.T @ oks.hcore @ X)[1][:, :oks.nocc]
    F1, P1 = ref.fd_forces(mol, "PBE0", Z, grid, h=4e-3, atoms=atoms, parts=True)
    F2, P2 = ref.fd_forces(mol, "PBE0", Z, grid, h=8e-3, atoms=atoms, parts=True)
    want = -(4 * P1 - P2) / 3
    ks = KS(mol, "PBE0", grid=grid, coulomb=df(chunk=None, engine=hip()))
    parts = gradient_parts(ks, SimpleNamespace(mo_coeff=torch.tensor(Z, device="cuda")), grid)
    for k, part in enumerate(PARTS):
        err = np.abs(parts[part] - want[k])[list(atoms)].max()
        print(f"  {part:13s} max |d| {err:.2e} of {np.abs(want[k]).max():.2e}", flush=True)
        assert err < TOL_FORCE, part
    assert np.abs(sum(parts.values()).sum(0)).max() < 1e-8


@pytest.mark.parametrize("natom,npts", [(1, 1), (2, 15), (5, 17), (128, 65), (129, 63), (513, 33)])
def test_becke_weights_edges(natom, npts):
    from dftax_amd import _native as N
    from oracle import ref
    rng = np.random.default_rng(natom)
    side = int(np.ceil(natom ** (1 / 3)))
    xyz = 2.5 * np.indices((side,) * 3).reshape(3, -1).T[:natom] + rng.uniform(-0.5, 0.5, (natom, 3))
    bragg = rng.choice([0.66140414, 1.32280829, 1.13383567], natom)
    own = rng.integers(0, natom, npts).astype(np.int32)
    pts = xyz[own] + rng.normal(0.0, 1.0, (npts, 3))
    raw = rng.uniform(0.1, 2.0, npts)
    P = ref.becke_partition(pts, xyz, bragg)
    want = raw * P[np.arange(npts), own] / P.sum(1)
    got = N.becke_weights(pts, raw, own, xyz, bragg)
    # about 10 natom roundings in each product of cell functions
    assert np.abs(got - want).max() < 20 * max(natom, 8) * 2.3e-16 * raw.max()


@pytest.mark.parametrize("far", [44, 46, 218])
def test_xc_gradient_with_far_atoms(far):
    """H2 molecules hundreds of Bohr away change nothing near a cluster: 62 and 64 atoms (four wavefronts and one
    in the Becke gradient's LDS) and 236 (distances not kept) against the cluster's 18 alone."""
    import torch
    from dftax_amd import KS, becke, df, hip
    from dftax_amd.forces import gradient_parts
    from dftax_amd.system import Molecule
    grid = becke(12, 26)
    near = _molecule("h18")
    rng = np.random.default_rng(3)
    Z0 = np.linalg.qr(rng.normal(size=(18, 9)))[0]

    def xc_grad(mol, extra):
        ks = KS(mol, "PBE0", grid=grid, coulomb=df(chunk=None, engine=hip()))
        Z = np.zeros((18 + extra, 9 + extra // 2))
        Z[:18, :9] = Z0
        for k in range(extra // 2):
            Z[18 + 2 * k:20 + 2 * k, 9 + k] = 0.55
        return gradient_parts(ks, SimpleNamespace(mo_coeff=torch.tensor(Z, device="cuda")), grid)["xc"]

    base = xc_grad(near, 0)
    k = np.arange(far)
    xyz = np.stack([300.0 + 60.0 * (k // 2) + 1.4 * (k % 2), 0 * k, 0 * k], 1)
    both = Molecule(["H"] * (18 + far), np.concatenate([near.coords, xyz]), "sto-3g", spherical=True)
    err = np.abs(xc_grad(both, far)[:18] - base).max()
    print(f"  {far} far atoms: max |d| {err:.2e} of {np.abs(base).max():.2e}", flush=True)
    assert err < TOL_FORCE
