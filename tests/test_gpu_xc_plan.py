"""The compact grid's plan (Morton sort, shells of each block, lists) on point sets around its tiles of 2048, blocks of
128 and wavefronts of 64 points: the XC term on blocks against the dense grid."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# the bound of the repository's kernel-against-kernel Fock checks, per unit of summed weight: the blocks leave out
# shells under 1e-14
TOL = 1e-11


@pytest.mark.parametrize("npts,shape", [(1, "cloud"), (63, "cloud"), (129, "cloud"), (2047, "cloud"), (2048, "plane"),
                                        (2049, "repeated"), (6000, "cloud"), (70000, "cloud")])
def test_plan_against_dense_grid(npts, shape):
    import torch
    from dftax_amd.basis import build_basis
    from dftax_amd.ks import HipDFKS, HipSpec
    from dftax_amd.system import Molecule
    from dftax_amd.xc import PBE0
    rng = np.random.default_rng(npts)
    xyz = np.array([[0.0, 0.0, 0.0], [1.4, 1.1, 0.0], [-1.4, 1.1, 0.1]])
    xyz = np.concatenate([xyz, xyz + [9.0, -3.0, 4.0], xyz[:, ::-1] + [25.0, 6.0, -2.0]])   # blocks of unequal width
    mol = Molecule(["O", "H", "H"] * 3, xyz, "def2-svp", spherical=True)
    pts = xyz[rng.integers(0, 9, npts)] + rng.normal(0.0, 1.5, (npts, 3))
    if shape == "plane":
        pts[:, 2] = 0.25
    if shape == "repeated":
        pts[npts // 2:] = pts[:npts - npts // 2]
    w = rng.uniform(0.0, 2.0 / npts, npts)
    orb, aux = (build_basis(mol.symbols, mol.coords, b, spherical=True) for b in ("def2-svp", "even-tempered-jk"))
    got = []
    for grid in ("blocks", "dense"):
        c = HipDFKS(orb, aux, mol, pts, w, PBE0(), 30, HipSpec(xc_grid=grid), chunk=None)
        g = torch.Generator(device=c.device).manual_seed(npts)
        Cf = torch.randn((c.nao, 15), dtype=torch.float64, device=c.device, generator=g) * 0.3
        got.append(c.energy_fock_factored(Cf))
    for a, b in zip(*got):
        assert float((a - b).abs().max()) < TOL * max(1.0, float(b.abs().max()))
