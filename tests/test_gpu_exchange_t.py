"""The FP64 exchange product by the tile as wide as the factor (gemm="mfma8d") and the reduction
of K's partials, against rocBLAS: factor widths around the 16-column groups and the 160-column
tile, an odd number of rows, and a fitted set shorter than a row tile."""
from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu

# the repository's bound for kernel against rocBLAS Fock matrices (the same FP64 terms in another order)
TOL = 1e-11


@pytest.fixture(scope="module")
def pairs():
    from dftax_amd import KS, Molecule, WATER, becke, df, hip, water_cluster
    mols = {"c2h": Molecule.from_xyz("C 0 0 0; C 0 0 1.2; H 0 0 2.27", "def2-svp", charge=-1, spherical=True),
            "water": Molecule.from_xyz(WATER, "def2-svp", spherical=True),
            "water4": water_cluster((2, 2, 1), seed=1, basis="def2-tzvp")}
    return {n: [KS(m, "PBE0", grid=becke(15, 50), coulomb=df(engine=hip(gemm=g))) for g in ("mfma8d", "rocblas")]
            for n, m in mols.items()}


@pytest.mark.parametrize("name,nf", [("c2h", 1), ("c2h", 16), ("c2h", 33), ("water", 5), ("water", 17), ("water4", 31),
                                     ("water4", 64), ("water4", 65), ("water4", 112), ("water4", 160),
                                     ("water4", 161)])
def test_factor_widths(pairs, name, nf):
    import torch
    got = []
    for k in pairs[name]:
        g = torch.Generator(device=k.device).manual_seed(nf)
        Cf = torch.randn((k.nao, nf), dtype=torch.float64, device=k.device, generator=g) * (0.5 / nf ** 0.5)
        got.append(k.coulomb.energy_fock_factored(Cf))
    for a, b in zip(*got):
        assert float((a - b).abs().max()) < TOL * max(1.0, float(b.abs().max()))


@pytest.mark.parametrize("nao,naux,nf", [(1, 3, 1), (63, 5, 3), (64, 16, 8), (65, 17, 1), (128, 7, 1), (129, 40, 33),
                                         (200, 130, 9)])
def test_exchange_k_tiles(nao, naux, nf):
    """K = T T^T on tiles of 64 functions and groups of 8 k: sizes on either side of both, rows that start on odd
    words, fewer k than splits."""
    import numpy as np
    import torch
    from dftax_amd.ks import HipDFKS, HipSpec
    from dftax_amd.system import Molecule
    from dftax_amd.xc import PBE0
    from test_gpu_eri_pair import _basis
    rng = np.random.default_rng(nao)
    mol = Molecule(["O"] * 2, np.array([[0.0, 0.0, 0.0], [0.0, 0.1, 2.1]]), "sto-3g")
    site = 1.6 * np.indices((6, 6, 6)).reshape(3, -1).T + rng.uniform(-0.1, 0.1, (216, 3))
    orb = _basis([(0, 0, x, [1.1]) for x in site[:nao]], True)
    aux = _basis([(0, 0, x, [0.9]) for x in site[:naux]], True)
    got = []
    for gemm in ("mfma8d", "rocblas"):
        c = HipDFKS(orb, aux, mol, np.zeros((1, 3)) + 5.0, np.ones(1), PBE0(), 2, HipSpec(gemm=gemm), chunk=None)
        g = torch.Generator(device=c.device).manual_seed(nf)
        Cf = torch.randn((c.nao, nf), dtype=torch.float64, device=c.device, generator=g) * (0.5 / nf ** 0.5)
        got.append(c.energy_fock_factored(Cf))
    for a, b in zip(*got):
        assert float((a - b).abs().max()) < TOL * max(1.0, float(b.abs().max()))
