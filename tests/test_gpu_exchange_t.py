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
