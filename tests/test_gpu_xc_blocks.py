"""FP64 XC on the compact grid: the one-launch block kernels against the per-bin rocBLAS
products, from blocks of one 32-column strip to several strips with a half one at the end."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# the bound of the repository's kernel-against-rocBLAS Fock checks: both sum the same FP64 terms
# (values up to ~20) in another order
TOL = 1e-11


def _mol(name):
    from dftax_amd import Molecule, WATER, tree_molecule, water_cluster
    if name == "h":
        return Molecule.from_xyz("H 0 0 0; H 0.74 0 0", "def2-svp", spherical=True)
    if name == "water":
        return Molecule.from_xyz(WATER, "def2-tzvp", spherical=True)
    if name == "water_cart":
        return Molecule.from_xyz(WATER, "sto-3g")
    if name == "tree":
        return tree_molecule(5, np.random.default_rng(5))
    return water_cluster((3, 1, 1), seed=2, basis="def2-tzvp")


@pytest.mark.parametrize("name,xc", [("h", "PBE"), ("water", "B3LYP"), ("water_cart", "PBE0"), ("tree", "PBE0"),
                                     ("water3", "B3LYP")])
def test_energy_and_response(name, xc):
    import torch
    from dftax_amd import KS, becke, df, hip
    from dftax_amd.scf import initial_density
    mol, grid = _mol(name), becke(30, 110)
    got = []
    for gemm in ("auto", "rocblas"):
        k = KS(mol, xc, grid=grid, coulomb=df(engine=hip(gemm=gemm)))
        P = initial_density(k, None)
        E, F = k.coulomb.energy_fock(P)
        g = torch.Generator(device=P.device).manual_seed(1)
        U, V = (torch.randn((k.nao, 2), dtype=torch.float64, device=P.device, generator=g) * 0.1 for _ in range(2))
        k.coulomb.response_begin(P)
        got.append((E, F, k.coulomb.response_fock(U, V)))
    for a, b in zip(*got):
        assert float((a - b).abs().max()) < TOL * max(1.0, float(b.abs().max()))


@pytest.mark.parametrize("spin,charge,name", [(1, 1, "tree"), (2, 0, "water")])
def test_spin_polarised(spin, charge, name):
    from dftax_amd import KS, Molecule, becke, df, hip
    from dftax_amd.scf import initial_density
    m = _mol(name)
    mol = Molecule(m.symbols, m.coords, m.basis, charge=charge, spin=spin, spherical=True)
    got = []
    for gemm in ("auto", "rocblas"):
        k = KS(mol, "B3LYP", grid=becke(30, 110), coulomb=df(engine=hip(gemm=gemm)))
        got.append(k.coulomb.energy_fock(initial_density(k, None)))
    for a, b in zip(*got):
        assert float((a - b).abs().max()) < TOL * max(1.0, float(b.abs().max()))


def test_what_is_not_finite_stays_with_its_blocks():
    """NaN in P[0][0] masks the points that function 0 reaches and no others: the columns that fill up a block to 32 are
    zero whatever P holds."""
    import ctypes
    import torch
    from dftax_amd import KS, _native, becke, df, hip, water_cluster
    from dftax_amd.scf import initial_density
    mol = water_cluster((3, 1, 1), seed=2, basis="def2-svp")
    got = []
    for gemm in ("auto", "rocblas"):
        k = KS(mol, "PBE", grid=becke(30, 110), coulomb=df(engine=hip(gemm=gemm)))
        c, P = k.coulomb, initial_density(k, None).contiguous().clone()
        P[0, 0] = float("nan")
        cm, signs = torch.zeros((1, c.nao), dtype=torch.float64, device=P.device), (ctypes.c_double * 1)(1.0)
        F = torch.empty_like(P)
        _native.check(c.L.dfks_energy_fock_factored(c.handle, ctypes.c_void_p(P.data_ptr()),
                                                    ctypes.c_void_p(cm.data_ptr()), signs, 1,
                                                    ctypes.c_void_p(c._E.data_ptr()), ctypes.c_void_p(F.data_ptr()),
                                                    c._stream()))
        got.append((float(c._E[4]), F.clone()))
    (a, Fa), (b, Fb) = got
    assert b < -1.0 and abs(a - b) < TOL * abs(b)
    assert float((Fa - Fb).abs().max()) < TOL * max(1.0, float(Fb.abs().max()))
