"""The SCF step's products by 32 x 32 tiles (X^T F X, the orbital gradient, P = C C^T) against rocBLAS (gemm="rocblas"):
converged solutions on either side of the tiles and of the groups of 8 functions."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["h2", "h2_svp", "water", "c2h", "water_svp", "water2", "water3_tzvp"])
def test_converged_solutions(name):
    from dftax_amd import KS, Molecule, WATER, becke, df, hip, scf, water_cluster
    mol = {"h2": lambda: Molecule.from_xyz("H 0 0 0; H 0.74 0 0", "sto-3g", spherical=True),          # 2 functions
           "h2_svp": lambda: Molecule.from_xyz("H 0 0 0; H 0.74 0 0", "def2-svp", spherical=True),    # 10
           "water": lambda: Molecule.from_xyz(WATER, "sto-3g", spherical=True),                       # 7
           "c2h": lambda: Molecule.from_xyz("C 0 0 0; C 0 0 1.2; H 0 0 2.27", "def2-svp", charge=-1, spherical=True),
           "water_svp": lambda: Molecule.from_xyz(WATER, "def2-svp", spherical=True),                 # 24
           "water2": lambda: water_cluster((2, 1, 1), seed=1, basis="def2-tzvp"),                     # 86
           "water3_tzvp": lambda: water_cluster((3, 1, 1), seed=2, basis="def2-tzvp")}[name]()        # 129
    got = [scf(KS(mol, "PBE0", grid=becke(20, 50), coulomb=df(engine=hip(gemm=g))), e_tol=1e-11, d_tol=1e-9)
           for g in ("auto", "rocblas")]
    assert all(r.converged for r in got)
    # the two converge to the same solution within the SCF's thresholds
    assert abs(got[0].e_tot - got[1].e_tot) < 1e-9
    assert float((got[0].P - got[1].P).abs().max()) < 1e-6
