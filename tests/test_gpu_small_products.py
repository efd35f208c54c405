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


@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True)])
@pytest.mark.parametrize("K", [1, 5, 8, 13, 66])
def test_infinities_in_the_last_group(ta, tb, K):
    """One infinite element at the last k of either operand reaches its row or column as an infinity, on both sides of
    the groups of 8 and of the tiles (k past the end is zero in both operands)."""
    import ctypes
    import torch
    from dftax_amd import _native
    f = _native.lib()["_ZN4dfks17launch_gemm_smallEbbiiidPKdlS1_ldPdlP12ihipStream_t"]
    f.restype, P, L = ctypes.c_int, ctypes.c_void_p, ctypes.c_int64
    f.argtypes = [ctypes.c_bool] * 2 + [ctypes.c_int] * 3 + [ctypes.c_double, P, L, P, L, ctypes.c_double, P, L, P]
    M, N = 33, 35
    g = torch.Generator().manual_seed(K)
    for which in ("a", "b"):
        A = torch.rand((M, K), dtype=torch.float64, generator=g) + 0.5
        B = torch.rand((K, N), dtype=torch.float64, generator=g) + 0.5
        (A if which == "a" else B)[(32, K - 1) if which == "a" else (K - 1, 34)] = float("-inf")
        want = A @ B
        # column-major operands and result
        a = (A if ta else A.T).contiguous().cuda()
        b = (B if tb else B.T).contiguous().cuda()
        c = torch.empty((N, M), dtype=torch.float64, device="cuda")
        assert f(ta, tb, M, N, K, 1.0, a.data_ptr(), a.shape[1], b.data_ptr(), b.shape[1], 0.0, c.data_ptr(), M,
                 torch.cuda.current_stream().cuda_stream) == 0
        got = c.T.cpu()
        assert torch.equal(got.isinf(), want.isinf()) and not got.isnan().any()
        # sums of K terms under 2.25
        assert (got - want)[want.isfinite()].abs().max() < 1e-14 * K
