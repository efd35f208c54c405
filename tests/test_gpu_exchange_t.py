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


@pytest.mark.parametrize("N", [3, 40, 80, 81, 150])
@pytest.mark.parametrize("K", [1, 15, 16, 18, 37])
def test_infinities_in_the_last_group_of_t(N, K):
    """One infinite element at the last k of either operand of T = A B^T reaches its row or column as an infinity, on
    whole and partial tiles of rows and on both sides of the groups of 16 (k past the end is zero in both operands)."""
    import ctypes
    import torch
    from dftax_amd import _native

    class Gemm(ctypes.Structure):
        _fields_ = [("M", ctypes.c_int), ("N", ctypes.c_int), ("K", ctypes.c_int64), ("A", ctypes.c_void_p),
                    ("lda", ctypes.c_int64), ("a_kcontig", ctypes.c_bool), ("B", ctypes.c_void_p),
                    ("ldb", ctypes.c_int64), ("b_kcontig", ctypes.c_bool)]

    class RowDot(ctypes.Structure):   # no row terms: out = null
        _fields_ = [("cf", ctypes.c_void_p), ("sg", ctypes.c_void_p), ("nao", ctypes.c_int), ("nq", ctypes.c_int),
                    ("out", ctypes.c_void_p)]

    f = _native.lib()["_ZN4dfks15launch_gemm_t64ERKNS_8GemmArgsEPdRKNS_6RowDotEP12ihipStream_t"]
    f.restype = ctypes.c_int
    f.argtypes = [ctypes.POINTER(Gemm), ctypes.c_void_p, ctypes.POINTER(RowDot), ctypes.c_void_p]
    M = 261   # one whole tile of rows, of 256 or 128, and a partial one
    g = torch.Generator().manual_seed(K)
    for at in ((0, 0), (258, N - 1)):
        for which in ("a", "b"):
            A = torch.rand((M, K), dtype=torch.float64, generator=g) + 0.5
            B = torch.rand((N, K), dtype=torch.float64, generator=g) + 0.5
            (A[at[0]] if which == "a" else B[at[1]])[K - 1] = float("inf")
            want = A @ B.T
            a, b = A.T.contiguous().cuda(), B.cuda()
            c = torch.empty((M, N), dtype=torch.float64, device="cuda")
            assert f(Gemm(M, N, K, a.data_ptr(), M, False, b.data_ptr(), K, True), c.data_ptr(),
                     RowDot(None, None, 0, 1, None),
                     torch.cuda.current_stream().cuda_stream) == 0
            got = c.cpu()
            assert torch.equal(got.isinf(), want.isinf()) and not got.isnan().any()
            # sums of K terms under 2.25
            assert (got - want)[want.isfinite()].abs().max() < 1e-14 * K
