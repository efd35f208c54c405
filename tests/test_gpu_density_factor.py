"""The factor of a density matrix behind energy_fock(P): ranks around the panel width, indefinite and
unsymmetric-to-rounding P, zero, and the row counts per thread, against the same Fock matrix from a
known factor or from the fitted tensor."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# kernel-against-kernel bound of the repository's Fock checks (relative to the largest element); the factor
# stops at 1e-14 of the largest diagonal element
TOL = 1e-11


def _handle(n_water, basis, zero_grid=True):
    """A Coulomb + exchange engine: one grid point of zero weight, so that F is linear in P."""
    from dftax_amd import water_cluster
    from dftax_amd.basis import build_basis
    from dftax_amd.ks import HipDFKS, HipSpec
    from dftax_amd.xc import PBE0
    m = water_cluster((n_water, 1, 1), seed=3, basis=basis)
    return HipDFKS(build_basis(m.symbols, m.coords, basis, spherical=True),
                   build_basis(m.symbols, m.coords, "even-tempered-jk", spherical=True), m,
                   np.zeros((1, 3)) + 1.0, np.zeros(1), PBE0(), m.nelectron, HipSpec(), chunk=None)


def _factor(c, nf, seed):
    import torch
    g = torch.Generator(device=c.device).manual_seed(seed)
    return torch.randn((c.nao, nf), dtype=torch.float64, device=c.device, generator=g) / max(nf, 1) ** 0.5


def _close(a, b):
    assert float((a - b).abs().max()) < TOL * max(1.0, float(b.abs().max()))


@pytest.mark.parametrize("n_water,basis,ranks", [(1, "def2-svp", (1, 2, 23, 24)),
                                                 (2, "def2-tzvp", (31, 32, 33, 64, 86)),
                                                 (12, "def2-tzvp", (60, 97)), (24, "def2-tzvp", (120, 128))])
def test_semidefinite(n_water, basis, ranks):
    c = _handle(n_water, basis)
    for r in ranks:
        E0, F0, P = c.energy_fock_factored(_factor(c, r, r))
        E, F = c.energy_fock(P)
        _close(F, F0)
        _close(E, E0)
    c.close()


@pytest.mark.parametrize("kind", ["indefinite", "zero_diagonal", "slightly_negative", "zero", "negative"])
def test_general(kind):
    import torch
    from dftax_amd import _native as N
    c = _handle(2, "def2-tzvp")
    n = c.nao
    A, D = _factor(c, 9, 1), _factor(c, 5, 2)
    P = {"indefinite": A @ A.T - D @ D.T, "negative": -(A @ A.T), "zero": torch.zeros_like(A @ A.T),
         "slightly_negative": A @ A.T - 1e-9 * (D @ D.T),
         "zero_diagonal": (lambda X: X - torch.diag(torch.diag(X)))(A @ A.T)}[kind]
    P = (0.5 * (P + P.T)).contiguous()
    E, F = c.energy_fock(P)
    B = c.matrix(N.DFKS_BFIT, (n, n, c.nfit))
    H = c.matrix(N.DFKS_HCORE, (n, n))
    gamma = torch.einsum("mnq,mn->q", B, P)
    J = B @ gamma
    X = (P @ B.reshape(n, n * c.nfit)).reshape(n, n, c.nfit)
    K = torch.zeros_like(P)
    for l in range(n):
        K += B[:, l] @ X[l].T
    _close(F, H + J - 0.125 * K)
    c.close()


@pytest.mark.parametrize("kind,size", [("antisymmetric", 1e-16), ("antisymmetric", 1e-13), ("antisymmetric", 1e-6),
                                       ("negative", 1e-15), ("negative", 1e-13), ("negative", 1e-12)])
def test_about_the_residual_limit(kind, size):
    """Parts that the residual limit (8e-14 of the largest diagonal element) lets pass as rounding and parts that it does
    not: an antisymmetric one, which J of a symmetric tensor and the symmetrised K do not see, and a negative one. What
    is dropped is at most its size times the largest integral sums, within the bound for a unit density."""
    import torch
    from dftax_amd import _native as N
    c = _handle(2, "def2-tzvp")
    n = c.nao
    A, D = _factor(c, 9, 1), _factor(c, 5, 2)
    S = A @ A.T
    R = D @ D.T if kind == "negative" else D @ A[:, :5].T - A[:, :5] @ D.T
    P = (S - size * float(S.diag().max()) * R / float(R.abs().max())).contiguous()
    E, F = c.energy_fock(P)
    P = 0.5 * (P + P.T)
    B = c.matrix(N.DFKS_BFIT, (n, n, c.nfit))
    H = c.matrix(N.DFKS_HCORE, (n, n))
    J = B @ torch.einsum("mnq,mn->q", B, P)
    X = (P @ B.reshape(n, n * c.nfit)).reshape(n, n, c.nfit)
    K = torch.zeros_like(P)
    for l in range(n):
        K += B[:, l] @ X[l].T
    want = H + J - 0.125 * K
    c.close()
    # an antisymmetric part beyond rounding goes to the eigenvectors of one triangle, whose own symmetric part it is
    slack = 0.0 if kind == "negative" or size < 1e-7 else 1e3 * size
    assert float((F - want).abs().max()) < (TOL + slack) * max(1.0, float(want.abs().max()))
