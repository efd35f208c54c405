"""Device memory that the library keeps between handles.

Buffers of 8 MiB and more are kept after a handle frees them and are handed to
the next handle that asks for the same size class (its stream first waits on
an event recorded where the block was freed).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SLACK = 1 << 30  # rocBLAS workspace, small pool blocks, torch's cached tensors


def _say(msg):
    print(msg, flush=True)


def test_kept_buffers_are_reused_and_counted(water_dimer_tzvp):
    """Two builds of the same molecule in a row: the second takes the first's
    kept buffers (with their old contents) and must give the same Fock matrix
    and energy. The memory the library reports it can obtain, which sizes the
    DF chunks and the serving budget, counts the kept buffers, so it returns to
    where it was once the handles are gone, although the device counts them as
    in use. After dfks_release_memory the device reports that memory free."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from dftax_amd import KS, _native, becke, df, hip
    from oracle import ref
    _say("case: water dimer def2-TZVP B3LYP, becke(35,110), built twice")
    torch.cuda.synchronize()
    before = _native.device_free(0)
    dev_before, _ = torch.cuda.mem_get_info(0)
    assert before >= dev_before - (64 << 20)
    g = becke(35, 110)
    out = []
    for _ in range(2):
        ks = KS(water_dimer_tzvp, "B3LYP", grid=g, coulomb=df(engine=hip(gemm="rocblas")))
        P0 = ref.minao_density(ks.mol, ks.basis)
        S = ks.S.cpu().numpy()
        P0 = torch.tensor(P0 * (ks.mol.nelectron / np.sum(P0 * S)), device="cuda")
        E, F = ks.coulomb.energy_fock(P0)
        torch.cuda.synchronize()
        out.append((E.cpu().numpy().copy(), F.cpu().numpy().copy()))
        ks.coulomb.close()
        del ks, E, F, P0
    torch.cuda.synchronize()
    after = _native.device_free(0)
    dev_after, _ = torch.cuda.mem_get_info(0)
    dF = np.abs(out[1][1] - out[0][1]).max()
    dE = np.abs(out[1][0] - out[0][0]).max()
    _say(f"library free {before / 1e9:.3f} -> {after / 1e9:.3f} GB, device free {dev_before / 1e9:.3f} -> "
         f"{dev_after / 1e9:.3f} GB; second build max|dF| {dF:.2e}, max|dE| {dE:.2e}")
    assert dF < 1e-12 and dE < 1e-10
    assert after >= before - SLACK
    assert after >= dev_after
    # released: the device itself reports the memory free again
    _native.release_memory(0)
    dev_released, _ = torch.cuda.mem_get_info(0)
    _say(f"after dfks_release_memory: device free {dev_released / 1e9:.3f} GB")
    assert dev_released >= after - SLACK


def test_mixed_build_takes_no_cholesky_work():
    """A handle with 32-bit products takes the metric's eigenvectors: its build holds (P|Q), the factor and the
    eigenvectors, whose buffer the factor's padded copy takes over, and none of the 5 naux^2 words of the Cholesky
    factor and its work. Every buffer that a build
    took stays with the library afterwards, so what the device counts as used is their sum (rocSOLVER's workspace, which
    stays with its handle, is in place before)."""
    import torch
    from dftax_amd import _native
    from dftax_amd.ks import HipDFKS, HipSpec
    from dftax_amd.system import Molecule
    from dftax_amd.xc import PBE0
    from test_gpu_eri_pair import _basis
    naux = 2048
    site = 1.6 * np.indices((13, 13, 13)).reshape(3, -1).T[:naux] + 0.0
    aux = _basis([(0, 0, x, [0.9]) for x in site], True)
    orb = _basis([(0, 0, x, [0.8]) for x in site[:2]], True)
    mol = Molecule(["O"] * 2, np.array([[0.0, 0.0, 0.0], [0.0, 0.1, 2.1]]), "sto-3g")

    def build():
        HipDFKS(orb, aux, mol, np.zeros((1, 3)) + 5.0, np.ones(1), PBE0(), 2, HipSpec(precision="mixed"),
                chunk=None).close()
        torch.cuda.synchronize()

    build()
    _native.release_memory(0)
    before, _ = torch.cuda.mem_get_info(0)
    build()
    after, _ = torch.cuda.mem_get_info(0)
    _say(f"taken by a build of {naux} fitting functions: {(before - after) / (8 * naux * naux):.2f} naux^2 words")
    assert 2 * 8 * naux * naux < before - after < 6 * 8 * naux * naux


def test_fresh_blocks_leave_room_for_the_runtime():
    """With 10.5 GB of the device free and more than that kept, a build that needs some 3.5 GB of fresh blocks gives kept
    ones back: 8 GiB stay free for what the runtime itself allocates (a queue's scratch, which ends the process when
    there is no room for it)."""
    import torch
    from dftax_amd import _native, water_cluster
    from dftax_amd.basis import build_basis
    from dftax_amd.ks import HipDFKS, HipSpec
    from dftax_amd.xc import PBE0

    def handle(n):
        m = water_cluster((n, 1, 1), seed=1, basis="def2-tzvp")
        return HipDFKS(*(build_basis(m.symbols, m.coords, b, spherical=True) for b in ("def2-tzvp", "even-tempered-jk")),
                       m, np.zeros((1, 3)) + 1.0, np.zeros(1), PBE0(), m.nelectron, HipSpec(), chunk=None)

    _native.release_memory(0)
    handle(24).close()
    torch.cuda.synchronize()
    free, _ = torch.cuda.mem_get_info(0)
    kept = _native.device_free(0) - free
    _say(f"kept {kept / 1e9:.1f} GB, device free {free / 1e9:.1f} GB")
    assert kept > 20e9
    fill = torch.empty(free - int(10.5e9), dtype=torch.uint8, device="cuda")
    try:
        c = handle(12)
        C = torch.eye(c.nao, 60, dtype=torch.float64, device="cuda")
        E, F, _ = c.energy_fock_factored(C)
        left, _ = torch.cuda.mem_get_info(0)
        _say(f"device free beside the second handle {left / 1e9:.1f} GB")
        assert bool(torch.isfinite(F).all())
        assert left > (8 << 30) - (256 << 20)   # blocks under 8 MiB come on top
        c.close()
    finally:
        del fill
        torch.cuda.empty_cache()
        _native.release_memory(0)
