"""The workloads that this framework's speed is measured on.

A case is one call (or one whole solve) as a user's program makes it, through the
public entry points, on one GPU. The listed cases cover what the framework is used
for: Fock builds of every kind from one water molecule to (H2O)_24 in def2-TZVP,
whole SCF solves in both precisions, requests of the serving loop, the build of a
molecule's integrals, the response products of the Newton solver and nuclear forces.
``draw`` gives further cases of the same kinds over the same ranges.

Molecules are the two generators of ``dftax_amd.system``: water clusters
(``molecule="water"``, size = number of molecules, def2-TZVP unless the case says
otherwise) and saturated C/N/O trees (``"tree"``, size = heavy atoms, def2-SVP).
Every seed is another geometry: the clusters are drawn anew, the trees (one molecule
a size) have their atoms displaced as a step of a geometry optimisation does.
"""

from __future__ import annotations

import math
import warnings

import numpy as np
import torch

from dftax_amd import KS, Molecule, df, forces, hip, scf, tree_molecule, water_cluster
from dftax_amd import _native
from dftax_amd.serve import Request, Server


def listed():
    return [
        # one water molecule, smallest basis: a Fock build is a chain of short launches
        {"name": "fock_water1_svp", "kind": "fock", "molecule": "water", "size": 1, "basis": "def2-svp", "xc": "PBE0"},
        # the largest resident system that fits a device several times: one Newton or property
        # step's Fock build from orbitals; the exchange products, J and the XC grid at full size
        {"name": "fock_water24_tzvp", "kind": "fock_orbitals", "molecule": "water", "size": 24, "basis": "def2-tzvp",
         "xc": "PBE0"},
        # a range-separated hybrid on an organic molecule: two fitted tensors, two exchange products
        {"name": "fock_tree10_camb3lyp", "kind": "fock", "molecule": "tree", "size": 10, "basis": "def2-svp",
         "xc": "CAM-B3LYP"},
        # a radical cation, spin-unrestricted: two densities, the spin-polarised functional
        {"name": "fock_tree8_uks", "kind": "fock_uks", "molecule": "tree", "size": 8, "basis": "def2-svp", "xc": "PBE0"},
        # integrals too large to keep: auxiliary slabs recomputed in the Fock build, screened bra pairs
        {"name": "fock_water12_recompute", "kind": "fock_recompute", "molecule": "water", "size": 12,
         "basis": "def2-tzvp", "xc": "PBE0", "chunk": 384},
        # a whole FP64 SCF converged tightly, as before forces or properties
        {"name": "scf_water8_tzvp", "kind": "scf", "molecule": "water", "size": 8, "basis": "def2-tzvp", "xc": "PBE0"},
        # the same in mixed precision with FP64 steps at the end
        {"name": "scf_water14_mixed", "kind": "scf_mixed", "molecule": "water", "size": 14, "basis": "def2-tzvp",
         "xc": "PBE0"},
        # requests of the serving loop, a small and a large one: build, mixed SCF, FP64 refinement
        {"name": "solve_tree3", "kind": "solve", "molecule": "tree", "size": 3, "basis": "def2-svp", "xc": "B3LYP"},
        {"name": "solve_tree20", "kind": "solve", "molecule": "tree", "size": 20, "basis": "def2-svp", "xc": "B3LYP"},
        # a molecule's integrals, metric, fitted tensor and grid, before any SCF
        {"name": "build_water8_tzvp", "kind": "build", "molecule": "water", "size": 8, "basis": "def2-tzvp",
         "xc": "PBE0"},
        # one Hessian-vector product of the Newton solver's inner loop
        {"name": "response_water10_tzvp", "kind": "response", "molecule": "water", "size": 10, "basis": "def2-tzvp",
         "xc": "PBE0"},
        # nuclear forces after an SCF, as in a geometry optimisation step
        {"name": "forces_tree6_svp", "kind": "forces", "molecule": "tree", "size": 6, "basis": "def2-svp",
         "xc": "B3LYP"},
    ]


# the range of sizes of each kind: (water molecules or None, heavy atoms of a tree or None)
_RANGES = {
    "fock": ((1, 20), (2, 24)),
    "fock_orbitals": ((1, 24), (2, 24)),
    "fock_uks": ((1, 8), (2, 14)),
    "fock_recompute": ((2, 12), (8, 20)),
    "scf": ((1, 10), (2, 20)),
    "scf_mixed": ((2, 14), (4, 24)),
    "solve": (None, (2, 22)),
    "build": ((1, 10), (2, 24)),
    "response": ((1, 12), (2, 24)),
    "forces": ((1, 3), (2, 8)),
}


def draw(rng):
    kind = rng.choice(sorted(_RANGES))
    water, tree = _RANGES[kind]
    mol = rng.choice([m for m, r in (("water", water), ("tree", tree)) if r])
    lo, hi = water if mol == "water" else tree
    size = max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))
    basis = rng.choice(["def2-tzvp", "def2-tzvp", "def2-svp"]) if mol == "water" else "def2-svp"
    xcs = ["PBE0", "B3LYP"] if kind in ("solve", "scf_mixed", "fock_uks", "forces") else ["PBE0", "B3LYP", "PBE"]
    if kind == "fock":
        xcs = xcs + ["CAM-B3LYP"]
    case = {"kind": kind, "molecule": mol, "size": size, "basis": basis, "xc": rng.choice(xcs)}
    if kind == "fock_recompute":
        case["chunk"] = rng.choice([96, 150, 256, 384, 500])
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _lattice(n):
    """The most compact a x b x c with a b c = n."""
    best = (n, 1, 1)
    for a in range(1, n + 1):
        for b in range(1, a + 1):
            if n % (a * b) == 0 and n // (a * b) <= b and a + b + n // (a * b) < sum(best):
                best = (a, b, n // (a * b))
    return best


def _molecule(case, seed):
    if case["molecule"] == "water":
        mol = water_cluster(_lattice(case["size"]), seed=seed, basis=case["basis"])
    else:
        mol = tree_molecule(case["size"], np.random.default_rng(case["size"]), basis=case["basis"])
        xyz = mol.coords + 0.05 * np.random.default_rng(seed).standard_normal(mol.coords.shape)   # Bohr
        mol = Molecule(mol.symbols, xyz, case["basis"], spherical=True)
    if case["kind"] == "fock_uks":
        mol = Molecule(mol.symbols, mol.coords, case["basis"], charge=1, spin=1, spherical=True)
    return mol


def _some_steps(ks, n, **kw):
    """A few SCF iterations: the densities and orbitals that Fock builds meet on the way."""
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        return scf(ks, max_iter=n, **kw)


def prepare(case, seed):
    kind = case["kind"]
    mol = _molecule(case, seed)
    if kind == "solve":
        return {"kind": kind, "server": Server(case["xc"], precision="mixed", slots=1), "mol": mol}
    if kind == "build":
        return {"kind": kind, "mol": mol, "xc": case["xc"]}
    coulomb = df(engine=hip(precision="mixed" if kind == "scf_mixed" else "fp64"))
    if kind == "fock_recompute":
        coulomb = df(chunk=case["chunk"], screen=1e-12)
    ks = KS(mol, case["xc"], coulomb=coulomb)
    state = {"kind": kind, "ks": ks, "mol": mol, "xc": case["xc"]}
    if kind in ("fock", "fock_uks"):
        state["P"] = _some_steps(ks, 3).P
    elif kind in ("fock_orbitals", "fock_recompute"):
        r = _some_steps(ks, 3)
        state["Cf"] = math.sqrt(2.0) * r.mo_coeff[0][:, : ks.nocc[0]]
    elif kind == "response":
        r = _some_steps(ks, 6)
        C, no = r.mo_coeff[0], ks.nocc[0]
        g = torch.Generator(device=C.device).manual_seed(seed)
        v = torch.randn((no, C.shape[1] - no), dtype=torch.float64, device=C.device, generator=g)
        state.update(P=r.P[0], U=C[:, :no].contiguous(), V=(-2.0 * (C[:, no:] @ v.T)).contiguous())
        ks.coulomb.response_begin(state["P"])
    elif kind == "forces":
        state["result"] = _some_steps(ks, 60, e_tol=1e-10, d_tol=1e-8)
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    ks = state.get("ks")
    if kind in ("fock", "fock_uks"):
        e, F = ks.energy_fock(state["P"])
        return {"e": e, "F": F}
    if kind in ("fock_orbitals", "fock_recompute"):
        E, F, P = ks.coulomb.energy_fock_factored(state["Cf"])
        return {"E": E, "F": F, "P": P}
    if kind in ("scf", "scf_mixed"):
        r = scf(ks, e_tol=1e-10, d_tol=1e-8)
        return {"e": r.e_tot, "P": r.P, "mo_energy": r.mo_energy}
    if kind == "solve":
        r = state["server"].solve(Request(rid=0, mol=state["mol"]))
        if r.error:
            raise RuntimeError(r.error)
        return {"e": r.e_tot}
    if kind == "build":
        k = KS(state["mol"], state["xc"], coulomb=df(engine=hip(keep_int3c=True)))
        c = k.coulomb
        return {"S": k.S, "hcore": k.hcore, "int2c": c.matrix(_native.DFKS_INT2C, (c.naux, c.naux)),
                "int3c": c.matrix(_native.DFKS_INT3C, (c.nao, c.nao, c.naux)), "e_nn": k.e_nn}
    if kind == "response":
        return {"R": ks.coulomb.response_fock(state["U"], state["V"])}
    return {"forces": forces(state["mol"], state["xc"], state["result"], ks=ks)}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
# functions per atom (orbital, fitting), electrons and grid points of the bases and the default grid
_PER_ATOM = {"def2-svp": {"H": 5, "X": 14}, "def2-tzvp": {"H": 6, "X": 31}}
_AUX = {"H": 15, "X": 85}
_GRID = {"H": 10500, "X": 11500}          # about what the weight cutoff leaves
_SCF_STEPS = 14


def work(case):
    n = case["size"]
    heavy, h = (n, 2 * n) if case["molecule"] == "water" else (n, int(1.9 * n) + 2)
    per = _PER_ATOM[case["basis"]]
    nao, naux = heavy * per["X"] + h * per["H"], heavy * _AUX["X"] + h * _AUX["H"]
    nocc = n * 5 if case["molecule"] == "water" else 4 * n + 1
    ng = heavy * _GRID["X"] + h * _GRID["H"]
    width = min(nao, 340 if case["basis"] == "def2-tzvp" else 170)   # functions that reach a grid point
    hybrid = case["xc"] != "PBE"
    tensors = 2 if case["xc"] == "CAM-B3LYP" else 1
    nn, kind = nao * nao, case["kind"]
    # the fitted tensor once (symmetric in its orbital pair), the AO values and gradients, P and F
    fock_b = 8 * (tensors * nn / 2 * naux + 4 * ng * width + 2 * nn)
    xc_f = 4.0 * ng * width * width
    # T = B^T C, K = T T^T (its upper half), J and gamma
    jk_f = (3.0 if hybrid else 2.0) * tensors * nn * naux * nocc + 2.0 * nn * naux
    # (mn|P) and B written once; B = (mn|P) L over the upper pairs, some 200 operations an integral
    build_b = 8 * (nn * naux + nn / 2 * naux + naux * naux + 4 * ng * width)
    build_f = nn * naux * naux + 4.0 * naux ** 3 + 100.0 * nn * naux + 30.0 * ng * (heavy + h) ** 2
    if kind in ("fock", "fock_orbitals"):
        return {"bytes": fock_b, "flops": jk_f + xc_f}
    if kind == "fock_uks":
        return {"bytes": fock_b + 16 * nn, "flops": 2 * (jk_f + xc_f)}
    if kind == "fock_recompute":
        return {"bytes": 8 * (4 * ng * width + 2 * nn + naux * naux),
                "flops": jk_f + xc_f + 100.0 * nn * naux + 2.0 * nao * naux * naux * nocc}
    if kind in ("scf", "scf_mixed"):
        return {"bytes": _SCF_STEPS * fock_b, "flops": _SCF_STEPS * (jk_f + xc_f + 20.0 * nao ** 3)}
    if kind == "solve":
        return {"bytes": build_b + _SCF_STEPS * fock_b,
                "flops": build_f + _SCF_STEPS * (jk_f + xc_f + 20.0 * nao ** 3)}
    if kind == "build":
        return {"bytes": build_b, "flops": build_f}
    if kind == "response":
        return {"bytes": fock_b, "flops": 2 * jk_f + xc_f}
    return {"bytes": 8 * (nn / 2 * naux + 10 * ng * width), "flops": 3 * jk_f + 4 * xc_f + 600.0 * nn * naux}


# ---------------------------------------------------------------------------
# the same in plain torch, 64 bits
# ---------------------------------------------------------------------------
# The fitted tensor, the AO rows, the grid and the core Hamiltonian of a handle are data here, as weights
# are to a network: everything from the density on is computed below. Solves, builds and forces have no
# value: their integrals in plain numpy would take minutes.
def _functional(xc, rho, sig):
    """rho * eps_xc of the closed-shell PBE, PBE0 and B3LYP."""
    pi2 = math.pi ** 2
    rs = (3.0 / (4.0 * math.pi * rho)) ** (1.0 / 3.0)
    kf = (3.0 * pi2 * rho) ** (1.0 / 3.0)
    lda = -0.75 * kf / math.pi
    if xc in ("PBE", "PBE0"):
        s2 = sig / (2.0 * kf * rho) ** 2
        kappa, mu = 0.804, 0.2195149727645171
        ex = lda * (1.0 + kappa - kappa / (1.0 + mu * s2 / kappa))
        A, a1, b = 0.0310907, 0.21370, (7.5957, 3.5876, 1.6382, 0.49294)
        q = rs.sqrt()
        ec = -2 * A * (1 + a1 * rs) * torch.log1p(1 / (2 * A * (b[0] * q + b[1] * rs + b[2] * rs * q + b[3] * rs * rs)))
        gam, beta = (1 - math.log(2.0)) / pi2, 0.06672455060314922
        t2 = sig / (4.0 * rho * rho * 4.0 * kf / math.pi)
        a = beta / (gam * torch.expm1(-ec / gam))
        f1 = t2 + a * t2 * t2
        ec = ec + gam * torch.log1p(beta * f1 / (gam * (1 + a * f1)))
        return rho * ((0.75 if xc == "PBE0" else 1.0) * ex + ec)
    r = 0.5 * rho
    x = 0.5 * (sig + 3e-60).sqrt() / r ** (4.0 / 3.0)
    b88 = (-0.75 * (6 / math.pi) ** (1 / 3) * r ** (1 / 3)
           - 0.0042 * r ** (1 / 3) * x * x / (1 + 6 * 0.0042 * x * torch.asinh(x)))
    A, b, c, x0 = 0.0310907, 13.0720, 42.7198, -0.409286
    y = rs.sqrt()
    X, X0, Q = y * y + b * y + c, x0 * x0 + b * x0 + c, math.sqrt(4 * c - b * b)
    at = torch.atan(Q / (2 * y + b))
    vwn = A * (torch.log(y * y / X) + 2 * b / Q * at
               - b * x0 / X0 * (torch.log((y - x0) ** 2 / X) + 2 * (b + 2 * x0) / Q * at))
    a_, b_, c_, d_ = 0.04918, 0.132, 0.2533, 0.349
    i3 = rho ** (-1 / 3)
    g = 1 / (1 + d_ * i3)
    om = torch.exp(-c_ * i3) * g * rho ** (-11 / 3)
    de = c_ * i3 + d_ * i3 * g
    lyp = -a_ * g - a_ * b_ * om * rho * (0.3 * (3 * pi2) ** (2 / 3) * rho ** (8 / 3) - sig * (3 + 7 * de) / 72)
    return rho * (0.08 * lda + 0.72 * b88 + 0.81 * lyp + 0.19 * vwn)


def _grad(f, *x):
    return torch.autograd.grad(f.sum(), x, create_graph=True)


def _xc(ks, xc, P, dP=None):
    """(E_xc, V_xc) at P, or the response of V_xc along dP."""
    n, dev = ks.nao, P.device
    w = torch.as_tensor(ks.grid_w, device=dev)
    ao = ks.coulomb.matrix(_native.DFKS_AO, (4, w.shape[0], n))
    V, e = torch.zeros((n, n), dtype=torch.float64, device=dev), 0.0
    for g0 in range(0, w.shape[0], 32768):
        phi, wg = ao[:, g0:g0 + 32768], w[g0:g0 + 32768]
        z = phi[0] @ P
        rho, drho = (z * phi[0]).sum(1), 2.0 * (z * phi[1:]).sum(2)
        keep = rho > 1e-10
        phi, wg, rho, drho = phi[:, keep], wg[keep], rho[keep], drho[:, keep]
        r, s = rho.clone().requires_grad_(), (drho * drho).sum(0).requires_grad_()
        f = _functional(xc, r, s)
        fr, fs = _grad(f, r, s)
        if dP is None:
            e = e + float((wg * f).sum())
            c0, cg = 0.5 * wg * fr, 2.0 * wg * fs * drho
        else:
            frr, frs = _grad(fr, r, s)
            fss = _grad(fs, s)[0]
            z1 = phi[0] @ dP
            r1, dr1 = (z1 * phi[0]).sum(1), 2.0 * (z1 * phi[1:]).sum(2)
            s1 = 2.0 * (drho * dr1).sum(0)
            c0 = 0.5 * wg * (frr * r1 + frs * s1)
            cg = 2.0 * wg * ((frs * r1 + fss * s1) * drho + fs * dr1)
        W = (c0.detach()[:, None] * phi[0]) + (cg.detach()[:, :, None] * phi[1:]).sum(0)
        V += phi[0].T @ W
    return e, V + V.T


def _jk(ks, P, hybrid):
    c, n = ks.coulomb, ks.nao
    B = c.matrix(_native.DFKS_BFIT, (n, n, c.nfit))
    gamma = P.reshape(-1) @ B.view(n * n, c.nfit)
    J = (B.view(n * n, c.nfit) @ gamma).view(n, n)
    K = torch.zeros_like(P)
    if hybrid:
        X = (P @ B.view(n, n * c.nfit)).view(n, n, c.nfit)
        for l in range(n):
            K += B[:, l] @ X[l].T
    return J, K


def exact(case, seed):
    kind, xc = case["kind"], case["xc"]
    if kind not in ("fock", "fock_orbitals", "fock_recompute", "response") or xc == "CAM-B3LYP":
        return None
    state = prepare(case, seed)
    ks = state["ks"]
    if kind == "fock_recompute":        # the same molecule with its tensor kept
        ks = KS(state["mol"], xc, coulomb=df(chunk=None))
    ax = {"PBE": 0.0, "PBE0": 0.25, "B3LYP": 0.2}[xc]
    if kind == "response":
        U, V = state["U"], state["V"]
        dP = U @ V.T + V @ U.T
        J, K = _jk(ks, dP, ax > 0)
        return {"R": J - 0.5 * ax * K + _xc(ks, xc, state["P"], dP)[1]}
    P = state["P"][0] if kind == "fock" else state["Cf"] @ state["Cf"].T
    J, K = _jk(ks, P, ax > 0)
    exc, V = _xc(ks, xc, P)
    F = ks.hcore + J - 0.5 * ax * K + V
    xyz, z = state["mol"].coords, state["mol"].atom_charges()
    d = np.linalg.norm(xyz[:, None] - xyz[None], axis=-1)[np.triu_indices(len(z), 1)]
    e = [float((P * ks.hcore).sum()), 0.5 * float((P * J).sum()), -0.25 * ax * float((P * K).sum()), exc,
         float(np.sum(np.outer(z, z)[np.triu_indices(len(z), 1)] / d))]
    if kind == "fock":
        return {"e": sum(e), "F": F}
    return {"E": torch.tensor([sum(e)] + e + [0.0, 0.0], dtype=torch.float64), "F": F, "P": P}
