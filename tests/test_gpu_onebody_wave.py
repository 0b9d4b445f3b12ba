"""One-electron kernels (a wave per shell pair) where their loops end: more
primitive pairs and more nuclei than a wave has lanes, one of each, pure and
cartesian shells up to f, against the host path (int1e.h's integrals and
derivative contractions) with the bars of the other one-electron tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _probe(natoms, nprim, lmax, pure):
    from qdk_chemistry_amd.basis import BasisSet, Shell, normalize_psi4
    from qdk_chemistry_amd.molecule import Structure
    i = np.arange(natoms)
    R = np.stack([2.1 * (i % 5), 2.3 * (i // 5 % 5), 1.9 * (i // 25)], 1) + 0.3 * np.cos(np.arange(3 * natoms)).reshape(-1, 3)
    mol = Structure(1 + i % 8, R)
    shells = []
    for l in range(lmax + 1):
        for atom in sorted({0, natoms // 2, natoms - 1}):
            n = nprim if atom == 0 else 1
            exps = 0.4 * 1.9 ** np.arange(n)[::-1] + 0.1 * l + 0.05 * atom / natoms
            c = normalize_psi4(l, exps, np.linspace(0.7, 0.2, n))
            shells.append(Shell(atom, l, exps, c, mol.coords[atom].copy()))
    return mol, BasisSet(name="probe", shells=shells, pure=pure, natoms=natoms)


@pytest.mark.parametrize("natoms,nprim,lmax,pure", [(1, 1, 0, True), (2, 9, 3, True), (63, 8, 2, False), (64, 1, 3, False),
                                                    (65, 9, 2, True), (130, 3, 3, True)])
def test_one_body_wave_kernels_vs_host(natoms, nprim, lmax, pure):
    from qdk_chemistry_amd.eri import one_body, one_body_gpu, one_body_grad, one_body_grad_gpu
    mol, b = _probe(natoms, nprim, lmax, pure)
    W = np.random.default_rng(natoms).uniform(-1, 1, (b.nbf, b.nbf))
    W = 0.5 * (W + W.T)
    for op in range(3):
        M, Mh = one_body_gpu(b, mol, op), one_body(b, mol, op)
        g, gh = one_body_grad_gpu(b, mol, op, W), one_body_grad(b, mol, op, W)
        dm = np.max(np.abs(M - Mh)) / max(1.0, np.max(np.abs(Mh)))
        dg = np.max(np.abs(g - gh)) / max(1.0, np.max(np.abs(gh)))
        print(f"{natoms} {nprim} {lmax} op {op}: rel dM {dm:.2e}, rel dg {dg:.2e}", flush=True)
        assert dm < 1e-11 and dg < 1e-9
