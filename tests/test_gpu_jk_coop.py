"""The cooperative J/K kernels (a block per shell quartet) against the
oracle's build_JK (libint2_direct.cpp:256-626) and against the segment
kernels: every class up to (ff|ff) over one small basis, with contraction
lengths that leave the last batch of (primitive quartet, root) combinations
full, short or alone, with both kinds of sums and null outputs."""
import numpy as np
import pytest

from conftest import random_density

pytestmark = pytest.mark.gpu


def _probe(lmax, nprim):
    from qdk_chemistry_amd.basis import BasisSet, Shell, normalize_psi4
    from qdk_chemistry_amd.molecule import Structure
    mol = Structure(np.array([8, 6, 1]), np.array([[0.0, 0.1, -0.2], [0.3, 1.9, 0.4], [-1.2, 0.2, 2.1]]))
    shells = []
    for l in range(lmax + 1):
        for atom, n in ((0, nprim), (1, 1), (2, 1 if l < 2 else 0)):
            if n == 0:
                continue
            exps = 0.9 * 2.7 ** np.arange(n)[::-1] + 0.1 * l
            c = normalize_psi4(l, exps, np.linspace(0.6, 0.3, n))
            shells.append(Shell(atom, l, exps, c, mol.coords[atom].copy()))
    return mol, BasisSet(name="probe", shells=shells, pure=True, natoms=3)


@pytest.mark.parametrize("atomics", [False, True])
@pytest.mark.parametrize("nprim", [1, 2, 5])
@pytest.mark.parametrize("lmax", [2, 3])
def test_small_basis_jk_vs_oracle(lmax, nprim, atomics):
    from oracle.oracle import OracleERI
    from qdk_chemistry_amd.eri import ERIConfig, compiled_max_l, create
    if compiled_max_l() < lmax:
        pytest.skip("library built without f-shell classes")
    mol, b = _probe(lmax, nprim)
    eng, o = create(b, mol, ERIConfig(use_atomics=atomics)), OracleERI(b, mol)
    P = random_density(b.nbf, 31, 0.2)
    J, K = eng.build_JK(P)
    Jr, Kr = o.build_JK(P)
    print(lmax, nprim, atomics, "max|dJ| %.2e max|dK| %.2e" % (np.max(np.abs(J - Jr)), np.max(np.abs(K - Kr))), flush=True)
    # both sides screen quartets at 1e-12: the bar of the other J/K tests
    assert np.max(np.abs(J - Jr)) < 1e-10 and np.max(np.abs(K - Kr)) < 1e-10
    J1, none = eng.build_JK(P, K=False)
    assert none is None
    none, K1 = eng.build_JK(P, J=False)
    assert none is None
    bar = 1e-12 if atomics else 0.0  # FP64 atomics round in any order; fixed-point sums do not
    assert np.max(np.abs(J1 - J)) <= bar and np.max(np.abs(K1 - K)) <= bar


def test_cooperative_and_segment_kernels_agree(monkeypatch):
    """(H2O)4/cc-pVDZ has classes on both sides of the dispatch; with
    QFE_COOP=0 all of them run in the segment kernels."""
    from qdk_chemistry_amd.basis import load_basis
    from qdk_chemistry_amd.eri import ERIConfig, create
    from qdk_chemistry_amd.molecule import water_cluster
    mol = water_cluster(4, 9)
    b = load_basis("cc-pvdz", mol.numbers, mol.coords)
    P = random_density(b.nbf, 37, 0.2)
    for cfg in (ERIConfig(), ERIConfig(use_atomics=True), ERIConfig(is_mix_precision=True)):
        monkeypatch.delenv("QFE_COOP", raising=False)
        J, K = create(b, mol, cfg).build_JK(P)
        monkeypatch.setenv("QFE_COOP", "0")
        J0, K0 = create(b, mol, cfg).build_JK(P)
        d = max(np.max(np.abs(J - J0)), np.max(np.abs(K - K0)))
        # mixed builds: the cooperative kernels evaluate FP32 tasks (bound 1e-6) in FP64
        assert d < (1e-8 if cfg.is_mix_precision else 1e-11), d
