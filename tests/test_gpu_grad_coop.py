"""The cooperative gradient kernels (a block per shell quartet) against the
oracle's ERI::get_gradients (libint2_direct.cpp:646-890): every class up to
(ff|ff) over one small basis, with contraction lengths that leave the last
batch of (primitive quartet, root) combinations full, short or alone."""
import numpy as np
import pytest

from conftest import random_density

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nprim", [1, 2, 5])
@pytest.mark.parametrize("lmax", [2, 3])
def test_small_basis_gradient_vs_oracle(lmax, nprim):
    from oracle.oracle import OracleERI
    from qdk_chemistry_amd.basis import BasisSet, Shell, normalize_psi4
    from qdk_chemistry_amd.eri import compiled_max_l, create
    from qdk_chemistry_amd.molecule import Structure
    if compiled_max_l() < lmax:
        pytest.skip("library built without f-shell classes")
    mol = Structure(np.array([8, 6, 1]), np.array([[0.0, 0.1, -0.2], [0.3, 1.9, 0.4], [-1.2, 0.2, 2.1]]))
    shells = []
    for l in range(lmax + 1):  # a contracted shell on the first centre, a primitive one on the others
        for atom, n in ((0, nprim), (1, 1), (2, 1 if l < 2 else 0)):
            if n == 0:
                continue
            exps = 0.9 * 2.7 ** np.arange(n)[::-1] + 0.1 * l
            c = normalize_psi4(l, exps, np.linspace(0.6, 0.3, n))
            shells.append(Shell(atom, l, exps, c, mol.coords[atom].copy()))
    b = BasisSet(name="probe", shells=shells, pure=True, natoms=3)
    eng, o = create(b, mol), OracleERI(b, mol)
    P = random_density(b.nbf, 23, 0.2)
    for D in (P, np.stack([P, random_density(b.nbf, 24, 0.1)])):
        dJ, dK = eng.get_gradients(D)
        rJ, rK = o.get_gradients(D, mode=1)
        print(lmax, nprim, D.shape, "max|ddJ| %.2e max|ddK| %.2e of %.2e" % (
            np.max(np.abs(dJ - rJ)), np.max(np.abs(dK - rK)), np.max(np.abs(rJ))), flush=True)
        # the engine and the oracle both screen quartets at 1e-12: the bar of the other gradient tests
        assert np.max(np.abs(dJ - rJ)) < 1e-10 and np.max(np.abs(dK - rK)) < 1e-10
