"""The dense AO tensor's class kernels (through the quarter transform) against
the oracle: s, p and d shells whose contraction lengths leave the last batch
of (primitive quartet, root) combinations full, short or alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lmax,nprim", [(0, 1), (1, 3), (2, 1), (2, 2), (2, 5)])
def test_quarter_trans_of_contracted_shells_vs_oracle(lmax, nprim):
    from oracle.oracle import OracleERI, quarter_trans
    from qdk_chemistry_amd.basis import BasisSet, Shell, normalize_psi4
    from qdk_chemistry_amd.eri import create
    from qdk_chemistry_amd.molecule import Structure
    mol = Structure(np.array([8, 6, 1]), np.array([[0.0, 0.1, -0.2], [0.3, 1.9, 0.4], [-1.2, 0.2, 2.1]]))
    shells = []
    for l in range(lmax + 1):
        for atom, n in ((0, nprim), (1, 1)):
            exps = 0.9 * 2.7 ** np.arange(n)[::-1] + 0.1 * l
            c = normalize_psi4(l, exps, np.linspace(0.6, 0.3, n))
            shells.append(Shell(atom, l, exps, c, mol.coords[atom].copy()))
    b = BasisSet(name="probe", shells=shells, pure=True, natoms=3)
    C = np.random.default_rng(nprim).uniform(-1.0, 1.0, (b.nbf, min(5, b.nbf)))
    got = create(b, mol).quarter_trans(C)
    ref = quarter_trans(OracleERI(b, mol).eri_full(), C)
    print(lmax, nprim, "max|diff| = %.2e" % np.max(np.abs(got - ref)), flush=True)
    assert np.max(np.abs(got - ref)) < 1e-11  # the bar of the other transform tests
