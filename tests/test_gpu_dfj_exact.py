"""Density-fitted J where the fit is exact: every product of two s functions of
one centre is a function of the auxiliary basis, so the fitted J of a density
without blocks between centres is the exact J (incore_impl_df.cpp:81-200).  The
sizes put the auxiliary functions below, at and above the rows of one block of
the triangular solve, and the pairs below and above one chunk of a row."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natoms,exps", [(1, (0.9,)), (1, (0.5, 2.2)), (42, (0.5, 2.2)), (128, (0.8,)), (43, (0.5, 2.2)),
                                         (64, (0.4, 1.8)), (129, (0.5, 2.2))])
def test_dfj_is_exact_for_products_in_the_auxiliary_basis(natoms, exps):
    from qdk_chemistry_amd.basis import BasisSet, Shell, normalize_psi4
    from qdk_chemistry_amd.eri import DFJ, create
    from qdk_chemistry_amd.molecule import Structure
    side = int(np.ceil(natoms ** (1.0 / 3.0) - 1e-9))
    g = np.array([(i // side // side, i // side % side, i % side) for i in range(natoms)], dtype=float)
    mol = Structure(np.full(natoms, 2), 3.1 * g + 0.2 * np.sin(np.arange(3 * natoms).reshape(natoms, 3)))

    def basis(name, exponents):
        return BasisSet(name=name, pure=True, natoms=natoms, shells=[
            Shell(a, 0, np.array([e]), normalize_psi4(0, np.array([e]), np.array([1.0])), mol.coords[a].copy())
            for a in range(natoms) for e in exponents])

    k = len(exps)
    b = basis("s", exps)
    aux = basis("products", [exps[i] + exps[j] for i in range(k) for j in range(i, k)])
    rng = np.random.default_rng(natoms + k)
    P = np.zeros((b.nbf, b.nbf))
    for a in range(natoms):
        m = rng.uniform(-0.5, 1.0, (k, k))
        P[a * k:(a + 1) * k, a * k:(a + 1) * k] = m + m.T
    dfj = DFJ(b, aux, mol)
    Jd, _ = dfj.build_JK(P)
    Je, _ = create(b, mol).build_JK(P, K=False)
    rel = np.max(np.abs(Jd - Je)) / np.max(np.abs(Je))
    print(natoms, b.nbf, dfj.naux, "max|J_df - J| / max|J| = %.2e" % rel, flush=True)
    assert rel < 1e-9  # the exact J drops quartets below 1e-12
    again, _ = dfj.build_JK(P)
    assert np.array_equal(again, Jd)
