"""The chunk kernels of the gradient (a thread per quartet and chunk) for
classes that would run in the cooperative kernels, with QFE_COOP=0: against
the oracle's ERI::get_gradients (libint2_direct.cpp:646-890) and against the
cooperative kernels, for one density and for a spin pair; and the strided loop
of larger classes."""
import numpy as np
import pytest

from conftest import decaying_density, random_density

pytestmark = pytest.mark.gpu


def _probe(nprim):
    from qdk_chemistry_amd.basis import BasisSet, Shell, normalize_psi4
    from qdk_chemistry_amd.molecule import Structure
    mol = Structure(np.array([8, 6, 1]), np.array([[0.0, 0.1, -0.2], [0.3, 1.9, 0.4], [-1.2, 0.2, 2.1]]))
    shells = []
    for l in range(3):
        for atom, n in ((0, nprim), (1, 1), (2, 2 if l < 2 else 1)):
            exps = 0.9 * 2.7 ** np.arange(n)[::-1] + 0.1 * l
            c = normalize_psi4(l, exps, np.linspace(0.6, 0.3, n))
            shells.append(Shell(atom, l, exps, c, mol.coords[atom].copy()))
    return mol, BasisSet(name="probe", shells=shells, pure=True, natoms=3)


@pytest.mark.parametrize("nprim", [1, 2, 5])
def test_chunk_kernels_of_every_class_up_to_d(monkeypatch, nprim):
    from oracle.oracle import OracleERI
    from qdk_chemistry_amd.eri import create
    mol, b = _probe(nprim)
    coop, o = create(b, mol), OracleERI(b, mol)
    monkeypatch.setenv("QFE_COOP", "0")
    chunks = create(b, mol)
    P = random_density(b.nbf, 23, 0.2)
    for D in (P, np.stack([P, random_density(b.nbf, 24, 0.1)])):
        dJ, dK = chunks.get_gradients(D)
        cJ, cK = coop.get_gradients(D)
        rJ, rK = o.get_gradients(D, mode=1)
        print(nprim, D.shape, "chunks vs oracle %.2e %.2e, vs cooperative %.2e %.2e" % (
            np.max(np.abs(dJ - rJ)), np.max(np.abs(dK - rK)), np.max(np.abs(dJ - cJ)), np.max(np.abs(dK - cK))),
            flush=True)
        # the engine and the oracle both screen quartets at 1e-12: the bar of the other gradient tests
        assert np.max(np.abs(dJ - rJ)) < 1e-10 and np.max(np.abs(dK - rK)) < 1e-10
        # one task list: the two kernels differ by rounding alone
        assert np.max(np.abs(dJ - cJ)) < 1e-11 and np.max(np.abs(dK - cK)) < 1e-11


def test_chunk_kernels_of_a_cluster_vs_oracle(monkeypatch):
    from oracle.oracle import OracleERI
    from qdk_chemistry_amd.basis import load_basis
    from qdk_chemistry_amd.eri import create
    from qdk_chemistry_amd.molecule import water_cluster
    mol = water_cluster(2, 5)
    b = load_basis("cc-pvdz", mol.numbers, mol.coords)
    monkeypatch.setenv("QFE_COOP", "0")
    D = np.stack([random_density(b.nbf, 31, 0.3), random_density(b.nbf, 32, 0.2)])
    dJ, dK = create(b, mol).get_gradients(D)
    rJ, rK = OracleERI(b, mol).get_gradients(D, mode=1)
    assert np.max(np.abs(dJ - rJ)) < 1e-10 and np.max(np.abs(dK - rK)) < 1e-10


def test_spin_pair_of_classes_beyond_one_grid():
    """(H2O)16/cc-pVDZ has classes of more quartets than one grid of the chunk
    kernels holds threads (524,288).  The spin pair's gradient is
    dJ[Pa + Pb] and 2 dK[Pa] + 2 dK[Pb] of the one-density gradients, which
    other tests hold to the oracle."""
    from qdk_chemistry_amd.basis import load_basis
    from qdk_chemistry_amd.eri import ERIConfig, create
    from qdk_chemistry_amd.molecule import water_cluster
    mol = water_cluster(16, 20261202)
    b = load_basis("cc-pvdz", mol.numbers, mol.coords)
    Pa, Pb = decaying_density(b, 7, 0.3), decaying_density(b, 8, 0.3)
    eng = create(b, mol, ERIConfig(eri_threshold=1e-15))
    sJ, sK = eng.get_gradients(np.stack([Pa, Pb]))
    eng.build_JK(Pa)
    assert max(nq for _, nq, _, _ in eng.class_stats(0)) > 524288
    aJ, aK = eng.get_gradients(Pa)
    bJ, bK = eng.get_gradients(Pb)
    tJ, _ = eng.get_gradients(Pa + Pb)
    print("max|ddJ| %.2e max|ddK| %.2e" % (np.max(np.abs(sJ - tJ)), np.max(np.abs(sK - 2 * aK - 2 * bK))), flush=True)
    assert np.max(np.abs(sJ - tJ)) < 1e-10 and np.max(np.abs(sK - 2 * aK - 2 * bK)) < 1e-10
