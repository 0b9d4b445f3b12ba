"""The variants of the segment J/K kernels with the cooperative kernels off
(QFE_COOP=0), so that classes with few quartets run in them too: exchange rows
in column tiles, density rows left out of LDS, J_cd by atomics instead of
share slots (also with the cooperative kernels, which have both ways).  Each
against the default variant and the oracle's build_JK (libint2_direct.cpp:
256-626), for a water cluster and for one small basis with every class up to
(ff|ff)."""
import numpy as np
import pytest

from conftest import random_density

pytestmark = pytest.mark.gpu


def _system(name):
    from qdk_chemistry_amd.basis import BasisSet, Shell, load_basis, normalize_psi4
    from qdk_chemistry_amd.eri import compiled_max_l
    from qdk_chemistry_amd.molecule import Structure, water_cluster
    if name == "h2o4":
        mol = water_cluster(4, 11)
        return mol, load_basis("cc-pvdz", mol.numbers, mol.coords)
    if compiled_max_l() < 3:
        pytest.skip("library built without f-shell classes")
    mol = Structure(np.array([8, 6, 1]), np.array([[0.0, 0.1, -0.2], [0.3, 1.9, 0.4], [-1.2, 0.2, 2.1]]))
    shells = []
    for l in range(4):
        for atom, n in ((0, 2), (1, 1), (2, 1 if l < 2 else 0)):
            if n:
                exps = 0.9 * 2.7 ** np.arange(n)[::-1] + 0.1 * l
                c = normalize_psi4(l, exps, np.linspace(0.6, 0.3, n))
                shells.append(Shell(atom, l, exps, c, mol.coords[atom].copy()))
    return mol, BasisSet(name="probe", shells=shells, pure=True, natoms=3)


def _compare(monkeypatch, system, coop, env, atomics, mix, same):
    """J and K with and without env, against each other and the oracle."""
    from oracle.oracle import OracleERI
    from qdk_chemistry_amd.eri import ERIConfig, create
    mol, b = _system(system)
    P = random_density(b.nbf, 14, 0.3)
    cfg = ERIConfig(use_atomics=atomics, is_mix_precision=mix)
    if not coop:
        monkeypatch.setenv("QFE_COOP", "0")
    J1, K1 = create(b, mol, cfg).build_JK(P)
    monkeypatch.setenv(*env)
    J0, K0 = create(b, mol, cfg).build_JK(P)
    Jr, Kr = OracleERI(b, mol).build_JK(P)
    d = max(np.max(np.abs(J1 - J0)), np.max(np.abs(K1 - K0)))
    r = max(np.max(np.abs(J0 - Jr)), np.max(np.abs(K0 - Kr)))
    print(system, "coop" if coop else "segments", env, atomics, mix, "vs default %.2e, vs oracle %.2e" % (d, r), flush=True)
    if same:
        assert d < 1e-12
    assert r < (1e-8 if mix else 1e-10)


@pytest.mark.parametrize("system", ["h2o4", "f"])
@pytest.mark.parametrize("atomics,mix", [(False, False), (True, False), (False, True)])
def test_column_tiles(monkeypatch, system, atomics, mix):
    # under mixed precision the tiled kernel evaluates FP32 tasks in FP64
    _compare(monkeypatch, system, False, ("QFE_KCOL_TILE", "20"), atomics, mix, not mix)


@pytest.mark.parametrize("system", ["h2o4", "f"])
@pytest.mark.parametrize("atomics,mix", [(False, False), (True, False), (False, True)])
def test_density_rows_out_of_lds(monkeypatch, system, atomics, mix):
    _compare(monkeypatch, system, False, ("QFE_SEGMENT_DIGEST", "0"), atomics, mix, True)


@pytest.mark.parametrize("coop", [False, True])
@pytest.mark.parametrize("system", ["h2o4", "f"])
@pytest.mark.parametrize("atomics,mix", [(False, False), (True, False), (False, True)])
def test_coulomb_shares_by_atomics(monkeypatch, system, atomics, mix, coop):
    _compare(monkeypatch, system, coop, ("QFE_JCD_SLOTS", "0"), atomics, mix, True)


@pytest.mark.parametrize("atomics", [False, True])
def test_nonsymmetric_density_in_both_kernels(monkeypatch, atomics):
    """Both kernels read the same blocks of the density, also where it is not
    symmetric."""
    from qdk_chemistry_amd.eri import ERIConfig, create
    mol, b = _system("f")
    P = np.random.default_rng(5).uniform(-0.3, 0.3, (b.nbf, b.nbf))
    J1, K1 = create(b, mol, ERIConfig(use_atomics=atomics)).build_JK(P)
    monkeypatch.setenv("QFE_COOP", "0")
    J0, K0 = create(b, mol, ERIConfig(use_atomics=atomics)).build_JK(P)
    assert max(np.max(np.abs(J1 - J0)), np.max(np.abs(K1 - K0))) < 1e-11


def test_shares_of_an_earlier_build_are_left_out(monkeypatch):
    """Share slots that an earlier, denser build filled do not enter the sums
    of a build whose density drops those quartets."""
    from oracle.oracle import OracleERI
    from qdk_chemistry_amd.eri import create
    mol, b = _system("h2o4")
    dense = random_density(b.nbf, 12, 0.3)
    molecule = np.concatenate([[s.atom // 3] * b.nfun(s.l) for s in b.shells])
    blk = np.where(molecule[:, None] == molecule[None, :], dense, 0.0)
    monkeypatch.setenv("QFE_COOP", "0")
    eng = create(b, mol)
    eng.build_JK(dense)
    many = eng.stats()["quartets"]
    J, K = eng.build_JK(blk)
    assert eng.stats()["quartets"] < many
    Jr, Kr = OracleERI(b, mol).build_JK(blk)
    assert np.max(np.abs(J - Jr)) < 1e-10 and np.max(np.abs(K - Kr)) < 1e-10
