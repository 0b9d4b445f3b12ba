"""The profiled count of evaluated primitive quartets follows the kernel that
ran: the cooperative kernels evaluate the full product of the two prefixes of
primitives that pass the engine's cut (libint2_direct.cpp:279-287) with their
best partner, the segment kernels leave out the pairs inside it that fail
together."""
import numpy as np
import pytest

from conftest import decaying_density

pytestmark = pytest.mark.gpu


def _counts(eng, P, prec):
    eng.build_JK(P)
    return {c: (nq, n, coop) for (c, nq, n, _), coop in zip(eng.class_stats(prec, executed=True),
                                                             eng.class_cooperative(prec)) if nq > 0}


def test_count_of_one_pair_is_that_of_the_kernel(monkeypatch):
    """One shell: one quartet, whose counts numpy forms from the cut."""
    from qdk_chemistry_amd.basis import BasisSet, Shell, normalize_psi4
    from qdk_chemistry_amd.eri import ERIConfig, create
    from qdk_chemistry_amd.molecule import Structure
    e = 0.2 * 4.0 ** np.arange(9)
    c = normalize_psi4(0, e, 10.0 ** -np.arange(9.0))
    mol = Structure(np.array([1]), np.zeros((1, 3)))
    b = BasisSet(name="s", pure=True, natoms=1, shells=[Shell(0, 0, e, c, np.zeros(3))])
    P = np.array([[2.0e-3]])
    p = (e[:, None] + e[None, :]).ravel()
    # 2 pi^(5/2) K_ab K_cd / (p q sqrt(p + q)) with p + q >= 2 sqrt(p q)
    sig = np.log(np.abs(np.outer(c, c)).ravel() / p) - 0.25 * np.log(p) + 0.5 * np.log(np.sqrt(2.0) * np.pi ** 2.5)
    lnp = np.log(np.finfo(float).eps / P[0, 0])
    walk = int(np.count_nonzero(sig[:, None] + sig[None, :] >= lnp))
    prefix = int(np.count_nonzero(sig + sig.max() >= lnp)) ** 2
    assert walk < prefix < sig.size ** 2
    cfg = ERIConfig(profile=True, eri_threshold=0.0)
    assert _counts(create(b, mol, cfg), P, 0) == {(0, 0, 0, 0): (1.0, float(prefix), True)}
    monkeypatch.setenv("QFE_COOP", "0")
    assert _counts(create(b, mol, cfg), P, 0) == {(0, 0, 0, 0): (1.0, float(walk), False)}


@pytest.mark.parametrize("mix", [False, True])
def test_counts_of_both_kernels_in_a_cluster(monkeypatch, mix):
    from qdk_chemistry_amd.basis import load_basis
    from qdk_chemistry_amd.eri import ERIConfig, create
    from qdk_chemistry_amd.molecule import water_cluster
    mol = water_cluster(4, 11)
    b = load_basis("cc-pvdz", mol.numbers, mol.coords)
    P = decaying_density(b, 17, 1.0)
    cfg = ERIConfig(profile=True, is_mix_precision=mix)
    eng = create(b, mol, cfg)
    with_coop = [_counts(eng, P, prec) for prec in (0, 1)]
    monkeypatch.setenv("QFE_COOP", "0")
    seg_eng = create(b, mol, cfg)
    kinds = set()
    for prec in (0, 1):
        seg = _counts(seg_eng, P, prec)
        assert seg.keys() == with_coop[prec].keys()
        for cls, (nq, n, coop) in with_coop[prec].items():
            assert nq == seg[cls][0] and not seg[cls][2]
            assert n >= seg[cls][1] if coop else n == seg[cls][1]
            kinds.add(coop)
    assert kinds == {True, False}


def test_flop_model_counts_a_cooperative_class_once():
    from qdk_chemistry_amd.flops import chunks, class_flops
    for cls in ((2, 2, 2, 2), (2, 1, 1, 1), (3, 2, 2, 1)):
        if max(cls) > 2:
            from qdk_chemistry_amd.eri import compiled_max_l
            if compiled_max_l() < 3:
                continue
        once, chunked = class_flops(*cls, coop=True)[0], class_flops(*cls)[0]
        print(cls, len(chunks(*cls)), once, chunked, flush=True)
        assert len(chunks(*cls)) == 1 or once < chunked
