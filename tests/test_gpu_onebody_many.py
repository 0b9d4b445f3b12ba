"""Overlap of more shell pairs in one class than one dimension of a launch
covers with a wave each (2^26 pairs are 2^32 threads), against the closed form
for s functions."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_overlap_of_more_than_2_to_26_pairs():
    from qdk_chemistry_amd.basis import BasisSet, Shell, normalize_psi4
    from qdk_chemistry_amd.eri import one_body_gpu
    from qdk_chemistry_amd.molecule import Structure
    n = 11586
    assert n * (n + 1) // 2 > 1 << 26
    i = np.arange(n)
    X = np.stack([1.7 * (i % 23), 1.9 * (i // 23 % 23), 2.1 * (i // 529)], 1) + 0.2 * np.sin(np.arange(3 * n)).reshape(n, 3)
    a = 0.3 + 0.8 * (i % 7)
    c = np.array([normalize_psi4(0, np.array([e]), np.array([1.0]))[0] for e in a])
    b = BasisSet(name="s", pure=True, natoms=1, shells=[
        Shell(0, 0, np.array([a[k]]), np.array([c[k]]), X[k].copy()) for k in range(n)])
    S = one_body_gpu(b, Structure(np.array([1]), X[:1].copy()), 0)
    rows = np.unique(np.concatenate([np.arange(0, n, 53), np.arange(64), np.arange(n - 64, n)]))
    worst = 0.0
    for r in rows:
        p = a[r] + a
        ref = c[r] * c * (np.pi / p) ** 1.5 * np.exp(-a[r] * a / p * np.sum((X[r] - X) ** 2, axis=1))
        worst = max(worst, np.max(np.abs(S[r] - ref)), np.max(np.abs(S[:, r] - ref)))
    print("max|dS| = %.2e over %d rows and columns" % (worst, len(rows)), flush=True)
    # exponents up to -37 before an element is below 1e-16: 37 roundings at most
    assert worst < 1e-14
