"""One-electron integrals between distant diffuse shells: the product of the
contraction coefficients and the Gaussian factor is below 1e-18 there while
the polynomials (|P - A|^la |P - B|^lb) and the extent (pi/p)^(3/2) of the
product bring the integrals back to 1e-9 and more, against the host path
(int1e.h's integrals and derivative contractions), which drops no primitive
pair."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pair(l, exp, nprim, factor):
    """Two shells of momentum l and smallest exponent exp, factor times as far
    apart as brings the product prefactor of their most diffuse primitives to
    1e-18, with an s shell and a nucleus on a third centre between them."""
    from qdk_chemistry_amd.basis import BasisSet, Shell, normalize_psi4
    from qdk_chemistry_amd.molecule import Structure
    exps = exp * 2.3 ** np.arange(nprim)[::-1]
    c = normalize_psi4(l, exps, np.linspace(0.4, 1.0, nprim))
    R = factor * np.sqrt(2.0 * np.log(c[-1] ** 2 * 1e18) / exp)
    u = np.array([2.0, 1.0, 2.0]) / 3.0
    X = np.array([[0.1, -0.2, 0.3], [0.0, 0.0, 0.0], [0.0, 0.0, 0.0]])
    X[1] = X[0] + R * u
    X[2] = X[0] + 0.45 * R * u + np.array([0.3, 0.9, -0.4])
    mol = Structure(np.array([6, 8, 1]), X)
    shells = [Shell(a, l, exps, c, X[a].copy()) for a in (0, 1)]
    e = np.array([1.1])
    shells.append(Shell(2, 0, e, normalize_psi4(0, e, np.array([1.0])), X[2].copy()))
    return mol, BasisSet(name="diffuse", shells=shells, pure=True, natoms=3)


@pytest.mark.parametrize("factor", [1.002, 1.15])
@pytest.mark.parametrize("l,exp,nprim", [(3, 0.05, 1), (3, 0.27, 1), (2, 0.02, 1), (2, 0.04, 3), (1, 0.003, 1)])
def test_distant_diffuse_shells_vs_host(l, exp, nprim, factor):
    from qdk_chemistry_amd.eri import one_body, one_body_gpu, one_body_grad, one_body_grad_gpu
    mol, b = _pair(l, exp, nprim, factor)
    n = b.shell_offsets[1]
    W = np.random.default_rng(l).uniform(-1, 1, (b.nbf, b.nbf))
    W = 0.5 * (W + W.T)
    Wf = np.zeros_like(W)  # the distant pair's block alone
    Wf[:n, n:2 * n] = W[:n, n:2 * n]
    Wf[n:2 * n, :n] = W[n:2 * n, :n]
    for op in range(3):
        M, Mh = one_body_gpu(b, mol, op), one_body(b, mol, op)
        far, farh = M[:n, n:2 * n], Mh[:n, n:2 * n]
        top = np.max(np.abs(farh))
        df = np.max(np.abs(far - farh)) / top
        print(f"l {l} exp {exp} x{nprim} R {np.linalg.norm(mol.coords[0] - mol.coords[1]):.1f} op {op}: "
              f"max|M_far| {top:.2e}, rel dM_far {df:.2e}", flush=True)
        # a few hundred roundings of sums without cancellation beyond two or three digits
        assert np.max(np.abs(M - Mh)) < 1e-13 * max(1.0, np.max(np.abs(Mh)))
        assert df < 1e-10
        for w in (W, Wf):
            g, gh = one_body_grad_gpu(b, mol, op, w), one_body_grad(b, mol, op, w)
            dg, gtop = np.max(np.abs(g - gh)), np.max(np.abs(gh))
            print(f"   max|g| {gtop:.2e}, dg {dg:.2e}", flush=True)
            assert dg < 1e-12 * max(1.0, gtop)
        assert dg < 1e-9 * gtop  # the distant pair's own force
