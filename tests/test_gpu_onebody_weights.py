"""One-electron derivative contractions with a weight matrix that is not
symmetric, against the host path (the *_integral_deriv(dm, res) contractions
of int1e.h): the derivatives by both shells are then weighted differently,
also where the shells sit on one atom."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("basis", ["cc-pvdz", "cc-pvtz"])
def test_derivatives_with_a_nonsymmetric_weight(water, basis):
    from qdk_chemistry_amd.basis import load_basis
    from qdk_chemistry_amd.eri import one_body_grad, one_body_grad_gpu
    b = load_basis(basis, water.numbers, water.coords)
    W = np.random.default_rng(3).uniform(-1, 1, (b.nbf, b.nbf))
    blocks = np.zeros_like(W)  # the blocks of the shells of one atom alone
    at = np.concatenate([[s.atom] * (b.shell_offsets[i + 1] - b.shell_offsets[i]) for i, s in enumerate(b.shells)])
    same = at[:, None] == at[None, :]
    blocks[same] = W[same]
    for op in range(3):
        for w in (W, blocks):
            g, gh = one_body_grad_gpu(b, water, op, w), one_body_grad(b, water, op, w)
            d = np.max(np.abs(g - gh))
            print(f"{basis} op {op}: max|g| {np.max(np.abs(gh)):.2e}, dg {d:.2e}", flush=True)
            assert d < 1e-9  # the bar of the other one-electron derivative tests
