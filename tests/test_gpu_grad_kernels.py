"""Kernels behind the differentiable one-gate functions against numpy."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import rand_state, rand_unitary, to_gpu, to_np
from oracle import statevector as O

pytestmark = pytest.mark.gpu


def gathered(v, n, bits):
    """Rows: the patterns on `bits` (bits[0] most significant)."""
    ax = [n - 1 - b for b in bits]
    rest = [a for a in range(n) if a not in ax]
    return np.transpose(v.reshape([2] * n), ax + rest).reshape(1 << len(bits), -1)


# every k at n = k (one item), one partial block, several blocks; any bit order
@pytest.mark.parametrize("n,bits", [
    (1, [0]), (11, [10]), (13, [0]), (20, [7]), (2, [0, 1]), (2, [1, 0]), (13, [3, 12]),
    (19, [18, 0]), (3, [1, 2, 0]), (14, [0, 13, 5]), (4, [3, 1, 0, 2]), (15, [14, 2, 9, 0])])
def test_matrix_grad(n, bits):
    from tyxonq_amd import _native as nat

    rng = np.random.default_rng(n)
    p, g = to_gpu(rand_state(rng, n)), to_gpu(rand_state(rng, n))
    ref = gathered(to_np(g), n, bits) @ gathered(to_np(p), n, bits).conj().T
    # exact FP64 products of the same complex64 values: sums to about 2^-52 per step
    np.testing.assert_allclose(nat.matrix_grad(p, g, bits), ref, atol=1e-13)
    with pytest.raises(ValueError):
        nat.matrix_grad(p, g, [0, 0])
    with pytest.raises(ValueError):
        nat.matrix_grad(p, g, [n])


@pytest.mark.parametrize("n", [1, 2, 9, 17])
def test_out_of_place_gates_and_z(n):
    import torch

    from tyxonq_amd import _native as nat

    rng = np.random.default_rng(n)
    v = to_gpu(rand_state(rng, n))
    for q in sorted({0, n // 2, n - 1}):
        U = rand_unitary(rng, 2)
        # 4 products and 3 sums of unit-norm rows at 2^-24 each
        np.testing.assert_allclose(to_np(nat.apply_1q_to(v, n - 1 - q, U)),
                                   O.apply_1q(to_np(v), U, q, n), atol=8 * 2.0 ** -24)
        ge = torch.tensor(-0.7, dtype=torch.float64, device="cuda")
        z = 1.0 - 2.0 * ((np.arange(1 << n) >> (n - 1 - q)) & 1)
        np.testing.assert_allclose(to_np(nat.z_grad(v, n - 1 - q, ge)), -1.4 * z * to_np(v),
                                   atol=2 * 2.0 ** -24)
        e = nat.expect_z_dev(v, n - 1 - q)
        assert e.is_cuda and e.dtype == torch.float64
        # the host entry point sums the same blocks
        assert float(e) == nat.expect_z(v, n - 1 - q)
    for a, b in [(0, 1), (1, 0), (0, n - 1)] if n > 1 else []:
        U = rand_unitary(rng, 4)
        np.testing.assert_allclose(to_np(nat.apply_2q_to(v, n - 1 - a, n - 1 - b, U)),
                                   O.apply_2q(to_np(v), U, a, b, n), atol=16 * 2.0 ** -24)
