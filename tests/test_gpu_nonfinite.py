"""Infinities and NaN reach only the amplitudes whose definition has them."""
from __future__ import annotations

import numpy as np
import pytest

from tests.gpu_util import rand_state, rand_unitary, to_gpu

pytestmark = pytest.mark.gpu


def _finite(t):
    return np.isfinite(t.cpu().numpy().view(np.float32).reshape(-1, 2)).all(axis=1)


def _group(n, qubits, i):
    """Indices that differ from i in the qubits' bits only."""
    m = sum(1 << (n - 1 - q) for q in qubits)
    return (np.arange(1 << n) & ~m) == (i & ~m)


# k = 3 at its smallest, with index bit 0 a target and not, and through LDS; the matrix cores, the
# general kernel (8-byte alignment), and the one- and two-qubit functions
@pytest.mark.parametrize("n,qubits,offset", [
    (3, [2, 0, 1], 0), (4, [0, 1, 2], 0), (12, [11, 0, 5], 0), (12, [3, 0, 5], 0),
    (12, [9, 11, 10], 0), (13, [8, 0, 9], 0), (12, [3, 0, 5], 1), (13, [2, 9, 5, 7], 0),
    (13, [1, 4, 12, 0, 7, 8], 0), (14, [5, 1, 4, 12, 0, 7, 8], 0), (12, [4], 0), (12, [7, 2], 0)])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_unitaries_keep_it_in_one_group(gpu, n, qubits, offset, bad):
    import torch

    from tyxonq_amd import kernels as K

    rng = np.random.default_rng(n)
    v = rand_state(rng, n).astype(np.complex64)
    i = int(rng.integers(1 << n))
    v[i] = bad
    buf = torch.zeros((1 << n) + offset, dtype=torch.complex64, device="cuda")
    src = buf[offset:]
    src.copy_(to_gpu(v))
    U = rand_unitary(rng, 1 << len(qubits))  # (no zero entries)
    out = K.apply_kqubit_unitary(src, U, qubits, n)
    np.testing.assert_array_equal(~_finite(out), _group(n, qubits, i))
