"""k-qubit unitaries on the matrix cores against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import rand_state, rand_unitary, to_gpu, to_np
from oracle import statevector as O

pytestmark = pytest.mark.gpu

# (n, qubits): the smallest tile of each k and one bit below it (general
# kernel), targets lowest, highest, interleaved and in descending order, chunks
# and row blocks of k >= 7, several tiles (19 qubits at k = 4: a work-group each;
# work-groups with several tiles are in test_work_groups_with_several_tiles)
CASES = [
    (3, [2, 0, 1]), (11, [0, 5, 10]), (12, [11, 10, 9]), (12, [0, 1, 2]),
    (11, [3, 1, 9, 4]), (12, [3, 1, 9, 4]), (12, [8, 9, 10, 11]), (19, [0, 18, 7, 3]),
    (12, [11, 0, 6, 3, 9]), (13, [4, 3, 2, 1, 0]), (11, [10, 8, 6, 4, 2]),
    (12, [0, 2, 4, 6, 8, 10]), (13, [12, 11, 10, 9, 8, 7]), (14, [5, 0, 13, 2, 9, 1]),
    (12, [0, 1, 2, 3, 4, 5, 6]), (13, [12, 1, 3, 5, 7, 9, 11]), (14, [0, 13, 1, 12, 2, 11, 3, 10]),
    (15, [14, 0, 2, 4, 6, 8, 10, 12, 13]), (16, [15, 3, 9, 0, 12, 6, 1, 7, 10, 4]),
]


@pytest.mark.parametrize("n,qubits", CASES)
@pytest.mark.parametrize("offset", [0, 1])  # 1: a state at 8-byte alignment (general kernel)
def test_kq_against_oracle(n, qubits, offset):
    import torch

    from tyxonq_amd import kernels as K

    rng = np.random.default_rng(100 * n + len(qubits))
    v, U = rand_state(rng, n), rand_unitary(rng, 1 << len(qubits))
    buf = torch.zeros((1 << n) + offset, dtype=torch.complex64, device="cuda")
    src = buf[offset:]
    src.copy_(to_gpu(v))
    out = to_np(K.apply_kqubit_unitary(src, U, qubits, n))
    ref = O.apply_kqubit(to_np(src), U, qubits, n)
    # unit-norm rows: 2^(k+1) FP32 products and sums of random sign, 2^-24 each
    tol = 4 * 2.0 ** -24 * np.sqrt(2.0 ** len(qubits))
    assert np.linalg.norm(out - ref) <= tol * np.linalg.norm(ref)
    np.testing.assert_array_equal(to_np(src), to_np(to_gpu(v)))


# index bits in each order: one thread's work with bit 0 a target (n = 3) and not
# (n = 4); LDS tiles at two targets below bit 5, one tile and several; bit 5 itself;
# part of a work-group
@pytest.mark.parametrize("n,bits", [
    (3, [0, 1, 2]), (3, [2, 0, 1]), (4, [3, 1, 2]), (4, [0, 3, 2]), (9, [8, 0, 4]),
    (11, [1, 2, 3]), (12, [1, 2, 3]), (12, [0, 11, 4]), (12, [4, 5, 11]), (12, [5, 0, 6]),
    (12, [11, 9, 10]), (15, [14, 4, 3]), (16, [2, 0, 1]), (17, [5, 16, 1]), (18, [17, 3, 10])])
def test_three_targets(n, bits):
    from tyxonq_amd import _native as nat

    rng = np.random.default_rng(n + bits[0])
    v, U = to_gpu(rand_state(rng, n)), rand_unitary(rng, 8)
    ref = O.apply_kqubit(to_np(v), U, [n - 1 - b for b in bits], n)
    # unit-norm rows: 16 FP32 products and sums of random sign, 2^-24 each
    assert np.linalg.norm(to_np(nat.apply_kq(v, bits, U)) - ref) <= 4 * 2.0 ** -24 * np.sqrt(8.0)


# more work than the grid of 1024 (16384 for k = 3): 2 and 4 tiles per work-group,
# U kept in registers over them; k >= 7: 2 tiles and 8 (interleaved over the XCDs),
# and 4 pieces of work per work-group
@pytest.mark.parametrize("n,qubits", [
    (23, [22, 3, 11, 0]), (24, [5, 23, 0, 12, 7]), (24, [23, 1, 8, 22, 15, 4]),
    (14, [13, 0, 6, 2, 9, 11, 4]), (16, [1, 15, 3, 8, 12, 0, 6]),
    (24, [2, 23, 10, 0, 17, 21, 6]), (24, [0, 22, 4, 18, 9, 13, 23, 2]),
    (27, [26, 24, 25])])
def test_work_groups_with_several_tiles(n, qubits):
    import torch

    from tyxonq_amd import kernels as K

    k, rng = len(qubits), np.random.default_rng(n + len(qubits))
    torch.manual_seed(n + k)
    v = torch.randn(1 << n, dtype=torch.complex64, device="cuda") * 2.0 ** (-n / 2)
    U = rand_unitary(rng, 1 << k)
    out = K.apply_kqubit_unitary(v, U, qubits, n)
    # complex128 products in plain torch, 2^22 amplitudes at a time (targets first)
    perm = list(qubits) + [a for a in range(n) if a not in qubits]
    x = v.reshape((2,) * n).permute(perm).reshape(1 << k, -1)
    y = out.reshape((2,) * n).permute(perm).reshape(1 << k, -1)
    Ut, d2, r2 = torch.tensor(U, device="cuda"), 0.0, 0.0
    for xs, ys in zip(x.split(1 << (22 - k), 1), y.split(1 << (22 - k), 1)):
        ref = Ut @ xs.to(torch.complex128)
        d2 += float((ys.to(torch.complex128) - ref).abs().square().sum())
        r2 += float(ref.abs().square().sum())
    assert d2 ** 0.5 <= 4 * 2.0 ** -24 * np.sqrt(2.0 ** k) * r2 ** 0.5


def test_kq_calls_in_flight_on_two_streams():
    """The tables of a call are staged until its kernel has run."""
    import torch

    from tyxonq_amd import kernels as K

    n, rng = 14, np.random.default_rng(3)
    v = to_gpu(rand_state(rng, n))
    Us = [rand_unitary(rng, 64) for _ in range(8)]
    qs = [[int(q) for q in rng.choice(n, 6, replace=False)] for _ in Us]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    outs = []
    for i, (U, q) in enumerate(zip(Us, qs)):
        with torch.cuda.stream(streams[i % 2]):
            outs.append(K.apply_kqubit_unitary(v, U, q, n))
    torch.cuda.synchronize()
    for U, q, out in zip(Us, qs, outs):
        ref = O.apply_kqubit(to_np(v), U, q, n)
        assert np.linalg.norm(to_np(out) - ref) <= 4 * 2.0 ** -24 * 8 * np.linalg.norm(ref)
