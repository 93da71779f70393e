"""Chains of stochastic channels and <Z> of every qubit against numpy."""
from __future__ import annotations

import math

import numpy as np
import pytest

from gpu_util import rand_state, to_gpu, to_np
from oracle import statevector as O

pytestmark = pytest.mark.gpu


def damping(g):
    return [np.array([[1, 0], [0, math.sqrt(1 - g)]], dtype=complex),
            np.array([[0, math.sqrt(g)], [0, 0]], dtype=complex)]


def depolarizing(p):
    P = [np.eye(2), np.array([[0, 1], [1, 0]]), np.array([[0, -1j], [1j, 0]]), np.diag([1, -1])]
    return [math.sqrt(w) * m.astype(complex) for w, m in zip([1 - p] + [p / 3] * 3, P)]


def reference(v, n, chain):
    for bit, ks, status in chain:
        cand = [O.apply_1q(v, K, n - 1 - bit, n) for K in ks]
        w = np.array([np.linalg.norm(c) ** 2 for c in cand])
        hit = np.nonzero(status <= np.cumsum(w / w.sum()))[0]
        sel = int(hit[0]) if len(hit) else 0
        v = cand[sel] / math.sqrt(w[sel]) if w[sel] > 0 else cand[sel]
    return v


# n = 1: no second bit; 2: one quad; 12, 13: one block and two; 17: several
# quads per thread; bits ascending, descending, repeated in a row
@pytest.mark.parametrize("n,bits", [
    (1, [0, 0, 0]), (2, [1, 0, 0, 1]), (5, [0, 4, 4, 2]), (12, list(range(12))),
    (13, [12, 0, 11, 1, 1]), (17, [16, 3, 9, 0, 16])])
def test_chain(n, bits):
    from tyxonq_amd import _native as nat

    rng = np.random.default_rng(n)
    v = to_gpu(rand_state(rng, n))
    # complex and non-diagonal operators as well
    H = np.array([[1, 1], [1, -1]]) / math.sqrt(2)
    S = np.diag([1, 1j])
    kinds = [damping(0.4), depolarizing(0.6), [H @ K @ S for K in damping(0.7)]]
    chain = [(b, kinds[j % 3], float(rng.random())) for j, b in enumerate(bits)]
    ref = reference(to_np(v), n, chain)
    nat.kraus_chain(v, chain)
    # per channel a 2x2 product and a scale in FP32
    assert np.linalg.norm(to_np(v) - ref) <= (len(bits) + 1) * 4 * 2.0 ** -24
    assert abs(np.linalg.norm(to_np(v)) - 1.0) <= 2.0 ** -23


def test_chain_edges():
    import torch

    from tyxonq_amd import _native as nat

    # no operator reaches the random number: the first one, as the reference
    v = to_gpu(rand_state(np.random.default_rng(1), 6))
    ref = reference(to_np(v), 6, [(2, damping(0.3), 1.5)])
    nat.kraus_chain(v, [(2, damping(0.3), 1.5)])
    assert np.linalg.norm(to_np(v) - ref) <= 8 * 2.0 ** -24
    # a zero state stays zero
    z = torch.zeros(64, dtype=torch.complex64, device="cuda")
    nat.kraus_chain(z, [(0, damping(0.3), 0.5), (1, damping(0.3), 0.5)])
    assert not z.any()
    with pytest.raises(ValueError):
        nat.kraus_chain(v, [(6, damping(0.3), 0.5)])
    with pytest.raises(ValueError):
        nat.kraus_chain(v, [(0, [], 0.5)])


def test_operators_of_another_size_are_refused():
    """Nothing is cut off or made up: the state stays as it is."""
    from tyxonq_amd import _native as nat

    v = to_gpu(rand_state(np.random.default_rng(2), 6))
    before = to_np(v)
    for bad in (np.eye(4), np.eye(3), np.eye(1)):
        with pytest.raises(ValueError, match="2x2"):
            nat.kraus_chain(v, [(0, [np.eye(2), bad], 0.5)])
    np.testing.assert_array_equal(to_np(v), before)


def test_long_tables_are_given_back():
    """16 MiB of operators on the device; what stays is bounded by a 10-qubit
    matrix (8 MiB) in each of two slots, filled here first."""
    import torch

    from tyxonq_amd import _native as nat

    v = to_gpu(rand_state(np.random.default_rng(4), 10))
    for _ in range(2):
        nat.apply_kq(v, list(range(10)), np.eye(1 << 10))
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    # 2^18 operators of weight 1e-18, then the identity, which is chosen
    ks = [np.array([[0, 1], [1, 0]]) * 1e-9] * (1 << 18) + [np.eye(2)]
    want = to_np(v)
    for _ in range(2):
        nat.kraus_chain(v, [(3, ks, 0.5)])
    torch.cuda.synchronize()
    assert np.linalg.norm(to_np(v) - want) <= 8 * 2.0 ** -24
    assert free - torch.cuda.mem_get_info()[0] <= 4 << 20


# below, at and above one chunk, several blocks, and chunks beyond the grid
@pytest.mark.parametrize("n", [1, 7, 12, 13, 18, 25])
def test_expect_z_all(n):
    from tyxonq_amd import _native as nat

    v = to_gpu(rand_state(np.random.default_rng(n), n)) if n < 20 else nat.new_state(n, 0)
    if n >= 20:  # a product state: <Z> = cos a per qubit
        for b in range(n):
            a = 0.1 * b
            nat.apply_1q(v, b, np.array([[math.cos(a / 2), -math.sin(a / 2)],
                                         [math.sin(a / 2), math.cos(a / 2)]]))
        # n rotations in FP32
        np.testing.assert_allclose(nat.expect_z_all(v), np.cos(0.1 * np.arange(n)),
                                   atol=n * 2.0 ** -23)
        return
    p = np.abs(to_np(v)) ** 2
    idx = np.arange(1 << n)
    ref = [np.sum(p * (1 - 2 * ((idx >> b) & 1))) for b in range(n)]
    np.testing.assert_allclose(nat.expect_z_all(v), ref, atol=1e-12)  # FP64 products and sums


@pytest.mark.parametrize("n", [1, 5, 13])
def test_run_with_one_and_with_every_qubit_measured(n):
    """The same values from the reduction of one qubit and the sweep of all."""
    import tyxonq_amd as tq
    from tyxonq_amd.engine import StatevectorEngine

    def run(measured):
        c = tq.Circuit(n)
        for q in range(n):
            c.ry(q, 0.3 + 0.2 * q)
        for q in measured:
            c.measure_z(q)
        return StatevectorEngine().run(c, shots=0)["expectations"]

    every = run(range(n))
    for q in range(n):
        one = run([q, q])
        assert list(one) == [f"Z{q}"]
        # FP64 sums of the same probabilities; n rotations in FP32
        assert one[f"Z{q}"] == pytest.approx(every[f"Z{q}"], abs=1e-12)
        assert one[f"Z{q}"] == pytest.approx(math.cos(0.3 + 0.2 * q), abs=n * 2.0 ** -23)
