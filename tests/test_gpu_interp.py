"""The interpreting tile-pass kernel: every slot bit, slot pair and flip mask of
a phase (lane bits and register bits), forward and adjoint, vs the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import statevector as O
from tests.gpu_util import (dense_apply_items, ops_from_items, rand_state, rand_unitary,
                            random_matrix_items, random_pauli_terms, to_gpu, to_np)

pytestmark = pytest.mark.gpu


# tile sizes with 256, 512 and 1024 threads, and 1024 threads in two turns; 0: automatic
@pytest.mark.parametrize("n,tile", [(11, 11), (12, 0), (13, 11), (13, 12), (13, 13), (14, 14),
                                    (15, 0), (15, 14)])
def test_matrices_on_all_slot_pairs(gpu, n, tile):
    from tyxonq_amd import _native as nat

    rng = np.random.default_rng(10 * n + tile)
    bits = [int(b) for b in rng.choice(n, 5, replace=False)]
    items = []
    for a in bits:
        for b in bits:
            if a != b:
                items.append(("m2", a, b, rand_unitary(rng, 4)))
        c = 1 << int(rng.choice([x for x in range(n) if x != n - 1 - a]))
        items.append(("m1", a, rand_unitary(rng, 2), c, c))
    items += random_matrix_items(rng, n, 40)
    v = rand_state(rng, n)
    psi = to_gpu(v)
    nat.Plan(n, ops_from_items(n, items), tile_bits=tile).run(psi)
    want = dense_apply_items(n, items, v)
    # about 70 gates, each rounding at 2^-24 of the norm a few times
    assert np.linalg.norm(to_np(psi) - want) <= 70 * 4 * 2.0 ** -24 * np.linalg.norm(want)


@pytest.mark.parametrize("n,tile", [(13, 0), (13, 11), (13, 12), (14, 13), (14, 0), (6, 0)])
def test_adjoint_over_all_flip_masks(gpu, n, tile):
    """(13, 0) and (6, 0) run in the batch kernel, the others as dual passes."""
    import torch

    import tyxonq_amd as tq

    rng = np.random.default_rng(n + 100 * tile)
    qs = [int(q) for q in rng.choice(n, 5, replace=False)]
    strings, groups = [], []
    for x in range(32):
        flip = [(("X", "Y")[int(rng.integers(2))], q) for j, q in enumerate(qs) if (x >> j) & 1]
        rest = [("Z", q) for q in range(n) if q not in [f[1] for f in flip] and rng.random() < 0.4]
        if flip or rest:
            strings.append(flip + rest)
        if len(flip) >= 2:  # a commuting partner: two letters exchanged, one rotation group
            other = [("Y" if P == "X" else "X", q) if k < 2 else (P, q)
                     for k, (P, q) in enumerate(flip)]
            groups.append((flip + rest, other + rest))

    def build(p):
        ops = [("ry", q, 0.3 + 0.1 * q) for q in range(n)]
        for k, s in enumerate(strings):
            ops.append(("pauli_rot", tuple(s), p[k]))
        for k, (s, t) in enumerate(groups):
            ops.append(("pauli_rot", tuple(s), p[len(strings) + k]))
            ops.append(("pauli_rot", tuple(t), p[len(strings) + k]))
        return ops

    from tyxonq_amd import _native as nat
    from tyxonq_amd.engine import lower
    from tyxonq_amd.pauli import PauliSum

    ns, ng = len(strings), len(groups)
    th = rng.normal(0.0, 0.7, ns + ng)
    terms = random_pauli_terms(rng, n, 20, maxw=3)
    t = [torch.tensor(v, requires_grad=True) for v in th]
    rows = lower(tq.Circuit(n, ops=build(t)), track_grad=True)[0].segments[0][1].copy()
    # the lowering numbers parameters by op: give the two members of a group one
    rows["param"][n:] = list(range(ns)) + [ns + k for k in range(ng) for _ in range(2)]
    rows["param"][:n] = -1
    batch = tile == 0 and n <= nat.BATCH_QUBITS
    plan = nat.Plan(n, rows, tile_bits=tile, min_qubits=nat.BATCH_QUBITS if batch else 0)
    ham = nat.Ham(n, *PauliSum(n, terms).to_masks())
    psi = nat.new_state(n, 0)
    if batch:
        e, g = nat.Batch().adjoint([plan], [ham], [psi], [ns + ng])[0]
    else:
        e, g = plan.adjoint(ham, psi, torch.empty_like(psi), ns + ng)

    def f(p):
        return O.pauli_sum_expectation(O.simulate(n, build(p))[0], terms, n)

    assert abs(e - f(th)) < 1e-5
    idx = list(range(0, len(th), 3))
    # complex128 differences: (h^2 / 6) |E'''| ~ 1e-7 at h = 1e-3 and 20 terms
    np.testing.assert_allclose(g[idx], O.central_fd_gradient(f, th, h=1e-3, indices=idx), atol=2e-5)
