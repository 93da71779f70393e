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


# the interpreting passes: every slot bit of a phase as target (lane and register
# bits), one tile and two
@pytest.mark.parametrize("n,tile", [(12, 12), (12, 11)])
@pytest.mark.parametrize("kind", ["real", "rxlike", "controlled"])
def test_real_matrices_keep_infinite_parts_apart(gpu, n, tile, kind):
    import torch

    from tests.gpu_util import ops_from_items
    from tyxonq_amd import _native as nat

    m = np.array([[1.5, 0.25], [-0.5, 2.0]])
    if kind == "rxlike":
        m = np.array([[1.5, 0.25j], [-0.5j, 2.0]])
    rng = np.random.default_rng(n)
    for q in range(n):
        v = rand_state(rng, n).astype(np.complex64)
        i = 0  # the control's value holds
        v[i] = complex(np.inf, 1.0)
        c = 1 << (n - 1 - (q + 1) % n) if kind == "controlled" else 0
        psi = to_gpu(v)
        nat.Plan(n, ops_from_items(n, [("m1", q, m, c, 0)]), tile_bits=tile, jit=-1).run(psi)
        out = torch.view_as_real(psi).cpu().numpy()
        j = 1 << (n - 1 - q)
        want = np.zeros((1 << n, 2), dtype=bool)
        want[i, 0] = want[j, 1 if kind == "rxlike" else 0] = True
        np.testing.assert_array_equal(~np.isfinite(out), want)


@pytest.mark.parametrize("tile", [11, 12])
@pytest.mark.parametrize("lo", range(5))
def test_rotation_groups_leave_other_patterns_alone(gpu, lo, tile):
    """A single excitation turns the patterns 01 and 10 into each other: an
    infinity at 00 or 11 stays where it is, and out of the gradient."""
    import torch

    import tyxonq_amd as tq
    from tyxonq_amd import _native as nat
    from tyxonq_amd.engine import lower

    n, th = 12, 0.7
    rng = np.random.default_rng(lo)
    a, b = n - 1 - lo, int(rng.choice([q for q in range(n) if q != n - 1 - lo]))
    t = [torch.tensor(x, requires_grad=True) for x in (th, -th)]
    rows = lower(tq.Circuit(n, ops=[("pauli_rot", (("X", a), ("Y", b)), t[0]),
                                    ("pauli_rot", (("Y", a), ("X", b)), t[1])]),
                 track_grad=True)[0].segments[0][1].copy()
    rows["param"] = 0  # one parameter, +- its value
    rows["gcoef"][1] *= -1
    plan = nat.Plan(n, rows, tile_bits=tile, jit=-1)
    for pattern in (0, 3):
        v = rand_state(rng, n).astype(np.complex64)
        lam = rand_state(rng, n).astype(np.complex64)
        bits = (1 << (n - 1 - a)) | (1 << (n - 1 - b))
        i = (int(rng.integers(1 << n)) & ~bits) | (bits if pattern else 0)
        ref = v.copy()
        v[i] = complex(np.inf, np.nan)
        psi = to_gpu(v)
        plan.run(psi)
        np.testing.assert_array_equal(np.nonzero(~_finite(psi))[0], [i])
        want = to_gpu(ref)
        plan.run(want)
        g = plan.vjp(psi, to_gpu(lam), 1)
        assert np.isfinite(g).all()
        # the patterns 00 and 11 have no part in the generator
        np.testing.assert_allclose(g, plan.vjp(want, to_gpu(lam), 1), rtol=0, atol=1e-7)
