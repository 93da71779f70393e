"""Tensors that torch conjugates or negates lazily (a flag on the same memory):
the kernel functions and their gradients against plain torch in complex128."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import statevector as O
from tests.gpu_util import rand_state, rand_unitary, to_gpu, to_np

pytestmark = pytest.mark.gpu

N = 6
# products and sums of unit-norm rows in FP32, forward and backward
TOL = 16 * 2.0 ** -24


def _apply(K, psi, U, qs):
    if len(qs) == 1:
        return K.apply_1q_statevector(None, psi, U, qs[0], N)
    if len(qs) == 2:
        return K.apply_2q_statevector(None, psi, U, qs[0], qs[1], N)
    return K.apply_kqubit_unitary(psi, U, qs, N)


def _dense(U, qs):
    """The full 2^N matrix of U on qs."""
    return np.stack([O.apply_kqubit(e, U, qs, N) for e in np.eye(1 << N)], axis=1)


def _view(v, view):
    """A lazy view and its values: conj, neg, or both."""
    c, t = np.asarray(v, dtype=np.complex64), to_gpu(v)
    if view != "neg":
        c, t = c.conj(), t.conj()
    if view != "conj":
        c, t = -c, torch._neg_view(t)
    assert t.is_conj() == (view != "neg") and t.is_neg() == (view != "conj")
    return t, c.astype(np.complex128)


@pytest.mark.parametrize("view", ["conj", "neg", "both"])
@pytest.mark.parametrize("qs", [[2], [4, 1], [5, 0, 3], [0, 2, 3, 5]])
def test_states_given_as_lazy_views(gpu, qs, view):
    from tyxonq_amd import kernels as K

    rng = np.random.default_rng(len(qs))
    U = rand_unitary(rng, 1 << len(qs))
    t, v = _view(rand_state(rng, N), view)
    out = _apply(K, t, U, qs)
    assert np.linalg.norm(to_np(out) - O.apply_kqubit(v, U, qs, N)) <= TOL
    # <Z> itself does not see the conjugation; its gradient 2 Z psi does
    s = t.clone().conj() if view == "conj" else t
    s = s.detach().requires_grad_()
    x = (s.conj() if view == "conj" else s)
    z = 1.0 - 2.0 * ((np.arange(1 << N) >> 2) & 1)
    e = K.expect_z_statevector(x, N - 1 - 2, N)
    assert abs(e.item() - float(np.sum(z * np.abs(v) ** 2))) <= 1e-12 + 4 * 2.0 ** -24
    e.backward()
    want = 2 * z * to_np(s)
    assert np.linalg.norm(to_np(s.grad) - want) <= TOL


LOSSES = {
    "conj_sum": lambda o, t: (o.conj() * t).sum(),
    "dot": lambda o, t: torch.dot(o.conj(), t),
    "einsum": lambda o, t: torch.einsum("i,i->", o.conj(), t),
    "matmul": lambda o, t: t @ o.conj(),
    "plain": lambda o, t: (o * t).sum(),
}


@pytest.mark.parametrize("loss", sorted(LOSSES))
@pytest.mark.parametrize("qs", [[2], [4, 1], [5, 0, 3]])
def test_gradients_with_conjugated_cotangents(gpu, qs, loss):
    from tyxonq_amd import kernels as K

    rng = np.random.default_rng(7 + len(qs))
    v, tv, U = rand_state(rng, N), rand_state(rng, N), rand_unitary(rng, 1 << len(qs))

    s = to_gpu(v).requires_grad_()
    g = torch.tensor(U, device="cuda", requires_grad=True)
    LOSSES[loss](_apply(K, s, g, qs), to_gpu(tv)).real.backward()

    s0 = torch.tensor(v.astype(np.complex64).astype(np.complex128), requires_grad=True)
    t0 = torch.tensor(tv.astype(np.complex64).astype(np.complex128))
    rows = torch.tensor(_dense(U, qs))
    LOSSES[loss](rows @ s0, t0).real.backward()
    assert np.linalg.norm(to_np(s.grad) - s0.grad.numpy()) <= TOL

    # gate gradient: g psi^dagger over the other qubits
    gout = torch.autograd.grad(LOSSES[loss](x := (rows @ s0).detach().requires_grad_(), t0).real, x)
    rest = [q for q in range(N) if q not in qs]

    def by_target(a):
        a = a.resolve_conj().numpy().reshape((2,) * N)
        return np.transpose(a, list(qs) + rest).reshape(1 << len(qs), -1)

    want = by_target(gout[0]) @ by_target(s0.detach()).conj().T
    assert np.linalg.norm(to_np(g.grad) - want) <= TOL


def test_expectation_with_a_negated_cotangent(gpu):
    """The imaginary part of a conjugated product hands a lazy negation down."""
    from tyxonq_amd import kernels as K

    v = rand_state(np.random.default_rng(3), N)
    s = to_gpu(v).requires_grad_()
    za, zb = K.expect_z_statevector(s, 0, N), K.expect_z_statevector(s, 1, N)
    w = (torch.complex(za, zb).conj() * (1.0 + 2.0j)).real  # za + 2 zb
    w.backward()
    idx = np.arange(1 << N)
    z = [1.0 - 2.0 * ((idx >> (N - 1 - q)) & 1) for q in (0, 1)]
    want = 2 * (z[0] + 2 * z[1]) * to_np(s)
    assert np.linalg.norm(to_np(s.grad) - want) <= TOL * np.linalg.norm(want)


def test_raw_entry_points_refuse_lazy_views(gpu):
    from tyxonq_amd import _native as nat
    from tyxonq_amd import kernels as K

    v, U = rand_state(np.random.default_rng(4), N), np.eye(2)
    for view in ("conj", "neg"):
        t, _ = _view(v, view)
        before = to_np(t)
        for call in (lambda: nat.apply_1q(t, 0, U), lambda: nat.dot(t, t), lambda: nat.norm2(t),
                     lambda: K.apply_1q_statevector_(t, U, 0, N),
                     lambda: K.apply_2q_statevector_(t, np.eye(4), 0, 1, N)):
            with pytest.raises(ValueError, match="lazy|lazily"):
                call()
        np.testing.assert_array_equal(to_np(t), before)
        # converted states are written out on the way
        for u in (t.cpu(), t.to(torch.complex128)):
            out = K.apply_1q_statevector_(u, U, 0, N)
            np.testing.assert_array_equal(to_np(out), before)
    with pytest.raises(ValueError, match="lazy"):
        nat.z_grad(to_gpu(v), 0, torch._neg_view(torch.ones((), dtype=torch.float64, device="cuda")))
