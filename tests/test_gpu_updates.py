"""Parameter updates and coefficient changes that are queued, not waited for:
many in flight on two streams, uses on another stream, and under capture."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N, LAYERS = 14, 6


def _rows(seed):
    import tyxonq_amd as tq
    from tyxonq_amd.engine import lower

    rng = np.random.default_rng(seed)
    c = tq.Circuit(N)
    for _ in range(LAYERS):
        for q in range(N):
            c.ry(q, float(rng.normal())).rz(q, float(rng.normal()))
        for q in range(N):
            c.cx(q, (q + 1) % N)
    return lower(c, mode="state")[0].segments[0][1]


def _fresh(seed):
    from tyxonq_amd import _native as nat

    psi = nat.new_state(N, 0)
    nat.Plan(N, _rows(seed)).run(psi)
    return psi


def _ham(scale):
    from tyxonq_amd import _native as nat
    from tyxonq_amd.pauli import PauliSum

    # 8 or more diagonal terms: the diagonal vector is rebuilt with new coefficients
    terms = [(1.0, [("Z", i), ("Z", (i + 1) % N)]) for i in range(N)] + \
        [(1.0, [("X", i)]) for i in range(N)]
    x, z, c = PauliSum(N, terms).to_masks()
    return nat.Ham(N, x, z, scale * np.linspace(0.5, 1.5, len(c))), len(c)


def test_many_updates_in_flight(gpu):
    """More program bytes than the staging ring holds, on two streams."""
    import torch

    from tyxonq_amd import _native as nat

    plans = [nat.Plan(N, _rows(0)) for _ in range(2)]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    outs = []
    for k in range(120):
        with torch.cuda.stream(streams[k % 2]):
            psi = nat.new_state(N, 0)
            plans[k % 2].update(_rows(k % 7))
            plans[k % 2].run(psi)
            outs.append(psi)
    torch.cuda.synchronize()
    ref = [_fresh(s) for s in range(7)]
    for k, psi in enumerate(outs):
        assert torch.equal(psi, ref[k % 7])


def test_update_used_on_another_stream_and_under_capture(gpu):
    import torch

    from tyxonq_amd import _native as nat

    plan = nat.Plan(N, _rows(1))
    ham, nt = _ham(1.0)
    psi, out = nat.new_state(N, 0), nat.new_state(N, 0)
    want = torch.empty_like(out)
    ham2, _ = _ham(-2.0)
    ham2.apply(_fresh(2), want)

    def go():
        nat.init_basis(psi, 0)
        plan.run(psi)
        ham.apply(psi, out)

    go()
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    plan.update(_rows(2))
    ham.set_coeffs(-2.0 * np.linspace(0.5, 1.5, nt))
    with torch.cuda.stream(side):
        go()
    side.synchronize()
    assert torch.equal(out, want)
    plan.update(_rows(2))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        go()
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        psi.normal_()  # eager work between the replays
    with pytest.raises(NotImplementedError):
        with torch.cuda.graph(torch.cuda.CUDAGraph()):
            plan.update(_rows(3))


def test_updates_between_replays_on_another_stream(gpu):
    """A replay passes no host call: updates of a captured plan and Hamiltonian
    are complete when they return."""
    import torch

    from tyxonq_amd import _native as nat

    plan = nat.Plan(N, _rows(0))
    ham, nt = _ham(1.0)
    psi, out = nat.new_state(N, 0), nat.new_state(N, 0)

    def go():
        nat.init_basis(psi, 0)
        plan.run(psi)
        ham.apply(psi, out)

    go()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        go()
    want = []
    for k in range(3):
        w = torch.empty_like(out)
        _ham(1.0 + k)[0].apply(_fresh(k), w)
        want.append(w)
    busy = torch.zeros(1 << 26, device="cuda")
    torch.cuda.synchronize()
    for k in (1, 2, 0, 1):
        with torch.cuda.stream(a):
            for _ in range(20):
                busy.add_(1.0)  # work in front of the copies
            plan.update(_rows(k))
            ham.set_coeffs((1.0 + k) * np.linspace(0.5, 1.5, nt))
        with torch.cuda.stream(b):
            graph.replay()
        b.synchronize()
        assert torch.equal(out, want[k])
    torch.cuda.synchronize()


@pytest.mark.parametrize("count", [0, 1, 7, 8, 40])
def test_update_many(gpu, count):
    """One thread, two threads and eight; a wrong op count fails and says so."""
    from tyxonq_amd import _native as nat

    rows = [_rows(s) for s in range(5)]
    plans = [nat.Plan(N, rows[0]) for _ in range(count)]
    nat.update_plans(plans, [rows[(k + 1) % 5] for k in range(count)])
    ref = [_fresh(s) for s in range(5)]
    for k, p in enumerate(plans):
        psi = nat.new_state(N, 0)
        p.run(psi)
        assert (psi == ref[(k + 1) % 5]).all()
    if count:
        with pytest.raises(ValueError, match="op count"):
            nat.update_plans(plans, [r[:-1] for r in [rows[0]] * count])
        bad = rows[1].copy()
        bad["kind"][3] = 99
        with pytest.raises(ValueError, match="op 3"):
            nat.update_plans(plans, [rows[2]] * (count - 1) + [bad])
        for k, p in enumerate(plans):  # the others are updated, the bad one is as it was
            psi = nat.new_state(N, 0)
            p.run(psi)
            assert (psi == ref[2 if k < count - 1 else (k + 1) % 5]).all()
    if count > 1:
        with pytest.raises(ValueError, match="repeated"):
            nat.update_plans([plans[0], plans[0]], [rows[0], rows[0]])


def test_batch_with_some_generated_plans(gpu, capfd, monkeypatch):
    """Plans that ask for generated kernels, behind one that does not: each
    distinct pass is compiled once."""
    import torch

    import tyxonq_amd as tq
    from tyxonq_amd import _native as nat
    from tyxonq_amd.engine import lower
    from tyxonq_amd.pauli import PauliSum

    n, count = 6, 12
    t = [torch.tensor(0.1 * q + 0.05, requires_grad=True) for q in range(n)]
    c = tq.Circuit(n)
    for q in range(n):
        c.ry(q, t[q])
    for q in range(n - 1):
        c.cx(q, q + 1)
    rows = lower(c, track_grad=True)[0].segments[0][1]
    ham = nat.Ham(n, *PauliSum(n, [(1.0, [("Z", q), ("X", (q + 1) % n)]) for q in range(n)]
                               + [(0.5, [("Z", q)]) for q in range(n)]).to_masks())
    monkeypatch.setenv("TQSV_JIT_VERBOSE", "1")
    res = []
    for jit in ([-1] * count, [-1] + [1] * (count - 1)):
        plans = [nat.Plan(n, rows, jit=j, min_qubits=nat.BATCH_QUBITS) for j in jit]
        capfd.readouterr()
        psis = [nat.new_state(n, 0) for _ in plans]
        res += nat.Batch().adjoint(plans, [ham] * count, psis, [n] * count)
        lines = [x.split("(hiprtc")[0] for x in capfd.readouterr().err.splitlines()
                 if x.startswith("tqsv jit: pass") and "mode 2" in x]
        assert len(lines) == len(set(lines))  # (one state tile: passes differ in their place)
    for e, g in res[1:]:
        assert e == res[0][0] and np.array_equal(g, res[0][1])
