"""Timed cases of the statevector framework: one pass each through its public
entry points, with inputs made from a seed and results in complex128 computed
here with plain torch / numpy.

Kinds of case (sizes below are the listed ones; `draw` spreads each kind over
its range):

  hea          a small variational step through Circuit and the engine
  serve_batch  many small energy+gradient requests in one batched launch
  serve        one mid-size energy+gradient request of the server
  vqe          an optimiser step on a kept plan: new angles, energy, gradient
  brickwork    a deep circuit on a large state and a Pauli-sum expectation
  qaoa         a circuit's state and its vector-Jacobian product (torch)
  ucc          a UCCSD energy and gradient through the chemistry runtime
  trajectory   one noise trajectory (Kraus ops) and <Z> of every qubit
  sample       shots from a state
  density      a noisy density matrix
  kq           a k-qubit unitary on a state
  gates        the kernel functions with gradients for state and gates
"""
from __future__ import annotations

import math

import numpy as np
import torch

SQ = 1.0 / math.sqrt(2.0)


def listed():
    return [
        # a 12-qubit hardware-efficient ansatz, open TFIM: the smallest
        # variational step, where latency and host work count
        {"name": "hea_12q", "kind": "hea", "n": 12, "layers": 4},
        # the server's batch lane: 48 requests of 2-13 qubits, depths 2-16
        {"name": "serve_batch_48", "kind": "serve_batch", "count": 48, "dmax": 16},
        # a mid-size request of the server (no kernels compiled for it)
        {"name": "serve_18q", "kind": "serve", "n": 18, "depth": 8, "ham": "heisenberg"},
        # 22 qubits x 12 RY/RZ/CX-ring layers, Heisenberg ring: one optimiser step
        {"name": "vqe_22q", "kind": "vqe", "n": 22, "layers": 12},
        # 30-qubit brickwork, 20 layers, and a 500-term 2-local Pauli sum
        {"name": "brickwork_30q", "kind": "brickwork", "n": 30, "layers": 20, "terms": 500},
        # a QAOA state on a random graph, differentiated through torch
        {"name": "qaoa_20q", "kind": "qaoa", "n": 20, "layers": 4},
        # UCCSD on 14 spin orbitals (7 spatial, 6 electrons)
        {"name": "ucc_14so", "kind": "ucc", "ns": 7, "no": 3},
        # a quantum trajectory: 3 layers with amplitude damping on every qubit
        {"name": "trajectory_20q", "kind": "trajectory", "n": 20, "layers": 3,
         "channel": "amplitude_damping"},
        # counts: 10^5 shots from a 26-qubit state
        {"name": "sample_26q", "kind": "sample", "n": 26, "shots": 100000},
        # a noisy 10-qubit density matrix (a 20-qubit vec(rho)), per-gate depolarizing
        {"name": "density_10q", "kind": "density", "n": 10, "layers": 3, "noise": "depolarizing"},
        # a dense 6-qubit unitary (state preparation, block encodings) on 24 qubits
        {"name": "kq6_24q", "kind": "kq", "n": 24, "k": 6},
        # the kernel functions, one layer of gates with gradients on 20 qubits
        {"name": "gates_20q", "kind": "gates", "n": 20, "layers": 1},
    ]


def draw(rng):
    def logint(a, b):
        return max(a, min(b, int(round(math.exp(rng.uniform(math.log(a), math.log(b + 0.49)))))))

    kind = rng.choice(["hea", "serve_batch", "serve", "vqe", "brickwork", "qaoa", "ucc",
                       "trajectory", "sample", "density", "kq", "gates"])
    if kind == "hea":
        return {"kind": kind, "n": rng.randint(2, 16), "layers": rng.randint(1, 8)}
    if kind == "serve_batch":
        return {"kind": kind, "count": logint(1, 200), "dmax": rng.randint(3, 16)}
    if kind == "serve":
        return {"kind": kind, "n": rng.randint(14, 24), "depth": rng.randint(2, 12),
                "ham": rng.choice(["tfim", "heisenberg"])}
    if kind == "vqe":
        return {"kind": kind, "n": rng.randint(22, 24), "layers": rng.randint(2, 4)}
    if kind == "brickwork":
        return {"kind": kind, "n": rng.randint(22, 28), "layers": rng.randint(3, 8),
                "terms": logint(20, 200)}
    if kind == "qaoa":
        return {"kind": kind, "n": rng.randint(8, 21), "layers": rng.randint(1, 6)}
    if kind == "ucc":
        ns = rng.randint(4, 8)
        return {"kind": kind, "ns": ns, "no": rng.randint(2, max(2, ns // 2))}
    if kind == "trajectory":
        return {"kind": kind, "n": rng.randint(8, 24), "layers": rng.randint(1, 3),
                "channel": rng.choice(["amplitude_damping", "depolarizing"])}
    if kind == "sample":
        return {"kind": kind, "n": rng.randint(10, 28), "shots": logint(1000, 1000000)}
    if kind == "density":
        return {"kind": kind, "n": rng.randint(3, 10), "layers": rng.randint(1, 4),
                "noise": rng.choice(["depolarizing", "amplitude_damping"])}
    if kind == "kq":
        k = rng.randint(3, 10)
        return {"kind": kind, "n": rng.randint(max(k, 10), min(27, 32 - k)), "k": k}
    return {"kind": kind, "n": rng.randint(6, 23), "layers": rng.randint(1, 2)}


# ---- inputs (plain data, used by prepare and by exact) -------------------------

def _rng(seed):
    return np.random.default_rng(seed)


def _state(n, seed, dtype=torch.complex64, tilt=False):
    """A normalised random state (complex64 values, also for `exact`); with
    `tilt` its qubits lean towards |0> or |1>, so that <Z> is of order one."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    v = torch.randn(1 << n, 2, generator=g, device="cuda", dtype=torch.float32)
    v /= math.sqrt(2.0 ** (n + 1))
    if tilt:
        for q, a in enumerate(_rng(seed).uniform(0.0, 0.5 * math.pi, n)):
            w = v.view(1 << q, 2, -1)
            w[:, 0] *= math.sqrt(2.0) * math.cos(a)
            w[:, 1] *= math.sqrt(2.0) * math.sin(a)
    return torch.view_as_complex(v).to(dtype)


def _unitary(rng, d):
    q, r = np.linalg.qr(rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d)))
    return q * (np.diag(r) / np.abs(np.diag(r)))


def _tfim(n, g=1.0):
    return [(-1.0, [("Z", i), ("Z", i + 1)]) for i in range(n - 1)] + \
        [(-g, [("X", i)]) for i in range(n)]


def _heisenberg(n, hz=0.5):
    t = [(1.0, [(P, i), (P, (i + 1) % n)]) for i in range(n) for P in "XYZ"]
    return t + [(hz, [("Z", i)]) for i in range(n)]


def _ring_ops(n, layers, th):
    """RY and RZ on every qubit, CX(q, q+1 mod n) per layer: (name, qubits, angle)."""
    ops, k = [], 0
    for _ in range(layers):
        for name in ("ry", "rz"):
            for q in range(n):
                ops.append((name, (q,), th[k]))
                k += 1
        ops += [("cx", (q, (q + 1) % n), None) for q in range(n)]
    return ops


def _requests(case, seed):
    """(n, depth, ham, g, angles) of a server case."""
    r = _rng(seed)
    if case["kind"] == "serve":
        dims = [(case["n"], case["depth"], case["ham"])]
    else:
        # the mix of sizes is the case's, so that every seed is the same work
        s = _rng(7919 + case["count"])
        dims = [(int(s.integers(2, 14)), int(s.integers(2, case["dmax"] + 1)),
                 "tfim" if s.random() < 0.5 else "heisenberg") for _ in range(case["count"])]
    return [(n, d, h, float(r.uniform(0.5, 1.5)), r.uniform(0.0, 2.0 * math.pi, 2 * n * d))
            for n, d, h in dims]


def _brickwork(case, seed):
    """Trotter-like angles in (-pi/2, pi/2); the Pauli strings are the problem's
    (the same for every seed), coefficients ~ N(0, 1)."""
    n, r = case["n"], _rng(seed)
    ang = r.uniform(-1.5, 1.5, size=(case["layers"], 2, n))
    ops = []
    for l in range(case["layers"]):
        for q in range(n):
            ops += [("rx", (q,), ang[l, 0, q]), ("rz", (q,), ang[l, 1, q])]
        ops += [("cz", (i, i + 1), None) for i in range(l % 2, n - 1, 2)]
    s = _rng(100003 + case["terms"])
    strings = []
    for _ in range(case["terms"]):
        i, j = sorted(int(v) for v in s.choice(n, 2, replace=False))
        strings.append((("XYZ"[int(s.integers(3))], i), ("XYZ"[int(s.integers(3))], j)))
    return ops, strings, r.normal(size=case["terms"])


def _qaoa(case, seed):
    """A random 3-regular-like graph (fixed per size), shared angles per layer,
    and the cotangent of the state."""
    n, L = case["n"], case["layers"]
    s = _rng(5000 + n)
    edges = sorted({tuple(sorted((i, int((i + d) % n)))) for d in (1, int(s.integers(2, n // 2 + 1)))
                    for i in range(n) if (i + d) % n != i})
    r = _rng(seed)
    return edges, r.normal(0.0, 0.4, L), r.normal(0.0, 0.4, L)


def _channel(name):
    if name == "amplitude_damping":
        g = 0.08
        return [np.array([[1, 0], [0, math.sqrt(1 - g)]], dtype=complex),
                np.array([[0, math.sqrt(g)], [0, 0]], dtype=complex)]
    p = 0.06
    return [math.sqrt(1 - p) * np.eye(2, dtype=complex), math.sqrt(p / 3) * PAULI["X"],
            math.sqrt(p / 3) * PAULI["Y"], math.sqrt(p / 3) * PAULI["Z"]]


def _trajectory(case, seed):
    n, r = case["n"], _rng(seed)
    ops = []
    for _ in range(case["layers"]):
        ops += [("ry", (q,), float(v)) for q, v in enumerate(r.normal(0.0, 0.6, n))]
        ops += [("cx", (q, q + 1), None) for q in range(n - 1)]
        ops += [("kraus", (q,), float(v)) for q, v in enumerate(r.random(n))]
    return ops


def _density(case, seed):
    n, r = case["n"], _rng(seed)
    ops = []
    for _ in range(case["layers"]):
        for q in range(n):
            ops += [("rx", (q,), float(r.uniform(-1.5, 1.5))), ("rz", (q,), float(r.uniform(-1.5, 1.5)))]
        ops += [("cx", (q, q + 1), None) for q in range(n - 1)]
    return ops


def _noise(case):
    return {"type": "depolarizing", "p": 0.01} if case["noise"] == "depolarizing" else \
        {"type": "amplitude_damping", "gamma": 0.02}


def _kq(case, seed):
    r = _rng(seed)
    return _unitary(r, 1 << case["k"]), [int(q) for q in r.choice(case["n"], case["k"], replace=False)]


def _gates(case, seed):
    """Per layer a random 1-qubit gate on every second qubit and a random
    2-qubit gate on a brick of neighbours."""
    n, r = case["n"], _rng(seed)
    one, two = [], []
    for l in range(case["layers"]):
        one += [(q, _unitary(r, 2)) for q in range(l % 2, n, 2)]
        two += [((q, q + 1), _unitary(r, 4)) for q in range(l % 2, n - 1, 4)]
    return one, two


_UCC = {}


def _ucc_problem(ns, no):
    """Spin-orbital Hamiltonian and excitations of a synthetic molecule."""
    if (ns, no) not in _UCC:
        from tyxonq_amd import chem

        h, g = chem.synthetic_integrals(ns, 1234)
        n = 2 * ns
        terms = [(c, [(P, n - 1 - q) for P, q in f]) for c, f in chem.molecular_hamiltonian(h, g)]
        _UCC[ns, no] = (terms,) + tuple(chem.uccsd_excitations(no, ns - no))
    return _UCC[ns, no]


def _theta_ucc(case, seed):
    ids = _ucc_problem(case["ns"], case["no"])[2]
    return _rng(seed).normal(0.0, 0.05, max(ids) + 1)


# ---- prepare and run -----------------------------------------------------------

def _circuit(n, ops, circ=None):
    """A Circuit of (name, qubits, angle) ops."""
    import tyxonq_amd as tq

    c = circ or tq.Circuit(n)
    for name, qs, th in ops:
        getattr(c, name)(*qs) if th is None else getattr(c, name)(*qs, th)
    return c


def _lowered(n, ops):
    """Op rows with one parameter per angle, as the engine lowers a circuit."""
    from tyxonq_amd.engine import lower

    t = [torch.tensor(th, dtype=torch.float64, requires_grad=True) if th is not None else None
         for _, _, th in ops]
    c = _circuit(n, [(a, q, v) for (a, q, _), v in zip(ops, t)])
    return lower(c, track_grad=True)[0].segments[0][1]


def prepare(case, seed):
    from tyxonq_amd import _native as nat

    kind = case["kind"]
    s = {"kind": kind, "case": case}
    if kind == "hea":
        from tyxonq_amd.engine import StatevectorEngine

        s["theta"] = _rng(seed).uniform(0.0, 2.0 * math.pi, case["n"] * case["layers"])
        s["terms"] = _tfim(case["n"])
        s["engine"] = StatevectorEngine("pytorch")
    elif kind in ("serve", "serve_batch"):
        from tyxonq_amd import serving

        s["reqs"] = [serving.Request(i, n, d, h, g, th)
                     for i, (n, d, h, g, th) in enumerate(_requests(case, seed))]
        s["cache"] = serving.Cache()
    elif kind == "vqe":
        n = case["n"]
        th = _rng(seed).normal(0.0, 0.3, 2 * n * case["layers"])
        s["ops"] = _lowered(n, _ring_ops(n, case["layers"], th))
        s["plan"] = nat.Plan(n, s["ops"])
        s["ham"] = _native_ham(n, _heisenberg(n))
        s["psi"] = nat.new_state(n, 0)
        s["lam"] = torch.empty_like(s["psi"])
    elif kind == "brickwork":
        n = case["n"]
        ops, strings, coef = _brickwork(case, seed)
        from tyxonq_amd.engine import lower

        s["plan"] = nat.Plan(n, lower(_circuit(n, [(a, q, None if t is None else float(t))
                                                   for a, q, t in ops]))[0].segments[0][1])
        s["ham"] = _native_ham(n, [(c, list(t)) for c, t in zip(coef, strings)])
        s["psi"] = nat.new_state(n, 0)
    elif kind == "qaoa":
        s["edges"], s["gamma"], s["beta"] = _qaoa(case, seed)
        s["cot"] = _state(case["n"], seed + 1)
    elif kind == "ucc":
        from tyxonq_amd.runtimes import UCCNumericRuntime

        terms, ex, ids = _ucc_problem(case["ns"], case["no"])
        s["theta"] = _theta_ucc(case, seed)
        s["rt"] = UCCNumericRuntime(2 * case["ns"], (case["no"], case["no"]),
                                    {tuple((q, P) for P, q in f): c for c, f in terms},
                                    ex_ops=ex, param_ids=ids)
    elif kind == "trajectory":
        from tyxonq_amd.engine import StatevectorEngine
        import tyxonq_amd as tq

        c = tq.Circuit(case["n"])
        ks = _channel(case["channel"])
        for name, qs, v in _trajectory(case, seed):
            if name == "kraus":
                c.kraus(qs[0], ks, status=v)
            else:
                _circuit(case["n"], [(name, qs, v)], c)
        for q in range(case["n"]):
            c.measure_z(q)
        s["circuit"], s["engine"] = c, StatevectorEngine()
    elif kind == "sample":
        s["psi"], s["seed"] = _state(case["n"], seed), seed
    elif kind == "density":
        from tyxonq_amd.density import DensityMatrixEngine

        s["circuit"] = _circuit(case["n"], _density(case, seed))
        for q in range(case["n"]):
            s["circuit"].measure_z(q)
        s["noise"], s["engine"] = _noise(case), DensityMatrixEngine()
    elif kind == "kq":
        s["psi"] = _state(case["n"], seed)
        s["U"], s["qubits"] = _kq(case, seed)
    else:
        one, two = _gates(case, seed)
        s["psi"] = _state(case["n"], seed + 1, tilt=True).requires_grad_(True)
        s["one"] = [(q, torch.tensor(U, requires_grad=True)) for q, U in one]
        s["two"] = [(q, torch.tensor(U, requires_grad=True)) for q, U in two]
        s["w"] = _rng(seed + 2).normal(size=case["n"])
    return s


def _native_ham(n, terms):
    from tyxonq_amd import _native as nat
    from tyxonq_amd.pauli import PauliSum

    return nat.Ham(n, *PauliSum(n, terms).to_masks())


def run(s):
    from tyxonq_amd import _native as nat

    kind, case = s["kind"], s["case"]
    if kind == "hea":
        n = case["n"]
        tt = torch.tensor(s["theta"], dtype=torch.float64, requires_grad=True)
        ops, k = [], 0
        for _ in range(case["layers"]):
            ops += [("ry", (q,), tt[k + q]) for q in range(n)]
            ops += [("cx", (q, q + 1), None) for q in range(n - 1)]
            k += n
        e, g = s["engine"].energy_and_grad(_circuit(n, ops), s["terms"])
        return np.concatenate([[e], g])
    if kind == "serve":
        from tyxonq_amd import serving

        e, g = serving.execute(s["reqs"][0], s["cache"])
        return np.concatenate([[e], g])
    if kind == "serve_batch":
        from tyxonq_amd import serving

        out = serving.execute_batch(s["reqs"], s["cache"])
        return np.concatenate([np.concatenate([[e], g]) for e, g in out])
    if kind == "vqe":
        s["plan"].update(s["ops"])
        nat.init_basis(s["psi"], 0)
        e, g = s["plan"].adjoint(s["ham"], s["psi"], s["lam"])
        return np.concatenate([[e], g])
    if kind == "brickwork":
        nat.init_basis(s["psi"], 0)
        s["plan"].run(s["psi"])
        _, norm, terms = s["ham"].expval(s["psi"], per_term=True)
        return {"state": s["psi"], "norm": norm, "terms": terms}
    if kind == "qaoa":
        import tyxonq_amd as tq

        n = case["n"]
        gam = torch.tensor(s["gamma"], requires_grad=True)
        bet = torch.tensor(s["beta"], requires_grad=True)
        c = tq.Circuit(n)
        for q in range(n):
            c.h(q)
        for l in range(case["layers"]):
            for a, b in s["edges"]:
                c.rzz(a, b, gam[l])
            for q in range(n):
                c.rx(q, bet[l])
        psi = c.state(backend="pytorch")
        psi.backward(s["cot"])
        return {"state": psi.detach(), "gamma": gam.grad, "beta": bet.grad}
    if kind == "ucc":
        e, g = s["rt"].energy_and_grad(s["theta"])
        return np.concatenate([[e], g])
    if kind == "trajectory":
        r = s["engine"].run(s["circuit"])
        z = np.array([r["expectations"]["Z%d" % q] for q in range(case["n"])])
        return {"z": z, "state": s["engine"].last_state}
    if kind == "sample":
        idx, cnt = nat.sample_counts(s["psi"], case["shots"], s["seed"])
        # one row per shot at most: the distinct states, then zeros
        out = np.zeros((2, case["shots"]), dtype=np.int64)
        out[0, :len(idx)], out[1, :len(cnt)] = idx, cnt
        return out
    if kind == "density":
        r = s["engine"].run(s["circuit"], use_noise=True, noise=s["noise"])
        z = np.array([r["expectations"]["Z%d" % q] for q in range(case["n"])])
        return {"z": z, "rho": s["engine"].last_vec}
    from tyxonq_amd import kernels as K

    n = case["n"]
    if kind == "kq":
        return K.apply_kqubit_unitary(s["psi"], s["U"], s["qubits"], n)
    psi = s["psi"]
    for q, U in s["one"]:
        psi = K.apply_1q_statevector(None, psi, U, q, n)
    for (a, b), U in s["two"]:
        psi = K.apply_2q_statevector(None, psi, U, a, b, n)
    z = [K.expect_z_statevector(psi, q, n) for q in range(n)]
    loss = sum(float(w) * v for w, v in zip(s["w"], z))
    gates = [U for _, U in s["one"]] + [U for _, U in s["two"]]
    grads = torch.autograd.grad(loss, [s["psi"]] + gates)
    m = len(s["one"])
    return {"z": torch.stack([v.detach() for v in z]), "dpsi": grads[0],
            "done": torch.stack(list(grads[1:1 + m])), "dtwo": torch.stack(list(grads[1 + m:]))}


# ---- work and tolerance --------------------------------------------------------

def work(case):
    """Inputs read once and outputs written once; flops of the gates as they
    are given: 14 per amplitude for a 2x2 gate, 6 for a diagonal one, 0 for a
    permutation, 8 * 2^k for a dense k-qubit matrix, 4 more per amplitude and
    parameter for a gradient (three sweeps: forward, and psi and lambda back)."""
    kind = case["kind"]

    def adjoint(n, one, diag, params, flips):
        return (3 * (14 * one + 6 * diag) + 4 * params + 8 * flips) * 2.0 ** n

    if kind == "hea":
        n, L = case["n"], case["layers"]
        return {"bytes": 16.0 * n * L, "flops": adjoint(n, n * L, 0, n * L, n + 1)}
    if kind in ("serve", "serve_batch"):
        f = b = 0.0
        for n, d, h, _, th in _requests(case, 0):
            f += adjoint(n, n * d, n * d, 2 * n * d, n + 1)
            b += 16.0 * th.size
        return {"bytes": b, "flops": f}
    if kind == "vqe":
        n, L = case["n"], case["layers"]
        return {"bytes": 32.0 * n * L, "flops": adjoint(n, n * L, n * L, 2 * n * L, n + 1)}
    if kind == "brickwork":
        n, L = case["n"], case["layers"]
        return {"bytes": 8.0 * 2 ** n,
                "flops": (L * (14 * n + 6 * n + 3 * (n - 1)) + 4 * case["terms"]) * 2.0 ** n}
    if kind == "qaoa":
        n, L = case["n"], case["layers"]
        e = len(_qaoa(case, 0)[0])
        return {"bytes": 16.0 * 2 ** n, "flops": adjoint(n, n * (L + 1), e * L, (n + e) * L, 0)}
    if kind == "ucc":
        terms, ex, _ = _ucc_problem(case["ns"], case["no"])
        n = 2 * case["ns"]
        # an excitation turns 2 of every 16 (4) amplitudes
        rot = sum(14.0 * (0.125 if len(t) == 4 else 0.5) for t in ex)
        flips = len({tuple(sorted(q for P, q in f if P != "Z")) for _, f in terms})
        return {"bytes": 16.0 * len(ex), "flops": (4 * rot + 8 * flips) * 2.0 ** n}
    if kind == "trajectory":
        n, L = case["n"], case["layers"]
        return {"bytes": 8.0 * 2 ** n, "flops": (L * n * (14 + 14) + 4 * n) * 2.0 ** n}
    if kind == "sample":
        return {"bytes": 8.0 * 2 ** case["n"] + 16.0 * case["shots"], "flops": 4.0 * 2 ** case["n"]}
    if kind == "density":
        n, L = case["n"], case["layers"]
        gates = L * (2 * n * 2 * 14 + (2 * n + 2 * (n - 1)) * 32)
        return {"bytes": 8.0 * 4 ** n, "flops": gates * 4.0 ** n}
    if kind == "kq":
        return {"bytes": 16.0 * 2 ** case["n"], "flops": 8.0 * 2 ** (case["n"] + case["k"])}
    n, L = case["n"], case["layers"]
    one, two = _gates(case, 0)
    # forward, U^dagger of the cotangent, and the outer product of each gate
    return {"bytes": 16.0 * 2 ** n,
            "flops": (3 * (14 * len(one) + 32 * len(two)) + 6 * n) * 2.0 ** n}


def tolerance(case):
    """Complex64 states and gates, FP64 sums: about 1e-7 per rounding, growing
    with the number of gates; about four times the measured distance from
    `exact`.  Counts are whole numbers."""
    if case["kind"] == "sample":
        return "exact"
    return {"rel": {"hea": 2e-6, "serve": 3e-6, "serve_batch": 2e-6, "vqe": 1e-5, "brickwork": 5e-6,
                    "qaoa": 1e-5, "ucc": 2e-6, "trajectory": 2e-6, "density": 5e-6, "kq": 1e-6,
                    "gates": 2e-6}[case["kind"]]}


# ---- results in 64 bits --------------------------------------------------------

PAULI = {"X": np.array([[0, 1], [1, 0]], dtype=complex),
         "Y": np.array([[0, -1j], [1j, 0]], dtype=complex),
         "Z": np.array([[1, 0], [0, -1]], dtype=complex)}
GEN = {"rx": "X", "ry": "Y", "rz": "Z"}


def _rot(P, t):
    return math.cos(t / 2) * np.eye(2) - 1j * math.sin(t / 2) * PAULI[P]


def _one(psi, q, U):
    """U on qubit q of a complex128 state (qubit 0 the most significant bit)."""
    v = psi.view(1 << q, 2, -1)
    a, b = v[:, 0], v[:, 1]
    out = torch.empty_like(v)
    for r in (0, 1):
        out[:, r] = complex(U[r, 0]) * a + complex(U[r, 1]) * b
    return out.view(-1)


def _kmat(psi, n, qubits, U):
    """A dense matrix on the given qubits (the first the most significant)."""
    k = len(qubits)
    rest = [q for q in range(n) if q not in qubits]
    t = psi.view([2] * n).permute(list(qubits) + rest).reshape(1 << k, -1)
    t = (torch.as_tensor(np.asarray(U), dtype=torch.complex128, device=psi.device) @ t).view([2] * n)
    inv = np.argsort(list(qubits) + rest).tolist()
    return t.permute(inv).reshape(-1)


def _op(psi, n, name, qs, th, sign=1.0):
    """A named gate, or with sign = -1 its inverse."""
    if name in GEN:
        return _one(psi, qs[0], _rot(GEN[name], sign * th))
    if name == "h":
        return _one(psi, qs[0], SQ * np.array([[1, 1], [1, -1]]))
    i = torch.arange(1 << n, device=psi.device)
    a, b = (n - 1 - q for q in qs)
    if name == "cx":
        return psi[i ^ (((i >> a) & 1) << b)]
    if name == "cz":
        return psi * (1 - 2 * ((i >> a) & (i >> b) & 1))
    s = 1 - 2 * (((i >> a) ^ (i >> b)) & 1)  # rzz
    return psi * torch.exp(-0.5j * sign * th * s.to(torch.complex128))


def _gen(psi, n, name, qs):
    """The generator P of exp(-i theta/2 P) on psi."""
    if name in GEN:
        return _one(psi, qs[0], PAULI[GEN[name]])
    i = torch.arange(1 << n, device=psi.device)
    return psi * (1 - 2 * (((i >> (n - 1 - qs[0])) ^ (i >> (n - 1 - qs[1]))) & 1))


def _pauli_sum(psi, n, terms, bit=None):
    """H psi; factors (P, q) on index bit `bit(q)` (default n-1-q)."""
    bit = bit or (lambda q: n - 1 - q)
    i = torch.arange(1 << n, device=psi.device)
    groups = {}
    for c, fac in terms:
        x = sum(1 << bit(q) for P, q in fac if P in "XY")
        z = sum(1 << bit(q) for P, q in fac if P in "YZ")
        groups.setdefault(x, []).append((c * 1j ** bin(x & z).count("1"), z))
    out = torch.zeros_like(psi)
    for x, zs in groups.items():
        j = i ^ x
        f = torch.zeros(1 << n, dtype=torch.complex128, device=psi.device)
        for c, z in zs:
            f += c * (1 - 2 * _parity(j & z))
        out += f * psi[j]
    return out


def _parity(v):
    for s in (32, 16, 8, 4, 2, 1):
        v = v ^ (v >> s)
    return v & 1


def _zero(n):
    psi = torch.zeros(1 << n, dtype=torch.complex128, device="cuda")
    psi[0] = 1
    return psi


def _reverse(psi, lam, n, ops, scale):
    """Im <lam|P|psi> * scale before each parametrised gate, in op order."""
    g = []
    for name, qs, th in reversed(ops):
        if th is not None:
            g.append(scale * float(torch.vdot(lam, _gen(psi, n, name, qs)).imag))
        psi, lam = _op(psi, n, name, qs, th, -1.0), _op(lam, n, name, qs, th, -1.0)
    return np.array(g[::-1])


def _energy_grad(n, ops, terms):
    psi = _zero(n)
    for name, qs, th in ops:
        psi = _op(psi, n, name, qs, th)
    lam = _pauli_sum(psi, n, terms)
    e = float(torch.vdot(psi, lam).real)
    return np.concatenate([[e], _reverse(psi, lam, n, ops, 1.0)])


def _exact_ucc(case, seed):
    terms, ex, ids = _ucc_problem(case["ns"], case["no"])
    n, no, th = 2 * case["ns"], case["no"], _theta_ucc(case, seed)
    i = torch.arange(1 << n, device="cuda")

    def ladder(idx, sgn, ok, p, create):
        occ = (idx >> p) & 1
        ok = ok & (occ == (0 if create else 1))
        return idx ^ (1 << p), sgn * (1 - 2 * _parity(idx & ((1 << p) - 1))), ok

    def turn(psis, t, f):
        """exp(t (T - T^dag)) on each state, and T - T^dag on the first."""
        m = len(f) // 2
        idx, sgn, ok = i, torch.ones_like(i), torch.ones_like(i, dtype=torch.bool)
        for k in reversed(range(2 * m)):
            idx, sgn, ok = ladder(idx, sgn, ok, f[k], k < m)
        a, s = i[ok], sgn[ok].to(torch.float64)
        b = idx[ok]
        out = []
        for v in psis:
            w = v.clone()
            w[a] = math.cos(t) * v[a] - math.sin(t) * s * v[b]
            w[b] = math.cos(t) * v[b] + math.sin(t) * s * v[a]
            out.append(w)
        d = torch.zeros_like(psis[0])
        d[b] = s * psis[0][a]
        d[a] = -s * psis[0][b]
        return out, d

    psi = torch.zeros(1 << n, dtype=torch.complex128, device="cuda")
    psi[sum(1 << k for k in range(no)) | sum(1 << (n // 2 + k) for k in range(no))] = 1
    for f, p in zip(ex, ids):
        (psi,), _ = turn([psi], th[p], f)
    lam = _pauli_sum(psi, n, terms, bit=lambda q: q)
    e = float(torch.vdot(psi, lam).real)
    g = np.zeros(len(th))
    for f, p in zip(reversed(ex), reversed(ids)):
        (psi, lam), d = turn([psi, lam], -th[p], f)
        g[p] += 2.0 * float(torch.vdot(lam, turn([psi], 0.0, f)[1]).real)
    return np.concatenate([[e], g])


def _exact_brickwork(case, seed):
    """Layers as dense 5-qubit blocks and a sign vector."""
    n = case["n"]
    ops, strings, _ = _brickwork(case, seed)
    psi, at = _zero(n), 0
    i = torch.arange(1 << n, device="cuda", dtype=torch.int32)  # n <= 30
    for _ in range(case["layers"]):
        U = [_rot("Z", ops[at + 2 * q + 1][2]) @ _rot("X", ops[at + 2 * q][2]) for q in range(n)]
        at += 2 * n
        for q in range(0, n, 5):
            m = min(5, n - q)
            B = U[q]
            for r in range(1, m):
                B = np.kron(B, U[q + r])
            B = torch.as_tensor(B, dtype=torch.complex128, device="cuda")
            v = psi.view(1 << q, 1 << m, -1)
            psi = (torch.matmul(B, v) if v.shape[2] > 1 else v[:, :, 0] @ B.T.contiguous()).reshape(-1)
        mask = i >> 1
        keep = 0
        while at < len(ops) and ops[at][0] == "cz":
            keep |= 1 << (n - 1 - ops[at][1][1])
            at += 1
        v = (i & mask) & keep
        for s in (16, 8, 4, 2, 1):
            v = v ^ (v >> s)
        psi *= (1 - 2 * (v & 1)).to(torch.float64)
        del v, mask
    del i
    out = []
    for (P, a), (Q, b) in strings:
        v = psi.view(1 << a, 2, 1 << (b - a - 1), 2, -1)
        M = np.kron(PAULI[P], PAULI[Q])
        acc = 0.0
        for r in range(4):
            c = int(np.nonzero(M[r])[0][0])
            if c < r:
                continue
            x = v[:, r >> 1, :, r & 1]
            y = v[:, c >> 1, :, c & 1]
            if c == r:
                acc += M[r, r].real * float((x.real.square() + x.imag.square()).sum())
            else:
                w = M[r, c]  # 2 Re(w conj(x) y), w real or imaginary
                t = (x.real * y.real + x.imag * y.imag) if w.imag == 0 else \
                    (x.imag * y.real - x.real * y.imag)
                acc += 2.0 * (w.real if w.imag == 0 else w.imag) * float(t.sum())
        out.append(acc)
    return {"state": psi, "norm": float(sum(c.abs().square().sum() for c in psi.chunk(16))),
            "terms": np.array(out)}


def _exact_trajectory(case, seed):
    n, ks = case["n"], _channel(case["channel"])
    psi = _zero(n)
    for name, qs, v in _trajectory(case, seed):
        if name != "kraus":
            psi = _op(psi, n, name, qs, v)
            continue
        cand = [_one(psi, qs[0], k) for k in ks]
        w = np.array([float(c.abs().square().sum()) for c in cand])
        sel = int(np.argmax(v <= np.cumsum(w / w.sum())))
        psi = cand[sel] / math.sqrt(w[sel])
    return {"z": _z(psi, n), "state": psi}


def _z(psi, n):
    p = psi.abs().square()
    out = []
    for q in range(n):
        v = p.view(1 << q, 2, -1)
        out.append(float(v[:, 0].sum() - v[:, 1].sum()))
    return np.array(out)


def _exact_density(case, seed):
    n = case["n"]
    noise = _noise(case)
    if noise["type"] == "depolarizing":
        p = noise["p"]
        ks = [math.sqrt(1 - p) * np.eye(2)] + [math.sqrt(p / 3) * PAULI[P] for P in "XYZ"]
    else:
        g = noise["gamma"]
        ks = [np.array([[1, 0], [0, math.sqrt(1 - g)]]), np.array([[0, math.sqrt(g)], [0, 0]])]
    rho = _zero(2 * n)
    for name, qs, th in _density(case, seed):
        rho = _op(rho, 2 * n, name, qs, th)
        # the column side: conj(U), i.e. rx and rz with -theta, cx itself
        rho = _op(rho, 2 * n, name, tuple(n + q for q in qs), th, -1.0)
        for q in qs:
            rho = sum(_one(_one(rho, q, k), n + q, k.conj()) for k in ks)
    d = torch.diagonal(rho.view(1 << n, 1 << n)).real
    z = []
    for q in range(n):
        v = d.reshape(1 << q, 2, -1)
        z.append(float(v[:, 0].sum() - v[:, 1].sum()))
    return {"z": np.array(z), "rho": rho}


def exact(case, seed):
    kind = case["kind"]
    if kind == "hea":
        n = case["n"]
        th = _rng(seed).uniform(0.0, 2.0 * math.pi, n * case["layers"])
        ops = []
        for l in range(case["layers"]):
            ops += [("ry", (q,), th[l * n + q]) for q in range(n)]
            ops += [("cx", (q, q + 1), None) for q in range(n - 1)]
        return _energy_grad(n, ops, _tfim(n))
    if kind in ("serve", "serve_batch"):
        out = []
        for n, d, h, g, th in _requests(case, seed):
            ops, t = [], th.reshape(d, 2, n)
            for l in range(d):
                ops += [("ry", (q,), t[l, 0, q]) for q in range(n)]
                ops += [("rz", (q,), t[l, 1, q]) for q in range(n)]
                ops += [("cx", (q, q + 1), None) for q in range(n - 1)]
            out.append(_energy_grad(n, ops, _tfim(n, g) if h == "tfim" else _heisenberg(n, g)))
        return np.concatenate(out)
    if kind == "vqe":
        n = case["n"]
        th = _rng(seed).normal(0.0, 0.3, 2 * n * case["layers"])
        return _energy_grad(n, _ring_ops(n, case["layers"], th), _heisenberg(n))
    if kind == "brickwork":
        return _exact_brickwork(case, seed)
    if kind == "qaoa":
        n = case["n"]
        edges, gam, bet = _qaoa(case, seed)
        ops = [("h", (q,), None) for q in range(n)]
        lab = []
        for l in range(case["layers"]):
            ops += [("rzz", e, gam[l]) for e in edges] + [("rx", (q,), bet[l]) for q in range(n)]
            lab += [(0, l)] * len(edges) + [(1, l)] * n
        psi = _zero(n)
        for name, qs, th in ops:
            psi = _op(psi, n, name, qs, th)
        g = _reverse(psi, _state(n, seed + 1, torch.complex128), n, ops, 0.5)
        out = np.zeros((2, case["layers"]))
        for (a, l), v in zip(lab, g):
            out[a, l] += v
        return {"state": psi, "gamma": out[0], "beta": out[1]}
    if kind == "ucc":
        return _exact_ucc(case, seed)
    if kind == "trajectory":
        return _exact_trajectory(case, seed)
    if kind == "sample":
        return None  # whole numbers
    if kind == "density":
        return _exact_density(case, seed)
    n = case["n"]
    if kind == "kq":
        U, qubits = _kq(case, seed)
        return _kmat(_state(n, seed, torch.complex128), n, qubits, U)
    one, two = _gates(case, seed)
    w = _rng(seed + 2).normal(size=n)
    seq = [((q,), U) for q, U in one] + [(qs, U) for qs, U in two]
    psis = [_state(n, seed + 1, torch.complex128, tilt=True)]
    for qs, U in seq:
        psis.append(_kmat(psis[-1], n, qs, U))
    psi = psis.pop()
    i = torch.arange(1 << n, device="cuda")
    f = torch.zeros(1 << n, dtype=torch.float64, device="cuda")
    for q in range(n):
        f += w[q] * (1 - 2 * ((i >> (n - 1 - q)) & 1))
    lam, grads = 2.0 * f * psi, []  # torch's gradient of a real loss
    for qs, U in reversed(seq):
        prev, k = psis.pop(), len(qs)
        rest = [q for q in range(n) if q not in qs]
        a = lam.view([2] * n).permute(list(qs) + rest).reshape(1 << k, -1)
        b = prev.view([2] * n).permute(list(qs) + rest).reshape(1 << k, -1)
        grads.append((a @ b.conj().T.contiguous()).cpu().numpy())
        lam = _kmat(lam, n, qs, U.conj().T)
    grads.reverse()
    return {"z": _z(psi, n), "dpsi": lam, "done": np.stack(grads[:len(one)]),
            "dtwo": np.stack(grads[len(one):])}
