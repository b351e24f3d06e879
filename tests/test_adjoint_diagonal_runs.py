"""Gradient terms of diagonal runs (k_adj_diag_terms) and Z-string observables
(k_apply_zterms) at every tile height, against numpy in 64 bits."""
import math
import random

import numpy as np
import pytest

import subquokka_dev_amd as sq

pytestmark = pytest.mark.gpu
REL = {"c128": 1e-11, "c64": 2e-5}   # FP64 sums of about 1e3 rounded gates; FP32 amplitudes


def parity(n, mask):
    p = np.arange(1 << n, dtype=np.uint64) & np.uint64(mask)
    for s in (32, 16, 8, 4, 2, 1):
        p ^= p >> np.uint64(s)
    return 1.0 - 2.0 * (p & np.uint64(1)).astype(np.float64)


def mask_of(qs):
    return sum(1 << q for q in qs)


def apply(a, g, back=False):
    name, qs, t = g[0], g[1], (-g[2] if back else g[2])
    n = a.size.bit_length() - 1
    if name == "H":
        m = 0.70710678118 * np.array([[1, 1], [1, -1]])
    elif name == "RX":
        m = np.array([[math.cos(t / 2), -1j * math.sin(t / 2)], [-1j * math.sin(t / 2), math.cos(t / 2)]])
    elif name == "RY":
        m = np.array([[math.cos(t / 2), -math.sin(t / 2)], [math.sin(t / 2), math.cos(t / 2)]])
    else:
        if name in ("RZ", "RZZ"):
            return a * np.exp(-0.5j * t * parity(n, mask_of(qs)))
        on = np.ones(1 << n, dtype=bool)
        for q in qs:
            on &= (np.arange(1 << n) >> q) & 1 == 1
        return np.where(on, a * np.exp(1j * t), a)   # P, CP
    v = a.reshape(-1, 2, 1 << qs[0])
    return np.stack([m[0, 0] * v[:, 0] + m[0, 1] * v[:, 1], m[1, 0] * v[:, 0] + m[1, 1] * v[:, 1]], axis=1).reshape(-1)


def derivative(lam, a, g):
    n = a.size.bit_length() - 1
    if g[0] in ("RZ", "RZZ"):
        return np.vdot(lam, parity(n, mask_of(g[1])) * a).imag
    if g[0] in ("P", "CP"):
        on = np.ones(1 << n, dtype=bool)
        for q in g[1]:
            on &= (np.arange(1 << n) >> q) & 1 == 1
        return -2.0 * np.vdot(lam[on], a[on]).imag
    v, w = a.reshape(-1, 2, 1 << g[1][0]), lam.reshape(-1, 2, 1 << g[1][0])
    if g[0] == "RX":
        return (np.vdot(w[:, 0], v[:, 1]) + np.vdot(w[:, 1], v[:, 0])).imag
    return (-1j * np.vdot(w[:, 0], v[:, 1]) + 1j * np.vdot(w[:, 1], v[:, 0])).imag


def circuit(n, seed):
    rng = random.Random(seed)
    gates = [("H", (q,), 0.0, -1) for q in range(n)]
    theta = []

    def add(name, qs, shared=None):
        if shared is None:
            theta.append(rng.uniform(-math.pi, math.pi))
            shared = len(theta) - 1
        gates.append((name, qs, theta[shared], shared))

    for _ in range(2):
        theta.append(rng.uniform(-1, 1))
        common = len(theta) - 1
        pairs = [(i, j) for i in range(n) for j in range(i + 1, n)]
        for p in rng.sample(pairs, min(len(pairs), 30)):
            add(rng.choice(["RZZ", "CP"]), p, common if rng.random() < 0.5 else None)
            if rng.random() < 0.3:
                gates.append(("CP", p, rng.uniform(-1, 1), -1))   # a fixed gate inside the run
        for q in rng.sample(range(n), min(n, 7)):
            add(rng.choice(["RZ", "P"]), (q,))
        for q in range(n):
            add(rng.choice(["RX", "RY"]), (q,))
        for q in rng.sample(range(n), 2):   # a short run
            add(rng.choice(["RZ", "P"]), (q,))
        gates.append(("H", (rng.randrange(n),), 0.0, -1))
    return gates, np.array(theta)


def strings(n, count, seed):
    rng = random.Random(seed)
    return [(rng.uniform(-1, 1), rng.sample(range(n), rng.randint(0, min(n, 5)))) for _ in range(count)]


@pytest.mark.parametrize("every", [0, 9])
@pytest.mark.parametrize("dtype,n", [("c128", 5), ("c128", 6), ("c64", 7), ("c128", 12), ("c64", 13), ("c128", 17),
                                     ("c64", 18), ("c128", 19), ("c64", 20)])
def test_gradient(dtype, n, every):
    gates, theta = circuit(n, n)
    terms = strings(n, 40, n)
    h = sum(c * parity(n, mask_of(qs)) for c, qs in terms)
    a = np.zeros(1 << n, dtype=np.complex128)
    a[0] = 1
    # H's coefficient is not exactly unitary (2 c^2 = 1 - 2e-11), so the state
    # un-applied through an H differs from the one before it: the reference
    # re-anchors to the forward states where the engine does
    pg = [i for i, g in enumerate(gates) if g[3] >= 0]
    anchors = set(pg[every::every]) if every else set()
    before = {}
    for i, g in enumerate(gates):
        if i in anchors:
            before[i] = a
        a = apply(a, g)
    energy, lam = float(np.sum(h * np.abs(a) ** 2)), h * a
    want = np.zeros(theta.size)
    for i, g in reversed(list(enumerate(gates))):
        a = before.get(i + 1, a)
        if g[3] >= 0:
            want[g[3]] += derivative(lam, a, g)
        a, lam = apply(a, g, True), apply(lam, g, True)
    text = "".join("%s %s%s\n" % (g[0], " ".join(map(str, g[1])), "" if g[0] == "H" else " %.17g" % g[2]) for g in gates)
    eng = sq.Engine(n, dtype=dtype)
    got_e, got = eng.adjoint_grad(text, [g[3] for g in gates], theta, terms, every)
    eng.close()
    scale = max(1.0, float(np.max(np.abs(want))))
    assert abs(got_e - energy) <= REL[dtype] * max(1.0, abs(energy))
    assert np.max(np.abs(got - want)) <= REL[dtype] * scale


@pytest.mark.parametrize("count", [0, 1, 70, 700])
@pytest.mark.parametrize("dtype,n", [("c128", 4), ("c128", 6), ("c64", 9), ("c128", 17), ("c64", 18), ("c128", 21)])
def test_expectation(dtype, n, count):
    s0 = sq.gen_state(n, 3)
    terms = strings(n, count, count + n) + [(0.25, [])] * (count > 0)
    p = np.abs(s0) ** 2
    want = sum(c * float(np.sum(parity(n, mask_of(qs)) * p)) for c, qs in terms)
    eng = sq.Engine(n, dtype=dtype)
    eng.set_state(s0)
    assert abs(eng.expect_z(terms) - want) <= (1e-12 if dtype == "c128" else 2e-6) * max(1, count)
    eng.close()
