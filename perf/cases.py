"""The engine's work as a user's program asks for it, one dict per case.

A case names what the program does ("do"), the circuit and its sizes:

  plain         a gate list on a state in HBM             Engine.apply_gates
  blocks        a subcircuit file (chunk-local blocks     Engine.apply_blocks
                and VSWAPs, the finder's output)
  fused         a gate list as fused passes (complex64)   Engine.apply_gates_fused
  fused_blocks  a planned file of five-qubit blocks       Engine.run_fused
  hea_gradient  energy and gradient of the hardware-      autograd.hea_energy
                efficient ansatz
  gradient      the same for a circuit given as text      autograd.circuit_energy
                with a Z-string observable
  measure       norm, expectations and shots of a state   norm2, expect_zz_ring, expect_z, sample
  stream        a gate list on a state in host memory     Engine.apply_gates, get_state

Circuits: qft (H, CP, SWAP), random (U1 on every qubit and CP(pi) on a random
perfect matching, per layer), qaoa (H, then RZZ on the edges and RX on every
qubit, per layer), hea (RY, RZ, ring of CNOTs written as U2, per layer).
"""
import math
import random

import numpy as np
import torch

import subquokka_dev_amd as sq
from subquokka_dev_amd.autograd import circuit_energy, hea_energy

H = 0.70710678118   # the H coefficient of the circuit grammar
DTYPES = {"c128": torch.complex128, "c64": torch.complex64}


def listed():
    return [
        # the smallest calls: a state of one workgroup, where launches and host work are all the time
        {"name": "qft11_c128", "do": "plain", "circuit": "qft", "qubits": 11, "layers": 0, "dtype": "c128"},
        # the 20-qubit QFT on a random state: controlled phases and swaps on a cache-resident state
        {"name": "qft20_c128", "do": "plain", "circuit": "qft", "qubits": 20, "layers": 0, "dtype": "c128"},
        # MaxCut ansatz on a complete graph, five layers at 21 qubits: mostly diagonal two-qubit gates
        {"name": "qaoa21_c128", "do": "plain", "circuit": "qaoa", "qubits": 21, "layers": 5, "dtype": "c128"},
        # random layers at an odd size in single precision
        {"name": "random25_c64", "do": "plain", "circuit": "random", "qubits": 25, "layers": 10, "dtype": "c64"},
        # the headline: 900 gates on 30 qubits, 16 GiB in double precision
        {"name": "random30_c128", "do": "plain", "circuit": "random", "qubits": 30, "layers": 20, "dtype": "c128"},
        # a subcircuit file that leaves the qubits permuted
        {"name": "blocks26_c128", "do": "blocks", "circuit": "qft", "qubits": 26, "layers": 0, "dtype": "c128", "chunk": 12},
        # the same headline circuit in single precision on the matrix cores
        {"name": "fused30_c64", "do": "fused", "circuit": "random", "qubits": 30, "layers": 20, "dtype": "c64"},
        # planned five-qubit blocks in double precision
        {"name": "fused_blocks25_c128", "do": "fused_blocks", "circuit": "random", "qubits": 25, "layers": 8, "dtype": "c128"},
        # a variational step: 24 qubits, 384 angles, single precision with checkpoints
        {"name": "hea_gradient24_c64", "do": "hea_gradient", "circuit": "hea", "qubits": 24, "layers": 8, "dtype": "c64", "every": 3},
        # a variational step of a MaxCut ansatz in double precision, angles shared by the gates of a layer
        {"name": "gradient18_c128", "do": "gradient", "circuit": "qaoa", "qubits": 18, "layers": 4, "dtype": "c128", "every": 0},
        # readout: expectations and 100000 shots
        {"name": "measure26_c128", "do": "measure", "circuit": "qaoa", "qubits": 26, "layers": 0, "dtype": "c128", "shots": 100000},
        # a state kept in host memory and streamed through the GPU, and read back
        {"name": "stream24_c128", "do": "stream", "circuit": "random", "qubits": 24, "layers": 6, "dtype": "c128", "resident": 20},
    ]


def draw(rng):
    do = rng.choice(["plain", "plain", "plain", "plain", "blocks", "fused", "fused_blocks", "hea_gradient",
                     "gradient", "gradient", "measure", "stream"])
    dtype = rng.choice(["c128", "c128", "c64"])
    if do == "plain":
        circuit = rng.choice(["qft", "random", "qaoa", "hea"])
        return {"do": do, "circuit": circuit, "qubits": rng.randint(7, 28),
                "layers": 0 if circuit == "qft" else rng.randint(1, 8), "dtype": dtype}
    if do == "blocks":
        circuit = rng.choice(["qft", "random", "qaoa"])
        return {"do": do, "circuit": circuit, "qubits": rng.randint(14, 26),
                "layers": 0 if circuit == "qft" else rng.randint(1, 5), "dtype": dtype, "chunk": rng.randint(6, 13)}
    if do == "fused":
        circuit = rng.choice(["random", "qaoa", "hea"])
        return {"do": do, "circuit": circuit, "qubits": rng.randint(14, 28), "layers": rng.randint(1, 8), "dtype": "c64"}
    if do == "fused_blocks":
        circuit = rng.choice(["random", "hea"])
        return {"do": do, "circuit": circuit, "qubits": rng.randint(8, 26), "layers": rng.randint(1, 8), "dtype": dtype}
    if do == "hea_gradient":
        return {"do": do, "circuit": "hea", "qubits": rng.randint(6, 23), "layers": rng.randint(1, 8), "dtype": dtype,
                "every": rng.choice([0, 1, 3])}
    if do == "gradient":
        circuit = rng.choice(["qaoa", "hea"])
        return {"do": do, "circuit": circuit, "qubits": rng.randint(6, 21), "layers": rng.randint(1, 5), "dtype": dtype,
                "every": rng.choice([0, 0, 20])}
    if do == "measure":
        return {"do": do, "circuit": "qaoa", "qubits": rng.randint(10, 27), "layers": 0, "dtype": dtype,
                "shots": int(10 ** rng.uniform(2, 5.5))}
    n = rng.randint(16, 23)
    return {"do": do, "circuit": "random", "qubits": n, "layers": rng.randint(2, 6), "dtype": dtype,
            "resident": rng.randint(14, n - 2)}


# ---------------------------------------------------------------------------
# circuits: a list of (name, qubits, numbers, index of the angle or -1)
# ---------------------------------------------------------------------------

CNOT = [1.0 if (r, c) in ((0, 0), (1, 1), (2, 3), (3, 2)) else 0.0 for r in range(4) for c in range(4)]
CNOT_REV = [1.0 if (r, c) in ((0, 0), (1, 3), (2, 2), (3, 1)) else 0.0 for r in range(4) for c in range(4)]


def edges_of(case, rng):
    """The graph of a qaoa circuit: complete up to 21 qubits, else 3n/2 random edges."""
    n = case["qubits"]
    pairs = [(i, j) for i in range(n) for j in range(i + 1, n)]
    return pairs if n <= 21 else sorted(rng.sample(pairs, 3 * n // 2))


def circuit_of(case, seed):
    """(gates, number of angles, edges)."""
    rng = random.Random(seed)
    n, layers, kind = case["qubits"], case["layers"], case["circuit"]
    angle = lambda: rng.uniform(-math.pi, math.pi)   # noqa: E731
    gates, count, edges = [], 0, []
    if kind == "qft":
        for i in range(n):
            gates.append(("H", (i,), (), -1))
            gates += [("CP", (i, j), (math.pi / 2 ** (j - i),), -1) for j in range(i + 1, n)]
        gates += [("SWAP", (i, n - 1 - i), (), -1) for i in range(n // 2)]
    elif kind == "random":
        for _ in range(layers):
            for q in range(n):
                th, ph, la = angle(), angle(), angle()
                c, s = math.cos(th / 2), math.sin(th / 2)
                gates.append(("U1", (q,), (c, 0.0, -math.cos(la) * s, -math.sin(la) * s, math.cos(ph) * s,
                                           math.sin(ph) * s, math.cos(ph + la) * c, math.sin(ph + la) * c), -1))
            order = list(range(n))
            rng.shuffle(order)
            gates += [("CP", (min(a, b), max(a, b)), (math.pi,), -1) for a, b in zip(order[::2], order[1::2])]
    elif kind == "qaoa":
        edges = edges_of(case, rng)
        gates += [("H", (q,), (), -1) for q in range(n)]
        for _ in range(layers):
            gamma, beta = angle(), angle()
            gates += [("RZZ", e, (gamma,), count) for e in edges]
            gates += [("RX", (q,), (beta,), count + 1) for q in range(n)]
            count += 2
    else:
        for _ in range(layers):
            for name in ("RY", "RZ"):
                gates += [(name, (q,), (angle(),), count + q) for q in range(n)]
                count += n
            for q in range(n):
                t = (q + 1) % n
                m = CNOT if q < t else CNOT_REV
                gates.append(("U2", (min(q, t), max(q, t)), tuple(v for x in m for v in (x, 0.0)), -1))
    return gates, count, edges


def text_of(gates):
    return "".join("%s %s%s\n" % (g[0], " ".join(map(str, g[1])), "".join(" %.17g" % v for v in g[2])) for g in gates)


def angles_of(gates, count):
    th = np.zeros(count)
    for g in gates:
        if g[3] >= 0:
            th[g[3]] = g[2][0]
    return th


# ---------------------------------------------------------------------------
# states
# ---------------------------------------------------------------------------

class _Memory:
    """The engine's state as torch reads it; keeps the engine alive."""

    def __init__(self, eng):
        self.eng = eng
        ptr, _ = eng.device_state()
        self.__cuda_array_interface__ = {"shape": (1 << eng.n,), "typestr": "<c16" if eng.dtype == "c128" else "<c8",
                                         "data": (ptr, False), "version": 3, "strides": None}


def state_of(eng):
    return torch.as_tensor(_Memory(eng), device="cuda")


def fill(amps, seed):
    """Gaussian amplitudes, normalised."""
    parts = torch.view_as_real(amps)
    parts.normal_(generator=torch.Generator(device=amps.device).manual_seed(seed))
    parts.mul_(1.0 / float(torch.linalg.vector_norm(parts[: 1 << 24], dtype=torch.float64))
               * math.sqrt(min(1.0, (1 << 24) / parts.shape[0])))
    return amps


def host_state(case, seed):
    amps = fill(torch.empty(1 << case["qubits"], dtype=DTYPES[case["dtype"]], device="cuda"), seed)
    return amps.cpu().numpy()


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def prepare(case, seed):
    n, do = case["qubits"], case["do"]
    gates, count, edges = circuit_of(case, seed)
    if do == "stream":
        eng = sq.Engine(n, dtype=case["dtype"], resident_qbit=case["resident"])
        eng.set_state(host_state(case, seed))
        parsed, _, ng, _ = sq.parse_circuit(text_of(gates), n)
        return {"do": do, "eng": eng, "gates": parsed, "ng": ng, "out": DTYPES[case["dtype"]]}
    eng = sq.Engine(n, dtype=case["dtype"], chunk=case.get("chunk", 0))
    st = {"do": do, "eng": eng}
    if do in ("plain", "blocks", "fused", "fused_blocks", "measure"):
        eng.sync()   # the engine's own |0...0> comes first
        fill(state_of(eng), seed)
        torch.cuda.synchronize()
    if do in ("plain", "fused"):
        st["gates"], _, st["ng"], _ = sq.parse_circuit(text_of(gates), n)
    elif do in ("blocks", "fused_blocks"):
        plan = sq.plan(text_of(gates), n, 0, case["chunk"]) if do == "blocks" else sq.plan(text_of(gates), n, 1, 5)
        st["gates"], st["blocks"], _, st["nb"] = sq.parse_circuit(plan, n, is_subcircuit=True)
    elif do in ("hea_gradient", "gradient"):
        st.update(theta=torch.tensor(angles_of(gates, count), requires_grad=True), layers=case["layers"],
                  every=case["every"], text=text_of(gates), param=[g[3] for g in gates],
                  terms=observable(case, edges))
    elif do == "measure":
        st.update(terms=observable(case, edges), shots=case["shots"], seed=seed)
    return st


def observable(case, edges):
    """Z strings [(coefficient, qubits)]: the cut of a graph, or a ring with fields."""
    n = case["qubits"]
    if case["circuit"] == "qaoa":
        return [(0.5, list(e)) for e in edges]
    return [(1.0, [q, (q + 1) % n]) for q in range(n)] + [(0.25, [q]) for q in range(n)]


def run(st):
    do, eng = st["do"], st["eng"]
    if do == "plain":
        eng.apply_gates(st["gates"], st["ng"])
        return state_of(eng)
    if do == "blocks":
        eng.apply_blocks(st["gates"], st["blocks"], st["nb"])
        return state_of(eng)
    if do == "fused":
        eng.apply_gates_fused(st["gates"], st["ng"])
        return state_of(eng)
    if do == "fused_blocks":
        eng.run_fused(st["gates"], st["blocks"], st["nb"])
        return state_of(eng)
    if do == "hea_gradient":
        energy = hea_energy(st["theta"], eng, st["layers"], st["every"])
        return [energy.detach(), torch.autograd.grad(energy, st["theta"])[0]]
    if do == "gradient":
        energy = circuit_energy(st["theta"], eng, st["text"], st["param"], st["terms"], st["every"])
        return [energy.detach(), torch.autograd.grad(energy, st["theta"])[0]]
    if do == "measure":
        return [eng.norm2(), eng.expect_zz_ring(), eng.expect_z(st["terms"]), eng.sample(st["shots"], st["seed"])]
    eng.apply_gates(st["gates"], st["ng"])
    return eng.get_state(np.complex128 if st["out"] == torch.complex128 else np.complex64)


def work(case):
    """State read and written once; gate arithmetic on every amplitude a gate changes."""
    n, amps = case["qubits"], 2.0 ** case["qubits"]
    size = amps * (16 if case["dtype"] == "c128" else 8)
    per = {"H": 6, "RX": 6, "RY": 6, "U1": 14, "RZ": 6, "RZZ": 6, "CP": 1.5, "SWAP": 0, "U2": 0}
    if case["do"] == "measure":
        return {"bytes": size, "flops": 8 * amps}
    flops = amps * sum(per[g[0]] for g in circuit_of(case, 0)[0])
    if case["do"] in ("hea_gradient", "gradient"):   # forward, two backward; the inner products
        angles = sum(g[3] >= 0 for g in circuit_of(case, 0)[0])
        return {"bytes": 2 * size, "flops": 3 * flops + 4 * amps * min(angles, 4 * n * case["layers"])}
    return {"bytes": 2 * size, "flops": flops}


# ---------------------------------------------------------------------------
# the same in 64 bits with torch alone
# ---------------------------------------------------------------------------

def _pair(a, q):
    v = a.view(-1, 2, 1 << q)
    return v[:, 0], v[:, 1]


def _quad(a, p, q):
    lo, hi = min(p, q), max(p, q)
    v = a.view(-1, 2, 1 << (hi - lo - 1), 2, 1 << lo)
    # [bit of p][bit of q]
    at = lambda bp, bq: v[:, bq if hi == q else bp, :, bp if hi == q else bq]   # noqa: E731
    return at


def _dense(a, q, m):
    x, y = _pair(a, q)
    u = m[0] * x + m[1] * y
    y.copy_(m[2] * x + m[3] * y)
    x.copy_(u)


def _swap(x, y):
    t = x.clone()
    x.copy_(y)
    y.copy_(t)


def apply(a, g, back=False):
    """One gate (or its inverse) on `a`, in place."""
    name, qs, v = g[0], g[1], g[2]
    sign = -1 if back else 1
    if name == "H":
        _dense(a, qs[0], (H, H, H, -H))
    elif name == "U1":
        m = [complex(v[2 * i], v[2 * i + 1]) for i in range(4)]
        _dense(a, qs[0], [m[0].conjugate(), m[2].conjugate(), m[1].conjugate(), m[3].conjugate()] if back else m)
    elif name in ("RX", "RY"):
        c, s = math.cos(v[0] / 2), sign * math.sin(v[0] / 2)
        _dense(a, qs[0], (c, -1j * s, -1j * s, c) if name == "RX" else (c, -s, s, c))
    elif name == "RZ":
        f = complex(math.cos(v[0] / 2), sign * math.sin(v[0] / 2))
        x, y = _pair(a, qs[0])
        x.mul_(f.conjugate())
        y.mul_(f)
    elif name in ("CP", "RZZ"):
        at = _quad(a, *qs)
        if name == "CP":
            at(1, 1).mul_(complex(math.cos(v[0]), sign * math.sin(v[0])))
        else:
            f = complex(math.cos(v[0] / 2), sign * math.sin(v[0] / 2))
            for b in (0, 1):
                at(b, b).mul_(f.conjugate())
                at(b, 1 - b).mul_(f)
    elif name == "U2":   # a CNOT: the first qubit of the pair is the high bit of the 4x4 basis
        at = _quad(a, *qs)
        if list(v[::2]) == CNOT:
            _swap(at(1, 0), at(1, 1))
        else:
            _swap(at(0, 1), at(1, 1))
    elif name in ("SWAP", "VSWAP_1_1"):
        at = _quad(a, *qs)
        _swap(at(0, 1), at(1, 0))
    elif name == "VSWAP_2_2":
        apply(a, ("SWAP", (qs[0], qs[2]), ()))
        apply(a, ("SWAP", (qs[1], qs[3]), ()))
    else:
        raise ValueError(name)


def file_gates(text):
    """The gates of a subcircuit file, in order."""
    arity = {"U2": 2, "SWAP": 2, "CP": 2, "RZZ": 2, "VSWAP_1_1": 2, "VSWAP_2_2": 4}
    out = []
    for line in text.splitlines():
        w = line.split()
        if len(w) > 1:
            k = arity.get(w[0], 1)
            out.append((w[0], tuple(map(int, w[1:1 + k])), tuple(map(float, w[1 + k:])), -1))
    return out


def _signs(n, qubits, device):
    i = torch.arange(1 << n, device=device)
    p = torch.zeros_like(i)
    for q in qubits:
        p ^= i >> q
    return 1.0 - 2.0 * (p & 1).double()


def _diagonal(n, terms, device):
    h = torch.zeros(1 << n, dtype=torch.float64, device=device)
    for c, qs in terms:
        h += c * _signs(n, qs, device)
    return h


def _generator(x, g):
    """P x for a rotation's generator P (exp(-i t P / 2))."""
    y = x.clone()
    name, qs = g[0], g[1]
    if name in ("RX", "RY"):
        _dense(y, qs[0], (0, 1, 1, 0) if name == "RX" else (0, -1j, 1j, 0))
    elif name == "RZ":
        _pair(y, qs[0])[1].neg_()
    else:
        at = _quad(y, *qs)
        at(0, 1).neg_()
        at(1, 0).neg_()
    return y


def exact(case, seed):
    n, do = case["qubits"], case["do"]
    gates, count, edges = circuit_of(case, seed)
    if n > 28:
        return None   # the whole state gate by gate takes too long
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    ring = [(1.0, [q, (q + 1) % n]) for q in range(n)]
    if do in ("hea_gradient", "gradient"):
        a = torch.zeros(1 << n, dtype=torch.complex128, device=dev)
        a[0] = 1
        for g in gates:
            apply(a, g)
        h = _diagonal(n, ring if do == "hea_gradient" else observable(case, edges), dev)
        energy = (h * (a.real.square() + a.imag.square())).sum()
        lam, grad = h * a, torch.zeros(count, dtype=torch.float64, device=dev)
        for g in reversed(gates):
            if g[3] >= 0:
                grad[g[3]] += torch.vdot(lam, _generator(a, g)).imag
            apply(a, g, back=True)
            apply(lam, g, back=True)
        return [energy.cpu(), grad.cpu()]
    a = fill(torch.empty(1 << n, dtype=DTYPES[case["dtype"]], device=dev), seed).to(torch.complex128)
    if do == "measure":
        p = a.real.square() + a.imag.square()
        return [float(p.sum()), float((_diagonal(n, ring, dev) * p).sum()),
                float((_diagonal(n, observable(case, edges), dev) * p).sum()), None]
    if do == "blocks":
        gates = file_gates(sq.plan(text_of(gates), n, 0, case["chunk"]))
    for g in gates:
        apply(a, g)
    return a.cpu().numpy() if do == "stream" else a
