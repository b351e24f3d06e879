"""Runs of diagonal gates applied as tables (PO_DIAG_TAB) in register passes:
every split of a gate's qubits between vector, lane, register and tile bits,
against the oracle (CPU emulation, GPU) and against one launch per gate (GPU).
"""
import math
import random

import numpy as np
import pytest

from helpers import Oracle
from test_cpu_emul import emul, run_case  # noqa: F401  (emul: the emulation build, a fixture)

TOL = {"c128": 1e-12, "c64": 2e-6}


def diagonal_circuit(n, dense, seed, layers=2):
    """Complete graphs of RZZ / CP / diagonal U2, P / RZ / Z on every qubit, dense gates between."""
    rng = random.Random(seed)
    out = []
    for layer in range(layers):
        for a in range(n):
            for b in range(a + 1, n):
                th = rng.uniform(-math.pi, math.pi)
                k = rng.random()
                if k < 0.5:
                    out.append(f"RZZ {a} {b} {th!r}")
                elif k < 0.9:
                    out.append(f"CP {a} {b} {th!r}")
                else:   # any diagonal of modulus 1, and now and then a scaled one (not a table's)
                    s = 1.0 if rng.random() < 0.8 else 0.5
                    d = [s * complex(math.cos(t), math.sin(t)) for t in (rng.uniform(-3, 3) for _ in range(4))]
                    m = [(d[r].real, d[r].imag) if r == c else (0.0, 0.0) for r in range(4) for c in range(4)]
                    out.append(f"U2 {a} {b} " + " ".join(repr(v) for z in m for v in z))
                    if s != 1.0:   # and back, so the norm stays
                        inv = [1 / z for z in d]
                        m = [(inv[r].real, inv[r].imag) if r == c else (0.0, 0.0) for r in range(4) for c in range(4)]
                        out.append(f"U2 {a} {b} " + " ".join(repr(v) for z in m for v in z))
        for q in range(n):
            out.append(rng.choice([f"P {q} {rng.uniform(-3, 3)!r}", f"RZ {q} {rng.uniform(-3, 3)!r}", f"Z {q}"]))
        for q in dense:
            out.append(rng.choice([f"RX {q} {rng.uniform(-3, 3)!r}", f"H {q}", f"RY {q} {rng.uniform(-3, 3)!r}"]))
    return "\n".join(out) + "\n"


@pytest.mark.parametrize("kh", [1, 3, 5])
@pytest.mark.parametrize("dtype,n", [("c128", 12), ("c64", 12), ("c128", 16), ("c64", 15)])
def test_emulated(emul, tmp_path, dtype, n, kh):
    first = 8   # lane gates cross lanes, which the emulation does not model
    text = diagonal_circuit(n, range(first, n), n + kh)
    got = run_case(emul, tmp_path, "plain", n, 4, dtype, text, seed=n, pass_qbits=kh)
    import subquokka_dev_amd as sq
    want = Oracle().run(sq.gen_state(n, n), n, text)
    assert np.max(np.abs(got - want)) <= TOL[dtype]


@pytest.mark.gpu
@pytest.mark.parametrize("kh", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("dtype,n", [("c128", 11), ("c128", 12), ("c64", 13), ("c128", 17), ("c64", 18)])
def test_gpu(dtype, n, kh):
    import subquokka_dev_amd as sq
    text = diagonal_circuit(n, range(n), 3 * n + kh)
    s0 = sq.gen_state(n, n)
    want = Oracle().run(s0, n, text)
    eng = sq.Engine(n, dtype=dtype, pass_qbits=kh)
    eng.set_state(s0)
    eng.apply_text(text)
    assert np.max(np.abs(eng.get_state() - want)) <= TOL[dtype]
    eng.close()


@pytest.mark.gpu
def test_gpu_many_tile_bits():
    # 24 qubits: tile bits up to the thirteenth, tables of every kind
    import subquokka_dev_amd as sq
    n = 24
    text = diagonal_circuit(n, range(0, n, 3), 5, layers=1)
    a, b = sq.Engine(n, dtype="c128"), sq.Engine(n, dtype="c128", sweep_mode=1)
    for e in (a, b):
        e.apply_text("".join(f"H {q}\n" for q in range(n)) + text)
    assert a.max_abs_diff(b) <= 1e-12
    a.close()
    b.close()
