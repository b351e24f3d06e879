"""CNOTs inside register passes (PO_CNOT): every target and control, between
rotations and phases that have to be applied before or may pass them, against
the oracle; alone they are an exact permutation."""
import itertools
import random

import numpy as np
import pytest

import subquokka_dev_amd as sq
from helpers import Oracle
from test_gpu_parity import cnot_line

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kh", [1, 2, 3, 4, 0])
@pytest.mark.parametrize("dtype,n", [("c128", 11), ("c64", 12), ("c128", 13), ("c64", 14)])
def test_alone_bit_exact(dtype, n, kh):
    pairs = list(itertools.permutations(range(n), 2))
    random.Random(n + kh).shuffle(pairs)
    s0 = sq.gen_state(n, 2)
    if dtype == "c64":
        s0 = s0.astype(np.complex64).astype(np.complex128)
    want = s0
    i = np.arange(1 << n)
    for c, t in pairs:
        want = want[i ^ (((i >> c) & 1) << t)]
    eng = sq.Engine(n, dtype=dtype, pass_qbits=kh)
    eng.set_state(s0)
    eng.apply_text("".join(cnot_line(c, t) + "\n" for c, t in pairs))
    assert np.array_equal(eng.get_state(), want)
    eng.close()


@pytest.mark.parametrize("kh", [2, 4, 0])
@pytest.mark.parametrize("dtype,n", [("c128", 12), ("c64", 13), ("c128", 16), ("c64", 17)])
def test_between_gates(dtype, n, kh):
    rng = random.Random(n * 7 + kh)
    lines = []
    for _ in range(250):
        a, b = rng.sample(range(n), 2)
        x = rng.uniform(-3, 3)
        lines.append(rng.choice([cnot_line(a, b)] * 4 + [f"RX {a} {x!r}", f"RY {a} {x!r}", f"H {a}", f"RZ {a} {x!r}", f"P {a} {x!r}",
                                                         f"CP {min(a, b)} {max(a, b)} {x!r}", f"RZZ {min(a, b)} {max(a, b)} {x!r}",
                                                         f"CP {min(a, b)} {max(a, b)} 3.141592653589793"]))
    text = "\n".join(lines) + "\n"
    s0 = sq.gen_state(n, 4)
    want = Oracle().run(s0, n, text)
    eng = sq.Engine(n, dtype=dtype, pass_qbits=kh)
    eng.set_state(s0)
    eng.apply_text(text)
    assert np.max(np.abs(eng.get_state() - want)) <= (1e-12 if dtype == "c128" else 2e-6)
    eng.close()
