"""Complex128 block lists that the register passes carry run as them; blocks
with other two-qubit gates, and smaller states, keep the composed 32x32 product:
both against one launch per gate, and the checks on blocks are the same."""
import ctypes
import random

import numpy as np
import pytest

import subquokka_dev_amd as sq
from test_gpu_parity import cnot_line

pytestmark = pytest.mark.gpu


def circuit(n, kinds, seed):
    rng = random.Random(seed)
    out = []
    for _ in range(120):
        a, b = sorted(rng.sample(range(n), 2))
        x = rng.uniform(-3, 3)
        k = rng.choice(kinds)
        if k == "CNOT":
            out.append(cnot_line(*rng.sample((a, b), 2)))
        elif k == "U2":   # a rotation by x about (XX + YY), not a CNOT and not diagonal
            c, s = np.cos(x), np.sin(x)
            m = [1, 0, 0, 0, 0, c, -1j * s, 0, 0, -1j * s, c, 0, 0, 0, 0, 1]
            out.append(f"U2 {a} {b} " + " ".join(f"{complex(z).real!r} {complex(z).imag!r}" for z in m))
        else:
            out.append(f"{k} {a} {b} {x!r}" if k in ("CP", "RZZ") else f"{k} {a} {b}" if k == "SWAP" else f"{k} {a} {x!r}" if k != "H" else f"H {a}")
    return "\n".join(out) + "\n"


@pytest.mark.parametrize("n", [24, 25])
@pytest.mark.parametrize("kinds,carried", [(["H", "RX", "RZ", "CP", "RZZ", "SWAP", "CNOT"], True), (["RY", "U2", "CP"], False)])
def test_blocks(n, kinds, carried):
    text = circuit(n, kinds, n)
    plan = sq.plan(text, n, 1, 5)
    gates, blocks, _, nb = sq.parse_circuit(plan, n, is_subcircuit=True)
    eng = sq.Engine(n, dtype="c128")
    eng.stats_enable(True)
    eng.run_fused(gates, blocks, nb)
    assert ("fused5_c128" in eng.stats()) == (not carried or n < 25)
    ref = sq.Engine(n, dtype="c128", sweep_mode=1)   # one launch per gate
    ref.apply_text(text)
    assert eng.max_abs_diff(ref) <= 1e-12
    eng.close()
    ref.close()


def test_wide_block_is_refused():
    n = 25
    gates, _, ng, _ = sq.parse_circuit("".join(f"H {q}\n" for q in range(6)), n)
    eng = sq.Engine(n, dtype="c128")
    with pytest.raises(sq.native.SqError) as err:
        eng.run_fused(gates, (ctypes.c_uint32 * 1)(ng), 1)
    assert err.value.code == sq.native.SQ_ERR_ARG
    eng.close()
