"""SWAPs of a plain list as a relabelling and one in-place permutation
(k_bitswap), and a subcircuit file's SWAP gates beside its VSWAPs, against the
oracle: single transpositions, disjoint ones, reversals and longer cycles, on
tiles smaller and larger than the state."""
import random

import numpy as np
import pytest

import subquokka_dev_amd as sq
from helpers import Oracle
from test_cpu_emul import emul, run_case  # noqa: F401  (emul: the emulation build, a fixture)

TOL = {"c128": 1e-12, "c64": 2e-6}


def swap_circuit(n, pairs, seed):
    rng = random.Random(seed)
    out = []
    for a, b in pairs:
        out += [f"RY {rng.randrange(n)} {rng.uniform(-3, 3)!r}", f"CP {a} {b} {rng.uniform(-3, 3)!r}"]
        out.append(f"SWAP {a} {b}")
        q = sorted(rng.sample(range(n), 2))
        out += [f"H {q[0]}", f"RZZ {q[0]} {q[1]} {rng.uniform(-3, 3)!r}", f"RX {b} {rng.uniform(-3, 3)!r}"]
    return "\n".join(out) + "\n"


def pairs_of(kind, n):
    rng = random.Random(n)
    if kind == "one":
        return [(0, n - 1)]
    if kind == "reversal":
        return [(i, n - 1 - i) for i in range(n // 2)]
    if kind == "cycle":
        return [(i, i + 1) for i in range(n - 1)]
    if kind == "back":
        return [(1, n - 2), (0, 3), (0, 3), (1, n - 2)]
    return [tuple(rng.sample(range(n), 2)) for _ in range(n)]


KINDS = ["one", "reversal", "cycle", "back", "random"]


@pytest.mark.parametrize("dtype,n", [("c128", 13), ("c64", 14)])
def test_in_bounds(emul, tmp_path, dtype, n):
    for kind in KINDS:   # addresses only: the tile crosses threads
        run_case(emul, tmp_path, "plain", n, 4, dtype, swap_circuit(n, pairs_of(kind, n), 3), seed=n, lane_moves=3)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("dtype,n", [("c128", 11), ("c64", 12), ("c128", 14), ("c64", 15), ("c128", 17), ("c64", 18)])
def test_plain_list(dtype, n, kind):
    text = swap_circuit(n, pairs_of(kind, n), n)
    s0 = sq.gen_state(n, n)
    want = Oracle().run(s0, n, text)
    gates, _, ng, _ = sq.parse_circuit(text, n)
    for call in ("apply_gates", "apply_gates_noalloc"):
        eng = sq.Engine(n, dtype=dtype)
        ptr = eng.device_state()[0]
        eng.set_state(s0)
        getattr(eng, call)(gates, ng)
        assert eng.device_state()[0] == ptr   # the state keeps its address
        assert np.max(np.abs(eng.get_state() - want)) <= TOL[dtype]
        eng.close()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["c128", "c64"])
def test_subcircuit_file_with_swap_gates(dtype):
    n, chunk = 14, 8
    text = sq.plan(swap_circuit(n, pairs_of("random", n), 5), n, 0, chunk)
    assert "VSWAP" in text and "\nSWAP" in text
    s0 = sq.gen_state(n, 1)
    want = Oracle().run(s0, n, text, chunk=chunk, sub=True)
    eng = sq.Engine(n, dtype=dtype, chunk=chunk)
    eng.set_state(s0)
    gates, blocks, _, nb = sq.parse_circuit(text, n, is_subcircuit=True)
    eng.apply_blocks(gates, blocks, nb)
    assert np.max(np.abs(eng.get_state() - want)) <= TOL[dtype]
    eng.close()
