"""The ansatz entry's passes (k_hea) at every register width and with partial
last qubit sets, against the general adjoint on complex128 (other kernels)."""
import numpy as np
import pytest

import subquokka_dev_amd as sq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("every", [0, 1])
@pytest.mark.parametrize("dtype,n", [("c128", 6), ("c128", 7), ("c128", 9), ("c128", 13), ("c128", 17), ("c128", 18),
                                     ("c128", 20), ("c64", 7), ("c64", 8), ("c64", 11), ("c64", 19), ("c64", 21)])
def test_against_general_adjoint(dtype, n, every):
    layers = 3
    rng = np.random.default_rng(n)
    theta = rng.uniform(-np.pi, np.pi, 2 * n * layers)
    text = sq.gen_circuit("hea", n, layers, theta=theta)
    param, k = [], 0
    for line in text.splitlines():
        param.append(k if line[0] == "R" else -1)
        k += line[0] == "R"
    ref = sq.Engine(n, dtype="c128")
    want_e, want = ref.adjoint_grad(text, param, theta, [(1.0, [q, (q + 1) % n]) for q in range(n)])
    eng = sq.Engine(n, dtype=dtype)
    got_e, got = eng.adjoint_grad_hea(layers, theta, every)
    assert abs(eng.hea_energy(layers, theta) - got_e) <= 1e-12 * n
    tol = 1e-11 if dtype == "c128" else 1e-4
    assert abs(got_e - want_e) <= tol * n
    assert np.max(np.abs(got - want)) <= tol * max(1.0, np.max(np.abs(want)))
    ref.close()
    eng.close()
