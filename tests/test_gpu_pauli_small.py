"""Pauli sums of states small enough for one workgroup (k_pauli_small) and the
sizes just past it: 12 and 13 qubits, 128 and 129 terms, 16 terms of 12 qubits
(the most work of one launch) and 17, every letter and power of i.  Against the
oracle at 1e-12 (complex128) and 1e-6 (complex64, summed in double) of the sum
of the coefficients' magnitudes."""
import numpy as np
import pytest

from conftest import random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n,count", [(1, 1), (1, 5), (2, 9), (5, 31), (6, 128), (9, 128), (9, 129), (10, 64),
                                     (10, 65), (11, 33), (12, 16), (12, 17), (13, 3)])
def test_pauli_sum_matches_oracle(oracle, dtype, n, count):
    from lightning_unification_amd import capi
    from lightning_unification_amd.circuits import Obs, pauli_word
    rs = np.random.default_rng(100 * n + count)
    words, coeffs = [], rs.normal(size=count).tolist()
    for _ in range(count):
        wt = int(rs.integers(1, n + 1))
        letters = "".join("XYZ"[int(rs.integers(3))] for _ in range(wt))
        words.append(pauli_word(letters, rs.choice(n, wt, replace=False).tolist()))
    ham = words[0] if count == 1 else Obs.hamiltonian(coeffs, words)
    s = random_state(n, n, dtype)
    exp = oracle.expval(s.astype(np.complex128), ham)
    tol = (1e-12 if dtype == np.complex128 else 1e-6) * max(1.0, np.abs(coeffs).sum())
    print(f"pauli n={n} terms={count} {np.dtype(dtype).name}", flush=True)
    with capi.DeviceStateVector.from_array(s) as sv:
        for _ in range(2):
            assert abs(sv.expval(ham) - exp) < tol
