"""Steps that go one by one because a pass would cost more (SweepCost): few on a
small state, and DoubleExcitations.  Every gate kind, alone and merged with
another of its place, forward through the per-gate kernels and backward through
k_sweep_step, at the counts where its instances and launches change (four and
eight states), against the oracle at 1e-12 (complex128; complex64 2e-5 forward
and 5e-5 backward, as the gates' and the adjoint's tests)."""
import numpy as np
import pytest

from conftest import random_state, rel_err
from lightning_unification_amd.circuits import Obs, Tape, pauli_word
from lightning_unification_amd.gates import GATE_ID, GATE_NAMES, GATE_NPARAMS, GATE_WIRES, GENERATOR_GATES

pytestmark = pytest.mark.gpu


def _gates(n, names, rs):
    tape = Tape()
    for g in names:
        k = GATE_WIRES[GATE_ID[g]]
        k = int(rs.integers(1, min(n, 6) + 1)) if k == -1 else k
        w = rs.choice(n, k, replace=False).tolist()
        for _ in range(1 + int(rs.integers(2))):  # some twice: one step
            tape.add(g, w, rs.uniform(-7, 7, GATE_NPARAMS[GATE_ID[g]]).tolist(), bool(rs.integers(2)))
    return tape


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n", [4, 11, 20])
def test_few_gates_match_oracle(oracle, dtype, n):
    from lightning_unification_amd import capi
    rs = np.random.default_rng(n)
    tol = 1e-12 if dtype == np.complex128 else 2e-5
    for g in GATE_NAMES:
        tape = _gates(n, [g] * 4, rs)
        while len(tape.ops) < 6:  # the shortest tape that is planned on a small state
            tape.ops += _gates(n, [g], rs).ops
        tape.ops = tape.ops[:6]
        s = random_state(n, GATE_ID[g], dtype)
        exp = oracle.apply_tape(s.astype(np.complex128), tape)
        with capi.DeviceStateVector.from_array(s) as sv:
            sv.apply_tape(tape)
            assert rel_err(sv.state(), exp, floor=0.1) < tol, g


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n,nobs", [(4, 1), (4, 9), (9, 4), (12, 5), (12, 8), (15, 3), (15, 17)])
def test_few_trainable_gates_match_oracle(oracle, dtype, n, nobs):
    from lightning_unification_amd import capi
    rs = np.random.default_rng(10 * n + nobs)
    tol = 1e-12 if dtype == np.complex128 else 5e-5
    obs = [pauli_word("XYZ"[k % 3], [k % n]) if k % 2 else Obs.named("PauliZ", [(5 * k) % n]) for k in range(nobs)]
    for g in GENERATOR_GATES:
        # the last gate is not trained, then one or two that are, then one that is not
        tape = _gates(n, ["CNOT", g, "CZ" if nobs % 2 else "SWAP"], rs)
        s = random_state(n, GATE_ID[g], dtype)
        oracle.apply_tape(s, tape)
        s128 = s.astype(np.complex128)
        dy = random_state(n, 3, dtype)
        tp = list(range(tape.num_params()))
        with capi.DeviceStateVector.from_array(s) as sv:
            assert rel_err(sv.adjoint_jacobian(tape, obs, tp), oracle.adjoint(s128, tape, obs, tp)) < tol, g
            assert rel_err(sv.vjp(tape, dy, tp), oracle.vjp(s128, tape, dy.astype(np.complex128), tp)) < tol, g
            assert np.array_equal(sv.state(), s)


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n,nobs", [(13, 2), (18, 12)])
def test_excitations_between_passes(oracle, dtype, n, nobs):
    """DoubleExcitations alone between passes of other gates."""
    from lightning_unification_amd import capi
    rs = np.random.default_rng(n)
    tape = Tape()
    for layer in range(3):
        for w in range(n):
            tape.add("RY", [w], [0.1 + w + layer])
            tape.add("CNOT", [w, (w + 1) % n])
        for _ in range(3):
            tape.add("DoubleExcitation", rs.choice(n, 4, replace=False).tolist(), [float(rs.uniform(0, 6))])
            tape.add("SingleExcitation", rs.choice(n, 2, replace=False).tolist(), [float(rs.uniform(0, 6))], True)
    s = random_state(n, 2, dtype)
    exp = oracle.apply_tape(s.astype(np.complex128), tape)
    obs = [Obs.named("PauliZ", [k]) for k in range(nobs)]
    tp = list(range(tape.num_params()))
    with capi.DeviceStateVector.from_array(s) as sv:
        sv.apply_tape(tape)
        assert rel_err(sv.state(), exp, floor=0.1) < (1e-12 if dtype == np.complex128 else 2e-5)
        got = sv.state()
        assert rel_err(sv.adjoint_jacobian(tape, obs, tp),
                       oracle.adjoint(got.astype(np.complex128), tape, obs, tp)) < (
                           1e-12 if dtype == np.complex128 else 5e-5)
