"""The backward sweep's tile passes (kernels_adjoint.hpp, sweep.hpp) where their
geometry changes: states smaller than a tile, one per number of wavefronts a
tile, several tiles and passes, two observables a workgroup, operations wider
than a step, wide parities, controls outside the tile, and runs that merge.
Jacobian and VJP against the oracle at 1e-12 (complex128, the parity contract)
and 5e-5 (complex64, as the other adjoint tests)."""
import numpy as np
import pytest

from conftest import random_state, rel_err
from lightning_unification_amd.circuits import Obs, Tape, pauli_word
from lightning_unification_amd.gates import GATE_ID, GATE_NPARAMS, GATE_WIRES
from test_gpu_adjoint import FIXED_GATES, PARAM_GATES

pytestmark = pytest.mark.gpu


def mixed_tape(n, nops, rs, wide=True):
    """Any gate that fits n wires; MultiRZ on up to n; now and then a run of
    gates on the wires just used, so that steps merge."""
    tape, last = Tape(), None
    for _ in range(nops):
        pool = PARAM_GATES if rs.uniform() < 0.7 else FIXED_GATES
        pool = [g for g in pool if (1 if GATE_WIRES[GATE_ID[g]] == -1 else GATE_WIRES[GATE_ID[g]]) <= n
                and (wide or "Double" not in g)]
        g = pool[rs.integers(len(pool))]
        k = GATE_WIRES[GATE_ID[g]]
        k = int(rs.integers(1, n + 1)) if k == -1 else k
        w = rs.choice(n, k, replace=False).tolist()
        if last and len(last) >= k and rs.uniform() < 0.4:
            w = last[:k]
        last = w
        tape.add(g, w, rs.uniform(0, 6.3, GATE_NPARAMS[GATE_ID[g]]), bool(rs.integers(2)))
    return tape


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n,nops,nobs", [(1, 12, 1), (2, 20, 2), (3, 30, 3), (8, 40, 2), (9, 60, 5), (10, 60, 1),
                                         (11, 80, 3), (12, 80, 4), (14, 120, 2), (18, 60, 1), (20, 24, 5)])
def test_sweep_geometries(oracle, dtype, n, nops, nobs):
    from lightning_unification_amd import capi
    rs = np.random.default_rng(100 * n + nobs)
    tape = mixed_tape(n, nops, rs, wide=n < 18)
    s = random_state(n, n, dtype)
    oracle.apply_tape(s, tape)
    obs = [Obs.named("PauliZ", [int(rs.integers(n))]) for _ in range(nobs)]
    if n > 1:
        obs[0] = pauli_word("XY", rs.choice(n, 2, replace=False).tolist())
    npar = tape.num_params()
    tp = sorted(rs.choice(npar, max(1, npar - 3), replace=False).tolist())
    tol = 1e-12 if dtype == np.complex128 else 5e-5
    s128 = s.astype(np.complex128)
    dy = random_state(n, n + 1, dtype)
    print(f"sweep n={n} {np.dtype(dtype).name}", flush=True)
    with capi.DeviceStateVector.from_array(s) as sv:
        assert rel_err(sv.adjoint_jacobian(tape, obs, tp), oracle.adjoint(s128, tape, obs, tp)) < tol
        assert rel_err(sv.vjp(tape, dy, tp), oracle.vjp(s128, tape, dy.astype(np.complex128), tp)) < tol
        assert np.array_equal(sv.state(), s)  # the state is not modified


def test_more_trainable_steps_than_a_pass_has_slots(oracle):
    """IsingZZ phases neither merge nor need tile bits: one pass could hold
    them all, so the slot limit splits it."""
    from lightning_unification_amd import capi
    n = 6
    tape = Tape()
    for layer in range(12):
        for a in range(n):
            tape.add("IsingZZ", [a, (a + 1 + layer % 4) % n], [0.1 + 0.01 * (layer * n + a)])
            tape.add("CRX", [a, (a + 2) % n], [0.2 + 0.01 * (layer * n + a)])
    s = random_state(n, 3)
    oracle.apply_tape(s, tape)
    tp = list(range(tape.num_params()))
    obs = [pauli_word("XX", [0, 3]), Obs.named("PauliY", [5])]
    with capi.DeviceStateVector.from_array(s) as sv:
        assert rel_err(sv.adjoint_jacobian(tape, obs, tp), oracle.adjoint(s, tape, obs, tp)) < 1e-12


def _wide_tape(n, nops, seed):
    """Entangled, with a parametrised gate in every step."""
    rs, tape = np.random.default_rng(seed), Tape()
    for i in range(nops):
        a, b = rs.choice(n, 2, replace=False).tolist()
        g = ["CRX", "IsingXX", "CRZ", "CRY"][i % 4]
        tape.add(g, [a, b], [0.2 + 0.1 * i])
    return tape


def _adjoint_pairwise(oracle, lam, tape, words):
    """The Jacobian of Pauli words (letters, wires), one parameter an operation,
    summed pairwise: at 2^23 coherent terms the oracle's running sum is 1e-11 off."""
    def gates(ops):
        t = Tape()
        for op in ops:
            t.add(*op)
        return t

    hs = []
    for letters, wires in words:
        hs.append(lam.copy())
        oracle.apply_tape(hs[-1], gates([("Pauli" + a, [w]) for a, w in zip(letters, wires)]))
    lam, jac = lam.copy(), np.zeros((len(words), len(tape.ops)))
    for i in reversed(range(len(tape.ops))):
        name, wires, _, params = tape.ops[i]
        mu = lam.copy()
        scale = oracle.apply_generator(mu, name, wires)
        jac[:, i] = [-2 * scale * np.sum(np.conj(h) * mu).imag for h in hs]
        for v in [lam] + hs:
            oracle.apply_tape(v, gates([(name, wires, params, True)]))
    return jac


@pytest.mark.parametrize("dtype,n", [(np.complex128, 23), (np.complex64, 24)])
def test_groups_of_a_large_state_one_by_one(oracle, dtype, n):
    """Past 64 MiB a state has one lambda: each group of observables is swept
    from it and the last one writes it.  Three and five observables, in pairs
    with one left over, over several passes, on a state whose wires all differ."""
    from lightning_unification_amd import capi
    prep, tape = Tape(), _wide_tape(n, 8, 5)
    for w in range(n):
        prep.add("RY", [w], [0.4 + 0.1 * w])
        prep.add("RZ", [w], [0.3 * w])
    s = np.zeros(1 << n, np.complex128)
    s[0] = 1
    oracle.apply_tape(s, prep)
    oracle.apply_tape(s, tape)
    used = [w for op in tape.ops for w in op[1]]
    words = [("Z", [used[1]]), ("XZ", [used[2], used[5]]), ("Y", [used[7]]), ("X", [used[9]]),
             ("YX", [used[12], used[15]])]
    exp = _adjoint_pairwise(oracle, s, tape, words)
    assert np.sum(np.abs(exp) > 1e-3) >= 5  # something to compare
    tol = 1e-12 if dtype == np.complex128 else 5e-5
    print(f"group by group: n={n} {np.dtype(dtype).name}", flush=True)
    obs = [pauli_word(letters, wires) for letters, wires in words]
    with capi.DeviceStateVector.from_array(s.astype(dtype)) as sv:
        for k in (3, 5):
            assert np.max(np.abs(sv.adjoint_jacobian(tape, obs[:k], list(range(8))) - exp[:k])) < tol


def test_partial_sums_are_added_up_during_the_sweep(oracle):
    """More trainable steps than the partial sums of 64 observables have room
    for at once."""
    from lightning_unification_amd import capi
    n = 16
    tape = _wide_tape(n, 100, 8)
    s = random_state(n, 4)
    oracle.apply_tape(s, tape)
    obs = [Obs.named("PauliZ", [k % n]) if k < n else pauli_word("XY", [k % n, (k + 1 + k // n) % n])
           for k in range(64)]
    with capi.DeviceStateVector.from_array(s) as sv:
        assert rel_err(sv.adjoint_jacobian(tape, obs, list(range(100))),
                       oracle.adjoint(s, tape, obs, list(range(100)))) < 1e-12
