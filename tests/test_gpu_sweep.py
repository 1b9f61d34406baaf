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
