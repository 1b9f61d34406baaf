"""Tapes as passes on register tiles (kernels_pass.hpp, the path of pl_sv_apply_ops
and of the default tiles) where their geometry changes: states smaller than a
tile, one per number of wavefronts a tile, several tiles and passes, every gate
form (pairs in one bit, two and four, phases, parities over bits outside the
tile, controls there, operations no step holds).  Against the oracle at 1e-12
(complex128) and 2e-5 (complex64, the gates' tolerance)."""
import numpy as np
import pytest

from conftest import random_state, rel_err
from lightning_unification_amd.circuits import Tape, random_layers
from test_gpu_sweep import mixed_tape

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n,nops", [(1, 9), (2, 20), (3, 30), (5, 60), (9, 80), (10, 80), (11, 80), (12, 80),
                                    (13, 100), (14, 120), (17, 120), (20, 60)])
def test_passes_match_oracle(oracle, dtype, n, nops):
    from lightning_unification_amd import capi
    rs = np.random.default_rng(n)
    tape = mixed_tape(n, nops, rs)
    for op in random_layers(n, 2, seed=n).ops if n > 2 else []:
        tape.ops.append(op)
    s = random_state(n, n, dtype)
    tol = 1e-12 if dtype == np.complex128 else 2e-5
    print(f"passes n={n} {np.dtype(dtype).name}", flush=True)
    with capi.DeviceStateVector.from_array(s) as sv, capi.DeviceStateVector.from_array(s) as tiled:
        sv.apply_tape(tape)
        tiled.apply_tape_tiled(tape)
        exp = s.copy()
        oracle.apply_tape(exp, tape)
        assert rel_err(sv.state(), exp, floor=0.1) < tol
        assert rel_err(tiled.state(), exp, floor=0.1) < tol
        # a second tape right behind the first: the program buffer is reused
        sv.apply_tape(tape)
        oracle.apply_tape(exp, tape)
        assert rel_err(sv.state(), exp, floor=0.1) < 2 * tol


def test_gates_before_a_refused_one_are_applied(oracle):
    """As gate by gate: the operations before one that does not lower stand."""
    from lightning_unification_amd import capi
    n = 6
    good = mixed_tape(n, 12, np.random.default_rng(4))
    tape = Tape()
    tape.ops = list(good.ops) + [("RX", [n], False, [0.3])] + [("RY", [0], False, [0.4])]
    s = random_state(n, 8)
    exp = s.copy()
    oracle.apply_tape(exp, good)
    with capi.DeviceStateVector.from_array(s) as sv:
        with pytest.raises(ValueError):
            sv.apply_tape(tape)
        assert rel_err(sv.state(), exp, floor=0.1) < 1e-12


def test_four_bit_members_at_every_window(oracle):
    """Double excitations mix four bits: two directly, two through a CNOT frame."""
    from lightning_unification_amd import capi
    n = 13
    rs = np.random.default_rng(2)
    tape = Tape()
    for i in range(30):
        g = ["DoubleExcitation", "DoubleExcitationMinus", "DoubleExcitationPlus", "CSWAP", "SWAP"][i % 5]
        k = {"CSWAP": 3, "SWAP": 2}.get(g, 4)
        tape.add(g, rs.choice(n, k, replace=False).tolist(), [0.3 + i] if k == 4 else [], bool(i & 1))
    s = random_state(n, 5)
    exp = s.copy()
    oracle.apply_tape(exp, tape)
    with capi.DeviceStateVector.from_array(s) as sv:
        sv.apply_tape(tape)
        assert rel_err(sv.state(), exp, floor=0.1) < 1e-12


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n", [9, 14])
def test_default_tiles_refuse_a_tape_whole(dtype, n):
    """The tiled executor leaves the state alone where an operation cannot be
    applied, wherever it stands in the tape; a low-bit count out of range is
    refused, one in range is the tiles'."""
    from lightning_unification_amd import capi
    good = random_layers(n, 2, seed=4)
    s = random_state(n, 8, dtype)
    with capi.DeviceStateVector.from_array(s) as sv:
        for op in (("RX", [n], False, [0.3]), ("RX", [-1], False, [0.3]), ("CNOT", [1], False, [])):
            for at in (0, 5, len(good.ops)):
                tape = Tape()
                tape.ops = list(good.ops[:at]) + [op] + list(good.ops[at:])
                with pytest.raises(ValueError):
                    sv.apply_tape_tiled(tape)
                assert np.array_equal(sv.state(), s)
        with pytest.raises(ValueError):
            sv.apply_tape_tiled(good, 0, 7)
        assert np.array_equal(sv.state(), s)
        k = min(n, 11 if dtype == np.complex128 else 12)
        assert sv.apply_tape_tiled(good, 0, 2) == len(capi.tile_plan(n, good, k, 2))
